// prefill.hip - the chunked prefill's kernels on gfx950: the int4 linear for many rows on the
// matrix cores, the causal attention of a chunk over the KV cache, and the chunk's embedding
// gather.
//
// Replaces the reference's prefill walk (src/runtime/prefill/step.h step_chunk, Engine::prefill
// src/runtime/engine.h:97-115): per chunk of T positions, the embedding gather and first norm,
// then per layer q||k||v, attn_prep, the chunk's causal attention, o + residual + norm,
// gate||up + SiLU, down + residual + norm; the last position's head and argmax leave the control
// block as decode's ingest of the same ids would (cur_token = the argmax, pos advanced by T).
//
// gemm_w4a16_kernel, gemm_w4a16_few_kernel: out[T][N] fp32 = x[T][K] (f16) . W[K][N] (int4 GPTQ g64,
// layout 0). The contraction is a dense GEMM here (2 T K N flops over K N / 2 weight bytes):
// MFMA-bound from some hundred rows, bound by the weights' stream and its latency below.
//   * each wave has 16 RI rows x 64 columns = RI x 4 v_mfma_f32_16x16x32_f16 tiles; 4 waves side by
//     side make tiles of 16 RI x 256 (RI 4, 6 or 8: up to 128 rows per weight unpacked). Where a launch
//     would leave CUs with one such work-group or none, 8 waves split the k-groups of 16 .. 96 rows in
//     two parts, or (few rows) 8 waves split the k-groups of a 64-column tile (pick_gemm);
//   * one 64-deep k-group per iteration (one scale per column). The activations go through LDS,
//     double-buffered (the next group's rows are loaded into registers while the current group
//     is multiplied, then written to the other buffer). The weights skip LDS: a B fragment of
//     v_mfma_f32_16x16x32_f16 is 8 consecutive k of one column, which is exactly one int4 word,
//     so each lane loads its own words two groups ahead (16 bytes: one word of each of its four
//     column tiles) and unpacks them into the fragments, half a group at a time between the
//     products of the half before. Every load is unconditional and stays where it is written, so
//     the waits count exactly the loads that may still be in flight;
//   * w = f16((q - 8) * scale): q - 8 exact in f16 (the magic-number unpack of the decode GEMV),
//     one f16 rounding of the product (the reference's prefill rounds the same product to bf16,
//     pf_dequant_slab.cl); the activations are permuted to the unpack's pair order
//     (k0,k4)(k1,k5)(k2,k6)(k3,k7) inside each 8-k chunk, so the products pair up;
//   * fp32 accumulation in MFMA order, the k parts' sums added in ascending k. A column's order
//     therefore depends on the shape that the rule takes, that is on T, K and N.
// gate||up + SwiGLU 5120 -> 34816 at 2048 rows 739 -> 672 us (1.09 PFLOP/s; the library's plain f16 product
// of these sizes 1.17; the other sizes stand at pick_gemm): a product of the matrix cores takes twice its
// issue time even so, since the clock falls under it.
//
// attn_prefill_kernel: causal GQA attention of T query rows at positions pos0 .. pos0+T-1 over
// the cache rows [0, pos0 + t] (the chunk's own rows written by attn_prep before it), f16 or the
// rotated int8 form. A work-group takes one kv head and the rows whose (row, q head) pairs fill its
// matrix columns, 16 per tile; its waves walk the same keys, 32 per step, staged in LDS for all of
// them: S^T = K Q^T with q as f16 high + low parts, an online softmax per column in fp32, O^T += V^T
// P^T with P as f16 high + low parts, so the result is fp32-accurate attention; keys past a row's
// position are -inf. What bounds it is the matrix cores and the softmax's vector instructions in
// turn (two waves per SIMD overlap them in part), at rows of 256 also the LDS reads:
//   * both products are 16x16x32: P V takes two 16-key score tiles as one operand (the order of
//     its 32 keys is free), with V^T from LDS rows through the transposing reads;
//   * at rows of 128 a wave has two column tiles on one set of LDS reads (rows of 256: one, two
//     would leave one wave per SIMD: 777 rows over 3778 int8 keys 128 -> 200 us);
//   * a step's keys are loaded two iterations ahead into registers and written to the other LDS
//     buffer after the products: one barrier per iteration, no wait for the load's latency;
//   * the accumulators follow the running maximum only when it has risen by more than 2^8, the
//     f16 parts come from v_cvt_pk_f16_f32 and v_fma_mix_f32.
// Measured (MI355X, 40 / 8 heads of 128, 2048 rows): 180 -> 84 us, 510 TFLOP/s of attention products or 1.0 PFLOP/s
// with the low parts (45 % of the matrix cores' cycles at 2.4 GHz, counters); 16 / 2 heads of 256, int8, 777 rows at
// position 3001: 375 -> 129 us; one step per 16 keys on 16x16x16 products before.
#include <algorithm>
#include <string>

#include "mi_capi_internal.h"
#include "mi_common.h"

namespace mi {
namespace {

// ---------------------------------------------------------------------------------------------
// the int4 linear for many rows
// ---------------------------------------------------------------------------------------------
constexpr uint32_t GBK = 64;
constexpr uint32_t GPAD = 8;             // f16 of padding per LDS row (a 144-byte stride)
constexpr uint32_t GROW = GBK + GPAD;    // LDS row length in f16

// 8 natural-order activations (x0..x7 in four u32) into the unpack's pair order.
__device__ __forceinline__ u4_t perm_pairs(u4_t v) {
  return u4_t{__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
              __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u)};
}

// The unpack's masks and magic, in registers and opaque: (w & mask) | magic then is one v_and_or_b32
// (known literals would become two instructions), and unlike inline assembly the scheduler can
// place it between matrix products.
struct DqConst {
  uint32_t lo = 0x000F000Fu, hi = 0x00F000F0u, magic = 0x64006400u;
  __device__ __forceinline__ DqConst() { asm("" : "+s"(lo), "+s"(hi), "+v"(magic)); }
};

// f16((q_i - 8) * s) of one word's 8 nibbles, pair order (q0,q4)(q1,q5)(q2,q6)(q3,q7)
__device__ __forceinline__ u4_t dequant_scaled(uint32_t w, h2_t s2, const DqConst& c) {
  const h2_t b1032 = {(half_t)1032.0f, (half_t)1032.0f};
  const h2_t s16 = {(half_t)0.0625f, (half_t)0.0625f};
  const h2_t b72 = {(half_t)-72.0f, (half_t)-72.0f};
  const uint32_t t = w >> 8;
  const h2_t p0 = as_h2((w & c.lo) | c.magic) - b1032;                               // q - 8, exact
  const h2_t p1 = __builtin_elementwise_fma(as_h2((w & c.hi) | c.magic), s16, b72);  // exact
  const h2_t p2 = as_h2((t & c.lo) | c.magic) - b1032;
  const h2_t p3 = __builtin_elementwise_fma(as_h2((t & c.hi) | c.magic), s16, b72);
  return u4_t{h2_bits(p0 * s2), h2_bits(p1 * s2), h2_bits(p2 * s2), h2_bits(p3 * s2)};
}

// outputs are stored in pieces of several elements at the elements' own alignment
typedef f4_t f4_any __attribute__((aligned(4)));
typedef uint32_t h2_any __attribute__((aligned(2)));
typedef u2_t h4_any __attribute__((aligned(2)));
typedef u4_t h8_any __attribute__((aligned(2)));

// A wave's 64 columns: lane (fr, fq) = (l % 16, l / 16) reads word row fq of a half group's four at
// columns 4 fr .. 4 fr + 3 (one 16-byte load), and column 4 fr + j is column fr of the wave's matrix
// tile j: the B operand is the lane's own word, and the lane ends with four adjacent columns.
struct BGroup {
  u4_t w[2];  // k half ks: the word rows 4 ks + fq
  u2_t s;     // the four columns' scales
};
// the operands of k half ks: four tiles' fragments
__device__ __forceinline__ void dequant_half(const BGroup& b, uint32_t ks, const DqConst& c, h8_t (&bf)[4]) {
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    const uint32_t sj = j < 2 ? b.s.x : b.s.y;
    const h2_t s2 = as_h2(__builtin_amdgcn_perm(sj, sj, j & 1u ? 0x03020302u : 0x01000100u));
    bf[j] = __builtin_bit_cast(h8_t, dequant_scaled(b.w[ks][j], s2, c));
  }
}
// Fixes the place where operands are formed: ahead of the loads that refill the registers they come
// from. (Sunk past those loads, to the products, they would make the loads take other registers,
// and the copies back at the loop's end would wait for the loads.)
template <uint32_t N>
__device__ __forceinline__ void pin(h8_t (&f)[N]) {
#pragma unroll
  for (uint32_t j = 0; j < N; ++j) asm volatile("" : "+v"(f[j]));
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ uint32_t f16_pair(float x, float y) { return (uint32_t)f2h(x) | ((uint32_t)f2h(y) << 16); }

// The lane's four adjacent columns ncol .. + 3 of one row. SILU: the columns are gate||up in the
// interleave16 order, so a gate lane (fr & 4 == 0) and the lane four on hold the gate and the up
// values of the same four outputs; it writes h [T][N/2] f16 = rne(rne(silu(rne(g))) * rne(u)) (the
// arithmetic of prep_silu_mul, prep.cl:384) instead of the fp32 output. The two lanes swap a pair of f16
// values and form two outputs each: four on the gate lane alone would leave half the lanes idle in
// the exponentials and divisions (64 -> 20096 at 1868 rows, nearly all epilogue, 52 -> 37 us; 1088 ->
// 25344 at 1542 137 -> 115; 5120 -> 34816 at 2048 693 -> 659). Every lane of the row's 16 calls it; `store`: the row and column exist.
template <bool SILU>
__device__ __forceinline__ void store_row4(f4_t v, bool store, float* out, uint16_t* h_out, uint32_t row, uint32_t ncol,
                                           uint32_t N) {
  if constexpr (SILU) {
    const bool up = ncol & 16u;
    const uint32_t p01 = f16_pair(v[0], v[1]), p23 = f16_pair(v[2], v[3]);
    const uint32_t own = up ? p23 : p01, send = up ? p01 : p23;
    // (row_shl:4 into the gate lanes, row_shr:4 into the up lanes)
    const int from = __builtin_amdgcn_update_dpp(0, (int)send, 0x104, 0xF, 0x5, true);
    const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(from, (int)send, 0x114, 0xF, 0xA, true);
    const uint32_t g = up ? got : own, u = up ? own : got;
    const float s0 = h2f(f2h(silu_f32(h2f((uint16_t)g)))), s1 = h2f(f2h(silu_f32(h2f((uint16_t)(g >> 16)))));
    const uint32_t n = ncol / 32u * 16u + ncol % 16u + (up ? 2u : 0u);
    if (store)
      *reinterpret_cast<h2_any*>(h_out + (size_t)row * (N / 2) + n) = f16_pair(s0 * h2f((uint16_t)u), s1 * h2f((uint16_t)(u >> 16)));
  } else {
    if (store) *reinterpret_cast<f4_any*>(out + (size_t)row * N + ncol) = v;
  }
}

// Tile: 16 RI rows x 256 columns, 4 waves of 16 RI x 64 per K part. KS = 2: 8 waves, waves 4 .. 7 the
// second half of the k-groups, the halves added at the end through LDS. DA: k-groups of activations in
// flight in registers ahead of the one multiplied (of weights two). ODD: a part has an odd number of
// groups, the last of which follows the loop over pairs (a second group of zeros instead took a fifth
// of the time at K = 64, 5 % at 1344; a branch for it inside the loop costs the waits their exact
// counts, 3 to 10 % at K = 5120, and the code after the loop alone 3 % at 333 rows, hence a kernel each).
template <bool SILU, uint32_t RI, uint32_t KS, uint32_t DA, bool ODD>
__global__ __launch_bounds__(256 * KS, 2) void gemm_w4a16_kernel(const uint32_t* __restrict__ qweight,
                                                                 const uint16_t* __restrict__ scales,
                                                                 const uint16_t* __restrict__ x,
                                                                 float* __restrict__ out, uint16_t* __restrict__ h_out,
                                                                 uint32_t T, uint32_t K, uint32_t N) {
  constexpr uint32_t BM = 16u * RI, AI = (BM + 31u) / 32u;
  __shared__ __align__(16) union {
    uint16_t As[KS][2][BM][GROW];
    f4_t part[KS > 1 ? 4 : 1][RI][4][64];
  } sm;
  // (readfirstlane: the compiler then knows that a wave's part and column block are uniform)
  const uint32_t t = threadIdx.x % 256u, lane = t & 63u, wn = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t kp = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / 256u) : 0u;
  const uint32_t n0 = blockIdx.x * 256u, m0 = blockIdx.y * BM;
  const uint32_t fr = lane & 15u, fq = lane >> 4;
  const uint32_t G = K / GBK, n_it = (G + KS - 1u) / KS;  // this part's groups: g0 .. g1 - 1
  const uint32_t g0 = kp * n_it, g1 = min(G, g0 + n_it);
  const uint32_t ncol = n0 + 64u * wn + 4u * fr;
  const bool col_in = n0 + 64u * wn < N;  // uniform per wave: the last tile may hold 128 columns

  // activations, staged through LDS: thread t takes rows (t >> 3) + 32 i, 8-k chunk t & 7. Buffer
  // loads: 32-bit offsets keep the addresses out of 64-bit registers; the row sits in the
  // per-thread offset, so a row at or past T lies outside the resource's T K elements and reads 0
  const uint32_t a_row = t >> 3, a_chunk = t & 7u;
  const __amdgpu_buffer_rsrc_t x_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, T * K * 2u, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(qweight), 0, (K / 8u) * N * 4u, 0x00020000);
  const __amdgpu_buffer_rsrc_t s_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(scales), 0, (K / GBK) * N * 2u, 0x00020000);
  const uint32_t a_voff = ((m0 + a_row) * K + 8u * a_chunk) * 2u;
  const uint32_t wcol = col_in ? ncol : 4u * fr;  // (a wave past N reads its own tile's words of column 0 ..)
  const uint32_t w_voff = (fq * N + wcol) * 4u, s_voff = wcol * 2u;
  u4_t a_st[DA][AI];
  BGroup b_st[2];
  // (a group at or past the part's end takes offsets outside the resource: zeros, so the loop needs
  // no branch around its loads or products)
  auto past = [&](uint32_t g) { return g < g1 ? 0u : 0x80000000u; };
  auto load_a = [&](uint32_t g, u4_t (&st)[AI]) {
    const uint32_t o = past(g);
    g = min(g, G - 1u);
#pragma unroll
    for (uint32_t i = 0; i < AI; ++i)
      st[i] = __builtin_bit_cast(
          u4_t, __builtin_amdgcn_raw_buffer_load_b128(x_rs, (a_voff + 32u * i * K * 2u) | o, g * GBK * 2u, 0));
  };
  auto load_b = [&](uint32_t g, BGroup& b) {
    const uint32_t o = past(g);
    g = min(g, G - 1u);
#pragma unroll
    for (uint32_t ks = 0; ks < 2; ++ks)
      b.w[ks] = __builtin_bit_cast(u4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rs, w_voff | o, (8u * g + 4u * ks) * N * 4u, 2));
    b.s = __builtin_bit_cast(u2_t, __builtin_amdgcn_raw_buffer_load_b64(s_rs, s_voff | o, g * N * 2u, 0));
  };
  auto store_a = [&](uint32_t buf, const u4_t (&st)[AI]) {
#pragma unroll
    for (uint32_t i = 0; i < AI; ++i)
      if (32u * (i + 1u) <= BM || a_row + 32u * i < BM)
        *reinterpret_cast<u4_t*>(&sm.As[kp][buf][a_row + 32u * i][8u * a_chunk]) = perm_pairs(st[i]);
  };

  f4_t acc[RI][4];
#pragma unroll
  for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};

  // Each half group's products run with the next half's weights becoming fragments between them (two
  // vector instructions hide behind each product; as phases of their own the products and the
  // unpack would add up). A group's weight registers are refilled, two groups on, once its second
  // half is unpacked.
  const DqConst dq;
  h8_t bf[2][4];
  load_b(g0, b_st[0]);
#pragma unroll
  for (uint32_t u = 0; u < DA; ++u) load_a(g0 + u, a_st[u]);
  __builtin_amdgcn_sched_barrier(0);
  load_b(g0 + 1u, b_st[1]);
  store_a(0, a_st[0]);
  dequant_half(b_st[0], 0, dq, bf[0]);
  pin(bf[0]);
  lds_barrier();
  for (uint32_t it0 = 0; it0 + (ODD ? 1u : 0u) < n_it; it0 += 2u) {
#pragma unroll
    for (uint32_t u = 0; u < 2u; ++u) {
      const uint32_t g = g0 + it0 + u;
      load_a(g + DA, a_st[u % DA]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t ks = 0; ks < 2; ++ks) {
        h8_t af[RI];
#pragma unroll
        for (uint32_t i = 0; i < RI; ++i)
          af[i] = *reinterpret_cast<const h8_t*>(&sm.As[kp][u][16u * i + fr][32u * ks + 8u * fq]);
#pragma unroll
        for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf[ks][j], acc[i][j], 0, 0, 0);
        dequant_half(b_st[ks ? u ^ 1u : u], ks ^ 1u, dq, bf[ks ^ 1u]);
        pin(bf[ks ^ 1u]);
        if (ks == 0) load_b(g + 2u, b_st[u]);
      }
      store_a(u ^ 1u, a_st[(u + 1u) % DA]);  // the other buffer was last read before the previous barrier
      lds_barrier();
    }
  }
  if constexpr (ODD) {  // the last group
#pragma unroll
    for (uint32_t ks = 0; ks < 2; ++ks) {
      if (ks) {
        dequant_half(b_st[0], 1, dq, bf[1]);
        pin(bf[1]);
      }
#pragma unroll
      for (uint32_t i = 0; i < RI; ++i) {
        const h8_t af = *reinterpret_cast<const h8_t*>(&sm.As[kp][0][16u * i + fr][32u * ks + 8u * fq]);
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf[ks][j], acc[i][j], 0, 0, 0);
      }
    }
    if constexpr (KS > 1) lds_barrier();  // (the merge reuses the staged activations)
  }
  if constexpr (KS > 1) {  // the second half's sums through LDS (the staged activations are done with)
    if (kp) {
#pragma unroll
      for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) sm.part[wn][i][j][lane] = acc[i][j];
    }
    lds_barrier();
    if (kp) return;
#pragma unroll
    for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) acc[i][j] += sm.part[wn][i][j][lane];
  }
  // lane holds rows 4 fq + r of columns ncol .. + 3 of each 16-row tile
#pragma unroll
  for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      const uint32_t row = m0 + 16u * i + 4u * fq + r;
      store_row4<SILU>(f4_t{acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]}, row < T && col_in, out, h_out, row,
                       ncol, N);
    }
}

// Few rows: 16 RI rows x 64 columns per work-group, its KW waves taking a KW-th of the k-groups
// each. Nothing is shared, so there is no LDS staging and no barrier in the loop: a wave loads its
// weights and its activations (in the A operand's own layout, from L2) D groups ahead. The waves'
// sums are added through LDS in ascending k.
template <bool SILU, uint32_t RI, uint32_t KW, uint32_t D>
__global__ __launch_bounds__(64 * KW, 2) void gemm_w4a16_few_kernel(
    const uint32_t* __restrict__ qweight, const uint16_t* __restrict__ scales, const uint16_t* __restrict__ x,
    float* __restrict__ out, uint16_t* __restrict__ h_out, uint32_t T, uint32_t K, uint32_t N) {
  constexpr uint32_t BM = 16u * RI;
  __shared__ f4_t red[KW][BM][16];
  const uint32_t lane = threadIdx.x & 63u, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fr = lane & 15u,
                 fq = lane >> 4;
  const uint32_t n0 = blockIdx.x * 64u, m0 = blockIdx.y * BM, ncol = n0 + 4u * fr;
  const uint32_t G = K / GBK, g0 = w * G / KW, g1 = (w + 1u) * G / KW;
  const __amdgpu_buffer_rsrc_t x_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, T * K * 2u, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(qweight), 0, (K / 8u) * N * 4u, 0x00020000);
  const __amdgpu_buffer_rsrc_t s_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(scales), 0, (K / GBK) * N * 2u, 0x00020000);
  const uint32_t a_voff = ((m0 + fr) * K + 8u * fq) * 2u, w_voff = (fq * N + ncol) * 4u, s_voff = ncol * 2u;
  const DqConst dq;
  u4_t a_st[D][2][RI];
  BGroup b_st[D];
  auto load = [&](uint32_t g, uint32_t u) {
    g = min(g, G - 1u);
#pragma unroll
    for (uint32_t ks = 0; ks < 2; ++ks)
      b_st[u].w[ks] =
          __builtin_bit_cast(u4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rs, w_voff, (8u * g + 4u * ks) * N * 4u, 2));
    b_st[u].s = __builtin_bit_cast(u2_t, __builtin_amdgcn_raw_buffer_load_b64(s_rs, s_voff, g * N * 2u, 0));
#pragma unroll
    for (uint32_t ks = 0; ks < 2; ++ks)
#pragma unroll
      for (uint32_t i = 0; i < RI; ++i)
        a_st[u][ks][i] = __builtin_bit_cast(
            u4_t, __builtin_amdgcn_raw_buffer_load_b128(x_rs, a_voff + 32u * i * K, (g * GBK + 32u * ks) * 2u, 0));
  };
  f4_t acc[RI][4];
#pragma unroll
  for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (uint32_t u = 0; u < D; ++u) {
    load(g0 + u, u);
    __builtin_amdgcn_sched_barrier(0);  // in the loop's order (as in gemm_w4a16_kernel)
  }
  for (uint32_t g = g0; g < g1; g += D) {
#pragma unroll
    for (uint32_t u = 0; u < D; ++u) {
      h8_t bf[2][4], af[2][RI];
#pragma unroll
      for (uint32_t ks = 0; ks < 2; ++ks) dequant_half(b_st[u], ks, dq, bf[ks]);
#pragma unroll
      for (uint32_t ks = 0; ks < 2; ++ks)
#pragma unroll
        for (uint32_t i = 0; i < RI; ++i) af[ks][i] = __builtin_bit_cast(h8_t, perm_pairs(a_st[u][ks][i]));
#pragma unroll
      for (uint32_t ks = 0; ks < 2; ++ks) {
        pin(bf[ks]);
        pin(af[ks]);
      }
      load(g + u + D, u);
      if (g + u < g1) {  // uniform
#pragma unroll
        for (uint32_t ks = 0; ks < 2; ++ks)
#pragma unroll
          for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[ks][i], bf[ks][j], acc[i][j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r)
      red[w][16u * i + 4u * fq + r][fr] = f4_t{acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
  __syncthreads();
  // (the lanes of a wave take 16 adjacent pieces of four rows at a time: BM * 16 pieces in all)
  for (uint32_t e = threadIdx.x; e < BM * 16u; e += 64u * KW) {
    const uint32_t row = e / 16u, c = e % 16u;
    f4_t v = red[0][row][c];
#pragma unroll
    for (uint32_t q = 1; q < KW; ++q) v += red[q][row][c];
    store_row4<SILU>(v, m0 + row < T, out, h_out, m0 + row, n0 + 4u * c, N);
  }
}

// ---------------------------------------------------------------------------------------------
// the chunk's MoE block, grouped by expert
// ---------------------------------------------------------------------------------------------
// The decode kernels take one row at a time through every expert it routes to, which for a
// chunk reads each expert's weights once per routed row. Here the chunk's (row, slot) pairs are
// grouped by expert first (moe_group_kernel), so each expert's weights stream once per 32, 64 or
// 96 of its pairs through the MFMA tile of gemm_w4a16_kernel (moe_gemm_kernel: layout-1 weights,
// gathered activation rows, scattered outputs), and the slot-ordered combine with the residual
// (moe.cl:383-470's epilogue, moe_ref.h:144-152) runs per row afterwards.
constexpr uint32_t kMoeRouteWords = 32, kMoeW = 8, kMoeSG = 16;  // the route row (moe.cl:49-56)
constexpr uint32_t kMoeTile = 136;                                 // layout 1: 128 words + 16 f16 scales
constexpr uint32_t kMoeMaxPairs = 2048u * 9u;                      // T <= 2048, top_k <= 8

// One work-group, a stable counting sort of the pairs p = t (top_k + 1) + s of T rows by expert:
// expert e's pairs go to list[off_e ..] in ascending p (the reference's (token, slot) order), its
// row tiles to tiles[] as {e, first list index, pair count}, the tile count to tiles_n[0]. Wave w (of
// 16) owns the pairs [w Q, (w + 1) Q): it counts them per expert, then places them 64 at a time, a
// lane's rank among the lanes of its expert coming from a match mask built from 9 ballots (one per
// bit of the expert index), so list[] is the same on every call. Latency-bound (2048 rows x 9 pairs):
// 31 us with the offsets summed by one thread and a division per pair, 22 now.
__global__ __launch_bounds__(1024) void moe_group_kernel(const uint32_t* __restrict__ route, uint32_t T,
                                                        uint32_t E, uint32_t top_k, uint32_t tile_rows,
                                                        uint32_t* __restrict__ list,
                                                        u4_t* __restrict__ tiles, uint32_t* __restrict__ tiles_n) {
  __shared__ uint16_t s_ex[kMoeMaxPairs];
  constexpr uint32_t kW = 16, kT = kW * 64;
  __shared__ uint32_t s_wc[kW][257], s_off[257], s_toff[257], s_cnt[257], s_wsum[kW][2];
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6, slots = top_k + 1, P = T * slots;
  for (uint32_t e = t; e <= E; e += kT)
    for (uint32_t w = 0; w < kW; ++w) s_wc[w][e] = 0;
  for (uint32_t r = t; r < T; r += kT) {  // a thread per row, its ids' loads together
    uint32_t id[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) id[k] = route[(size_t)r * kMoeRouteWords + k];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k)
      if (k < top_k) s_ex[r * slots + k] = (uint16_t)min(id[k], E);  // (an id outside [0, E): the shared expert)
    s_ex[r * slots + top_k] = (uint16_t)E;
  }
  __syncthreads();
  const uint32_t Q = (P + kW - 1u) / kW, lo = min(P, wave * Q), hi = min(P, lo + Q);
  for (uint32_t p = lo + lane; p < hi; p += 64u) atomicAdd(&s_wc[wave][s_ex[p]], 1u);  // counts only
  __syncthreads();
  // the experts' first list indices and tiles: exclusive sums over the experts, thread e expert e
  // (the lanes of a wave by shuffles, then the waves before it; E <= 256 < kT)
  uint32_t c = 0;
  if (t <= E)
    for (uint32_t w = 0; w < kW; ++w) c += s_wc[w][t];
  const uint32_t ct = (c + tile_rows - 1u) / tile_rows;
  uint32_t o = c, to = ct;
#pragma unroll
  for (uint32_t d = 1; d < 64u; d *= 2) {
    const uint32_t po = __shfl_up(o, d, 64), pt = __shfl_up(to, d, 64);
    if (lane >= d) {
      o += po;
      to += pt;
    }
  }
  if (lane == 63u) {
    s_wsum[wave][0] = o;
    s_wsum[wave][1] = to;
  }
  __syncthreads();
  for (uint32_t w = 0; w < wave; ++w) {
    o += s_wsum[w][0];
    to += s_wsum[w][1];
  }
  if (t <= E) {
    s_cnt[t] = c;
    s_off[t] = o - c;
    s_toff[t] = to - ct;
  }
  if (t == E) tiles_n[0] = to;
  __syncthreads();
  for (uint32_t e = t; e <= E; e += kT) {  // s_wc becomes each wave's next list index per expert
    uint32_t b = s_off[e];
    for (uint32_t w = 0; w < kW; ++w) {
      const uint32_t c = s_wc[w][e];
      s_wc[w][e] = b;
      b += c;
    }
  }
  __syncthreads();
  const uint64_t below = lane ? (~0ull >> (64u - lane)) : 0ull;
  for (uint32_t p0 = lo; p0 < hi; p0 += 64u) {
    const uint32_t p = p0 + lane;
    const bool valid = p < hi;
    const uint32_t e = valid ? s_ex[p] : 511u;  // 511: no expert index (E <= 256)
    uint64_t same = __ballot(valid);
#pragma unroll
    for (uint32_t b = 0; b < 9u; ++b) {
      const uint64_t bal = __ballot((e >> b) & 1u);
      same &= ((e >> b) & 1u) ? bal : ~bal;
    }
    const uint32_t rank = (uint32_t)__popcll(same & below);
    const uint32_t base = valid ? s_wc[wave][e] : 0u;
    if (valid) list[base + rank] = p;
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0) s_wc[wave][e] = base + (uint32_t)__popcll(same);
    __builtin_amdgcn_wave_barrier();
  }
  for (uint32_t e = t; e <= E; e += kT) {
    const uint32_t n = s_cnt[e];
    for (uint32_t k = 0; k * tile_rows < n; ++k)
      tiles[s_toff[e] + k] = u4_t{e, s_off[e] + k * tile_rows, min(tile_rows, n - k * tile_rows), 0u};
  }
}

// out rows = pairs of one expert (a row tile) x that expert's layout-1 block (K x N, columns in
// 16-column tiles of 64-k groups: word j of the group's tile holds k 8 j .. 8 j + 7 of column c
// at j 16 + c, its f16 scale at half-word 256 + c). A row of a pair p is row p / slots of x
// (GATE_UP) or row p of h (down). GATE_UP: N = 2 inter in interleave16 order, SwiGLU in the
// epilogue into h[p][inter] (the dense GEMM's epilogue); down: d[p][N] rounded to f16 (the
// combine's first rounding of a slot's value, so nothing is lost). Tile: up to 96 pairs x 256
// columns, 4 waves side by side, the dense GEMM's loop for the tile's 16-row blocks (1 .. 6, uniform):
// at top 8 of 256 experts a 2048-row chunk has 64 +- 8 pairs per expert, one tile of 4 or 5 blocks,
// where tiles of 64 rows took a second, nearly empty one for half of the experts. Bound by the
// products and the weights' latency (77 + 39 GFLOP over 428 MB there): gate||up 166 -> 135 us, down
// 98 -> 85 at 2048 rows; 512 rows: the block 230 -> 178.
struct MoeGemm {
  const u4_t* tiles;
  const uint32_t *tiles_n, *list, *blocks;
  const uint16_t* a;
  uint16_t *h_out, *d_out;
  size_t block_u32;
  uint32_t a_rows, slots, K, N;
};

template <bool GATE_UP, uint32_t RI, uint32_t ROWS>
__device__ __forceinline__ void moe_gemm_tile(const MoeGemm& m, const u4_t& tile, uint16_t (&As)[2][ROWS][GROW]) {
  constexpr uint32_t BM = 16u * RI, AI = (BM + 31u) / 32u;
  const uint32_t e = tile.x, first = tile.y, cnt = tile.z, K = m.K, N = m.N, G = K / GBK;
  const uint32_t t = threadIdx.x, lane = t & 63u, wn = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t fr = lane & 15u, fq = lane >> 4, n0 = blockIdx.x * 256u + 64u * wn;

  // activations: thread t stages pairs (t >> 3) + 32 i, 8-k chunk t & 7; a pair past the tile's
  // count gets an offset outside the resource and reads zeros
  const uint32_t a_row = t >> 3, a_chunk = t & 7u;
  const __amdgpu_buffer_rsrc_t x_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(m.a), 0, m.a_rows * K * 2u, 0x00020000);
  uint32_t a_voff[AI];
#pragma unroll
  for (uint32_t i = 0; i < AI; ++i) {
    const uint32_t r = a_row + 32u * i, p = m.list[first + min(r, cnt - 1u)];
    a_voff[i] = r < cnt ? ((GATE_UP ? p / m.slots : p) * K + 8u * a_chunk) * 2u : 0x80000000u;
  }
  // weights: lane (fr, fq) takes columns n0 + 4 fr .. + 3 (as in the dense GEMM): 16-column tile
  // fr / 4 of the wave's four, word row fq of a half group's, its columns 4 (fr % 4) ..
  const __amdgpu_buffer_rsrc_t w_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(m.blocks + (size_t)e * m.block_u32), 0, (uint32_t)(m.block_u32 * 4u), 0x00020000);
  const uint32_t t_voff = (fr >> 2) * G * kMoeTile * 4u, w_voff = t_voff + (fq * 16u + 4u * (fr & 3u)) * 4u;
  const uint32_t s_voff = t_voff + (256u + 4u * (fr & 3u)) * 2u, base = n0 / 16u * G * kMoeTile * 4u;
  u4_t a_st[AI];
  BGroup b_st[2];
  auto load_a = [&](uint32_t g) {  // (a group past the last re-reads it and is not multiplied)
    const uint32_t so = min(g, G - 1u) * GBK * 2u;
#pragma unroll
    for (uint32_t i = 0; i < AI; ++i)
      a_st[i] = __builtin_bit_cast(u4_t, __builtin_amdgcn_raw_buffer_load_b128(x_rs, a_voff[i], so, 0));
  };
  auto load_b = [&](uint32_t g, BGroup& b) {
    const uint32_t so = base + min(g, G - 1u) * kMoeTile * 4u;
#pragma unroll
    for (uint32_t ks = 0; ks < 2; ++ks)
      b.w[ks] = __builtin_bit_cast(u4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rs, w_voff, so + 256u * ks, 2));
    b.s = __builtin_bit_cast(u2_t, __builtin_amdgcn_raw_buffer_load_b64(w_rs, s_voff, so, 0));
  };
  auto store_a = [&](uint32_t buf) {
#pragma unroll
    for (uint32_t i = 0; i < AI; ++i)
      if (32u * (i + 1u) <= BM || a_row + 32u * i < BM)
        *reinterpret_cast<u4_t*>(&As[buf][a_row + 32u * i][8u * a_chunk]) = perm_pairs(a_st[i]);
  };

  f4_t acc[RI][4];
#pragma unroll
  for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
  const DqConst dq;
  h8_t bf[2][4];
  load_b(0, b_st[0]);
  load_a(0);
  __builtin_amdgcn_sched_barrier(0);
  load_b(1, b_st[1]);
  store_a(0);
  dequant_half(b_st[0], 0, dq, bf[0]);
  pin(bf[0]);
  lds_barrier();
  // (G is even: hidden a multiple of 512, inter of 128)
  for (uint32_t g0 = 0; g0 < G; g0 += 2u) {
#pragma unroll
    for (uint32_t u = 0; u < 2u; ++u) {
      const uint32_t g = g0 + u;
      load_a(g + 1u);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t ks = 0; ks < 2; ++ks) {
        h8_t af[RI];
#pragma unroll
        for (uint32_t i = 0; i < RI; ++i)
          af[i] = *reinterpret_cast<const h8_t*>(&As[u][16u * i + fr][32u * ks + 8u * fq]);
#pragma unroll
        for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf[ks][j], acc[i][j], 0, 0, 0);
        dequant_half(b_st[ks ? u ^ 1u : u], ks ^ 1u, dq, bf[ks ^ 1u]);
        pin(bf[ks ^ 1u]);
        if (ks == 0) load_b(g + 2u, b_st[u]);
      }
      store_a(u ^ 1u);
      lds_barrier();
    }
  }
  // lane holds pairs 4 fq + r of columns n0 + 4 fr .. + 3 of each 16-row block
#pragma unroll
  for (uint32_t i = 0; i < RI; ++i)
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      const uint32_t q = 16u * i + 4u * fq + r, p = m.list[first + min(q, cnt - 1u)];
      const f4_t v = {acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
      if constexpr (GATE_UP) {
        store_row4<true>(v, q < cnt, nullptr, m.h_out, p, n0 + 4u * fr, N);
      } else if (q < cnt) {
        *reinterpret_cast<h4_any*>(m.d_out + (size_t)p * N + n0 + 4u * fr) =
            u2_t{(uint32_t)f2h(v[0]) | ((uint32_t)f2h(v[1]) << 16), (uint32_t)f2h(v[2]) | ((uint32_t)f2h(v[3]) << 16)};
      }
    }
}

// RMAX: the most 16-row blocks of a work-group's tile. Its registers set the waves in flight, so
// few pairs per expert, where the weights' stream is the bound, take RMAX 2: half of a 64-row tile
// per work-group (grid z), five waves per SIMD.
template <bool GATE_UP, uint32_t RMAX>
__global__ __launch_bounds__(256, RMAX == 2 ? 4 : RMAX == 4 ? 3 : 2) void moe_gemm_kernel(MoeGemm m) {
  __shared__ __align__(16) uint16_t As[2][16u * RMAX][GROW];
  if (blockIdx.y >= m.tiles_n[0]) return;  // uniform: the grid is sized for the most tiles
  u4_t tile = m.tiles[blockIdx.y];
  if constexpr (RMAX == 2) {
    const uint32_t skip = 32u * blockIdx.z;
    if (skip >= tile.z) return;
    tile.y += skip;
    tile.z = min(32u, tile.z - skip);
  }
  const uint32_t ri = (tile.z + 15u) / 16u;
  if (ri == 1u) moe_gemm_tile<GATE_UP, 1>(m, tile, As);
  else if (RMAX == 2 || ri == 2u) moe_gemm_tile<GATE_UP, 2>(m, tile, As);
  if constexpr (RMAX > 2) {
    if (ri == 3u) moe_gemm_tile<GATE_UP, 3>(m, tile, As);
    else if (ri == 4u) moe_gemm_tile<GATE_UP, 4>(m, tile, As);
  }
  if constexpr (RMAX > 4) {
    if (ri == 5u) moe_gemm_tile<GATE_UP, 5>(m, tile, As);
    else if (ri > 5u) moe_gemm_tile<GATE_UP, 6>(m, tile, As);
  }
}

// resid[t][n] += the slot-ordered combine of row t's pair outputs (moe_down_kernel's epilogue,
// moe_ref.h:144-152): sum_k rne(rne(d_k) w_k) in slot order, + rne(rne(d_shared) s)
// Eight columns per thread, the slots' pieces loaded together: bound by the pair outputs' bytes
// (2048 rows x 9 x 2048: 75 MB; 16 us, 30 with a column per thread).
__global__ __launch_bounds__(256) void moe_combine_kernel(const uint32_t* __restrict__ route,
                                                          const uint16_t* __restrict__ d, uint16_t* __restrict__ resid,
                                                          uint32_t T, uint32_t top_k, uint32_t hidden) {
  const uint32_t h8 = hidden / 8u, i = blockIdx.x * 256u + threadIdx.x, t = i / h8, n = 8u * (i - t * h8);
  if (t >= T) return;
  const uint32_t* row = route + (size_t)t * kMoeRouteWords;
  const uint32_t slots = top_k + 1;
  const uint16_t* dp = d + (size_t)t * slots * hidden + n;
  h8_any* rp = reinterpret_cast<h8_any*>(resid + (size_t)t * hidden + n);
  u4_t v[9];
#pragma unroll
  for (uint32_t k = 0; k < 9; ++k) v[k] = *reinterpret_cast<const h8_any*>(dp + (size_t)min(k, top_k) * hidden);
  const u4_t rv = *rp;
  float wk[8];
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) wk[k] = __builtin_bit_cast(float, row[kMoeW + k]);
  const float sg = __builtin_bit_cast(float, row[kMoeSG]);
  u4_t o;
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q) {
    uint32_t half[2];
#pragma unroll
    for (uint32_t c = 0; c < 2; ++c) {
      auto at = [&](const u4_t& u) { return h2f((uint16_t)(u[q] >> (16u * c))); };
      float sum = 0.f;
#pragma unroll
      for (uint32_t k = 0; k < 8; ++k)
        if (k < top_k) sum += h2f(f2h(at(v[k]) * wk[k]));
      // (v[8]: slot top_k, as every piece from top_k on)
      const uint16_t r_b = f2h(sum), sh_b = f2h(at(v[8]) * sg);
      const uint16_t o_b = f2h(h2f(r_b) + h2f(sh_b));
      half[c] = f2h(at(rv) + h2f(o_b));
    }
    o[q] = half[0] | (half[1] << 16);
  }
  *rp = o;
}

// ---------------------------------------------------------------------------------------------
// the chunk's causal attention
// ---------------------------------------------------------------------------------------------

struct PrefillAttnArgs {
  const float* attn_q;  // [T][q_heads][HD] fp32
  const void* kv_k;     // f16, or int8 (KV8)
  const void* kv_v;
  const uint32_t* pages;
  uint16_t* attn_out;   // [T][q_heads * HD] f16
  size_t row_stride, head_stride;
  uint32_t page, T, pos0, q_heads;
  float scale;
  // KV8: fp16 row scales at row * sc_row_stride + head * sc_head_stride, and the output in
  // the output in the cache's rotated basis, fp32 [T][q_heads][HD]
  const uint16_t* k_scale;
  const uint16_t* v_scale;
  size_t sc_row_stride, sc_head_stride;
  float* out_rot;
};

// 8 int8 values (two u32) widened exactly to f16: each biased byte u = q8 + 128 under an f16
// exponent byte 0x64 is 1024 + u; subtracting 1152 leaves q8 (f16 integers up to 2048 are exact)
__device__ __forceinline__ u4_t widen_i8x8(uint32_t x0, uint32_t x1) {
  x0 ^= 0x80808080u;
  x1 ^= 0x80808080u;
  const uint32_t hi = 0x64646464u;
  const h2_t bias = {(half_t)1152.0f, (half_t)1152.0f};
  return u4_t{h2_bits(as_h2(__builtin_amdgcn_perm(hi, x0, 0x04010400u)) - bias),
              h2_bits(as_h2(__builtin_amdgcn_perm(hi, x0, 0x04030402u)) - bias),
              h2_bits(as_h2(__builtin_amdgcn_perm(hi, x1, 0x04010400u)) - bias),
              h2_bits(as_h2(__builtin_amdgcn_perm(hi, x1, 0x04030402u)) - bias)};
}

// (v_maximum3_f32: fmaxf would quieten each operand first, an instruction per operand)
__device__ __forceinline__ float max3(float x, float y, float z) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(x, y), z);
}
// the max over the four lanes l % 16 + 16 k that hold one column's scores
__device__ __forceinline__ float col_max(float x) {
  float a0 = x, a1 = x;
  lane_swap16(a0, a1);
  float b0 = __builtin_elementwise_maximum(a0, a1), b1 = b0;
  lane_swap32(b0, b1);
  return __builtin_elementwise_maximum(b0, b1);
}

// 8 consecutive elements of a cache row as loaded, and as f16
template <int KV8>
struct KvPiece {
  typedef u4_t type;
  static __device__ __forceinline__ u4_t f16(u4_t v) { return v; }
};
template <>
struct KvPiece<1> {
  typedef u2_t type;
  static __device__ __forceinline__ u4_t f16(u2_t v) { return widen_i8x8(v.x, v.y); }
};

// KV8: the K and V rows are int8 with one fp16 scale per (position, kv head), the attn_prep_kv8
// form (kv8.cl): the rows are widened exactly to f16 in LDS, a score is scaled by its key's K
// scale and a weight by its key's V scale before P V (the decode reader's order); the output goes
// to out_rot in the rotated basis and, un-rotated (FWHT(s * y) / 16, kv8.cl:814-860), to attn_out.
//
// CT: 16-column tiles per wave, which share every LDS read of K and V; NS: 4 NS waves, wave w
// taking the column tiles of w % 4 and the keys 32 (w / 4) .. of each 32 NS-key iteration (the NS
// partial results of a column merge through LDS at the end, in ascending key part).
template <int HD, int GQA, int KV8, int NC, int CT, int NS>
__global__ __launch_bounds__(64 * NC * NS, 2) void attn_prefill_kernel(PrefillAttnArgs a) {
  constexpr uint32_t KK = HD / 32, NT = HD / 16;
  constexpr uint32_t COLS = 16 * CT * NC, RB = COLS / GQA;  // columns and rows per work-group
  constexpr uint32_t KB = 32 * NS;                      // keys per iteration
  constexpr uint32_t KROW = HD + 8;   // K row in LDS (f16): 16 rows' 16-byte reads fall on distinct banks
  constexpr uint32_t VROW = HD + 16;  // V row: the transposing reads of 16 rows' 32 bytes likewise
  constexpr uint32_t TPR = 2 * NC, CH = HD / (8 * TPR);  // staging threads per row, pieces of 8 elements per thread
  struct Stage {
    uint16_t k[KB * KROW];
    uint16_t v[KB * VROW];
    float ks[KV8 ? KB : 4], vs[KV8 ? KB : 4];
  };
  __shared__ __align__(16) union {
    Stage st[2];
    struct {
      float acc[CT * NT * 4][64], m[CT][64], l[CT][64];
    } part[NS > 1 ? NC * (NS - 1) : 1];
  } sm;
  // the last row blocks see the most keys: they are dispatched first, so the short blocks fill
  // the tail of the grid
  const uint32_t j = blockIdx.x, t0 = (gridDim.y - 1u - blockIdx.y) * RB;
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6, cw = wave % NC, ks = wave / NC;
  const uint32_t qi = lane & 15u, qq = lane >> 4;
  const uint32_t rows_here = min(RB, a.T - t0);
  const uint32_t kend = a.pos0 + t0 + rows_here;  // keys [0, kend) cover every row of the block
  // staging: TPR threads per key row, each its 8-element pieces TPR apart; the next
  // iteration's rows are in flight in registers while this one's are multiplied, and go to the
  // other LDS buffer afterwards. A key past kend re-reads the last one (its scores are -inf).
  const uint32_t srow = t / TPR, sch = t % TPR;
  auto cache_row = [&](uint32_t kb) -> size_t {
    const uint32_t key = min(kb + srow, kend - 1u);
    return a.pages ? (size_t)a.pages[key / a.page] * a.page + key % a.page : (size_t)key;
  };
  constexpr uint32_t EB = KV8 ? 1u : 2u;  // bytes per cache element
  const size_t hoff = (size_t)j * a.head_stride;
  typename KvPiece<KV8>::type kr[CH], vr[CH];
  uint16_t ksr = 0, vsr = 0;
  auto load_tile = [&](size_t crow) {
    const size_t off = (crow * a.row_stride + hoff) * EB + 8u * EB * sch;
#pragma unroll
    for (uint32_t i = 0; i < CH; ++i) {
      kr[i] = *reinterpret_cast<const typename KvPiece<KV8>::type*>(static_cast<const unsigned char*>(a.kv_k) + off + 8u * TPR * EB * i);
      vr[i] = *reinterpret_cast<const typename KvPiece<KV8>::type*>(static_cast<const unsigned char*>(a.kv_v) + off + 8u * TPR * EB * i);
    }
    if constexpr (KV8 == 1) {  // (all 8 threads of a row: one address)
      const size_t so = crow * a.sc_row_stride + (size_t)j * a.sc_head_stride;
      ksr = a.k_scale[so];
      vsr = a.v_scale[so];
    }
  };
  auto store_tile = [&](Stage& s) {
#pragma unroll
    for (uint32_t i = 0; i < CH; ++i) {
      const uint32_t e = 8u * (sch + TPR * i);
      *reinterpret_cast<u4_t*>(s.k + srow * KROW + e) = KvPiece<KV8>::f16(kr[i]);
      *reinterpret_cast<u4_t*>(s.v + srow * VROW + e) = KvPiece<KV8>::f16(vr[i]);
    }
    if constexpr (KV8 == 1) {
      if (sch == 0) {
        s.ks[srow] = h2f(ksr);
        s.vs[srow] = h2f(vsr);
      }
    }
  };

  // the first rows and the page table's entries of the next two iterations go out before q
  size_t crow = cache_row(KB);
  const size_t crow2 = cache_row(2u * KB);
  load_tile(cache_row(0));
  // a weight is 2^(c s - m) with s the unscaled score: one fma per key, m the running max of c s
  // (c > 0: a negative scale's sign goes to q; a zero scale keeps -inf times c at -inf)
  const float sl = a.scale * 1.4426950408889634f, sgn = sl < 0.f ? -1.f : 1.f;
  const float c = sl == 0.f ? 1e-37f : fabsf(sl);
  const bool computes = 16u * CT * cw < rows_here * GQA;  // a wave without a live column only stages
  float neg1 = -1.f;
  asm("" : "+s"(neg1));
  // this lane's columns: pair p = 16 (CT cw + ct) + qi -> row t0 + p / GQA, q head j GQA + p % GQA
  uint32_t prow[CT], ph[CT], lim[CT];
  bool live[CT];
  h8_t qh[CT][KK], ql[CT][KK];  // q as the B operand (f16 high and low parts): k = 32 kk + 8 qq + e
#pragma unroll
  for (uint32_t ct = 0; ct < CT; ++ct) {
    const uint32_t p = 16u * (CT * cw + ct) + qi;
    prow[ct] = p / GQA;
    ph[ct] = j * GQA + p % GQA;
    live[ct] = prow[ct] < rows_here;
    lim[ct] = live[ct] ? a.pos0 + t0 + prow[ct] : kend - 1u;  // the last key the column sees
    // (a dead column reads the first row's q and is never written)
    const float* qp = a.attn_q + ((size_t)(t0 + (live[ct] ? prow[ct] : 0u)) * a.q_heads + ph[ct]) * HD + 8u * qq;
#pragma unroll
    for (uint32_t kk = 0; kk < KK; ++kk) {
      const f4_t q0 = *reinterpret_cast<const f4_t*>(qp + 32u * kk) * sgn;
      const f4_t q1 = *reinterpret_cast<const f4_t*>(qp + 32u * kk + 4) * sgn;
      u4_t h, l;
      uint32_t hh, ll;
      f16_parts(q0.x, q0.y, neg1, hh, ll); h.x = hh; l.x = ll;
      f16_parts(q0.z, q0.w, neg1, hh, ll); h.y = hh; l.y = ll;
      f16_parts(q1.x, q1.y, neg1, hh, ll); h.z = hh; l.z = ll;
      f16_parts(q1.z, q1.w, neg1, hh, ll); h.w = hh; l.w = ll;
      qh[ct][kk] = __builtin_bit_cast(h8_t, h);
      ql[ct][kk] = __builtin_bit_cast(h8_t, l);
    }
  }

  // m_run: the column's reference exponent. It is raised to the largest c s seen only when that
  // exceeds it by more than kSlack (the threshold of FlashAttention-4's conditional rescaling; f16 rows:
  // weights up to 2^kSlack lose nothing in fp32 or in the f16 high and low parts), so after a few keys
  // the accumulators are hardly ever rescaled and the maximum over the column's four lanes hardly ever
  // formed. An int8 row's weight becomes f16 times its V scale, which passes f16's 65504 from a scale
  // of 256 on: a lane with a scale above kSlackScale among its eight keys takes no slack, so its
  // weights stay within 1 (c_up, c_dn: the largest c s rounded up) and no scale overflows (seven
  // instructions per 32 keys: 777 rows over 3778 keys 127.1 -> 127.7 us).
  constexpr float kNoKey = -1e30f, kSlack = 8.f, kSlackScale = 255.f;
  const float c_up = KV8 ? c * 1.0000002384f : c, c_dn = KV8 ? c * 0.9999997616f : c;
  float m_run[CT], l_run[CT];
  f4_t acc[CT][NT];
#pragma unroll
  for (uint32_t ct = 0; ct < CT; ++ct) {
    m_run[ct] = kNoKey;
    l_run[ct] = 0.f;
#pragma unroll
    for (uint32_t tt = 0; tt < NT; ++tt) acc[ct][tt] = f4_t{0.f, 0.f, 0.f, 0.f};
  }

  store_tile(sm.st[0]);
  load_tile(crow);
  crow = crow2;
  lds_barrier();
  for (uint32_t kb = 0, it = 0; kb < kend; kb += KB, ++it) {
    const Stage& s = sm.st[it & 1u];
    const uint32_t g0 = kb + 32u * ks;  // this wave's 32 keys
    if (computes && (NS == 1 || g0 < kend)) {  // uniform per wave
      // scores S^T[key g0 + 16 g + 4 qq + r][column qi]
      f4_t d[CT][2];
#pragma unroll
      for (uint32_t ct = 0; ct < CT; ++ct) d[ct][0] = d[ct][1] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (uint32_t kk = 0; kk < KK; ++kk)
#pragma unroll
        for (uint32_t g = 0; g < 2; ++g) {
          const h8_t kh = *reinterpret_cast<const h8_t*>(s.k + (32u * ks + 16u * g + qi) * KROW + 32u * kk + 8u * qq);
#pragma unroll
          for (uint32_t ct = 0; ct < CT; ++ct) d[ct][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qh[ct][kk], d[ct][g], 0, 0, 0);
#pragma unroll
          for (uint32_t ct = 0; ct < CT; ++ct) d[ct][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, ql[ct][kk], d[ct][g], 0, 0, 0);
        }
      f4_t kscale[2], vscale[2];
      if constexpr (KV8 == 1) {
#pragma unroll
        for (uint32_t g = 0; g < 2; ++g) {
          kscale[g] = *reinterpret_cast<const f4_t*>(s.ks + 32u * ks + 16u * g + 4u * qq);
          vscale[g] = *reinterpret_cast<const f4_t*>(s.vs + 32u * ks + 16u * g + 4u * qq);
        }
      }
      float slack = kSlack;
      if constexpr (KV8 == 1) {  // (the largest of the lane's eight keys' scales, whose weights it forms)
        auto abs3 = [](float x, float y, float z) { return max3(fabsf(x), fabsf(y), fabsf(z)); };
        const f4_t v0 = vscale[0], v1 = vscale[1];
        if (max3(abs3(v0[0], v0[1], v0[2]), abs3(v0[3], v1[0], v1[1]), abs3(v1[2], v1[3], v1[3])) > kSlackScale) slack = 0.f;
      }
      const bool masked = g0 + 31u > a.pos0 + t0;  // uniform: some column does not see every key
      u4_t bh[CT], bl[CT];
#pragma unroll
      for (uint32_t ct = 0; ct < CT; ++ct) {
        float w[8];
#pragma unroll
        for (uint32_t e = 0; e < 8; ++e) {
          w[e] = d[ct][e / 4][e % 4];
          if constexpr (KV8 == 1) w[e] *= kscale[e / 4][e % 4];
        }
        if (masked) {
#pragma unroll
          for (uint32_t e = 0; e < 8; ++e)
            w[e] = g0 + 16u * (e / 4) + 4u * qq + e % 4 <= lim[ct] ? w[e] : -INFINITY;
        }
        float mx = max3(max3(w[0], w[1], w[2]), max3(w[3], w[4], w[5]), max3(w[6], w[7], w[7]));
        mx *= mx > 0.f ? c_up : c_dn;
        if (const uint64_t over = __ballot(mx > m_run[ct] + slack)) {
          // (each column by its own four lanes, whatever its neighbours need)
          const uint32_t o = (uint32_t)over | (uint32_t)(over >> 32);
          const float cm = col_max(mx), m_new = ((o | o >> 16) >> qi) & 1u ? fmaxf(m_run[ct], cm) : m_run[ct];
          const float alpha = __builtin_amdgcn_exp2f(m_run[ct] - m_new);
          m_run[ct] = m_new;
          l_run[ct] *= alpha;
#pragma unroll
          for (uint32_t tt = 0; tt < NT; ++tt) acc[ct][tt] *= alpha;
        }
#pragma unroll
        for (uint32_t e = 0; e < 8; ++e) w[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(w[e], c, -m_run[ct]));
        l_run[ct] += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
        if constexpr (KV8 == 1) {
#pragma unroll
          for (uint32_t e = 0; e < 8; ++e) w[e] *= vscale[e / 4][e % 4];
        }
        uint32_t hh, ll;
        f16_parts(w[0], w[1], neg1, hh, ll); bh[ct].x = hh; bl[ct].x = ll;
        f16_parts(w[2], w[3], neg1, hh, ll); bh[ct].y = hh; bl[ct].y = ll;
        f16_parts(w[4], w[5], neg1, hh, ll); bh[ct].z = hh; bl[ct].z = ll;
        f16_parts(w[6], w[7], neg1, hh, ll); bh[ct].w = hh; bl[ct].w = ll;
      }
      // O^T += V^T P^T: the products' 32 k are the keys 4 qq + e of the two groups, which is how
      // the lanes hold the weights; V^T of 4 keys comes from one transposing read (lane 4 jj + h
      // of a 16-lane group supplies key 4 qq + jj, dims 4 h ..; lane i receives dim i of 4 keys)
      typedef short v4s_t __attribute__((ext_vector_type(4)));
      typedef v4s_t __attribute__((address_space(3)))* v4s_lds;
      const uint16_t* vb = s.v + (32u * ks + 4u * qq + (qi >> 2)) * VROW + 4u * (qi & 3u);
#pragma unroll
      for (uint32_t tt = 0; tt < NT; ++tt) {
        const v4s_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s_lds)(vb + 16u * tt));
        const v4s_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s_lds)(vb + 16u * VROW + 16u * tt));
        const h8_t av = __builtin_bit_cast(h8_t, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (uint32_t ct = 0; ct < CT; ++ct) {
          acc[ct][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(h8_t, bh[ct]), acc[ct][tt], 0, 0, 0);
          acc[ct][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(h8_t, bl[ct]), acc[ct][tt], 0, 0, 0);
        }
      }
    }
    // (the other buffer was last read before the previous barrier)
    if (kb + KB < kend) {
      store_tile(sm.st[(it + 1u) & 1u]);
      if (kb + 2u * KB < kend) {
        load_tile(crow);
        crow = cache_row(kb + 3u * KB);
      }
    }
    lds_barrier();
  }

  float l[CT];
#pragma unroll
  for (uint32_t ct = 0; ct < CT; ++ct) {
    float a0 = l_run[ct], a1 = l_run[ct];
    lane_swap16(a0, a1);
    float b0 = a0 + a1, b1 = b0;
    lane_swap32(b0, b1);
    l[ct] = b0 + b1;
  }
  if constexpr (NS > 1) {
    // the key parts 1 .. NS - 1 hand their state over through LDS (the staged keys are done with)
    if (ks) {
      auto& pt = sm.part[NC * (ks - 1u) + cw];
#pragma unroll
      for (uint32_t ct = 0; ct < CT; ++ct) {
        pt.m[ct][lane] = m_run[ct];
        pt.l[ct][lane] = l[ct];
#pragma unroll
        for (uint32_t tt = 0; tt < NT; ++tt)
#pragma unroll
          for (uint32_t r = 0; r < 4; ++r) pt.acc[(ct * NT + tt) * 4u + r][lane] = acc[ct][tt][r];
      }
    }
    lds_barrier();
    if (ks) return;
#pragma unroll
    for (uint32_t q = 0; q + 1u < NS; ++q) {
      const auto& pt = sm.part[NC * q + cw];
#pragma unroll
      for (uint32_t ct = 0; ct < CT; ++ct) {
        // (a part without a key of the column: kNoKey, weight 0)
        const float mq = pt.m[ct][lane], m = fmaxf(m_run[ct], mq);
        const float f0 = __builtin_amdgcn_exp2f(m_run[ct] - m), f1 = __builtin_amdgcn_exp2f(mq - m);
        m_run[ct] = m;
        l[ct] = __builtin_fmaf(pt.l[ct][lane], f1, l[ct] * f0);
#pragma unroll
        for (uint32_t tt = 0; tt < NT; ++tt)
#pragma unroll
          for (uint32_t r = 0; r < 4; ++r)
            acc[ct][tt][r] = __builtin_fmaf(pt.acc[(ct * NT + tt) * 4u + r][lane], f1, acc[ct][tt][r] * f0);
      }
    }
  }
#pragma unroll
  for (uint32_t ct = 0; ct < CT; ++ct) {
    // the lane holds dims 16 tt + 4 qq + r of its column
    const float inv = 1.0f / l[ct];
    const size_t o = ((size_t)(t0 + prow[ct]) * a.q_heads + ph[ct]) * HD + 4u * qq;
#pragma unroll
    for (uint32_t tt = 0; tt < NT; ++tt) acc[ct][tt] *= inv;
    if constexpr (KV8 == 1) {
      if (live[ct]) {
#pragma unroll
        for (uint32_t tt = 0; tt < NT; ++tt) *reinterpret_cast<f4_any*>(a.out_rot + o + 16u * tt) = acc[ct][tt];
      }
      // FWHT(s * y): the stages h = 1 .. 128 in order, the pair (i, i + h) becoming (a + c, a - c):
      // h = 1, 2 inside the four values, 4 and 8 across the lane groups (four swaps together: apart, their
      // wait states took 0.6 us of a few rows' 9.4), 16 .. 128 across the tiles
#pragma unroll
      for (uint32_t tt = 0; tt < NT; ++tt) {
        f4_t y;
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) y[r] = kv8_flip(acc[ct][tt][r], kv8_sign_neg(16u * tt + 4u * qq + r));
        const f4_t y1 = {y[0] + y[1], y[0] - y[1], y[2] + y[3], y[2] - y[3]};
        float u0[4] = {y1[0] + y1[2], y1[1] + y1[3], y1[0] - y1[2], y1[1] - y1[3]}, u1[4], v0[4], v1[4];
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) u1[r] = u0[r];
        lane_swap16(u0, u1);
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) v0[r] = v1[r] = (qq & 1u) ? u0[r] - u1[r] : u0[r] + u1[r];
        lane_swap32(v0, v1);
        f4_t y2;
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) y2[r] = (qq & 2u) ? v0[r] - v1[r] : v0[r] + v1[r];
        acc[ct][tt] = y2;
      }
#pragma unroll
      for (uint32_t h = 1; h < NT; h *= 2)
#pragma unroll
        for (uint32_t tt = 0; tt < NT; ++tt)
          if (!(tt & h)) {
            const f4_t u = acc[ct][tt], v = acc[ct][tt + h];
            acc[ct][tt] = u + v;
            acc[ct][tt + h] = u - v;
          }
#pragma unroll
      for (uint32_t tt = 0; tt < NT; ++tt) acc[ct][tt] *= 0.0625f;
    }
    if (live[ct]) {
#pragma unroll
      for (uint32_t tt = 0; tt < NT; ++tt) {
        const u2_t w = {(uint32_t)f2h(acc[ct][tt][0]) | ((uint32_t)f2h(acc[ct][tt][1]) << 16),
                        (uint32_t)f2h(acc[ct][tt][2]) | ((uint32_t)f2h(acc[ct][tt][3]) << 16)};
        *reinterpret_cast<h4_any*>(a.attn_out + o + 16u * tt) = w;
      }
    }
  }
}

template <int HD, int GQA, int KV8>
void launch_prefill_gqa(const PrefillAttnArgs& a, uint32_t kv_heads, uint32_t cus, hipStream_t st) {
  // Measured (40 / 8 heads of 128 or 16 / 2 of 256; us): two column tiles per wave where they still give
  // every CU a work-group (2048 rows: 86 against 97 at one tile); below that the keys in two parts,
  // which doubles the waves, until one part fills the CUs (777 rows over 3778 int8 keys: 133 against
  // 175 in one part; 333 rows over 1333: 32 / 44), but not for 64 keys or fewer (64 rows at position
  // 0: 6.6 / 7.4, int8 12.4 / 14.9); up to 32 columns at rows of 128 two column tiles and the keys in
  // four parts (3 rows over 8003: 77 / 131; 6 over 506: 11.1 / 13.5).
  constexpr uint32_t R1 = 64 / GQA;
  const uint32_t narrow = (a.T + R1 - 1) / R1;
  if constexpr (HD == 128) {
    constexpr uint32_t R2 = 128 / GQA;
    const uint32_t wide = (a.T + R2 - 1) / R2;
    if (kv_heads * wide > cus) {
      attn_prefill_kernel<HD, GQA, KV8, 4, 2, 1><<<dim3(kv_heads, wide), 256, 0, st>>>(a);
      return;
    }
  }
  if (kv_heads * narrow > cus || a.pos0 + a.T <= 64) {
    attn_prefill_kernel<HD, GQA, KV8, 4, 1, 1><<<dim3(kv_heads, narrow), 256, 0, st>>>(a);
    return;
  }
  if constexpr (HD == 128) {
    if (a.T * GQA <= 32) {
      attn_prefill_kernel<HD, GQA, KV8, 2, 1, 4><<<dim3(kv_heads, 1), 512, 0, st>>>(a);
      return;
    }
  }
  attn_prefill_kernel<HD, GQA, KV8, 4, 1, 2><<<dim3(kv_heads, narrow), 512, 0, st>>>(a);
}

template <int HD, int KV8>
int launch_prefill_attn(const PrefillAttnArgs& a, uint32_t gqa, uint32_t kv_heads, uint32_t cus, hipStream_t st) {
  switch (gqa) {
    case 1: launch_prefill_gqa<HD, 1, KV8>(a, kv_heads, cus, st); return 0;
    case 2: launch_prefill_gqa<HD, 2, KV8>(a, kv_heads, cus, st); return 0;
    case 4: launch_prefill_gqa<HD, 4, KV8>(a, kv_heads, cus, st); return 0;
    case 5: launch_prefill_gqa<HD, 5, KV8>(a, kv_heads, cus, st); return 0;
    case 6: launch_prefill_gqa<HD, 6, KV8>(a, kv_heads, cus, st); return 0;
    case 8: launch_prefill_gqa<HD, 8, KV8>(a, kv_heads, cus, st); return 0;
    default: return -1;
  }
}

// attn_prep for the chunk's rows (prep.cl attn_prep, attn.cl:361-372) with one wave per (head,
// row): grid (q_heads + 2 kv_heads, ceil(T / 4)), 256 lanes; wave w of work-group (hh, y) takes
// row 4 y + w of head hh (q heads, then k, then v), lane l elements l + 64 k. The chain is
// attn_prep's operation for operation on a one-slice fold (qkv [T][qkv_n] fp32): q/k rounded to
// f16, the RMSNorm with the 256-lane tree's order (a lane's own elements, then the 64-lane
// shuffle tree), RoPE's rotate_half pairs, q -> attn_q fp32, k and v -> the f16 cache row of
// position pos0 + t. No work-group barrier: the waves are independent.
template <int HD>
__global__ __launch_bounds__(256) void prep_rows_kernel(const float* __restrict__ qkv, uint32_t T, uint32_t pos0,
                                                        uint32_t q_heads, uint32_t kv_heads, uint32_t rot_dim,
                                                        uint32_t qkv_n, const float* __restrict__ q_norm,
                                                        const float* __restrict__ k_norm, const float* __restrict__ rope,
                                                        float* __restrict__ attn_q, uint16_t* __restrict__ kv_k,
                                                        uint16_t* __restrict__ kv_v, size_t row_stride, size_t head_stride,
                                                        const uint32_t* __restrict__ pages, uint32_t page, float eps) {
  constexpr uint32_t EPL = HD / 64u;
  __shared__ float s_row[4][HD];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t hh = blockIdx.x, t = blockIdx.y * 4u + wave;
  if (t >= T) return;  // uniform per wave
  const bool is_q = hh < q_heads, is_k = !is_q && hh < q_heads + kv_heads;
  const uint32_t h = is_q ? hh : (is_k ? hh - q_heads : hh - q_heads - kv_heads);
  const float* src = qkv + (size_t)t * qkv_n + (size_t)hh * HD;  // q || k || v, HD columns per head
  const uint32_t p = pos0 + t;
  const size_t crow = pages ? (size_t)pages[p / page] * page + p % page : (size_t)p;
  float raw[EPL];
#pragma unroll
  for (uint32_t k = 0; k < EPL; ++k) raw[k] = src[lane + 64u * k];
  if (!is_q && !is_k) {
#pragma unroll
    for (uint32_t k = 0; k < EPL; ++k) kv_v[crow * row_stride + h * head_stride + lane + 64u * k] = f2h(raw[k]);
    return;
  }
  const float* nw = is_q ? q_norm : k_norm;
  const uint32_t half = rot_dim / 2u;
  const float* cs = rope + (size_t)p * 2u * half;
  float wn[EPL], rc[EPL], rsn[EPL], xf[EPL], nv[EPL];
#pragma unroll
  for (uint32_t k = 0; k < EPL; ++k) {
    const uint32_t e = lane + 64u * k;
    wn[k] = nw ? nw[e] : 0.f;
    rc[k] = 1.f;
    rsn[k] = 0.f;
    if (e < rot_dim) {
      const uint32_t ii = e < half ? e : e - half;
      rc[k] = cs[ii];
      rsn[k] = cs[half + ii];
    }
    xf[k] = h2f(f2h(raw[k]));
  }
  if (nw) {
    float sq[EPL];
#pragma unroll
    for (uint32_t k = 0; k < EPL; ++k) sq[k] = xf[k] * xf[k];
    float acc;
    if constexpr (EPL == 4) acc = (sq[0] + sq[2]) + (sq[1] + sq[3]);
    else acc = sq[0] + sq[1];
    const float tot = wave_tree64(acc);
    const float rstd = 1.0f / sqrtf(tot / (float)HD + eps);
#pragma unroll
    for (uint32_t k = 0; k < EPL; ++k) nv[k] = h2f(f2h(xf[k] * rstd * wn[k]));
  } else {
#pragma unroll
    for (uint32_t k = 0; k < EPL; ++k) nv[k] = xf[k];
  }
  float* nrm = s_row[wave];
#pragma unroll
  for (uint32_t k = 0; k < EPL; ++k) nrm[lane + 64u * k] = nv[k];
  wave_lds_sync();
#pragma unroll
  for (uint32_t k = 0; k < EPL; ++k) {
    const uint32_t e = lane + 64u * k;
    float out;
    if (e < half) {
      const float tt = nrm[e + half] * rsn[k];
      out = __builtin_fmaf(nv[k], rc[k], -tt);
    } else if (e < rot_dim) {
      const float tt = nrm[e - half] * rsn[k];
      out = __builtin_fmaf(nv[k], rc[k], tt);
    } else {
      out = nv[k];
    }
    if (is_q)
      attn_q[((size_t)t * q_heads + h) * HD + e] = out;
    else
      kv_k[crow * row_stride + h * head_stride + e] = f2h(out);
  }
}

// grid (T), 256 lanes: resid[t] = embed[ids[t]]; an id outside the table leaves the row and
// sets the flag word (the caller's host check rejects such ids before launching)
__global__ __launch_bounds__(256) void embed_rows_kernel(const uint32_t* __restrict__ ids,
                                                         const uint16_t* __restrict__ embed,
                                                         uint16_t* __restrict__ resid, uint32_t hidden,
                                                         uint32_t vocab, uint32_t* flag) {
  const uint32_t row = ids[blockIdx.x];
  if (row >= vocab) {
    if (threadIdx.x == 0 && flag) *flag = 0xDEAD0001u;
    return;
  }
  const u4_t* s4 = reinterpret_cast<const u4_t*>(embed + (size_t)row * hidden);
  u4_t* d4 = reinterpret_cast<u4_t*>(resid + (size_t)blockIdx.x * hidden);
  for (uint32_t k = threadIdx.x; k < hidden / 8u; k += 256u) d4[k] = s4[k];
}

}  // namespace
}  // namespace mi

using namespace mi;

// the CUs of the current device, which the launch rules fill
static int cu_count(uint32_t* cus, const char* name) {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return mi_hip((int)hipGetLastError(), name);
  *cus = n > 0 ? (uint32_t)n : 1u;
  return 0;
}

// The work-group shape of the GEMM: rows per tile 16 ri, k parts ks (or the few-rows kernel). A CU's
// work-groups are r = ceil(work-groups / CUs); the rule takes the shape with the least
//   launch + (r / 2) (pair + K / 64 pair_step) + (r % 2) (round + K / 64 step).
// Two 4-wave work-groups share a CU (pair: one's ends and waits run beside the other's products), the
// others run one after the other (pair = 2 round); a round's own cost is the pipeline's fill, the
// parts' merge and the epilogue. The ns were fitted on a 256-CU part to every shape's times at 888 random
// sizes (8..2048 rows, K 64..17408, N 512..57344, plain and SwiGLU): the choice is 0.5 % off the best
// shape on average (fitted to two thirds of them, 0.6 % on the rest), 24 % at most, at a few us.
// Measured (us, the 4-wave kernel of 64..128-row tiles with 4-byte weight loads / this rule's choice; K -> N):
//   5120 -> 7168: 8 rows 65.6 / 12.1 (few, 16 rows), 64: 65.9 / 20.7 (few, 32), 100: 66.8 / 27.1 (few, 64),
//   200: 66.8 / 32.9 (32 x 256), 333: 67.2 / 38.2 (48), 500: 68.3 / 44.3 (64), 777: 84.8 / 59.1 (96),
//   1500: 128 / 111 (96 in one part), 2048: 163 / 141 (128);
//   17408 -> 5120: 8 rows 217 / 26.6, 64: 218 / 48.2, 333: 222 / 105, 777: 268 / 170, 2048: 421 / 363;
//   12864 -> 2816: 8 rows 161 / 20.2, 64: 161 / 26.2, 1024: 183 / 105;
//   SwiGLU: 1344 -> 16896 at 546 rows 41.9 / 38.5, 1600 -> 32128 at 270 53.0 / 39.1, 1728 -> 29952 at 772 112 / 104.
// The geometric mean over 250 other sizes from K = 512 on is 2.4, none slower; below K = 448 nine of 83 are,
// by 3 to 12 % (at most 2 us: a round's ends are nearly all of them).
struct GemmPick {
  bool few;
  uint32_t ri, ks;
};
static GemmPick pick_gemm(uint32_t T, uint32_t K, uint32_t N, uint32_t cus) {
  static constexpr struct {
    GemmPick p;
    int64_t launch, pair, pair_step, round, step;  // ns
  } kShapes[] = {{{true, 1, 8}, 1899, 5116, 186, 2558, 93}, {{true, 2, 8}, 1392, 9904, 238, 4952, 119},
                 {{true, 4, 8}, 0, 10230, 412, 5115, 206}, {{false, 1, 2}, 3203, 1614, 484, 807, 242},
                 {{false, 2, 2}, 3793, 2156, 700, 1078, 350}, {{false, 3, 2}, 1186, 8206, 832, 4103, 416},
                 {{false, 4, 2}, 558, 10852, 998, 5426, 499}, {{false, 6, 2}, 0, 13074, 1294, 6537, 647},
                 {{false, 4, 1}, 3373, 4409, 934, 1666, 585}, {{false, 6, 1}, 1048, 7432, 1254, 4493, 738},
                 {{false, 8, 1}, 1189, 13167, 1452, 6702, 926}};
  GemmPick best{false, 8, 1};
  int64_t least = INT64_MAX;
  for (const auto& s : kShapes) {
    const uint64_t rows = (T + 16u * s.p.ri - 1u) / (16u * s.p.ri);
    if (rows > 65535u) continue;  // the grid's limit
    const uint64_t wg = rows * (s.p.few ? N / 64u : (N + 255u) / 256u);
    const int64_t r = (int64_t)((wg + cus - 1u) / cus), G = K / GBK;
    const int64_t t = s.launch + r / 2 * (s.pair + G * s.pair_step) + r % 2 * (s.round + G * s.step);
    if (t < least) {
      least = t;
      best = s.p;
    }
  }
  return best;
}

template <bool SILU>
static int launch_gemm(const char* name, const uint32_t* qweight, const uint16_t* scales, const uint16_t* x,
                       float* out, uint16_t* h, uint32_t T, uint32_t K, uint32_t N, void* stream) {
  if (!qweight || !scales || !x || (!out && !h) || T == 0) return mi_fail(MI_ERR_ARG, (std::string(name) + ": bad arguments").c_str());
  if (K == 0 || K % GBK || N == 0 || N % 128u)
    return mi_fail(MI_ERR_SHAPE, (std::string(name) + ": K must be a multiple of 64 and N of 128").c_str());
  if (reinterpret_cast<uintptr_t>(qweight) % 16 || reinterpret_cast<uintptr_t>(x) % 16 ||
      reinterpret_cast<uintptr_t>(scales) % 8)
    return mi_fail(MI_ERR_ARG, (std::string(name) + ": qweight/x need 16-byte, scales 8-byte alignment").c_str());
  if ((T + 63u) / 64u > 65535u) return mi_fail(MI_ERR_SHAPE, (std::string(name) + ": too many rows").c_str());
  // the kernels' buffer loads take 32-bit byte offsets: x (with the last tile's rows past T) and
  // the packed weights stay below 2 GiB
  if (((uint64_t)T + 128u) * K * 2u >= (1ull << 31) || (uint64_t)K * N / 2u >= (1ull << 31))
    return mi_fail(MI_ERR_SHAPE, (std::string(name) + ": x or qweight beyond 2 GiB").c_str());
  uint32_t cus = 0;
  if (int e = cu_count(&cus, name)) return e;
  hipStream_t st = (hipStream_t)stream;
  const GemmPick p = pick_gemm(T, K, N, cus);
  const dim3 grid(p.few ? N / 64u : (N + 255u) / 256u, (T + 16u * p.ri - 1u) / (16u * p.ri));
  const bool odd = (K / GBK + p.ks - 1u) / p.ks & 1u;  // k-groups per part
#define MI_GEMM(RI, KS, DA)                                                                                    \
  if (odd) gemm_w4a16_kernel<SILU, RI, KS, DA, true><<<grid, 256 * KS, 0, st>>>(qweight, scales, x, out, h, T, K, N); \
  else gemm_w4a16_kernel<SILU, RI, KS, DA, false><<<grid, 256 * KS, 0, st>>>(qweight, scales, x, out, h, T, K, N)
#define MI_GEMM_FEW(RI, D) \
  gemm_w4a16_few_kernel<SILU, RI, 8, D><<<grid, 512, 0, st>>>(qweight, scales, x, out, h, T, K, N)
  switch ((p.few ? 100u : 10u * p.ks) + p.ri) {
    case 101: MI_GEMM_FEW(1, 4); break;
    case 102: MI_GEMM_FEW(2, 4); break;
    case 104: MI_GEMM_FEW(4, 2); break;
    case 21: MI_GEMM(1, 2, 2); break;
    case 22: MI_GEMM(2, 2, 2); break;
    case 23: MI_GEMM(3, 2, 2); break;
    case 24: MI_GEMM(4, 2, 2); break;
    case 26: MI_GEMM(6, 2, 1); break;
    case 14: MI_GEMM(4, 1, 2); break;
    case 16: MI_GEMM(6, 1, 1); break;
    default: MI_GEMM(8, 1, 1); break;
  }
#undef MI_GEMM
#undef MI_GEMM_FEW
  return mi_hip((int)hipGetLastError(), name);
}

extern "C" {

int mi_gemm_w4a16(const uint32_t* qweight, const uint16_t* scales, const uint16_t* x, float* out, uint32_t T,
                  uint32_t K, uint32_t N, void* stream) {
  return launch_gemm<false>("gemm_w4a16", qweight, scales, x, out, nullptr, T, K, N, stream);
}

int mi_gemm_w4a16_silu(const uint32_t* qweight, const uint16_t* scales, const uint16_t* x, uint16_t* h, uint32_t T,
                       uint32_t K, uint32_t N, void* stream) {
  if (!h) return mi_fail(MI_ERR_ARG, "gemm_w4a16_silu: bad arguments");
  return launch_gemm<true>("gemm_w4a16_silu", qweight, scales, x, nullptr, h, T, K, N, stream);
}

int mi_moe_prefill(const uint32_t* route, const uint16_t* x, const uint32_t* gu_blocks, const uint32_t* dn_blocks,
                   uint16_t* resid, uint32_t T, uint32_t experts, uint32_t top_k, uint32_t hidden, uint32_t inter,
                   uint32_t* list, uint32_t* tiles, uint32_t* tiles_n, uint16_t* h, uint16_t* d, void* stream) {
  if (!route || !x || !gu_blocks || !dn_blocks || !resid || !list || !tiles || !tiles_n || !h || !d)
    return mi_fail(MI_ERR_ARG, "moe_prefill: null pointer");
  if (T == 0 || T > 2048u) return mi_fail(MI_ERR_SHAPE, "moe_prefill: T must be 1..2048");
  if (experts < 16 || experts > 256 || (experts & (experts - 1)))
    return mi_fail(MI_ERR_SHAPE, "moe_prefill: experts must be a power of two in [16, 256]");
  if (top_k < 1 || top_k > 8) return mi_fail(MI_ERR_SHAPE, "moe_prefill: top_k must be 1..8");
  if (hidden == 0 || hidden % 512 || hidden > 4096)
    return mi_fail(MI_ERR_SHAPE, "moe_prefill: hidden must be a multiple of 512 up to 4096");
  if (inter == 0 || inter % 128 || inter > 1024)
    return mi_fail(MI_ERR_SHAPE, "moe_prefill: inter must be a multiple of 128 up to 1024");
  if (reinterpret_cast<uintptr_t>(tiles) % 16 || reinterpret_cast<uintptr_t>(x) % 16 ||
      reinterpret_cast<uintptr_t>(h) % 16 || reinterpret_cast<uintptr_t>(gu_blocks) % 4 ||
      reinterpret_cast<uintptr_t>(dn_blocks) % 4)
    return mi_fail(MI_ERR_ARG, "moe_prefill: tiles, x and h need 16-byte, gu_blocks and dn_blocks 4-byte alignment");
  const uint32_t slots = top_k + 1, P = T * slots;
  // The tile's most 16-row blocks by the mean pairs per expert. Measured at 2 / 4 / 6 (us, the whole block, pairs
  // spread evenly): 256 experts, top 8, 2048 -> 512: 8 pairs 114 / 120 / 141, 16: 125 / 129 / 152, 32: 188 / 153 / 176,
  // 46: 248 / 186 / 202, 64: 309 / 242 / 230; ten other shapes of 16..256 experts cross at 16..24 and 48..72. Six
  // blocks pay where one tile then holds an expert's pairs (32 experts, top 8, 2048 -> 512: 80 pairs 69 / 61 at 4 / 6,
  // 96: 71 / 63). From there to 140 both take two tiles, and those of four blocks have more waves in flight (112: 71 / 90,
  // 128: 73 / 91; tiles of 64 rows in the kernel before: 85, 87). Beyond, six save a tile, which pays where a tile
  // works long (hidden x inter 2^21 on: 64 experts, top 8, 3072 -> 768 at 176: 278 / 260; 32 experts, 2048 -> 512: 89 / 96).
  const uint32_t mean = T * top_k / experts;
  const bool one96 = mean > 52u && mean <= 96u, long96 = mean > 140u && hidden * inter >= 1u << 21;
  const uint32_t rmax = mean <= 20u ? 2u : one96 || long96 ? 6u : 4u;
  const uint32_t tile_rows = rmax == 6u ? 96u : 64u;
  const uint32_t max_tiles = (P + tile_rows - 1u) / tile_rows + experts + 1u;
  const size_t gu_block = (size_t)(2u * inter / 16u) * (hidden / GBK) * kMoeTile;
  const size_t dn_block = (size_t)(hidden / 16u) * (inter / GBK) * kMoeTile;
  hipStream_t st = (hipStream_t)stream;
  u4_t* tl = reinterpret_cast<u4_t*>(tiles);
  moe_group_kernel<<<1, 1024, 0, st>>>(route, T, experts, top_k, tile_rows, list, tl, tiles_n);
  const MoeGemm up{tl, tiles_n, list, gu_blocks, x, h, nullptr, gu_block, T, slots, hidden, 2u * inter};
  const MoeGemm down{tl, tiles_n, list, dn_blocks, h, nullptr, d, dn_block, P, slots, inter, hidden};
  const dim3 up_grid(2u * inter / 256u, max_tiles, rmax == 2u ? 2u : 1u), down_grid(hidden / 256u, max_tiles, up_grid.z);
  if (rmax == 2u) {
    moe_gemm_kernel<true, 2><<<up_grid, 256, 0, st>>>(up);
    moe_gemm_kernel<false, 2><<<down_grid, 256, 0, st>>>(down);
  } else if (rmax == 4u) {
    moe_gemm_kernel<true, 4><<<up_grid, 256, 0, st>>>(up);
    moe_gemm_kernel<false, 4><<<down_grid, 256, 0, st>>>(down);
  } else {
    moe_gemm_kernel<true, 6><<<up_grid, 256, 0, st>>>(up);
    moe_gemm_kernel<false, 6><<<down_grid, 256, 0, st>>>(down);
  }
  moe_combine_kernel<<<(T * (hidden / 8u) + 255u) / 256u, 256, 0, st>>>(route, d, resid, T, top_k, hidden);
  return mi_hip((int)hipGetLastError(), "moe_prefill");
}

int mi_attn_prefill(const float* attn_q, const uint16_t* kv_k, const uint16_t* kv_v, size_t row_stride,
                    size_t head_stride, const uint32_t* pages, uint32_t page, uint32_t T, uint32_t pos0,
                    const mi_attn_shape* shape, uint16_t* attn_out, void* stream) {
  if (!attn_q || !kv_k || !kv_v || !attn_out || !shape || T == 0)
    return mi_fail(MI_ERR_ARG, "attn_prefill: bad arguments");
  if (shape->act) return mi_fail(MI_ERR_SHAPE, "attn_prefill: f16 activations only");
  const uint32_t HD = shape->head_dim;
  if (HD != 128 && HD != 256) return mi_fail(MI_ERR_SHAPE, "attn_prefill: head_dim must be 128 or 256");
  const uint32_t gqa = shape->kv_heads ? shape->q_heads / shape->kv_heads : 0;
  if (shape->kv_heads == 0 || shape->q_heads % shape->kv_heads ||
      !(gqa == 1 || gqa == 2 || gqa == 4 || gqa == 5 || gqa == 6 || gqa == 8))
    return mi_fail(MI_ERR_SHAPE, "attn_prefill: q_heads / kv_heads must be 1, 2, 4, 5, 6 or 8");
  if (pages && page == 0) return mi_fail(MI_ERR_ARG, "attn_prefill: page size 0");
  if ((row_stride % 8) || (head_stride % 8))
    return mi_fail(MI_ERR_ARG, "attn_prefill: KV strides must keep 8-element alignment");
  PrefillAttnArgs a{attn_q, kv_k, kv_v, pages, attn_out, row_stride, head_stride, page, T, pos0,
                    shape->q_heads, shape->scale, nullptr, nullptr, 0, 0, nullptr};
  hipStream_t st = (hipStream_t)stream;
  uint32_t cus = 0;
  if (int e = cu_count(&cus, "attn_prefill")) return e;
  const int r = HD == 128 ? launch_prefill_attn<128, 0>(a, gqa, shape->kv_heads, cus, st)
                          : launch_prefill_attn<256, 0>(a, gqa, shape->kv_heads, cus, st);
  if (r) return mi_fail(MI_ERR_SHAPE, "attn_prefill: unsupported GQA");
  return mi_hip((int)hipGetLastError(), "attn_prefill");
}

int mi_attn_prefill_kv8(const float* attn_q, const int8_t* kv_k, const int8_t* kv_v, const uint16_t* k_scale,
                        const uint16_t* v_scale, size_t row_stride, size_t head_stride, size_t sc_row_stride,
                        size_t sc_head_stride, const uint32_t* pages, uint32_t page, uint32_t T, uint32_t pos0,
                        const mi_attn_shape* shape, float* out_rot, uint16_t* attn_out, void* stream) {
  if (!attn_q || !kv_k || !kv_v || !k_scale || !v_scale || !out_rot || !attn_out || !shape || T == 0)
    return mi_fail(MI_ERR_ARG, "attn_prefill_kv8: bad arguments");
  if (shape->act) return mi_fail(MI_ERR_SHAPE, "attn_prefill_kv8: f16 activations only");
  if (shape->head_dim != 256) return mi_fail(MI_ERR_SHAPE, "attn_prefill_kv8: the rotation is defined for head_dim 256");
  const uint32_t gqa = shape->kv_heads ? shape->q_heads / shape->kv_heads : 0;
  if (shape->kv_heads == 0 || shape->q_heads % shape->kv_heads ||
      !(gqa == 1 || gqa == 2 || gqa == 4 || gqa == 5 || gqa == 6 || gqa == 8))
    return mi_fail(MI_ERR_SHAPE, "attn_prefill_kv8: q_heads / kv_heads must be 1, 2, 4, 5, 6 or 8");
  if (pages && page == 0) return mi_fail(MI_ERR_ARG, "attn_prefill_kv8: page size 0");
  if ((row_stride % 16) || (head_stride % 16))
    return mi_fail(MI_ERR_ARG, "attn_prefill_kv8: int8 KV strides must keep 16-byte alignment");
  PrefillAttnArgs a{attn_q, kv_k, kv_v, pages, attn_out, row_stride, head_stride, page, T, pos0,
                    shape->q_heads, shape->scale, k_scale, v_scale, sc_row_stride, sc_head_stride, out_rot};
  hipStream_t st = (hipStream_t)stream;
  uint32_t cus = 0;
  if (int e = cu_count(&cus, "attn_prefill_kv8")) return e;
  if (launch_prefill_attn<256, 1>(a, gqa, shape->kv_heads, cus, st))
    return mi_fail(MI_ERR_SHAPE, "attn_prefill_kv8: unsupported GQA");
  return mi_hip((int)hipGetLastError(), "attn_prefill_kv8");
}

int mi_attn_prep_rows(const float* qkv, uint32_t T, uint32_t pos0, const mi_attn_shape* shape, const float* q_norm,
                      const float* k_norm, const float* rope, float* attn_q, uint16_t* kv_k, uint16_t* kv_v,
                      size_t row_stride, size_t head_stride, const uint32_t* pages, uint32_t page, void* stream) {
  if (!qkv || !shape || !rope || !attn_q || !kv_k || !kv_v || T == 0)
    return mi_fail(MI_ERR_ARG, "attn_prep_rows: bad arguments");
  if (shape->act) return mi_fail(MI_ERR_SHAPE, "attn_prep_rows: f16 activations only");
  const uint32_t HD = shape->head_dim;
  if (HD != 128 && HD != 256) return mi_fail(MI_ERR_SHAPE, "attn_prep_rows: head_dim must be 128 or 256");
  if (shape->gated || shape->kv_heads == 0 || shape->k_off != shape->q_heads * HD ||
      shape->v_off != (shape->q_heads + shape->kv_heads) * HD || shape->qkv_n != shape->v_off + shape->kv_heads * HD)
    return mi_fail(MI_ERR_SHAPE, "attn_prep_rows: a plain q||k||v layout (not gated)");
  if (shape->rot_dim > HD || shape->rot_dim % 2) return mi_fail(MI_ERR_SHAPE, "attn_prep_rows: bad rot_dim");
  if (pages && page == 0) return mi_fail(MI_ERR_ARG, "attn_prep_rows: page size 0");
  const dim3 grid(shape->q_heads + 2 * shape->kv_heads, (T + 3) / 4);
  hipStream_t st = (hipStream_t)stream;
  if (HD == 128)
    prep_rows_kernel<128><<<grid, 256, 0, st>>>(qkv, T, pos0, shape->q_heads, shape->kv_heads, shape->rot_dim,
                                                shape->qkv_n, q_norm, k_norm, rope, attn_q, kv_k, kv_v, row_stride,
                                                head_stride, pages, page, shape->eps);
  else
    prep_rows_kernel<256><<<grid, 256, 0, st>>>(qkv, T, pos0, shape->q_heads, shape->kv_heads, shape->rot_dim,
                                                shape->qkv_n, q_norm, k_norm, rope, attn_q, kv_k, kv_v, row_stride,
                                                head_stride, pages, page, shape->eps);
  return mi_hip((int)hipGetLastError(), "attn_prep_rows");
}

int mi_embed_rows(const uint32_t* ids, const uint16_t* embed, uint16_t* resid, uint32_t T, uint32_t hidden,
                  uint32_t vocab, uint32_t* flag, void* stream) {
  if (!ids || !embed || !resid || T == 0 || hidden == 0 || hidden % 8)
    return mi_fail(MI_ERR_ARG, "embed_rows: bad arguments (hidden a multiple of 8)");
  embed_rows_kernel<<<T, 256, 0, (hipStream_t)stream>>>(ids, embed, resid, hidden, vocab, flag);
  return mi_hip((int)hipGetLastError(), "embed_rows");
}

}  // extern "C"
