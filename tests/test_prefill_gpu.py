"""The chunked prefill on the GPU: the int4 linear for many rows on the matrix cores, the chunk's
causal attention, and Engine::prefill against decode's ingest of the same ids on one engine
(tests/prefill/prefill_consistency_test.cc's comparison: prefill against decode-ingest, same
engine, same prompt).

Bars: the GEMM within 2^-16 sum |x w| of the fp64 product of the same f16-rounded weights
(w = f16((q - 8) scale)), exact where every operation is exact; the attention within rel 2e-3 of
fp64 causal softmax attention, cosine >= 0.99999, paged bitwise the contiguous cache; the engine's
prefill leaves the control block as ingest does (pos, cur_token unless the last logits' top two are
closer than the tolerance), the KV rows and the last logits within the two paths' rounding
difference (prefill rounds each dequantised weight to f16; decode's GEMV multiplies the exact
integers and scales once per group)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from mipkg import dev, empty, host, mi, ptr, stream, sync
from test_engine_gpu import OracleModel, close, small_desc

pytestmark = pytest.mark.gpu
F16 = O.ORC_F16


def weights(K, N, seed, exact=False):
    rng = np.random.default_rng(seed)
    qw = rng.integers(0, 2**32, size=(K // 8, N), dtype=np.uint64).astype(np.uint32)
    if exact:
        sc = np.full((K // 64, N), O.f32_to_f16_bits(np.float32(1 / 16)), np.uint16)
    else:
        sc = O.f32_to_f16_bits(rng.uniform(0.002, 0.02, size=(K // 64, N)).astype(np.float32))
    return qw, sc


def dequant16(qw, sc):
    """w[k][n] = f16((q - 8) * s): the product of two f16 values is exact in fp32, so one
    rounding to f16 is the correctly rounded f16 product"""
    K = qw.shape[0] * 8
    k = np.arange(K)
    q = (qw[k // 8, :] >> (4 * (k % 8))[:, None]) & 0xF
    s = O.f16_bits_to_f32(sc)[k // 64, :]
    return ((q.astype(np.float32) - 8) * s).astype(np.float16).astype(np.float64)


# small and large grids, a last column tile of 128 (N % 256 != 0), ragged T, odd group counts
@pytest.mark.parametrize("T,K,N", [(1, 256, 128), (3, 64, 256), (9, 320, 384), (37, 1024, 384), (130, 2048, 256),
                                   (256, 5120, 512), (1000, 192, 14336), (2000, 64, 5120)])
def test_gemm_vs_fp64(T, K, N):
    qw, sc = weights(K, N, T + K)
    x = O.f32_to_f16_bits(np.random.default_rng(T).standard_normal((T, K)).astype(np.float32))
    print(f"gemm T={T} K={K} N={N}", flush=True)
    dq, ds, dx = dev(qw), dev(sc), dev(x)
    out = empty((T, N), np.float32)
    mi.call("mi_gemm_w4a16", ptr(dq), ptr(ds), ptr(dx), ptr(out), T, K, N, stream())
    sync()
    got = host(out, np.float32).astype(np.float64)
    w = dequant16(qw, sc)
    xf = O.f16_bits_to_f32(x).astype(np.float64)
    want = xf @ w
    bound = 2.0 ** -16 * (np.abs(xf) @ np.abs(w)) + 1e-30
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) / bound)


# the launch rule's work-group shapes on a 256-CU part, with those of the list below: full and ragged
# rows, odd group counts, fewer groups than waves or parts, a last tile of 128 columns
@pytest.mark.parametrize("T,K,N", [(16, 448, 384), (5, 64, 128), (17, 576, 7296), (64, 320, 7168), (33, 64, 7168),
                                   (100, 832, 7168), (16, 1856, 34816), (11, 2112, 34944), (30, 1856, 34816),
                                   (48, 1856, 34816), (35, 2112, 34944), (64, 1856, 34816), (511, 1088, 7296),
                                   (700, 1088, 7168), (673, 64, 7296), (1000, 320, 14464)])
def test_gemm_work_group_shapes(T, K, N):
    """Each shape against the fp64 product (test_gemm_vs_fp64's bound), and its SwiGLU form bitwise
    mi_silu_mul of the fp32 output."""
    qw, sc = weights(K, N, T + K)
    x = O.f32_to_f16_bits(np.random.default_rng(T).standard_normal((T, K)).astype(np.float32))
    print(f"gemm shapes T={T} K={K} N={N}", flush=True)
    dq, ds, dx = dev(qw), dev(sc), dev(x)
    out, h, hw = empty((T, N), np.float32), empty((T, N // 2), np.uint16), empty((T, N // 2), np.uint16)
    mi.call("mi_gemm_w4a16", ptr(dq), ptr(ds), ptr(dx), ptr(out), T, K, N, stream())
    mi.call("mi_gemm_w4a16_silu", ptr(dq), ptr(ds), ptr(dx), ptr(h), T, K, N, stream())
    mi.call("mi_silu_mul", ptr(out), ptr(hw), T, N // 2, 1, stream())
    sync()
    got = host(out, np.float32)
    w, xf = dequant16(qw, sc), O.f16_bits_to_f32(x).astype(np.float64)
    bound = 2.0 ** -16 * (np.abs(xf) @ np.abs(w)) + 1e-30
    over = np.abs(got - xf @ w) / bound
    assert np.all(over <= 1), over.max()
    assert np.array_equal(host(h, np.uint16), host(hw, np.uint16))


# k parts of an even number of groups for each number of rows, then the rest of the rule's shapes: 64, 96 and
# 128 rows in one part, 96 in two, 32 and 64 with the k-groups over 8 waves
@pytest.mark.parametrize("T,K,N", [(17, 192, 9472), (17, 192, 34816), (129, 192, 14464), (50, 768, 34816), (79, 768, 34816),
                                   (50, 128, 34816), (50, 64, 34944), (64, 192, 34816), (79, 128, 34816), (95, 64, 34944),
                                   (850, 384, 14464), (333, 448, 34816), (79, 832, 34816), (50, 832, 34816), (17, 1536, 9472),
                                   (17, 1600, 9472), (33, 2048, 9472), (33, 2112, 9472)])
def test_gemm_work_group_shapes_more(T, K, N):
    test_gemm_work_group_shapes(T, K, N)


def test_gemm_outputs_at_their_own_alignment():
    """Outputs one element off 16 bytes: the same values."""
    T, K, N = 40, 128, 384
    qw, sc = weights(K, N, 1)
    dq, ds = dev(qw), dev(sc)
    dx = dev(O.f32_to_f16_bits(np.random.default_rng(0).standard_normal((T, K)).astype(np.float32)))
    for call, dt, n in (("mi_gemm_w4a16", np.float32, N), ("mi_gemm_w4a16_silu", np.uint16, N // 2)):
        a, b = empty(T * n + 1, dt), empty(T * n + 1, dt)
        mi.call(call, ptr(dq), ptr(ds), ptr(dx), ptr(a), T, K, N, stream())
        mi.call(call, ptr(dq), ptr(ds), ptr(dx), ptr(b) + dt().itemsize, T, K, N, stream())
        sync()
        assert np.array_equal(host(b, dt)[1:], host(a, dt)[:-1])


@pytest.mark.parametrize("T,K,N", [(70, 512, 256), (70, 512, 384), (1000, 128, 14336), (2000, 64, 5120)])
def test_gemm_exact_arithmetic(T, K, N):
    """Small-integer activations and scale 1/16: every product and partial sum is exact in fp32,
    so the GEMM equals the fp64 product bit for bit (any misplaced nibble, row or column shows)."""
    qw, sc = weights(K, N, 3, exact=True)
    x = O.f32_to_f16_bits(np.random.default_rng(4).integers(-3, 4, size=(T, K)).astype(np.float32))
    dq, ds, dx = dev(qw), dev(sc), dev(x)
    out = empty((T, N), np.float32)
    mi.call("mi_gemm_w4a16", ptr(dq), ptr(ds), ptr(dx), ptr(out), T, K, N, stream())
    sync()
    want = O.f16_bits_to_f32(x).astype(np.float64) @ dequant16(qw, sc)
    assert np.array_equal(host(out, np.float32).astype(np.float64), want)


@pytest.mark.parametrize("T,K,I", [(77, 1024, 640), (70, 512, 576), (1000, 128, 7168), (2000, 64, 2560)])
def test_gemm_silu_is_gemm_then_silu_mul(T, K, I):
    """mi_gemm_w4a16_silu: SwiGLU in the GEMM's epilogue, bitwise mi_gemm_w4a16 followed by
    mi_silu_mul (the interleave16 gate||up columns), on each work-group tile."""
    qw, sc = weights(K, 2 * I, 8)
    x = O.f32_to_f16_bits(np.random.default_rng(8).standard_normal((T, K)).astype(np.float32))
    dq, ds, dx = dev(qw), dev(sc), dev(x)
    out = empty((T, 2 * I), np.float32)
    want = empty((T, I), np.uint16)
    got = empty((T, I), np.uint16)
    mi.call("mi_gemm_w4a16", ptr(dq), ptr(ds), ptr(dx), ptr(out), T, K, 2 * I, stream())
    mi.call("mi_silu_mul", ptr(out), ptr(want), T, I, 1, stream())
    mi.call("mi_gemm_w4a16_silu", ptr(dq), ptr(ds), ptr(dx), ptr(got), T, K, 2 * I, stream())
    sync()
    assert np.array_equal(host(got, np.uint16), host(want, np.uint16))


@pytest.mark.parametrize("QH,KVH,HD,rot,qk,paged", [(40, 8, 128, 128, True, False), (16, 2, 256, 64, False, True)])
def test_attn_prep_rows_is_attn_prep(QH, KVH, HD, rot, qk, paged):
    """mi_attn_prep_rows (one wave per head and row): bitwise mi_attn_prep on the same one-slice
    fold, for T rows at pos0 (attn_q and the written cache rows; the other rows untouched)."""
    sh = O.attn_shape(QH, KVH, HD, rot_dim=rot)
    T, pos0, Lm, P = 37, 100, 256, 64
    rng = np.random.default_rng(QH + HD)
    qkv = rng.standard_normal((T, sh.qkv_n)).astype(np.float32)
    qn = (1 + 0.05 * rng.standard_normal(HD)).astype(np.float32) if qk else None
    kn = (1 + 0.05 * rng.standard_normal(HD)).astype(np.float32) if qk else None
    rope = O.rope_table(1e6, rot, Lm)
    pages = rng.permutation(Lm // P).astype(np.uint32) if paged else None
    kk = O.f32_to_f16_bits(rng.standard_normal((KVH, Lm, HD)).astype(np.float32))
    keep = [dev(qkv), dev(qn), dev(kn), dev(rope), dev(pages)]
    pp = [ptr(k) if k is not None else None for k in keep]
    c = np.zeros(64, np.uint32)
    c[0], c[1] = pos0, T
    ctrl = dev(c)
    q1, k1, v1 = empty((T, QH, HD), np.float32), dev(kk), dev(kk)
    q2, k2, v2 = empty((T, QH, HD), np.float32), dev(kk), dev(kk)
    print(f"attn_prep_rows {QH}/{KVH}x{HD}", flush=True)
    mi.call("mi_attn_prep", ptr(ctrl), pp[0], 1, T, mi.shape_ref(sh), pp[1], pp[2], pp[3], ptr(q1), None, ptr(k1),
            ptr(v1), HD, Lm * HD, pp[4], P if paged else 0, Lm, stream())
    mi.call("mi_attn_prep_rows", pp[0], T, pos0, mi.shape_ref(sh), pp[1], pp[2], pp[3], ptr(q2), ptr(k2), ptr(v2), HD,
            Lm * HD, pp[4], P if paged else 0, stream())
    sync()
    assert np.array_equal(host(q2, np.uint32), host(q1, np.uint32))
    assert np.array_equal(host(k2, np.uint16), host(k1, np.uint16))
    assert np.array_equal(host(v2, np.uint16), host(v1, np.uint16))


def test_gemm_refuses_bad_shapes():
    with pytest.raises(mi.MiError):
        mi.call("mi_gemm_w4a16", 16, 16, 16, 16, 4, 100, 128, None)
    with pytest.raises(mi.MiError):
        mi.call("mi_gemm_w4a16", 16, 16, 16, 16, 4, 128, 100, None)


def prefill_attention(sh, q, k, v, T, pos0, pages=None, page=0):
    HD, QH = sh.head_dim, sh.q_heads
    Lm = k.shape[1]
    dq, dk, dv, dpg = dev(q), dev(k), dev(v), dev(pages)
    out = empty((T, QH * HD), np.uint16)
    mi.call("mi_attn_prefill", ptr(dq), ptr(dk), ptr(dv), HD, Lm * HD, ptr(dpg), page, T, pos0, mi.shape_ref(sh),
            ptr(out), stream())
    sync()
    return host(out, np.uint16)


@pytest.mark.parametrize("QH,KVH,HD,T,pos0", [(40, 8, 128, 37, 100), (40, 8, 128, 130, 0), (16, 2, 256, 20, 64),
                                              (8, 8, 128, 65, 3)])
def test_attn_prefill_vs_fp64(QH, KVH, HD, T, pos0):
    sh = O.attn_shape(QH, KVH, HD)
    Lm = 256
    rng = np.random.default_rng(QH + T)
    k = O.f32_to_f16_bits(rng.standard_normal((KVH, Lm, HD)).astype(np.float32))
    v = O.f32_to_f16_bits(rng.standard_normal((KVH, Lm, HD)).astype(np.float32))
    q = rng.standard_normal((T, QH, HD)).astype(np.float32)
    print(f"attn_prefill {QH}/{KVH}x{HD} T={T} pos0={pos0}", flush=True)
    got = prefill_attention(sh, q, k, v, T, pos0)
    G = QH // KVH
    want = np.zeros((T, QH, HD))
    for t in range(T):
        for h in range(QH):
            O.lib().orc_attend64(C.byref(sh), O._p(np.ascontiguousarray(q[t, h])), h // G, pos0 + t + 1, 0, F16,
                                 O._p(k), O._p(v), None, None, HD, Lm * HD, 1, Lm, None, 0, O._p(want[t, h]))
    g = O.f16_bits_to_f32(got).astype(np.float64).reshape(T, QH, HD)
    err = np.abs(g - want)
    assert np.all(err <= 2e-3 * np.abs(want) + 2e-3 * np.abs(want).max(axis=-1, keepdims=True)), err.max()
    cos = (g * want).sum(-1) / np.sqrt((g * g).sum(-1) * (want * want).sum(-1))
    assert cos.min() >= 0.99999


def unrotate64():
    """y -> H_256 diag(s) y / 16 as an fp64 matrix (the int8 cache's rotation, kv8.h:1-26)."""
    words = (0xA197D809, 0xA6850592, 0xB205A73E, 0x20AFA769, 0x45C2CF64, 0xBEAEAACB, 0x75F39ADD, 0x2385A70C)
    sign = np.array([-1.0 if words[j // 32] >> (j % 32) & 1 else 1.0 for j in range(256)])
    h = np.ones((1, 1))
    for _ in range(8):
        h = np.block([[h, h], [h, -h]])
    return h * sign[None, :] / 16


# each work-group shape of the launch rule on a 256-CU part: 32 columns or fewer with the keys in four
# parts (1..6 rows at GQA 5) around its 128-key iteration, 64 keys in one part against 65 in two, 64
# columns with the keys in two parts, 64 and 128 columns in one; key counts around the iterations' edges
@pytest.mark.parametrize("QH,KVH,HD,T,pos0,int8", [
    (40, 8, 128, 6, 122, 0), (40, 8, 128, 6, 123, 0), (40, 8, 128, 1, 64, 0), (40, 8, 128, 64, 0, 0),
    (40, 8, 128, 65, 0, 0), (40, 8, 128, 7, 185, 0), (40, 8, 128, 400, 33, 0), (40, 8, 128, 810, 0, 0),
    (12, 2, 128, 3, 500, 0), (16, 2, 256, 5, 59, 0), (16, 2, 256, 33, 95, 0), (16, 2, 256, 1030, 0, 0),
    (16, 2, 256, 1, 0, 1), (16, 2, 256, 9, 119, 1), (16, 2, 256, 1030, 31, 1), (24, 4, 256, 37, 290, 1)])
def test_attn_prefill_work_group_shapes_vs_fp64(QH, KVH, HD, T, pos0, int8):
    """Scores that grow along the keys (the running maximum keeps rising, so the accumulators are
    rescaled again and again) and span about 2^30, against fp64 causal attention; the last cache row
    holds what no row may read."""
    sh = O.attn_shape(QH, KVH, HD)
    Lm = pos0 + T + 1
    rng = np.random.default_rng(QH + T + pos0)
    q = 2 * rng.standard_normal((T, QH, HD)).astype(np.float32)
    ramp = np.linspace(0.3, 1.5, Lm)[None, :, None]
    k = ramp * rng.standard_normal((KVH, Lm, HD))
    if int8:
        s16 = O.f32_to_f16_bits((np.abs(k).max(-1) / 127).astype(np.float32))
        k8 = np.clip(np.rint(k / O.f16_bits_to_f32(s16)[..., None]), -127, 127).astype(np.int8)
        v8 = rng.integers(-127, 128, size=(KVH, Lm, HD)).astype(np.int8)
        vs = O.f32_to_f16_bits(rng.uniform(0.005, 0.05, (KVH, Lm)).astype(np.float32))
        s16[:, -1] = vs[:, -1] = 0x7E00  # NaN scales in the row past the last
        kf = k8 * O.f16_bits_to_f32(s16).astype(np.float64)[..., None]
        vf = v8 * O.f16_bits_to_f32(vs).astype(np.float64)[..., None]
    else:
        k16, v16 = O.f32_to_f16_bits(k.astype(np.float32)), O.f32_to_f16_bits(rng.standard_normal(k.shape).astype(np.float32))
        k16[:, -1] = v16[:, -1] = 0x7E00
        kf, vf = O.f16_bits_to_f32(k16).astype(np.float64), O.f16_bits_to_f32(v16).astype(np.float64)
    print(f"attn_prefill {QH}/{KVH}x{HD} T={T} pos0={pos0} int8={int8}", flush=True)
    if int8:
        keep = [dev(a) for a in (q, k8, v8, s16, vs)]
        rot, out = empty((T, QH, HD), np.float32), empty((T, QH * HD), np.uint16)
        mi.call("mi_attn_prefill_kv8", *[ptr(a) for a in keep], HD, Lm * HD, 1, Lm, None, 0, T, pos0, mi.shape_ref(sh),
                ptr(rot), ptr(out), stream())
        sync()
        got = host(out, np.uint16)
    else:
        got = prefill_attention(sh, q, k16, v16, T, pos0)
    g = O.f16_bits_to_f32(got).astype(np.float64).reshape(T, QH, HD)
    keys = pos0 + T
    hidden = np.arange(keys)[None, :] > pos0 + np.arange(T)[:, None]
    for h in range(QH):
        s = q[:, h].astype(np.float64) @ kf[h // (QH // KVH), :keys].T * float(sh.scale)
        s[hidden] = -np.inf
        w = np.exp(s - s.max(-1, keepdims=True))
        w /= w.sum(-1, keepdims=True)
        kh, vh = kf[h // (QH // KVH), :keys], vf[h // (QH // KVH), :keys]
        want = w @ vh
        # a score's error: 2^-21 sum |q k| scale (q in two f16 parts is good to 2^-22, the fp32 sums of
        # its products to about as much); a weight's is that of its own and of the largest score; the
        # weights' parts and the sums over the keys add 2^-20. The parts are f16 values down to 2^-24, so
        # a weight (int8: times its V scale) is also off by up to 2^-25 of the largest one, whatever its
        # size: independent over the keys, 8 standard deviations of 2^-25 / sqrt(3) each
        ds = 2.0 ** -21 * np.where(hidden, 0, np.abs(q[:, h]).astype(np.float64) @ np.abs(kh).T * float(sh.scale))
        bound = (2 * ds.max(-1, keepdims=True) + 2.0 ** -20) * (w @ np.abs(vh))
        vraw = v8[h // (QH // KVH), :keys].astype(np.float64) if int8 else vh
        bound += 8 * 2.0 ** -25 / 3 ** 0.5 * np.sqrt(~hidden @ np.square(vraw))
        if int8:
            rot_err = np.abs(host(rot, np.float32).reshape(T, QH, HD)[:, h] - want)
            assert np.all(rot_err <= bound), (h, (rot_err / bound).max())
            R = unrotate64()
            want, bound = want @ R.T, bound @ np.abs(R).T
        err = np.abs(g[:, h] - want)
        bound = bound + 2.0 ** -11 * np.abs(want) + 2.0 ** -25  # the f16 rounding of the output
        assert np.all(err <= bound), (h, (err / bound).max())


# keys in one part and in two, 64 columns per work-group; the key counts end inside an iteration
@pytest.mark.parametrize("T,pos0", [(5, 259), (100, 301), (1030, 231)])
@pytest.mark.parametrize("big", [255, 256, 300, 8000, 65504])
def test_attn_prefill_int8_large_v_scales(T, pos0, big):
    """V scales up to f16's largest under scores that rise by 7.9 in log2 units after the first 128
    keys (a weight times its V scale must stay an f16 value), every third key's scale large, against
    fp64 attention on the fp32 rotated output (the f16 one overflows by itself)."""
    QH, KVH, HD, keys = 16, 2, 256, pos0 + T
    sh = O.attn_shape(QH, KVH, HD)
    rng = np.random.default_rng(T)
    u = rng.choice([-1, 1], (KVH, 1, HD)) * rng.integers(64, 120, (KVH, 1, HD))
    k8 = (u + rng.integers(-3, 4, (KVH, keys, HD))).astype(np.int8)
    v8 = rng.integers(-127, 128, (KVH, keys, HD)).astype(np.int8)
    rise = np.clip((np.arange(keys) - 128) / 32, 0.002, 1) * 7.9 / np.log2(np.e)
    ks = O.f32_to_f16_bits(np.tile((0.05 * rise / rise[-1]).astype(np.float32), (KVH, 1)))
    vs = O.f32_to_f16_bits(np.where(np.arange(keys) % 3 == 0, big, 0.03)[None].repeat(KVH, 0).astype(np.float32))
    # q along u, so that the last keys' score is rise[-1]
    gain = rise[-1] / (0.05 * np.square(u.astype(np.float64)).sum(-1) * float(sh.scale))
    q = (np.repeat((u[:, 0] * gain).astype(np.float32), QH // KVH, 0)[None] * np.linspace(0.97, 1, T)[:, None, None]).astype(np.float32)
    print(f"attn_prefill_kv8 V scale {big} T={T} pos0={pos0}", flush=True)
    keep = [dev(a) for a in (q, k8, v8, ks, vs)]
    rot, out = empty((T, QH, HD), np.float32), empty((T, QH * HD), np.uint16)
    mi.call("mi_attn_prefill_kv8", *[ptr(a) for a in keep], HD, keys * HD, 1, keys, None, 0, T, pos0, mi.shape_ref(sh),
            ptr(rot), ptr(out), stream())
    sync()
    got = host(rot, np.float32).reshape(T, QH, HD).astype(np.float64)
    assert np.isfinite(got).all()
    hidden = np.arange(keys)[None, :] > pos0 + np.arange(T)[:, None]
    for h in range(0, QH, QH // KVH):
        j = h // (QH // KVH)
        kh = k8[j] * O.f16_bits_to_f32(ks[j]).astype(np.float64)[:, None]
        vh = v8[j] * O.f16_bits_to_f32(vs[j]).astype(np.float64)[:, None]
        s = q[:, h].astype(np.float64) @ kh.T * float(sh.scale)
        s[hidden] = -np.inf
        w = np.exp(s - s.max(-1, keepdims=True))
        w /= w.sum(-1, keepdims=True)
        # test_attn_prefill_work_group_shapes_vs_fp64's bound
        ds = 2.0 ** -21 * np.where(hidden, 0, np.abs(q[:, h]).astype(np.float64) @ np.abs(kh).T * float(sh.scale))
        bound = (2 * ds.max(-1, keepdims=True) + 2.0 ** -20) * (w @ np.abs(vh))
        bound += 8 * 2.0 ** -25 / 3 ** 0.5 * np.sqrt(~hidden @ np.square(v8[j].astype(np.float64)))
        err = np.abs(got[:, h] - w @ vh)
        assert np.all(err <= bound), (h, (err / bound).max())


@pytest.mark.parametrize("QH,KVH,HD,T,pos0,int8", [
    (40, 8, 128, 6, 123, 0), (40, 8, 128, 65, 0, 0), (40, 8, 128, 810, 0, 0), (16, 2, 256, 33, 95, 0),
    (16, 2, 256, 9, 119, 1), (16, 2, 256, 1030, 31, 1)])
def test_attn_prefill_columns_do_not_depend_on_their_neighbours(QH, KVH, HD, T, pos0, int8):
    """A (row, head)'s bits are the same whatever the other rows and heads of its work-group hold: half
    of them, drawn at random, with 30 times the q, whose maxima rise where the others' do not."""
    sh = O.attn_shape(QH, KVH, HD)
    keys = pos0 + T
    rng = np.random.default_rng(T)
    q = rng.standard_normal((T, QH, HD)).astype(np.float32)
    loud = rng.random((T, QH)) < 0.5
    print(f"attn_prefill neighbours {QH}/{KVH}x{HD} T={T} pos0={pos0} int8={int8}", flush=True)

    def run(q):
        if not int8:
            return prefill_attention(sh, q, k16, v16, T, pos0)
        rot, out = empty((T, QH, HD), np.float32), empty((T, QH * HD), np.uint16)
        mi.call("mi_attn_prefill_kv8", *[ptr(a) for a in [dev(q), *keep]], HD, keys * HD, 1, keys, None, 0, T, pos0,
                mi.shape_ref(sh), ptr(rot), ptr(out), stream())
        sync()
        return host(out, np.uint16)

    if int8:
        keep = [dev(rng.integers(-127, 128, (KVH, keys, HD)).astype(np.int8)) for _ in range(2)]
        keep += [dev(O.f32_to_f16_bits(rng.uniform(0.005, 0.05, (KVH, keys)).astype(np.float32))) for _ in range(2)]
    else:
        k16, v16 = (O.f32_to_f16_bits(rng.standard_normal((KVH, keys, HD)).astype(np.float32)) for _ in range(2))
    a = run(q).reshape(T, QH, HD)
    b = run(np.where(loud[..., None], 30 * q, q).astype(np.float32)).reshape(T, QH, HD)
    assert np.array_equal(a[~loud], b[~loud])


def test_attn_prefill_paged_bitwise():
    sh = O.attn_shape(40, 8, 128)
    Lm, P, T, pos0 = 512, 64, 50, 300
    rng = np.random.default_rng(5)
    k = O.f32_to_f16_bits(rng.standard_normal((8, Lm, 128)).astype(np.float32))
    v = O.f32_to_f16_bits(rng.standard_normal((8, Lm, 128)).astype(np.float32))
    q = rng.standard_normal((T, 40, 128)).astype(np.float32)
    a = prefill_attention(sh, q, k, v, T, pos0)
    pages = rng.permutation(Lm // P).astype(np.uint32)
    phys = np.concatenate([np.arange(pg * P, pg * P + P) for pg in pages])
    kp, vp = np.empty_like(k), np.empty_like(v)
    kp[:, phys], vp[:, phys] = k, v
    b = prefill_attention(sh, q, kp, vp, T, pos0, pages, P)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("P", [16, 64])
@pytest.mark.parametrize("QH,KVH,HD,T,pos0,int8", [
    (40, 8, 128, 6, 123, 0), (40, 8, 128, 64, 0, 0), (40, 8, 128, 7, 185, 0), (40, 8, 128, 810, 0, 0), (16, 2, 256, 5, 59, 0),
    (16, 2, 256, 33, 95, 0), (16, 2, 256, 1030, 0, 0), (16, 2, 256, 1, 0, 1), (16, 2, 256, 9, 119, 1), (16, 2, 256, 1030, 31, 1),
    (24, 4, 256, 37, 290, 1)])
def test_attn_prefill_work_group_shapes_paged_bitwise(QH, KVH, HD, T, pos0, int8, P):
    """Each work-group shape through a permuted page table, keys ending inside a page: bitwise the
    contiguous cache. Every row that no key has holds NaN (int8: NaN scales)."""
    sh = O.attn_shape(QH, KVH, HD)
    keys = pos0 + T
    npg = -(-keys // P) + 3
    rng = np.random.default_rng(T + pos0 + P)
    pages = rng.permutation(npg).astype(np.uint32)
    phys = (pages[:, None] * P + np.arange(P)).ravel()[:keys]
    q = rng.standard_normal((T, QH, HD)).astype(np.float32)
    print(f"attn_prefill paged {QH}/{KVH}x{HD} T={T} pos0={pos0} int8={int8} P={P}", flush=True)

    def paged(a, fill):
        b = np.full((KVH, npg * P) + a.shape[2:], fill, a.dtype)
        b[:, phys] = a
        return b

    if int8:
        kv = [rng.integers(-127, 128, (KVH, keys, HD)).astype(np.int8) for _ in range(2)]
        sc = [O.f32_to_f16_bits(rng.uniform(0.005, 0.05, (KVH, keys)).astype(np.float32)) for _ in range(2)]

        def run(kv, sc, Lm, pages, P):
            keep = [dev(a) for a in (q, *kv, *sc)]
            rot, out, dpg = empty((T, QH, HD), np.float32), empty((T, QH * HD), np.uint16), dev(pages)
            mi.call("mi_attn_prefill_kv8", *[ptr(a) for a in keep], HD, Lm * HD, 1, Lm, ptr(dpg), P, T, pos0, mi.shape_ref(sh),
                    ptr(rot), ptr(out), stream())
            sync()
            return host(out, np.uint16), host(rot, np.uint32)

        want = run(kv, sc, keys, None, 0)
        got = run([paged(a, 127) for a in kv], [paged(a, 0x7E00) for a in sc], npg * P, pages, P)
        assert np.array_equal(got[1], want[1])
        got, want = got[0], want[0]
    else:
        k, v = (O.f32_to_f16_bits(rng.standard_normal((KVH, keys, HD)).astype(np.float32)) for _ in range(2))
        want = prefill_attention(sh, q, k, v, T, pos0)
        got = prefill_attention(sh, q, paged(k, 0x7E00), paged(v, 0x7E00), T, pos0, pages, P)
    assert np.array_equal(got, want)
    assert np.isfinite(O.f16_bits_to_f32(want)).all()


def kv_rows(eng, p0, n):
    d = eng.desc
    k = eng.to_host(mi.T_KV_K, 0, np.uint16).reshape(d.layers, d.kv_heads, d.max_len, d.head_dim)
    v = eng.to_host(mi.T_KV_V, 0, np.uint16).reshape(d.layers, d.kv_heads, d.max_len, d.head_dim)
    f = lambda a: O.f16_bits_to_f32(a[:, :, p0:p0 + n]).astype(np.float64)
    return f(k), f(v)


@pytest.mark.parametrize("n,chunk,p0", [(40, 0, 0), (40, 16, 0), (33, 8, 100)])
def test_prefill_matches_ingest(n, chunk, p0):
    eng = mi.Engine(small_desc(max_len=512), seed=11)
    eng.capture(1)
    ids = np.random.default_rng(n + chunk).integers(0, eng.desc.vocab_used, n).astype(np.uint32)
    print(f"prefill vs ingest n={n} chunk={chunk} p0={p0}", flush=True)
    eng.reset(p0, 0)
    eng.ingest(ids)
    c_ing = eng.ctrl()
    lg_ing = eng.logits(1)[0].astype(np.float64)
    k_ing, v_ing = kv_rows(eng, p0, n)
    eng.reset(p0, 0)
    eng.prefill(ids, chunk)
    c_pf = eng.ctrl()
    lg_pf = eng.logits(1)[0].astype(np.float64)
    k_pf, v_pf = kv_rows(eng, p0, n)
    assert c_pf[mi.CTRL_POS] == c_ing[mi.CTRL_POS] == p0 + n
    assert c_pf[mi.CTRL_NACT] == 1
    # the two paths differ by the f16 rounding of the dequantised weights (2^-11 relative each)
    for a, b in ((k_pf, k_ing), (v_pf, v_ing)):
        assert np.all(np.abs(a - b) <= 0.02 * np.abs(b) + 0.02 * np.abs(b).max()), np.abs(a - b).max()
    scale = np.abs(lg_ing).max()
    assert np.all(np.abs(lg_pf - lg_ing) <= 0.01 * scale), np.abs(lg_pf - lg_ing).max() / scale
    top2 = np.sort(lg_ing)[-2:]
    if top2[1] - top2[0] > 0.02 * scale:
        assert c_pf[mi.CTRL_CUR] == c_ing[mi.CTRL_CUR] == int(np.argmax(lg_ing))
    # decode continues from the prefilled cache as from the ingested one
    eng.close()


@pytest.mark.parametrize("n,chunk,p0,qk_norm", [(40, 0, 0, 1), (40, 16, 0, 1), (33, 8, 100, 0)])
def test_prefill_vs_oracle_prefill(n, chunk, p0, qk_norm):
    """The engine's chunked prefill against the oracle's prefill walk (orc_prefill_chunk, chunk by
    chunk on the same cache): the last position's logits and every K/V row written, at the
    north star's rel 2e-3, and the control block as ingest leaves it."""
    eng = mi.Engine(small_desc(max_len=512, qk_norm=qk_norm), seed=13)
    orc = OracleModel(eng)
    ids = np.random.default_rng(n + chunk + 1).integers(0, eng.desc.vocab_used, n).astype(np.uint32)
    print(f"prefill vs oracle n={n} chunk={chunk} p0={p0} qk_norm={qk_norm}", flush=True)
    eng.reset(p0, 0)
    eng.prefill(ids, chunk)
    c = eng.ctrl()
    lg = eng.logits(1)[0].astype(np.float64)
    k_pf, v_pf = kv_rows(eng, p0, n)
    step = chunk or n
    want = np.zeros(eng.desc.vocab, np.float32)
    for c0 in range(0, n, step):
        part = np.ascontiguousarray(ids[c0:c0 + step])
        am = O.lib().orc_prefill_chunk(O.ORC_F16, C.byref(orc.m), O._p(part), len(part), p0 + c0, O._p(orc.kv_k),
                                       O._p(orc.kv_v), O._p(want))
    d = eng.desc
    kw = orc.kv_k.reshape(d.layers, d.kv_heads, d.max_len, d.head_dim)[:, :, p0:p0 + n]
    vw = orc.kv_v.reshape(d.layers, d.kv_heads, d.max_len, d.head_dim)[:, :, p0:p0 + n]
    for a, b in ((k_pf, kw), (v_pf, vw)):
        b = O.f16_bits_to_f32(b).astype(np.float64)
        assert np.all(np.abs(a - b) <= 2e-3 * np.abs(b) + 2e-3 * np.abs(b).max()), np.abs(a - b).max()
    w = want.astype(np.float64)
    assert close(lg, w), np.abs(lg - w).max() / np.abs(w).max()
    assert c[mi.CTRL_POS] == p0 + n and c[mi.CTRL_NACT] == 1
    top2 = np.sort(w)[-2:]
    if top2[1] - top2[0] > 4e-3 * np.abs(w).max():
        assert c[mi.CTRL_CUR] == am
    eng.close()


def test_prefill_refusals():
    eng = mi.Engine(small_desc(max_len=256), seed=2)
    eng.reset(250, 0)
    with pytest.raises(mi.MiError):
        eng.prefill(np.arange(10, dtype=np.uint32))  # past the cache
    eng.reset(0, 0)
    with pytest.raises(mi.MiError):
        eng.prefill(np.array([eng.desc.vocab], np.uint32))  # outside the vocabulary
    with pytest.raises(mi.MiError):
        eng.prefill(np.arange(4, dtype=np.uint32), 4096)  # chunk above the cap
    eng.close()


def test_moe_prefill_matches_ingest():
    """A mixture-of-experts model: the expert kernels run over the chunk's rows in slices. Layer
    0's K/V rows come before any routing and hold the dense bar; later layers sit behind top-k
    routing, where a near-tied expert choice may flip between the two roundings, so the last
    logits are held to a cosine bar there."""
    from test_engine_gpu import moe_small_desc
    eng = mi.Engine(moe_small_desc(max_len=512), seed=12)
    eng.capture(1)
    n, p0 = 37, 20
    ids = np.random.default_rng(3).integers(0, eng.desc.vocab_used, n).astype(np.uint32)
    print(f"moe prefill vs ingest n={n} p0={p0}", flush=True)
    eng.reset(p0, 0)
    eng.ingest(ids)
    c_ing, lg_ing = eng.ctrl(), eng.logits(1)[0].astype(np.float64)
    k_ing, v_ing = kv_rows(eng, p0, n)
    eng.reset(p0, 0)
    eng.prefill(ids, 16)
    c_pf, lg_pf = eng.ctrl(), eng.logits(1)[0].astype(np.float64)
    k_pf, v_pf = kv_rows(eng, p0, n)
    assert c_pf[mi.CTRL_POS] == c_ing[mi.CTRL_POS] == p0 + n
    for a, b in ((k_pf[0], k_ing[0]), (v_pf[0], v_ing[0])):
        assert np.all(np.abs(a - b) <= 0.02 * np.abs(b) + 0.02 * np.abs(b).max()), np.abs(a - b).max()
    cos = (lg_pf * lg_ing).sum() / np.sqrt((lg_pf * lg_pf).sum() * (lg_ing * lg_ing).sum())
    assert cos >= 0.99, cos
    eng.close()


def test_moe_prefill_vs_oracle_prefill():
    """The MoE model's chunked prefill against the oracle's prefill walk (orc_prefill_chunk with
    the experts as orc_moe_prefill, pinned to pf_moe_ref.h): every K/V row and the last logits
    at rel 2e-3."""
    from test_engine_gpu import moe_small_desc
    eng = mi.Engine(moe_small_desc(max_len=512), seed=12)
    orc = OracleModel(eng)
    n, p0, chunk = 37, 20, 16
    ids = np.random.default_rng(3).integers(0, eng.desc.vocab_used, n).astype(np.uint32)
    print(f"moe prefill vs oracle n={n} p0={p0}", flush=True)
    eng.reset(p0, 0)
    eng.prefill(ids, chunk)
    lg = eng.logits(1)[0].astype(np.float64)
    k_pf, v_pf = kv_rows(eng, p0, n)
    want = np.zeros(eng.desc.vocab, np.float32)
    for c0 in range(0, n, chunk):
        part = np.ascontiguousarray(ids[c0:c0 + chunk])
        O.lib().orc_prefill_chunk(O.ORC_F16, C.byref(orc.m), O._p(part), len(part), p0 + c0, O._p(orc.kv_k),
                                  O._p(orc.kv_v), O._p(want))
    d = eng.desc
    kw = orc.kv_k.reshape(d.layers, d.kv_heads, d.max_len, d.head_dim)[:, :, p0:p0 + n]
    vw = orc.kv_v.reshape(d.layers, d.kv_heads, d.max_len, d.head_dim)[:, :, p0:p0 + n]
    for a, b in ((k_pf, kw), (v_pf, vw)):
        b = O.f16_bits_to_f32(b).astype(np.float64)
        assert np.all(np.abs(a - b) <= 2e-3 * np.abs(b) + 2e-3 * np.abs(b).max()), np.abs(a - b).max()
    w = want.astype(np.float64)
    assert close(lg, w), np.abs(lg - w).max() / np.abs(w).max()
    eng.close()


def test_attn_prefill_kv8_rows_match_the_decode_reader():
    """mi_attn_prefill_kv8 over the int8 rotated cache: row t equals the decode reader's
    (attn_decode int8 + attn_reduce_kv8, itself held to fp64 attention with an fp64
    un-rotation in test_kv8_gpu) at position pos0 + t, within rel 2e-3 / cosine 0.99999."""
    QH, KVH, HD, Lm, T, pos0 = 16, 2, 256, 256, 20, 64
    sh = O.attn_shape(QH, KVH, HD)
    rng = np.random.default_rng(31)
    k8 = rng.integers(-127, 128, size=(KVH, Lm, HD)).astype(np.int8)
    v8 = rng.integers(-127, 128, size=(KVH, Lm, HD)).astype(np.int8)
    ks = O.f32_to_f16_bits(rng.uniform(0.005, 0.05, (KVH, Lm)).astype(np.float32))
    vs = O.f32_to_f16_bits(rng.uniform(0.005, 0.05, (KVH, Lm)).astype(np.float32))
    q = rng.standard_normal((T, QH, HD)).astype(np.float32)
    dk, dv, dks, dvs, dq = dev(k8), dev(v8), dev(ks), dev(vs), dev(q)
    rot = empty((T, QH, HD), np.float32)
    out = empty((T, QH * HD), np.uint16)
    print("attn_prefill_kv8", flush=True)
    mi.call("mi_attn_prefill_kv8", ptr(dq), ptr(dk), ptr(dv), ptr(dks), ptr(dvs), HD, Lm * HD, 1, Lm, None, 0, T,
            pos0, mi.shape_ref(sh), ptr(rot), ptr(out), stream())
    sync()
    got = O.f16_bits_to_f32(host(out, np.uint16)).astype(np.float64).reshape(T, QH, HD)
    tgt = 16
    for t in (0, 7, T - 1):
        c = np.zeros(64, np.uint32)
        c[0], c[1] = pos0 + t, 1
        ctrl = dev(c)
        qt = dev(np.ascontiguousarray(q[t:t + 1]))
        part = empty((QH, tgt, 1, HD + 2), np.float32)
        want16 = empty((1, QH * HD), np.uint16)
        mi.call("mi_attn_decode", ptr(ctrl), ptr(qt), 1, ptr(dk), ptr(dv), ptr(dks), ptr(dvs), HD, Lm * HD, 1, Lm,
                None, 0, Lm, ptr(part), 1, tgt, mi.shape_ref(sh), stream())
        mi.call("mi_attn_reduce_kv8", ptr(ctrl), ptr(part), None, ptr(want16), 1, tgt, Lm, mi.shape_ref(sh), stream())
        sync()
        want = O.f16_bits_to_f32(host(want16, np.uint16)).astype(np.float64).reshape(QH, HD)
        g = got[t]
        err = np.abs(g - want)
        assert np.all(err <= 2e-3 * np.abs(want) + 2e-3 * np.abs(want).max(axis=-1, keepdims=True)), (t, err.max())
        cos = (g * want).sum(-1) / np.sqrt((g * g).sum(-1) * (want * want).sum(-1))
        assert cos.min() >= 0.99999, t


def test_int8_cache_prefill_matches_ingest():
    eng = mi.Engine(small_desc(max_len=256, head_dim=256, q_heads=8, kv_heads=2, kv_int8=1), seed=13)
    eng.capture(1)
    d = eng.desc
    n, p0 = 30, 10
    ids = np.random.default_rng(9).integers(0, d.vocab_used, n).astype(np.uint32)
    print(f"int8-cache prefill vs ingest n={n} p0={p0}", flush=True)

    def rows():
        k = eng.to_host(mi.T_KV_K, 0, np.int8).reshape(d.layers, d.kv_heads, d.max_len, d.head_dim)
        ks = O.f16_bits_to_f32(eng.to_host(mi.T_KV_KS, 0, np.uint16).reshape(d.layers, d.kv_heads, d.max_len))
        return k[:, :, p0:p0 + n].astype(np.float64) * ks[:, :, p0:p0 + n, None]

    eng.reset(p0, 0)
    eng.ingest(ids)
    c_ing, lg_ing, k_ing = eng.ctrl(), eng.logits(1)[0].astype(np.float64), rows()
    eng.reset(p0, 0)
    eng.prefill(ids, 16)
    c_pf, lg_pf, k_pf = eng.ctrl(), eng.logits(1)[0].astype(np.float64), rows()
    assert c_pf[mi.CTRL_POS] == c_ing[mi.CTRL_POS] == p0 + n
    assert np.all(np.abs(k_pf - k_ing) <= 0.03 * np.abs(k_ing).max()), np.abs(k_pf - k_ing).max()
    scale = np.abs(lg_ing).max()
    assert np.all(np.abs(lg_pf - lg_ing) <= 0.01 * scale), np.abs(lg_pf - lg_ing).max() / scale
    eng.close()
