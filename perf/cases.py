"""The workloads whose speed this library is judged by: single layers and blocks through the C entries
that a host engine binds, and whole engine calls, over the sizes that its configurations use.

  linear             a W4A16 linear at 1..16 rows (plain decode steps, speculative verification) and its fold
  prefill_linear     a W4A16 linear over a prompt chunk's rows
  prefill_mlp        gate||up with SwiGLU over a chunk's rows
  prefill_attention  a chunk's causal attention over the cache (f16, or the rotated int8 one)
  decode_attention   a step's attention over the cache (f16 or int8, contiguous or paged), with its merge
  moe_decode         the token boundary and one mixture-of-experts block of a decode step
  moe_prefill        the same of a prompt chunk
  generate           one token of Engine.generate, to its logits
  prefill            Engine.prefill of a whole prompt, to its logits and cache rows

Weights, activations and caches have the distributions of the synthetic models: uniform nibbles with
scales U(0.002, 0.02), activations and keys and values N(0, 1), int8 caches uniform with scales
U(0.005, 0.05), a router of N(0, 0.02).
"""
import importlib
import math

import torch

mi = importlib.import_module("intel-arc-inference-server_amd")

PAGE = 64           # positions per cache page (the paged configurations)
TGT = 64            # attention blocks per kv head
EPS = 1e-6
VOCAB = 151936
HIDDEN, INTER, Q_HEADS, KV_HEADS, HEAD_DIM = 5120, 17408, 40, 8, 128  # the 27B-shape decoder's layer
MOE_TABLE = 8192    # embedding rows a mixture-of-experts block draws its tokens from
ROUTE_WORDS = 32


def listed():
    return [
        # the smallest call: one square projection of one token
        {"name": "linear_token", "kind": "linear", "rows": 1, "K": 4096, "N": 4096},
        # gate||up of the 27B shape over the longest verification list of one launch
        {"name": "linear_verify16", "kind": "linear", "rows": 16, "K": 5120, "N": 34816},
        # q||k||v over an ordinary, ragged prompt
        {"name": "prefill_qkv_333", "kind": "prefill_linear", "rows": 333, "K": 5120, "N": 7168},
        # gate||up + SwiGLU over the largest chunk
        {"name": "prefill_mlp_2048", "kind": "prefill_mlp", "rows": 2048, "K": 5120, "N": 34816},
        # a 2048-token prompt's attention in the 27B shape
        {"name": "prefill_attn_2048", "kind": "prefill_attention", "rows": 2048, "pos": 0, "q_heads": 40, "kv_heads": 8,
         "head_dim": 128, "int8": False, "paged": False},
        # a ragged second chunk over the rotated int8 cache of the mixture-of-experts shape
        {"name": "prefill_attn_int8_777", "kind": "prefill_attention", "rows": 777, "pos": 3001, "q_heads": 16,
         "kv_heads": 2, "head_dim": 256, "int8": True, "paged": False},
        # long-context decode: int8, paged in 64-token blocks
        {"name": "decode_attn_128k", "kind": "decode_attention", "rows": 1, "keys": 131072, "q_heads": 40, "kv_heads": 8,
         "head_dim": 128, "int8": True, "paged": True},
        # a four-row verification step at an ordinary context
        {"name": "decode_attn_verify4", "kind": "decode_attention", "rows": 4, "keys": 4099, "q_heads": 40,
         "kv_heads": 8, "head_dim": 128, "int8": False, "paged": False},
        # one token through a block of 256 experts, top 8 and a shared one
        {"name": "moe_token", "kind": "moe_decode", "rows": 1, "experts": 256, "top_k": 8, "hidden": 2048, "inter": 512},
        # the largest chunk through the same block
        {"name": "moe_prefill_2048", "kind": "moe_prefill", "rows": 2048, "experts": 256, "top_k": 8, "hidden": 2048,
         "inter": 512},
        # streaming generation, token by token: eight layers of the 27B shape at context 4096
        {"name": "generate_token", "kind": "generate", "layers": 8, "pos": 4095, "int8_head": False},
        # a prompt from its ids to the first token's logits: four layers of the 27B shape
        {"name": "prefill_prompt_1500", "kind": "prefill", "layers": 4, "tokens": 1500},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "prefill_linear", "prefill_mlp", "prefill_attention", "decode_attention", "moe_decode",
                       "moe_prefill", "generate", "prefill"])
    c = {"kind": kind}
    if kind in ("linear", "prefill_linear", "prefill_mlp"):
        step = 64 if kind == "linear" else 128
        c["rows"] = rng.randint(1, 16) if kind == "linear" else _log_int(rng, 1, 2048)
        c["K"] = 64 * _log_int(rng, 16, 272)
        c["N"] = step * _log_int(rng, 1024 // step, min(34816, HIDDEN * 34816 // c["K"]) // step)
        if kind == "prefill_mlp" and rng.random() < 0.5:
            c["K"], c["N"] = HIDDEN, 2 * INTER
    elif kind == "prefill_attention":
        c.update(rng.choice([{"q_heads": 40, "kv_heads": 8, "head_dim": 128, "int8": False},
                             {"q_heads": 32, "kv_heads": 8, "head_dim": 128, "int8": False},
                             {"q_heads": 16, "kv_heads": 2, "head_dim": 256, "int8": False},
                             {"q_heads": 16, "kv_heads": 2, "head_dim": 256, "int8": True},
                             {"q_heads": 24, "kv_heads": 4, "head_dim": 256, "int8": True}]))
        c["rows"] = _log_int(rng, 1, 2048)
        c["pos"] = 0 if rng.random() < 0.4 else _log_int(rng, 1, 8192)
        c["paged"] = rng.random() < 0.3
    elif kind == "decode_attention":
        c.update(rng.choice([{"q_heads": 40, "kv_heads": 8, "head_dim": 128, "int8": False},
                             {"q_heads": 40, "kv_heads": 8, "head_dim": 128, "int8": True},
                             {"q_heads": 16, "kv_heads": 2, "head_dim": 256, "int8": False},
                             {"q_heads": 16, "kv_heads": 2, "head_dim": 256, "int8": True}]))
        c["rows"] = rng.choice([1, 1, 2, 3, 4, 5, 8])
        c["keys"] = _log_int(rng, 16, 131072 if c["int8"] else 65536)
        c["paged"] = rng.random() < 0.5
    elif kind in ("moe_decode", "moe_prefill"):
        c["rows"] = rng.randint(1, 8) if kind == "moe_decode" else _log_int(rng, 9, 2048)
        c["experts"] = rng.choice([32, 64, 128, 256, 256])
        c["top_k"] = rng.choice([2, 4, 6, 8, 8])
        c["hidden"] = 512 * rng.randint(2, 4)
        c["inter"] = 128 * rng.randint(2, 6)
    elif kind == "generate":
        c["layers"] = rng.randint(1, 8)
        c["pos"] = _log_int(rng, 1, 4400)
        c["int8_head"] = rng.random() < 0.3
    else:
        c["layers"] = rng.randint(1, 4)
        c["tokens"] = _log_int(rng, 2, 1500)
    return c


# ---- inputs -------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _words(g, *shape):
    return torch.randint(-2 ** 31, 2 ** 31, shape, generator=g, device="cuda", dtype=torch.int32)


def _uniform16(g, lo, hi, *shape):
    return torch.empty(shape, device="cuda").uniform_(lo, hi, generator=g).half()


def _normal16(g, *shape, std=1.0):
    return torch.empty(shape, device="cuda", dtype=torch.float16).normal_(0.0, std, generator=g)


def _norm_weights(g, n):
    return torch.empty(n, device="cuda").normal_(1.0, 0.02, generator=g).half().float()


def _int4(g, K, N):
    return _words(g, K // 8, N), _uniform16(g, 0.002, 0.02, K // 64, N)


def _expert_blocks(g, blocks, K, N):
    """Layout 1: per 16-column tile and 64-k group 128 nibble words and 16 f16 scales."""
    w = _words(g, blocks * (N // 16) * (K // 64), 136)
    w[:, 128:] = _uniform16(g, 0.002, 0.02, w.shape[0], 16).view(torch.int32)
    return w


def _router_tiles(w):
    """[N][K] f16 -> [N/16][K/8][8][16]"""
    N, K = w.shape
    return w.view(N // 16, 16, K // 8, 8).permute(0, 2, 3, 1).contiguous()


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, device="cuda", dtype=dtype)


def _shape(c):
    qh, kvh, hd = c["q_heads"], c["kv_heads"], c["head_dim"]
    sh = mi.AttnShape(qh, kvh, hd, hd, 0, (qh + 2 * kvh) * hd, qh * hd, (qh + kvh) * hd, hd ** -0.5, EPS, 0)
    return sh, mi.C.byref(sh)


def _cache(g, c, keys):
    """K and V rows [kv_heads][keys][head_dim] (the last page whole), their scales, the page table."""
    n, kvh, hd = -(-keys // PAGE) * PAGE, c["kv_heads"], c["head_dim"]
    s = {"len": n, "pages": None, "ks": None, "vs": None}
    for k in ("k", "v"):
        if c["int8"]:
            s[k] = torch.randint(-127, 128, (kvh, n, hd), generator=g, device="cuda", dtype=torch.int8)
            s[k + "s"] = _uniform16(g, 0.005, 0.05, kvh, n)
        else:
            s[k] = _normal16(g, kvh, n, hd)
    if c["paged"]:
        s["pages"] = torch.randperm(n // PAGE, generator=g, device="cuda", dtype=torch.int32)
    return s


def _ctrl(pos, rows, ids=None):
    c = torch.zeros(mi.CTRL_WORDS, device="cuda", dtype=torch.int32)
    c[mi.CTRL_POS], c[mi.CTRL_NACT] = pos, rows
    if ids is not None:
        c[mi.CTRL_CUR:mi.CTRL_CUR + rows] = ids
    return c


class _DeviceArray:
    """An engine's device buffer, as torch takes it (the tensor keeps this object, and so the engine)."""

    def __init__(self, engine, ptr, shape, typestr):
        self.engine = engine
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _device_tensor(engine, kind, layer, typestr, *shape):
    return torch.as_tensor(_DeviceArray(engine, engine.tensor(kind, layer)[0], shape, typestr), device="cuda")


def _engine(c, seed):
    if c["kind"] == "generate":
        max_len, head8 = 4608, int(c["int8_head"])
    else:
        max_len, head8 = c["tokens"] + 8, 0
    d = mi.dense_desc(c["layers"], HIDDEN, Q_HEADS, KV_HEADS, HEAD_DIM, INTER, VOCAB, max_len, attn_tgt=TGT,
                      lm_head_int8=head8)
    e = mi.Engine(d, seed=seed % 100003 + 17)
    # a quarter of the synthetic scales, so that the random model's residual stays far inside f16's range
    for li in range(c["layers"]):
        for kind in (mi.T_QKV_S, mi.T_O_S, mi.T_GU_S, mi.T_DOWN_S):
            p, n = e.tensor(kind, li)
            mi.call("mi_fill_f16", p, n // 2, seed + 8 * li + kind, 0, 0.0005, 0.005, e.stream)
    mi.call("mi_stream_sync", e.stream)
    logits = _device_tensor(e, mi.T_LOGITS, 0, "<f4", VOCAB)
    kv = [_device_tensor(e, k, 0, "<f2", c["layers"], KV_HEADS, max_len, HEAD_DIM) for k in (mi.T_KV_K, mi.T_KV_V)]
    return {"engine": e, "logits": logits, "kv": kv}


def _tokens(c, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, VOCAB, (c.get("tokens", 1),), generator=g).to(torch.int32).numpy()


def prepare(case, seed):
    c, g = dict(case), _gen(seed)
    kind, rows = c["kind"], c.get("rows")
    s = {"c": c, "stream": torch.cuda.current_stream().cuda_stream}
    if kind == "linear":
        K, N = c["K"], c["N"]
        s["q"], s["s"] = _int4(g, K, N)
        s["x"] = _normal16(g, rows, K)
        s["S"] = mi.lib().mi_gemv_pick_s(K, N)
        s["part"], s["out"] = _empty(s["S"], rows, N), _empty(rows, N, dtype=torch.float16)
    elif kind in ("prefill_linear", "prefill_mlp"):
        K, N = c["K"], c["N"]
        s["q"], s["s"] = _int4(g, K, N)
        s["x"] = _normal16(g, rows, K)
        s["out"] = _empty(rows, N) if kind == "prefill_linear" else _empty(rows, N // 2, dtype=torch.float16)
    elif kind in ("prefill_attention", "decode_attention"):
        qh, hd = c["q_heads"], c["head_dim"]
        keys = c["pos"] + rows if kind == "prefill_attention" else max(c["keys"], rows)
        s.update(_cache(g, c, keys))
        s["shape"], s["shape_ref"] = _shape(c)
        s["aq"] = torch.empty(rows, qh, hd, device="cuda").normal_(generator=g).half().float()
        s["out"] = _empty(rows, qh, hd, dtype=torch.float16)
        if kind == "prefill_attention":
            s["rot"] = _empty(rows, qh, hd)
        else:
            s["ctrl"] = _ctrl(keys - rows, rows)
            s["part"] = _empty(qh * TGT * rows * (hd + 2))
    elif kind in ("moe_decode", "moe_prefill"):
        H, I, E, slots = c["hidden"], c["inter"], c["experts"], c["top_k"] + 1
        R = s["R"] = -(-(E + 1) // 16) * 16
        s["router_rows"] = torch.zeros(R, H, device="cuda", dtype=torch.float16)
        s["router_rows"][:E + 1] = _normal16(g, E + 1, H, std=0.02)
        s["router"] = _router_tiles(s["router_rows"])
        s["gu"], s["dn"] = _expert_blocks(g, E + 1, H, 2 * I), _expert_blocks(g, E + 1, I, H)
        s["embed"] = _normal16(g, MOE_TABLE, H)
        s["w0"], s["w1"] = _norm_weights(g, H), _norm_weights(g, H)
        s["ids"] = torch.randint(0, MOE_TABLE, (rows,), generator=g, device="cuda", dtype=torch.int32)
        s["resid"], s["x"], s["y"] = (_empty(rows, H, dtype=torch.float16) for _ in range(3))
        s["logits"], s["route"] = _empty(rows, R), _empty(rows, ROUTE_WORDS, dtype=torch.int32)
        s["h"] = _empty(rows * slots, I, dtype=torch.float16)
        if kind == "moe_decode":
            s["ctrl"], s["rstd"] = _ctrl(0, rows, s["ids"]), _empty(rows)
            s["words"] = _empty(rows, H // 2)
            mi.call("mi_gemv_handoff_init", s["words"].data_ptr(), s["words"].numel(), s["stream"])
        else:
            s["list"], s["n"] = _empty(rows * slots, dtype=torch.int32), _empty(1, dtype=torch.int32)
            s["tiles"] = _empty((rows * slots + 63) // 64 + E + 1, 4, dtype=torch.int32)
            s["d"] = _empty(rows * slots, H, dtype=torch.float16)
    else:
        s.update(_engine(c, seed))
        s["ids"] = _tokens(c, seed)
        if kind == "generate":
            s["engine"].capture(1)
    return s


# ---- one pass -----------------------------------------------------------------------------------
def _p(t):
    return None if t is None else t.data_ptr()


def run(s):
    c, st = s["c"], s["stream"]
    kind, rows = c["kind"], c.get("rows")
    if kind == "linear":
        mi.call("mi_gemv_w4a16", _p(s["q"]), _p(s["s"]), _p(s["x"]), _p(s["part"]), rows, c["K"], c["N"], s["S"], st)
        mi.call("mi_fold_partials", _p(s["part"]), _p(s["out"]), None, s["S"], rows, c["N"], st)
        return s["out"]
    if kind in ("prefill_linear", "prefill_mlp"):
        mi.call("mi_gemm_w4a16" if kind == "prefill_linear" else "mi_gemm_w4a16_silu", _p(s["q"]), _p(s["s"]), _p(s["x"]),
                _p(s["out"]), rows, c["K"], c["N"], st)
        return s["out"]
    if kind == "prefill_attention":
        hd, n = c["head_dim"], s["len"]
        if c["int8"]:
            mi.call("mi_attn_prefill_kv8", _p(s["aq"]), _p(s["k"]), _p(s["v"]), _p(s["ks"]), _p(s["vs"]), hd, n * hd, 1, n,
                    _p(s["pages"]), PAGE, rows, c["pos"], s["shape_ref"], _p(s["rot"]), _p(s["out"]), st)
        else:
            mi.call("mi_attn_prefill", _p(s["aq"]), _p(s["k"]), _p(s["v"]), hd, n * hd, _p(s["pages"]), PAGE, rows,
                    c["pos"], s["shape_ref"], _p(s["out"]), st)
        return s["out"]
    if kind == "decode_attention":
        hd, n = c["head_dim"], s["len"]
        mi.call("mi_attn_decode", _p(s["ctrl"]), _p(s["aq"]), int(c["int8"]), _p(s["k"]), _p(s["v"]), _p(s["ks"]),
                _p(s["vs"]), hd, n * hd, 1, n, _p(s["pages"]), PAGE, n, _p(s["part"]), rows, TGT, s["shape_ref"], st)
        rotated = c["int8"] and hd == 256
        mi.call("mi_attn_reduce_kv8" if rotated else "mi_attn_reduce", _p(s["ctrl"]), _p(s["part"]), None, _p(s["out"]),
                rows, TGT, n, s["shape_ref"], st)
        return s["out"]
    if kind == "moe_decode":
        H, I, E, k = c["hidden"], c["inter"], c["experts"], c["top_k"]
        mi.call("mi_embed_norm", _p(s["ctrl"]), _p(s["embed"]), _p(s["resid"]), _p(s["w0"]), _p(s["x"]), _p(s["rstd"]),
                rows, H, MOE_TABLE, EPS, st)
        mi.call("mi_gemv_f16w", _p(s["router"]), _p(s["x"]), _p(s["logits"]), rows, H, s["R"], 16, st)
        mi.call("mi_moe_gate_up_routed", _p(s["logits"]), s["R"], _p(s["route"]), _p(s["x"]), _p(s["gu"]), _p(s["h"]),
                rows, E, k, H, I, st)
        mi.call("mi_moe_down_norm", _p(s["route"]), _p(s["h"]), _p(s["dn"]), _p(s["resid"]), rows, E, k, H, I,
                _p(s["w1"]), _p(s["y"]), _p(s["rstd"]), EPS, _p(s["words"]), None, 0, 0, st)
        return s["logits"], s["resid"], s["y"]
    if kind == "moe_prefill":
        H, I, E, k = c["hidden"], c["inter"], c["experts"], c["top_k"]
        mi.call("mi_embed_rows", _p(s["ids"]), _p(s["embed"]), _p(s["resid"]), rows, H, MOE_TABLE, None, st)
        mi.call("mi_res_norm", None, _p(s["resid"]), _p(s["w0"]), _p(s["x"]), rows, H, 0, EPS, st)
        mi.call("mi_gemv_f16w", _p(s["router"]), _p(s["x"]), _p(s["logits"]), rows, H, s["R"], 16, st)
        mi.call("mi_moe_route", _p(s["logits"]), _p(s["route"]), rows, E, k, s["R"], st)
        mi.call("mi_moe_prefill", _p(s["route"]), _p(s["x"]), _p(s["gu"]), _p(s["dn"]), _p(s["resid"]), rows, E, k, H, I,
                _p(s["list"]), _p(s["tiles"]), _p(s["n"]), _p(s["h"]), _p(s["d"]), st)
        mi.call("mi_res_norm", None, _p(s["resid"]), _p(s["w1"]), _p(s["y"]), rows, H, 0, EPS, st)
        return s["logits"], s["resid"], s["y"]
    e = s["engine"]
    if kind == "generate":
        e.reset(c["pos"], int(s["ids"][0]))
        e.generate(1)
        return s["logits"]
    e.reset(0, 0)
    e.prefill(s["ids"])
    return s["logits"], s["kv"]


# ---- what a pass cannot do without ---------------------------------------------------------------
def work(case):
    c = dict(case)
    kind, T = c["kind"], c.get("rows")

    def int4(K, N):
        return K * N * 17 / 32

    if kind in ("linear", "prefill_linear", "prefill_mlp"):
        K, N = c["K"], c["N"]
        out = {"linear": 2 * N, "prefill_linear": 4 * N, "prefill_mlp": N}[kind]
        return {"bytes": int4(K, N) + T * (2 * K + out), "flops": 2 * T * K * N}
    if kind in ("prefill_attention", "decode_attention"):
        qh, kvh, hd = c["q_heads"], c["kv_heads"], c["head_dim"]
        keys = c["pos"] + T if kind == "prefill_attention" else max(c["keys"], T)
        pairs = T * keys - T * (T - 1) // 2
        return {"bytes": 2 * kvh * keys * (hd + 2 if c["int8"] else 2 * hd) + T * qh * hd * 6, "flops": 4 * qh * hd * pairs}
    if kind in ("moe_decode", "moe_prefill"):
        H, I, E, slots = c["hidden"], c["inter"], c["experts"], c["top_k"] + 1
        used = 1 + E * (1 - (1 - c["top_k"] / E) ** T)  # experts that T rows' routes name, and the shared one
        return {"bytes": used * 3 * int4(H, I) + 2 * H * (E + 1) + T * (10 * H + 4 * (E + 1)),
                "flops": 2 * T * (slots * 3 * H * I + H * (E + 1))}
    qkv = (Q_HEADS + 2 * KV_HEADS) * HEAD_DIM
    layer = HIDDEN * qkv + Q_HEADS * HEAD_DIM * HIDDEN + 3 * HIDDEN * INTER
    T, keys = (1, c["pos"] + 1) if kind == "generate" else (c["tokens"], c["tokens"])
    pairs = T * keys - T * (T - 1) // 2
    head = HIDDEN * VOCAB * (1 if c.get("int8_head") else 17 / 32)
    return {"bytes": c["layers"] * (int4(layer, 1) + 4 * KV_HEADS * HEAD_DIM * keys) + head + 4 * VOCAB + T * 2 * HIDDEN,
            "flops": 2 * (c["layers"] * (T * layer + 2 * Q_HEADS * HEAD_DIM * pairs) + HIDDEN * VOCAB)}


def tolerance(case):
    # about four times the measured distance to the 64-bit results: one f16 rounding of an output is
    # 2e-4, the MLP rounds four times, the blocks once per operation, a prompt through every layer
    return {"rel": {"linear": 1e-3, "prefill_linear": 1e-3, "prefill_mlp": 2e-3, "prefill_attention": 1e-3,
                    "decode_attention": 1e-3, "moe_decode": 3e-3, "moe_prefill": 3e-3, "generate": 5e-4,
                    "prefill": 8e-3}[case["kind"]]}


# ---- the same in 64 bits -------------------------------------------------------------------------
def _deq(q, s):
    """Layout-0 words [K/8][N] and scales [K/64][N] as f64 [K][N]."""
    K8, N = q.shape
    sh = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    n = (q[:, None, :] >> sh[None, :, None]) & 15
    w = (n - 8).view(K8 // 8, 64, N).double() * s.double()[:, None, :]
    return w.view(K8 * 8, N)


def _deq_block(b, K, N):
    """One layout-1 block as f64 [K][N]."""
    t = b.view(N // 16, K // 64, 136)
    q = t[:, :, :128].reshape(N // 16, K // 64, 8, 16).permute(1, 2, 0, 3).reshape(K // 8, N)
    s = t[:, :, 128:].contiguous().view(torch.float16).view(N // 16, K // 64, 16).permute(1, 0, 2).reshape(K // 64, N)
    return _deq(q, s)


def _swiglu(gu):
    """Columns in blocks of 16: gate, up, gate, up, ..."""
    b = gu.view(gu.shape[0], -1, 2, 16)
    return (torch.nn.functional.silu(b[:, :, 0]) * b[:, :, 1]).reshape(gu.shape[0], -1)


def _rms(v, w):
    return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS) * w.double()


def _attend(q, k, v, first):
    """q [T][QH][HD], k and v [KVH][keys][HD] in f64; row t sees keys 0 .. first + t."""
    T, QH, HD = q.shape
    G, keys = QH // k.shape[0], k.shape[1]
    hidden = torch.arange(keys, device="cuda")[None, :] > first + torch.arange(T, device="cuda")[:, None]
    out = torch.empty_like(q)
    for h in range(QH):
        w = (q[:, h] @ k[h // G].T * HD ** -0.5).masked_fill_(hidden, -math.inf).softmax(-1)
        out[:, h] = w @ v[h // G]
    return out


def _unrotate():
    """The f64 matrix that takes a rotated head row back: y -> H_256 diag(s) y / 16."""
    words = (0xA197D809, 0xA6850592, 0xB205A73E, 0x20AFA769, 0x45C2CF64, 0xBEAEAACB, 0x75F39ADD, 0x2385A70C)
    sign = torch.tensor([-1.0 if words[j // 32] >> (j % 32) & 1 else 1.0 for j in range(256)], dtype=torch.float64)
    h = torch.ones(1, 1, dtype=torch.float64)
    for _ in range(8):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (h * sign[None, :] / 16).cuda()


def _cache64(s, c, keys):
    rows = torch.arange(keys, device="cuda")
    if s["pages"] is not None:
        rows = s["pages"].long()[rows // PAGE] * PAGE + rows % PAGE
    k, v = s["k"][:, rows].double(), s["v"][:, rows].double()
    if c["int8"]:
        k, v = k * s["ks"][:, rows, None].double(), v * s["vs"][:, rows, None].double()
    return k, v


def _moe64(s, c):
    H, I, E, top = c["hidden"], c["inter"], c["experts"], c["top_k"]
    r = s["embed"][s["ids"].long()].double()
    # x and the logits are stored as f16: without these two roundings near-ties route otherwise
    x = _rms(r, s["w0"]).half().double()
    logits = x @ s["router_rows"].double().T
    lg = logits[:, :E + 1].half().double()
    p, ids = torch.sort(lg[:, :E].softmax(-1), dim=-1, descending=True, stable=True)
    p, ids = p[:, :top], ids[:, :top]
    w = p / p.sum(-1, keepdim=True)
    gu, dn = s["gu"].view(E + 1, -1), s["dn"].view(E + 1, -1)
    for e in range(E + 1):
        t, k = torch.nonzero(ids == e, as_tuple=True) if e < E else (torch.arange(r.shape[0], device="cuda"), None)
        if t.numel():
            d = _swiglu(x[t] @ _deq_block(gu[e], H, 2 * I)) @ _deq_block(dn[e], I, H)
            r[t] += d * (w[t, k, None] if e < E else torch.sigmoid(lg[:, E:]))
    return logits, r, _rms(r, s["w1"])


def _forward64(c, seed):
    """The dense model's walk over the tokens, from the engine's own weights: (logits, K, V)."""
    s = _engine(c, seed)
    e, ids = s["engine"], torch.from_numpy(_tokens(c, seed)).long().cuda()

    def take(kind, layer, typestr, *shape):
        return _device_tensor(e, kind, layer, typestr, *shape)

    def lin(kind, layer, K, N):
        return _deq(take(kind, layer, "<i4", K // 8, N), take(kind + 1, layer, "<f2", K // 64, N))

    T, pos = ids.numel(), c.get("pos", 0)
    QD, KD, half = Q_HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM, HEAD_DIM // 2
    a = torch.arange(pos, pos + T, device="cuda").double()[:, None] * 1e6 ** (
        -torch.arange(half, device="cuda").double() / half)
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    kc, vc = (t.double() for t in s["kv"])
    r = take(mi.T_EMBED, 0, "<f2", VOCAB, HIDDEN)[ids].double()
    for li in range(c["layers"]):
        def norm(v, kind, n):
            return _rms(v, take(kind, li, "<f4", n))

        def rope(v, kind):
            v = norm(v.reshape(T, -1, HEAD_DIM), kind, HEAD_DIM)
            lo, hi = v[..., :half], v[..., half:]
            return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], -1)

        qkv = norm(r, mi.T_IN_NORM, HIDDEN) @ lin(mi.T_QKV_Q, li, HIDDEN, QD + 2 * KD)
        kc[li, :, pos:pos + T] = rope(qkv[:, QD:QD + KD], mi.T_K_NORM).transpose(0, 1)
        vc[li, :, pos:pos + T] = qkv[:, QD + KD:].reshape(T, KV_HEADS, HEAD_DIM).transpose(0, 1)
        o = _attend(rope(qkv[:, :QD], mi.T_Q_NORM), kc[li, :, :pos + T], vc[li, :, :pos + T], pos)
        r = r + o.reshape(T, QD) @ lin(mi.T_O_Q, li, QD, HIDDEN)
        h = _swiglu(norm(r, mi.T_POST_NORM, HIDDEN) @ lin(mi.T_GU_Q, li, HIDDEN, 2 * INTER))
        r = r + h @ lin(mi.T_DOWN_Q, li, INTER, HIDDEN)
    x = _rms(r[-1:], take(mi.T_FINAL_NORM, 0, "<f4", HIDDEN))[0]
    if c.get("int8_head"):
        # [N/16][K/64][lane][16]: lane l holds column l % 16 at k = 8 (l / 16) + e and 32 + 8 (l / 16) + e
        w = take(mi.T_LM_I8, 0, "|i1", VOCAB // 16, HIDDEN // 64, 4, 16, 2, 8)
        xk = x.view(HIDDEN // 64, 2, 4, 8)
        logits = torch.cat([torch.einsum("ngqchk,ghqk->nc", b.double(), xk) for b in w.split(1024)]).reshape(-1)
        logits = logits * take(mi.T_LM_I8_S, 0, "<f4", VOCAB).double()
    else:
        logits = x @ lin(mi.T_LM_Q, 0, HIDDEN, VOCAB)
    torch.cuda.synchronize()
    e.close()
    return logits, kc, vc


def exact(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind in ("generate", "prefill"):
        logits, k, v = _forward64(c, seed)
        return logits if kind == "generate" else (logits, [k, v])
    s = prepare(case, seed)
    if kind in ("linear", "prefill_linear", "prefill_mlp"):
        y = s["x"].double() @ _deq(s["q"], s["s"])
        return _swiglu(y) if kind == "prefill_mlp" else y
    if kind in ("prefill_attention", "decode_attention"):
        T = c["rows"]
        keys = c["pos"] + T if kind == "prefill_attention" else max(c["keys"], T)
        o = _attend(s["aq"].double(), *_cache64(s, c, keys), keys - T)
        return o @ _unrotate().T if c["int8"] and c["head_dim"] == 256 else o
    return _moe64(s, c)
