"""Workloads of this backend that are timed and checked: what a program that serves a quantized MoE model makes of its
public entry points (`HipBackend`, `qwen3moe.Model`), from one matrix-vector product to the whole 48-layer stack.

Kinds of case, and what they stand for:
  gemv          y[t] = W x[t] for 1 to 4 tokens (`gemv` / `gemvn`): a decode token's projection, or the lm head over
                the few tokens of a speculative step
  dense         `gemm_dense` of n tokens, x quantized inside the call: a projection of a prefill chunk, of a short
                prompt, or of a batch of decoding sequences
  moe           one routed-MoE block from the hidden rows to the combined expert outputs: FFN norm, F32 router, top-k,
                sort by expert, gate/up with SwiGLU, down, weighted combine; one token runs the decode launches
  attn_prefill  causal attention of a chunk of t tokens at position pos over the f16 KV cache (GQA)
  attn_decode   attention of nt decode tokens over a long f16 KV cache
  prefill       `Model.prefill` of a prompt: embedding, layers, the output norm and the lm head
  decode        `Model.decode_step` (the recorded graph) at a position of a filled KV cache

Weights are seeded random GGUF blocks whose scale fields give values of the size that trained weights have; the
experts' load is skewed as a Zipf law (s = 1.1) skews it. Whole models have few layers here: with random weights a
change of the last bit in one layer's attention changes the routing of some token in the next ones, and 48 layers turn
that into other logits (0.3 of them, against 0.03 for up to four layers).
"""
import math

import numpy as np
import torch

from rustingstrata_amd import ggml
from rustingstrata_amd.backend import ACT_STORE, X_Q, F32_TYPE, GpuTensor, HipBackend
from rustingstrata_amd.qwen3moe import Config, Model, Weights

DEV = "cuda"
EPS = 1e-6
TYPES = {n: t for t, n in ggml.NAMES.items()}
_HIP = None


def _hip():
    """The program's one backend context."""
    global _HIP
    if _HIP is None:
        _HIP = HipBackend(0)
    return _HIP


# ---- the cases ----
def listed():
    return [
        # a decode token's attention projection in the most used type: one launch, latency counts
        {"name": "gemv_q4k_4096", "kind": "gemv", "ty": "Q4_K", "rows": 4096, "cols": 4096, "nt": 1},
        # the lm head over the 3 tokens of a speculative step
        {"name": "gemvn_head_q6k_x3", "kind": "gemv", "ty": "Q6_K", "rows": 151936, "cols": 2048, "nt": 3},
        # the MoE block of one decode token
        {"name": "moe_1_q5k_q6k", "kind": "moe", "ty_gu": "Q5_K", "ty_d": "Q6_K", "t": 1, "E": 128, "k": 8, "H": 2048, "F": 768},
        # the MoE block of a short prompt (a chat turn, odd length)
        {"name": "moe_27_q2k_q3k", "kind": "moe", "ty_gu": "Q2_K", "ty_d": "Q3_K", "t": 27, "E": 128, "k": 8, "H": 2048, "F": 768},
        # the MoE block of an ordinary prompt, codebook experts
        {"name": "moe_512_iq4xs", "kind": "moe", "ty_gu": "IQ4_XS", "ty_d": "IQ4_XS", "t": 512, "E": 128, "k": 8, "H": 2048, "F": 768},
        # the MoE block of a full prefill chunk
        {"name": "moe_4096_q5k_q6k", "kind": "moe", "ty_gu": "Q5_K", "ty_d": "Q6_K", "t": 4096, "E": 128, "k": 8, "H": 2048, "F": 768},
        # a q/k/v projection of a short prompt or of a batch of decoding sequences
        {"name": "dense_24_q6k", "kind": "dense", "ty": "Q6_K", "rows": 5120, "cols": 2048, "n": 24},
        # a projection of a prefill chunk in the 8-bit type
        {"name": "dense_4096_q8_0", "kind": "dense", "ty": "Q8_0", "rows": 2048, "cols": 2048, "n": 4096},
        # attention of a full prefill chunk from position 0
        {"name": "attn_prefill_4096", "kind": "attn_prefill", "t": 4096, "pos": 0, "nh": 32, "nkv": 4, "hd": 128, "win": 0},
        # attention of one decode token over a long context
        {"name": "attn_decode_32k", "kind": "attn_decode", "nt": 1, "pos": 32700, "nh": 32, "nkv": 4, "hd": 128, "win": 0},
        # whole calls of the model, logits out: a prompt of odd length through one layer and the head, and one token at
        # the end of a 4096-token context through four layers and the head
        {"name": "prefill_1501", "kind": "prefill", "t": 1501, "layers": 1},
        {"name": "decode_at_4095", "kind": "decode", "pos": 4095, "layers": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "dense", "dense", "moe", "moe", "moe", "attn_prefill", "attn_decode", "prefill", "decode"])
    quants = ["Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q2_K", "Q3_K", "IQ4_XS", "IQ3_S", "IQ2_XXS"]
    if kind == "gemv":
        return {"kind": kind, "ty": rng.choice(quants), "rows": _log(rng, 500, 151936), "cols": rng.choice([768, 2048, 2048, 4096, 6144]), "nt": rng.choice([1, 1, 2, 3, 4])}
    if kind == "dense":
        return {"kind": kind, "ty": rng.choice(quants), "rows": rng.choice([512, 1000, 2048, 4096, 5120]), "cols": rng.choice([768, 2048, 4096]), "n": _log(rng, 5, 4096)}
    if kind == "moe":
        gu, d = rng.choice([("Q4_K", "Q6_K"), ("Q5_K", "Q6_K"), ("Q2_K", "Q3_K"), ("Q4_K", "Q5_K"), ("IQ4_XS", "IQ4_XS"), ("IQ3_S", "IQ4_XS"), ("IQ2_XXS", "IQ3_S")])
        E, k, H, F = rng.choice([(128, 8, 2048, 768), (128, 8, 2048, 768), (64, 6, 2048, 1024), (32, 4, 1024, 512)])
        return {"kind": kind, "ty_gu": gu, "ty_d": d, "t": _log(rng, 1, 4096), "E": E, "k": k, "H": H, "F": F}
    nh, nkv, hd = rng.choice([(32, 4, 128), (32, 4, 128), (32, 8, 128), (16, 8, 64), (16, 16, 128)])
    win = rng.choice([0, 0, 0, 1024])
    if kind == "attn_prefill":
        return {"kind": kind, "t": _log(rng, 16, 4096), "pos": rng.choice([0, 0, rng.randrange(1, 4096)]), "nh": nh, "nkv": nkv, "hd": hd, "win": win}
    if kind == "attn_decode":
        return {"kind": kind, "nt": rng.choice([1, 1, 2, 4]), "pos": _log(rng, 100, 32700), "nh": nh, "nkv": nkv, "hd": hd, "win": win}
    if kind == "prefill":
        return {"kind": kind, "t": _log(rng, 16, 4096), "layers": 1}
    return {"kind": kind, "pos": rng.randrange(64, 4096), "layers": rng.choice([1, 2, 4])}


# ---- inputs ----
def _gen(seed, part):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1009 + part) % (1 << 62))
    return g


def _randn(seed, part, *shape):
    return torch.randn(*shape, device=DEV, dtype=torch.float32, generator=_gen(seed, part))


# f16 scales (d, then dmin as a multiple of d, which centres the values) that give weights a deviation near 0.02
SCALES = {"Q8_0": (2.2e-4, 3.2e-4, 0), "Q2_K": (1.6e-3, 2.2e-3, 1.5), "Q3_K": (4.0e-4, 5.5e-4, 0), "Q4_K": (8e-5, 1.2e-4, 7.5),
          "Q5_K": (4e-5, 6e-5, 15.5), "Q6_K": (1.2e-5, 1.8e-5, 0), "IQ2_XXS": (3e-4, 4.5e-4, 0), "IQ3_S": (1.5e-4, 2.2e-4, 0),
          "IQ4_XS": (1.2e-5, 1.8e-5, 0)}


def _blocks(name, rows, cols, seed, part):
    """Random GGUF blocks [rows, row_bytes] of the type."""
    ty = TYPES[name]
    bb = ggml.block_bytes(ty)
    nb = rows * cols // ggml.block_elems(ty)
    g = _gen(seed, part)
    w = torch.randint(0, 1 << 62, ((nb * bb + 7) // 8,), device=DEV, dtype=torch.int64, generator=g)
    w = w.view(torch.uint8)[:nb * bb].view(nb, bb)
    w.bitwise_xor_(w.roll(3, 1))  # the words' top bits are not random; mix the bytes
    lo, hi, mn = SCALES[name]
    d = torch.empty(nb, device=DEV, dtype=torch.float32).uniform_(lo, hi, generator=g)
    for i, off in enumerate(ggml.F16_FIELDS[ty]):
        f = (d if i == 0 else d * mn).to(torch.float16)
        w[:, off:off + 2] = f.view(torch.uint8).view(nb, 2)
    return w.view(rows, -1)


class _View:
    """A device buffer of the backend, seen by torch."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(buf), False), "version": 2, "strides": None}


def _tensor(buf, shape, typestr="<f4"):
    return torch.as_tensor(_View(buf, shape, typestr), device=DEV)


def _weight(name, blocks):
    ty = TYPES[name]
    rows = blocks.shape[0]
    return GpuTensor(ty, rows, blocks.shape[1] // ggml.block_bytes(ty) * ggml.block_elems(ty), blocks.data_ptr())


def _moe_inputs(c, seed):
    E, H, F = c["E"], c["H"], c["F"]
    x = _randn(seed, 1, c["t"], H)
    nw = 1.0 + 0.1 * _randn(seed, 2, H)
    router = _randn(seed, 3, E, H) / math.sqrt(H)
    # channel 0 is a constant one that carries the experts' bias: 8 * rank^-1.1 over a permutation of the experts
    x[:, 0] = 2.0
    rank = torch.randperm(E, device=DEV, generator=_gen(seed, 4)).to(torch.float32) + 1.0
    router[:, 0] = 4.0 * rank ** -1.1
    gate_up = _blocks(c["ty_gu"], 2 * E * F, H, seed, 5)
    down = _blocks(c["ty_d"], E * H, F, seed, 6)
    return x, nw, router, gate_up, down


def _attn_inputs(c, seed):
    nt = c["t"] if c["kind"] == "attn_prefill" else c["nt"]
    n = c["pos"] + nt
    q = 1.5 * _randn(seed, 1, nt, c["nh"] * c["hd"])
    k = _randn(seed, 2, n, c["nkv"] * c["hd"]).to(torch.float16)
    v = (0.5 * _randn(seed, 3, n, c["nkv"] * c["hd"])).to(torch.float16)
    return q, k, v


def _config(c):
    return Config.qwen3_30b_a3b(n_layer=c["layers"])


class _State:
    pass


def prepare(case, seed):
    hip, c, s = _hip(), case, _State()
    s.c, kind = case, case["kind"]
    empty = lambda *shape, dtype=torch.float32: torch.empty(*shape, device=DEV, dtype=dtype)  # noqa: E731
    if kind == "gemv":
        s.blocks = _blocks(c["ty"], c["rows"], c["cols"], seed, 1)
        s.w = _weight(c["ty"], s.blocks)
        s.x = _randn(seed, 2, c["nt"], c["cols"])
        s.y = empty(c["nt"], c["rows"])
    elif kind == "dense":
        s.blocks = _blocks(c["ty"], c["rows"], c["cols"], seed, 1)
        s.w = _weight(c["ty"], s.blocks)
        s.x = _randn(seed, 2, c["n"], c["cols"])
        s.y = empty(c["n"], c["rows"])
    elif kind == "moe":
        t, E, k, H, F = c["t"], c["E"], c["k"], c["H"], c["F"]
        s.x, s.nw, s.rw, s.gu, s.dn = _moe_inputs(c, seed)
        s.router = GpuTensor(F32_TYPE, E, H, s.rw.data_ptr())
        s.ty_gu, s.ty_d = TYPES[c["ty_gu"]], TYPES[c["ty_d"]]
        s.e_gu, s.e_d = F * ggml.row_bytes(s.ty_gu, H), H * ggml.row_bytes(s.ty_d, F)
        s.acc = hip.alloc(t * H * 4)  # the block's output rows, cleared and added into
        s.out = _tensor(s.acc, (t, H))
        s.h, s.hq = empty(t, H), empty(t * (H + H // 8), dtype=torch.uint8)
        s.logits = empty(t, E)
        s.ids, s.wts = empty(t * k, dtype=torch.int32), empty(t * k)
        s.ge, s.ye = empty(2 if t == 1 else 1, t * k, F), empty(t * k, H)
        if t == 1:
            s.zero = torch.zeros(H, device=DEV)
            s.table = torch.arange(E, device=DEV, dtype=torch.int32)
            s.slots, s.wh = empty(k, dtype=torch.int32), empty(k)
        else:
            s.max_tiles = t * k // 64 + E
            s.off, s.xrow, s.inv = empty(E + 1, dtype=torch.int32), empty(t * k, dtype=torch.int32), empty(t * k, dtype=torch.int32)
            s.tiles = torch.zeros(2 * s.max_tiles * 2, device=DEV, dtype=torch.int64)
            s.ntd, s.err = torch.zeros(1, device=DEV, dtype=torch.int32), torch.zeros(1, device=DEV, dtype=torch.int32)
    elif kind == "attn_prefill":
        s.q, s.k, s.v = _attn_inputs(c, seed)
        s.step = torch.tensor([c["pos"], 0], device=DEV, dtype=torch.int32)
        s.out = torch.empty_like(s.q)
    elif kind == "attn_decode":
        s.q, s.k, s.v = _attn_inputs(c, seed)
        s.step = torch.tensor([[c["pos"] + i, 0] for i in range(c["nt"])], device=DEV, dtype=torch.int32)
        s.out = torch.empty_like(s.q)
        s.part = empty(c["nt"] * hip.attn_part_floats(c["nh"], c["hd"]))
    elif kind == "prefill":
        cfg = _config(c)
        s.m = Model(hip, Weights.random(hip, cfg, seed=int(seed) % 1000003), ctx=c["t"], chunk=min(c["t"], 4096))
        s.tokens = np.random.default_rng(int(seed)).integers(0, cfg.n_vocab, c["t"]).astype(np.int32)
        s.logits = _tensor(s.m.logits, (cfg.n_vocab,))
    elif kind == "decode":
        cfg = _config(c)
        s.m = Model(hip, Weights.random(hip, cfg, seed=int(seed) % 1000003), ctx=4096, chunk=16)
        kv = cfg.n_head_kv * cfg.head_dim
        for i in range(cfg.n_layer):  # the context before the token
            _tensor(s.m.kc[i], (4096, kv), "<f2").copy_(_randn(seed, 10 + 2 * i, 4096, kv))
            _tensor(s.m.vc[i], (4096, kv), "<f2").copy_(0.5 * _randn(seed, 11 + 2 * i, 4096, kv))
        s.token = np.random.default_rng(int(seed)).integers(0, cfg.n_vocab, 1).astype(np.int32)
        s.logits = _tensor(s.m.logits, (cfg.n_vocab,))
        # the program's first token, which records the decode graph; the KV row it writes is the one every pass writes
        hip.htod(s.token, s.m.tok)
        s.m.pos = c["pos"]
        s.m.decode_step(graph=False)
        s.m.pos = c["pos"]
        hip.htod(s.token, s.m.tok)
        s.m.decode_step()
    return s


# ---- one pass ----
def run(s):
    hip, c, kind = _hip(), s.c, s.c["kind"]
    if kind == "gemv":
        if c["nt"] == 1:
            hip.gemv(s.w, s.x.data_ptr(), s.y.data_ptr())
        else:
            hip.gemvn(s.w, s.x.data_ptr(), c["cols"], s.y.data_ptr(), c["rows"], c["nt"])
        return s.y
    if kind == "dense":
        hip.gemm_dense(s.w, c["n"], s.x.data_ptr(), c["cols"], s.y.data_ptr(), c["rows"], ACT_STORE)
        return s.y
    if kind == "moe":
        return _moe_decode(hip, s) if c["t"] == 1 else _moe_prefill(hip, s)
    if kind == "attn_prefill":
        hip.attn_prefill(s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), 0, s.out.data_ptr(), s.step.data_ptr(), c["t"], c["nh"],
                         c["nkv"], c["hd"], 1.0 / math.sqrt(c["hd"]), win=c["win"])
        return s.out
    if kind == "attn_decode":
        hip.attn_decode(s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), 0, s.out.data_ptr(), s.part.data_ptr(), s.step.data_ptr(),
                        c["nh"], c["nkv"], c["hd"], 1.0 / math.sqrt(c["hd"]), c["nt"], win=c["win"])
        return s.out
    if kind == "prefill":
        s.m.reset()
        s.m.prefill(s.tokens)
        return s.logits
    hip.htod(s.token, s.m.tok)
    s.m.pos = c["pos"]
    s.m.decode_step()
    return s.logits


def _moe_decode(hip, s):
    c = s.c
    k, H, F, E = c["k"], c["H"], c["F"], c["E"]
    p = lambda t: t.data_ptr()  # noqa: E731
    g = p(s.ge)
    hip.memset(s.acc)
    hip.rms_norm_q_gemv_f32(p(s.x), p(s.zero), p(s.nw), p(s.h), p(s.hq), H, EPS, s.router, p(s.logits))
    hip.moe_route_gemv(p(s.logits), E, k, 0.0, p(s.table), p(s.ids), p(s.wts), p(s.slots), p(s.wh), s.ty_gu, F, H, p(s.gu), s.e_gu,
                       p(s.h), g, pair=(E * s.e_gu, k * F * 4), xq=p(s.hq))
    hip.moe_down_swiglu_combine(s.ty_d, H, F, p(s.dn), s.e_d, p(s.slots), k, g, g + k * F * 4, p(s.ye), s.acc, p(s.wh), 0, 0, 1)
    return s.out


def _moe_prefill(hip, s):
    c = s.c
    t, k, H, F, E = c["t"], c["k"], c["H"], c["F"], c["E"]
    p = lambda x: x.data_ptr()  # noqa: E731
    hip.memset(s.acc)
    hip.rms_norm_q(p(s.x), H, p(s.nw), p(s.h), H, H, t, EPS, xq=p(s.hq))
    hip.gemm_dense(s.router, t, p(s.h), H, p(s.logits), E, ACT_STORE)
    hip.router_topk(p(s.logits), E, k, 0.0, p(s.ids), p(s.wts), t)
    chunk, small = hip.moe_tile_plan(t, k, E)
    hip.moe_sort(p(s.ids), t, k, E, p(s.off), p(s.xrow), p(s.inv), [(p(s.gu), s.e_gu), (p(s.dn), s.e_d)], p(s.tiles), s.max_tiles,
                 p(s.ntd), err_dev=p(s.err), chunk=chunk)
    hip.gemm_grouped_gate_up(s.ty_gu, F, H, p(s.tiles), s.max_tiles, p(s.ntd), p(s.hq), H, t, p(s.xrow), p(s.ge), F, E * s.e_gu,
                             flags=X_Q | small)
    hip.gemm_grouped(s.ty_d, H, F, p(s.tiles) + s.max_tiles * 16, s.max_tiles, p(s.ntd), p(s.ge), F, t * k, 0, p(s.ye), H,
                     ACT_STORE | small)
    hip.moe_combine_seq(s.acc, p(s.ye), p(s.wts), p(s.inv), k, 0, 0, H, t)
    return s.out


# ---- what a pass cannot do without ----
def _experts_used(c, t):
    """Experts that t tokens reach, at the skew of the cases: the skewed ones always, the rest as uniform draws would."""
    return c["E"] * (1.0 - (1.0 - c["k"] / c["E"]) ** (0.6 * t + 0.4))


def work(case):
    c, kind = case, case["kind"]
    if kind in ("gemv", "dense"):
        n = c["nt"] if kind == "gemv" else c["n"]
        return {"bytes": c["rows"] * ggml.row_bytes(TYPES[c["ty"]], c["cols"]) + 4 * n * (c["rows"] + c["cols"]),
                "flops": 2 * n * c["rows"] * c["cols"]}
    if kind == "moe":
        return _moe_work(c)
    if kind in ("attn_prefill", "attn_decode"):
        nt = c["t"] if kind == "attn_prefill" else c["nt"]
        keys = sum(min(c["pos"] + i + 1, c["win"] or 1 << 60) for i in range(nt))
        seen = min(c["pos"] + nt, (c["win"] or 1 << 60) + nt - 1)
        return {"bytes": 4 * seen * c["nkv"] * c["hd"] + 8 * nt * c["nh"] * c["hd"], "flops": 4 * keys * c["nh"] * c["hd"]}
    cfg = _config(c)
    H, a, kv = cfg.n_embd, cfg.n_head * cfg.head_dim, cfg.n_head_kv * cfg.head_dim
    t = c["t"] if kind == "prefill" else 1
    pos = 0 if kind == "prefill" else c["pos"]
    moe = _moe_work({"t": t, "E": cfg.n_expert, "k": cfg.n_expert_used, "H": H, "F": cfg.n_ff_exp, "ty_gu": "Q2_K", "ty_d": "Q3_K"})
    proj = (a + 2 * kv) * ggml.row_bytes(cfg.ty_attn, H) + H * ggml.row_bytes(cfg.ty_attn, a)
    keys = t * pos + t * (t + 1) // 2
    layer_b = moe["bytes"] + proj + 4 * (pos + t) * kv
    layer_f = moe["flops"] + 2 * t * H * (2 * a + 2 * kv) + 4 * keys * a
    head = cfg.n_vocab * ggml.row_bytes(cfg.ty_out, H)
    return {"bytes": cfg.n_layer * layer_b + head, "flops": cfg.n_layer * layer_f + 2 * cfg.n_vocab * H}


def _moe_work(c):
    t, E, k, H, F = c["t"], c["E"], c["k"], c["H"], c["F"]
    expert = 2 * F * ggml.row_bytes(TYPES[c["ty_gu"]], H) + H * ggml.row_bytes(TYPES[c["ty_d"]], F)
    return {"bytes": _experts_used(c, t) * expert + 4 * E * H + 8 * t * H, "flops": t * (6 * k * H * F + 2 * E * H)}


# ---- what another correct implementation may differ by ----
def tolerance(case):
    kind = case["kind"]
    if kind in ("gemv", "dense"):
        # int8 products, 32-bit sums in another order: 1e-7 from the sums in 64 bits
        return {"rel": 2e-6, "max": 4e-5}
    if kind == "moe":
        # a SwiGLU or norm value that rounds to the next int8 step now and then: 5e-4 from the block in 64 bits
        return {"rel": 2e-3, "max": 0.1}
    if kind in ("attn_prefill", "attn_decode"):
        # 32-bit softmax and sums in another order: 5e-7 from the sums in 64 bits
        return {"rel": 3e-6, "max": 1e-4}
    # whole calls: a last-bit change in the attention becomes an int8 step, or another expert at the edge of the top k
    # (the attention's scale changed by 1e-7 to 1e-6: up to 0.025 over 16 models of one to four layers)
    return {"rel": 0.03, "max": 0.5}


# ---- the same in 64 bits, plainly ----
def _dequant(name, w, rows, cols):
    """Values of GGUF blocks [rows, row_bytes] as float64 [rows, cols], as the formats define them."""
    ty = TYPES[name]
    b = w.reshape(-1, ggml.block_bytes(ty))
    f16 = lambda o: b[:, o:o + 2].contiguous().view(torch.float16).to(torch.float64)  # noqa: E731
    u = lambda o, n: b[:, o:o + n].to(torch.int32)  # noqa: E731
    n = b.shape[0]
    if name == "Q8_0":
        v = f16(0) * b[:, 2:34].contiguous().view(torch.int8).to(torch.float64)
    elif name in ("Q4_K", "Q5_K"):
        s = u(4, 12)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = u(16 if name == "Q4_K" else 48, 128).view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32)
        if name == "Q5_K":
            q = q + 16 * ((u(16, 32).view(n, 1, 32) >> torch.arange(8, device=w.device).view(1, 8, 1)) & 1)
        v = (f16(0) * sc).unsqueeze(2) * q - (f16(2) * mn).unsqueeze(2)
    elif name == "Q6_K":
        ql, qh = u(0, 128).view(n, 2, 1, 2, 32), u(128, 64).view(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2).view(n, 2, 4, 32)
        q = (lo | (((qh >> (2 * torch.arange(4, device=w.device)).view(1, 1, 4, 1)) & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        v = f16(208).unsqueeze(2) * sc.unsqueeze(2) * q.reshape(n, 16, 16)
    elif name in ("Q2_K", "Q3_K"):
        sh = (2 * torch.arange(4, device=w.device)).view(1, 1, 4, 1)
        q = (u(16 if name == "Q2_K" else 32, 64).view(n, 2, 1, 32) >> sh) & 3
        if name == "Q2_K":
            s = u(0, 16)
            v = (f16(80) * (s & 15)).unsqueeze(2) * q.reshape(n, 16, 16) - (f16(82) * (s >> 4)).unsqueeze(2)
        else:
            hm = (u(0, 32).view(n, 1, 32) >> torch.arange(8, device=w.device).view(1, 8, 1)) & 1
            q = q.reshape(n, 8, 32) - 4 * (1 - hm)
            s = u(96, 12)
            lo = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
            hi = torch.cat([(s[:, 8:12] >> (2 * i)) & 3 for i in range(4)], 1)
            v = (f16(108) * ((lo | (hi << 4)) - 32)).unsqueeze(2) * q.reshape(n, 16, 16)
    elif name == "IQ4_XS":
        kv = torch.tensor([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113], device=w.device, dtype=torch.float64)
        i8 = torch.arange(8, device=w.device).view(1, 8)
        h = (u(2, 1) | (u(3, 1) << 8))
        ls = ((u(4, 4).repeat_interleave(2, 1) >> (4 * (i8 & 1))) & 15) | (((h >> (2 * i8)) & 3) << 4)
        qs = u(8, 128).view(n, 8, 16)
        v = (f16(0) * (ls - 32)).unsqueeze(2) * kv[torch.cat([qs & 15, qs >> 4], 2).long()]
    else:
        return None
    return v.reshape(rows, cols)


def _q8k(x):
    """Activations as every product reads them: int8 steps of one scale per 256 values, -127 / the value of largest magnitude."""
    n = x.shape[1]
    b = torch.nn.functional.pad(x.to(torch.float32), (0, -n % 256)).view(x.shape[0], -1, 256)
    top = torch.gather(b, 2, b.abs().argmax(2, keepdim=True))
    f = torch.where(top == 0, torch.zeros_like(top), -127.0 / top)
    q = torch.round(b * f).clamp(max=127.0)
    d = torch.where(top == 0, torch.zeros_like(top), 1.0 / f)
    return (q.to(torch.float64) * d.to(torch.float64)).view(x.shape[0], -1)[:, :n]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("gemv", "dense"):
        w = _dequant(c["ty"], _blocks(c["ty"], c["rows"], c["cols"], seed, 1), c["rows"], c["cols"])
        return None if w is None else _q8k(_randn(seed, 2, c["nt"] if kind == "gemv" else c["n"], c["cols"])) @ w.T
    if kind == "moe":
        return _moe_exact(c, seed)
    if kind in ("attn_prefill", "attn_decode"):
        q, k, v = (a.to(torch.float64) for a in _attn_inputs(c, seed))
        nt, nh, nkv, hd = q.shape[0], c["nh"], c["nkv"], c["hd"]
        out = torch.empty_like(q)
        at = c["pos"] + torch.arange(nt, device=DEV).view(-1, 1)
        key = torch.arange(k.shape[0], device=DEV).view(1, -1)
        hidden = (key > at) | (key <= at - c["win"] if c["win"] else key < 0)
        for h in range(nh):
            g = h // (nh // nkv)
            sc = (q[:, h * hd:(h + 1) * hd] @ k[:, g * hd:(g + 1) * hd].T) / math.sqrt(hd)
            out[:, h * hd:(h + 1) * hd] = torch.softmax(sc.masked_fill_(hidden, -math.inf), 1) @ v[:, g * hd:(g + 1) * hd]
        return out
    return None


def _moe_exact(c, seed):
    if c["ty_gu"] in ("IQ3_S", "IQ2_XXS") or c["ty_d"] in ("IQ3_S", "IQ2_XXS"):
        return None
    x, nw, router, gate_up, down = _moe_inputs(c, seed)
    E, H, F = c["E"], c["H"], c["F"]
    x = x.to(torch.float64)
    h = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * nw
    p, ids = torch.softmax(h @ router.to(torch.float64).T, 1).topk(c["k"], 1)
    p = p / p.sum(1, keepdim=True)
    hq, y = _q8k(h), torch.zeros_like(x)
    gate_up, down = gate_up.view(2, E, F, -1), down.view(E, H, -1)
    for e in range(E):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if len(tok):
            g, u = (hq[tok] @ _dequant(c["ty_gu"], gate_up[i, e], F, H).T for i in range(2))
            act = _q8k(g / (1.0 + torch.exp(-g)) * u)
            y.index_add_(0, tok, (act @ _dequant(c["ty_d"], down[e], H, F).T) * p[tok, slot].unsqueeze(1))
    return y
