"""The calls whose speed is watched: the LM's decode step and its layers'
projections, attention in its three forms, the DiT's block and projections,
and the depth decoder's stack, each through the package's public entry points.

A case's `kind` says which entry point it takes:

  lm       Lm.decode: one batched CFG decode step of the Qwen3-8B-shape LM
           (2 sets at the same position), logits and hidden states on the host
  proj     mmhip.mul_mat: the projections of one layer of a model (the LM's
           qkv, o, gate_up, down; the depth decoder's q, gate, down; the DiT's
           qkv, o, ff_in, ff_out), one product each on M tokens
  decode   mmhip.flash_attn_ext with one query token per set, the caches of
           several layers in turn
  prefill  mmhip.flash_attn_ext, causal over a key window padded to 256
  dit      mmhip.flash_attn_ext, bidirectional
  block    OpGraph.compute: the DiT block
  depth    OpGraph.compute: the depth decoder's four layers
"""
import ctypes
import importlib
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

PKG_DIR = pathlib.Path(__file__).resolve().parent.parent / "minimaxmusic.cpp_amd"


def _package():
    name = "mmcpp_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, PKG_DIR / "__init__.py",
                                                      submodule_search_locations=[str(PKG_DIR)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _module(name):
    return importlib.import_module(_package().__name__ + "." + name)


F32, F16, Q8_0, Q4_K, Q5_K, Q6_K, BF16 = 0, 1, 8, 12, 13, 14, 30
TYPES = {"q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K, "bf16": BF16, "q5_k_m": Q5_K}
BLOCKS = {Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), BF16: (1, 2)}

# LM: hidden 4096, 32 query / 8 KV heads of 128, FFN 12288, vocab 151936
LM_H, LM_NH, LM_NKV, LM_D, LM_FFN, LM_VOCAB, LM_MAX_SEQ = 4096, 32, 8, 128, 12288, 151936, 4608
LM_EPS, LM_THETA = 1e-6, 1e6
# (rows, columns) of the weights of one layer
PROJ = {"lm": [(6144, 4096), (4096, 4096), (24576, 4096), (4096, 12288)],
        "depth": [(4096, 4096), (6144, 4096), (4096, 6144)],
        "dit": [(6144, 2048), (2048, 2048), (16384, 2048), (2048, 8192)],
        "dit_qkv": [(6144, 2048)]}


def listed():
    return [
        # the reference's batched CFG decode step at a long context, Q8_0 file
        {"name": "lm_decode_q8_0_kv4096", "kind": "lm", "wtype": "q8_0", "layers": 36, "kv": 4096},
        # the Light preset's LM file early in a song: a ragged, short context
        {"name": "lm_decode_q5_k_m_kv691", "kind": "lm", "wtype": "q5_k_m", "layers": 36, "kv": 691},
        # one decoder layer's projections for the CFG pair
        {"name": "lm_proj_q8_0_m2", "kind": "proj", "model": "lm", "wtype": "q8_0", "tokens": 2},
        # the same for a short text prompt (40 tokens is the reference's logged prefill)
        {"name": "lm_proj_q8_0_m40", "kind": "proj", "model": "lm", "wtype": "q8_0", "tokens": 40},
        # and for a longer prompt, a length that fills no tile, the Q6_K file
        {"name": "lm_proj_q6_k_m333", "kind": "proj", "model": "lm", "wtype": "q6_k", "tokens": 333},
        # the DiT's QKV projection over two long sequences, Q4_K file
        {"name": "dit_qkv_q4_k_m8192", "kind": "proj", "model": "dit_qkv", "wtype": "q4_k", "tokens": 8192},
        # decode attention of eight layers
        {"name": "attn_decode_kv2048", "kind": "decode", "batch": 2, "heads": 32, "kv_heads": 8, "dim": 128,
         "kv": 2048, "layers": 8},
        # causal prefill attention
        {"name": "attn_prefill_s1024", "kind": "prefill", "batch": 2, "heads": 32, "kv_heads": 8, "dim": 128,
         "tokens": 1024, "past": 0},
        # bidirectional attention over a long song
        {"name": "attn_dit_s4096_d128", "kind": "dit", "batch": 2, "heads": 16, "dim": 128, "tokens": 4096},
        # and at the DiT's own head size, 689 latent frames and the timestep token
        {"name": "attn_dit_s690_d64", "kind": "dit", "batch": 2, "heads": 32, "dim": 64, "tokens": 690},
        # a DiT block of a diffusion step, CFG pair
        {"name": "dit_block_q8_0_s690", "kind": "block", "wtype": "q8_0", "tokens": 690, "batch": 2},
        # the depth decoder's stack at its last position, CFG pair
        {"name": "depth_q8_0_s8", "kind": "depth", "tokens": 8, "batch": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lm", "proj", "proj", "proj", "decode", "prefill", "dit", "block", "depth"])
    if kind == "lm":
        return {"kind": kind, "wtype": rng.choice(["q8_0", "q6_k", "q5_k_m", "bf16"]), "layers": rng.randint(2, 12),
                "kv": _log(rng, 33, 4096)}
    if kind == "proj":
        model = rng.choice(["lm", "lm", "depth", "dit"])
        wtype = rng.choice(["q8_0", "q4_k"] if model == "dit" else ["q8_0", "q4_k", "q5_k", "q6_k"])
        most = {"lm": 1024, "depth": 64, "dit": 4096}[model]
        return {"kind": kind, "model": model, "wtype": wtype, "tokens": _log(rng, 1, most)}
    if kind == "decode":
        return {"kind": kind, "batch": rng.choice([1, 2]), "heads": 32, "kv_heads": 8, "dim": 128,
                "kv": _log(rng, 40, 8192), "layers": rng.randint(4, 12)}
    if kind == "prefill":
        return {"kind": kind, "batch": rng.choice([1, 2]), "heads": 32, "kv_heads": 8, "dim": 128,
                "tokens": _log(rng, 17, 2048), "past": rng.choice([0, 0, _log(rng, 20, 1500)])}
    if kind == "dit":
        heads, dim = rng.choice([(16, 128), (32, 64)])
        return {"kind": kind, "batch": rng.choice([1, 2]), "heads": heads, "dim": dim, "tokens": _log(rng, 120, 4000)}
    if kind == "block":
        return {"kind": kind, "wtype": rng.choice(["q8_0", "q8_0", "bf16"]), "tokens": _log(rng, 60, 1500),
                "batch": rng.choice([1, 2, 2])}
    return {"kind": kind, "tokens": rng.randint(1, 8), "batch": rng.choice([1, 2, 2])}


# ---------------------------------------------------------------- sizes

def _weight_bytes(t, n, k):
    be, bb = BLOCKS[t]
    return n * (k // be) * bb


def _bumped(layer, n):
    """Layers of a Q5_K_M file whose V and down projections are Q6_K."""
    return layer < n // 9 or layer >= n - n // 7 or layer % 3 == 0


def _lm_weights(case):
    """(bytes, multiplications per token) of the LM's matrices."""
    n, t = case["layers"], TYPES[case["wtype"]]
    total, mults = _weight_bytes(t, LM_VOCAB, LM_H), LM_VOCAB * LM_H
    for l in range(n):
        high = Q6_K if case["wtype"] == "q5_k_m" and _bumped(l, n) else t
        for (rows, k), ty in (((5120, 4096), t), ((1024, 4096), high), ((4096, 4096), t), ((24576, 4096), t),
                              ((4096, 12288), high)):
            total += _weight_bytes(ty, rows, k)
            mults += rows * k
    return total, mults


def _window(case):
    """Keys of a prefill: past and new ones, padded to 256 as the LM pads."""
    return -(-(case["past"] + case["tokens"]) // 256) * 256


def work(case):
    kind = case["kind"]
    if kind == "lm":
        weights, mults = _lm_weights(case)
        kv = 2 * 2 * case["layers"] * LM_NKV * case["kv"] * LM_D * 2
        attn = 2 * case["layers"] * 4 * LM_NH * case["kv"] * LM_D
        return {"bytes": weights + kv + 2 * (2 * LM_H + LM_VOCAB) * 4, "flops": 2 * 2 * mults + attn}
    if kind == "proj":
        m, t = case["tokens"], TYPES[case["wtype"]]
        shapes = PROJ[case["model"]]
        return {"bytes": sum(_weight_bytes(t, n, k) + m * (n + k) * 4 for n, k in shapes),
                "flops": sum(2 * m * n * k for n, k in shapes)}
    if kind == "decode":
        b, h, d = case["batch"], case["heads"], case["dim"]
        one = 2 * b * h * d * 4 + 2 * b * case["kv_heads"] * case["kv"] * d * 2
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 4 * b * h * case["kv"] * d}
    if kind == "prefill":
        b, h, d, s, p = case["batch"], case["heads"], case["dim"], case["tokens"], case["past"]
        pairs = s * p + s * (s + 1) // 2
        return {"bytes": 2 * b * h * s * d * 4 + 2 * b * case["kv_heads"] * (s + p) * d * 2 + s * _window(case) * 2,
                "flops": 4 * b * h * d * pairs}
    if kind == "dit":
        b, h, d, s = case["batch"], case["heads"], case["dim"], case["tokens"]
        return {"bytes": b * h * s * d * (4 + 2 + 2 + 4), "flops": 4 * b * h * s * s * d}
    if kind == "block":
        m, dim, ff = case["tokens"] * case["batch"], 2048, 8192
        weights = [(dim, dim)] * 4 + [(2 * ff, dim), (dim, ff)]
        return {"bytes": sum(_weight_bytes(TYPES[case["wtype"]], n, k) for n, k in weights) + 2 * m * dim * 4,
                "flops": sum(2 * m * n * k for n, k in weights) + 4 * m * case["tokens"] * dim}
    m, dim, ff = case["tokens"] * case["batch"], 4096, 6144
    one = 4 * dim * dim + 3 * dim * ff
    return {"bytes": 4 * one * 34 // 32 + 2 * m * dim * 4, "flops": 4 * 2 * m * one}


def tolerance(case):
    kind = case["kind"]
    if kind == "lm":
        # int8 activation codes move with the last bits of what they code, and
        # with them all later layers: the whole step is 3e-2 from 64 bits
        return {"rel": 0.03}
    if kind == "proj":
        # up to 16 tokens the integer products are exact and only the order of
        # the 32-bit sums is free; above, operands rounded to f16 lie 3e-4
        # from 64 bits
        return {"rel": 2e-5} if case["tokens"] <= 16 else {"rel": 1.2e-3}
    if kind in ("decode", "prefill", "dit"):
        return {"rel": 1.2e-3}  # probabilities and V in f16: 3e-4 from 64 bits
    if kind == "block":
        # f16 operands, 8e-5 from 64 bits beside the residual; bf16: 1.9e-3
        return {"rel": 4e-4 if case["wtype"] != "bf16" else 8e-3}
    return {"rel": 0.02}  # int8 activations in four chained layers: 8e-3 from 64 bits


# --------------------------------------------------------------- inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _blocks(t, n, k, seed):
    """GGUF rows of a synthetic weight as device bytes; BF16: the values' bits."""
    if t == BF16:
        w = torch.randn((n, k), device="cuda", generator=_generator(seed)) * 0.02
        return w.bfloat16().view(torch.uint8).view(-1)
    return _module("synth").gguf_blocks_torch(t, n, k, seed)


class _DeviceArray:
    """A graph tensor's memory as torch.as_tensor takes it; the graph, whose
    buffer that is, lives as long."""

    def __init__(self, graph, tensor, shape):
        self.graph = graph
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "version": 2,
                                         "data": (int(tensor.contents.data), False)}


def _prepare_lm(case, seed):
    lm_mod = _module("lm")
    cfg = dict(lm_mod.QWEN3_8B, n_layers=case["layers"], wtype=TYPES[case["wtype"]],
               bump_type=Q6_K if case["wtype"] == "q5_k_m" else 0, max_seq=LM_MAX_SEQ)
    lm = lm_mod.Lm(seed=seed, **cfg)
    for s in (0, 1):
        lm.fill_kv(s, case["kv"] - 1, seed=seed * 2 + s)
    embeds = np.random.default_rng(seed).standard_normal((2, LM_H)).astype(np.float32)
    return {"lm": lm, "embeds": embeds, "pos": case["kv"] - 1}


def _prepare_proj(case, seed):
    mm = _package().mmhip
    t, m = TYPES[case["wtype"]], case["tokens"]
    g = _generator(seed)
    calls = []
    for i, (n, k) in enumerate(PROJ[case["model"]]):
        raw = _blocks(t, n, k, seed * 8 + i)
        w = mm.QuantWeight.from_gguf(t, raw, n, k)
        x = torch.randn((m, k), device="cuda", generator=g)
        out = torch.empty((m, n), device="cuda")
        need = mm.load().mmhip_mul_mat_workspace(t, n, k, m)
        calls.append((w, x, out, torch.empty(need, dtype=torch.uint8, device="cuda") if need else None))
    return {"mul_mat": mm.mul_mat, "calls": calls}


def _prepare_attn(case, seed):
    mm = _package().mmhip
    g = _generator(seed)
    kind, b, h, d = case["kind"], case["batch"], case["heads"], case["dim"]
    kvh = case.get("kv_heads", h)
    nq = 1 if kind == "decode" else case["tokens"]
    nkv = case["kv"] if kind == "decode" else _window(case) if kind == "prefill" else case["tokens"]
    mask = None
    if kind == "prefill":
        keys = torch.arange(nkv, device="cuda")[None, :]
        last = torch.arange(nq, device="cuda")[:, None] + case["past"]
        mask = torch.zeros((nq, nkv), device="cuda").masked_fill_(keys > last, float("-inf")).half().view(1, 1, nq, nkv)
    calls = []
    for _ in range(case.get("layers", 1)):
        q = torch.randn((b, h, nq, d), device="cuda", generator=g)
        k = torch.randn((b, kvh, nkv, d), device="cuda", generator=g).half()
        v = torch.randn((b, kvh, nkv, d), device="cuda", generator=g).half()
        out = torch.empty((b, nq, h, d), device="cuda")
        views = [mm.view_of(x) for x in (q, k, v)]
        need = mm.load().mmhip_flash_attn_workspace(*(ctypes.byref(x) for x in views))
        calls.append((q, k, v, out, torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")))
    return {"attn": mm.flash_attn_ext, "calls": calls, "mask": mask, "scale": float(np.float32(1 / np.sqrt(d)))}


def _block_weights(case):
    """(attribute, rows, columns or 0 for a vector) of a block's or layer's tensors."""
    if case["kind"] == "block":
        dim, ff = 2048, 8192
        mats = [("wq", dim, dim), ("wk", dim, dim), ("wv", dim, dim), ("wo", dim, dim), ("ff_in_w", 2 * ff, dim),
                ("ff_out_w", dim, ff)]
        vecs = [("norm1_w", dim), ("norm1_b", dim), ("norm2_w", dim), ("norm2_b", dim), ("ff_in_b", 2 * ff),
                ("ff_out_b", dim)]
    else:
        dim, ff = 4096, 6144
        mats = [("wq", dim, dim), ("wk", dim, dim), ("wv", dim, dim), ("wo", dim, dim), ("w_gate", ff, dim),
                ("w_up", ff, dim), ("w_down", dim, ff)]
        vecs = [("attn_norm", dim), ("ffn_norm", dim)]
    return mats, vecs


def _layer_arrays(case, seed, layer):
    """Device arrays of one layer: GGUF bytes of the matrices, f32 vectors."""
    mats, vecs = _block_weights(case)
    t = TYPES[case.get("wtype", "q8_0")]
    got = {n: _blocks(t, rows, k, (seed * 4 + layer) * 8 + i) for i, (n, rows, k) in enumerate(mats)}
    g = _generator(seed * 4 + layer)
    for n, size in vecs:
        base = 0.0 if n.endswith("_b") else 1.0
        got[n] = base + 0.05 * torch.randn(size, device="cuda", generator=g)
    return got


def _rows_in(case, seed):
    dim = 2048 if case["kind"] == "block" else 4096
    return torch.randn((case["batch"], case["tokens"], dim), device="cuda", generator=_generator(seed + 77))


def _prepare_graph(case, seed):
    og, dit = _module("opgraph"), case["kind"] == "block"
    kind = _module("ditgraph" if dit else "depthgraph")
    s, b, n_layers = case["tokens"], case["batch"], 1 if dit else 4
    g = og.OpGraph(n_tensors=100 * n_layers)
    layers = [kind.Block(g, wtype=TYPES[case["wtype"]]) if dit else kind.Layer(g) for _ in range(n_layers)]
    x = g.tensor(F32, [kind.DIM, s, b])
    pos = g.tensor(26, [s]) if dit else None  # GGML_TYPE_I32
    out = x
    for lw in layers:
        out = kind.build_block(g, lw, out, pos, s, b) if dit else kind.build_layer(g, lw, out, s, b)
    g.build([out])
    for i, lw in enumerate(layers):
        lw.upload(g, {n: a.cpu().numpy() for n, a in _layer_arrays(case, seed, i).items()})
    g.set(x, _rows_in(case, seed).cpu().numpy())
    if dit:
        g.set(pos, np.arange(s, dtype=np.int32))
    view = torch.as_tensor(_DeviceArray(g, out, (b, s, kind.DIM)), device="cuda")
    view.graph = g  # the outputs may outlive the state
    return {"graph": g, "out": view}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "lm":
        return _prepare_lm(case, seed)
    if kind == "proj":
        return _prepare_proj(case, seed)
    if kind in ("block", "depth"):
        return _prepare_graph(case, seed)
    return _prepare_attn(case, seed)


def run(state):
    if "lm" in state:
        lm = state["lm"]
        lm.set_pos(0, state["pos"])
        lm.set_pos(1, state["pos"])
        logits, hidden = lm.decode(state["embeds"], [0, 1])
        return {"logits": logits, "hidden": hidden}
    if "mul_mat" in state:
        return [state["mul_mat"](w, x, out=out, workspace=ws) for w, x, out, ws in state["calls"]]
    if "attn" in state:
        return [state["attn"](q, k, v, state["mask"], state["scale"], out=out, workspace=ws)
                for q, k, v, out, ws in state["calls"]]
    state["graph"].compute()
    return state["out"]


# ------------------------------------------------- the same in 64 bits

def _half_at(b, at):
    return b[..., at:at + 2].contiguous().view(torch.float16).double()


def _scales_k4(b):
    """The eight 6-bit (scale, min) pairs of 12 packed bytes."""
    b = b.to(torch.int32)
    lo, mid, hi = b[..., 0:4], b[..., 4:8], b[..., 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | (lo >> 6 << 4)], -1)
    mn = torch.cat([mid & 63, (hi >> 4) | (mid >> 6 << 4)], -1)
    return sc.double(), mn.double()


def _dequantize(t, raw, n, k):
    """GGUF rows (device bytes) to f64 [n, k]."""
    if t == BF16:
        return raw.view(torch.bfloat16).view(n, k).double()
    be, bb = BLOCKS[t]
    b = raw.view(n, k // be, bb)
    if t == Q8_0:
        return (b[..., 2:].contiguous().view(torch.int8).double() * _half_at(b, 0)).view(n, k)
    if t in (Q4_K, Q5_K):
        sc, mn = _scales_k4(b[..., 4:16])
        qs = b[..., -128:].to(torch.int32).view(n, -1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3).view(n, -1, 8, 32)
        if t == Q5_K:
            bit = torch.arange(8, device=b.device).view(1, 1, 8, 1)
            q = q + ((b[..., 16:48].to(torch.int32)[:, :, None] >> bit & 1) << 4)
        return (_half_at(b, 0)[..., None] * sc[..., None] * q.double() - _half_at(b, 2)[..., None] * mn[..., None]).view(n, k)
    ql = b[..., :128].to(torch.int32).view(n, -1, 2, 2, 32)
    qh = b[..., 128:192].to(torch.int32).view(n, -1, 2, 32)
    parts = [ql[..., 0, :] & 15, ql[..., 1, :] & 15, ql[..., 0, :] >> 4, ql[..., 1, :] >> 4]
    q = torch.stack([p | (qh >> 2 * i & 3) << 4 for i, p in enumerate(parts)], 3) - 32
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    return (q.double().view(n, -1, 16, 16) * (sc * _half_at(b, 208))[..., None]).view(n, k)


def _linear(t, raw, n, k, x):
    """x [m, k] f64 times the weight's rows, some rows at a time."""
    be, bb = BLOCKS[t]
    step, stride = 16384, k // be * bb
    return torch.cat([x @ _dequantize(t, raw[i * stride:(i + step) * stride], min(step, n - i), k).T
                      for i in range(0, n, step)], 1)


def _attention(q, k, v, mask, scale):
    """q [B, H, S, D], k, v [B, Hkv, N, D] -> [B, S, H, D], a head at a time."""
    b, h, s, d = q.shape
    out = torch.empty((b, s, h, d), dtype=torch.float64, device=q.device)
    for i in range(b):
        for j in range(h):
            kj, vj = (x[i, j // (h // k.shape[1])].double() for x in (k, v))
            p = q[i, j].double() @ kj.T * scale
            out[i, :, j] = torch.softmax(p if mask is None else p + mask.double(), -1) @ vj
    return out


def _rms(x, w, eps=LM_EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos, dims, base):
    """x [..., T, H, D]: NeoX pairs (i, i + dims / 2) of the first dims."""
    half = dims // 2
    ang = pos.double()[:, None] * base ** (-2.0 * torch.arange(half, device=x.device).double() / dims)
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :half], x[..., half:dims]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., dims:]], -1)


def _exact_lm(case, state):
    lm, pos = state["lm"], state["pos"]

    def dev(name):
        return torch.from_numpy(lm.get(name)).cuda()

    def vec(name):
        return dev(name).view(torch.float32)

    def lin(name, n, k, x):
        return _linear(lm.type_of(name), dev(name), n, k, x)

    h = torch.from_numpy(state["embeds"]).cuda().double()
    where = torch.full((2,), pos, device="cuda")
    for l in range(case["layers"]):
        p = "blk.%d." % l
        x = _rms(h, vec(p + "attn_norm"))
        if lm.has(p + "qkv"):
            qkv = lin(p + "qkv", 6144, LM_H, x)
        else:
            qkv = torch.cat([lin(p + "qk", 5120, LM_H, x), lin(p + "v", 1024, LM_H, x)], 1)
        q = _rope(_rms(qkv[:, :4096].view(2, LM_NH, LM_D), vec(p + "q_norm")), where, LM_D, LM_THETA)
        k = _rope(_rms(qkv[:, 4096:5120].view(2, LM_NKV, LM_D), vec(p + "k_norm")), where, LM_D, LM_THETA)
        v = qkv[:, 5120:].view(2, LM_NKV, LM_D)
        ck, cv = (dev("kv_%s4_%d" % (c, l)).view(torch.float16).view(2, LM_NKV, LM_MAX_SEQ, LM_D)[:, :, :pos].double()
                  for c in "kv")
        o = _attention(q[:, :, None], torch.cat([ck, k[:, :, None]], 2), torch.cat([cv, v[:, :, None]], 2), None,
                       1 / math.sqrt(LM_D))
        h = h + lin(p + "o_proj", LM_H, 4096, o.reshape(2, 4096))
        gu = lin(p + "gate_up", 2 * LM_FFN, LM_H, _rms(h, vec(p + "ffn_norm")))
        h = h + lin(p + "down", LM_H, LM_FFN, torch.nn.functional.silu(gu[:, :LM_FFN]) * gu[:, LM_FFN:])
    h = _rms(h, vec("output_norm"))
    return {"logits": lin("lm_head", LM_VOCAB, LM_H, h), "hidden": h}


def _exact_block(case, seed):
    w = _layer_arrays(case, seed, 0)
    t, dim, ff, nh, d = TYPES[case["wtype"]], 2048, 8192, 32, 64
    b, s = case["batch"], case["tokens"]

    def norm(x, i):
        x = torch.nn.functional.layer_norm(x, (dim,), eps=1e-5)
        return x * w["norm%d_w" % i].double() + w["norm%d_b" % i].double()

    def lin(name, n, k, x):
        return _linear(t, w[name], n, k, x)

    x = _rows_in(case, seed).double().view(b * s, dim)
    h = norm(x, 1)
    pos = torch.arange(s, device="cuda")
    q, k, v = (lin(n, dim, dim, h).view(b, s, nh, d) for n in ("wq", "wk", "wv"))
    q, k = (_rope(a, pos, 32, 10000.0) for a in (q, k))
    o = _attention(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), None, 1 / math.sqrt(d))
    x = x + lin("wo", dim, dim, o.reshape(b * s, dim))
    f = lin("ff_in_w", 2 * ff, dim, norm(x, 2)) + w["ff_in_b"].double()
    act = torch.nn.functional.silu(f[:, ff:]) * f[:, :ff]
    return (x + lin("ff_out_w", dim, ff, act) + w["ff_out_b"].double()).view(b, s, dim)


def _exact_depth(case, seed):
    dim, ff, nh, d = 4096, 6144, 16, 256
    b, s = case["batch"], case["tokens"]
    x = _rows_in(case, seed).double().view(b * s, dim)
    mask = torch.full((s, s), float("-inf"), device="cuda").triu(1)
    for layer in range(4):
        w = _layer_arrays(case, seed, layer)

        def lin(name, n, k, a):
            return _linear(Q8_0, w[name], n, k, a)

        h = _rms(x, w["attn_norm"])
        q, k, v = (lin(n, dim, dim, h).view(b, s, nh, d).transpose(1, 2) for n in ("wq", "wk", "wv"))
        x = x + lin("wo", dim, dim, _attention(q, k, v, mask, 1 / math.sqrt(d)).reshape(b * s, dim))
        h = _rms(x, w["ffn_norm"])
        act = torch.nn.functional.silu(lin("w_gate", ff, dim, h)) * lin("w_up", ff, dim, h)
        x = x + lin("w_down", dim, ff, act)
    return x.view(b, s, dim)


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        return _exact_block(case, seed)
    if kind == "depth":
        return _exact_depth(case, seed)
    if kind == "proj":
        t = TYPES[case["wtype"]]
        got = []
        for i, (_, x, _, _) in enumerate(_prepare_proj(case, seed)["calls"]):
            n, k = PROJ[case["model"]][i]
            got.append(_linear(t, _blocks(t, n, k, seed * 8 + i), n, k, x.double()))
        return got
    state = prepare(case, seed)
    if kind == "lm":
        return _exact_lm(case, state)
    mask = None if state["mask"] is None else state["mask"][0, 0]
    return [_attention(q, k, v, mask, state["scale"]) for q, k, v, _, _ in state["calls"]]
