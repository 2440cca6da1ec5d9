"""What this framework's users have it do, as cases that can be timed and compared.

A case is a whole decode step, or one block of a Llama graph (an MLP, an attention layer, a
product, a soft_max, a weight load, a product routed to experts), through the package's entry
points.  The shapes are those of the repository's two decoder configurations (SmolLM2-135M and
Llama 1B) and its prefill workload, ragged prompt lengths among them.  Every result is an LNS
code or its F32 value, formed in a fixed term order, so two correct implementations agree in
every bit: tolerance() is "exact" throughout.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "xlns-ggml-backend_amd"))

import lnship  # noqa: E402
from lnship.llama import LlamaConfig, LlamaLNS16, n_kv_for  # noqa: E402

DEV = "cuda"
STD = 0.02        # weights N(0, STD^2), as in the decoder configurations
EPS = 1e-5
THETA = 10000.0


def listed():
    return [
        # one user's chat: the next token after a 128-token prompt, SmolLM2-135M shape
        {"name": "decode_sum32", "kind": "decode", "mode": "sum32", "seqs": 1, "past": 128},
        # eight users' next tokens in one step, after 256-token prompts
        {"name": "decode8_monte", "kind": "decode", "mode": "monte", "seqs": 8, "past": 256},
        # the smallest product of a decode step: one token's key (or value) projection
        {"name": "gemv_base_kv", "kind": "mm16", "mode": "base", "K": 576, "M": 192, "N": 1},
        # prefill throughput: 512 tokens against a 2048 x 8192 matrix
        {"name": "gemm_sum32", "kind": "mm16", "mode": "sum32", "K": 2048, "M": 8192, "N": 512},
        # a down projection of a ragged prompt
        {"name": "gemm_base_ragged", "kind": "mm16", "mode": "base", "K": 1536, "M": 576, "N": 131},
        # a SmolLM2 MLP (norm, up | gate, swiglu, down, residual) over a ragged prompt
        {"name": "ffn_lpvip", "kind": "ffn16", "mode": "lpvip", "E": 576, "F": 1536, "N": 201},
        # a SmolLM2 attention layer over a ragged prompt: rope, cache stores, kq, soft_max, kqv
        {"name": "attn_sum32", "kind": "attn16", "mode": "sum32", "H": 9, "HKV": 3, "D": 64, "T": 203, "past": 0},
        # the longest chains of an LNS32 decode step: the Llama-1B down projection
        {"name": "gemv_lns32_down", "kind": "mm32", "K": 8192, "M": 2048, "N": 1},
        # a Llama-1B MLP in LNS32 over a short prompt
        {"name": "ffn_lns32", "kind": "ffn32", "E": 2048, "F": 8192, "N": 64},
        # prefill scores of 32 heads under a causal mask
        {"name": "soft_max_base", "kind": "soft_max", "mode": "base", "H": 32, "T": 512, "n_kv": 512},
        # loading a model: one half-precision matrix into the weight cache
        {"name": "pack16", "kind": "pack", "width": 16, "half": True, "K": 2048, "M": 8192},
        # a mixture-of-experts projection: 37 tokens, each to 2 of 8 experts
        {"name": "moe_monte", "kind": "moe", "mode": "monte", "K": 576, "M": 1536, "T": 37, "experts": 8, "used": 2},
    ]


# MACs a drawn case may cost: the largest listed product's, less for the slower adders
MACS = {"base": 8e9, "monte": 6e9, "lpvip": 2.5e9, "sum32": 8e9, "lns32": 8e9}


def draw(rng):
    mode = rng.choice(["base", "monte", "lpvip", "sum32"])
    kind = rng.choice(["decode", "mm16", "mm16", "ffn16", "attn16", "mm32", "ffn32", "soft_max", "pack", "moe"])

    def size(lo, hi):   # spread over the logarithm, odd ones among them
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "decode":   # one or a few sequences at some position of a 512-cell context (as far as a step costs no more than the listed ones)
        mode = rng.choice(["base", "monte", "sum32"])
        if mode == "sum32":
            return {"kind": kind, "mode": mode, "seqs": 1, "past": rng.randint(2, 250)}
        return {"kind": kind, "mode": mode, "seqs": rng.choice([1, 1, 2, 3, 5, 8]), "past": rng.randint(2, 250)}
    if kind in ("mm16", "mm32"):
        K, M = size(32, 8192), size(16, 8192)
        top = MACS[mode if kind == "mm16" else "lns32"]
        N = 1 if rng.random() < 0.3 else max(1, min(size(2, 512), int(top // (K * M))))
        c = {"kind": kind, "K": K, "M": M, "N": N}
        return dict(c, mode=mode) if kind == "mm16" else c
    if kind in ("ffn16", "ffn32"):
        E, F = (576, 1536) if rng.random() < 0.5 else (8 * size(16, 256), 8 * size(32, 1024))
        N = max(1, min(size(2, 512), int(MACS[mode if kind == "ffn16" else "lns32"] // (3 * E * F))))
        c = {"kind": kind, "E": E, "F": F, "N": N}
        return dict(c, mode=mode) if kind == "ffn16" else c
    if kind == "attn16":
        HKV = rng.choice([1, 2, 3, 4, 8])
        T = size(2, 400)
        return {"kind": kind, "mode": mode, "H": HKV * rng.choice([1, 2, 3, 4]), "HKV": HKV, "D": rng.choice([32, 64, 64, 128]),
                "T": T, "past": rng.choice([0, rng.randint(1, 100)])}
    if kind == "soft_max":
        n_kv = size(16, 1024)
        return {"kind": kind, "mode": mode if rng.random() < 0.8 else "lns32", "H": rng.randint(1, 32),
                "T": min(size(1, 512), n_kv), "n_kv": n_kv}
    if kind == "pack":
        return {"kind": kind, "width": rng.choice([16, 16, 32]), "half": rng.random() < 0.5, "K": size(64, 8192), "M": size(64, 2048)}
    experts = rng.choice([4, 8, 16])
    return {"kind": "moe", "mode": mode if rng.random() < 0.8 else "lns32", "K": size(64, 2048), "M": size(64, 1536),
            "T": size(1, 128), "experts": experts, "used": rng.choice([1, 2, 4])}


# ---- inputs ---------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) + 1)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _mask(T, past, n_kv):
    j = torch.arange(n_kv, device=DEV)
    t = torch.arange(past, past + T, device=DEV)
    return torch.where(j[None, :] <= t[:, None], 0.0, float("-inf")).to(torch.float32)


def _config(case):
    return LlamaConfig(n_ctx=512)   # the SmolLM2-135M shape


def _llama_weights(cfg, g):
    """Weights of the architecture, random-initialised on the GPU, as the decoder takes them (host arrays)."""
    e, f, d = cfg.n_embd, cfg.n_ff, cfg.head_dim
    nq, nkv = cfg.n_head * d, cfg.n_head_kv * d

    def m(rows, cols):
        return _normal(g, rows, cols, std=STD)

    w = {"tok_embd": m(cfg.n_vocab, e), "out_norm": torch.ones(e, device=DEV), "layers": []}
    for _ in range(cfg.n_layer):
        w["layers"].append({"attn_norm": torch.ones(e, device=DEV), "wq": m(nq, e), "wk": m(nkv, e), "wv": m(nkv, e), "wo": m(e, nq),
                            "ffn_norm": torch.ones(e, device=DEV), "w_gate": m(f, e), "w_up": m(f, e), "w_down": m(e, f)})
    return w


def _decode_inputs(case, seed):
    cfg, g = _config(case), _gen(seed)
    w = _llama_weights(cfg, g)
    prompts = torch.randint(0, cfg.n_vocab, (case["seqs"], case["past"]), generator=g, device=DEV)
    nxt = torch.randint(0, cfg.n_vocab, (case["seqs"],), generator=g, device=DEV, dtype=torch.int32)
    return cfg, w, prompts, nxt


def _mm_inputs(case, seed):
    g = _gen(seed)
    return _normal(g, case["M"], case["K"], std=STD), _normal(g, case["N"], case["K"])


def _ffn_inputs(case, seed):
    g, E, F = _gen(seed), case["E"], case["F"]
    return _normal(g, case["N"], E), 1.0 + _normal(g, E, std=0.1), _normal(g, 2 * F, E, std=STD), _normal(g, E, F, std=STD)


def _attn_inputs(case, seed):
    g, w = _gen(seed), (case["H"] + 2 * case["HKV"]) * case["D"]
    return _normal(g, case["T"], w), _normal(g, max(case["past"], 1), w)


def _soft_max_inputs(case, seed):
    x = _normal(_gen(seed), 1, case["H"], case["T"], case["n_kv"], std=3.0)
    return x, _mask(case["T"], case["n_kv"] - case["T"], case["n_kv"])


def _pack_inputs(case, seed):
    w = _normal(_gen(seed), case["M"], case["K"], std=STD)
    return w.half() if case["half"] else w


def _moe_inputs(case, seed):
    g, E = _gen(seed), case["experts"]
    w = _normal(g, E, case["M"], case["K"], std=STD)
    x = _normal(g, case["T"], 1, case["K"])
    # a router's choice: each token's `used` best experts of random scores, distinct
    ids = torch.rand(case["T"], E, generator=g, device=DEV).topk(case["used"], dim=1).indices.to(torch.int32)
    return w, x, ids


def prepare(case, seed):
    lnship.init()
    kind = case["kind"]
    mode = lnship.MODES.get(case.get("mode"))   # None: LNS32
    s = {"case": dict(case), "mode": mode, "lfsr": 7 + int(seed) % 60000}
    empty = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=DEV)  # noqa: E731
    if kind == "decode":
        cfg, w, prompts, nxt = _decode_inputs(case, seed)
        host = lambda v: v.cpu().numpy() if isinstance(v, torch.Tensor) else v  # noqa: E731
        w = {"tok_embd": host(w["tok_embd"]), "out_norm": host(w["out_norm"]),
             "layers": [{k: host(v) for k, v in L.items()} for L in w["layers"]]}
        m = LlamaLNS16(cfg, w, mode=mode, lfsr=s["lfsr"], n_seq=case["seqs"])
        for i, p in enumerate(prompts.cpu().tolist()):
            m.eval(p, seq=i)
        s.update(model=m, next=nxt)
    elif kind in ("mm16", "mm32"):
        w, x = _mm_inputs(case, seed)
        s.update(x=x, w=(lnship.pack16 if kind == "mm16" else lnship.pack32)(w))
    elif kind in ("ffn16", "ffn32"):
        x, nw, ug, down = _ffn_inputs(case, seed)
        pack = lnship.pack16 if kind == "ffn16" else lnship.pack32
        E, F, N = case["E"], case["F"], case["N"]
        s.update(x=x, norm=nw, wug=pack(ug), wdown=pack(down), h=empty(N, E), ug=empty(N, 2 * F), sw=empty(N, F), y=empty(N, E))
    elif kind == "attn16":
        qkv, old = _attn_inputs(case, seed)
        H, HKV, D, T, past = (case[k] for k in ("H", "HKV", "D", "T", "past"))
        n_ctx = 512
        n_kv = n_kv_for(past + T, n_ctx)
        rope = np.empty(n_ctx * D, np.float32)
        lnship.check(lnship.lib().lnship_rope_table(THETA, D, n_ctx, ctypes.c_void_p(rope.ctypes.data)))
        s.update(qkv=qkv, rope=torch.from_numpy(rope).to(DEV), n_ctx=n_ctx, n_kv=n_kv, q=empty(T, H * D), kq=empty(H, T, n_kv),
                 att=empty(T, H * D), mask=empty(T, n_kv), k=torch.zeros(HKV, lnship.kp(D) * n_ctx, dtype=torch.int16, device=DEV),
                 v=torch.zeros(HKV, lnship.kp(n_ctx) * D, dtype=torch.int16, device=DEV),
                 pos=torch.arange(past, past + T, dtype=torch.int32, device=DEV))
        if past:   # the cells of the tokens before
            _store(s, old, torch.arange(past, dtype=torch.int32, device=DEV), empty(past, H * D))
    elif kind == "soft_max":
        x, mask = _soft_max_inputs(case, seed)
        s.update(x=x, mask=mask)
    elif kind == "pack":
        s.update(x=_pack_inputs(case, seed))
    else:
        w, x, ids = _moe_inputs(case, seed)
        s.update(x=x, ids=ids, w=(lnship.pack32 if mode is None else lnship.pack16)(w))
    return s


# ---- one pass -------------------------------------------------------------------------------

def _p(t, off=0):
    return ctypes.c_void_p(t.data_ptr() + off * t.element_size())


def _store(s, qkv, pos, q):
    """The query rope and the key / value cache stores of qkv's tokens."""
    c = s["case"]
    H, HKV, D = c["H"], c["HKV"], c["D"]
    a = lnship.QkvStoreArgs(_p(qkv), (H + 2 * HKV) * D, _p(pos), pos.numel(), H, HKV, D, D, _p(s["rope"]), _p(q), _p(s["k"]), _p(s["v"]),
                            s["n_ctx"], s["k"].shape[1], s["v"].shape[1], None, 0)
    lnship.check(lnship.lib().lnship16_rope_store_kv(ctypes.byref(a), lnship._stream()))


def _seed_after(s, draws):
    """Where the next Monte node's draws start (graph order)."""
    now = s["now"]
    s["now"] = lnship.lfsr_jump(now, draws) if s["mode"] == lnship.MONTE else now
    return now


def _ffn(s):
    c, L, st, mode = s["case"], lnship.lib(), lnship._stream(), s["mode"]
    E, F, N = c["E"], c["F"], c["N"]
    if c["kind"] == "ffn32":
        lnship.check(L.lnship32_rms_norm_mul(_p(s["x"]), _p(s["norm"]), _p(s["h"]), E, N, EPS, st))
        lnship.mul_mat32_raw(_p(s["wug"]), _p(s["h"]), _p(s["ug"]), E, 2 * F, N, stream=st)
        lnship.check(L.lnship32_swiglu(_p(s["ug"], F), 2 * F, _p(s["ug"]), 2 * F, _p(s["sw"]), F, N, st))
        lnship.mul_mat32_raw(_p(s["wdown"]), _p(s["sw"]), _p(s["y"]), F, E, N, stream=st, residual=_p(s["x"]))
        return s["y"]
    s["now"] = s["lfsr"]
    seed = _seed_after(s, L.lnship16_rms_norm_draws(mode, E, N))
    lnship.check(L.lnship16_rms_norm_mul(mode, _p(s["x"]), _p(s["norm"]), _p(s["h"]), E, N, EPS, seed, None, 0, st))
    seed = _seed_after(s, L.lnship16_mul_mat_draws(mode, E, 2 * F, N, 1, 1))
    lnship.mul_mat16_raw(mode, _p(s["wug"]), _p(s["h"]), _p(s["ug"]), E, 2 * F, N, seed=seed, stream=st)
    lnship.check(L.lnship16_swiglu(_p(s["ug"], F), 2 * F, _p(s["ug"]), 2 * F, _p(s["sw"]), F, N, st))
    seed = _seed_after(s, L.lnship16_mul_mat_draws(mode, F, E, N, 1, 1))
    lnship.mul_mat16_raw(mode, _p(s["wdown"]), _p(s["sw"]), _p(s["y"]), F, E, N, seed=seed, stream=st, residual=_p(s["x"]))
    return s["y"]


def _attn(s):
    c, L, st, mode = s["case"], lnship.lib(), lnship._stream(), s["mode"]
    H, HKV, D, T, n_kv = c["H"], c["HKV"], c["D"], c["T"], s["n_kv"]
    s["now"] = s["lfsr"]
    _store(s, s["qkv"], s["pos"], s["q"])
    lnship.check(L.lnship_causal_mask(_p(s["pos"]), T, n_kv, _p(s["mask"]), st))
    seed = _seed_after(s, L.lnship16_mul_mat_draws(mode, D, n_kv, T, H, 1))
    lnship.mul_mat16_raw(mode, _p(s["k"]), _p(s["q"]), _p(s["kq"]), D, n_kv, T, ne02=HKV, ne12=H, x_ld=H * D, x_slice=D, seed=seed,
                         w_mstride=s["n_ctx"], w_slice=s["k"].shape[1], stream=st)
    seed = _seed_after(s, L.lnship16_soft_max_draws(mode, n_kv, T * H))
    p = lnship.soft_max16(mode, s["kq"].view(1, H, T, n_kv), s["mask"].view(1, 1, T, n_kv), 1.0 / math.sqrt(D), seed=seed)
    seed = _seed_after(s, L.lnship16_mul_mat_draws(mode, n_kv, D, T, H, 1))
    lnship.mul_mat16_raw(mode, _p(s["v"]), _p(p), _p(s["att"]), n_kv, D, T, ne02=HKV, ne12=H, x_ld=n_kv, x_slice=T * n_kv, seed=seed,
                         w_slice=s["v"].shape[1], dst_ld=H * D, dst_slice=D, stream=st)
    return {"att": s["att"], "k": s["k"], "v": s["v"]}


def run(s):
    c, mode = s["case"], s["mode"]
    kind = c["kind"]
    if kind == "decode":   # the same position again, as a program that samples another continuation does
        m = s["model"]
        m.restart(lfsr=s["lfsr"])
        m.past = [c["past"]] * c["seqs"]
        return m.decode_graph(s["next"]) if c["seqs"] == 1 else m.decode_graph_batch(s["next"])
    if kind == "mm16":
        return lnship.mul_mat16(mode, s["w"], s["x"], c["K"], c["M"], seed=s["lfsr"])
    if kind == "mm32":
        return lnship.mul_mat32(s["w"], s["x"], c["K"], c["M"])
    if kind in ("ffn16", "ffn32"):
        return _ffn(s)
    if kind == "attn16":
        return _attn(s)
    if kind == "soft_max":
        mask, scale = s["mask"].view(1, 1, c["T"], c["n_kv"]), 0.125
        if mode is None:
            return lnship.soft_max32(s["x"], mask, scale)
        return lnship.soft_max16(mode, s["x"], mask, scale, seed=s["lfsr"])
    if kind == "pack":
        return lnship.pack16(s["x"]) if c["width"] == 16 else lnship.pack32(s["x"])
    return lnship.mul_mat_id(mode, s["w"], s["x"], s["ids"], c["K"], c["M"], c["experts"], seed=s["lfsr"])


# ---- what a pass cannot do without ----------------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    if kind == "decode":
        g = _config(case)
        e, f, d, B = g.n_embd, g.n_ff, g.head_dim, c["seqs"]
        macs = g.n_layer * ((g.n_head + 2 * g.n_head_kv) * d * e + e * g.n_head * d + 3 * e * f) + g.n_vocab * e
        cells = c["past"] + 1
        return {"bytes": 2 * macs + B * (g.n_layer * 2 * g.n_head_kv * d * cells * 2 + 4 * g.n_vocab),
                "flops": 2 * B * (macs + g.n_layer * 2 * g.n_head * d * cells)}
    if kind in ("mm16", "mm32"):
        K, M, N = c["K"], c["M"], c["N"]
        return {"bytes": (2 if kind == "mm16" else 4) * K * M + 4 * N * (K + M), "flops": 2 * K * M * N}
    if kind in ("ffn16", "ffn32"):
        E, F, N = c["E"], c["F"], c["N"]
        return {"bytes": (2 if kind == "ffn16" else 4) * 3 * E * F + 4 * (2 * N * E + E), "flops": 6 * E * F * N + 4 * N * E}
    if kind == "attn16":
        H, HKV, D, T, past = (c[k] for k in ("H", "HKV", "D", "T", "past"))
        pairs = T * past + T * (T + 1) // 2   # (query, visible cell)
        return {"bytes": 4 * T * (2 * H + 2 * HKV) * D + 2 * 2 * HKV * D * (2 * T + past), "flops": H * pairs * (4 * D + 5)}
    if kind == "soft_max":
        n = c["H"] * c["T"] * c["n_kv"]
        return {"bytes": 8 * n + 4 * c["T"] * c["n_kv"], "flops": 5 * n}
    if kind == "pack":
        n = c["K"] * c["M"]
        return {"bytes": ((2 if c["half"] else 4) + c["width"] // 8) * n, "flops": n}
    K, M, T = c["K"], c["M"], c["T"]
    hit = min(c["experts"], T * c["used"])
    return {"bytes": (4 if c["mode"] == "lns32" else 2) * hit * K * M + 4 * T * (K + c["used"] * M), "flops": 2 * K * M * T * c["used"]}


def tolerance(case):
    return "exact"   # LNS codes in the reference's term order: whole numbers, whatever the kernel


# ---- the same in 64 bits --------------------------------------------------------------------

def _rope64(x, pos, D):
    """x [T, heads, D] rotated in pairs (2j, 2j + 1) at positions pos."""
    inv = THETA ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D)
    a = pos.double()[:, None] * inv[None, :]
    cos, sin = a.cos()[:, None, :], a.sin()[:, None, :]
    y = torch.empty_like(x)
    y[..., 0::2] = x[..., 0::2] * cos - x[..., 1::2] * sin
    y[..., 1::2] = x[..., 0::2] * sin + x[..., 1::2] * cos
    return y


def _attend64(q, k, v, mask, H, HKV, D):
    """q [T, H, D], k and v [cells, HKV, D] -> [T, H * D]."""
    out = []
    for h in range(H):
        p = torch.softmax(q[:, h] @ k[:, h // (H // HKV)].t().contiguous() / math.sqrt(D) + mask, dim=-1)
        out.append(p @ v[:, h // (H // HKV)].contiguous())
    return torch.stack(out, 1).reshape(q.shape[0], H * D)


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _ffn64(x, nw, ug, down):
    F = down.shape[1]
    u = _norm64(x, nw) @ ug.t()
    return torch.nn.functional.silu(u[:, F:]) * u[:, :F] @ down.t() + x


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        # an LNS16 code holds 7 fraction bits, and each of the 30 layers rounds to it several times:
        # the format's own distance from a 64-bit decoder (0.10 in sum32, 0.14 in monte) says
        # nothing about an implementation of it
        return None
    if case.get("mode") == "lpvip":
        # Mitchell's approximation of the Gaussian logs is far off by itself (an MLP's outputs by
        # more than their size): no 64-bit value stands for what it gives
        return None
    if kind in ("mm16", "mm32"):
        w, x = _mm_inputs(case, seed)
        return x.double() @ w.double().t()
    if kind in ("ffn16", "ffn32"):
        return _ffn64(*(t.double() for t in _ffn_inputs(case, seed)))
    if kind == "attn16":
        qkv, old = (t.double() for t in _attn_inputs(case, seed))
        H, HKV, D, T, past = (case[k] for k in ("H", "HKV", "D", "T", "past"))
        rows = torch.cat([old[:past], qkv]).reshape(past + T, H + 2 * HKV, D)
        pos = torch.arange(past + T, device=DEV)
        q, k, v = _rope64(rows[:, :H], pos, D)[past:], _rope64(rows[:, H:H + HKV], pos, D), rows[:, H + HKV:]
        # (the caches hold LNS codes, which have no 64-bit value of their own)
        return {"att": _attend64(q, k, v, _mask(T, past, past + T).double(), H, HKV, D), "k": None, "v": None}
    if kind == "soft_max":
        x, mask = _soft_max_inputs(case, seed)
        return torch.softmax(x.double() * 0.125 + mask.double(), dim=-1)
    if kind == "pack":
        return None   # LNS codes
    w, x, ids = _moe_inputs(case, seed)
    return torch.stack([torch.stack([w[e].double() @ x[t, 0].double() for e in row]) for t, row in enumerate(ids.tolist())])
