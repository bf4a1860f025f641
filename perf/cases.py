"""Performance cases of the verify/draft hot path, through the Python entry
points a program calls: the RMSNorm -> linear family (fp32, bf16 / f16 and
fp8-e4m3 weights, grouped INT4) from a single decode row to a prompt, one
draft step, the multi-token verify over a whole vocabulary, and the decode,
fp8-KV, masked and tree-verify attention.

A case is a dict of sizes and options; `listed()` names the fixed ones and
`draw(rng)` gives more of the same ranges. Inputs are made on the GPU from
the seed alone. All sizes are this repository's workloads, tests and
benchmark, or generic transformer sizes.
"""
import math
import os
import sys

import torch

# The package lives in a directory of the working tree's root (its name has a
# dash, so it is put on the path rather than imported by name).
_PKG = os.path.join(os.getcwd(), "mtp-engine_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from mtp_hip import fused_verify as FV  # noqa: E402
from mtp_hip import kernels as MK  # noqa: E402
from mtp_hip import ops  # noqa: E402

DEV = "cuda"
_DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_BYTES = {"f32": 4.0, "bf16": 2.0, "f16": 2.0, "fp8": 1.0}
EPS = 1e-6


def listed():
    return [
        # The engine's default head: fp32 (TF32 off), a handful of positions
        # through a small draft head. The smallest call: latency and host work.
        {"name": "head_fp32", "kind": "linear", "x": "f32", "w": "f32", "M": 16, "N": 4096,
         "K": 1024, "gamma": True, "bias": False},
        # One greedy draft step of 8 sequences: norm(hidden + embedding), head,
        # argmax and the next embedding lookup.
        {"name": "draft_step_bf16", "kind": "draft", "x": "bf16", "M": 8, "V": 32000, "K": 4096},
        # A 64-node verify tree through an fp8 MLP projection.
        {"name": "verify_linear_fp8", "kind": "linear", "x": "bf16", "w": "fp8", "M": 64,
         "N": 14336, "K": 4096, "gamma": True, "bias": False},
        # A 2048-token prompt through the same projection in bf16.
        {"name": "prefill_linear_bf16", "kind": "linear", "x": "bf16", "w": "bf16", "M": 2048,
         "N": 14336, "K": 4096, "gamma": True, "bias": False},
        # A ragged prompt (or several sequences' trees in one call) on fp8 weights.
        {"name": "prefill_linear_fp8", "kind": "linear", "x": "bf16", "w": "fp8", "M": 517,
         "N": 14336, "K": 4096, "gamma": True, "bias": False},
        # Decode of 8 rows on INT4 weights (group 128, fp16 scales) with the norm.
        {"name": "int4_decode", "kind": "int4", "x": "bf16", "M": 8, "N": 28672, "K": 8192,
         "group": 128, "scales": "f16", "norm": True},
        # The chain verify of 8 sequences with 4 drafts over a whole vocabulary.
        {"name": "multi_verify_bf16", "kind": "verify", "x": "bf16", "B": 8, "D": 4, "K": 4096,
         "V": 128256},
        # Decode attention of 8 sequences over a paged KV cache.
        {"name": "paged_decode_bf16", "kind": "paged", "x": "bf16", "B": 8, "H": 32, "D": 128,
         "L": 4096, "page": 16},
        # The same over a KV cache held in fp8 with per-head scales.
        {"name": "kv_fp8_decode", "kind": "kvfp8", "x": "bf16", "B": 8, "H": 32, "D": 128,
         "L": 4096},
        # The engine's default dtype: fp32 masked attention of one tree node per
        # sequence over context and draft nodes.
        {"name": "tree_attention_fp32", "kind": "tree", "x": "f32", "B": 4, "H": 16, "D": 64,
         "L": 2048},
        # 64 tree nodes over a 2048-token paged context under one softmax.
        {"name": "tree_verify_bf16", "kind": "treeverify", "x": "bf16", "N": 64, "H": 32,
         "D": 128, "L": 2048, "page": 16},
    ]


def _logint(rng, lo, hi, step=1):
    """An integer multiple of step, uniform over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / step) * step)))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "prefill", "head", "draft", "int4", "verify", "paged",
                       "kvfp8", "tree", "treeverify"])
    if kind == "head":  # fp32 heads, a few rows to a small tree
        return {"kind": "linear", "x": "f32", "w": "f32", "M": _logint(rng, 1, 64),
                "N": _logint(rng, 256, 8192), "K": _logint(rng, 256, 4096, 64),
                "gamma": rng.random() < 0.5, "bias": rng.random() < 0.5}
    if kind in ("decode", "prefill"):
        x = rng.choice(["bf16", "bf16", "f16"])
        lo, hi = (1, 64) if kind == "decode" else (65, 2048)
        return {"kind": "linear", "x": x, "w": rng.choice(["fp8", x]), "M": _logint(rng, lo, hi),
                "N": _logint(rng, 512, 14336), "K": _logint(rng, 512, 4096, 64),
                "gamma": rng.random() < 0.7, "bias": rng.random() < 0.3}
    if kind == "draft":
        return {"kind": "draft", "x": rng.choice(["bf16", "f16"]), "M": rng.randint(1, 16),
                "V": _logint(rng, 8000, 64000), "K": _logint(rng, 512, 4096, 64)}
    if kind == "int4":
        group = rng.choice([32, 64, 128])
        return {"kind": "int4", "x": rng.choice(["bf16", "f16"]), "M": _logint(rng, 1, 256),
                "N": _logint(rng, 1024, 28672), "K": _logint(rng, 1024, 8192, 128),
                "group": group, "scales": rng.choice(["f16", "f32"]), "norm": rng.random() < 0.5}
    if kind == "verify":
        return {"kind": "verify", "x": rng.choice(["bf16", "f16"]), "B": _logint(rng, 1, 16),
                "D": rng.randint(1, 7), "K": _logint(rng, 512, 4096, 64),
                "V": _logint(rng, 8000, 128256)}
    if kind in ("paged", "kvfp8"):
        c = {"kind": kind, "x": rng.choice(["bf16", "f16", "f32"] if kind == "paged" else
                                           ["bf16", "f16", "f32"]),
             "B": _logint(rng, 1, 8), "H": rng.choice([8, 16, 32]), "D": rng.choice([64, 128]),
             "L": _logint(rng, 100, 4096)}
        if kind == "paged":
            c["page"] = rng.choice([16, 32, 64])
        return c
    if kind == "tree":
        return {"kind": "tree", "x": rng.choice(["f32", "f32", "bf16"]), "B": _logint(rng, 1, 8),
                "H": rng.choice([8, 16, 32]), "D": rng.choice([64, 128]),
                "L": _logint(rng, 100, 2048)}
    return {"kind": "treeverify", "x": rng.choice(["bf16", "f16"]), "N": _logint(rng, 2, 64),
            "H": rng.choice([8, 16, 32]), "D": rng.choice([64, 128]), "L": _logint(rng, 100, 4096),
            "page": 16}


# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    """std N(0, 1) in dtype, made in slices of the first dimension."""
    out = torch.empty(shape, dtype=dtype, device=DEV)
    rows = max(1, (1 << 26) // max(1, math.prod(shape[1:])))
    for r in range(0, shape[0], rows):
        n = min(rows, shape[0] - r)
        out[r:r + n] = std * torch.randn(n, *shape[1:], generator=g, device=DEV)
    return out


def _peaked(g, W, target, dtype):
    """Hidden rows whose logits peak at `target`, as a trained head's do: a
    unit of noise plus half of its length along the target's head row."""
    K = W.shape[1]
    rows = W[target].float()
    along = rows / rows.norm(dim=-1, keepdim=True) * (0.5 * math.sqrt(K))
    return (torch.randn(*target.shape, K, generator=g, device=DEV) + along).to(dtype)


def _pages(g, c, B, dtype):
    """Pages of a cache a little larger than the context, physically shuffled."""
    L, ps = c["L"], c["page"]
    n = -(-L // ps)
    P = n + max(1, n // 8)
    k = _randn(g, P, B, c["H"], ps, c["D"], dtype=dtype)
    v = _randn(g, P, B, c["H"], ps, c["D"], dtype=dtype)
    perm = torch.stack([torch.randperm(P, generator=g, device=DEV)[:n] for _ in range(B)])
    table = perm.repeat_interleave(ps, dim=1)[:, :L].to(torch.int32).contiguous()
    return k, v, table


def _tree_mask(g, n):
    """Ancestor-or-self mask of a tree whose node i hangs below an earlier node."""
    parent = [0] + [int(p * i) for i, p in
                    enumerate(torch.rand(n - 1, generator=g, device=DEV).tolist(), 1)]
    m = torch.zeros(n, n)
    for i in range(n):
        if i:
            m[i] = m[parent[i]]
        m[i, i] = 1.0
    return m.to(DEV)


def prepare(case, seed):
    c, g = case, _gen(seed)
    dt = _DT[c["x"]]
    s = {"case": c}
    k = c["kind"]
    if k == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        s["x"] = _randn(g, M, K, dtype=dt)
        if c["w"] == "fp8":
            s["w"], s["wscale"] = MK.quantize_fp8_rows(_randn(g, N, K, std=0.02))
        else:
            s["w"] = _randn(g, N, K, dtype=_DT[c["w"]], std=0.02)
        s["gamma"] = 1.0 + _randn(g, K, std=0.1) if c["gamma"] else None
        s["bias"] = _randn(g, N, dtype=dt, std=0.1) if c["bias"] else None
    elif k == "draft":
        s["w"] = _randn(g, c["V"], c["K"], dtype=dt, std=0.02)
        s["table"] = _randn(g, c["V"], c["K"], dtype=dt)
        t = torch.randint(0, c["V"], (c["M"],), generator=g, device=DEV)
        s["emb"] = s["table"][torch.randint(0, c["V"], (c["M"],), generator=g, device=DEV)]
        s["hidden"] = (2.0 * _peaked(g, s["w"], t, torch.float32)).to(dt)
        s["norm_w"] = (1.0 + _randn(g, c["K"], std=0.1)).to(dt)
    elif k == "int4":
        M, N, K = c["M"], c["N"], c["K"]
        w, sc = MK.quantize_int4(_randn(g, N, K, std=0.02), c["group"])
        s["w"] = w ^ 0x88  # the decoder's offset-8 nibbles of the quantizer's signed ones
        s["scales"] = sc.to(_DT[c["scales"]])
        s["x"] = _randn(g, M, K, dtype=dt)
        s["gamma"] = 1.0 + _randn(g, K, std=0.1) if c["norm"] else None
    elif k == "verify":
        B, S, V = c["B"], c["D"] + 1, c["V"]
        s["w"] = _randn(g, V, c["K"], dtype=dt, std=0.02)
        top = torch.randint(0, V, (B, S), generator=g, device=DEV)
        s["hidden"] = _peaked(g, s["w"], top, dt)
        good = torch.rand(B, c["D"], generator=g, device=DEV) < 0.6
        other = torch.randint(0, V, (B, c["D"]), generator=g, device=DEV)
        s["draft"] = torch.where(good, top[:, 1:], other).to(torch.int32)
    elif k == "paged":
        s["q"] = _randn(g, c["B"], c["H"], c["D"], dtype=dt)
        s["k"], s["v"], s["table"] = _pages(g, c, c["B"], dt)
    elif k == "kvfp8":
        B, H, D, L = c["B"], c["H"], c["D"], c["L"]
        s["q"] = _randn(g, B, H, D, dtype=dt)
        # |N(0, 1)| stays below 7, so 7 / 448 scales use the whole e4m3 range
        s["ks"] = torch.full((H,), 7.0 / 448.0, device=DEV) * (1.0 + 0.1 * _randn(g, H).abs())
        s["vs"] = torch.full((H,), 7.0 / 448.0, device=DEV) * (1.0 + 0.1 * _randn(g, H).abs())
        for n, sc in (("k", s["ks"]), ("v", s["vs"])):
            t = _randn(g, B, H, L, D) / sc[None, :, None, None]
            s[n] = t.clamp(-448, 448).to(torch.float8_e4m3fn)
    elif k == "tree":
        B, H, D, L = c["B"], c["H"], c["D"], c["L"]
        s["q"] = _randn(g, B, H, D, dtype=dt)
        s["k"] = _randn(g, B, H, L, D, dtype=dt)
        s["v"] = _randn(g, B, H, L, D, dtype=dt)
        s["mask"] = torch.ones(L, device=DEV)
        n = min(64, L // 2)  # the last n keys are draft nodes, some of them ancestors
        s["mask"][L - n:] = _tree_mask(g, n)[-1]
    elif k == "treeverify":
        N, H, D = c["N"], c["H"], c["D"]
        s["q"] = _randn(g, N, H, D, dtype=dt)
        s["kt"] = _randn(g, N, H, D, dtype=dt)
        s["vt"] = _randn(g, N, H, D, dtype=dt)
        s["k"], s["v"], s["table"] = _pages(g, c, 1, dt)
        s["mask"] = _tree_mask(g, N)
    else:
        raise ValueError(k)
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "linear":
        if c["w"] == "fp8":
            return MK.fused_rmsnorm_linear_fp8(s["x"], s["w"], s["wscale"], s["bias"], EPS,
                                               gamma=s["gamma"])
        return MK.fused_rmsnorm_linear(s["x"], s["w"], s["bias"], EPS, gamma=s["gamma"])
    if k == "draft":
        h = MK.fused_add_rmsnorm(s["hidden"], s["emb"], s["norm_w"], EPS)
        logits = MK.fused_rmsnorm_linear(h, s["w"], None, EPS, norm=False)
        tokens, emb = ops.argmax(logits, s["table"])
        return {"hidden": h, "logits": logits, "tokens": tokens, "emb": emb}
    if k == "int4":
        return MK.fused_int4_matmul(s["x"], s["w"], s["scales"], c["K"], c["group"],
                                    gamma=s["gamma"], norm=c["norm"], eps=EPS)
    if k == "verify":
        a, n, t, top = FV.fused_multi_verify(s["hidden"], s["w"], s["draft"], return_top=True)
        return {"accept": a, "accepted_n": n, "corrected": t, "top": top}
    if k == "paged":
        return MK.fused_paged_attention(s["q"], s["k"], s["v"], s["table"], c["page"])
    if k == "kvfp8":
        return MK.fused_causal_attention_fp8(s["q"], s["k"], s["v"], s["ks"], s["vs"])
    if k == "tree":
        return MK.fused_tree_attention(s["q"], s["k"], s["v"], s["mask"])
    return MK.tree_verify_attention(s["q"], s["k"], s["v"], s["table"], c["page"], s["kt"],
                                    s["vt"], s["mask"])


def work(case):
    c = case
    k, xb = c["kind"], _BYTES[c["x"]]
    if k == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        extra = (4 * N if c["w"] == "fp8" else 0) + (4 * K if c["gamma"] else 0) + \
            (xb * N if c["bias"] else 0)
        return {"bytes": M * K * xb + N * K * _BYTES[c["w"]] + M * N * xb + extra,
                "flops": 2.0 * M * N * K}
    if k == "draft":
        M, V, K = c["M"], c["V"], c["K"]
        # hidden and embedding in, normed hidden and next embedding out (and its
        # table rows), the head, the logits
        return {"bytes": xb * (5 * M * K + K + V * K + M * V) + 8 * M, "flops": 2.0 * M * V * K}
    if k == "int4":
        M, N, K = c["M"], c["N"], c["K"]
        sb = _BYTES[c["scales"]] * N * -(-K // c["group"])
        return {"bytes": M * K * xb + N * K / 2 + sb + M * N * xb + (4 * K if c["norm"] else 0),
                "flops": 2.0 * M * N * K}
    if k == "verify":
        M = c["B"] * (c["D"] + 1)
        return {"bytes": xb * (M * c["K"] + c["V"] * c["K"]) + 4 * M + 5 * c["B"] * c["D"] +
                8 * c["B"], "flops": 2.0 * M * c["V"] * c["K"]}
    H, D, L = c["H"], c["D"], c["L"]
    if k == "treeverify":
        N = c["N"]
        return {"bytes": xb * H * D * (2 * L + 4 * N) + 4 * L + 4 * N * N,
                "flops": 4.0 * N * H * D * (L + N)}
    B = c["B"]
    kb = 1.0 if k == "kvfp8" else xb
    return {"bytes": 2 * B * H * L * D * kb + 2 * B * H * D * xb +
            {"paged": 4 * B * L, "kvfp8": 8 * H, "tree": 4 * L}[k],
            "flops": 4.0 * B * H * L * D}


def tolerance(case):
    c = case
    k = c["kind"]
    if k == "verify":
        return "exact"
    # About four times the error against 64 bits (2-norm) that was measured.
    if c["x"] == "f32":
        # fp32 sums over K or L of some thousands: 1.6e-7 for the head; 1.2e-6
        # for attention, whose exp turns a score's absolute error into a
        # relative one
        return {"rel": 1e-6 if k == "linear" else 5e-6}
    # 16-bit outputs, rounded to 8 (bf16) or 11 (f16) bits, on top of x * gamma
    # or the probabilities rounded once to the same type: 2.4e-3 and 2.9e-4
    return {"rel": 1e-2 if c["x"] == "bf16" else 1.2e-3}


# ---------------------------------------------------------------------------
def _softmax_av(scores, v):
    return torch.softmax(scores, dim=-1).unsqueeze(-2).matmul(v).squeeze(-2)


def exact(case, seed):
    s, c = prepare(case, seed), case
    k = c["kind"]

    def f(t):
        return None if t is None else t.double()

    def norm(x, gamma):
        y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
        return y if gamma is None else y * gamma

    if k == "linear":
        w = f(s["w"]) if c["w"] != "fp8" else s["w"].float().double() * f(s["wscale"])[:, None]
        y = norm(f(s["x"]), f(s["gamma"])) @ w.t()
        return y if s["bias"] is None else y + f(s["bias"])
    if k == "draft":
        h = norm(f(s["hidden"]) + f(s["emb"]), f(s["norm_w"]))
        return {"hidden": h, "logits": h @ f(s["w"]).t(), "tokens": None, "emb": None}
    if k == "int4":
        N, K = c["N"], c["K"]
        w = torch.empty(N, K, dtype=torch.float64, device=DEV)
        w[:, 0::2] = (s["w"] & 0xF).double() - 8
        w[:, 1::2] = (s["w"] >> 4).double() - 8
        w *= f(s["scales"]).repeat_interleave(c["group"], dim=1)[:, :K]
        x = f(s["x"])
        return (norm(x, f(s["gamma"])) if c["norm"] else x) @ w.t()
    if k == "verify":
        return None
    scale = 1.0 / math.sqrt(c["D"])
    if k in ("paged", "treeverify"):
        B = c.get("B", 1)
        t = torch.arange(c["L"], device=DEV) % c["page"]
        b = torch.arange(B, device=DEV)[:, None]
        # [B, L, H, D] rows of the pages -> [B, H, L, D]
        kk = f(s["k"][s["table"].long(), b, :, t[None, :]]).transpose(1, 2)
        vv = f(s["v"][s["table"].long(), b, :, t[None, :]]).transpose(1, 2)
    if k == "paged":
        return _softmax_av((kk @ f(s["q"]).unsqueeze(-1)).squeeze(-1) * scale, vv)
    if k == "kvfp8":
        kk = s["k"].float().double() * f(s["ks"])[None, :, None, None]
        vv = s["v"].float().double() * f(s["vs"])[None, :, None, None]
        return _softmax_av((kk @ f(s["q"]).unsqueeze(-1)).squeeze(-1) * scale, vv)
    if k == "tree":
        sc = (f(s["k"]) @ f(s["q"]).unsqueeze(-1)).squeeze(-1) * scale
        return _softmax_av(sc.masked_fill(s["mask"] <= 0.5, -math.inf), f(s["v"]))
    q = f(s["q"]).transpose(0, 1)  # [H, N, D]
    kt, vt = f(s["kt"]).transpose(0, 1), f(s["vt"]).transpose(0, 1)
    sc = torch.cat([q @ kk[0].transpose(1, 2).contiguous(),
                    (q @ kt.transpose(1, 2).contiguous()).masked_fill(s["mask"] <= 0.5, -math.inf)],
                   dim=-1) * scale
    return (torch.softmax(sc, dim=-1) @ torch.cat([vv[0], vt], dim=1)).transpose(0, 1)
