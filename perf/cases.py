"""The work that programs built on this framework have it do, as measurable cases.

A case is one pass through public entry points: the training-side ops of a layer over both streams
(the state fork, complementary-mask attention), the prefill and the denoising step of the cached
decoder (the chunked rule, block-causal attention, the small-M projections), the fp32 runs of the
equivalence harness, and two whole calls (a cached denoising step, the two-stream forward).

The head geometries are those of the repository's workloads: 27B-class (16 key / 48 value GDN heads
of 128, 24 query / 4 key-value attention heads of 256, hidden 5120, MLP 17408), 0.8B-class (16 / 16
GDN heads of 128), the small fp32 layer (4 heads of 64) and the attention head sizes 64 and 128 of
the tests. Inputs are drawn as the benchmark draws them: N(0, 1) projections, beta = sigmoid(N(0, 1)),
g = -softplus(N(0, 1) + 1), conv weights U(-0.5, 0.5), linear weights N(0, 0.02).
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dllm-qwen38_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dllm_qwen38_amd import attention, blockdiff, decode, gdn, gemm_tuning, model  # noqa: E402

DEV = "cuda"
EPS = 1e-6


def listed():
    return [
        # --- training / scoring side: both streams of one layer
        # the benchmarked GDN layer: conv + state fork with every block's state kept
        _fork("fork 27B states", "bf16", 4, 4096, 32, 16, 48, 128, True),
        # the GDN layer inside the two-stream forward at B = 1 (no states leave the layer)
        _fork("fork 27B in stack", "bf16", 1, 2048, 32, 16, 48, 128, False),
        # the equivalence harness's GDN layer: fp32 at the 27B-class heads, a short sequence
        _fork("fork fp32 harness", "fp32", 1, 256, 32, 16, 48, 128, True),
        # the gated attention layer's core over cat([x_t, x_0])
        _bd("attention 27B gated", "bf16", 2, 4096, 32, 24, 4, 256),
        # the equivalence harness's attention layer: fp32
        _bd("attention fp32 harness", "fp32", 1, 256, 32, 24, 4, 256),
        # --- the cached decoder
        # prompt prefill of one GDN layer: the chunked rule over 61 blocks, states kept for the commit
        _rule("rule prefill", "bf16", 1, 1952, 32, 16, 48, 128, False, True),
        # the same layer in a denoising step: one 32-token block from the cached state
        _rule("rule decode", "bf16", 1, 32, 32, 16, 48, 128, True, False),
        # prompt prefill of one attention layer: block-causal, 61 blocks
        _bc("attention prefill", 1, 1952, 1952, 32, 24, 4, 256),
        # a denoising step's attention: one block against a long cached prefix
        _bc("attention decode", 1, 32, 4128, 32, 24, 4, 256),
        # MLP of a denoising step for two sequences (64 token rows): gate | up with SwiGLU, then down + residual + norm
        _mlp("mlp decode 64 rows", 64, 5120, 17408),
        # --- whole calls, on four 27B-class layers (three GDN, one attention)
        # one cached denoising step over a 2048-token prefix, logits of the block
        _step("decode step", 1, 2048, 32, 4),
        # the two-stream forward, logits of both streams
        _stack("two-stream forward", 1, 2048, 32, 4),
    ]


def _fork(name, dtype, B, L, block, Hk, Hv, D, states):
    return {"name": name, "kind": "fork", "dtype": dtype, "B": B, "L": L, "block": block, "Hk": Hk, "Hv": Hv, "D": D,
            "states": states}


def _bd(name, dtype, B, L, block, Hq, Hkv, d):
    return {"name": name, "kind": "bd", "dtype": dtype, "B": B, "L": L, "block": block, "Hq": Hq, "Hkv": Hkv, "d": d}


def _rule(name, dtype, B, T, chunk, Hk, Hv, D, init, states):
    return {"name": name, "kind": "rule", "dtype": dtype, "B": B, "T": T, "chunk": chunk, "Hk": Hk, "Hv": Hv, "D": D,
            "init": init, "states": states}


def _bc(name, B, M, N, block, Hq, Hkv, d):
    return {"name": name, "kind": "bc", "B": B, "M": M, "N": N, "block": block, "Hq": Hq, "Hkv": Hkv, "d": d}


def _mlp(name, rows, hidden, inter):
    return {"name": name, "kind": "mlp", "rows": rows, "hidden": hidden, "inter": inter}


def _step(name, B, prefix, block, layers):
    return {"name": name, "kind": "step", "B": B, "prefix": prefix, "block": block, "layers": layers}


def _stack(name, B, L, block, layers):
    return {"name": name, "kind": "stack", "B": B, "L": L, "block": block, "layers": layers}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed kinds: sequence lengths of any number of blocks, blocks 8 to 32, the
    repository's head geometries, one to four sequences, ragged decoder shapes."""
    kind = rng.choice(["fork", "fork", "bd", "bd", "rule", "rule", "bc", "bc", "mlp", "step"])
    block = rng.choice([32, 32, 32, 16, 8])
    fp32 = rng.random() < 0.25
    if kind == "fork":
        if fp32:
            Hk, Hv, D = rng.choice([(4, 4, 64), (16, 48, 128), (16, 16, 128)])
            c = _fork("", "fp32", rng.choice([1, 2]), block * _log(rng, 2, 512 // block), block, Hk, Hv, D, True)
        else:
            Hk, Hv, D = rng.choice([(16, 48, 128), (16, 16, 128)])
            B = rng.choice([1, 2, 4])
            c = _fork("", "bf16", B, block * _log(rng, 4, (4096 if B < 4 else 2048) // block), block, Hk, Hv, D,
                      rng.random() < 0.6 and block == 32)
    elif kind == "bd":
        Hq, Hkv, d = rng.choice([(24, 4, 256), (24, 4, 256), (16, 4, 128), (8, 2, 64)])
        B = rng.choice([1, 2])
        top = 512 if fp32 else 4096 // B
        c = _bd("", "fp32" if fp32 else "bf16", B, block * _log(rng, 2, top // block), block, Hq, Hkv, d)
    elif kind == "rule":
        Hk, Hv = rng.choice([(16, 48), (16, 16)])
        B = rng.choice([1, 1, 2])
        T = 32 if rng.random() < 0.4 else block * _log(rng, 2, 4096 // block)
        c = _rule("", "bf16", B, T, min(block, T), Hk, Hv, 128, rng.random() < 0.5, T > 32)
    elif kind == "bc":
        Hq, Hkv, d = rng.choice([(24, 4, 256), (24, 4, 256), (16, 4, 128), (8, 2, 64)])
        B = rng.choice([1, 1, 2, 4])
        if rng.random() < 0.5:  # a denoising step after a prefix of any number of blocks
            c = _bc("", B, block, block * _log(rng, 4, 8192 // block), block, Hq, Hkv, d)
        else:  # a prompt
            n = block * _log(rng, 4, 4096 // B // block)
            c = _bc("", B, n, n, block, Hq, Hkv, d)
    elif kind == "mlp":
        hidden, inter = rng.choice([(5120, 17408), (1024, 3584), (2048, 6144)])
        c = _mlp("", rng.randint(1, 64), hidden, inter)
    else:
        c = _step("", rng.choice([1, 2]), 32 * _log(rng, 2, 64), 32, 4)
    del c["name"]
    return c


# ------------------------------------------------------------------------------------------ inputs
def _dt(case):
    return torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _gates(g, *shape, dtype):
    beta = torch.sigmoid(_randn(g, *shape)).to(dtype).float()
    return beta, -F.softplus(_randn(g, *shape) + 1.0)


def _tables(L, rd, dtype):
    inv = 1.0 / (1e7 ** (torch.arange(0, rd, 2, dtype=torch.float32, device=DEV) / rd))
    fr = torch.arange(L, dtype=torch.float32, device=DEV)[:, None] * inv[None]
    e = torch.cat([fr, fr], -1)
    return e.cos().to(dtype), e.sin().to(dtype)


def _rd(case):
    """Rotary dims of the gated core: a quarter of the head, at least the 64 that the fused core takes."""
    return max(64, case["d"] // 4)


def prepare(case, seed):
    g, dt, k = _gen(seed), _dt(case), case["kind"]
    if k == "fork":
        B, L, Hk, Hv, D = (case[x] for x in ("B", "L", "Hk", "Hv", "D"))
        Cd = 2 * Hk * D + Hv * D
        s = {"raw0": _randn(g, B, L, Cd, dtype=dt), "rawt": _randn(g, B, L, Cd, dtype=dt)}
        s["beta0"], s["g0"] = _gates(g, B, L, Hv, dtype=dt)
        s["betat"], s["gt"] = _gates(g, B, L, Hv, dtype=dt)
        s["w"] = (torch.rand(Cd, 4, generator=g, device=DEV) - 0.5).to(dt)
    elif k == "rule":
        B, T, Hk, Hv, D = (case[x] for x in ("B", "T", "Hk", "Hv", "D"))
        # q | k | v channel blocks of one post-conv buffer, as the mixer hands them over
        mixed = F.silu(_randn(g, B, T, 2 * Hk * D + Hv * D)).to(dt)
        s = {"q": mixed[..., :Hk * D].unflatten(-1, (Hk, D)), "k": mixed[..., Hk * D:2 * Hk * D].unflatten(-1, (Hk, D)),
             "v": mixed[..., 2 * Hk * D:].unflatten(-1, (Hv, D))}
        s["beta"], s["g"] = _gates(g, B, T, Hv, dtype=dt)
        s["init"] = 0.05 * _randn(g, B, Hv, D, D) if case["init"] else None
    elif k == "bd":
        B, L, Hq, Hkv, d = (case[x] for x in ("B", "L", "Hq", "Hkv", "d"))
        # the q_proj output holds each head's query and gate side by side
        qg = _randn(g, B, 2 * L, Hq, 2 * d, dtype=dt)
        s = {"q": qg[..., :d], "gate": qg[..., d:], "k": _randn(g, B, 2 * L, Hkv, d, dtype=dt),
             "v": _randn(g, B, 2 * L, Hkv, d, dtype=dt), "qw": 0.1 * _randn(g, d, dtype=dt)}
        s["qw"] = s["qw"].to(dt)
        s["cos"], s["sin"] = _tables(L, _rd(case), dt)
    elif k == "bc":
        B, M, N, Hq, Hkv, d = (case[x] for x in ("B", "M", "N", "Hq", "Hkv", "d"))
        qg = _randn(g, B, M, Hq, 2 * d, dtype=dt)
        cap = N + 2 * case["block"]  # the cache has room past the segment
        kc, vc = _randn(g, B, cap, Hkv, d, dtype=dt), _randn(g, B, cap, Hkv, d, dtype=dt)
        s = {"q": _randn(g, B, M, Hq, d, dtype=dt), "gate": qg[..., d:], "k": kc[:, :N], "v": vc[:, :N]}
    elif k == "mlp":
        M, H, I = case["rows"], case["hidden"], case["inter"]
        s = {"x": _randn(g, M, H, dtype=dt), "res": _randn(g, M, H, dtype=dt), "nw": (0.1 * _randn(g, H)).to(dt)}
        s["gate"], s["up"] = (0.02 * _randn(g, I, H)).to(dt), (0.02 * _randn(g, I, H)).to(dt)
        s["down"] = (0.02 * _randn(g, H, I)).to(dt)
    else:
        cfg = model.config_27b_truncated(case["layers"])
        tm, head = model.build(cfg, device=DEV, dtype=torch.bfloat16, seed=int(seed))
        tm.requires_grad_(False)
        head.requires_grad_(False)
        s = {"tm": tm, "head": head}
        if k == "stack":
            gemm_tuning.enable()  # the committed choices for the library's GEMMs, as the benchmark runs it
            ids = torch.randint(0, cfg.vocab_size - 1, (case["B"], case["L"]), generator=g, device=DEV)
            t = torch.rand(case["B"], case["L"] // case["block"], 1, generator=g, device=DEV)
            u = torch.rand(case["B"], case["L"] // case["block"], case["block"], generator=g, device=DEV)
            noised = (u < t).reshape(case["B"], case["L"])
            s["x0"], s["xt"] = ids, torch.where(noised, cfg.vocab_size - 1, ids)
        else:
            P, n = case["prefix"], case["block"]
            ids = torch.randint(0, cfg.vocab_size - 1, (case["B"], P + n), generator=g, device=DEV)
            s["ids"] = ids
            s["cache"] = decode.PrefixCache(tm, batch=case["B"], capacity=P + n, block=n)
            decode.forward_segment(tm, head, s["cache"], ids[:, :P], commit=True, logits=False)
            s["xt"] = ids[:, P:].contiguous()
    s["case"] = dict(case)
    return s


# ------------------------------------------------------------------------------------------ a pass
def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "fork":
        r = gdn.gdn_state_fork(s["raw0"], s["rawt"], s["w"], s["beta0"], s["betat"], s["g0"], s["gt"],
                               num_k_heads=c["Hk"], num_v_heads=c["Hv"], head_k_dim=c["D"], head_v_dim=c["D"],
                               block=c["block"], need_states=c["states"], need_tails=c["states"])
        return {n: r[n] for n in (("o0", "ot", "states", "tails") if c["states"] else ("o0", "ot"))}
    if k == "rule":
        out, st = gdn.chunk_gated_delta_rule_with_states(s["q"], s["k"], s["v"], s["g"], s["beta"], c["chunk"],
                                                         initial_state=s["init"], need_states=c["states"])
        return {"out": out, "states": st} if c["states"] else {"out": out}
    if k == "bd":
        if c["dtype"] == "fp32":
            return attention.bd_attention(s["q"], s["k"], s["v"], block=c["block"])
        return attention.bd_attention_gated(s["q"], s["k"], s["v"], s["gate"], block=c["block"], q_norm_weight=s["qw"],
                                            q_norm_eps=EPS, cos=s["cos"], sin=s["sin"])
    if k == "bc":
        return attention.block_causal_attention(s["q"], s["k"], s["v"], block=c["block"], q_offset=c["N"] - c["M"],
                                                gate=s["gate"])
    if k == "mlp":
        act = decode.decode_linear_multi(s["x"], [s["gate"], s["up"]], swiglu=True)
        y, h = decode.decode_linear_rmsnorm(act, s["down"], s["res"], s["nw"], EPS)
        return {"act": act, "y": y, "h": h}
    if k == "step":
        return decode.forward_segment(s["tm"], s["head"], s["cache"], s["xt"], commit=False)
    lt, l0 = blockdiff.block_diffusion_forward(s["tm"], s["head"], s["x0"], s["xt"], c["block"])
    return {"noised": lt, "clean": l0}


# ------------------------------------------------------------------------- what a pass cannot do without
def _pairs_bd(L, block):
    nb = L // block
    return block * block * (nb + nb * (nb - 1) // 2 + nb * (nb + 1) // 2)


def _pairs_bc(M, N, block):
    q0 = N - M
    return sum(min(N, ((q0 + i) // block + 1) * block) for i in range(M))


def _rule_flops(T, H, D, C, noised):
    """Chunk contractions of T tokens and H heads: Gram, inverse applied, state products, update."""
    return (T // C) * H * ((4 if noised else 6) * C * D * D + 8 * C * C * D)


def _layer_params(cfg, kind):
    D, I = cfg.hidden_size, cfg.intermediate_size
    n = 3 * D * I
    if kind == model.FULL:
        q = cfg.num_attention_heads * cfg.head_dim
        return n + D * (2 * q + 2 * cfg.num_key_value_heads * cfg.head_dim) + q * D
    kd, vd = cfg.linear_num_key_heads * cfg.linear_key_head_dim, cfg.linear_num_value_heads * cfg.linear_value_head_dim
    return n + D * (2 * kd + 2 * vd + 2 * cfg.linear_num_value_heads) + vd * D


def work(case):
    k, e = case["kind"], 4 if case.get("dtype") == "fp32" else 2
    if k == "fork":
        B, L, C, Hk, Hv, D = (case[x] for x in ("B", "L", "block", "Hk", "Hv", "D"))
        Cd, T = 2 * Hk * D + Hv * D, B * L
        n = 2 * T * Cd * e + 2 * T * Hv * 8 + 2 * T * Hv * D * e + Cd * 4 * e
        if case["states"]:
            n += (T // C) * (Hv * D * D * 4 + Cd * 3 * e)
        return {"bytes": n, "flops": _rule_flops(T, Hv, D, C, False) + _rule_flops(T, Hv, D, C, True)}
    if k == "rule":
        B, T, C, Hk, Hv, D = (case[x] for x in ("B", "T", "chunk", "Hk", "Hv", "D"))
        n = B * T * ((2 * Hk + 2 * Hv) * D * e + Hv * 8)
        n += B * Hv * D * D * 4 * (int(case["init"]) + (T // C if case["states"] else 0))
        return {"bytes": n, "flops": _rule_flops(B * T, Hv, D, C, False)}
    if k == "bd":
        B, L, Hq, Hkv, d = (case[x] for x in ("B", "L", "Hq", "Hkv", "d"))
        rows = B * 2 * L * d * e
        heads = 2 * Hq + 2 * Hkv + (Hq if e == 2 else 0)  # q, out, k, v and (bf16) the gate
        return {"bytes": rows * heads, "flops": 4 * d * B * Hq * _pairs_bd(L, case["block"])}
    if k == "bc":
        B, M, N, Hq, Hkv, d = (case[x] for x in ("B", "M", "N", "Hq", "Hkv", "d"))
        return {"bytes": B * d * 2 * (3 * M * Hq + 2 * N * Hkv), "flops": 4 * d * B * Hq * _pairs_bc(M, N, case["block"])}
    if k == "mlp":
        M, H, I = case["rows"], case["hidden"], case["inter"]
        return {"bytes": 2 * (3 * H * I + M * (H + I + 3 * H)), "flops": 6 * M * H * I}
    cfg = model.config_27b_truncated(case["layers"])
    params = sum(_layer_params(cfg, t) for t in cfg.layer_types)
    head = cfg.hidden_size * cfg.vocab_size
    att = cfg.layer_types.count(model.FULL)
    gd = cfg.layer_types.count(model.LINEAR)
    Hv, D = cfg.linear_num_value_heads, cfg.linear_key_head_dim
    if k == "step":
        B, P, n = case["B"], case["prefix"], case["block"]
        rows = B * n
        state = B * (att * 2 * (P + n) * cfg.num_key_value_heads * cfg.head_dim * 2 + gd * Hv * D * D * 4)
        fl = 2 * rows * (params + head) + att * 4 * cfg.head_dim * B * cfg.num_attention_heads * n * (P + n)
        return {"bytes": 2 * (params + head) + state + rows * (cfg.vocab_size + cfg.hidden_size) * 2,
                "flops": fl + gd * _rule_flops(rows, Hv, D, n, False)}
    B, L, n = case["B"], case["L"], case["block"]
    rows = 2 * B * L
    fl = 2 * rows * (params + head) + att * 4 * cfg.head_dim * B * cfg.num_attention_heads * _pairs_bd(L, n)
    fl += gd * (_rule_flops(B * L, Hv, D, n, False) + _rule_flops(B * L, Hv, D, n, True))
    return {"bytes": 2 * (params + head) + rows * (cfg.vocab_size + cfg.hidden_size) * 2, "flops": fl}


def tolerance(case):
    k = case["kind"]
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5}
    if k in ("step", "stack"):
        # a different rounding in one of the layers travels through those after it
        return {"rel": 4e-2}
    return {"rel": 1e-2}


# ------------------------------------------------------------------------- the same in 64 bits
def _l2(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _rule64(q, k, v, g, beta, C, init=None):
    """Gated delta rule over chunks of C, float64. q, k [B, T, Hk, D], v [B, T, Hv, D], g, beta
    [B, T, Hv]; returns out [B, T, Hv, D] and the state after every chunk [B, T/C, Hv, D, D]."""
    B, T, Hk, D = k.shape
    Hv = v.shape[2]
    n = T // C
    q, k = _l2(q) * D ** -0.5, _l2(k)
    q, k = (x.repeat_interleave(Hv // Hk, 2) for x in (q, k))
    # [B, n, Hv, C, .]
    q, k, v = (x.reshape(B, n, C, Hv, D).transpose(2, 3).contiguous() for x in (q, k, v))
    g, beta = (x.reshape(B, n, C, Hv).transpose(2, 3) for x in (g, beta))
    gam = g.cumsum(-1)
    low = torch.tril(torch.ones(C, C, dtype=torch.bool, device=q.device))
    dec = (gam[..., :, None] - gam[..., None, :]).masked_fill(~low, -math.inf).exp()
    kt = k.transpose(-1, -2).contiguous()
    A = torch.tril((k @ kt) * dec * beta[..., None], -1)
    eye = torch.eye(C, dtype=q.dtype, device=q.device)
    T_ = torch.linalg.solve_triangular(A + eye, eye.expand_as(A).contiguous(), upper=False, unitriangular=True)
    U = T_ @ (v * beta[..., None])
    W = T_ @ (k * (beta * gam.exp())[..., None])
    P = (q @ kt) * dec
    qe = q * gam.exp()[..., None]
    ke = (k * (gam[..., -1:] - gam).exp()[..., None]).transpose(-1, -2).contiguous()
    lam = gam[..., -1].exp()[..., None, None]
    S = torch.zeros(B, Hv, D, D, dtype=q.dtype, device=q.device) if init is None else init
    out, states = torch.empty_like(v), []
    for i in range(n):
        vn = U[:, i] - W[:, i] @ S
        out[:, i] = qe[:, i] @ S + P[:, i] @ vn
        S = S * lam[:, i] + ke[:, i] @ vn
        states.append(S)
    return out.transpose(2, 3).reshape(B, T, Hv, D), states


def _conv64(x, w, before):
    """Causal depthwise conv + SiLU of x [N, T, C] with w [C, K], the K - 1 rows `before` [N, K - 1, C] first."""
    K, T = w.shape[1], x.shape[1]
    e = torch.cat([before, x], 1)
    return F.silu(sum(e[:, j:j + T] * w[:, j] for j in range(K)))


def _fork64(raw0, rawt, w, beta0, betat, g0, gt, Hk, Hv, D, block):
    B, L, Cd = raw0.shape
    nb = L // block
    zero = raw0.new_zeros(B, 3, Cd)
    y0 = _conv64(raw0, w, zero)
    pad = torch.cat([zero, raw0], 1)
    before = torch.stack([pad[:, k * block:k * block + 3] for k in range(nb)], 1)  # [B, nb, 3, Cd]
    yt = _conv64(rawt.reshape(B * nb, block, Cd), w, before.reshape(B * nb, 3, Cd))

    def split(y):
        return (y[..., :Hk * D].unflatten(-1, (Hk, D)), y[..., Hk * D:2 * Hk * D].unflatten(-1, (Hk, D)),
                y[..., 2 * Hk * D:].unflatten(-1, (Hv, D)))

    o0, st = _rule64(*split(y0), g0, beta0, block)
    states = torch.stack(st, 1)
    del st
    init = torch.cat([torch.zeros_like(states[:, :1]), states[:, :-1]], 1).reshape(B * nb, Hv, D, D)
    ot, _ = _rule64(*split(yt), gt.reshape(B * nb, block, Hv), betat.reshape(B * nb, block, Hv), block, init)
    return o0, ot.reshape(B, L, Hv, D), states, before.reshape(B * nb, 3, Cd).transpose(1, 2)


def _rms64(x, w, unit=1.0):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * (unit + w)


def _rope64(x, cos, sin):
    """x [B, S, H, d] with tables [S, rd]."""
    rd = cos.shape[-1]
    a, rest = x[..., :rd], x[..., rd:]
    rot = torch.cat([-a[..., rd // 2:], a[..., :rd // 2]], -1)
    return torch.cat([a * cos[None, :, None] + rot * sin[None, :, None], rest], -1)


def _attend64(q, k, v, seen):
    """Softmax attention, one query head at a time; seen [S, N] bool."""
    B, S, Hq, d = q.shape
    rep = Hq // k.shape[2]
    out = torch.empty_like(q)
    for b in range(B):
        for h in range(Hq):
            kt = k[b, :, h // rep].transpose(0, 1).contiguous()
            sc = (q[b, :, h] @ kt * d ** -0.5).masked_fill(~seen, -math.inf)
            out[b, :, h] = torch.softmax(sc, -1) @ v[b, :, h // rep].contiguous()
    return out


def _seen_bd(L, block):
    i = torch.arange(L, device=DEV) // block
    top = torch.cat([i[None] == i[:, None], i[None] < i[:, None]], 1)
    return torch.cat([top, torch.cat([torch.zeros(L, L, dtype=torch.bool, device=DEV), i[None] <= i[:, None]], 1)], 0)


def _seen_bc(M, N, block):
    return torch.arange(N, device=DEV)[None] // block <= (N - M + torch.arange(M, device=DEV))[:, None] // block


def _stack64(tm, head, x0, xt, block, clean_rows=None):
    """Both streams through the layers in float64: (noised, clean) logits; with clean_rows, only
    the clean logits of the last so many rows."""
    B, L = x0.shape
    cfg = tm.config
    W = lambda lin: lin.weight.double()  # noqa: E731
    D = cfg.linear_key_head_dim
    h = F.embedding(torch.cat([xt, x0]), W(tm.embed_tokens))  # rows 0..B-1 noised, B..2B-1 clean
    rd = int(cfg.head_dim * cfg.partial_rotary_factor)
    cos, sin = (t.double() for t in _tables(L, rd, torch.bfloat16))
    cos, sin = torch.cat([cos, cos]), torch.cat([sin, sin])
    for i, kind in enumerate(cfg.layer_types):
        ly = tm.layers[i]
        n = _rms64(h, W(ly.input_layernorm))
        if kind == model.LINEAR:
            m = ly.linear_attn
            raw, z = n @ W(m.in_proj_qkv).t(), n @ W(m.in_proj_z).t()
            beta = torch.sigmoid(n @ W(m.in_proj_b).t())
            g = -m.A_log.double().exp() * F.softplus(n @ W(m.in_proj_a).t() + m.dt_bias.double())
            o0, ot, _, _ = _fork64(raw[B:], raw[:B], W(m.conv1d).squeeze(1), beta[B:], beta[:B], g[B:], g[:B],
                                   m.num_k_heads, m.num_v_heads, D, block)
            o = _rms64(torch.cat([ot, o0]), W(m.norm), 0.0) * F.silu(z.reshape(2 * B, L, m.num_v_heads, D))
            h = h + o.reshape(2 * B, L, -1) @ W(m.out_proj).t()
        else:
            a = ly.self_attn
            x = torch.cat([n[:B], n[B:]], 1)  # [B, 2L, D]
            qg = (x @ W(a.q_proj).t()).reshape(B, 2 * L, -1, 2 * a.head_dim)
            k = (x @ W(a.k_proj).t()).reshape(B, 2 * L, -1, a.head_dim)
            v = (x @ W(a.v_proj).t()).reshape(B, 2 * L, -1, a.head_dim)
            q = _rope64(_rms64(qg[..., :a.head_dim], W(a.q_norm)), cos, sin)
            k = _rope64(_rms64(k, W(a.k_norm)), cos, sin)
            o = _attend64(q, k, v, _seen_bd(L, block)) * torch.sigmoid(qg[..., a.head_dim:])
            o = o.reshape(B, 2 * L, -1) @ W(a.o_proj).t()
            h = h + torch.cat([o[:, :L], o[:, L:]])
        n = _rms64(h, W(ly.post_attention_layernorm))
        h = h + (F.silu(n @ W(ly.mlp.gate_proj).t()) * (n @ W(ly.mlp.up_proj).t())) @ W(ly.mlp.down_proj).t()
    h = _rms64(h, W(tm.norm))
    if clean_rows:
        return None, h[B:, -clean_rows:] @ W(head).t()
    y = h @ W(head).t()
    return y[:B], y[B:]


@torch.no_grad()
def exact(case, seed):
    s, k = prepare(case, seed), case["kind"]
    d = {n: t.double() for n, t in s.items() if isinstance(t, torch.Tensor) and t.is_floating_point()}
    if k == "fork":
        o0, ot, st, tails = _fork64(d["raw0"], d["rawt"], d["w"], d["beta0"], d["betat"], d["g0"], d["gt"], case["Hk"],
                                    case["Hv"], case["D"], case["block"])
        return {"o0": o0, "ot": ot, "states": st, "tails": tails} if case["states"] else {"o0": o0, "ot": ot}
    if k == "rule":
        out, st = _rule64(d["q"], d["k"], d["v"], d["g"], d["beta"], case["chunk"], d.get("init"))
        return {"out": out, "states": torch.stack(st, 1)} if case["states"] else {"out": out}
    if k == "bd":
        seen = _seen_bd(case["L"], case["block"])
        if case["dtype"] == "fp32":
            return _attend64(d["q"], d["k"], d["v"], seen)
        cos, sin = torch.cat([d["cos"], d["cos"]]), torch.cat([d["sin"], d["sin"]])
        q = _rope64(_rms64(d["q"], d["qw"]), cos, sin)
        return _attend64(q, d["k"], d["v"], seen) * torch.sigmoid(d["gate"])
    if k == "bc":
        return _attend64(d["q"], d["k"], d["v"], _seen_bc(case["M"], case["N"], case["block"])) * torch.sigmoid(d["gate"])
    if k == "mlp":
        act = F.silu(d["x"] @ d["gate"].t()) * (d["x"] @ d["up"].t())
        h = act @ d["down"].t() + d["res"]
        return {"act": act, "y": _rms64(h, d["nw"]), "h": h}
    if k == "step":
        ids = s["ids"]
        return _stack64(s["tm"], s["head"], ids, ids, case["block"], clean_rows=case["block"])[1]
    lt, l0 = _stack64(s["tm"], s["head"], s["x0"], s["xt"], case["block"])
    return {"noised": lt, "clean": l0}
