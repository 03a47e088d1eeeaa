"""The calls that a user of this library makes, as measurable cases.

Four kinds, each through the library's public entry points (glacier_attn.py):

  attn   the attention layer on device tensors: a forward that saves nothing
         (evaluation, and the first sweep of a checkpointed step), a training
         step (forward that saves lse and the rotated q and k, then backward),
         or a checkpointed layer (forward, recompute forward, backward)
  host   the drop-in host entry points on float32 arrays, as the C# engine
         calls them: forward that saves, then backward
  proj   the q/k/v projections with LoRA adapters, forward and backward
  norm   residual add + RMSNorm, forward and backward
  block  the whole attention sub-block of a training step: norm, q/k/v
         projections, attention, O projection, residual + norm, and back

A case is a dict of plain values; `lengths` is the packed batch's sequence
lengths and `outs` the projections' widths, as comma-separated text.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("glacier.tune_amd"))
import glacier_attn as ga  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
PRECISIONS = {"bf16": ga.PREC_BF16, "fp32": ga.PREC_FP32}
EPS = 1.0e-6


def _attn(lengths, heads_q, heads_kv, head_dim, dtype="bf16", mode="step", theta=1.0e6):
    return {"kind": "attn", "mode": mode, "lengths": lengths, "heads_q": heads_q,
            "heads_kv": heads_kv, "head_dim": head_dim, "theta": theta, "dtype": dtype}


def _host(tokens, heads_q, heads_kv, head_dim, precision="bf16", theta=1.0e6):
    return {"kind": "host", "lengths": str(tokens), "heads_q": heads_q, "heads_kv": heads_kv,
            "head_dim": head_dim, "theta": theta, "dtype": "fp32", "precision": precision}


def _proj(tokens, hidden, outs, rank, dtype="bf16"):
    return {"kind": "proj", "tokens": tokens, "hidden": hidden, "outs": outs, "rank": rank,
            "dtype": dtype}


def _norm(rows, width, dtype="bf16"):
    return {"kind": "norm", "rows": rows, "width": width, "dtype": dtype}


def _block(lengths, hidden, heads_q, heads_kv, head_dim, rank, dtype="bf16", theta=1.0e6):
    return {"kind": "block", "lengths": lengths, "hidden": hidden, "heads_q": heads_q,
            "heads_kv": heads_kv, "head_dim": head_dim, "rank": rank, "theta": theta,
            "dtype": dtype}


def listed():
    named = {
        # a short prompt's evaluation, 14/2 heads of 64: launches and latency
        "attn_fwd_short": _attn("37", 14, 2, 64, mode="forward"),
        # the smaller model's layer, one training step (few heads, small grid)
        "attn_step_14h_d64_s512": _attn("512", 14, 2, 64),
        # the larger model's layer, one training step: the library's headline
        "attn_step_28h_d128_s512": _attn("512", 28, 4, 128),
        # a checkpointed layer over a packed batch of ragged sequences
        "attn_ckpt_28h_d128_packed": _attn("365,425,74,426", 28, 4, 128, mode="checkpoint"),
        # long context
        "attn_step_28h_d128_s4096": _attn("4096", 28, 4, 128),
        # the fp32-operand mode, which runs are checked with
        "attn_step_28h_d128_s512_fp32": _attn("512", 28, 4, 128, dtype="fp32"),
        # the widest head size the library is built for
        "attn_step_8h_d256_s512": _attn("512", 8, 2, 256),
        # the drop-in under the C# training loop: float32 host arrays
        "host_step_28h_d128_s512": _host(512, 28, 4, 128),
        # q/k/v projections with rank-16 adapters, the larger model
        "proj_3584_t512": _proj(512, 3584, "3584,512,512", 16),
        # the smaller model's projections in fp32, a ragged token count
        "proj_896_t201_fp32": _proj(201, 896, "896,128,128", 8, dtype="fp32"),
        # the residual add and RMSNorm either side of the sub-block
        "norm_512x3584": _norm(512, 3584),
        # the whole sub-block, two sequences of 2048, 32/8 heads
        "block_4096_b2_s2048": _block("2048,2048", 4096, 32, 8, 128, 16, theta=5.0e5),
    }
    return [dict(case, name=name) for name, case in named.items()]


HEADS = [(14, 2), (28, 4), (32, 8), (12, 3), (8, 2), (16, 16), (7, 1), (40, 8)]
OTHER_HEAD_DIMS = [32, 48, 80, 96, 112, 256]
# hidden size, q/k/v widths, block heads (query, kv, size)
MODELS = [(896, "896,128,128", (14, 2, 64)), (3584, "3584,512,512", (28, 4, 128)),
          (4096, "4096,1024,1024", (32, 8, 128)), (1000, "1000,200,200", (10, 2, 100)),
          (2048, "2048,512,512", (32, 8, 64))]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _split(rng, tokens):
    """tokens as one to four sequences."""
    n = min(rng.choice([1, 1, 2, 4]), tokens)
    cuts = sorted(rng.sample(range(1, tokens), n - 1)) if n > 1 else []
    ends = [0] + cuts + [tokens]
    return ",".join(str(b - a) for a, b in zip(ends, ends[1:]))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "attn_fp32", "attn_other", "host", "proj", "proj",
                       "proj_fp32", "norm", "block", "block"])
    hq, hkv = rng.choice(HEADS)
    theta = rng.choice([1.0e4, 5.0e5, 1.0e6])
    mode = rng.choice(["forward", "step", "step", "checkpoint"])
    hidden, outs, (bq, bkv, bd) = rng.choice(MODELS)
    rank = rng.choice([4, 8, 16, 16, 32, 64])
    if kind == "attn":
        return _attn(_split(rng, _log_int(rng, 16, 4096)), hq, hkv, rng.choice([64, 128]),
                     mode=mode, theta=theta)
    if kind == "attn_fp32":
        return _attn(_split(rng, _log_int(rng, 16, 1024)), hq, hkv, rng.choice([64, 96, 128]),
                     dtype="fp32", mode=mode, theta=theta)
    if kind == "attn_other":
        return _attn(_split(rng, _log_int(rng, 16, 2048)), hq, hkv, rng.choice(OTHER_HEAD_DIMS),
                     mode=mode, theta=theta)
    if kind == "host":
        return _host(_log_int(rng, 16, 1024), hq, hkv, rng.choice([64, 128]),
                     rng.choice(["bf16", "fp32"]), theta)
    if kind == "proj":
        return _proj(_log_int(rng, 16, 4096), hidden, outs, rank)
    if kind == "proj_fp32":
        return _proj(_log_int(rng, 16, 1024), hidden, outs, rank, dtype="fp32")
    if kind == "norm":
        return _norm(_log_int(rng, 16, 16384), rng.choice([128, 896, 1000, 3584, 4096]),
                     rng.choice(["bf16", "bf16", "fp32"]))
    dtype = rng.choice(["bf16", "bf16", "fp32"])
    tokens = _log_int(rng, 16, 512 if dtype == "fp32" else 4096)
    return _block(_split(rng, tokens), hidden, bq, bkv, bd, rank, dtype, theta)


# ---- inputs --------------------------------------------------------------


def _lengths(case):
    return [int(n) for n in case["lengths"].split(",")]


def _cu_seqlens(lengths):
    """None for one sequence, else the packed batch's offsets."""
    return None if len(lengths) == 1 else np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)


def _normal(seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def make(*shape, std=1.0, mean=0.0, dtype=torch.float32):
        t = torch.randn(*shape, device="cuda", generator=gen)
        return t.mul_(std).add_(mean).to(dtype)

    return make


def _attn_inputs(case, seed):
    rnd, dt = _normal(seed), DTYPES[case["dtype"]]
    T, hq, hkv, d = sum(_lengths(case)), case["heads_q"], case["heads_kv"], case["head_dim"]
    return {"q": rnd(T, hq, d, dtype=dt), "k": rnd(T, hkv, d, dtype=dt),
            "v": rnd(T, hkv, d, dtype=dt), "d_out": rnd(T, hq, d, std=0.01, dtype=dt)}


def _projections(rnd, n_in, outs, rank, dt, bias):
    """Frozen weights and trained adapters (B away from its zero start); the
    adapters' gradients are views of one flat buffer, zeroed as one."""
    projs = []
    for o in outs:
        projs.append({"w": rnd(o, n_in, std=n_in ** -0.5, dtype=dt),
                      "bias": rnd(o, std=0.1) if bias else None,
                      "a": rnd(n_in, rank, std=n_in ** -0.5), "b": rnd(rank, o, std=0.1),
                      "scaling": 2.0})
    return projs


def _bind_grads(projs):
    sizes = [t.numel() for p in projs for t in (p["a"], p["b"])]
    flat = torch.zeros(sum(sizes), device="cuda")
    views = iter(torch.split(flat, sizes))
    for p in projs:
        p["grad_a"] = next(views).view_as(p["a"])
        p["grad_b"] = next(views).view_as(p["b"])
    return flat


def _proj_inputs(case, seed):
    rnd, dt = _normal(seed), DTYPES[case["dtype"]]
    outs = [int(o) for o in case["outs"].split(",")]
    T = case["tokens"]
    x = rnd(T, case["hidden"], dtype=dt)
    projs = _projections(rnd, case["hidden"], outs, case["rank"], dt, bias=True)
    for p, o in zip(projs, outs):
        p["dy"] = rnd(T, o, std=0.01, dtype=dt)
    return x, projs


def _norm_inputs(case, seed):
    rnd, dt = _normal(seed), DTYPES[case["dtype"]]
    shape = (case["rows"], case["width"])
    return {"x": rnd(*shape, dtype=dt), "delta": rnd(*shape, std=0.5, dtype=dt),
            "dy": rnd(*shape, dtype=dt), "d_residual": rnd(*shape, std=0.3, dtype=dt),
            "weight": rnd(case["width"], std=0.2, mean=1.0)}


def _block_inputs(case, seed):
    rnd, dt = _normal(seed), DTYPES[case["dtype"]]
    T, H, d = sum(_lengths(case)), case["hidden"], case["head_dim"]
    q_out, kv_out = case["heads_q"] * d, case["heads_kv"] * d
    return {"x": rnd(T, H, dtype=dt), "d_n2": rnd(T, H, std=0.01, dtype=dt),
            "d_x1": rnd(T, H, std=0.01, dtype=dt),
            "w1": rnd(H, std=0.2, mean=1.0), "w2": rnd(H, std=0.2, mean=1.0),
            "qkv": _projections(rnd, H, (q_out, kv_out, kv_out), case["rank"], dt, bias=True),
            "o": _projections(rnd, q_out, (H,), case["rank"], dt, bias=False)}


# ---- prepare and run -----------------------------------------------------


def prepare(case, seed):
    return {"attn": _prepare_attn, "host": _prepare_host, "proj": _prepare_proj,
            "norm": _prepare_norm, "block": _prepare_block}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_attn(case, seed):
    t = _attn_inputs(case, seed)
    cu, theta = _cu_seqlens(_lengths(case)), case["theta"]
    eng = ga.GpuAttentionEngine(0, PRECISIONS[case["dtype"]])
    q, k = t["q"], t["k"]
    out = {"out": torch.empty_like(q)}
    if case["mode"] == "forward":
        calls = [eng.bind_forward(q, k, t["v"], out["out"], theta, cu_seqlens=cu)]
    else:
        out.update(lse=torch.empty(q.shape[1], q.shape[0], device="cuda"),
                   q_rot=torch.empty_like(q), k_rot=torch.empty_like(k),
                   dq=torch.empty_like(q), dk=torch.empty_like(k), dv=torch.empty_like(k))
        fwd = dict(q=q, k=k, v=t["v"], **{n: out[n] for n in ("out", "lse", "q_rot", "k_rot")})
        bwd = dict(d_out=t["d_out"], **{n: out[n] for n in ("dq", "dk", "dv")})
        calls = [eng.bind_step(fwd, bwd, theta, cu_seqlens=cu)]
        if case["mode"] == "checkpoint":
            # the forward sweep's output goes on to the next layer
            out["sweep_out"] = torch.empty_like(q)
            calls.insert(0, eng.bind_forward(q, k, t["v"], out["sweep_out"], theta,
                                             cu_seqlens=cu))
    return {"run": _run_attn, "engine": eng, "inputs": t, "calls": calls, "outputs": out}


def _run_attn(state):
    for call in state["calls"]:
        call()
    return state["outputs"]


def _prepare_host(case, seed):
    t = {n: x.cpu() for n, x in _attn_inputs(case, seed).items()}
    T, hq, hkv, d = sum(_lengths(case)), case["heads_q"], case["heads_kv"], case["head_dim"]
    # the projection writes q and k, the forward turns them in place
    work = {"q": torch.empty_like(t["q"]), "k": torch.empty_like(t["k"])}
    out = {"out": torch.empty_like(t["q"]), "lse": torch.empty(hq, T),
           "dq": torch.empty_like(t["q"]), "dk": torch.empty_like(t["k"]),
           "dv": torch.empty_like(t["v"])}
    arrays = {n: x.numpy() for n, x in (*work.items(), *out.items())}
    arrays["v"], arrays["d_out"] = t["v"].numpy(), t["d_out"].numpy()
    return {"run": _run_host, "engine": ga.GpuAttentionEngine(0, PRECISIONS[case["precision"]]),
            "inputs": t, "work": work, "arrays": arrays, "shape": (T, hq, hkv, d, case["theta"])}


def _run_host(state):
    eng, a, shape = state["engine"], state["arrays"], state["shape"]
    for n, x in state["work"].items():
        x.copy_(state["inputs"][n])
    eng.forward_attention(0, a["q"], a["k"], a["v"], a["out"], a["lse"], *shape)
    eng.backward_attention(0, a["d_out"], a["q"], a["k"], a["v"], a["out"], a["lse"], a["dq"],
                           a["dk"], a["dv"], *shape)
    return {n: a[m] for n, m in (("out", "out"), ("lse", "lse"), ("q_rot", "q"), ("k_rot", "k"),
                                 ("dq", "dq"), ("dk", "dk"), ("dv", "dv"))}


def _prepare_proj(case, seed):
    x, projs = _proj_inputs(case, seed)
    for p in projs:
        p["y"] = torch.empty_like(p["dy"])
    return {"run": _run_proj, "engine": ga.GpuAttentionEngine(0, PRECISIONS[case["dtype"]]),
            "x": x, "projs": projs, "rank": case["rank"], "grads": _bind_grads(projs),
            "dx": torch.empty_like(x)}


def _run_proj(state):
    eng, x, projs = state["engine"], state["x"], state["projs"]
    state["grads"].zero_()  # the optimiser step before this one
    ys = eng.proj_forward(x, projs, state["rank"])
    dx = eng.proj_backward(x, projs, state["rank"], dx=state["dx"])
    out = {"dx": dx}
    for i, p in enumerate(projs):
        out[f"y{i}"], out[f"grad_a{i}"], out[f"grad_b{i}"] = ys[i], p["grad_a"], p["grad_b"]
    return out


def _prepare_norm(case, seed):
    t = _norm_inputs(case, seed)
    out = {n: torch.empty_like(t["x"]) for n in ("x1", "y", "dx")}
    return {"run": _run_norm, "engine": ga.GpuAttentionEngine(0, PRECISIONS[case["dtype"]]),
            "inputs": t, "outputs": out}


def _run_norm(state):
    eng, t, out = state["engine"], state["inputs"], state["outputs"]
    eng.rmsnorm_forward(t["x"], t["weight"], EPS, delta=t["delta"], x1=out["x1"], y=out["y"])
    eng.rmsnorm_backward(t["dy"], out["x1"], t["weight"], EPS, d_residual=t["d_residual"],
                         dx=out["dx"])
    return out


def _prepare_block(case, seed):
    t = _block_inputs(case, seed)
    lengths = _lengths(case)
    return {"run": _run_block, "engine": ga.GpuAttentionEngine(0, PRECISIONS[case["dtype"]]),
            "inputs": t, "grads": _bind_grads(t["qkv"] + t["o"]), "rank": case["rank"],
            "theta": case["theta"], "cu": _cu_seqlens(lengths),
            "heads": (sum(lengths), -1, case["head_dim"])}


def _run_block(state):
    """Forward and backward as a training program writes them: every
    intermediate is a new tensor."""
    eng, t, rank, heads = state["engine"], state["inputs"], state["rank"], state["heads"]
    theta, cu = state["theta"], state["cu"]
    qkv = [dict(p) for p in t["qkv"]]
    o = [dict(p) for p in t["o"]]
    state["grads"].zero_()
    _, n1 = eng.rmsnorm_forward(t["x"], t["w1"], EPS)
    q, k, v = (y.view(heads) for y in eng.proj_forward(n1, qkv, rank))
    att, lse, q_rot, k_rot = eng.forward(q, k, v, theta, cu_seqlens=cu)
    att_rows = att.view(att.shape[0], -1)
    (delta,) = eng.proj_forward(att_rows, o, rank)
    x1, n2 = eng.rmsnorm_forward(t["x"], t["w2"], EPS, delta=delta)

    d_x1 = eng.rmsnorm_backward(t["d_n2"], x1, t["w2"], EPS, d_residual=t["d_x1"])
    o[0]["dy"] = d_x1
    d_att = eng.proj_backward(att_rows, o, rank)
    grads = eng.backward(d_att.view_as(att), q_rot, k_rot, v, att, lse, theta, cu_seqlens=cu)
    for p, g in zip(qkv, grads):
        p["dy"] = g.view(g.shape[0], -1)
    d_n1 = eng.proj_backward(n1, qkv, rank)
    dx = eng.rmsnorm_backward(d_n1, t["x"], t["w1"], EPS, d_residual=d_x1)
    out = {"x1": x1, "n2": n2, "dx": dx}
    for i, p in enumerate(qkv + o):
        out[f"grad_a{i}"], out[f"grad_b{i}"] = p["grad_a"], p["grad_b"]
    return out


# ---- what a pass cannot do without ---------------------------------------


def _attn_flops(case, per_pair):
    """per_pair * head_dim flops for each unmasked (query, key, head)."""
    pairs = sum(n * (n + 1) // 2 for n in _lengths(case))
    return per_pair * case["head_dim"] * case["heads_q"] * pairs


def _proj_flops(T, n_in, outs, rank):
    """Base products both ways (dX only: W is frozen) and six low-rank ones."""
    return sum(4 * T * n_in * o + 6 * T * rank * (n_in + o) for o in outs)


def _proj_weights(n_in, outs, rank, size):
    """Bytes of the weights and biases, and of the adapters (read once) and
    their gradients (written once)."""
    return sum(n_in * o * size + 4 * o + 2 * 4 * rank * (n_in + o) for o in outs)


def work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    kind = case["kind"]
    if kind in ("attn", "host"):
        T, hq, hkv, d = sum(_lengths(case)), case["heads_q"], case["heads_kv"], case["head_dim"]
        mode = case.get("mode", "step")
        q_rows, kv_rows = T * hq * d * size, T * hkv * d * size
        if mode == "forward":
            return {"bytes": 2 * q_rows + 2 * kv_rows, "flops": _attn_flops(case, 4)}
        # q, k, v, d_out in; out, lse, q_rot, k_rot, dq, dk, dv out
        moved = 5 * q_rows + 5 * kv_rows + 4 * T * hq
        if mode == "checkpoint":
            return {"bytes": moved + q_rows, "flops": _attn_flops(case, 16)}
        return {"bytes": moved, "flops": _attn_flops(case, 12)}
    if kind == "proj":
        outs = [int(o) for o in case["outs"].split(",")]
        T, n_in, rank = case["tokens"], case["hidden"], case["rank"]
        return {"bytes": T * (2 * n_in + 2 * sum(outs)) * size + _proj_weights(n_in, outs, rank, size),
                "flops": _proj_flops(T, n_in, outs, rank)}
    if kind == "norm":
        cells = case["rows"] * case["width"]
        return {"bytes": 7 * cells * size + 4 * case["width"], "flops": 16 * cells}
    T, H, d = sum(_lengths(case)), case["hidden"], case["head_dim"]
    q_out, kv_out = case["heads_q"] * d, case["heads_kv"] * d
    qkv, rank = (q_out, kv_out, kv_out), case["rank"]
    return {"bytes": 6 * T * H * size + 8 * H + _proj_weights(H, qkv, rank, size)
            + _proj_weights(q_out, (H,), rank, size),
            "flops": _attn_flops(case, 12) + _proj_flops(T, H, qkv, rank)
            + _proj_flops(T, q_out, (H,), rank)}


# ---- the same in 64 bits -------------------------------------------------


# The largest 2-norm error of any output against 64 bits, seen over the listed
# cases and drawn ones: attention 4.3e-3 in bf16 (8.5e-7 in fp32), projections
# and norm 1.7e-3 (1.1e-6; the norm 6.5e-8), the block 8.3e-3 (2.2e-6).
REL = {"attn": {"bf16": 1.7e-2, "fp32": 4.0e-6}, "host": {"bf16": 1.7e-2, "fp32": 4.0e-6},
       "proj": {"bf16": 7.0e-3, "fp32": 4.0e-6}, "norm": {"bf16": 7.0e-3, "fp32": 4.0e-7},
       "block": {"bf16": 3.3e-2, "fp32": 1.0e-5}}


def tolerance(case):
    """About four times that error."""
    return {"rel": REL[case["kind"]][case.get("precision", case["dtype"])]}


def _rope(x, lengths, theta):
    """Half-split rotation by position * theta^(-2i/d); the angles are float32
    (that is the interface's definition), the rest is 64-bit."""
    half = x.shape[-1] // 2
    power = torch.arange(0, 2 * half, 2, dtype=torch.float32) / x.shape[-1]
    freq = 1.0 / torch.pow(torch.tensor(theta, dtype=torch.float64), power.double()).float()
    pos = torch.cat([torch.arange(n) for n in lengths]).float()
    angle = (pos[:, None] * freq[None, :]).double().to(x.device)[:, None, :]
    c, s = torch.cos(angle), torch.sin(angle)
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., 2 * half:]], dim=-1)


def _attention(q, k, v, lengths, theta):
    """Causal grouped-query attention of packed sequences, head by head."""
    q_rot, k_rot = _rope(q, lengths, theta), _rope(k, lengths, theta)
    group, scale = q.shape[1] // k.shape[1], q.shape[2] ** -0.5
    outs, lses, start = [], [], 0
    for n in lengths:
        rows = slice(start, start + n)
        start += n
        future = torch.ones(n, n, dtype=torch.bool, device=q.device).triu(1)
        heads, stats = [], []
        for h in range(q.shape[1]):
            g = h // group
            scores = torch.mm(q_rot[rows, h], k_rot[rows, g].t().contiguous()) * scale
            scores = scores.masked_fill(future, -math.inf)
            lse = torch.logsumexp(scores, dim=1)
            heads.append(torch.mm(torch.exp(scores - lse[:, None]), v[rows, g]))
            stats.append(lse)
        outs.append(torch.stack(heads, dim=1))
        lses.append(torch.stack(stats))
    return torch.cat(outs), torch.cat(lses, dim=1), q_rot, k_rot


def _linear(x, p):
    y = x @ p["w"].t() + p["scaling"] * ((x @ p["a"]) @ p["b"])
    return y if p["bias"] is None else y + p["bias"]


def _rmsnorm(x, weight):
    return x * torch.rsqrt(x.pow(2).mean(dim=1, keepdim=True) + EPS) * weight


def _wide(t, grad=True):
    return t.double().requires_grad_(grad)


def _wide_projections(projs):
    return [{"w": p["w"].double(), "bias": None if p["bias"] is None else p["bias"].double(),
             "a": _wide(p["a"]), "b": _wide(p["b"]), "scaling": p["scaling"]} for p in projs]


def _adapter_grads(projs):
    out = {}
    for i, p in enumerate(projs):
        out[f"grad_a{i}"], out[f"grad_b{i}"] = p["a"].grad, p["b"].grad
    return out


def exact(case, seed):
    out = {"attn": _exact_attn, "host": _exact_attn, "proj": _exact_proj, "norm": _exact_norm,
           "block": _exact_block}[case["kind"]](case, seed)
    return {n: t.detach() for n, t in out.items()}


def _exact_attn(case, seed):
    t = _attn_inputs(case, seed)
    mode = case.get("mode", "step")
    q, k, v = (_wide(t[n], mode != "forward") for n in ("q", "k", "v"))
    out, lse, q_rot, k_rot = _attention(q, k, v, _lengths(case), case["theta"])
    if mode == "forward":
        return {"out": out}
    torch.autograd.backward(out, t["d_out"].double())
    res = {"out": out, "lse": lse, "q_rot": q_rot, "k_rot": k_rot, "dq": q.grad, "dk": k.grad,
           "dv": v.grad}
    if mode == "checkpoint":
        res["sweep_out"] = out
    return res


def _exact_proj(case, seed):
    x, projs = _proj_inputs(case, seed)
    x, dys = _wide(x), [p["dy"].double() for p in projs]
    projs = _wide_projections(projs)
    ys = [_linear(x, p) for p in projs]
    torch.autograd.backward(ys, dys)
    return {"dx": x.grad, **{f"y{i}": y for i, y in enumerate(ys)}, **_adapter_grads(projs)}


def _exact_norm(case, seed):
    t = {n: x.double() for n, x in _norm_inputs(case, seed).items()}
    # the norm is taken of x1 as it is stored
    x1 = (t["x"] + t["delta"]).to(DTYPES[case["dtype"]]).double().requires_grad_()
    y = _rmsnorm(x1, t["weight"])
    torch.autograd.backward(y, t["dy"])
    return {"x1": x1, "y": y, "dx": x1.grad + t["d_residual"]}


def _exact_block(case, seed):
    t = _block_inputs(case, seed)
    lengths, d = _lengths(case), case["head_dim"]
    x = _wide(t["x"])
    qkv, o = _wide_projections(t["qkv"]), _wide_projections(t["o"])
    n1 = _rmsnorm(x, t["w1"].double())
    q, k, v = (_linear(n1, p).view(x.shape[0], -1, d) for p in qkv)
    att, _, _, _ = _attention(q, k, v, lengths, case["theta"])
    x1 = x + _linear(att.reshape(x.shape[0], -1), o[0])
    n2 = _rmsnorm(x1, t["w2"].double())
    torch.autograd.backward([n2, x1], [t["d_n2"].double(), t["d_x1"].double()])
    return {"x1": x1, "n2": n2, "dx": x.grad, **_adapter_grads(qkv + o)}
