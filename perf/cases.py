"""The workloads whose speed counts: what a program that uses this package has it do, through
the public entry points, from the smallest calls to the largest.

Every case is a dict with a ``kind``:

* ``op``       the KDA operator in training: forward and exact backward (``kda``, autograd);
* ``prefill``  the operator on a prompt at inference: forward with the final state;
* ``decode``   one recurrent step of the operator, the state updated in place;
* ``mixer``    a ``KimiDeltaAttention`` block in training: forward and every gradient;
* ``prompt``   the block on a prompt at inference: output and the ``KDAState`` it leaves;
* ``step``     the block on one token with a carried ``KDAState``;
* ``gpt``      the 6-layer decoder's one-token step with its ``KVCache``: logits and states;
* ``loss``     the trainer's soft-capped cross entropy: loss and logit gradient.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from experiment_swa_kda_amd.kda import KDAState, KimiDeltaAttention, kda
from experiment_swa_kda_amd.model import GPT, GPTConfig, KVCache, softcap_cross_entropy

LOWER = -5.0
CAP = 15.0


def _op(name, B, T, H, D, gate, state=False, lens=""):
    c = {"kind": "op", "B": B, "T": T, "H": H, "D": D, "gate": gate, "state": state, "lens": lens}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest training call: a unit-test or tiny-model layer, where launches count
        _op("op_b1_t256_h2_d64", 1, 256, 2, 64, "precomputed"),
        # one layer of the 6-layer trainer, the benchmark's default workload
        _op("op_b2_t4096_h3_d128", 2, 4096, 3, 128, "precomputed"),
        # a layer of a larger model on a full card: as many chunks as a real batch brings, K3 gate
        _op("op_b4_t8192_h6_d128", 4, 8192, 6, 128, "k3"),
        # one long document, few heads: the recurrence is one long chain
        _op("op_b1_t32768_h1_d128", 1, 32768, 1, 128, "k3"),
        # packed documents of uneven lengths (16,384 tokens, lengths from U(128, 8192) at seed 7)
        _op("op_packed_16384_h8_d128", 1, 16384, 8, 128, "precomputed", lens="7748,5169,3467"),
        # a head size between the two main ones, a ragged length, state carried in and out
        _op("op_b2_t1999_h3_d96", 2, 1999, 3, 96, "k3", state=True),
        # prompt prefill of a serving batch through the operator
        {"name": "prefill_b64_t1024_h3_d128", "kind": "prefill", "B": 64, "T": 1024, "H": 3, "D": 128, "gate": "precomputed",
         "state": False},
        # the decode loop's step at a serving batch
        {"name": "decode_b64_h3_d128", "kind": "decode", "B": 64, "H": 3, "D": 128, "gate": "k3"},
        # the trainer's mixer block: projections, convolution, operator, gated norm, every gradient
        {"name": "mixer_b2_t4096_h3_d128", "kind": "mixer", "B": 2, "T": 4096, "H": 3, "D": 128},
        # a prompt through the block at inference, which leaves the state that decoding continues from
        {"name": "prompt_b4_t1000_h3_d128", "kind": "prompt", "B": 4, "T": 1000, "H": 3, "D": 128},
        # token generation with the whole decoder: embedding to logits for one token per sequence
        {"name": "gpt_step_b8", "kind": "gpt", "B": 8, "P": 48, "L": 6, "H": 3, "D": 128, "vocab": 32768},
        # the loss over a micro-batch's logits, the largest tensor of the trainer
        {"name": "loss_8192x32768", "kind": "loss", "rows": 8192, "vocab": 32768},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _chunks(c):
    return c["B"] * -(-c["T"] // 64) * c["H"]


# the training calls' recurrences (sequences x heads) and the chunks of any call: what one
# device takes of a layer, the rest being other devices' share
MOST_RECURRENCES, MOST_CHUNKS = 24, 3072


def draw(rng):
    kind = rng.choice(["op", "op", "op", "packed", "long", "prefill", "decode", "mixer", "prompt", "step", "gpt", "loss"])
    if kind in ("op", "packed", "long"):
        D = rng.choice([64, 96, 128, 128])
        gate = rng.choice(["k3", "precomputed"])
        state = rng.random() < 0.3
        if kind == "long":
            return _op("", 1, _log(rng, 8192, 32768), rng.choice([1, 2, 3]), D, gate, state)
        if kind == "packed":
            T, H = _log(rng, 1024, 16384), rng.choice([2, 3, 4])
            lens, left = [], T
            while left > 0:
                n = min(left, rng.randint(T // 8, T // 2))
                lens.append(n if len(lens) + 1 < MOST_RECURRENCES // H else left)
                left -= lens[-1]
            return _op("", 1, T, H, D, gate, state, ",".join(map(str, lens)))
        while True:
            c = _op("", rng.randint(1, 8), _log(rng, 64, 8192), rng.choice([1, 2, 3, 4, 6, 8, 12, 16]), D, gate, state)
            if _chunks(c) <= MOST_CHUNKS and c["B"] * c["H"] <= MOST_RECURRENCES:
                return c
    if kind == "prefill":
        while True:
            c = {"kind": kind, "B": _log(rng, 1, 64), "T": _log(rng, 16, 4096), "H": rng.choice([2, 3, 4, 8]),
                 "D": rng.choice([64, 128]), "gate": rng.choice(["k3", "precomputed"]), "state": rng.random() < 0.5}
            if _chunks(c) <= MOST_CHUNKS:
                return c
    if kind == "decode":
        return {"kind": kind, "B": _log(rng, 1, 256), "H": rng.choice([2, 3, 4, 8]), "D": rng.choice([64, 128]),
                "gate": rng.choice(["k3", "precomputed"])}
    if kind in ("mixer", "prompt"):
        while True:
            c = {"kind": kind, "B": rng.randint(1, 4), "T": _log(rng, 64, 4096), "H": rng.choice([2, 3, 4, 6, 8]),
                 "D": rng.choice([64, 128])}
            if _chunks(c) <= 1024 and c["B"] * c["H"] <= MOST_RECURRENCES:
                return c
    if kind == "step":
        return {"kind": kind, "B": _log(rng, 1, 128), "H": rng.choice([2, 3, 4, 6, 8]), "D": rng.choice([64, 128])}
    if kind == "gpt":
        return {"kind": kind, "B": _log(rng, 1, 64), "P": rng.randint(8, 96), "L": rng.choice([2, 4, 6]),
                "H": rng.choice([2, 3, 6]), "D": 128, "vocab": rng.choice([8192, 32768])}
    return {"kind": "loss", "rows": _log(rng, 256, 8192), "vocab": rng.choice([4096, 8000, 16384, 32000, 32768])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _op_inputs(c, seed):
    """q, k unit per head, v and the beta logits ~ N(0, 1); the precomputed gate is
    -exp(A) softplus(N(0, 1)) with A ~ U(-1, 1), the raw K3 gate ~ N(0, 1)."""
    g = _rng(seed)
    B, T, H, D = c["B"], c.get("T", 1), c["H"], c["D"]
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    t = {"q": F.normalize(r(B, T, H, D), dim=-1).bfloat16(), "k": F.normalize(r(B, T, H, D), dim=-1).bfloat16(),
         "v": r(B, T, H, D).bfloat16()}
    A = torch.rand(H, device="cuda", generator=g) * 2 - 1
    z = r(B, T, H, D)
    t["gate"] = z.bfloat16() if c["gate"] == "k3" else -A.exp().view(H, 1) * F.softplus(z)
    t["beta"] = r(B, T, H).bfloat16()
    t["A_log"], t["dt_bias"] = A, 0.3 * r(H * D)
    n = len(c["lens"].split(",")) if c.get("lens") else B
    t["s0"] = 0.05 * r(n, H, D, D) if c.get("state") or c["kind"] == "decode" else None
    if c["kind"] == "op":
        t["do"] = r(B, T, H, D).bfloat16()
        t["ds"] = 0.05 * r(n, H, D, D) if c["state"] else None
    return t


def _cu(c):
    if not c.get("lens"):
        return None
    cu = [0]
    for n in c["lens"].split(","):
        cu.append(cu[-1] + int(n))
    return cu


def _mixer_weights(c, seed, g):
    """Weights of one block by name, at the trainer's initial scale (the output projection
    and the gate parameters as after some training, not zero)."""
    d, H, D = c["H"] * c["D"], c["H"], c["D"]
    s = 3 ** 0.5 * d ** -0.5
    u = lambda *sh: (torch.rand(*sh, device="cuda", generator=g) * 2 - 1) * s  # noqa: E731
    w = {n + ".weight": u(d, d) for n in ("q_proj", "k_proj", "v_proj", "g_proj", "o_proj")}
    w.update({"f_a_proj.weight": u(D, d), "f_b_proj.weight": u(d, D), "b_proj.weight": u(H, d)})
    w.update({n + "_conv1d.weight": 0.5 * torch.randn(d, 1, 4, device="cuda", generator=g) for n in "qkv"})
    w["A_log"] = 0.2 * torch.randn(H, device="cuda", generator=g)
    w["dt_bias"] = 0.3 * torch.randn(d, device="cuda", generator=g)
    w["o_norm.weight"] = 1 + 0.1 * torch.randn(D, device="cuda", generator=g)
    return w


def _mixer(c, w):
    with torch.device("cuda"):
        layer = KimiDeltaAttention(c["H"] * c["D"], c["H"], c["D"], mode="project_chunk", allow_fallback=False)
    layer.load_state_dict(w)
    return layer


def _mixer_state(c, g):
    B, H, D = c["B"], c["H"], c["D"]
    return [0.05 * torch.randn(B, H, D, D, device="cuda", generator=g)] + \
        [torch.randn(B, H * D, 4, device="cuda", generator=g).bfloat16() for _ in range(3)]


def _block_inputs(c, seed):
    g = _rng(seed)
    B, T, d = c["B"], c.get("T", 1), c["H"] * c["D"]
    w = _mixer_weights(c, seed, g)
    x = torch.randn(B, T, d, device="cuda", generator=g).bfloat16()
    extra = torch.randn(B, T, d, device="cuda", generator=g).bfloat16() if c["kind"] == "mixer" else None
    state = _mixer_state(c, g) if c["kind"] == "step" else None
    return w, x, extra, state


def _gpt_inputs(c, seed):
    g = _rng(seed)
    d, L = c["H"] * c["D"], c["L"]
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    w = {"transformer.wte.weight": (0.8 * r(c["vocab"], d)).bfloat16(), "lm_head.weight": 0.05 * r(c["vocab"], d)}
    for i in range(L):
        p = f"transformer.h.{i}."
        w.update({p + "attn." + n: t for n, t in _mixer_weights(c, seed, g).items()})
        w[p + "mlp.c_fc.weight"] = 0.5 * d ** -0.5 * r(4 * d, d)
        w[p + "mlp.c_proj.weight"] = 0.5 * d ** -0.5 * r(d, 4 * d)
    w["resid_lambdas"] = 1.15 - 0.10 * torch.rand(L, device="cuda", generator=g)
    w["x0_lambdas"] = 0.20 * torch.rand(L, device="cuda", generator=g)
    w["smear_gate.weight"] = 0.3 * r(1, 24)
    w["smear_lambda"], w["backout_lambda"] = 0.5 + 0.1 * r(1), 0.2 + 0.02 * r(1)
    idx = torch.randint(0, c["vocab"], (c["B"], c["P"] + 1), device="cuda", generator=g)
    return w, idx


def _loss_inputs(c, seed):
    g = _rng(seed)
    cols = -(-c["vocab"] // 64) * 64
    logits = torch.empty(c["rows"], cols, device="cuda", dtype=torch.bfloat16).normal_(0, 2.0, generator=g)
    targets = torch.randint(0, c["vocab"], (c["rows"],), device="cuda", generator=g)
    targets[torch.rand(c["rows"], device="cuda", generator=g) < 0.05] = -1
    return logits, targets


def prepare(case, seed):
    c = case
    if c["kind"] in ("op", "prefill", "decode"):
        t = _op_inputs(c, seed)
        if c["kind"] == "op":
            names = ["q", "k", "v", "gate", "beta"] + (["A_log", "dt_bias"] if c["gate"] == "k3" else []) + \
                (["s0"] if c["state"] else [])
            t["leaves"] = [t[n].requires_grad_() for n in names]
            cu = _cu(c)
            t["cu"] = None if cu is None else torch.tensor(cu, dtype=torch.int32, device="cuda")
        return c, t
    if c["kind"] in ("mixer", "prompt", "step"):
        w, x, dy, state = _block_inputs(c, seed)
        layer = _mixer(c, w)
        if c["kind"] == "mixer":
            return c, layer, [x.requires_grad_()] + list(layer.parameters()), dy
        return c, layer, x, None if state is None else KDAState(*state)
    if c["kind"] == "gpt":
        w, idx = _gpt_inputs(c, seed)
        d = c["H"] * c["D"]
        with torch.device("cuda"):
            model = GPT(GPTConfig(sequence_len=4096, vocab_size=c["vocab"], n_layer=c["L"], n_head=c["H"], n_embd=d))
        model.transformer.wte.to(dtype=torch.bfloat16)
        model.load_state_dict(w)
        model.cache_bf16_weights()  # as a server does: the weights are cast once
        cache = KVCache(c["B"], c["H"], 4096, c["D"], c["L"], "cuda", torch.bfloat16, inplace_state=True)
        with torch.no_grad():
            model(idx[:, :-1], kv_cache=cache)
        return c, model, cache, idx[:, -1:].contiguous()
    logits, targets = _loss_inputs(c, seed)
    return c, logits.requires_grad_(), targets


def run(state):
    c = state[0]
    if c["kind"] == "op":
        t = state[1]
        out, fin = kda(t["q"], t["k"], t["v"], t["gate"], t["beta"], t["A_log"], t["dt_bias"], initial_state=t["s0"],
                       output_final_state=c["state"], mode="project_chunk", lower_bound=LOWER, cu_seqlens=t["cu"],
                       gate=c["gate"])
        outs, ups = ((out, fin), (t["do"], t["ds"])) if c["state"] else ((out,), (t["do"],))
        return outs + torch.autograd.grad(outs, t["leaves"], ups)
    if c["kind"] in ("prefill", "decode"):
        t = state[1]
        with torch.no_grad():
            return kda(t["q"], t["k"], t["v"], t["gate"], t["beta"], t["A_log"], t["dt_bias"], initial_state=t["s0"],
                       output_final_state=True, mode="project_chunk" if c["kind"] == "prefill" else "project_recurrent",
                       lower_bound=LOWER, gate=c["gate"], state_in_place=c["kind"] == "decode")
    if c["kind"] == "mixer":
        _, layer, leaves, dy = state
        y, _ = layer(leaves[0])
        return (y,) + torch.autograd.grad(y, leaves, dy)
    if c["kind"] in ("prompt", "step"):
        _, layer, x, carried = state
        mode = "project_recurrent" if c["kind"] == "step" else "project_chunk"
        with torch.no_grad():
            y, st = layer(x, state=carried, output_final_state=True, mode=mode)
        return y, st.memory, st.q_conv, st.k_conv, st.v_conv
    if c["kind"] == "gpt":
        _, model, cache, token = state
        with torch.no_grad():
            logits = model(token, kv_cache=cache)
        states = [cache.get_kda_state(i) for i in range(c["L"])]
        return logits, [s.memory for s in states], [s.q_conv for s in states], [s.k_conv for s in states], \
            [s.v_conv for s in states]
    _, logits, targets = state
    loss = softcap_cross_entropy(logits, targets, c["vocab"], CAP, -1, expected_grad=1.0)
    return loss, torch.autograd.grad(loss, logits)[0]


# ---------------------------------------------------------------------------
# the work and the tolerances
# ---------------------------------------------------------------------------

def _core_flops(chunks, D):
    """Chunked delta rule, forward, per 64-token chunk and head: A, M, W, U, the triangular
    solve, W S, K^T delta, Q S, A delta."""
    return chunks * (4 * 2 * 64 * 64 * D + 64 ** 3 // 3 + 3 * 2 * 64 * D * D + 2 * 64 * 64 * D)


def work(case):
    c = case
    if c["kind"] == "loss":
        n = c["rows"] * (-(-c["vocab"] // 64) * 64)
        return {"bytes": 4 * n + 8 * c["rows"], "flops": 20 * n}
    B, T, H, D = c["B"], c.get("T", 1), c["H"], c["D"]
    n, d = B * T * H * D, H * D
    seqs = len(c["lens"].split(",")) if c.get("lens") else B
    chunks = sum(-(-int(m) // 64) for m in c["lens"].split(",")) * H if c.get("lens") else B * -(-T // 64) * H
    s_bytes = 4 * seqs * H * D * D
    gate = 4 if c.get("gate") == "precomputed" else 2
    if c["kind"] == "op":
        # q, k, v, gate, beta, dO in; o and five gradients out; states and their gradients
        return {"bytes": n * (3 * 2 + gate + 2 + 2 + 3 * 2 + gate) + 4 * B * T * H + (4 * s_bytes if c["state"] else 0),
                "flops": 3 * _core_flops(chunks, D)}
    if c["kind"] == "prefill":
        return {"bytes": n * (4 * 2 + gate) + 2 * B * T * H + s_bytes * (2 if c["state"] else 1),
                "flops": _core_flops(chunks, D)}
    if c["kind"] == "decode":
        return {"bytes": 2 * s_bytes + n * (4 * 2 + gate) + 2 * B * H, "flops": 7 * B * H * D * D}
    weights = 5 * d * d + 2 * d * D + H * d + 12 * d
    gemm = 2 * B * T * (weights - 12 * d)
    if c["kind"] == "mixer":  # x, dy, the f32 weights in; y, dx, the f32 weight gradients out
        return {"bytes": 4 * 2 * B * T * d + 8 * weights, "flops": 3 * (gemm + _core_flops(chunks, D))}
    if c["kind"] == "prompt":
        return {"bytes": 2 * 2 * B * T * d + 4 * weights + s_bytes + 3 * 2 * B * d * 4,
                "flops": gemm + _core_flops(chunks, D)}
    if c["kind"] == "step":
        return {"bytes": 2 * 2 * B * d + 4 * weights + 2 * s_bytes + 2 * 3 * 2 * B * d * 4,
                "flops": gemm + 7 * B * H * D * D}
    layer = 2 * (weights + 8 * d * d) + 2 * s_bytes + 2 * 3 * 2 * B * d * 4
    return {"bytes": c["L"] * layer + 2 * d * c["vocab"] + 4 * B * c["vocab"],
            "flops": c["L"] * (gemm + 2 * B * 8 * d * d + 7 * B * H * D * D) + 2 * B * d * c["vocab"]}


def tolerance(case):
    """bf16 activations and gradients, f32 sums.  Stated at about four times the largest
    error against exact() over the listed and some twenty drawn cases: the operator's
    outputs and gradients 4.2e-3 (up to 8.2e-3 for dA_log, a sum of few terms of both
    signs), a block 5.0e-3 and its parameter gradients 6e-3 to 1.3e-2, the decoder's logits
    8.6e-3 and its states 1.2e-2, a decode step 1.7e-3, the logit gradient 2.4e-3."""
    rel = {"prefill": 1.6e-2, "decode": 6e-3, "mixer": 3e-2, "prompt": 2e-2, "step": 2e-2, "gpt": 3e-2, "loss": 1e-2}
    if case["kind"] == "op":
        return {"rel": 3e-2 if case["gate"] == "k3" else 1.6e-2}
    return {"rel": rel[case["kind"]]}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _unit(x):
    return x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)


def _kda64(q, k, v, g, beta, s0, C=16):
    """The gated delta rule of [B, T, H, *] float64 inputs: chunks of C tokens in WY form.
    Returns (o [B, T, H, V], state [B, H, V, K])."""
    B, T, H, K = q.shape
    pad = -T % C
    N = (T + pad) // C

    def chunked(x):
        x = F.pad(x, (0, 0, 0, 0, 0, pad)) if pad else x
        return x.reshape(B, N, C, H, x.shape[-1]).permute(1, 0, 3, 2, 4)  # [N, B, H, C, *]

    q, k, v, g = chunked(_unit(q) * K ** -0.5), chunked(_unit(k)), chunked(v), chunked(g)
    b = chunked(beta.unsqueeze(-1))
    G = g.cumsum(3)
    up, last = G.exp(), G[:, :, :, -1:]
    kp, km, qp = k * up, k / up, q * up
    eye = torch.eye(C, dtype=q.dtype, device=q.device)
    P = -(b * (kp @ km.transpose(-1, -2))).tril(-1)
    inv, n = eye + P, 1
    while 2 * n < C:
        P, n = P @ P, 2 * n
        inv = inv @ (eye + P)
    A = (qp @ km.transpose(-1, -2)).tril()
    U, W = inv @ (b * v), inv @ (b * kp)
    kd, lam = (k * (last - G).exp()).transpose(-1, -2), last.exp().transpose(-1, -2)
    S = s0.transpose(-1, -2) if s0 is not None else q.new_zeros(B, H, K, v.shape[-1])
    outs = []
    for u, w, a, x, y, z in zip(U.unbind(0), W.unbind(0), A.unbind(0), qp.unbind(0), kd.unbind(0), lam.unbind(0)):
        delta = u - w @ S
        outs.append(x @ S + a @ delta)
        S = z * S + y @ delta
    o = torch.stack(outs).permute(1, 0, 3, 2, 4).reshape(B, N * C, H, v.shape[-1])[:, :T]
    return o, S.transpose(-1, -2)


def _k3(z, A_log, dt_bias):
    H, D = z.shape[-2:]
    return LOWER * torch.sigmoid(A_log.exp().view(H, 1) * (z + dt_bias.view(H, D)))


def _op64(c, t, s0):
    g = _k3(t["gate"], t["A_log"], t["dt_bias"]) if c["gate"] == "k3" else t["gate"]
    cu = _cu(c)
    args = (t["q"], t["k"], t["v"], g, torch.sigmoid(t["beta"]))
    if cu is None:
        return _kda64(*args, s0)
    parts = [_kda64(*(x[:, a:b] for x in args), None if s0 is None else s0[i:i + 1])
             for i, (a, b) in enumerate(zip(cu[:-1], cu[1:]))]
    return torch.cat([p[0] for p in parts], 1), torch.cat([p[1] for p in parts], 0)


def _conv64(x, w, before):
    """Causal depthwise convolution + SiLU; returns the activations and the last inputs."""
    W = w.shape[-1]
    z = torch.cat([before, x.transpose(1, 2)], 2)
    y = sum(z[:, :, j:j + x.shape[1]] * w[:, 0, j:j + 1] for j in range(W))
    return F.silu(y).transpose(1, 2), F.pad(z, (max(0, W - z.shape[2]), 0))[:, :, -W:]


def _block64(x, w, H, state):
    """The mixer block on float64 [B, T, d] and float64 weights (a dict by parameter name)."""
    B, T, d = x.shape
    D = d // H
    act, wins = [], []
    for i, n in enumerate("qkv"):
        before = x.new_zeros(B, d, 3) if state is None else state[1 + i][:, :, 1:]
        a, win = _conv64(x @ w[n + "_proj.weight"].T, w[n + "_conv1d.weight"], before)
        act.append(a.reshape(B, T, H, D))
        wins.append(win)
    z = (x @ w["f_a_proj.weight"].T @ w["f_b_proj.weight"].T).reshape(B, T, H, D)
    g = _k3(z, w["A_log"], w["dt_bias"])
    o, mem = _kda64(*act, g, torch.sigmoid(x @ w["b_proj.weight"].T), None if state is None else state[0])
    o = o * (o.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * w["o_norm.weight"]
    o = o * torch.sigmoid((x @ w["g_proj.weight"].T).reshape(B, T, H, D))
    return o.reshape(B, T, d) @ w["o_proj.weight"].T, [mem] + wins


def _as64(w):
    """Weights as the package multiplies with them: matrices and taps rounded to bf16."""
    return {n: (t.bfloat16() if t.ndim > 1 else t).double() for n, t in w.items()}


def _rms64(x):
    return x * (x.square().mean(-1, keepdim=True) + torch.finfo(torch.float32).eps).rsqrt()


def _gpt64(c, w, idx):
    """Logits of the last token and every layer's state after it."""
    H, L = c["H"], c["L"]
    # the two-term scalars enter in f32; the smear scalar is rounded to bf16 where it is used
    w64 = _as64(w)
    x = _rms64(w64["transformer.wte.weight"][idx])
    weight = w64["smear_lambda"] * torch.sigmoid(x[..., :24] @ w64["smear_gate.weight"].T)
    # the prompt smears within itself; the decoded token with the one before it
    smeared = torch.cat([x[:, :1], x[:, 1:] + weight[:, 1:] * x[:, :-1]], 1)
    x = x0 = smeared
    mid_out, states = None, []
    for i in range(L):
        p = f"transformer.h.{i}."
        x = w64["resid_lambdas"][i] * x + w64["x0_lambdas"][i] * x0
        layer = {n[len(p) + 5:]: t for n, t in w64.items() if n.startswith(p + "attn.")}
        mixed, st = _block64(_rms64(x), layer, H, None)
        states.append(st)
        x = x + mixed
        x = x + F.relu(_rms64(x) @ w64[p + "mlp.c_fc.weight"].T).square() @ w64[p + "mlp.c_proj.weight"].T
        mid_out = x if i == L // 2 else mid_out
    if mid_out is not None:
        x = x - w64["backout_lambda"] * mid_out
    logits = _rms64(x[:, -1:]) @ w64["lm_head.weight"].T
    return (CAP * torch.tanh(logits[..., :c["vocab"]] / CAP), *[[s[j] for s in states] for j in range(4)])


def exact(case, seed):
    c = case
    if c["kind"] in ("op", "prefill", "decode"):
        t = {n: None if x is None else x.double() for n, x in _op_inputs(c, seed).items()}
        if c["kind"] != "op":
            return _op64(c, t, t["s0"])
        names = ["q", "k", "v", "gate", "beta"] + (["A_log", "dt_bias"] if c["gate"] == "k3" else []) + \
            (["s0"] if c["state"] else [])
        leaves = [t[n].requires_grad_() for n in names]
        out, fin = _op64(c, t, t["s0"])
        outs, ups = ((out, fin), (t["do"], t["ds"])) if c["state"] else ((out,), (t["do"],))
        return tuple(o.detach() for o in outs) + torch.autograd.grad(outs, leaves, ups)
    if c["kind"] in ("mixer", "prompt", "step"):
        w, x, dy, state = _block_inputs(c, seed)
        w64, x = _as64(w), x.double()
        if c["kind"] != "mixer":
            y, st = _block64(x, w64, c["H"], None if state is None else [s.double() for s in state])
            return (y, *st)
        order = [n for n, _ in KimiDeltaAttention(c["H"] * c["D"], c["H"], c["D"]).named_parameters()]
        leaves = [x.requires_grad_()] + [w64[n].requires_grad_() for n in order]
        y, _ = _block64(x, w64, c["H"], None)
        return (y.detach(),) + torch.autograd.grad(y, leaves, dy.double())
    if c["kind"] == "gpt":
        return _gpt64(c, *_gpt_inputs(c, seed))
    logits, targets = _loss_inputs(c, seed)
    keep = targets >= 0
    loss, grad = 0.0, torch.zeros(logits.shape, dtype=torch.float64, device="cuda")
    n = keep.sum().double()
    for a in range(0, c["rows"], 1024):  # rows in blocks, so that the float64 copies stay small
        z = (CAP * torch.tanh(logits[a:a + 1024, :c["vocab"]].double() / CAP))
        lse, tgt, m = z.logsumexp(-1), targets[a:a + 1024].clamp_min(0), keep[a:a + 1024].double()
        loss = loss + (m * (lse - z.gather(1, tgt[:, None])[:, 0])).sum() / n
        p = (z - lse[:, None]).exp()
        p[torch.arange(len(tgt), device="cuda"), tgt] -= 1
        grad[a:a + 1024, :c["vocab"]] = p * (1 - (z / CAP).square()) * (m / n)[:, None]
    return loss, grad
