"""The work this framework is timed on: calls of its public entry points, over the sizes and types they are used with.

Each case is one call, or one training step (forward and backward), of

- ``diag``: the layer with diagonal dynamics, ``fused_diagonal_bayesian`` (key dims 1, 2, 4, 8 with 8 value columns;
  float32, or bfloat16 / float8 keys, values and queries at key dim 4; learned or fixed dynamics; training, or
  inference that carries a belief: prefill and decode);
- ``d64``: the wide layer (64 x 64 belief), ``bayesian_layer``;
- ``rotation``: rotation dynamics, ``bayesian_layer``;
- ``scan``: the static associative scan, ``associative_static_bayesian_cuda``;
- ``readout`` and ``block``: the mixer from its bfloat16 projections to the gated readout, without and with the
  causal depthwise-4 filter (``bayes_mixer_readout``, ``bayes_mixer_block``).

``exact`` restates each in float64 torch operations.
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

sys.path.insert(0, os.path.join(os.getcwd(), "bayes-ssm_amd"))

DEVICE = "cuda:0"
FLOOR = 1e-6


def listed():
    return [
        # One new token for 64 requests of a 64-head layer: the belief is carried from call to call.
        {"name": "decode_d4", "path": "diag", "d": 4, "n": 4096, "t": 1, "dtype": "f32", "fixed": False,
         "train": False},
        # A prompt of odd length, one request of a 64-head layer.
        {"name": "prefill_d4", "path": "diag", "d": 4, "n": 64, "t": 437, "dtype": "f32", "fixed": False,
         "train": False},
        # The scalar-key layer's training step at batch 64, 64 heads.
        {"name": "train_d1", "path": "diag", "d": 1, "n": 4096, "t": 512, "dtype": "f32", "fixed": False,
         "train": True},
        # The D = 2 variant on sequences of an odd length (a batch cut at its longest document).
        {"name": "train_d2_odd", "path": "diag", "d": 2, "n": 8192, "t": 509, "dtype": "f32", "fixed": False,
         "train": True},
        # The training shape: batch 256, 64 heads, 512 tokens.
        {"name": "train_d4", "path": "diag", "d": 4, "n": 16384, "t": 512, "dtype": "f32", "fixed": False,
         "train": True},
        # bfloat16 projections of a next-token batch (512 tokens less the last one) at batch 32.
        {"name": "train_d4_bf16_odd", "path": "diag", "d": 4, "n": 2048, "t": 511, "dtype": "bf16", "fixed": False,
         "train": True},
        # The D = 8 variant at the training shape.
        {"name": "train_d8", "path": "diag", "d": 8, "n": 16384, "t": 512, "dtype": "f32", "fixed": False,
         "train": True},
        # The wide layer: 32 sequences of 8 heads.
        {"name": "train_d64", "path": "d64", "n": 256, "t": 512, "train": True},
        # Rotation dynamics at the training shape.
        {"name": "train_rotation", "path": "rotation", "d": 4, "n": 16384, "t": 512, "train": True},
        # The static scan over longer sequences, with gradients.
        {"name": "train_scan", "path": "scan", "b": 16, "t": 1000, "d": 16, "m": 16, "train": True},
        # The mixer's gated readout on a next-token batch, from separate projections.
        {"name": "readout_odd", "path": "readout", "b": 32, "t": 511, "h": 64, "train": True},
        # The whole Bayes block between its fused projection and out_proj: batch 256, width 512.
        {"name": "train_block", "path": "block", "b": 256, "t": 512, "h": 64, "train": True},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the ranges above; never more sequences x tokens than the listed case of its path and size."""
    path = rng.choice(["diag", "diag", "diag", "diag", "d64", "rotation", "scan", "readout", "block"])
    train = rng.random() < 0.8
    if path == "diag":
        d = rng.choice([1, 2, 4, 4, 8])
        t = _log_int(rng, 1, 1024) if not train else _log_int(rng, 32, 1024)
        n = _log_int(rng, 32, min(32768, max(64, 16384 * 512 // t)))
        dtype = rng.choice(["f32", "f32", "bf16", "e4m3"]) if d == 4 else "f32"
        return {"path": path, "d": d, "n": n, "t": t, "dtype": dtype, "fixed": rng.random() < 0.2, "train": train}
    if path == "d64":
        t = _log_int(rng, 16, 512)
        return {"path": path, "n": _log_int(rng, 8, 256), "t": t, "train": train}
    if path == "rotation":
        d = rng.choice([2, 4, 8])
        t = _log_int(rng, 32, 1024)
        return {"path": path, "d": d, "n": _log_int(rng, 32, 16384 * 512 // max(t, 512) * 4 // max(d, 4)), "t": t,
                "train": train}
    if path == "scan":
        t = _log_int(rng, 16, 1000)
        return {"path": path, "b": _log_int(rng, 1, 16), "t": t, "d": rng.choice([3, 4, 8, 12, 16]),
                "m": rng.choice([4, 8, 16, 32]), "train": train}
    t = _log_int(rng, 16, 1024)
    h = rng.choice([16, 32, 48, 64, 64, 24])
    top = (256 if path == "block" else 64) * 512 * 64 // (max(t, 512) * h)
    if t % 4 or h % 16:  # the widest calls of a batch that is not cut to whole tiles
        top = min(top, 32 * 512 * 64 // (max(t, 512) * h))
    return {"path": path, "b": _log_int(rng, 1, max(2, top)), "t": t, "h": h, "train": train}


# ------------------------------------------------------------------------------------------------- inputs

_KQV = {"f32": torch.float32, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn}


def _diag_inputs(g, n, t, d, m, dtype, key_scale=1.0):
    """k, v, q through bfloat16 (what a model's projections give), positive noise, decay below one."""
    def rn(*shape):
        return torch.randn(*shape, device=DEVICE, generator=g)

    k, v, q = (key_scale * rn(n, t, d)).bfloat16(), rn(n, t, m).bfloat16(), (key_scale * rn(n, t, d)).bfloat16()
    dec = torch.sigmoid(rn(n, t, d) + 2.0)
    p = F.softplus(rn(n, t) - 3.0)
    r = 1e-4 + F.softplus(rn(n, t))
    return [k.to(dtype), v.to(dtype), q.to(dtype), dec, p, r]


def _inputs(case, seed):
    """(leaves, others): the tensors that a training step differentiates, and the rest."""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    path = case["path"]

    def rn(*shape):
        return torch.randn(*shape, device=DEVICE, generator=g)

    if path in ("diag", "d64"):
        d = case.get("d", 64)
        m = 64 if path == "d64" else 8
        n, t = case["n"], case["t"]
        leaves = _diag_inputs(g, n, t, d, m, _KQV[case.get("dtype", "f32")], 0.125 if path == "d64" else 1.0)
        if path == "diag" and not case["train"]:
            # The belief that earlier calls left: a mean and a positive definite covariance.
            a = 0.3 * rn(n, d, d)
            m0, c0 = rn(n, d, m), a @ a.transpose(1, 2) + 0.2 * torch.eye(d, device=DEVICE)
            c0 = 0.5 * (c0 + c0.transpose(1, 2))
        else:
            m0 = torch.zeros(n, d, m, device=DEVICE)
            c0 = torch.eye(d, device=DEVICE).expand(n, d, d).contiguous()
        return leaves, {"m0": m0, "c0": c0, "gy": rn(n, t, m)}
    if path == "rotation":
        n, t, d, j = case["n"], case["t"], case["d"], case["d"] // 2
        k, v, q = rn(n, t, d) / d ** 0.5, rn(n, t, 8), rn(n, t, d)
        radius = torch.exp(-F.softplus(rn(n, t, j) - 2.0))
        angle = rn(n, t, j)
        p, r = 1e-4 + F.softplus(rn(n, t, j) - 3.0), 1e-4 + F.softplus(rn(n, t))
        return [k, v, q, radius, angle, p, r], {"gy": rn(n, t, 8)}
    if path == "scan":
        b, t, d, m = case["b"], case["t"], case["d"], case["m"]
        leaves = [rn(b, t, d) / d ** 0.5, rn(b, t, m), rn(b, t, d), 1e-4 + F.softplus(rn(b, t))]
        return leaves, {"gy": rn(b, t, m)}
    b, t, h = case["b"], case["t"], case["h"]
    bf = torch.bfloat16
    if path == "readout":
        leaves = [rn(b, t, 4 * h), rn(b, t, 4 * h), rn(b, t, 8 * h), rn(b, t, 4 * h) - 4.0,
                  rn(b, t, 2 * h), rn(b, t, 8 * h)]
        leaves[4][..., ::2] -= 2.0
        leaves = [x.to(bf) for x in leaves] + [(1.0 + 0.1 * rn(8)).to(bf)]
    else:
        core, state = 16 * h, 4 * h
        projected = rn(b, t, 30 * h)
        projected[..., core:core + state] -= 4.0
        projected[..., core + state:core + state + 2 * h:2] -= 2.0
        leaves = [projected.to(bf), (0.5 * rn(core, 1, 4)).to(bf), (1.0 + 0.1 * rn(8)).to(bf),
                  (0.1 * rn(6 * h)).to(bf)]
    return leaves, {"gy": rn(b, t, 8 * h).to(bf)}


def prepare(case, seed):
    import bayes_ssm  # noqa: F401  (loads the kernels' library)

    leaves, rest = _inputs(case, seed)
    if case["train"]:
        leaves = [x.requires_grad_(True) for x in leaves]
    return {"case": case, "leaves": leaves, **rest}


# -------------------------------------------------------------------------------------------------- calls

def _forward(state):
    case, x = state["case"], state["leaves"]
    path = case["path"]
    if path == "diag":
        from bayes_ssm.fused_cuda import fused_diagonal_bayesian

        return fused_diagonal_bayesian(*x, state["m0"], state["c0"], chunk_length=64, denominator_floor=FLOOR,
                                       fixed_dynamics=case["fixed"])
    if path == "d64":
        import bayes_ssm

        k, v, q, dec, p, r = x
        return bayes_ssm.bayesian_layer(k, v, q, transition_diagonals=dec, process_variances=p,
                                        observation_variances=r, chunk_length=64, optimized=True)
    if path == "rotation":
        import bayes_ssm

        k, v, q, radius, angle, p, r = x
        return bayes_ssm.bayesian_layer(k, v, q, rotation_radii=radius, rotation_angles=angle, process_variances=p,
                                        observation_variances=r, chunk_length=64, optimized=True)
    if path == "scan":
        from bayes_ssm.replay_ssm import associative_static_bayesian_cuda

        return associative_static_bayesian_cuda(x[0], x[1], x[2], observation_variances=x[3])
    if path == "readout":
        from bayes_ssm.mixer import bayes_mixer_readout

        return bayes_mixer_readout(*x, heads=case["h"])
    from bayes_ssm.mixer import bayes_mixer_block

    return bayes_mixer_block(x[0], x[1], x[2], heads=case["h"], aux_bias=x[3])


def run(state):
    if not state["case"]["train"]:
        with torch.no_grad():
            return list(_forward(state))
    out = _forward(state)
    grads = torch.autograd.grad(out[0], state["leaves"], state["gy"])
    return [o.detach() for o in out] + list(grads)


# --------------------------------------------------------------------------------------------- work, bounds

def _layer_flops(d, m):
    """(forward, backward) operations per token and sequence of the dense recurrence, a multiply-add as two."""
    fwd = d + 2 * d * d + 3 * d + 2 * d + 2 * d * m + 3 * d * m + 4 * d * d + 2 * d * m
    return fwd, (fwd - 2 * d * m) + 16 * d * m + 14 * d * d


def work(case):
    path, train = case["path"], case["train"]
    if path in ("diag", "d64"):
        d, m = case.get("d", 64), 64 if path == "d64" else 8
        size = {"f32": 4, "bf16": 2, "e4m3": 1}[case.get("dtype", "f32")]
        tokens, state = case["n"] * case["t"], case["n"] * (d * m + d * d) * 4
        kqv, dyn = (2 * d + m) * size, 0 if case.get("fixed") else (d + 2) * 4
        fwd, bwd = _layer_flops(d, m)
        per = kqv + dyn + 4 * m
        if train:
            # The gradients of the dynamics are written (as zeros) also where the dynamics are fixed.
            per += 4 * m + kqv + (d + 2) * 4
        return {"bytes": tokens * per + 2 * state, "flops": tokens * (fwd + (bwd if train else 0))}
    if path == "rotation":
        d = case["d"]
        tokens, state = case["n"] * case["t"], case["n"] * (8 * d + d * d) * 4
        ins = (2 * d + 8 + 3 * (d // 2) + 1) * 4
        fwd, bwd = _layer_flops(d, 8)
        return {"bytes": tokens * (ins + 32 + ((32 + ins) if train else 0)) + state,
                "flops": tokens * (fwd + (bwd if train else 0))}
    if path == "scan":
        b, t, d, m = case["b"], case["t"], case["d"], case["m"]
        ins = (2 * d + m + 1) * 4
        # Per token: the prefix terms, a factorization and the solves of the value columns (twice with gradients).
        flops = 3 * d * d + 3 * d * m + d * d * d / 3 + 2 * d * d * m + 2 * d * m
        return {"bytes": b * t * (ins + 4 * m + ((ins + 4 * m) if train else 0)) + b * (d * d + d * m) * 4,
                "flops": b * t * flops * (3 if train else 1)}
    b, t, h = case["b"], case["t"], case["h"]
    ins = 30 * h * 2  # q, k, v, decay, noise and gate columns
    fwd, bwd = _layer_flops(4, 8)
    # Projections in, gated readout out; with gradients its gradient in and the projections' out.
    return {"bytes": b * t * (ins + 16 * h + ((ins + 16 * h) if train else 0)) + b * h * 48 * 4,
            "flops": b * t * h * (fwd + (bwd if train else 0))}


def tolerance(case):
    """Measured against ``exact`` over the listed and some drawn cases; about four times what two roundings give."""
    path = case["path"]
    if path in ("readout", "block"):
        # bfloat16 outputs and gradients (2^-9 each, 3e-3 to 5e-3 with the chain's other roundings); the gradient
        # through the normalization of a key near zero magnifies single elements.
        return {"rel": 0.02, "max": 0.9}
    if path == "scan":
        return {"rel": 1e-5, "max": 3e-4}  # seen 1.1e-6 and 3.6e-5: sums over up to a thousand tokens, then solves
    if path == "diag" and case["train"] and case["dtype"] == "bf16":
        return {"rel": 3e-4, "max": 0.016}  # a value beside a rounding boundary moves one step, 2^-8
    if path == "diag" and case["train"] and case["dtype"] == "e4m3":
        return {"rel": 2e-3, "max": 0.26}  # the same, 2^-3
    return {"rel": 5e-6, "max": 1e-4}  # seen 2.7e-7 and 1.1e-5


# ------------------------------------------------------------------------------------- the same in 64 bits

def _layer(k, v, q, transition, p, r, m0, c0):
    """The exact recurrence, token by token; ``transition(t)`` gives x -> A_t x on the row axis."""
    mean, cov, ys = m0, c0, []
    for t in range(k.shape[1]):
        rows = transition(t)
        kt, qt = k[:, t], q[:, t]
        mean = rows(mean)
        cov = rows(rows(cov).transpose(1, 2)) + torch.diag_embed(p[:, t])
        u = (cov @ kt.unsqueeze(-1)).squeeze(-1)
        s = (r[:, t] + (kt * u).sum(-1)).clamp_min(FLOOR)
        e = v[:, t] - (kt.unsqueeze(1) @ mean).squeeze(1)
        mean = mean + u.unsqueeze(-1) * (e / s.unsqueeze(-1)).unsqueeze(1)
        cov = cov - u.unsqueeze(-1) * (u / s.unsqueeze(-1)).unsqueeze(1)
        ys.append((qt.unsqueeze(1) @ mean).squeeze(1))
    return torch.stack(ys, 1), mean, cov


def _diagonal(k, v, q, dec, p, r, m0, c0):
    d = k.shape[2]
    return _layer(k, v, q, lambda t: lambda x: dec[:, t].unsqueeze(-1) * x, p.unsqueeze(-1).expand(-1, -1, d), r, m0,
                  c0)


def _rotation(k, v, q, radius, angle, p, r, m0, c0):
    rho = radius.clamp(max=1.0)
    c, s = rho * angle.cos(), rho * angle.sin()

    def at(t):
        def rows(x):
            even, odd = x[:, 0::2], x[:, 1::2]
            ct, st = c[:, t].unsqueeze(-1), s[:, t].unsqueeze(-1)
            return torch.stack((ct * even - st * odd, st * even + ct * odd), 2).reshape(x.shape)
        return rows

    noise = torch.stack((p, torch.zeros_like(p)), -1).reshape(k.shape)
    return _layer(k, v, q, at, noise, r, m0, c0)


def _in_parts(fn, args, size):
    """fn over parts of the sequences, each replayed in its backward: the history of one part at a time."""
    parts = [checkpoint(fn, *(x[i:i + size] for x in args), use_reentrant=False)
             for i in range(0, args[0].shape[0], size)]
    return [torch.cat(z) for z in zip(*parts)]


def _scan(k, v, q, r):
    d = k.shape[-1]
    wk = k / r.unsqueeze(-1)
    lam = torch.eye(d, device=k.device, dtype=k.dtype) + (k.unsqueeze(-1) * wk.unsqueeze(-2)).cumsum(1)
    nat = (wk.unsqueeze(-1) * v.unsqueeze(-2)).cumsum(1)
    mean = torch.linalg.solve(lam, nat)
    return ((q.unsqueeze(-2) @ mean).squeeze(-2), mean[:, -1], torch.linalg.inv(lam[:, -1]))


def _readout(q, k, v, decay, noise, gate, weight, h, part):
    b, t = q.shape[:2]

    def heads(x):
        return x.reshape(b, t, h, -1).transpose(1, 2).reshape(b * h, t, -1)

    unit = [F.normalize(heads(F.silu(x)), dim=-1) for x in (k, q)]
    pr = heads(F.softplus(noise) + 1e-4)
    n = b * h
    m0 = torch.zeros(n, 4, 8, device=q.device, dtype=q.dtype)
    c0 = torch.eye(4, device=q.device, dtype=q.dtype).expand(n, 4, 4)
    y, mean, cov = _in_parts(_diagonal, (unit[0], heads(F.silu(v)), unit[1], heads(torch.exp(-F.softplus(decay))),
                                         pr[..., 0], pr[..., 1], m0, c0), part)
    y = y.reshape(b, h, t, 8).transpose(1, 2)
    norm = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + torch.finfo(torch.float32).eps) * weight
    return (norm * F.silu(gate.reshape(b, t, h, 8))).reshape(b, t, 8 * h), mean, cov


def exact(case, seed):
    path = case["path"]
    leaves, rest = _inputs(case, seed)
    leaves = [x.double().requires_grad_(case["train"]) for x in leaves]
    with torch.set_grad_enabled(case["train"]):
        if path in ("diag", "d64"):
            args = list(leaves)
            if case.get("fixed"):  # the constants that a layer with fixed dynamics uses
                args[3:] = [torch.full_like(x, c) for x, c in zip(args[3:], (0.97, 0.1, 1.0))]
            out = _in_parts(_diagonal, (*args, rest["m0"].double(), rest["c0"].double()),
                            32 if path == "d64" else 4096)
        elif path == "rotation":
            n, d = case["n"], case["d"]
            m0 = torch.zeros(n, d, 8, device=DEVICE, dtype=torch.float64)
            c0 = torch.eye(d, device=DEVICE, dtype=torch.float64).expand(n, d, d)
            out = _in_parts(_rotation, (*leaves, m0, c0), 4096)
        elif path == "scan":
            out = _scan(*leaves)
        else:
            h = case["h"]
            if path == "readout":
                args = leaves
            else:
                projected, taps, weight, bias = leaves
                core, state = 16 * h, 4 * h
                x = F.pad(projected[..., :core], (0, 0, 3, 0))
                t = case["t"]
                # The filter's output and the biased columns are bfloat16 tensors of the block.
                x = sum(x[:, j:j + t] * taps[:, 0, j] for j in range(4)).to(torch.bfloat16).double()
                aux = (projected[..., core:core + 6 * h] + bias).to(torch.bfloat16).double()
                args = (x[..., :state], x[..., state:2 * state], x[..., 2 * state:], aux[..., :state],
                        aux[..., state:], projected[..., core + 6 * h:], weight)
            out = _readout(*args, h, 4096)
        if not case["train"]:
            return [o.detach() for o in out]
        grads = torch.autograd.grad(out[0], leaves, rest["gy"].double(), allow_unused=True)
    return [o.detach() for o in out] + [torch.zeros_like(x) if g is None else g for g, x in zip(grads, leaves)]
