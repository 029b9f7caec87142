"""The mixer's small-batch kernels through the C entry points (BSSM_ROW_KERNELS): a given prior and its gradients,
float32 (precise) and bfloat16 results, gradients without the dynamics; off whole tiles and on them, one group of 4 heads
to a workgroup and two.  Against the float64 oracle, as the tile kernels in test_gpu_mixer.py."""
from __future__ import annotations

import pytest
import torch

from oracle import bssm_oracle as O
from tests.test_gpu_mixer import CHUNK, EPS32, _device_views, _gate_inputs, _lds, _state, close

pytestmark = pytest.mark.gpu

# Batch, tokens, heads, row padding of the projections and of the gate; the last two have more than 256 groups.
CASES = [(1, 1, 4, 8, 0), (2, 7, 8, 0, 8), (1, 17, 12, 8, 0), (3, 16, 20, 8, 8), (2, 36, 16, 0, 0), (65, 9, 16, 0, 0),
         (33, 12, 32, 8, 0)]
NAMES = ["g_q", "g_k", "g_v", "g_decay_logits", "g_noise"]


def _chunk():
    from bayes_ssm import _hip

    return CHUNK | _hip.ANY_SHAPE | _hip.ROW_KERNELS


def _pairs(dv, lds):
    return [y for x, ld in zip(dv, lds) for y in (x.data_ptr(), ld)]


def _beliefs(n, t, dev):
    nb = -(-t // CHUNK)
    return (torch.empty(n, 4, 8, device=dev), torch.empty(n, 4, 4, device=dev),
            torch.empty(n, nb + 1, 4, 8, device=dev), torch.empty(n, nb + 1, 4, 4, device=dev))


def _grads(dv, f32, dyn):
    dtype = torch.float32 if f32 else torch.bfloat16
    return [torch.empty(x.shape, device=x.device, dtype=dtype) if i < 3 or dyn else None for i, x in enumerate(dv)]


def _forward(dv, lds, d, b, t, h):
    from bayes_ssm import _hip

    read = torch.empty(b, t, h * 8, device=dv[0].device)
    bel = _beliefs(b * h, t, dv[0].device)
    P = _hip.ptr
    _hip.call("bssm_mixer_forward", *_pairs(dv, lds), P(d["m0"]), P(d["c0"]), P(read), *map(P, bel), b, t, h, _chunk(),
              1e-6, _hip.stream_of(dv[0].device))
    return (read, *bel)


def _backward(dv, lds, d, bm, bc, b, t, h, *, f32, dyn=True, final=True):
    from bayes_ssm import _hip

    grads = _grads(dv, f32, dyn)
    initial = [torch.empty_like(d["m0"]), torch.empty_like(d["c0"])] if final else [None, None]
    ends = [d["gmf"], d["gcf"]] if final else [None, None]
    P = _hip.ptr
    _hip.call("bssm_mixer_backward", *_pairs(dv, lds), P(d["m0"]), P(d["c0"]), P(bm), P(bc), P(d["gy"]), *map(P, ends),
              *map(P, grads), *map(P, initial), b, t, h, _chunk(), 1e-6, int(f32), _hip.stream_of(dv[0].device))
    return grads + initial


def _gated_forward(dv, lds, gate, d, b, t, h, precise):
    from bayes_ssm import _hip

    dev = dv[0].device
    out = torch.empty(b, t, h * 8, device=dev, dtype=torch.float32 if precise else torch.bfloat16)
    yb = torch.empty(b, t, h * 8, device=dev, dtype=torch.bfloat16)
    bel = _beliefs(b * h, t, dev)
    P = _hip.ptr
    _hip.call("bssm_mixer_gated_forward", *_pairs(dv, lds), P(gate), gate.stride(1), P(d["w"]), EPS32, P(d["m0"]),
              P(d["c0"]), P(out), P(yb), *map(P, bel), b, t, h, _chunk(), 1e-6, int(precise), _hip.stream_of(dev))
    return (out, yb, *bel)


def _gated_backward(dv, lds, gate, d, bm, bc, yb, b, t, h, precise, dyn=True):
    from bayes_ssm import _hip

    dev = dv[0].device
    grads = _grads(dv, precise, dyn)
    ggate = torch.empty(b, t, h * 8, device=dev, dtype=torch.float32 if precise else torch.bfloat16)
    part = torch.full((4 * b * (-(-h // 16)), 8), float("nan"), device=dev)  # every row is written
    gm0, gc0 = torch.empty_like(d["m0"]), torch.empty_like(d["c0"])
    P = _hip.ptr
    _hip.call("bssm_mixer_gated_backward", *_pairs(dv, lds), P(gate), gate.stride(1), P(d["w"]), EPS32, P(d["m0"]),
              P(d["c0"]), P(bm), P(bc), P(yb), P(d["gout"]), P(d["gmf"]), P(d["gcf"]), *map(P, grads), P(ggate),
              P(part), P(gm0), P(gc0), b, t, h, _chunk(), 1e-6, int(precise), _hip.stream_of(dev))
    return grads + [ggate, part.sum(0), gm0, gc0]


def _inputs(b, t, h, pad, device):
    views, g_read = O.make_mixer_inputs(b, t, h, seed=500 + t, ld_pad=pad)
    m0, c0, gmf, gcf = _state(b * h, seed=t)
    dv = _device_views(views, device)
    d = {k: x.to(device) for k, x in dict(m0=m0, c0=c0, gmf=gmf, gcf=gcf, gy=g_read).items()}
    return views, g_read, (m0, c0, gmf, gcf), dv, d


@pytest.mark.parametrize("b,t,h,pad,gpad", CASES)
def test_core(cuda_device, b, t, h, pad, gpad):
    print(f"mixer row abi core b={b} t={t} h={h}", flush=True)
    views, g_read, (m0, c0, gmf, gcf), dv, d = _inputs(b, t, h, pad, cuda_device)
    lds = _lds(views)
    read, mT, cT, bm, bc = _forward(dv, lds, d, b, t, h)
    g32, g16 = (_backward(dv, lds, d, bm, bc, b, t, h, f32=f) for f in (True, False))
    lean = _backward(dv, lds, d, bm, bc, b, t, h, f32=True, dyn=False, final=False)
    torch.cuda.synchronize()
    e_read, e_mT, e_cT, e_grads = O.mixer_grads(*views, h, m0, c0, g_read, gmf, gcf)
    close(read.view(b, t, h, 8), e_read, "read")
    close(mT, e_mT, "mean_T")
    close(cT, e_cT, "cov_T")
    e_bm, e_bc = O.checkpoints(*O.mixer_inputs(*views, h), m0.double(), c0.double(), CHUNK, 1e-6)
    close(bm, e_bm, "bmean")
    close(bc, e_bc, "bcov")
    for name, a, e in zip(NAMES + ["g_mean0", "g_cov0"], g32, e_grads):
        close(a, e, name)
    for name, a, e in zip(NAMES, g16, g32):
        assert torch.equal(a, e.bfloat16()), f"{name} (bf16) is not the float32 gradient rounded"
    for a, e in zip(g16[5:], g32[5:]):
        assert torch.equal(a, e)
    _, _, _, e_lean = O.mixer_grads(*views, h, m0, c0, g_read)
    for name, a, e in zip(NAMES[:3], lean, e_lean):
        close(a, e, f"lean {name}")


@pytest.mark.parametrize("b,t,h,pad,gpad", CASES)
def test_gated(cuda_device, b, t, h, pad, gpad):
    print(f"mixer row abi gated b={b} t={t} h={h}", flush=True)
    views, _, (m0, c0, gmf, gcf), dv, d = _inputs(b, t, h, pad, cuda_device)
    lds = _lds(views)
    gate, w, gout = _gate_inputs(b, t, h, seed=t, gate_pad=gpad)
    gate_d = _device_views([gate], cuda_device)[0] if gpad else gate.to(cuda_device)
    d["w"], d["gout"] = w.to(cuda_device), gout.to(cuda_device)
    o32, yb, mT, cT, bm, bc = _gated_forward(dv, lds, gate_d, d, b, t, h, True)
    o16, yb2, *_ = _gated_forward(dv, lds, gate_d, d, b, t, h, False)
    g32, g16 = (_gated_backward(dv, lds, gate_d, d, bm, bc, yb, b, t, h, f) for f in (True, False))
    fixed = _gated_backward(dv, lds, gate_d, d, bm, bc, yb, b, t, h, True, dyn=False)
    torch.cuda.synchronize()
    leaves = [x.detach().double().requires_grad_(True) for x in (*views, gate, w, m0, c0)]
    read, e_mT, e_cT = O.mixer_core(*leaves[:5], h, leaves[7], leaves[8])
    e_out = O.mixer_readout(read, leaves[5], leaves[6], EPS32, read_bf16=yb.cpu())
    close(yb.view(b, t, h, 8), read, "read_bf16", rtol=2 ** -8, atol=1e-6)
    close(o32, e_out, "out")
    close(mT, e_mT, "mean_T")
    close(cT, e_cT, "cov_T")
    assert torch.equal(yb, yb2)
    assert torch.equal(o16, o32.bfloat16()), "bf16 out is not the float32 product rounded"
    loss = (e_out * gout.double()).sum() + (e_mT * gmf.double()).sum() + (e_cT * gcf.double()).sum()
    e_grads = torch.autograd.grad(loss, leaves)
    names = NAMES + ["g_gate", "g_norm_weight", "g_mean0", "g_cov0"]
    for name, a, e in zip(names, g32, e_grads):
        # The weight gradient sums b t h terms of order one.
        close(a, e, name, atol=max(1e-4, 1e-7 * b * t * h) if name == "g_norm_weight" else 1e-4)
    for name, a, e in zip(names[:6], g16, g32):
        assert torch.equal(a, e.bfloat16()), f"{name} (bf16) is not the float32 gradient rounded"
    for a, e in zip(g16[6:], g32[6:]):
        assert torch.equal(a, e)
    # Without the dynamics' gradients: the others as they were.
    assert fixed[3] is None and fixed[4] is None
    for name, a, e in zip(names, fixed, g32):
        if a is not None:
            assert torch.equal(a, e), name
