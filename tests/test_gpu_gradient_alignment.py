"""Upstream gradients that are contiguous but start off a 16-byte boundary (what
a concatenation of an odd number of elements and an output hands back): off whole
tiles, and at T not a multiple of 4 in bfloat16, the kernels' calls take them, bit
for bit the results of the same gradients on a boundary."""
from __future__ import annotations

import pytest
import torch

from oracle import bssm_oracle as O
from tests.test_gpu_mixer_shapes import _inputs, _spy

pytestmark = pytest.mark.gpu


def _shifted(x):
    """The values of x on a contiguous buffer that starts one element past a boundary."""
    y = torch.empty(x.numel() + 1, device=x.device, dtype=x.dtype)[1:].view(x.shape)
    y.copy_(x)
    assert y.is_contiguous() and y.data_ptr() % 8
    return y


def _compare(outs, leaves, seeds):
    want = torch.autograd.grad(outs, leaves, seeds, retain_graph=True)
    got = torch.autograd.grad(outs, leaves, [_shifted(x) for x in seeds])
    for i, (x, e) in enumerate(zip(got, want)):
        assert torch.equal(x, e), i


@pytest.mark.parametrize("kind", ["core", "readout", "block"])
@pytest.mark.parametrize("b,t,h", [(2, 7, 8), (1, 33, 16), (2, 16, 12)])
def test_mixer(cuda_device, monkeypatch, kind, b, t, h):
    from bayes_ssm import mixer
    from tests.test_gpu_block import _inputs as block_inputs

    print(f"gradient alignment {kind} b={b} t={t} h={h}", flush=True)
    g = torch.Generator().manual_seed(t)
    gm, gc = torch.randn(b * h, 4, 8, generator=g).to(cuda_device), torch.randn(b * h, 4, 4, generator=g).to(cuda_device)
    if kind == "block":
        projected, taps, weight, bias, gout = block_inputs(b, t, h, seed=t, device=cuda_device)
        leaves = [x.requires_grad_(True) for x in (projected, taps, weight, bias)]
        calls = _spy(monkeypatch, mixer._MixerBlockFunction)
        outs = mixer.bayes_mixer_block(*leaves[:3], heads=h, aux_bias=leaves[3])
    else:
        _, dev, gout = _inputs(b, t, h, seed=t, device=cuda_device, pad=8)
        gout = gout.to(cuda_device)
        leaves = [x.detach().requires_grad_(True) for x in dev]
        if kind == "core":
            calls = _spy(monkeypatch, mixer._MixerCoreFunction)
            outs = mixer.bayes_mixer_core(*leaves, heads=h)
        else:
            gate = torch.randn(b, t, 8 * h, generator=g).to(torch.bfloat16).to(cuda_device)
            weight = (1 + 0.1 * torch.randn(8, generator=g)).to(torch.bfloat16).to(cuda_device)
            leaves += [x.requires_grad_(True) for x in (gate, weight)]
            gout = gout.reshape(b, t, 8 * h).to(torch.bfloat16)
            calls = _spy(monkeypatch, mixer._MixerReadoutFunction)
            outs = mixer.bayes_mixer_readout(*leaves, heads=h)
    assert calls, "the fused kernels were not used"
    _compare(outs, leaves, [gout.view_as(outs[0]), gm, gc])


@pytest.mark.parametrize("t", [7, 33, 509])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_narrow(cuda_device, monkeypatch, dtype, t):
    from bayes_ssm import fused_cuda

    print(f"gradient alignment {dtype} t={t}", flush=True)
    k, v, q, d, p, r, gy = O.make_inputs(6, t, 4, seed=t)
    leaves = [x.to(cuda_device).requires_grad_(True) for x in (k.to(dtype), v.to(dtype), q.to(dtype), d, p, r)]
    m0, c0 = torch.zeros(6, 4, 8, device=cuda_device), torch.eye(4, device=cuda_device).expand(6, 4, 4).contiguous()
    calls = _spy(monkeypatch, fused_cuda._ChunkedBayesianBF16Function)
    outs = fused_cuda.fused_diagonal_bayesian(*leaves, m0, c0, chunk_length=64, denominator_floor=1e-6)
    assert calls, "the narrow kernels were not used"
    g = torch.Generator().manual_seed(t)
    seeds = [gy, torch.randn(6, 4, 8, generator=g), torch.randn(6, 4, 4, generator=g)]
    _compare(outs, leaves, [x.to(cuda_device) for x in seeds])
