"""The gated readout and the block with ``norm_eps = 0``: 1 / rms is infinite
where a head's values are all zero, and the kernels read zeros for tokens past
T and for heads past the row's last.  Both kernel families (small batch, large
batch) against the float64 oracle, at sequence lengths and head counts that end
inside chunks, tiles and waves."""
from __future__ import annotations

import pytest
import torch

from oracle import bssm_oracle as O
from tests.test_gpu_mixer_row import limits  # noqa: F401  (fixture)
from tests.test_gpu_mixer_shapes import _inputs, _spy

pytestmark = pytest.mark.gpu

SHAPES = [(2, t, h) for t in (7, 12, 17, 33) for h in (8, 16, 24)]


def _gradients_close(got, want, what):
    """As the small-batch readout's test against the large-batch kernels: a readout beside a bfloat16 rounding boundary
    may move one step (2^-7 of its value), which the gradients take over as a share of their largest."""
    assert torch.isfinite(got).all(), what
    torch.testing.assert_close(got.double().cpu(), want.double(), rtol=2 ** -6,
                               atol=2 ** -7 * want.abs().max().item(), msg=lambda m: f"{what}: {m}")


@pytest.mark.parametrize("b,t,h", SHAPES)
@pytest.mark.parametrize("small", [False, True])
def test_readout(cuda_device, monkeypatch, limits, b, t, h, small):  # noqa: F811
    from bayes_ssm import mixer

    print(f"norm_eps 0 readout b={b} t={t} h={h} small={small}", flush=True)
    limits(small)
    views, dev, _ = _inputs(b, t, h, seed=13 * t + h, device=cuda_device, pad=8)
    g = torch.Generator().manual_seed(t)
    gate, gy = (torch.randn(b, t, 8 * h, generator=g).to(torch.bfloat16) for _ in range(2))
    weight = (1 + 0.1 * torch.randn(8, generator=g)).to(torch.bfloat16)
    leaves = [x.detach().clone(memory_format=torch.preserve_format).requires_grad_(True)
              for x in (*dev, gate.to(cuda_device), weight.to(cuda_device))]
    calls = _spy(monkeypatch, mixer._MixerReadoutFunction)
    out, _, _ = mixer.bayes_mixer_readout(*leaves, heads=h, norm_eps=0.0)
    assert calls, "the fused kernels were not used"
    grads = torch.autograd.grad(out, leaves, gy.to(cuda_device))

    e_leaves = [x.double().requires_grad_(True) for x in (*views, gate, weight)]
    read, _, _ = O.mixer_core(*e_leaves[:5], h)
    e_out = O.mixer_readout(read, e_leaves[5], e_leaves[6], 0.0,
                            read_bf16=read.detach().to(torch.bfloat16).reshape(b, t, 8 * h))
    e_grads = torch.autograd.grad(e_out, e_leaves, gy.double().reshape(e_out.shape))
    _gradients_close(out, e_out.detach().reshape(out.shape), "out")
    for got, want, what in zip(grads, e_grads, ("q", "k", "v", "decay", "noise", "gate", "weight")):
        _gradients_close(got, want, what)


@pytest.mark.parametrize("b,t,h", SHAPES)
@pytest.mark.parametrize("small", [False, True])
def test_block(cuda_device, monkeypatch, limits, b, t, h, small):  # noqa: F811
    """The block's results with a zero epsilon are those with one far below every mean square: bit for bit in the same
    kernels, within a bfloat16 rounding where the zero takes others (whole tiles)."""
    from bayes_ssm import mixer
    from tests.test_gpu_block import _inputs as block_inputs
    from tests.test_gpu_block import _bf16_close, _leaves

    print(f"norm_eps 0 block b={b} t={t} h={h} small={small}", flush=True)
    limits(small)
    projected, weight, norm_w, aux_bias, gout = block_inputs(b, t, h, seed=t + h, device=cuda_device)

    def run(eps):
        leaves, view, bias = _leaves(projected, weight, norm_w, aux_bias, False)
        calls = _spy(monkeypatch, mixer._MixerBlockFunction)
        out, _, _ = mixer.bayes_mixer_block(view, leaves[1], leaves[2], heads=h, aux_bias=bias, norm_eps=eps)
        assert calls, "the block kernels were not used"
        return (out, *torch.autograd.grad(out, leaves + [bias], gout))

    for i, (got, want) in enumerate(zip(run(0.0), run(1e-30))):
        assert torch.isfinite(got).all(), i
        if t % 4:
            assert torch.equal(got, want), i
        else:
            _bf16_close(got, want, f"result {i}")
