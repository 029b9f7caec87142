"""The mixer's small-batch kernels (a workgroup per one or two groups of 4
heads) against the float64 oracle and against the fused kernels of larger
batches, which the same calls take when the small-batch limits are zero: one
group and two to a workgroup, an odd number of groups, head counts whose last
group leaves partial rows empty, and sequences that end inside chunks and
tiles.  float32 outputs at the parity tolerance (1e-5 relative, 1e-4
absolute), bfloat16 ones within their roundings besides."""
from __future__ import annotations

import pytest
import torch

from oracle import bssm_oracle as O
from tests.test_gpu_mixer_shapes import _bf16_close, _inputs, _spy
from tests.test_gpu_parity import close

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 4), (3, 7, 4), (1, 7, 16), (2, 8, 20), (1, 9, 16), (1, 16, 36), (2, 17, 12), (5, 33, 8), (257, 21, 4),
          (65, 41, 16)]


@pytest.fixture
def limits():
    """set(small): both small-batch limits as far up as any size, or zero."""
    from bayes_ssm import _hip

    lib = _hip.load()
    old = [lib.bssm_small_batch_limit(d, -1) for d in (2, 3)]

    def put(small):
        for d in (2, 3):
            lib.bssm_small_batch_limit(d, 1 << 30 if small else 0)

    yield put
    for d, n in zip((2, 3), old):
        lib.bssm_small_batch_limit(d, n)


def _small_kernels(b, t, h):
    """Whether both directions of a call off whole tiles take the small-batch kernels."""
    from bayes_ssm import _hip, mixer

    return all(mixer._chunk_arg(b, h, t, backward=x) & _hip.ROW_KERNELS for x in (False, True))


@pytest.mark.parametrize("b,t,h", SHAPES)
@pytest.mark.parametrize("final_grads", [False, True])
def test_core_matches_oracle(cuda_device, monkeypatch, limits, b, t, h, final_grads):
    from bayes_ssm import mixer

    print(f"mixer row core b={b} t={t} h={h} final_grads={final_grads}", flush=True)
    limits(True)
    calls = _spy(monkeypatch, mixer._MixerCoreFunction)
    views, dev, g_read = _inputs(b, t, h, seed=5 * t + h, device=cuda_device, pad=8)
    g = torch.Generator().manual_seed(t)
    gmf, gcf = torch.randn(b * h, 4, 8, generator=g), torch.randn(b * h, 4, 4, generator=g)
    leaves = [x.detach().requires_grad_(True) for x in dev]
    read, mT, cT = mixer.bayes_mixer_core(*leaves, heads=h)
    assert calls and _small_kernels(b, t, h), "the small-batch kernels were not used"
    outs, seeds = [read], [g_read.to(cuda_device).view_as(read)]
    if final_grads:
        outs, seeds = [read, mT, cT], seeds + [gmf.to(cuda_device), gcf.to(cuda_device)]
    grads = torch.autograd.grad(outs, leaves, seeds)
    m0, c0 = torch.zeros(b * h, 4, 8), torch.eye(4).expand(b * h, 4, 4)  # (other priors: test_gpu_mixer_row_abi.py)
    e_read, e_mT, e_cT, e_grads = O.mixer_grads(*views, h, m0.double(), c0.double(), g_read,
                                                gmf if final_grads else None, gcf if final_grads else None)
    close(read.reshape(e_read.shape), e_read, "read")
    close(mT, e_mT, "mean_T")
    close(cT, e_cT, "cov_T")
    for got, want, what in zip(grads, e_grads, ("q", "k", "v", "decay", "noise")):
        _bf16_close(got, want.reshape(got.shape), what)


@pytest.mark.parametrize("b,t,h", SHAPES)
@pytest.mark.parametrize("dynamics", [True, False])
def test_readout_is_the_large_batch_kernels(cuda_device, monkeypatch, limits, b, t, h, dynamics):
    from bayes_ssm import mixer

    print(f"mixer row readout b={b} t={t} h={h} dynamics={dynamics}", flush=True)
    _, dev, _ = _inputs(b, t, h, seed=7 * t + h, device=cuda_device, pad=8)
    g = torch.Generator().manual_seed(t)
    gate, gy = (torch.randn(b, t, 8 * h, generator=g).to(torch.bfloat16).to(cuda_device) for _ in range(2))
    weight = (1 + 0.1 * torch.randn(8, generator=g)).to(torch.bfloat16).to(cuda_device)
    calls = _spy(monkeypatch, mixer._MixerReadoutFunction)

    def run(small):
        limits(small)
        assert _small_kernels(b, t, h) == small
        leaves = [x.detach().clone(memory_format=torch.preserve_format).requires_grad_(dynamics or i not in (3, 4))
                  for i, x in enumerate((*dev, gate, weight))]
        out = mixer.bayes_mixer_readout(*leaves, heads=h)
        return (*out, *torch.autograd.grad(out[0], [x for x in leaves if x.requires_grad], gy))

    got, want = run(True), run(False)
    assert len(calls) == 2, "the fused kernels were not used"
    # The two routes round in float32 differently, so that a readout may fall on the other side of a bfloat16 rounding
    # boundary: one step of it, up to 2^-7 of the value, and another when the product of the epilogue is rounded; the
    # gradients are linear in gy, which moves with the readout by up to 2^-7 of its terms.
    for i, (x, e) in enumerate(zip(got[:-1], want[:-1])):
        if x.dtype == torch.float32:
            close(x, e, f"output {i}")
        else:
            scale = 2 ** -7 * e.float().abs().max().item() if i >= 3 else 0.0
            torch.testing.assert_close(x.float(), e.float(), rtol=2 ** -6, atol=scale + 2e-4)
    # The weight gradient sums b t h terms of both signs in another order, and is rounded to bfloat16 (a step is up to 2^-7
    # of the value).
    torch.testing.assert_close(got[-1].float(), want[-1].float(), rtol=2 ** -7, atol=2e-6 * b * t * h)


@pytest.mark.parametrize("b,t,h", SHAPES)
@pytest.mark.parametrize("with_bias", [False, True])
def test_block_is_the_large_batch_kernels(cuda_device, monkeypatch, limits, b, t, h, with_bias):
    from bayes_ssm import mixer
    from tests.test_gpu_block import _inputs as block_inputs
    from tests.test_gpu_block import _leaves

    print(f"mixer row block b={b} t={t} h={h} bias={with_bias}", flush=True)
    projected, weight, norm_w, aux_bias, gout = block_inputs(b, t, h, seed=t + h, device=cuda_device)
    calls = _spy(monkeypatch, mixer._MixerBlockFunction)

    def run(small):
        limits(small)
        assert _small_kernels(b, t, h) == small
        leaves, view, bias = _leaves(projected, weight, norm_w, aux_bias if with_bias else None, False)
        out = mixer.bayes_mixer_block(view, leaves[1], leaves[2], heads=h, aux_bias=bias)
        return (*out, *torch.autograd.grad(out[0], leaves + ([bias] if with_bias else []), gout))

    got, want = run(True), run(False)
    assert len(calls) == 2, "the block kernels were not used"
    # As in the readout's test; the projection's gradient passes the filter's bfloat16 gradient besides.
    torch.testing.assert_close(got[0].float(), want[0].float(), rtol=2 ** -6, atol=2e-4)
    close(got[1], want[1], "mean_T")
    close(got[2], want[2], "cov_T")
    for x, e in zip(got[3:], want[3:]):
        torch.testing.assert_close(x.float(), e.float(), rtol=2 ** -6, atol=2 ** -7 * e.float().abs().max().item())
