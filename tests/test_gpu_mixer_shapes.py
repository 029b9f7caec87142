"""The mixer's fused kernels off whole tiles: heads a multiple of 4, any T.

The last wave of a batch row holds 4, 8 or 12 heads, rows end inside pieces,
chunks and tiles.  Against the float64 oracle at the parity tolerance (1e-5
relative, 1e-4 absolute; bfloat16 gradients within their rounding) and bit for
bit against the whole-tile kernels on padded inputs, with the kernels' route
asserted; values that the op chain refuses are still refused.
"""
from __future__ import annotations

import pytest
import torch

from oracle import bssm_oracle as O
from tests.test_gpu_parity import close

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 4), (2, 3, 8), (1, 7, 12), (2, 17, 16), (3, 30, 20), (1, 33, 64), (2, 24, 24), (1, 61, 36)]


def _inputs(b, t, h, seed, device, pad=0):
    views, g_read = O.make_mixer_inputs(b, t, h, seed=seed, ld_pad=pad)
    base = views[0]._base.to(device)
    dev = [torch.as_strided(base, x.shape, x.stride(), x.storage_offset()) for x in views]
    return views, dev, g_read


def _spy(monkeypatch, cls):
    calls = []
    orig = cls.apply
    monkeypatch.setattr(cls, "apply", staticmethod(lambda *a: calls.append(1) or orig(*a)))
    return calls


def _bf16_close(got, want, what):
    """Within one bfloat16 rounding (2^-8 of the value) and the parity tolerance."""
    torch.testing.assert_close(got.double().cpu(), want.double().cpu(), rtol=2 ** -8, atol=2e-4,
                               msg=lambda m: f"{what}: {m}")


@pytest.mark.parametrize("b,t,h", SHAPES)
@pytest.mark.parametrize("final_grads", [False, True])
def test_core_matches_oracle(cuda_device, monkeypatch, b, t, h, final_grads):
    from bayes_ssm import mixer

    print(f"mixer core b={b} t={t} h={h} final_grads={final_grads}", flush=True)
    calls = _spy(monkeypatch, mixer._MixerCoreFunction)
    # A row stride that is a multiple of 8 elements (22 H + pad).
    views, dev, g_read = _inputs(b, t, h, seed=3 * t + h, device=cuda_device, pad=8)
    leaves = [x.detach().requires_grad_(True) for x in dev]
    read, mT, cT = mixer.bayes_mixer_core(*leaves, heads=h)
    assert calls, "the fused kernels were not used"
    g = torch.Generator().manual_seed(t)
    gmf, gcf = torch.randn(b * h, 4, 8, generator=g), torch.randn(b * h, 4, 4, generator=g)
    outs, seeds = [read], [g_read.to(cuda_device).view_as(read)]
    if final_grads:
        outs, seeds = [read, mT, cT], seeds + [gmf.to(cuda_device), gcf.to(cuda_device)]
    grads = torch.autograd.grad(outs, leaves, seeds)
    zero = torch.zeros(b * h, 4, 8, dtype=torch.float64)
    eye = torch.eye(4, dtype=torch.float64).expand(b * h, 4, 4).contiguous()
    e_read, e_mT, e_cT, e_grads = O.mixer_grads(*views, h, zero, eye, g_read, gmf if final_grads else None,
                                                gcf if final_grads else None)
    close(read.reshape(e_read.shape), e_read, "read")
    close(mT, e_mT, "mean_T")
    close(cT, e_cT, "cov_T")
    for got, want, what in zip(grads, e_grads, ("q", "k", "v", "decay", "noise")):
        assert got.dtype == torch.bfloat16
        _bf16_close(got, want.reshape(got.shape), what)


@pytest.fixture
def large_batch_kernels():
    """The small-batch kernels (test_gpu_mixer_row.py), which round differently, off."""
    from bayes_ssm import _hip

    lib = _hip.load()
    old = [lib.bssm_small_batch_limit(d, 0) for d in (2, 3)]
    yield
    for d, n in zip((2, 3), old):
        lib.bssm_small_batch_limit(d, n)


@pytest.mark.parametrize("b,t,h", SHAPES)
def test_readout_is_the_whole_tile_kernels(cuda_device, monkeypatch, large_batch_kernels, b, t, h):
    """Bit for bit the whole-tile kernels on inputs padded with zeros to a multiple of 16 heads and of 4 tokens: heads
    are independent, and tokens past T whose gradient is zero leave the others' results alone."""
    from bayes_ssm import mixer

    print(f"mixer readout b={b} t={t} h={h}", flush=True)
    _, dev, _ = _inputs(b, t, h, seed=11 * t + h, device=cuda_device, pad=8)
    g = torch.Generator().manual_seed(t)
    gate = torch.randn(b, t, 8 * h, generator=g).to(torch.bfloat16).to(cuda_device)
    gy = torch.randn(b, t, 8 * h, generator=g).to(torch.bfloat16).to(cuda_device)
    weight = (1 + 0.1 * torch.randn(8, generator=g)).to(torch.bfloat16).to(cuda_device)
    hp, tp = -(-h // 16) * 16, -(-t // 4) * 4

    def padded(x):
        w = x.shape[2] // h
        y = torch.zeros(b, tp, hp * w, device=cuda_device, dtype=x.dtype)
        y[:, :t, :h * w] = x
        return y

    def run(streams, heads, gout):
        leaves = [x.detach().clone(memory_format=torch.preserve_format).requires_grad_(True)
                  for x in (*streams, weight)]
        calls = _spy(monkeypatch, mixer._MixerReadoutFunction)
        out, mT, cT = mixer.bayes_mixer_readout(*leaves, heads=heads)
        assert calls, "the fused kernels were not used"
        return out, mT, cT, torch.autograd.grad(out, leaves, gout)

    out, mT, cT, grads = run((*dev, gate), h, gy)
    e_out, e_mT, e_cT, e_grads = run([padded(x) for x in (*dev, gate)], hp, padded(gy))
    assert torch.equal(out, e_out[:, :t, :8 * h])
    if t == tp:
        assert torch.equal(mT, e_mT.view(b, hp, 4, 8)[:, :h].reshape(mT.shape))
        assert torch.equal(cT, e_cT.view(b, hp, 4, 4)[:, :h].reshape(cT.shape))
    for i, (got, want) in enumerate(zip(grads[:6], e_grads[:6])):
        assert torch.equal(got, want[:, :t, :got.shape[2]]), i
    # The weight gradient sums the same terms (zeros among them) over another number of partial rows.
    torch.testing.assert_close(grads[6].float(), e_grads[6].float(), rtol=2 ** -8, atol=1e-5)


@pytest.mark.parametrize("b,t,h", SHAPES)
@pytest.mark.parametrize("with_bias", [False, True])
def test_block_is_its_stages(cuda_device, monkeypatch, b, t, h, with_bias):
    """One call per direction against the filter and the readout called apart, bit for bit; the weight gradients
    (other orders of summation) within one bfloat16 rounding of the sums."""
    from bayes_ssm import mixer
    from tests.test_gpu_block import _inputs as block_inputs
    from tests.test_gpu_block import _leaves, _staged

    print(f"mixer block b={b} t={t} h={h} bias={with_bias}", flush=True)
    projected, weight, norm_w, aux_bias, gout = block_inputs(b, t, h, seed=t + h, device=cuda_device)
    aux_bias = aux_bias if with_bias else None
    leaves, view, bias = _leaves(projected, weight, norm_w, aux_bias, False)
    calls = _spy(monkeypatch, mixer._MixerBlockFunction)
    out, mT, cT = mixer.bayes_mixer_block(view, leaves[1], leaves[2], heads=h, aux_bias=bias)
    assert calls, "the block kernels were not used"
    grads = torch.autograd.grad(out, leaves + ([bias] if with_bias else []), gout)
    e_out, e_mT, e_cT, e_grads, e_bias = _staged(projected, weight, norm_w, aux_bias, gout, h)
    e_grads = e_grads + ([e_bias] if with_bias else [])
    assert torch.equal(out, e_out) and torch.equal(mT, e_mT) and torch.equal(cT, e_cT)
    assert torch.equal(grads[0], e_grads[0])
    for got, want in zip(grads[1:], e_grads[1:]):
        torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -7, atol=2 ** -8 * want.abs().max().item())


@pytest.mark.parametrize("stream", ["q", "k", "v", "decay", "noise"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), 3e38])
def test_values_are_judged_by_the_op_chain(cuda_device, monkeypatch, stream, value):
    """A non-finite or enormous projection: the same error, or the same result, as the op chain gives."""
    from bayes_ssm import mixer

    b, t, h = 2, 19, 8
    _, dev, _ = _inputs(b, t, h, seed=5, device=cuda_device, pad=8)
    dev = [x.clone() for x in dev]
    dev[("q", "k", "v", "decay", "noise").index(stream)][1, 11, 5] = value

    def run(fused):
        with monkeypatch.context() as m:
            if not fused:
                m.setattr(mixer, "_any_shape_call", lambda *a: False)
            try:
                return mixer.bayes_mixer_core(*dev, heads=h)
            except ValueError as e:
                return str(e)

    got, want = run(True), run(False)
    if isinstance(want, str):
        assert got == want
    else:
        for a, e in zip(got, want):
            assert torch.equal(a, e)
