"""Off whole tiles, gradients of the mixer's final state alone: the gate and the norm weight, which it does not depend on,
have none, on the kernels as in the op chain (an optimizer skips such a parameter; a zero gradient it would apply)."""
from __future__ import annotations

import pytest
import torch

from tests.test_gpu_mixer_shapes import _inputs, _spy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("state", [1, 2])
@pytest.mark.parametrize("b,t,h", [(2, 7, 8), (1, 12, 20), (1, 33, 16)])
def test_readout(cuda_device, monkeypatch, b, t, h, state):
    from bayes_ssm import mixer

    print(f"unused readout b={b} t={t} h={h} state={state}", flush=True)
    _, dev, _ = _inputs(b, t, h, seed=t + h, device=cuda_device, pad=8)
    gate = torch.randn(b, t, 8 * h, device=cuda_device).to(torch.bfloat16)
    weight = torch.ones(8, device=cuda_device, dtype=torch.bfloat16)
    leaves = [x.detach().requires_grad_(True) for x in (*dev, gate, weight)]
    calls = _spy(monkeypatch, mixer._MixerReadoutFunction)
    final = mixer.bayes_mixer_readout(*leaves, heads=h)[state]
    assert calls, "the fused kernels were not used"
    grads = torch.autograd.grad(final, leaves, torch.ones_like(final), allow_unused=True)
    assert grads[5] is None and grads[6] is None
    assert all(x is not None and torch.isfinite(x).all() for x in grads[:5]) and grads[1].abs().max() > 0


@pytest.mark.parametrize("b,t,h", [(2, 7, 8), (1, 12, 20)])
def test_block(cuda_device, monkeypatch, b, t, h):
    from bayes_ssm import mixer
    from tests.test_gpu_block import _inputs as block_inputs

    print(f"unused block b={b} t={t} h={h}", flush=True)
    projected, weight, norm_w, aux_bias, _ = block_inputs(b, t, h, seed=t + h, device=cuda_device)
    leaves = [x.detach().requires_grad_(True) for x in (projected, weight, norm_w, aux_bias)]
    calls = _spy(monkeypatch, mixer._MixerBlockFunction)
    final = mixer.bayes_mixer_block(*leaves[:3], heads=h, aux_bias=leaves[3])[1]
    assert calls, "the block kernels were not used"
    grads = torch.autograd.grad(final, leaves, torch.ones_like(final), allow_unused=True)
    assert grads[2] is None
    assert all(grads[i] is not None and grads[i].abs().max() > 0 for i in (0, 1, 3))
