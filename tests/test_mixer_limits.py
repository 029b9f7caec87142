"""Which mixer calls off whole tiles go to the kernels: the sizes that the C entry points take (asked here with an empty
batch, which launches nothing); others run the op chain."""
from __future__ import annotations

import ctypes

import pytest
import torch

from bayes_ssm import _hip, mixer

F = ctypes.c_float(1e-6)
# T at and beside each limit: T * heads * 32, (T + 16) * ld * 2, checkpoint records.
CASES = [(h, ld, t + step) for h, ld in ((4, 32), (64, 22 * 64), (64, 30 * 64), (20, 30 * 20))
         for t in ((1 << 31) // (32 * h), (1 << 31) // (2 * ld) - 16, (1 << 31) // 2048 * 8 - 8, 511)
         for step in (-9, -8, -1, 0, 1, 8)]


def _entry_takes(name, t, heads, ld):
    lib = _hip.load()
    chunk = _hip.preferred_checkpoint(4) | _hip.ANY_SHAPE
    if name == "core":
        rc = [lib.bssm_mixer_forward(*[None, ld] * 5, *[None] * 7, 0, t, heads, chunk, F, None),
              lib.bssm_mixer_backward(*[None, ld] * 5, *[None] * 14, 0, t, heads, chunk, F, 0, None)]
    elif name == "readout":
        rc = [lib.bssm_mixer_gated_forward(*[None, ld] * 6, None, F, *[None] * 8, 0, t, heads, chunk, F, 0, None),
              lib.bssm_mixer_gated_backward(*[None, ld] * 6, None, F, *[None] * 17, 0, t, heads, chunk, F, 0, None)]
    else:
        rc = [lib.bssm_mixer_block_forward(None, ld, *[None] * 3, F, *[None] * 9, 0, t, heads, chunk, F, None),
              lib.bssm_mixer_block_backward(None, ld, *[None] * 4, F, *[None] * 10, ld, *[None] * 6, 0, None, None, 0,
                                            t, heads, chunk, F, None)]
    return all(r == 0 for r in rc)


@pytest.mark.parametrize("name", ["core", "readout", "block"])
@pytest.mark.parametrize("heads,ld,t", CASES)
def test_limits_are_the_entry_points(name, heads, ld, t):
    if name == "block" and ld < 30 * heads:
        pytest.skip("the block's rows hold 30 columns a head")
    assert mixer._in_limits(t, heads, ld) == _entry_takes(name, t, heads, ld)


def test_an_empty_batch_is_left_to_the_op_chain():
    """The block's weight gradients would come back unwritten from a call without work."""
    assert mixer._any_shape_call(1, 8, 7, None, None, None, 1e-6, True)
    assert not mixer._any_shape_call(0, 8, 7, None, None, None, 1e-6, True)


class _OpChain(Exception):
    pass


@pytest.mark.gpu
def test_long_calls_go_to_the_op_chain(cuda_device, monkeypatch):
    """A row of 64 heads in a fused projection just past the 32-bit offsets: the op chain, as before any T was fused."""
    def reached(*a):
        raise _OpChain

    monkeypatch.setattr(mixer, "mixer_layer_inputs", reached)
    h, t = 64, 559_241
    projected = torch.empty(1, t, 30 * h, device=cuda_device, dtype=torch.bfloat16)
    cuts = [0, 4 * h, 8 * h, 16 * h, 20 * h, 22 * h, 30 * h]
    q, k, v, d, n, gate = [projected[..., i:j] for i, j in zip(cuts, cuts[1:])]
    with pytest.raises(_OpChain):
        mixer.bayes_mixer_core(q, k, v, d, n, heads=h)
    with pytest.raises(_OpChain):
        mixer.bayes_mixer_readout(q, k, v, d, n, gate, torch.ones(8, device=cuda_device, dtype=torch.bfloat16), heads=h)
