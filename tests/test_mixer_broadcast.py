"""Mixer projections whose rows overlap (broadcast over time) cannot be addressed by the kernels: the op chain takes
them."""
from __future__ import annotations

import pytest
import torch

from bayes_ssm import mixer
from oracle import bssm_oracle as O


def test_overlapping_rows_are_not_addressable():
    base = torch.zeros(2, 1, 64, dtype=torch.bfloat16)
    assert mixer._row_stride(base.expand(2, 1, 64), 1) == 64
    assert mixer._row_stride(torch.zeros(1, 1, 64, dtype=torch.bfloat16).expand(1, 7, 64), 7) is None
    assert mixer._row_stride(torch.zeros(200, dtype=torch.bfloat16).as_strided((1, 7, 64), (56, 8, 1)), 7) is None


@pytest.mark.gpu
@pytest.mark.parametrize("t,h", [(7, 8), (511, 16), (8, 12)])
def test_projections_broadcast_over_time(cuda_device, t, h):
    """Decay logits and noise of one row for all tokens (row stride 0): the results of the written-out rows."""
    views, _ = O.make_mixer_inputs(2, t, h, seed=t)
    q, k, v, d, n = [x.contiguous().to(cuda_device) for x in views]
    d, n = d[:1, :1].expand(2, t, -1), n[:1, :1].expand(2, t, -1)
    got = mixer.bayes_mixer_core(q, k, v, d, n, heads=h)
    want = mixer.bayes_mixer_core(q, k, v, d.contiguous(), n.contiguous(), heads=h)
    for x, e in zip(got, want):
        torch.testing.assert_close(x, e, rtol=1e-5, atol=1e-4)
