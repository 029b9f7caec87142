"""The D = M = 64 backward's four-token prediction blocks at their edges: rows
that end inside, at and past a block, keys that repeat within a block (the
block's innovations are differences then), and an initial covariance that is
not symmetric, against the one-wave kernel that other checkpoint intervals
take and predicts token by token (parity tolerance, 1e-5 relative and 1e-4
absolute)."""
from __future__ import annotations

import pytest
import torch

from tests.test_gpu_d64 import _case, close, ext  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fixed", [False, True])
@pytest.mark.parametrize("t", [1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 17, 24])
def test_blocks_match_single_tokens(ext, cuda_device, t, fixed):  # noqa: F811
    print(f"d64 blocks t={t} fixed={fixed}", flush=True)
    _, dev = _case(3, t, seed=50 + t, device=cuda_device)
    k = dev["k"].clone()
    k[1, 1::2] = k[1, :1]  # one direction again and again
    g = torch.Generator().manual_seed(t)
    c0 = dev["c0"] + 0.05 * torch.randn(3, 64, 64, generator=g).to(cuda_device)
    fwd = ext.forward_chunked_fixed if fixed else ext.forward_chunked
    bwd = ext.backward_chunked_fixed if fixed else ext.backward_chunked
    grads = []
    for chunk in (8, 5):
        args = (k, dev["v"], dev["q"], dev["d"], dev["p"], dev["r"], dev["m0"], c0)
        bm, bc = fwd(*args, chunk, 1e-6)[3:]
        grads.append(bwd(*args, bm, bc, dev["gy"], dev["gmf"], dev["gcf"], chunk, 1e-6))
    for name, a, b in zip(("gk", "gv", "gq", "gd", "gp", "gr", "gm0", "gc0"), *grads):
        close(a, b, name)
