"""bfloat16 and float8 calls on slices of a batch: at T not a multiple of 4 the
rows of such a slice start at other offsets from a 16-byte boundary in each
stream.  Such calls are taken, with the results of the same values on aligned
buffers (parity tolerance, and a step of the narrow type in its gradients)."""
from __future__ import annotations

import pytest
import torch

from oracle import bssm_oracle as O

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn}


def _call(streams, gy):
    from bayes_ssm.fused_cuda import fused_diagonal_bayesian

    leaves = [x.detach().requires_grad_(True) for x in streams]
    n, _, d = leaves[0].shape
    m0, c0 = torch.zeros(n, d, 8, device=gy.device), torch.eye(d, device=gy.device).expand(n, d, d).contiguous()
    out, mT, cT = fused_diagonal_bayesian(*leaves, m0, c0, chunk_length=64, denominator_floor=1e-6)
    return out, mT, cT, torch.autograd.grad(out, leaves, gy)


@pytest.mark.parametrize("first", [1, 2, 3, 4])
@pytest.mark.parametrize("t", [508, 509, 510, 511])
@pytest.mark.parametrize("dtype", ["bf16", "e4m3"])
def test_batch_slice(cuda_device, dtype, t, first):
    print(f"narrow slice {dtype} t={t} first={first}", flush=True)
    k, v, q, d, p, r, *_ = O.make_inputs(9, t, 4, seed=t)
    narrow = DTYPES[dtype]
    whole = [x.to(cuda_device) for x in (k.to(narrow), v.to(narrow), q.to(narrow), d, p, r)]
    part = [x[first:] for x in whole]
    gy = torch.randn(9 - first, t, 8, generator=torch.Generator().manual_seed(t)).to(cuda_device)
    got = _call(part, gy)
    # The same values on buffers of their own, which are aligned.
    want = _call([x.clone() for x in part], gy)
    for x, e in zip((*got[:3], *got[3][3:]), (*want[:3], *want[3][3:])):
        torch.testing.assert_close(x, e, rtol=1e-5, atol=1e-4)
    # One step of the narrow type (up to 2^-7 of the value with 8 significant bits, 2^-3 with 4), where the two routes'
    # float32 gradients round to different sides.
    rtol, atol = (2 ** -7, 2e-4) if dtype == "bf16" else (2 ** -3, 2 ** -9)
    for x, e in zip(got[3][:3], want[3][:3]):
        assert x.dtype == e.dtype == narrow
        torch.testing.assert_close(x.float(), e.float(), rtol=rtol, atol=atol)
