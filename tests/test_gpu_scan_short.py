"""The static scan's two families of kernels, a wave per token for short sequences and a workgroup per 64 tokens: either
side of the rule that chooses one, over batches that fill the GPU and that do not, exact and padded key dimensions.
Forward, final state and all gradients against the float64 oracle at the parity tolerance (1e-5 relative, 1e-4
absolute)."""
from __future__ import annotations

import pytest
import torch

import bayes_ssm
from oracle import bssm_oracle as O
from tests.test_gpu_parity import close

pytestmark = pytest.mark.gpu

SHAPES = [
    # A wave per token, both ways; the last five backward only.
    (3, 1, 1, 1), (2, 3, 2, 3), (2, 2, 3, 9), (3, 5, 4, 8), (2, 4, 5, 17), (3, 6, 8, 8), (2, 9, 8, 64), (1, 14, 7, 64),
    (2, 16, 16, 16), (3, 33, 16, 32), (1, 28, 12, 64), (1, 80, 16, 64), (700, 2, 2, 4), (600, 4, 8, 16),
    (400, 8, 16, 64), (2, 4, 3, 5), (3, 8, 8, 8), (1, 40, 12, 64), (1, 90, 16, 64), (300, 10, 16, 16),
    # A workgroup per 64 tokens.
    (2, 30, 1, 8), (2, 41, 4, 16), (2, 60, 8, 33), (1, 64, 13, 4), (700, 6, 4, 8), (300, 14, 16, 16), (40, 65, 16, 32),
    (20, 130, 16, 64),
]


@pytest.mark.parametrize("b,t,d,m", SHAPES)
@pytest.mark.parametrize("with_final", [False, True])
def test_matches_oracle(cuda_device, b, t, d, m, with_final):
    print(f"scan short b={b} t={t} d={d} m={m} final={with_final}", flush=True)
    k, v, q, r = O.make_scan_inputs(b, t, d, m, seed=t + d)
    g = torch.Generator().manual_seed(m)
    a = torch.randn(b, d, d, generator=g) / d ** 0.5
    c0 = a @ a.transpose(-1, -2) + 0.5 * torch.eye(d)
    m0 = torch.randn(b, d, m, generator=g)
    gy, gm, gc = (torch.randn(*s, generator=g) for s in ((b, t, m), (b, d, m), (b, d, d)))
    leaves = [x.to(cuda_device).requires_grad_(True) for x in (k, v, q, r, m0, c0)]
    out = bayes_ssm.associative_static_bayesian_cuda(
        leaves[0], leaves[1], leaves[2], observation_variances=leaves[3], initial_mean=leaves[4],
        initial_covariance=leaves[5])
    el = [x.double().requires_grad_(True) for x in (k, v, q, r, m0, c0)]
    expected = O.associative_static(*el)
    n = 3 if with_final else 1
    torch.autograd.backward(out[:n], [x.to(cuda_device) for x in (gy, gm, gc)][:n])
    torch.autograd.backward(expected[:n], [x.double() for x in (gy, gm, gc)][:n])
    for name, x, e in zip(("y", "mean", "cov"), out, expected):
        close(x, e, name)
    # The gradients of k and v are sums divided by r, that of r is one divided by r^2 whose terms cancel (r reaches 1e-2
    # here): the parity tolerance is that of the sums.
    r64 = el[3].detach().unsqueeze(-1)
    scale = {"k": r64, "v": r64, "r": el[3].detach() ** 2}
    for name, x, e in zip(("k", "v", "q", "r", "mean0", "cov0"), leaves, el):
        w = scale.get(name, torch.ones((), dtype=torch.float64))
        close(x.grad.double().cpu() * w, e.grad * w, "grad " + name)


def test_token_that_is_not_finite_stays_in_its_row(cuda_device):
    k, v, q, r = (x.to(cuda_device) for x in O.make_scan_inputs(3, 12, 16, 16, seed=9))
    clean = bayes_ssm.associative_static_bayesian_cuda(k, v, q, observation_variances=r)[0]
    bad = v.clone()
    bad[1, 5, 3] = float("nan")
    y = bayes_ssm.associative_static_bayesian_cuda(k, bad, q, observation_variances=r)[0]
    hit = torch.zeros_like(y, dtype=torch.bool)
    hit[1, 5:, 3] = True
    assert torch.isnan(y[hit]).all()
    assert torch.equal(y[~hit], clean[~hit])
