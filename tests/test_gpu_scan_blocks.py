"""The static scan's 64-token workgroups: sequences that end inside, at and
past a block, odd and padded key dimensions, value columns that do not divide
over the waves.  Forward, final state and all gradients against the float64
oracle at the parity tolerance (1e-5 relative, 1e-4 absolute)."""
from __future__ import annotations

import pytest
import torch

import bayes_ssm
from oracle import bssm_oracle as O
from tests.test_gpu_parity import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,d,m,with_final", [
    (2, 1, 16, 16, True), (1, 2, 8, 4, True), (2, 63, 4, 4, True), (3, 64, 8, 12, True), (2, 65, 16, 32, True),
    (1, 127, 16, 4, False), (2, 128, 2, 3, True), (1, 129, 1, 64, True), (2, 191, 3, 5, True),
    (1, 192, 12, 16, True), (1, 193, 16, 64, True), (2, 320, 7, 1, False), (1, 700, 16, 17, True),
    (1, 1500, 4, 8, True)])
def test_scan_blocks(cuda_device, b, t, d, m, with_final):
    print(f"scan blocks b={b} t={t} d={d} m={m} final={with_final}", flush=True)
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
    for name, x, e in zip(("k", "v", "q", "r", "mean0", "cov0"), leaves, el):
        close(x.grad, e.grad, "grad " + name)


def test_scan_token_that_is_not_finite_stays_in_its_row(cuda_device):
    """A NaN key reaches the tokens from its own on, in its batch row only."""
    k, v, q, r = (x.to(cuda_device) for x in O.make_scan_inputs(3, 150, 8, 8, seed=9))
    clean = bayes_ssm.associative_static_bayesian_cuda(k, v, q, observation_variances=r)[0]
    bad = v.clone()
    bad[1, 70, 3] = float("nan")
    y = bayes_ssm.associative_static_bayesian_cuda(k, bad, q, observation_variances=r)[0]
    hit = torch.zeros_like(y, dtype=torch.bool)
    hit[1, 70:, 3] = True
    assert torch.isnan(y[hit]).all()
    assert torch.equal(y[~hit], clean[~hit])
