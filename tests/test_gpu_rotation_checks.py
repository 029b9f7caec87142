"""The rotation forward's own value checks (D = 4 row kernel): each input with
one bad entry, at the edges of tiles, pieces and waves, raises what the check
pass of the other key dimensions raises, and clean inputs raise nothing."""
from __future__ import annotations

import importlib

import pytest
import torch

import bayes_ssm

bl = importlib.import_module("bayes_ssm.bayesian_layer")

pytestmark = pytest.mark.gpu

NAMES = ("keys", "values", "queries", "rotation_radii", "rotation_angles", "process_variances",
         "observation_variances")


def _inputs(n, t, d, device):
    g = torch.Generator().manual_seed(n + t)
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    u = lambda *s: torch.rand(*s, generator=g)  # noqa: E731
    xs = (r(n, t, d), r(n, t, 8), r(n, t, d), u(n, t, d // 2), r(n, t, d // 2), u(n, t, d // 2), 0.5 + u(n, t))
    return [x.to(device) for x in xs]


def _run(xs, d=4):
    return bayes_ssm.bayesian_layer(*xs[:3], rotation_radii=xs[3], rotation_angles=xs[4], process_variances=xs[5],
                                    observation_variances=xs[6], chunk_length=16, optimized=True)


@pytest.mark.parametrize("n,t", [(1, 1), (3, 5), (4, 16), (5, 17), (6, 31), (9, 64)])
def test_a_bad_entry_is_found(cuda_device, monkeypatch, n, t):
    passes = []
    orig = bl._device_value_stats
    monkeypatch.setattr(bl, "_device_value_stats", lambda xs: passes.append(len(xs)) or orig(xs))
    clean = _inputs(n, t, 4, cuda_device)
    zero = [x.clone() for x in clean]
    zero[5].zero_()  # a process variance of zero is allowed
    for xs in (clean, zero):
        _run(xs)
    assert not passes, "the forward made its checks itself"
    for which, name in enumerate(NAMES):
        flat = clean[which].numel()
        for at in sorted({0, flat // 2, flat - 1}):
            values = [float("nan"), float("inf"), -float("inf")]
            values += [-1e-30] if which >= 5 else []
            values += [0.0] if which == 6 else []
            for value in values:
                xs = [x.clone() for x in clean]
                xs[which].view(-1)[at] = value
                with pytest.raises(ValueError) as e:
                    _run(xs)
                kind = ("contain only finite values" if value != value or abs(value) == float("inf")
                        else "be nonnegative" if which == 5 else "be strictly positive")
                assert str(e.value) == f"{name} must {kind}"


def test_first_fault_in_order_and_other_tensors(cuda_device):
    """Several faults: the first argument's; an initial mean, which the kernel does not check, after them."""
    xs = _inputs(4, 20, 4, cuda_device)
    xs[6][2, 3] = -1.0
    xs[2][1, 7, 2] = float("nan")
    with pytest.raises(ValueError, match="queries must contain only finite values"):
        _run(xs)
    xs = _inputs(4, 20, 4, cuda_device)
    mean = torch.zeros(4, 4, 8, device=cuda_device)
    mean[3, 1, 2] = float("inf")
    with pytest.raises(ValueError, match="initial_mean must contain only finite values"):
        bayes_ssm.bayesian_layer(*xs[:3], rotation_radii=xs[3], rotation_angles=xs[4], process_variances=xs[5],
                                 observation_variances=xs[6], initial_mean=mean, chunk_length=16, optimized=True)


@pytest.mark.parametrize("d", [2, 8])
def test_other_key_dimensions_keep_the_pass(cuda_device, monkeypatch, d):
    """... and have no probe: its kernel makes no checks for them."""
    from bayes_ssm import fused_cuda

    monkeypatch.setattr(fused_cuda.RotationProbe, "__init__", lambda *a: pytest.fail("a probe was made"))
    xs = _inputs(3, 9, d, cuda_device)
    _run(xs)
    xs[6][1, 4] = 0.0
    with pytest.raises(ValueError, match="observation_variances must be strictly positive"):
        _run(xs)
