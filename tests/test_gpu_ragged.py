"""Sequence lengths that are not a multiple of the kernels' pieces, chunks and tiles.

Rows then start off a 16-byte boundary, the last piece of a row straddles its
end, and the last chunk of the backward is filled up with neutral tokens
(k = q = v = gy = 0, d = 1, p = 0).  Every kernel that takes such a T is
compared with the float64 oracle at the parity tolerance (1e-5 relative,
1e-4 absolute); N leaves idle slots in the last wave, and all rows are
compared, so a store past a row's end shows in its neighbour.
"""
from __future__ import annotations

import pytest
import torch

from oracle import bssm_oracle as O
from tests._layouts import LAYOUTS, layout
from tests.test_gpu_floor import NAMES
from tests.test_gpu_parity import ABIS, _case, _fixed_dynamics, _oracle_forward, close

pytestmark = pytest.mark.gpu

# One token; around the 4-token pieces, the 8-token chunks and the 16-token tiles.
TIMES = [1, 3, 6, 7, 9, 13, 15, 17, 23, 30, 33, 51]
CHUNK = {1: 16, 2: 8, 4: 8, 8: 8}


def _ext(d):
    from bayes_ssm import fused_cuda

    return fused_cuda._load_extension(d)


def _run(d, dev, abi, final_grads):
    name, fixed, nout = abi
    ext = _ext(d)
    args = (dev["k"], dev["v"], dev["q"], dev["d"], dev["p"], dev["r"], dev["m0"], dev["c0"])
    y, mT, cT, bm, bc = (ext.forward_chunked_fixed if fixed else ext.forward_chunked)(*args, CHUNK[d], 1e-6)
    gmf, gcf = (dev["gmf"], dev["gcf"]) if final_grads else (None, None)
    grads = ext._backward("bssm_" + name, fixed, nout, *args, bm, bc, (), dev["gy"], gmf, gcf, CHUNK[d], 1e-6)
    torch.cuda.synchronize()
    return (y, mT, cT, bm, bc), grads


def _check(cpu, outs, grads, abi, chunk, final_grads):
    name, fixed, nout = abi
    ref = _fixed_dynamics(cpu) if fixed else cpu
    f64 = {k: x.double() for k, x in ref.items()}
    core = [f64[k] for k in ("k", "v", "q", "d", "p", "r", "m0", "c0")]
    ey, em, ec, eg = O.diagonal_grads(*core, f64["gy"], f64["gmf"] if final_grads else None,
                                      f64["gcf"] if final_grads else None)
    ebm, ebc = O.checkpoints(*core, chunk, 1e-6)
    for got, want, what in zip(outs, (ey, em, ec, ebm, ebc), ("y", "mean_T", "cov_T", "bmean", "bcov")):
        close(got, want, what)
    assert len(grads) == nout
    for g, e, what in zip(grads, eg, NAMES):
        if fixed and what in ("gd", "gp", "gr"):
            assert torch.count_nonzero(g) == 0, what
        else:
            close(g, e, what)


@pytest.mark.parametrize("t", TIMES)
@pytest.mark.parametrize("final_grads", [False, True])
@pytest.mark.parametrize("abi", ABIS, ids=[a[0] for a in ABIS])
@pytest.mark.parametrize("name", list(LAYOUTS))
def test_d4_matches_oracle(cuda_device, name, abi, final_grads, t):
    print(f"ragged D4 {name} {abi[0]} final_grads={final_grads} t={t}", flush=True)
    cpu, dev = _case(21, t, 4, seed=900 + t, device=cuda_device)
    with layout(name):
        outs, grads = _run(4, dev, abi, final_grads)
    _check(cpu, outs, grads, abi, 8, final_grads)


@pytest.mark.parametrize("t", TIMES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("name", ["split", "quad"])
def test_d4_narrow_is_the_float32_kernel_on_the_widened_values(cuda_device, name, dtype, t):
    """Outputs and float32 gradients bit for bit, the narrow gradients those rounded (as torch casts them)."""
    from bayes_ssm.fused_cuda import fused_diagonal_bayesian

    print(f"ragged D4 narrow {name} {dtype} t={t}", flush=True)
    cpu, dev = _case(21, t, 4, seed=950 + t, device=cuda_device)
    narrow = [dev[x].to(dtype) for x in ("k", "v", "q")]
    results = []
    with layout(name):
        for wide in (False, True):
            kvq = [x.float() if wide else x.clone() for x in narrow]
            leaves = [x.detach().requires_grad_(True) for x in (*kvq, dev["d"], dev["p"], dev["r"])]
            out = fused_diagonal_bayesian(*leaves, dev["m0"], dev["c0"], chunk_length=64, denominator_floor=1e-6)
            grads = torch.autograd.grad([out[0], out[1]], leaves, [dev["gy"], dev["gmf"]])
            results.append((out, grads))
    torch.cuda.synchronize()
    (out, grads), (eout, egrads) = results
    for a, b in zip(out, eout):
        assert torch.equal(a, b)
    for i, (a, b) in enumerate(zip(grads, egrads)):
        assert torch.equal(a.float(), b.to(a.dtype).float()), i


@pytest.mark.parametrize("t", TIMES + [63, 65, 97])
@pytest.mark.parametrize("final_grads", [False, True])
@pytest.mark.parametrize("abi", ABIS, ids=[a[0] for a in ABIS])
@pytest.mark.parametrize("d", [1, 2, 8])
def test_other_dims_match_oracle(cuda_device, d, abi, final_grads, t):
    """The dedicated kernels; fixed dynamics with final-state gradients take the generic backward."""
    print(f"ragged D{d} {abi[0]} final_grads={final_grads} t={t}", flush=True)
    cpu, dev = _case(21, t, d, seed=970 + t + d, device=cuda_device)
    outs, grads = _run(d, dev, abi, final_grads)
    _check(cpu, outs, grads, abi, CHUNK[d], final_grads)


@pytest.mark.parametrize("t", [1, 7, 18, 33])
@pytest.mark.parametrize("chunk", [1, 3, 5, 64])
@pytest.mark.parametrize("d", [1, 2, 4, 8])
def test_generic_kernels_match_oracle(cuda_device, monkeypatch, d, chunk, t):
    """Checkpoint chunks the dedicated backwards do not take, on streams that start 4 bytes off a 16-byte boundary."""
    print(f"ragged generic D{d} chunk={chunk} t={t}", flush=True)
    cpu, dev = _case(21, t, d, seed=990 + t + d, device=cuda_device)
    for x in ("k", "v", "q", "d", "p", "r", "gy"):
        buf = torch.full((dev[x].numel() + 9,), float("nan"), device=cuda_device)
        buf[1:1 + dev[x].numel()] = dev[x].flatten()
        dev[x] = buf[1:1 + dev[x].numel()].view(dev[x].shape)
    monkeypatch.setitem(CHUNK, d, chunk)
    abi = ("backward_chunked", False, 8)
    outs, grads = _run(d, dev, abi, True)
    _check(cpu, outs, grads, abi, chunk, True)


@pytest.mark.parametrize("t", [1, 3, 7, 9, 17, 30, 33])
@pytest.mark.parametrize("d", [2, 4, 8])
@pytest.mark.parametrize("name", ["row", "quad"])
def test_rotation_matches_oracle(cuda_device, name, d, t):
    from bayes_ssm import _hip
    from tests.test_gpu_rotation import _case as rotation_case
    from tests.test_gpu_rotation import _run as run_rotation

    print(f"ragged rotation {name} D{d} t={t}", flush=True)
    ins, gy, gmf, gcf = rotation_case(21, t, d, seed=40 * d + t)
    with layout(name):
        y, mT, cT, _, _, grads = run_rotation(ins, gy, gmf, gcf, _hip.load().bssm_rotation_checkpoint(d), cuda_device)
    leaves = [x.double().requires_grad_(True) for x in ins]
    ey, em, ec = O.run_rotation(*leaves, 1e-6)
    loss = (ey * gy.double()).sum() + (em * gmf.double()).sum() + (ec * gcf.double()).sum()
    for got, want, what in zip((y, mT, cT, *grads), (ey, em, ec, *torch.autograd.grad(loss, leaves)),
                               ("y", "mean_T", "cov_T", "gk", "gv", "gq", "g_radii", "g_angles", "g_process",
                                "g_observation", "gm0", "gc0")):
        close(got, want, what)
