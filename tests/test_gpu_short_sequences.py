"""Either side of the rules that choose between kernels by the number of sequences and a last chunk or tile that is not
whole: D = 1 backward (filled up, or generic), D = 4 backward (row or rotated layout), D = 8 forward of less than a tile.
Against the float64 oracle at the parity tolerance; N leaves idle slots in the last wave."""
from __future__ import annotations

import pytest

from tests.test_gpu_parity import ABIS, _case
from tests.test_gpu_ragged import CHUNK, _check, _run

pytestmark = pytest.mark.gpu

CASES = [(1, n, t) for n, t in ((21, 5), (21, 6), (6143, 20), (6147, 20), (12290, 28), (12290, 30), (6147, 36))]
CASES += [(4, n, t) for n, t in ((21, 4), (2047, 8), (2053, 8), (4095, 20), (4099, 20), (4099, 36), (4099, 28))]
CASES += [(8, n, t) for n, t in ((4095, 12), (4099, 12), (4099, 13), (8195, 8))]


@pytest.mark.parametrize("d,n,t", CASES)
@pytest.mark.parametrize("final_grads", [False, True])
def test_matches_oracle(cuda_device, d, n, t, final_grads):
    print(f"short sequences D{d} n={n} t={t} final_grads={final_grads}", flush=True)
    cpu, dev = _case(n, t, d, seed=600 + t, device=cuda_device)
    outs, grads = _run(d, dev, ABIS[0], final_grads)
    _check(cpu, outs, grads, ABIS[0], CHUNK[d], final_grads)


@pytest.mark.parametrize("t", [4, 8, 12, 20])
@pytest.mark.parametrize("final_grads", [False, True])
@pytest.mark.parametrize("abi", ABIS, ids=[a[0] for a in ABIS])
def test_d2_whole_pieces(cuda_device, abi, final_grads, t):
    """T a multiple of 4 runs the D = 2 backward's pieces as they are, fixed dynamics with final-state gradients too."""
    print(f"short sequences D2 {abi[0]} t={t} final_grads={final_grads}", flush=True)
    cpu, dev = _case(21, t, 2, seed=650 + t, device=cuda_device)
    outs, grads = _run(2, dev, abi, final_grads)
    _check(cpu, outs, grads, abi, CHUNK[2], final_grads)
