"""Either side of the rules that choose a kernel's ragged form (a template parameter): sequence lengths that are whole
pieces but not whole chunks, or whole chunks but not whole blocks and tiles.  Against the float64 oracle at the parity
tolerance."""
from __future__ import annotations

import pytest

from tests._layouts import layout
from tests.test_gpu_parity import ABIS, _case
from tests.test_gpu_ragged import CHUNK, _check, _run

pytestmark = pytest.mark.gpu

NAMES = [a[0] for a in ABIS]


@pytest.mark.parametrize("t", [4, 12, 16, 20, 32, 36, 48, 52])
@pytest.mark.parametrize("final_grads", [False, True])
@pytest.mark.parametrize("abi", ABIS, ids=NAMES)
def test_d1(cuda_device, abi, final_grads, t):
    print(f"tail d1 {abi[0]} final_grads={final_grads} t={t}", flush=True)
    cpu, dev = _case(13, t, 1, seed=700 + t, device=cuda_device)
    outs, grads = _run(1, dev, abi, final_grads)
    _check(cpu, outs, grads, abi, CHUNK[1], final_grads)


@pytest.mark.parametrize("n,t", [(21, 8), (21, 16), (21, 24), (21, 28), (21, 40), (1030, 24), (1030, 28)])
@pytest.mark.parametrize("final_grads", [False, True])
@pytest.mark.parametrize("abi", ABIS, ids=NAMES)
@pytest.mark.parametrize("name", ["row", "split"])
def test_d4_small_batch(cuda_device, name, abi, final_grads, n, t):
    print(f"tail d4 {name} {abi[0]} final_grads={final_grads} n={n} t={t}", flush=True)
    cpu, dev = _case(n, t, 4, seed=750 + t, device=cuda_device)
    with layout(name):
        outs, grads = _run(4, dev, abi, final_grads)
    _check(cpu, outs, grads, abi, CHUNK[4], final_grads)
