"""Either side of the rules that choose a kernel's ragged form (a template parameter): sequence lengths that are whole
pieces but not whole chunks, or whole chunks but not whole blocks and tiles.  Against the float64 oracle at the parity
tolerance."""
from __future__ import annotations

import pytest

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
