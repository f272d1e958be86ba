"""Large results while every CPU is busy: a result is whole, and does not wait
for threads of the pool that have not run yet."""
import threading

import numpy as np
import pytest

import gpuvh
from parity import Case
from test_resident_gpu import state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(128, 64, 16), (128, 64, 17), (160, 128, 57)])
def test_results_under_load(nx, ny, nz):
    """One chunk, one and a part, and more than the slots."""
    case = Case(nx, ny, nz, 0.2, 0.2, 0.01, 0.5, 0.16, bulk=True, eos=gpuvh.EOS_TABLE,
                zeta_tpeak=0.16 / gpuvh.HBARC)
    st = state(case)
    ctx = case.context(gpuvh.FP64)
    ctx.set_initial_state(case.t0, *st)
    stop = threading.Event()
    a = np.ones(1 << 16)

    def spin():
        while not stop.is_set():
            np.sqrt(a)

    load = [threading.Thread(target=spin) for _ in range(32)]
    for t in load:
        t.start()
    try:
        for _ in range(5):
            assert np.array_equal(ctx.get(gpuvh.E), st[0])
            assert np.array_equal(ctx.get(gpuvh.UX), st[3])
    finally:
        stop.set()
        for t in load:
            t.join()
    ctx.close()
