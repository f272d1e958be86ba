"""Results around the sizes at which a read changes its route: 64 KiB (packed
into pinned memory), 1 MiB (pinned slots emptied by threads) and the eight
slots' turn; pageable and pinned destinations; two contexts read by two threads
at once."""
import ctypes as C
import threading

import numpy as np
import pytest

import gpuvh

pytestmark = pytest.mark.gpu

# interior cells around 8192 (64 KiB), 131072 (1 MiB) and 9 MiB
SHAPES = [(8191, 1, 1), (8192, 1, 1), (8193, 1, 1), (131071, 1, 1), (1024, 128, 1), (131073, 1, 1),
          (523, 251, 9)]


def context(shape, precision):
    L = gpuvh.lattice(*shape, 0.1, 0.1, 0.1, 0.01)
    ctx = gpuvh.Context(L, gpuvh.hydro(0.5, 0.2), gpuvh.options(gpuvh.EOS_CONFORMAL, True, precision))
    n = int(np.prod(shape))
    e = (1.0 + np.arange(n, dtype=np.float64)).reshape(shape, order="F")
    one, zero = np.ones(shape), np.zeros(shape)
    Pi = (0.25 * np.arange(n) % 97).reshape(shape, order="F")
    ctx.set_initial_state(0.5, e, e / 3, one, zero, zero, zero, None, Pi)
    return ctx, e, Pi


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision", [gpuvh.FP64, gpuvh.MIXED])
def test_sizes(shape, precision):
    ctx, e, Pi = context(shape, precision)
    for _ in range(2):
        assert np.array_equal(ctx.get(gpuvh.E), e)
        assert np.array_equal(ctx.get(gpuvh.PI), Pi)
        assert np.array_equal(ctx.get(gpuvh.E, ghosted=True)[2:-2, 2:-2, 2:-2], e)
    ctx.close()


def test_pinned_destination():
    ctx, e, _ = context((523, 251, 3), gpuvh.FP64)
    hip = C.CDLL("libamdhip64.so.7")
    p = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), C.c_size_t(e.nbytes), C.c_uint(0)) == 0
    out = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (e.size,))
    assert gpuvh.lib().gvh_get_field(ctx.h, gpuvh.E, 0, gpuvh._ptr(out)) == 0
    assert np.array_equal(out, e.ravel(order="F"))
    ctx.close()
    assert hip.hipHostFree(p) == 0


def test_two_threads():
    made = [context((523, 251, 9), gpuvh.FP64), context((401, 333, 7), gpuvh.MIXED)]
    bad = []

    def read(ctx, e):
        for _ in range(5):
            if not np.array_equal(ctx.get(gpuvh.E), e):
                bad.append(1)

    threads = [threading.Thread(target=read, args=m[:2]) for m in made]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
