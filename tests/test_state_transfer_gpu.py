"""Initial state and field reads: every conserved and primitive field on the
ghosted grid against numpy, bit by bit, for one-point axes, odd sizes and a
block's last partial wave; also after steps and a second initial state on the
same context, and reads between steps that leave the evolution alone."""
import numpy as np
import pytest

import gpuvh

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(11)


def primitives(shape, bulk, with_pi):
    e = 10.0 + 0.01 * RNG.standard_normal(shape)
    p = e / 3 + RNG.uniform(-0.01, 0.01, shape)
    ux, uy, un = (0.001 * RNG.standard_normal(shape) for _ in range(3))
    ut = np.sqrt(1 + ux ** 2 + uy ** 2 + 0.25 * un ** 2)
    pi = [0.01 * RNG.standard_normal(shape) for _ in range(10)] if with_pi else None
    Pi = 0.01 * RNG.standard_normal(shape) if with_pi else None
    return e, p, ut, ux, uy, un, pi, Pi


def ghosted(a):
    """Zero-gradient face ghosts, zero edges and corners."""
    nx, ny, nz = a.shape
    out = np.zeros((nx + 4, ny + 4, nz + 4))
    full = np.pad(a, 2, mode="edge")
    i, j, k = np.ogrid[:nx + 4, :ny + 4, :nz + 4]
    outside = [((x < 2) | (x >= n + 2)).astype(int) for x, n in ((i, nx), (j, ny), (k, nz))]
    face = sum(outside) <= 1
    out[face] = full[face]
    return out


def expected(st, bulk, mixed):
    e, p, ut, ux, uy, un, pi, Pi = st
    zero = np.zeros(e.shape)
    pi = pi or [zero] * 10
    Pi = Pi if bulk and Pi is not None else zero
    P = p + Pi
    T = [(e + P) * ut * ut - P + pi[0]] + [(e + P) * ut * u + pi[1 + m]
                                           for m, u in enumerate((ux, uy, un))]
    kept = [np.float32(a).astype(np.float64) if mixed else a for a in pi + [Pi]]
    return dict(zip(range(gpuvh.TTT, gpuvh.UN + 1), T + kept + [e, p, ut, ux, uy, un]))


@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 1, 1), (5, 4, 3), (17, 13, 1), (61, 33, 9)])
@pytest.mark.parametrize("precision", [gpuvh.FP64, gpuvh.MIXED])
@pytest.mark.parametrize("bulk", [True, False])
def test_state_and_reads(shape, precision, bulk):
    L = gpuvh.lattice(*shape, 0.1, 0.1, 0.1, 0.005)
    ctx = gpuvh.Context(L, gpuvh.hydro(0.5, 0.2), gpuvh.options(gpuvh.EOS_TABLE, bulk, precision))
    for with_pi in (True, False):
        st = primitives(shape, bulk, with_pi)
        ctx.set_initial_state(0.5, *st)
        want = expected(st, bulk, precision != gpuvh.FP64)
        for f, a in want.items():
            assert np.array_equal(ctx.get(f), a), gpuvh.FIELD_NAMES[f]
            assert np.array_equal(ctx.get(f, ghosted=True), ghosted(a)), gpuvh.FIELD_NAMES[f]
        for m, f in enumerate((gpuvh.UTP, gpuvh.UXP, gpuvh.UYP, gpuvh.UNP)):
            prev = np.zeros(tuple(n + 4 for n in shape))
            prev[2:-2, 2:-2, 2:-2] = st[2 + m]
            assert np.array_equal(ctx.get(f, ghosted=True), prev), gpuvh.FIELD_NAMES[f]
        ctx.steps(0.5, 0, 3)  # the next round starts on a used context
    ctx.close()


@pytest.mark.parametrize("precision", [gpuvh.FP64, gpuvh.MIXED])
def test_reads_between_steps(precision):
    shape = (33, 21, 5)
    L = gpuvh.lattice(*shape, 0.1, 0.1, 0.1, 0.005)
    st = primitives(shape, True, False)
    out = []
    for reads in (False, True):
        ctx = gpuvh.Context(L, gpuvh.hydro(0.5, 0.2), gpuvh.options(gpuvh.EOS_TABLE, True, precision))
        ctx.set_initial_state(0.5, *st)
        for n in range(4):
            ctx.step(0.5 + 0.005 * n)
            if reads:
                for f in (gpuvh.E, gpuvh.PIXX, gpuvh.UX):
                    ctx.get(f)
                    ctx.get(f, ghosted=True)
        out.append([ctx.get(f, ghosted=True) for f in range(gpuvh.TTT, gpuvh.UNP + 1)])
        ctx.close()
    for f, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b, equal_nan=True), gpuvh.FIELD_NAMES[f]
