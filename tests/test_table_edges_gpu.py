"""The table lookup where it leaves its branch-free range: short tables whose
first and last nodes lie inside the energy densities of the event, so that
cells and half-site states fall below the first node, between the last two
and beyond the last, in the same waves as ordinary ones.  FP64 against the
oracle at the parity bar; the mixed form at its accuracy criterion, 1e-4 in e
and in u^mu/u^tau."""
import numpy as np
import pytest

import gpuvh
from parity import PI_FIELDS, U_FIELDS, Case, compare, hotspot_state, run_both

pytestmark = pytest.mark.gpu

FULL = gpuvh.EosTable()


class Cut:
    """Nodes [k0, k1) of the full table; k0 starts an octave."""

    def __init__(self, octave, n):
        k0 = (octave - FULL.emin_exp) * FULL.per_octave
        self.e, self.p, self.cs2, self.T = (a[k0:k0 + n].copy()
                                            for a in (FULL.e, FULL.p, FULL.cs2, FULL.T))
        self.n, self.per_octave, self.emin_exp = n, FULL.per_octave, octave


def cases():
    # (first octave, nodes): within one octave, one past it, a whole number of
    # octaves and one node more, wide, and the full table
    for octave, n in ((2, 2), (2, 3), (2, 50), (2, 51), (1, 101), (1, 117)):
        yield octave, n


def gentle_state(case):
    """Seeded hotspots with e between 1.5 and 12 fm^-4: near enough to the
    tables for their linear continuations to be an equation of state."""
    e, _, ut, ux, uy, un, pi10, Pi = hotspot_state(case, seed=7, n_hot=8, amp=6.0)
    e = 1.5 + 10.5 * (e - e.min()) / (e.max() - e.min())
    return e, case.pressure(e), ut, ux, uy, un, pi10, Pi


@pytest.mark.parametrize("octave,n", cases())
@pytest.mark.parametrize("nz", [1, 5])
def test_short_tables(octave, n, nz):
    case = Case(37, 11, nz, 0.2, 0.2, 0.01, 0.5, 0.16, bulk=True, eos=gpuvh.EOS_TABLE,
                zeta_tpeak=0.16 / gpuvh.HBARC)
    case.table = Cut(octave, n)
    state = gentle_state(case)
    e0 = state[0]
    # the event does reach past both ends of the table
    assert (e0 < case.table.e[0]).any() and (e0 > case.table.e[-1]).any()
    orc, ctx = run_both(case, state, 3)
    errs = compare(orc, ctx, [gpuvh.E] + U_FIELDS + PI_FIELDS + [gpuvh.PI], tau=0.53)
    assert max(errs.values()) <= 1e-10, errs
    L = gpuvh.lattice(case.nx, case.ny, nz, case.dx, case.dx, case.dz, case.dt)
    mixed = gpuvh.Context(L, gpuvh.hydro(0.5, 0.16),
                          gpuvh.options(gpuvh.EOS_TABLE, True, gpuvh.MIXED, case.zeta_tpeak,
                                        table=case.table))
    mixed.set_initial_state(0.5, *state)
    mixed.steps(0.5, 0, 3)
    e, ut = ctx.get(gpuvh.E), ctx.get(gpuvh.UT)
    assert np.max(np.abs(mixed.get(gpuvh.E) - e) / e) <= 1e-4
    for f in U_FIELDS:
        assert np.max(np.abs(mixed.get(f) - ctx.get(f)) / ut) <= 1e-4
