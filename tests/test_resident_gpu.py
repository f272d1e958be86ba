"""The resident stage kernel (lattices of many tiles, tabulated EoS) against
the oracle: sizes a little above the line from which it runs, rows that are no
multiple of a wave, strips that do not divide y, 2+1D and 3+1D, with and
without bulk.  FP64 at the parity bar; the mixed forms at their accuracy
criterion, 1e-4 in e and in u^mu/u^tau.  The order in which waves take tiles
differs from run to run, the results may not."""
import numpy as np
import pytest

import gpuvh
from parity import PI_FIELDS, U_FIELDS, Case, compare, run_both

pytestmark = pytest.mark.gpu


def state(case):
    x = (np.arange(case.nx) - case.nx / 2)[:, None, None] / case.nx
    y = (np.arange(case.ny) - case.ny / 2)[None, :, None] / case.ny
    z = (np.arange(case.nz) - case.nz / 2)[None, None, :] / case.nz
    e = 40.0 * np.exp(-6 * (x * x + y * y) - 2 * z * z)
    e = e * (1 + 0.2 * np.sin(40 * x) * np.cos(31 * y)) + 1e-2 + 0 * z
    zero = np.zeros(e.shape)
    ux, uy = 0.3 * x + 0 * e, 0.2 * y + 0 * e
    un = 0.1 * z + 0 * e
    ut = np.sqrt(1 + ux ** 2 + uy ** 2 + (case.t0 * un) ** 2)
    return e, case.pressure(e), ut, ux, uy, un, [zero] * 10, zero


@pytest.mark.parametrize("nx,ny,nz,bulk", [(101, 101, 65, True), (333, 37, 55, True),
                                           (65, 161, 67, False), (815, 815, 1, True),
                                           (1201, 547, 1, False)])
def test_resident_against_oracle(nx, ny, nz, bulk):
    case = Case(nx, ny, nz, 0.2, 0.2, 0.01, 0.5, 0.16, bulk=bulk, eos=gpuvh.EOS_TABLE,
                zeta_tpeak=0.16 / gpuvh.HBARC)
    st = state(case)
    orc, ctx = run_both(case, st, 2)
    fields = [gpuvh.E] + U_FIELDS + PI_FIELDS + ([gpuvh.PI] if bulk else [])
    errs = compare(orc, ctx, fields, tau=0.52)
    assert max(errs.values()) <= 1e-10, errs
    first = [ctx.get(f) for f in fields]
    ctx.set_initial_state(case.t0, *st)
    ctx.steps(case.t0, 0, 2)
    for f, a in zip(fields, first):
        assert np.array_equal(ctx.get(f), a), gpuvh.FIELD_NAMES[f]
    e, ut = orc.get(gpuvh.E), orc.get(gpuvh.UT)
    for precision in (gpuvh.MIXED, gpuvh.MIXED_F64_ROOTS):
        m = case.context(precision)
        m.set_initial_state(case.t0, *st)
        m.steps(case.t0, 0, 2)
        assert np.max(np.abs(m.get(gpuvh.E) - e) / e) <= 1e-4
        for f in U_FIELDS:
            assert np.max(np.abs(m.get(f) - orc.get(f)) / ut) <= 1e-4
        m.close()
