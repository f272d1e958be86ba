"""The stage kernel of small lattices, with a wave for the sources and one for
each direction, against the oracle: single cells and rows, tiles that are not
full, both sides of the numbers of tiles up to which it runs, 2+1D and 3+1D,
every EoS.  FP64 at the parity bar; the mixed forms at their accuracy
criterion, 1e-4 in e and in u^mu/u^tau."""
import numpy as np
import pytest

import gpuvh
from parity import PI_FIELDS, U_FIELDS, Case, compare, run_both
from test_resident_gpu import state

pytestmark = pytest.mark.gpu
TABLE, WB, CONFORMAL = gpuvh.EOS_TABLE, gpuvh.EOS_WB, gpuvh.EOS_CONFORMAL


@pytest.mark.parametrize("nx,ny,nz,eos,bulk", [
    (1, 1, 1, TABLE, True), (5, 3, 1, CONFORMAL, False), (63, 1, 2, TABLE, True),
    (64, 9, 1, WB, True), (65, 7, 3, TABLE, False), (33, 21, 5, CONFORMAL, False),
    (17, 19, 9, WB, True),
    # 512 tiles and the next number of them, in FP64; 1536 and the next in FP32
    (64, 512, 1, TABLE, True), (64, 513, 1, TABLE, True), (64, 64, 8, TABLE, True),
    (64, 64, 9, WB, False), (64, 1536, 1, TABLE, False), (65, 1536, 1, CONFORMAL, False),
    (64, 64, 24, CONFORMAL, False), (64, 64, 25, TABLE, True)])
def test_split_against_oracle(nx, ny, nz, eos, bulk):
    case = Case(nx, ny, nz, 0.2, 0.2, 0.01, 0.5, 0.16, bulk=bulk, eos=eos,
                zeta_tpeak=0.16 / gpuvh.HBARC)
    st = state(case)
    orc, ctx = run_both(case, st, 2)
    fields = [gpuvh.E] + U_FIELDS + PI_FIELDS + ([gpuvh.PI] if bulk else [])
    errs = compare(orc, ctx, fields, tau=0.52)
    assert max(errs.values()) <= 1e-10, errs
    e, ut = orc.get(gpuvh.E), orc.get(gpuvh.UT)
    for precision in (gpuvh.MIXED, gpuvh.MIXED_F64_ROOTS):
        m = case.context(precision)
        m.set_initial_state(case.t0, *st)
        m.steps(case.t0, 0, 2)
        assert np.max(np.abs(m.get(gpuvh.E) - e) / e) <= 1e-4
        for f in U_FIELDS:
            assert np.max(np.abs(m.get(f) - orc.get(f)) / ut) <= 1e-4
        m.close()
