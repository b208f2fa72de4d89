"""The FP64 paths' near lists as they are built (MI355X): large and long cells, whose
atoms the build tries in runs of 64.

Two-phase against single_phase (the plain kernel, every pair): FP64 sums of some 1e3 terms in
another order, 1e-9 as for the FP64 results against the oracle."""
import pytest

import pureadsorb_amd as pa
from pureadsorb_amd import synth

pytestmark = pytest.mark.gpu
T = 298.15
FIELDS = ("mu_ex", "mu_ex_err", "K_H", "K_H_err", "q_st", "q_st_err", "ln_K_H")


def _system(guest="co2"):
    ff = synth.synthetic_forcefield(12.0, guest=guest)
    return ff, synth.co2_guest(ff) if guest == "co2" else synth.ch4_guest(ff), pa.EwaldParams(12.0, 1e-6)


# more than 64 runs, so that a wavefront tries them in two rounds; runs longer than the cell is
# wide; a skewed cell; fewer atoms than a run; no atoms at all
@pytest.mark.parametrize("cell,atoms", [((60.0, 62.0, 58.0, 90, 90, 90), 6200), ((24.1, 24.3, 260.0, 90, 90, 90), 700),
                                        ((41.0, 47.0, 43.0, 66, 104, 72), 1500), ((25.0, 25.0, 25.0, 90, 90, 90), 20),
                                        ((25.0, 25.0, 25.0, 90, 90, 90), 0)])
@pytest.mark.parametrize("guest", ["co2", "ch4"])
def test_lists_of_large_and_long_cells(cell, atoms, guest):
    ff, g, ew = _system(guest)
    fw = synth.synthetic_framework(*cell, atoms, 5, charge_sd=0.1 if guest == "co2" else 0.0)
    small = synth.synthetic_framework(26.0, 25.0, 27.0, 80, 95, 100, 130, 6, charge_sd=0.1)
    b = pa.FrameworkBatch([small, fw, small], ff, g, ew)
    kw = dict(T=T, ninsert=3 * 2_000, seed=4, nblocks=3, precision="f64")
    near, plain = pa.widom(b, g, **kw), pa.widom(b, g, **kw, single_phase=True)
    for r, p in zip(near, plain):
        for k in FIELDS:
            assert getattr(r, k) == pytest.approx(getattr(p, k), rel=1e-9, abs=1e-9 if k == "q_st_err" else 1e-300), k
