"""Phase 0 from the coldest call to the warmest (MI355X): the cells' lists hold the rejection radii of 0 K and
are cut short at those of 77 and 273 K, and calls at and beside those temperatures take one part or
the other. Bars as in test_gpu_reject.py: the device
rejects nothing that the oracle's brute-force check does not, and two-phase and single-phase mixed
results are the same."""
import numpy as np
import pytest

import pureadsorb_amd as pa
from conftest import oracle_for, oracle_threads
from pureadsorb_amd import synth

pytestmark = pytest.mark.gpu


def _system(cell, guest):
    """hex: cells of 1.2 Å; long: 64 cells of 3.2 Å on one axis (their cap)."""
    ff = synth.synthetic_forcefield(12.0, guest=guest)
    g = synth.co2_guest(ff) if guest == "co2" else synth.ch4_guest(ff)
    if cell == "hex":
        fw = pa.replicate(synth.synthetic_framework(13.0, 13.0, 15.0, 90, 90, 120, 60, 42, charge_sd=0.2), (3, 3, 2))
    else:
        fw = synth.synthetic_framework(24.5, 24.5, 205.0, 90, 90, 90, 2600, 5, charge_sd=0.1 if guest == "co2" else 0.0)
    return fw, ff, g, pa.EwaldParams(12.0, 1e-6)


@pytest.mark.parametrize("T", [1.0, 20.0, 76.0, 77.0, 78.0, 272.0, 273.0, 274.0, 500.0])
@pytest.mark.parametrize("cell,guest", [("hex", "co2"), ("hex", "ch4"), ("long", "ch4"), ("long", "co2")])
def test_cold_flags_and_results(cell, guest, T):
    fw, ff, g, ew = _system(cell, guest)
    b = pa.FrameworkBatch([fw, fw], ff, g, ew)
    o = oracle_for(fw, ff, g, ew)
    n, kT = 3000, pa.KB * T
    dev = pa.hardcore_flags(b, 1, 11, T, 7, n).astype(bool)
    _, rho2 = o.rejection_tables(kT, 1.1920929e-07)
    ref = o.hardcore_flags(11, 1, 7, n, rho2, nthreads=oracle_threads()).astype(bool)
    warm = pa.hardcore_flags(b, 1, 11, 298.15, 7, n).astype(bool)
    print(f"{cell} {guest} {T} K: device rejects {dev.sum()}, oracle {ref.sum()} of {n}, at 298 K {warm.sum()}", flush=True)
    assert not np.any(dev & ~ref) and dev.sum() >= 0.97 * ref.sum()
    # radii shrink as it gets warmer
    assert not np.any(warm & ~dev if T < 298.15 else dev & ~warm)
    if T < 5.0:  # weights overflow Float64
        return
    kw = dict(T=T, ninsert=50_000, seed=5, nblocks=4)
    assert pa.widom(b, g, **kw) == pa.widom(b, g, **kw, single_phase=True)
    f64 = pa.widom(b, g, **kw, precision="f64")
    for r, s in zip(f64, pa.widom(b, g, **kw, precision="f64", single_phase=True)):
        assert r.ln_K_H == pytest.approx(s.ln_K_H, rel=1e-9) and r.q_st == pytest.approx(s.q_st, rel=1e-9)
