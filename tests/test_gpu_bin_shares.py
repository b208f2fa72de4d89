"""Mixed Widom path: workgroups that share a bin's insertions, and the bin scale a long call takes."""
import numpy as np
import pytest

import pureadsorb_amd as pa
from pureadsorb_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def porous():
    """80 atoms per hexagonal cell: about 1% of CO2 insertions bind."""
    ff = synth.synthetic_forcefield(12.0)
    g = synth.co2_guest(ff)
    fw = pa.replicate(synth.synthetic_framework(13.0, 13.0, 15.0, 90, 90, 120, 80, 42, charge_sd=0.5), (3, 3, 3))
    return fw, ff, g, pa.EwaldParams(12.0, 1e-6)


@pytest.mark.parametrize("n", [1, 11, 13, 97, 700, 5000, 30_000])
def test_shared_bins_match_f64(porous, n):
    """Bins from one (every insertion in it, eight shares, most of them empty at the smallest n) to
    too many to share: on binding poses the mixed energy stays within 3e-6 eV of the FP64 one (its
    FP32 pair terms), and every insertion is written."""
    fw, ff, g, ew = porous
    b = pa.FrameworkBatch([fw], ff, g, ew)
    ref = pa.widom_energies(b, 0, 42, 0, n, precision="f64")
    kT = pa.KB * 298.15
    for scale in (8.0, 1.0):
        b.bin_scale = scale
        dU = pa.widom_energies(b, 0, 42, 0, n, precision="mixed")
        bind = ref < 10 * kT
        print(n, scale, int(bind.sum()), np.max(np.abs(dU - ref)[bind], initial=0.0), flush=True)
        assert np.all(np.abs(dU - ref)[bind] <= 3e-6)
        assert not np.any(np.isnan(dU)) and np.all(dU[~bind] > 9 * kT)


@pytest.mark.parametrize("nfw", [1, 3])
def test_long_call_repeats_at_its_reported_scale(porous, nfw):
    """A long call on an unpinned batch, and on one pinned to the scale that it reports: equal bits."""
    fw, ff, g, ew = porous
    other = pa.replicate(synth.synthetic_framework(11.0, 12.0, 14.0, 80, 95, 100, 30, 7, charge_sd=0.3), (3, 3, 3))
    fws = [fw, other, fw][:nfw]
    b = pa.FrameworkBatch(fws, ff, g, ew)
    r = pa.widom(b, g, T=298.15, ninsert=300_000, seed=3)
    k = b.bin_scale
    again = pa.widom(b, g, T=298.15, ninsert=300_000, seed=3)
    pinned = pa.FrameworkBatch(fws, ff, g, ew)
    pinned.bin_scale = k
    print("scale", k, flush=True)
    assert 0.75 <= k <= 2.5
    assert r == again == pa.widom(pinned, g, T=298.15, ninsert=300_000, seed=3)
