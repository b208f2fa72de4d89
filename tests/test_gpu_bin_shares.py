"""Mixed Widom path: the bin scale a long call takes."""
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
