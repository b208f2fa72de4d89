"""The FP64 paths over the near lists and the move kernel's variants (MI355X).

Skewed cells replicated to just over twice the cutoff are where a list could miss an atom: the
nearest image to the bin's centre and the image a site sees differ there. The two-phase FP64 call
is held to the plain kernel (single_phase), which tests every pair. Both sum some 1e3 FP64 terms
per insertion in different orders and skip only weights that are exactly zero, so results agree
to 1e-9, the tolerance of the FP64 results against the oracle.

The move kernel has one variant for up to 256 chains without exchange moves, one with, and one
for more chains; the same chain must take the same decisions in each (dU within 1e-9 of
1 + |dU|, FP64 sums in another order)."""
import numpy as np
import pytest

import pureadsorb_amd as pa
from pureadsorb_amd import synth

pytestmark = pytest.mark.gpu
T = 298.15
CELLS = {"cubic": (12.4, 12.4, 12.4, 90, 90, 90, 40), "hex": (13.0, 13.0, 15.0, 90, 90, 120, 50),
         "skew": (14.2, 17.1, 13.3, 62, 108, 71, 60), "flat": (29.0, 8.7, 31.0, 100, 75, 112, 120)}


def _system(cell, guest, fullk=False, nsys=1, width=24.0):
    a, b, c, al, be, ga, n = CELLS[cell]
    uc = synth.synthetic_framework(a, b, c, al, be, ga, n, 11, charge_sd=0.2)
    fw = pa.replicate(uc, synth.replication_for_width(uc, width))
    ff = synth.synthetic_forcefield(12.0, guest=guest)
    g = synth.co2_guest(ff) if guest == "co2" else synth.ch4_guest(ff)
    return pa.FrameworkBatch([fw] * nsys, ff, g, pa.EwaldParams(12.0, 1e-6), fullk=fullk), g


@pytest.mark.parametrize("cell", list(CELLS))
@pytest.mark.parametrize("guest,ninsert", [("co2", 4099), ("ch4", 40_001)])
def test_f64_near_lists_match_the_plain_kernel(cell, guest, ninsert):
    b, g = _system(cell, guest)
    near = pa.widom(b, g, T=T, ninsert=ninsert, seed=5, nblocks=4, precision="f64")[0]
    plain = pa.widom(b, g, T=T, ninsert=ninsert, seed=5, nblocks=4, precision="f64", single_phase=True)[0]
    print(f"{cell} {guest}: ln K_H {near.ln_K_H:.12f} plain {plain.ln_K_H:.12f}", flush=True)
    for k in ("mu_ex", "mu_ex_err", "K_H", "K_H_err", "q_st", "q_st_err", "ln_K_H"):
        assert getattr(near, k) == pytest.approx(getattr(plain, k), rel=1e-9, abs=1e-300), k
    assert near.nsamples == plain.nsamples == ninsert


def test_f64_near_lists_over_system_boundaries():
    """Wavefronts whose insertions belong to more than one system, and a chunk that cuts one."""
    b, g = _system("skew", "co2", nsys=7)
    kw = dict(T=T, ninsert=7 * 61 + 5, seed=3, nblocks=3, run=1, precision="f64")
    near = pa.widom(b, g, **kw, chunk=100)
    plain = pa.widom(b, g, **kw, single_phase=True)
    for r, p in zip(near, plain):
        assert r.ln_K_H == pytest.approx(p.ln_K_H, rel=1e-9) and r.nsamples == p.nsamples


@pytest.mark.parametrize("cell", ["hex", "skew"])
@pytest.mark.parametrize("guest", ["co2", "ch4"])
@pytest.mark.parametrize("move", [pa.MOVE_TRANSLATION, pa.MOVE_REINSERTION, pa.MOVE_INSERTION, pa.MOVE_DELETION])
def test_move_kernel_variants_agree(cell, guest, move):
    nmany, load, n = 260, 150, 70
    out = []
    for nsys in (1, nmany):
        b, g = _system(cell, guest, fullk=True, nsys=nsys)
        st = pa.SystemState(b, g, [0] * nsys, T=T, seed=9, capacities=[200] * nsys)
        pa.mc_moves(st, pa.MOVE_INSERTION, load, T=T, fugacity=3e6)
        tr = pa.mc_moves(st, move, n, T=T, step_trans=0.4, step_rot=0.3, fugacity=1e6, trace=True)[0]
        res = pa.run_gcmc(st, T=T, n_warmup=0, n_production=12, n_audit=1000, step_trans=0.5, step_rot=0.3, fugacity=1e6,
                          min_cycle_length=4, nblocks=2)[0]
        # the running energies against the poses (host rebuild)
        assert np.allclose(pa.total_energy(st), st.energy(), rtol=1e-9, atol=1e-9)
        out.append((tr, res, st.info(0), st.sk(0)))
        st.close()
        b.close()
    (t1, r1, i1, s1), (t2, r2, i2, s2) = out
    assert np.array_equal(t1[:, [0, 1, 3]], t2[:, [0, 1, 3]])
    fin = np.isfinite(t1[:, 2])
    assert np.array_equal(fin, np.isfinite(t2[:, 2]))
    assert np.all(np.abs(t1[fin, 2] - t2[fin, 2]) <= 1e-9 * (1 + np.abs(t1[fin, 2])))
    assert r1.accepted == r2.accepted and r1.attempted == r2.attempted
    assert i1["occupancy"] == i2["occupancy"] and i1["rng_counter"] == i2["rng_counter"]
    assert i1["energy"] == pytest.approx(i2["energy"], rel=1e-9, abs=1e-9)
    assert np.allclose(s1, s2, rtol=0, atol=1e-10)
