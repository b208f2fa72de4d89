"""Launches in which one wavefront takes several insertions (MI355X): from 32,768 insertions on it takes
two, and their count doubles with the launch. The same insertions in smaller launches take one
each. Also the move kernel's variant for more than 256 chains with guests of other site counts."""
import numpy as np
import pytest

import pureadsorb_amd as pa
from pureadsorb_amd import synth
from test_gpu_guests import _guest

pytestmark = pytest.mark.gpu
T = 298.15
FIELDS = ("mu_ex", "mu_ex_err", "K_H", "K_H_err", "q_st", "q_st_err", "ln_K_H", "nsamples")


def _porous(n=40, reps=(3, 3, 2)):
    return pa.replicate(synth.synthetic_framework(13.0, 13.0, 15.0, 90, 90, 120, n, 42, charge_sd=0.2), reps)


def test_charged_insertions_of_several_systems():
    """140,010 insertions: wavefronts of 4 (2 in chunks), boundaries of the three unlike systems and the last
    batch off their multiples. Launches of 20,000 take one each, and every insertion is evaluated on
    its own: the same bits. Against the plain kernel 1e-9, FP64 sums in another order."""
    ff = synth.synthetic_forcefield(12.0)
    g = synth.co2_guest(ff)
    skew = synth.synthetic_framework(27.0, 26.0, 28.0, 75, 100, 95, 200, 3, charge_sd=0.15)
    b = pa.FrameworkBatch([_porous(), skew, _porous(60)], ff, g, pa.EwaldParams(12.0, 1e-6))
    kw = dict(T=T, ninsert=3 * 46_670, seed=9, nblocks=7, run=1, precision="f64")
    whole = pa.widom(b, g, **kw)
    assert whole == pa.widom(b, g, **kw, chunk=20_000) == pa.widom(b, g, **kw, chunk=50_001)
    for r, p in zip(whole, pa.widom(b, g, **kw, single_phase=True)):
        for k in FIELDS:
            assert getattr(r, k) == pytest.approx(getattr(p, k), rel=1e-9), k


def test_chain_insertions_across_cycles_and_systems():
    """Four chains, five cycles of 2,001 insertions: 40,020 in one launch, wavefronts of two that hold the end
    of one cycle or chain and the start of the next. The first two chains alone make 20,010, one each:
    the same chains and poses, so the same sums to the last bit."""
    ff = synth.synthetic_forcefield(12.0)
    g = synth.co2_guest(ff)
    out = []
    for nsys in (4, 2):
        b = pa.FrameworkBatch([_porous()] * nsys, ff, g, pa.EwaldParams(12.0, 1e-6), fullk=True)
        st = pa.SystemState(b, g, [6, 4, 5, 3][:nsys], T=T, seed=5, capacities=[20] * nsys)
        pa.run_nvt(b, st, g, ff, T=T, n_warmup=0, n_production=5, n_widom_per_cycle=2001, n_audit=1000, step_trans=0.4,
                   step_rot=0.3, min_cycle_length=8, widom_seed=99, nblocks=2)
        out.append([np.array(pa.nvt_samples(st, n, 5)) for n in range(2)])
        if nsys == 4:
            assert pa.nvt_last_timing(st)["insertion_launches"] == 1
            # given poses, 40,000 and 5,000 at a time
            rng = np.random.default_rng(1)
            pos, q = rng.random((40_001, 3)) @ _porous().cell.T, rng.normal(size=(40_001, 4))
            q /= np.linalg.norm(q, axis=1)[:, None]
            whole = pa.widom_chain_energies(st, 2, pos, q)
            parts = [pa.widom_chain_energies(st, 2, pos[i:i + 5000], q[i:i + 5000]) for i in range(0, 40_001, 5000)]
            assert np.array_equal(whole, np.concatenate(parts), equal_nan=True)
    assert np.array_equal(out[0], out[1]) and np.all(np.isfinite(out[0]))


@pytest.mark.parametrize("ns", [1, 2, 4, 5, 6])
def test_move_variants_of_other_guests(ns):
    """One chain, and the same one first among 260: the same decisions, dU within 1e-9 of 1 + |dU|."""
    ff = synth.synthetic_forcefield(11.0)
    g = _guest(ff, ns)
    fw = pa.replicate(synth.synthetic_framework(12.0, 12.0, 12.0, 90, 90, 90, 40, 5, charge_sd=0.5), (2, 2, 2))
    out = []
    for nsys in (1, 260):
        b = pa.FrameworkBatch([fw] * nsys, ff, g, pa.EwaldParams(11.0), fullk=True)
        st = pa.SystemState(b, g, [4] + [0] * (nsys - 1), T=T, seed=9, capacities=[30] * nsys)
        tr = [pa.mc_moves(st, mt, 70, T=T, step_trans=0.3, step_rot=0.2, fugacity=f, trace=True)[0]
              for mt, f in ((1, 1e5), (4, 1e8), (2, 1e5), (3, 1e5), (5, 1e2))]
        assert np.allclose(pa.total_energy(st), st.energy(), rtol=1e-9, atol=1e-9)
        out.append((np.concatenate(tr), st.info(0)))
    (t1, i1), (t2, i2) = out
    assert np.array_equal(t1[:, [0, 1, 3]], t2[:, [0, 1, 3]])
    fin = np.isfinite(t1[:, 2])
    assert np.array_equal(fin, np.isfinite(t2[:, 2]))
    assert np.all(np.abs(t1[fin, 2] - t2[fin, 2]) <= 1e-9 * (1 + np.abs(t1[fin, 2])))
    assert i1["occupancy"] == i2["occupancy"] and i1["rng_counter"] == i2["rng_counter"]


def test_chain_insertions_into_a_very_long_cell():
    """A cell of 3,420 Å whose k-vectors' phase tables for six sites (over 100 KB) LDS does not hold: without
    guests a chain insertion is a Widom insertion (1e-10 as in test_gpu_nvt.py)."""
    ff = synth.synthetic_forcefield(12.0)
    g = _guest(ff, 6)
    fw = synth.synthetic_framework(24.1, 24.2, 3420.0, 90, 90, 90, 3000, 5, charge_sd=0.1)
    b = pa.FrameworkBatch([fw], ff, g, pa.EwaldParams(12.0, 1e-6), fullk=True)
    st = pa.SystemState(b, g, [0], T=T, seed=5, capacities=[2])
    pos, quat = pa.widom_poses(b, 0, 777, 0, 200)
    dU = pa.widom_chain_energies(st, 0, pos, quat)
    ref = pa.widom_energies(b, 0, 777, 0, 200, precision="f64")
    fin = np.isfinite(ref) & (np.abs(ref) < 1e8)
    assert fin.sum() > 100
    assert np.all(np.abs(dU[fin] - ref[fin]) <= 1e-10 * (1 + np.abs(ref[fin])))
