"""The FP64 paths' near lists as the batch's creation builds them (MI355X): large and long cells, whose
atoms the build tries in runs of 64, and what finds the lists: a no-allocation call that comes
first, and states made on several host threads.

Two-phase against single_phase (the plain kernel, every pair): FP64 sums of some 1e3 terms in
another order, 1e-9 as for the FP64 results against the oracle."""
import threading

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


@pytest.mark.parametrize("precision", ["f64", "mixed"])
def test_first_call_without_allocation(precision):
    """On a batch that has made no other call, then beside pa_widom, then again: the same fields."""
    ff, g, ew = _system()
    fws = [pa.replicate(synth.synthetic_framework(13.0, 13.0, 15.0, 90, 90, 120, n, 42, charge_sd=0.2), (3, 3, 2))
           for n in (40, 300)]
    # (the second one binds nothing, which the mixed path refuses)
    b = pa.FrameworkBatch(fws if precision == "f64" else fws[:1], ff, g, ew)
    kw = dict(T=T, ninsert=10_000, seed=3, nblocks=5, precision=precision)
    first = pa.widom(b, g, **kw, no_alloc=True)
    assert first == pa.widom(b, g, **kw) == pa.widom(b, g, **kw, no_alloc=True)


def test_states_made_on_several_threads():
    ff, g, ew = _system()
    fw = pa.replicate(synth.synthetic_framework(13.0, 13.0, 15.0, 90, 90, 120, 40, 42, charge_sd=0.2), (3, 3, 2))
    b = pa.FrameworkBatch([fw] * 4, ff, g, ew, fullk=True)
    want = pa.SystemState(b, g, [3] * 4, T=T, seed=7, capacities=[20] * 4)
    got, errors = [None] * 6, []

    def make(i):
        try:
            got[i] = pa.SystemState(b, g, [3] * 4, T=T, seed=7, capacities=[20] * 4)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=make, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    ref = pa.mc_moves(want, pa.MOVE_TRANSLATION, 40, T=T, step_trans=0.5, trace=True)
    for st in got:
        assert (pa.mc_moves(st, pa.MOVE_TRANSLATION, 40, T=T, step_trans=0.5, trace=True) == ref).all()
