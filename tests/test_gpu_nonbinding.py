"""Float64 Widom where nothing binds (MI355X): cells so dense that the best insertion lies some 100
to 700 eV up.

Phase 0 rejects insertions whose weight exp(-dU/kT) is zero in Float64; the estimators are sums
relative to the system's best insertion, which here is often a rejected one. The two-phase call is
held to single_phase, which evaluates every insertion. Tolerance: an energy is a sum of FP64 terms
of its own size, taken in another order with some 20 ulp, so -dU/kT (up to 700 eV / 0.0257 eV)
agrees to 20 * 2.2e-16 * 2.7e4 = 1.2e-10, and with it every weight: 1e-9.

q_st_err is the root of vU/U^2 + vW/W^2 - 2 cov/(U W), times |q_st|/sqrt(nblocks). Where one insertion
holds all the weight each term is nblocks (up to a factor 2) and they cancel, so that what is left
is rounding: four terms of nblocks to 8 ulp, 32 eps q_st^2 in the square. Its square is compared
to that, beside 1e-9."""
import sys

import pytest

import pureadsorb_amd as pa
from pureadsorb_amd import synth

pytestmark = pytest.mark.gpu
T = 298.15
FIELDS = ("mu_ex", "mu_ex_err", "K_H", "K_H_err", "q_st", "ln_K_H", "nsamples", "nblocks")


def _cell(atoms, seed, charge_sd=0.0):
    return pa.replicate(synth.synthetic_framework(12.9, 12.9, 12.9, 90, 90, 90, atoms, seed, charge_sd=charge_sd), (2, 2, 2))


def _batch(fws, guest):
    ff = synth.synthetic_forcefield(12.0, guest=guest)
    g = synth.co2_guest(ff) if guest == "co2" else synth.ch4_guest(ff)
    return pa.FrameworkBatch(fws, ff, g, pa.EwaldParams(12.0, 1e-6)), g


def _same(got, want):
    assert len(got) == len(want)
    for r, w in zip(got, want):
        for k in FIELDS:
            assert getattr(r, k) == pytest.approx(getattr(w, k), rel=1e-9, abs=1e-300), k
        noise = 32 * sys.float_info.epsilon * w.q_st**2
        assert r.q_st_err**2 == pytest.approx(w.q_st_err**2, rel=2e-9, abs=noise)


@pytest.mark.parametrize("guest,atoms,fw_seed,seed,n", [
    ("ch4", 320, 7, 0, 5000),  # every insertion rejected
    ("ch4", 300, 7, 1, 1000), ("ch4", 300, 7, 2, 1000), ("ch4", 300, 7, 3, 20),
    ("ch4", 260, 3, 4, 1000),  # the best one rejected, another left
    ("co2", 300, 1, 3, 1000), ("co2", 300, 2, 5, 40_000)])
def test_two_phase_equals_single_phase_without_binding(guest, atoms, fw_seed, seed, n):
    b, g = _batch([_cell(atoms, fw_seed, 0.15 if guest == "co2" else 0.0)], guest)
    kw = dict(T=T, ninsert=n, seed=seed, nblocks=4, precision="f64")
    want = pa.widom(b, g, **kw, single_phase=True)
    print(guest, atoms, n, "ln K_H", want[0].ln_K_H, flush=True)
    assert want[0].ln_K_H < -697.0
    _same(pa.widom(b, g, **kw), want)


def test_binding_and_other_systems_in_one_batch():
    """Dense systems first, in the middle side by side, and last, and a chunk that cuts them."""
    dense, porous = [_cell(300, 7, 0.15), _cell(290, 8, 0.15)], _cell(40, 9, 0.15)
    fws = [dense[0], porous, dense[1], dense[0], porous, dense[1]]
    b, g = _batch(fws, "co2")
    kw = dict(T=T, ninsert=6 * 211 + 5, seed=3, nblocks=3, run=1, precision="f64")
    want = pa.widom(b, g, **kw, single_phase=True)
    assert [r.ln_K_H < -697.0 for r in want] == [True, False, True, True, False, True]
    got = pa.widom(b, g, **kw, chunk=100)
    _same(got, want)
    # gradients carry the same call's results
    grad = pa.widom_grad(b, g, **kw)
    assert [x.result for x in grad] == pa.widom(b, g, **kw)
    _same([x.result for x in grad], want)
