"""Batches of millions of atoms (MI355X): the phase-0 lists are limited to 2^31 entries, which is what they
hold and not what a box around them could."""
import ctypes as C

import numpy as np
import pytest

from pureadsorb_amd import _lib

pytestmark = pytest.mark.gpu


def test_seventeen_million_atoms():
    """A 400 Å cell of 17.3 million atoms with small radii: some 3 lists an atom, where the box of cells
    within reach has 125. Mixed and two-phase FP64 results against the plain FP64 kernel: 1e-4 (mixed,
    as in test_gpu_guests.py) and 1e-9."""
    n, L = 17_300_000, 400.0
    rng = np.random.default_rng(3)
    frac = rng.random((n, 3))
    types, charges = np.zeros(n, dtype=np.int32), np.zeros(n)
    sig = np.array([0.30, 0.32, 0.32, 0.34])
    eps = np.array([0.004, 0.005, 0.005, 0.006])
    fw = _lib.PaFramework((C.c_double * 9)(L, 0, 0, 0, L, 0, 0, 0, L), n, frac.ctypes.data, types.ctypes.data,
                          charges.ctypes.data, (C.c_int32 * 3)(1, 1, 1))
    ff = _lib.PaForcefield(2, sig.ctypes.data, eps.ctypes.data, 6.0, 0)
    site, gtype, q = np.zeros(3), np.array([1], dtype=np.int32), np.zeros(1)
    guest = _lib.PaGuest(1, site.ctypes.data, gtype.ctypes.data, q.ctypes.data)
    ew = _lib.PaEwald(6.0, 1e-4)
    lib, h = _lib.lib(), C.c_void_p()
    _lib.check(lib.pa_batch_create(C.byref(fw), 1, C.byref(ff), C.byref(guest), C.byref(ew), 0, C.byref(h)))
    try:
        def ln_kh(precision):
            out = _lib.PaWidomResult()
            _lib.check(lib.pa_widom(h, C.byref(guest), 298.15, 64, 5, 4, 0, 0, precision, C.byref(out)))
            return out.ln_K_H

        # 64 insertions would share one bin, whose list of all atoms takes thousands of passes: bins of 4 Å
        _lib.check(lib.pa_batch_set_bin_scale(h, 0.01))
        plain = ln_kh(_lib.PA_PREC_F64 | _lib.PA_SINGLE_PHASE)
        near, mixed = ln_kh(_lib.PA_PREC_F64), ln_kh(_lib.PA_PREC_MIXED)
        print("ln K_H", plain, near, mixed, flush=True)
        assert near == pytest.approx(plain, rel=1e-9)
        assert mixed == pytest.approx(plain, rel=1e-4)
    finally:
        lib.pa_batch_destroy(h)
