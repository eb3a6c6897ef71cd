"""Host-side limits of the pull form, on the CPU: what its kernels address
must lie within the buffers that the library's own sizes give them."""

import math
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "openfermion-fqe_amd", "fqe_amd", "libfqehip.so")

pytestmark = pytest.mark.skipif(not os.path.exists(LIB),
                                reason="libfqehip.so not built")


def sector(norb, na, nb, npull):
    import torch  # noqa: F401  (binds the library to torch's HIP runtime)
    from fqe_amd import _lib
    s = _lib.Sector()
    s.norb, s.nalpha, s.nbeta = norb, na, nb
    s.lena, s.lenb = math.comb(norb, na), math.comb(norb, nb)
    s.npull = npull
    return s


def fits(norb, na, lenb, npull, complex_op):
    """One accumulator row and one W tile (k steps of 4 pairs, 64 doubles a
    step) in 160 KB of LDS beside the row tables."""
    ks = (na * (norb - na) + 4) // 4
    return (16 * lenb + ks * 512 * (2 if complex_op else 1) + 64 * 16 + 80 * 4
            + 32) <= 160 * 1024


@pytest.mark.parametrize("norb", range(1, 25))
def test_target_words_within_their_table(norb):
    """The row kernel takes the W tiles in equal passes (9 tiles of 16 pairs
    as 2 x 5), which is more than the table of target words may have.  It
    must read all rows of that table, npair rounded up to 16, and no word
    past them: the bounds check of the loads does not cover the row part of
    their address."""
    from fqe_amd import _lib
    plans = 0
    for complex_op, npull in ((0, norb * (norb + 1) // 2), (0, norb * norb),
                              (1, norb * norb)):
        for na in range(norb + 1):
            for nb in range(norb + 1):
                s = sector(norb, na, nb, npull)
                if not fits(norb, na, s.lenb, npull, complex_op):
                    continue
                n = _lib.lib().fqehip_pull_table_count(s, complex_op)
                plans += 1
                assert n == (npull + 15) // 16 * 16 * s.lenb, (na, nb, npull)
    assert plans


def test_fits_is_what_the_sector_with_tables_gets():
    """fqehip_pull_fits_supported without pointers answers as
    fqehip_pull_supported does with them."""
    import ctypes
    from fqe_amd import _lib
    lib = _lib.lib()
    op = _lib.Operator()
    op.a = 256
    seen = set()
    for norb in range(1, 25):
        for na in range(norb + 1):
            for nb in range(norb + 1):
                s = sector(norb, na, nb, norb * (norb + 1) // 2)
                fits = bool(lib.fqehip_pull_fits_supported(s, 0))
                s.pull_w = s.haa = s.hbb = s.pull_fwd = s.dexc_a = 256
                assert fits == bool(lib.fqehip_pull_supported(
                    _lib.C128, ctypes.byref(s), ctypes.byref(op))), (norb, na,
                                                                     nb)
                seen.add(fits)
    assert seen == {True, False}
