"""Gram products of interleaved and planar rows, on the GPU, at the edges of
their tiles: 32-row blocks, 8-element wave steps, 32-element workgroup steps,
chunks; general and with one block against itself.  Tolerance: FP64 sums of
n products of magnitude about 1, each rounded to 1.1e-16, over the square
root of n in norm, so 1e-14 sqrt(n) per element is ample and catches any
lost or repeated element (about 1)."""

import numpy
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fqe():
    import torch
    assert torch.cuda.is_available()
    import fqe_amd
    return fqe_amd


@pytest.mark.parametrize("k", [1, 15, 32, 33, 65, 101])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 33, 255, 257, 4099])
def test_gram_rows(fqe, k, n):
    import torch
    from fqe_amd import _lib, engine
    rng = numpy.random.default_rng(1000 * k + n)
    a, b = (rng.normal(size=(k, n)) + 1j * rng.normal(size=(k, n))
            for _ in range(2))
    dev = _lib.device()
    da, db = (torch.from_numpy(x).to(dev) for x in (a, b))
    pa, pb = (torch.stack((x.real, x.imag), 1).contiguous() for x in (da, db))
    tol = 1e-14 * numpy.sqrt(n)
    for got, ref in ((engine.gram(da, db), a.conj() @ b.T),
                     (engine.gram_planar(pa, pb), a.conj() @ b.T),
                     (engine.gram(da, da), a.conj() @ a.T),
                     (engine.gram_planar(pb, pb), b.conj() @ b.T)):
        assert numpy.max(numpy.abs(got - ref)) < 10 * tol
