"""Operator and string tables that one stream builds and another reads, and
tables first needed under capture.  The tables are built by kernels at the
first apply that needs them and kept; a second stream must wait for them."""

import numpy
import pytest

from oracle import fqe_oracle as fo
from tests.test_gpu_pull import prepared, tensors

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fqe():
    import torch
    assert torch.cuda.is_available()
    import fqe_amd
    return fqe_amd


def problem(fqe, kind, na, nb, norb):
    """Coefficients on the device and two equal operators, neither with
    tables, on string tables of their own."""
    from fqe_amd import fci_graph
    fci_graph._TABLE_CACHE.clear()
    rng = numpy.random.default_rng(norb)
    d = fqe.FqeData(na, nb, norb, dtype=numpy.complex128)
    d.coeff = fo.synthetic_coeff(d.lena(), d.lenb(), rng)
    x = d.device_coeff()
    h = tensors(kind, norb, rng)
    return d.get_fcigraph(), x, prepared(fqe, kind, h, norb), prepared(
        fqe, kind, h, norb)


@pytest.mark.parametrize("kind,engine_kind,na,nb,norb", [
    ("real", "fp64", 5, 4, 9), ("real", "ozaki", 4, 5, 9),
    ("complex", "fp64", 4, 5, 9), ("nonsymmetric", "fp64", 5, 5, 10),
    ("spin", "fp64", 5, 4, 9), ("spin_complex", "fp64", 4, 4, 9)])
def test_second_stream_waits_for_the_tables(fqe, kind, engine_kind, na, nb,
                                            norb):
    """Stream 1 is held back, then asked to build the tables; stream 2
    applies the operator at once.  Same kernels, hence the same bits as an
    apply on one stream."""
    import torch
    from fqe_amd import engine, settings
    print(f"streams {kind} {engine_kind}", flush=True)
    saved = settings.contraction, settings.ozaki_min_determinants
    settings.contraction, settings.ozaki_min_determinants = engine_kind, 0
    try:
        graph, x, op, _ = problem(fqe, kind, na, nb, norb)
        streams = [torch.cuda.Stream() for _ in range(2)]
        outs = [torch.empty_like(x) for _ in range(3)]
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[0]):
            torch.cuda._sleep(5000000)
            engine.apply_sector(graph, x, op, outs[0])
        with torch.cuda.stream(streams[1]):
            engine.apply_sector(graph, x, op, outs[1])
        torch.cuda.synchronize()
        engine.apply_sector(graph, x, op, outs[2])
    finally:
        settings.contraction, settings.ozaki_min_determinants = saved
    want = outs[2].cpu().numpy()
    assert numpy.isfinite(want).all() and want.any()
    for out in outs[:2]:
        assert numpy.array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("kind", ["real", "complex", "spin"])
def test_tables_first_needed_under_capture(fqe, kind):
    """A captured apply whose tables are missing builds them in the graph and
    keeps none: an eager apply before the replay must not find tables that
    nothing has filled.  Replays on new coefficients, with eager work between
    them, against eager applies."""
    import torch
    from fqe_amd import engine
    print(f"capture {kind}", flush=True)
    graph, x, op, other = problem(fqe, kind, 4, 3, 8)
    out, eager = torch.empty_like(x), torch.empty_like(x)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            engine.apply_sector(graph, x, op, out)
    assert len(op._tables) == 0
    engine.apply_sector(graph, x, op, eager)
    want = torch.empty_like(x)
    engine.apply_sector(graph, x, other, want)
    assert numpy.array_equal(eager.cpu().numpy(), want.cpu().numpy())
    for k in range(3):
        g.replay()
        engine.apply_sector(graph, x, other, want)
        torch.cuda.synchronize()
        assert numpy.array_equal(out.cpu().numpy(), want.cpu().numpy()), k
        x.mul_(0.5 - 1j)


@pytest.mark.parametrize("how", ["deepcopy", "pickle"])
def test_copies_of_an_applied_hamiltonian(fqe, how):
    """A Hamiltonian that holds its device tables copies and pickles, and
    the copy applies with the same bits."""
    import copy
    import pickle
    rng = numpy.random.default_rng(3)
    h = tensors("real", 7, rng)
    wfn = fqe.Wavefunction([[7, 1, 7]])
    wfn.set_wfn("random")
    ham = fqe.get_restricted_hamiltonian(h)
    want = wfn.apply(ham).get_coeff((7, 1))
    other = (copy.deepcopy(ham) if how == "deepcopy" else
             pickle.loads(pickle.dumps(ham)))
    assert numpy.array_equal(wfn.apply(other).get_coeff((7, 1)), want)
