"""The pull form of the complex128 apply (k_same_spin_f64 and
k_pull_rows_f64), on the GPU, against the oracle where it is small enough
and against the slot-row and unfused kernels elsewhere.

Sizes: one to several 16-column tiles with remainders, one and several
passes over the W tiles (npair 3 to 196), one and several accumulator rows,
4- and 8-wave workgroups, no off-diagonal alpha pair (empty or full alpha
shell).  Tolerance 1e-12 normwise, as for every FP64 kernel here (sums of at
most a few thousand products of random signs, each rounded to 1.1e-16).
"""

import copy

import numpy
import pytest

from oracle import fqe_oracle as fo

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module")
def fqe():
    import torch
    assert torch.cuda.is_available()
    import fqe_amd
    return fqe_amd


def rel(a, b):
    return numpy.linalg.norm(a - b) / numpy.linalg.norm(b)


def tensors(kind, norb, rng):
    h1, h2 = fo.synthetic_hamiltonian(norb, norb, rng)
    if kind == "real":
        return h1, h2
    if kind == "nonsymmetric":
        return (h1 + 0.1 * rng.normal(size=h1.shape),
                h2 + 0.02 * rng.normal(size=h2.shape))
    if kind == "complex":
        return (h1 + 0.1j * rng.normal(size=h1.shape),
                h2 + 0.02j * rng.normal(size=h2.shape))
    m = 2 * norb
    h1 = rng.normal(size=(m, m)) + 1j * rng.normal(size=(m, m))
    h2 = rng.normal(size=(m,) * 4) + 1j * rng.normal(size=(m,) * 4)
    return (h1.real, h2.real) if kind == "spin" else (h1, h2)


def sector(fqe, na, nb, norb, seed):
    rng = numpy.random.default_rng(seed)
    g = fo.OracleGraph(na, nb, norb)
    d = fqe.FqeData(na, nb, norb, dtype=numpy.complex128)
    c = fo.synthetic_coeff(g.lena, g.lenb, rng)
    d.coeff = c
    return d, c, g, rng


def prepared(fqe, kind, h, norb):
    from fqe_amd import _lib, engine
    make = (engine.prepare_spin_operator if kind.startswith("spin") else
            engine.prepare_operator)
    return make(h, norb, _lib.device())


def takes_pull(d, op):
    import ctypes
    from fqe_amd import _lib, engine
    s, keep = engine.sector_struct(d.get_fcigraph(), op, _lib.C128)
    return bool(_lib.lib().fqehip_pull_supported(
        _lib.C128, ctypes.byref(s), ctypes.byref(op.c_struct())))


@pytest.mark.parametrize("kind", ["real", "nonsymmetric", "complex", "spin",
                                  "spin_complex"])
@pytest.mark.parametrize("na,nb,norb", [(1, 1, 2), (1, 2, 3), (2, 1, 5),
                                        (3, 3, 6), (6, 2, 6), (2, 6, 7),
                                        (5, 3, 7), (4, 3, 8), (3, 7, 9)])
def test_pull_matches_oracle(fqe, kind, na, nb, norb):
    print(f"pull {kind} {na} {nb} {norb}", flush=True)
    d, c, g, rng = sector(fqe, na, nb, norb, 31 * norb + 7 * na + nb)
    h = tensors(kind, norb, rng)
    op = prepared(fqe, kind, h, norb)
    assert takes_pull(d, op)
    ref = (fo.apply_spin12(c, h[0], h[1], g) if kind.startswith("spin") else
           fo.apply_12(c, h[0], h[1], g))
    outs = []
    for _ in range(2):
        e = copy.deepcopy(d)
        e.apply_inplace_scaled(h, op=op)
        outs.append(e.coeff)
    assert rel(outs[0], ref) < TOL
    assert numpy.array_equal(outs[0], outs[1])
    # the separate epilogue (in place, with accumulation and norm) and the
    # one in the row kernel
    from fqe_amd import engine
    import torch
    x = d.device_coeff().clone()
    acc = torch.zeros_like(x)
    n = engine.norm_partials_count(x.numel())
    part = torch.zeros(max(n, 1), dtype=torch.float64, device=x.device)
    engine.apply_sector(d.get_fcigraph(), x, op, x, alpha=0.5 - 2j,
                        acc=torch.view_as_real(acc), partials=part)
    want = (0.5 - 2j) * ref
    assert rel(x.cpu().numpy(), want) < TOL
    assert rel(acc.cpu().numpy(), want) < TOL
    norm = numpy.sqrt(part.sum().item())
    assert abs(norm - numpy.linalg.norm(want)) < TOL * norm
    y = torch.empty_like(x)
    engine.apply_sector(d.get_fcigraph(), d.device_coeff(), op, y,
                        alpha=0.5 - 2j, beta=1.5j, cin=d.device_coeff())
    assert rel(y.cpu().numpy(), want + 1.5j * c) < TOL


@pytest.mark.parametrize("kind,na,nb,norb", [
    ("real", 5, 6, 12), ("real", 7, 6, 13), ("real", 7, 7, 14),
    ("real", 2, 8, 15), ("real", 3, 10, 15), ("nonsymmetric", 4, 6, 13),
    ("complex", 5, 5, 11), ("complex", 6, 7, 14), ("spin", 5, 4, 11),
    ("spin_complex", 3, 4, 12), ("nonsymmetric", 5, 1, 12),
    ("complex", 1, 6, 12), ("spin_complex", 4, 4, 9), ("real", 4, 4, 13)])
def test_pull_matches_other_kernels(fqe, kind, na, nb, norb):
    """Sectors too large for the oracle: the same operator on the slot-row
    kernels (real symmetric) or the unfused ones."""
    from fqe_amd import settings
    print(f"pull {kind} {na} {nb} {norb}", flush=True)
    d, c, g, rng = sector(fqe, na, nb, norb, 17 * norb + 3 * na + nb)
    h = tensors(kind, norb, rng)
    op = prepared(fqe, kind, h, norb)
    assert takes_pull(d, op)
    e = copy.deepcopy(d)
    e.apply_inplace_scaled(h, op=op)
    saved = settings.split_tile_fp64
    settings.split_tile_fp64 = 0
    try:
        assert not takes_pull(d, op)
        d.apply_inplace_scaled(h, op=op)
    finally:
        settings.split_tile_fp64 = saved
    assert rel(e.coeff, d.coeff) < TOL


@pytest.mark.parametrize("shape", ["synthetic", "constant"])
@pytest.mark.parametrize("blocks", [True, False])
@pytest.mark.parametrize("na,nb,norb", [(1, 1, 2), (1, 2, 3), (3, 2, 5),
                                        (6, 1, 6), (4, 4, 8), (3, 7, 9),
                                        (8, 5, 9), (6, 6, 11), (8, 2, 15)])
def test_digit_rows_edges(fqe, na, nb, norb, blocks, shape):
    """The digit kernels on every sector (ozaki_min_determinants = 0):
    fewer than 64 columns or strings, ragged tiles, 3 to 120 pairs, 2 to 64
    de-excitation rows; and the largest possible sums (every integral and
    every coefficient equal).  Tolerance 3e-11 normwise: operator rounding
    2^-39 of the row's largest element, data rounding 2^-47 of the largest
    coefficient, dropped digit pairs below both, times the spread between
    the largest element and the norm of a row (up to some hundreds here).  Integer sums: the same bits
    on every run."""
    from fqe_amd import settings
    print(f"digit rows {na} {nb} {norb} {blocks} {shape}", flush=True)
    d, c, g, rng = sector(fqe, na, nb, norb, 11 * norb + 5 * na + nb)
    h = tensors("real", norb, rng)
    if shape == "constant":
        h = (numpy.full_like(h[0], 0.3), numpy.full_like(h[1], -0.3))
        c = numpy.full_like(c, 1 + 1j) / numpy.sqrt(2.0 * c.size)
        d.coeff = c
    op = prepared(fqe, "real", h, norb)
    saved = (settings.contraction, settings.ozaki_beta,
             settings.ozaki_min_determinants)
    settings.contraction, settings.ozaki_beta = "ozaki", blocks
    settings.ozaki_min_determinants = 0
    outs = []
    try:
        for _ in range(2):
            e = copy.deepcopy(d)
            e.apply_inplace_scaled(h, op=op)
            outs.append(e.coeff)
    finally:
        (settings.contraction, settings.ozaki_beta,
         settings.ozaki_min_determinants) = saved
    d.apply_inplace_scaled(h, op=op)
    assert rel(outs[0], d.coeff) < 3e-11
    assert numpy.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("blocks", [True, False])
@pytest.mark.parametrize("zero", ["alpha", "beta", "both", "all"])
@pytest.mark.parametrize("na,nb,norb", [(4, 3, 8), (3, 5, 9), (5, 5, 10)])
def test_digit_rows_with_empty_strings(fqe, na, nb, norb, zero, blocks):
    """Alpha strings, beta strings, or both without any amplitude (every
    string that occupies orbital 0), and a vector of zeros: a zero row or
    column of C has no digit scale.  Tolerance as in test_digit_rows_edges;
    of zeros, exactly zeros."""
    from fqe_amd import settings
    print(f"empty strings {na} {nb} {norb} {zero} {blocks}", flush=True)
    d, c, g, rng = sector(fqe, na, nb, norb, 11 * norb + 5 * na + nb)
    h = tensors("real", norb, rng)
    c = c.copy()
    core = d.get_fcigraph()
    if zero in ("alpha", "both"):
        c[core.string_alpha_all() & numpy.uint64(1) == 1, :] = 0.0
    if zero in ("beta", "both"):
        c[:, core.string_beta_all() & numpy.uint64(1) == 1] = 0.0
    if zero == "all":
        c[:] = 0.0
    d.coeff = c
    op = prepared(fqe, "real", h, norb)
    saved = (settings.contraction, settings.ozaki_beta,
             settings.ozaki_min_determinants)
    settings.contraction, settings.ozaki_beta = "ozaki", blocks
    settings.ozaki_min_determinants = 0
    try:
        e = copy.deepcopy(d)
        e.apply_inplace_scaled(h, op=op)
    finally:
        (settings.contraction, settings.ozaki_beta,
         settings.ozaki_min_determinants) = saved
    d.apply_inplace_scaled(h, op=op)
    if zero == "all":
        assert not e.coeff.any()
    else:
        assert rel(e.coeff, d.coeff) < 3e-11


@pytest.mark.parametrize("large", [1e3, 1e5, 1e6, 1e9])
@pytest.mark.parametrize("na,nb,norb", [(4, 3, 8), (3, 5, 9), (5, 5, 10)])
def test_digit_rows_beside_a_large_integral(fqe, na, nb, norb, large):
    """One local integral (00|00) far above the others, and no determinant of
    the vector with orbital 0 occupied.  Only the row (00) of W is rounded as
    coarsely as that integral asks; it reaches beta strings that occupy
    orbital 0, and on the others the result keeps the tolerance of
    test_digit_rows_edges.  Past the range of the digits the sector runs in
    FP64."""
    from fqe_amd import _lib, engine, settings
    print(f"digit rows {na} {nb} {norb} large {large}", flush=True)
    d, c, g, rng = sector(fqe, na, nb, norb, 11 * norb + 5 * na + nb)
    h1, h2 = tensors("real", norb, rng)
    h2 = h2.copy()
    h2[0, 0, 0, 0] = -large * numpy.abs(h2).max()
    c = c.copy()
    core, bit = d.get_fcigraph(), numpy.uint64(1)
    c[core.string_alpha_all() & bit == 1, :] = 0.0
    beta = core.string_beta_all() & bit == 0
    c[:, ~beta] = 0.0
    d.coeff = c
    op = prepared(fqe, "real", (h1, h2), norb)
    saved = settings.contraction, settings.ozaki_min_determinants
    settings.contraction, settings.ozaki_min_determinants = "ozaki", 0
    try:
        s, keep = engine.sector_struct(d.get_fcigraph(), op, _lib.C128)
        assert bool(s.w_oz) == (large < 1e8)
        e = copy.deepcopy(d)
        e.apply_inplace_scaled((h1, h2), op=op)
    finally:
        settings.contraction, settings.ozaki_min_determinants = saved
    d.apply_inplace_scaled((h1, h2), op=op)
    assert rel(e.coeff[:, beta], d.coeff[:, beta]) < 3e-11
    if large > 1e8:
        assert numpy.array_equal(e.coeff, d.coeff)


@pytest.mark.parametrize("nterms", [0, 1, 2, 5])
@pytest.mark.parametrize("group", [True, False])
def test_batch_terms(fqe, nterms, group):
    """Pull-form sectors of a batch: alternating term buffers for every
    parity of the last term, groups of one and several sectors of each W
    tile count, sectors past the groups (8-wave workgroups), items without
    the apply.  Against applies one by one; 1e-13 as the kernels are the
    same and only the epilogue's order of additions differs."""
    import ctypes
    import torch
    from fqe_amd import _lib, batched
    rng = numpy.random.default_rng(5)
    shapes = [(2, 1, 1), (3, 1, 2), (4, 2, 2), (4, 2, 0), (5, 5, 2), (6, 3, 3),
              (7, 3, 4), (8, 4, 3), (9, 4, 4), (10, 5, 4), (6, 1, 3), (6, 3, 3)]
    specs = []
    for norb, na, nb in shapes:
        h1, h2 = fo.synthetic_hamiltonian(norb, norb, rng)
        g = fo.OracleGraph(na, nb, norb)
        specs.append(batched.SectorSpec(
            norb=norb, nalpha=na, nbeta=nb, h1=h1, h2=h2,
            coeff=fo.synthetic_coeff(g.lena, g.lenb, rng)))
    tiles = {f"{n},{a},{b}": "split" for n, a, b in shapes}
    bt = batched.BatchedTaylor(specs, 0.1, nterms=nterms,
                               dtype=torch.complex128, tiles=tiles, nstreams=3,
                               group=group)
    items = []
    for i, p in enumerate(bt.sectors):
        it = p.item()
        if i % 3 == 2:
            it.d_apply_out = None
            p.apply_out.fill_(7.0)
        items.append(it)
    arr = (_lib.BatchItem * len(items))(*items)
    handle = ctypes.c_void_p()
    torch.cuda.synchronize()
    _lib.call("fqehip_batch_create", bt.prec, len(items), arr, bt.time, nterms,
              3, int(group), _lib.stream_ptr(), ctypes.byref(handle))
    bt._batch = handle
    for _ in range(2):
        bt.launch()
        got = bt.results()
        torch.zeros(1000, device="cuda").sum().item()
    bt.run_sequential()
    for i, ((a0, e0), (a1, e1)) in enumerate(zip(got, bt.results())):
        assert rel(e0, e1) < 1e-13, shapes[i]
        if i % 3 == 2:
            assert (a0 == 7.0).all(), shapes[i]
        else:
            assert rel(a0, a1) < 1e-13, shapes[i]
    bt.close()


@pytest.mark.parametrize("na,nb,norb", [
    (2, 2, 4), (3, 3, 7), (4, 4, 8),                   # one launch a term
    (4, 3, 9), (5, 2, 10), (2, 5, 10), (6, 1, 12),     # same-spin kernel first
    (6, 0, 13), (5, 1, 13)])                           # test in its own launch
def test_series_terms(fqe, na, nb, norb):
    """A Taylor series whose terms are tested for convergence at the start
    of the next term's kernel: the sum against applies one by one, summed
    in the same order and stopped at the same norm (1e-13: the kernels are
    the same but for the epilogue), and no convergence where one term fewer
    is allowed than it takes."""
    rng = numpy.random.default_rng(50 * norb + na)
    h1, h2 = fo.synthetic_hamiltonian(norb, norb, rng)
    ham = fqe.get_restricted_hamiltonian((h1, h2))
    d, c, g, rng = sector(fqe, na, nb, norb, 7)
    key = (na + nb, na - nb)
    wfn = fqe.Wavefunction([[na + nb, na - nb, norb]])
    wfn.set_wfn("from_data", {key: c / numpy.linalg.norm(c)})
    t = 0.01
    term, acc, nterms = wfn, wfn.get_coeff(key).copy(), 0
    for order in range(1, 30):
        term = term.apply(ham)
        term.scale(-1j * t / order)
        acc = acc + term.get_coeff(key)
        nterms = order
        if term.norm() < 1e-12:
            break
    got = wfn.apply_generated_unitary(t, "taylor", ham, accuracy=1e-12,
                                      expansion=nterms + 1)
    assert rel(got.get_coeff(key), acc) < 1e-13
    longer = wfn.apply_generated_unitary(t, "taylor", ham, accuracy=1e-12,
                                         expansion=nterms + 6)
    assert numpy.array_equal(longer.get_coeff(key), got.get_coeff(key))
    with pytest.raises(RuntimeError):
        wfn.apply_generated_unitary(t, "taylor", ham, accuracy=1e-12,
                                    expansion=nterms)


@pytest.mark.parametrize("kind", ["real", "complex"])
@pytest.mark.parametrize("na,nb,norb", [(3, 3, 6), (6, 1, 12), (5, 5, 11)])
def test_accumulate_onto_the_input(fqe, kind, na, nb, norb):
    """acc += alpha H C where acc is C (and where it overlaps C in part):
    every row of C is read before any is written.  In the row kernel's
    epilogue it would race with the rows that still read C.  Sectors whose
    rows run in one wave of workgroups and in several.  1e-13: the same
    kernels as the separate buffers', other epilogue."""
    import torch
    from fqe_amd import _lib, engine
    print(f"acc on input {kind} {na} {nb} {norb}", flush=True)
    d, c, g, rng = sector(fqe, na, nb, norb, 3 * norb + na)
    op = prepared(fqe, kind, tensors(kind, norb, rng), norb)
    assert takes_pull(d, op)
    x = d.device_coeff()
    n = x.numel()
    want = torch.empty_like(x)
    engine.apply_sector(d.get_fcigraph(), x, op, want, alpha=0.5 - 2j)
    want = want.cpu().numpy()
    for shift in (0, n // 2):
        # C at the start of a longer buffer, acc `shift` elements after it
        buf = torch.zeros(2 * n, dtype=x.dtype, device=x.device)
        buf[:n] = x.reshape(-1)
        before = buf.cpu().numpy()
        out = torch.empty_like(x)
        s, keep = engine.sector_struct(d.get_fcigraph(), op, _lib.C128)
        ws = engine.workspace(s, _lib.C128, x.device)
        _lib.call("fqehip_apply", _lib.C128, engine._as_ref(s),
                  engine._as_ref(op.c_struct()), _lib.ptr(buf), 0.5, -2.0,
                  0.0, 0.0, None, _lib.ptr(out), _lib.ptr(buf) + 16 * shift,
                  None, None, _lib.ptr(ws), _lib.stream_ptr())
        before[shift:shift + n] += want.reshape(-1)
        assert rel(out.cpu().numpy(), want) < 1e-13
        assert rel(buf.cpu().numpy(), before) < 1e-13


@pytest.mark.parametrize("na,nb,norb", [(5, 8, 16), (8, 5, 16)])
def test_no_blocks_past_the_limits(fqe, na, nb, norb):
    """A sector that the pull form refuses (12870 strings of one spin) builds
    none of its tables: Haa or Hbb would take 1.3 GB for nothing."""
    import torch
    from fqe_amd import _lib, engine, settings
    from fqe_amd.fci_graph import FciGraph
    graph = FciGraph(na, nb, norb)
    op = prepared(fqe, "real", tensors("real", norb,
                                       numpy.random.default_rng(1)), norb)
    before = torch.cuda.memory_allocated()
    assert op.pull_tables(graph) is None
    s, keep = engine.sector_struct(graph, op, _lib.C128)
    assert not s.pull_w and not s.haa and not s.hbb
    # the string tables of the unfused path, npair rows each
    tables = 3 * op.npair * 4 * (graph.lena() + graph.lenb())
    assert torch.cuda.memory_allocated() - before <= tables + (1 << 20)
    # within the limits again: one electron fewer
    small = FciGraph(2, 2, norb)
    assert op.pull_tables(small) is not None


@pytest.mark.parametrize("nterms", [1, 4])
@pytest.mark.parametrize("contraction,group,norb,na,nb,kernels,extra", [
    ("fp64", True, 8, 4, 4, 1, 0),      # rows with their same-spin part
    ("fp64", True, 9, 4, 4, 2, 0),      # same-spin products, rows
    ("fp64", False, 8, 4, 4, 1, 1),     # on its own: the result's start value
    ("fp64", False, 9, 4, 4, 2, 1),
    # row maxima, column maxima, digits and product of C, of C^T, rows
    ("ozaki", True, 9, 4, 4, 7, 1)])
def test_batch_node_count(fqe, contraction, group, norb, na, nb, kernels,
                          extra, nterms):
    """fqehip_batch_nodes is the number of launches of the recorded graph:
    `kernels` for the apply and each term, `extra` beside them."""
    import torch
    from fqe_amd import batched, settings
    rng = numpy.random.default_rng(5)
    h1, h2 = fo.synthetic_hamiltonian(norb, norb, rng)
    g = fo.OracleGraph(na, nb, norb)
    spec = batched.SectorSpec(norb=norb, nalpha=na, nbeta=nb, h1=h1, h2=h2,
                              coeff=fo.synthetic_coeff(g.lena, g.lenb, rng))
    saved = settings.ozaki_min_determinants
    settings.ozaki_min_determinants = 0
    try:
        bt = batched.BatchedTaylor([spec], 0.1, nterms=nterms,
                                   dtype=torch.complex128,
                                   tiles={f"{norb},{na},{nb}": "split"},
                                   nstreams=1, group=group,
                                   contraction=contraction)
    finally:
        settings.ozaki_min_determinants = saved
    bt.build()
    assert bt.nodes() == kernels * (nterms + 1) + extra
    bt.close()


@pytest.mark.parametrize("value", [numpy.inf, numpy.nan])
@pytest.mark.parametrize("kind,contraction,na,nb,norb", [
    ("real", "fp64", 3, 3, 6), ("real", "fp64", 5, 4, 9),
    ("complex", "fp64", 4, 4, 9), ("spin", "fp64", 4, 3, 8),
    ("real", "ozaki", 4, 5, 9)])
def test_coefficients_that_are_not_finite(fqe, kind, contraction, na, nb,
                                          norb, value):
    """One infinite or NaN coefficient: every determinant that H connects it
    with is not finite, and outside its row and column of C (the digit
    engine: and the rows that an alpha excitation reaches) the others keep
    the values they have without it (1e-13: the same sums)."""
    from fqe_amd import settings
    print(f"not finite {kind} {contraction} {value}", flush=True)
    d, c, g, rng = sector(fqe, na, nb, norb, 5 * norb + na)
    h = tensors(kind, norb, rng)
    op = prepared(fqe, kind, h, norb)
    ia, ib = c.shape[0] // 3, c.shape[1] // 2

    def apply(x):
        e = copy.deepcopy(d)
        e.coeff = x
        e.apply_inplace_scaled(h, op=op)
        return e.coeff
    unit = numpy.zeros_like(c)
    unit[ia, ib] = 1.0
    connected = numpy.abs(apply(unit)) > 1e-12
    bad = c.copy()
    bad[ia, ib] = value
    clean = c.copy()
    clean[ia, ib] = 0.0
    want = apply(clean)
    saved = settings.contraction, settings.ozaki_min_determinants
    settings.contraction, settings.ozaki_min_determinants = contraction, 0
    try:
        got = apply(bad)
    finally:
        settings.contraction, settings.ozaki_min_determinants = saved
    assert not numpy.isfinite(got[connected]).any()
    rest = ~connected
    rest[ia, :] = rest[:, ib] = False
    if contraction == "ozaki":
        rest[connected.any(axis=1), :] = False
    assert rest.any()
    tol = 3e-11 if contraction == "ozaki" else 1e-13
    assert rel(got[rest], want[rest]) < tol


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("na,nb,norb", [(4, 3, 8), (3, 5, 9), (6, 1, 12)])
def test_series_in_digits(fqe, na, nb, norb, graph):
    """A Taylor series on the digit kernels (norm test in its own launch,
    second term buffer behind the digit planes) against the FP64 one: the
    same number of terms, and 3e-11 as for one apply (each term's error is
    that of its apply, and the terms after the first few are small)."""
    from fqe_amd import settings
    print(f"series in digits {na} {nb} {norb} {graph}", flush=True)
    rng = numpy.random.default_rng(50 * norb + na)
    h1, h2 = fo.synthetic_hamiltonian(norb, norb, rng)
    ham = fqe.get_restricted_hamiltonian((h1, h2))
    d, c, g, rng = sector(fqe, na, nb, norb, 7)
    key = (na + nb, na - nb)
    wfn = fqe.Wavefunction([[na + nb, na - nb, norb]])
    wfn.set_wfn("from_data", {key: c / numpy.linalg.norm(c)})
    want = wfn.time_evolve(0.05, ham)
    saved = (settings.contraction, settings.ozaki_min_determinants,
             settings.taylor_graph)
    settings.contraction, settings.ozaki_min_determinants = "ozaki", 0
    settings.taylor_graph = graph
    try:
        for _ in range(2):
            got = wfn.time_evolve(0.05, ham)
            assert got._taylor_terms == want._taylor_terms
            assert rel(got.get_coeff(key), want.get_coeff(key)) < 3e-11
            assert not numpy.array_equal(got.get_coeff(key),
                                         want.get_coeff(key))
    finally:
        (settings.contraction, settings.ozaki_min_determinants,
         settings.taylor_graph) = saved


@pytest.mark.parametrize("kind", ["real", "nonsymmetric", "complex"])
@pytest.mark.parametrize("nele,norb", [
    (0, 3), (1, 1), (1, 2), (2, 3), (3, 3), (0, 6), (6, 6), (0, 8), (8, 8),
    (3, 6), (4, 8), (1, 8), (7, 8), (2, 9), (6, 9), (5, 10)])
def test_spin_block_elements(fqe, kind, nele, norb):
    """Every element of fqehip_spin_block against the same sum of dense
    pair matrices, from the library's forward table, in numpy: no, one and
    two excitations, empty and full shells, shells of one electron or one
    hole, and 36 pairs as 8 compressed or 6 plain orbitals.  1e-13 of the
    largest element (sums of at most norb^2 + 4 norb products)."""
    from fqe_amd import engine
    from fqe_amd.fci_graph import FciGraph
    print(f"spin block {kind} {nele} {norb}", flush=True)
    rng = numpy.random.default_rng(100 * norb + nele)
    op = prepared(fqe, kind, tensors(kind, norb, rng), norb)
    tab = FciGraph(nele, nele, norb).tables(True)
    got = op._spin_block(tab, True).cpu().numpy().T       # by target, source
    fwd = tab.fused_tables(op.compressed)[0].cpu().numpy()
    a = op.a.cpu().numpy()
    if op.complex_op:
        a = a[::2, ::2] + 1j * a[1::2, ::2]
    n = tab.length
    pair = numpy.zeros((op.npair, n, n))
    p, src = numpy.nonzero(fwd)
    f = fwd[p, src]
    pair[p, numpy.abs(f) - 1, src] = numpy.sign(f)
    want = numpy.einsum("q,qij->ij", a[-1], pair)
    for q in range(op.npair):
        want = want + numpy.einsum("p,pij->ij", a[:-1, q], pair) @ pair[q]
    scale = max(numpy.abs(want).max(), 1e-300)
    assert numpy.abs(got - want).max() <= 1e-13 * scale


@pytest.mark.parametrize("na,nb,norb", [(1, 5, 10), (1, 6, 13), (2, 5, 11),
                                        (2, 6, 12), (0, 5, 10), (10, 4, 10)])
def test_digit_rows_in_segments(fqe, na, nb, norb):
    """Few alpha strings and several 128-column chunks: a row's chunks are
    shared among workgroups (two, all, uneven shares, and a single row), in
    every form of the epilogue and in a Taylor series.  Tolerance and bits
    as in test_digit_rows_edges and test_series_in_digits."""
    import torch
    from fqe_amd import _lib, engine, settings
    print(f"digit segments {na} {nb} {norb}", flush=True)
    d, c, g, rng = sector(fqe, na, nb, norb, 11 * norb + 5 * na + nb)
    h = tensors("real", norb, rng)
    op = prepared(fqe, "real", h, norb)
    graph, x = d.get_fcigraph(), d.device_coeff()
    key = (na + nb, na - nb)
    wfn = fqe.Wavefunction([[na + nb, na - nb, norb]])
    wfn.set_wfn("from_data", {key: c / numpy.linalg.norm(c)})
    ham = fqe.get_restricted_hamiltonian(h)

    def run():
        out = torch.empty_like(x)
        acc = torch.ones_like(x)
        engine.apply_sector(graph, x, op, out, alpha=0.5 - 2j, beta=1.5j,
                            cin=x, acc=torch.view_as_real(acc))
        inplace = x.clone()
        n = engine.norm_partials_count(x.numel())
        part = torch.zeros(max(n, 1), dtype=torch.float64, device=x.device)
        engine.apply_sector(graph, inplace, op, inplace, alpha=2.0,
                            partials=part)
        ev = wfn.time_evolve(0.05, ham)
        return [t.cpu().numpy() for t in (out, acc, inplace)] + [
            ev.get_coeff(key), numpy.sqrt(part.sum().item())], \
            ev._taylor_terms
    want, terms = run()
    saved = settings.contraction, settings.ozaki_min_determinants
    settings.contraction, settings.ozaki_min_determinants = "ozaki", 0
    try:
        s, keep = engine.sector_struct(graph, op, _lib.C128)
        assert s.w_oz and s.haa_oz and s.hbb_oz
        got, got_terms = run()
        again, _ = run()
    finally:
        settings.contraction, settings.ozaki_min_determinants = saved
    assert got_terms == terms
    for a, b, w in zip(got, again, want):
        assert rel(a, w) < 3e-11
        assert numpy.array_equal(a, b)


def test_which_sectors_run_on_digits(fqe):
    """The rule at the sizes beside its measured crossings."""
    from fqe_amd import settings
    for lena, lenb, digits in (
            (462, 462, False), (220, 924, False), (364, 1001, True),
            (792, 792, True), (13, 1716, True), (66, 924, False),
            (91, 2002, True), (3432, 14, False), (3432, 91, False),
            (6435, 15, False), (6435, 105, True)):
        assert settings.runs_digits(lena, lenb) == digits, (lena, lenb)


def test_batch_items_that_share_scratch(fqe):
    """One branch runs its items one after another, so they may share the
    term buffer and the workspace; a group's launches run them at once, so
    those items stay out of it.  Against items with buffers of their own,
    1e-13 as in test_batch_terms."""
    import ctypes
    import torch
    from fqe_amd import _lib, batched
    rng = numpy.random.default_rng(8)
    shapes = [(8, 4, 4), (7, 3, 4), (9, 4, 4), (6, 3, 3), (8, 4, 3)]
    specs = []
    for norb, na, nb in shapes:
        h1, h2 = fo.synthetic_hamiltonian(norb, norb, rng)
        g = fo.OracleGraph(na, nb, norb)
        specs.append(batched.SectorSpec(
            norb=norb, nalpha=na, nbeta=nb, h1=h1, h2=h2,
            coeff=fo.synthetic_coeff(g.lena, g.lenb, rng)))
    tiles = {f"{n},{a},{b}": "split" for n, a, b in shapes}
    own = batched.BatchedTaylor(specs, 0.1, nterms=4, dtype=torch.complex128,
                                tiles=tiles, nstreams=2)
    own.build()
    own.launch()
    want = own.results()
    bt = batched.BatchedTaylor(specs, 0.1, nterms=4, dtype=torch.complex128,
                               tiles=tiles, nstreams=1)
    items = [p.item() for p in bt.sectors]
    ws = max((p.ws for p in bt.sectors[:4]), key=lambda t: t.numel())
    term = max((p.term for p in bt.sectors[:4]), key=lambda t: t.numel())
    for it in items[:4]:                     # the last keeps its own
        it.d_workspace, it.d_term = _lib.ptr(ws), _lib.ptr(term)
    handle = ctypes.c_void_p()
    torch.cuda.synchronize()
    _lib.call("fqehip_batch_create", bt.prec, len(items),
              (_lib.BatchItem * len(items))(*items), bt.time, 4, 1, 1,
              _lib.stream_ptr(), ctypes.byref(handle))
    bt._batch = handle
    for _ in range(2):
        bt.launch()
        for (a0, e0), (a1, e1) in zip(bt.results(), want):
            assert rel(a0, a1) < 1e-13 and rel(e0, e1) < 1e-13
    own.close()
    bt.close()
