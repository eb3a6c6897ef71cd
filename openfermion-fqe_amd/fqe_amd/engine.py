"""Device form of the operator and the per-sector apply / Taylor drivers.

The operator of a spatial (h1, h2) tuple is put in the dvec form the
reference's Python path uses (``src/fqe/fqe_data.py:646-683``):

    H C = sum_ij h1'[i,j] E_ij C + sum_ijkl V[ij,kl] E_ij E_kl C,
    V[i,j,k,l] = -h2[i,k,j,l],  h1' = h1 - einsum('ikkj', V).

Pair basis.  When V[ij,kl] = V[ji,kl] = V[ij,lk] and h1' is symmetric
(real molecular integrals) the n(n+1)/2 unordered pairs carry the same
operator exactly (reference ``:659-681`` assumes this for any real h; here
it is checked, so a real non-symmetric h takes the ordered n^2 basis and
matches the reference's C path).  GEMM matrix A: rows = output pairs plus
one row for h1', columns = input pairs; complex operators use the real
2x2-block form [[Re, -Im], [Im, Re]] on the planar (re, im) dvec.
"""

from __future__ import annotations

from typing import Optional, Sequence, Tuple

import numpy
import torch

from . import _lib
from . import settings


class PreparedOperator:
    """GEMM matrix (2-body) or pair vector (1-body) on the device."""

    def __init__(self, norb: int, compressed: bool, complex_op: bool,
                 a: Optional[torch.Tensor], h1: Optional[torch.Tensor],
                 spin: bool = False):
        self.norb = norb
        self.compressed = compressed
        self.complex_op = complex_op
        self.a = a
        self.h1 = h1
        # spin: pairs of alpha orbitals, then pairs of beta orbitals
        self.spin = spin
        self.npair = (2 * norb * norb if spin else
                      norb * (norb + 1) // 2 if compressed else norb * norb)
        # A[p][q] == A[q][p] exactly (p, q < npair): the split apply applies
        self.pair_symmetric = False
        # opposite-spin coupling W[p][q] = V[p][q] + V[q][p] (device, alpha
        # pair p, beta pair q) of a two-body operator: the pull form
        self.coupling: Optional[torch.Tensor] = None
        self.coupling_host: Optional[numpy.ndarray] = None
        self._in_range: Optional[bool] = None
        on = a if a is not None else h1
        self._tables = _lib.TableCache(on.device)

    def beta_block(self, graph):
        """Beta-beta block of this operator on the beta strings of
        ``graph`` (fqehip_beta_block): (bfloat16 hi, bfloat16 lo, ldh, beta
        forward table, FP64 columns, the GEMM matrix), cached per nbeta;
        None when the split apply does not apply."""
        if not self.pair_symmetric or self.a is None or self.complex_op:
            return None
        lenb = graph.lenb()
        if (lenb + self.npair) * 8 > 160 * 1024:
            return None
        return self._tables.get(("hbb", graph.nbeta()), self._build_hbb,
                                graph.tables(False))

    def _build_hbb(self, tables):
        lenb = tables.length
        fwb, _ = tables.fused_tables(self.compressed)
        ldh = int(_lib.call("fqehip_beta_block_ld", lenb))
        hcol = torch.empty((lenb, lenb), dtype=torch.float64,
                           device=self.a.device)
        hhi = torch.empty((ldh, ldh), dtype=torch.int16, device=self.a.device)
        hlo = torch.empty_like(hhi)
        _lib.call("fqehip_beta_block", self.npair, lenb, _lib.ptr(fwb),
                  _lib.ptr(self.a), _lib.ptr(hcol), _lib.ptr(hhi),
                  _lib.ptr(hlo), ldh, _lib.stream_ptr())
        return hhi, hlo, ldh, fwb, hcol, self.a

    def pull_digits(self, graph):
        """Digits of the pull form (W, Haa, Hbb; fqehip_pull_digits and
        fqehip_beta_block_digits) on the sector of ``graph``, cached per
        electron count; None where the digit kernels do not apply."""
        tabs = self.pull_tables(graph)
        if (tabs is None or self.complex_op or self.spin
                or not self.pair_symmetric or self.coupling.shape[0] > 128
                or max(graph.lena(), graph.lenb()) >= 26214
                or not self._digit_range()):
            return None
        return [self._tables.get("w_oz", self._build_coupling_digits)] + [
            self._tables.get(("digits", nele), self._build_block_digits, block)
            for nele, block in ((graph.nalpha(), tabs[1]),
                                (graph.nbeta(), tabs[2]))]

    def _digit_range(self) -> bool:
        """Whether W's digits resolve its rows.  Their products are summed as
        integers whose unit can be as fine as 2^-62 sum |W|: down to rows
        whose largest element is 2^-23 sum |W| that is finer than the row's
        own 38-bit digits (integrals of canonical orbitals: 2^-10 to 2^-14).
        Beside one integral 10^7 times the others, as a penalty on an
        orbital, the typical row is past that, and the sector runs in
        FP64."""
        if self._in_range is None:
            w = numpy.abs(self.coupling_host)
            rows = w.max(axis=0, initial=0.0)
            rows = rows[rows > 0.0]
            self._in_range = (rows.size == 0 or
                              bool(w.sum() <= 2.0**23 * numpy.median(rows)))
        return self._in_range

    def _build_coupling_digits(self) -> torch.Tensor:
        npull = self.coupling.shape[0]
        woz = torch.empty(int(_lib.call("fqehip_pull_digits_bytes", npull)),
                          dtype=torch.uint8, device=self.a.device)
        _lib.call("fqehip_pull_digits", npull, _lib.ptr(self.coupling),
                  _lib.ptr(woz), _lib.stream_ptr())
        return woz

    def _build_block_digits(self, block: torch.Tensor) -> torch.Tensor:
        n = block.shape[0]
        nbytes = int(_lib.call("fqehip_beta_block_digits_bytes", n))
        hoz = torch.empty(max(nbytes, 16), dtype=torch.uint8,
                          device=self.a.device)
        _lib.call("fqehip_beta_block_digits", n, _lib.ptr(block),
                  _lib.ptr(hoz), _lib.stream_ptr())
        return hoz

    def _spin_block(self, tables, alpha: bool) -> torch.Tensor:
        """Matrix of this two-body operator on the strings of one spin, by
        source string (fqehip_spin_block)."""
        n, npull = tables.length, self.coupling.shape[0]
        w = 2 if self.complex_op else 1
        lda = self.a.shape[1]
        # spin-orbital operators: the beta block of A follows the alpha one
        first = w * npull if self.spin and not alpha else 0
        fwd, _ = tables.fused_tables(self.compressed)
        out = torch.empty((n, n), device=self.a.device,
                          dtype=torch.complex128 if self.complex_op else
                          torch.float64)
        pairs = _lib.ptr(self.a) + 8 * first * (lda + 1)
        one_body = _lib.ptr(self.a) + 8 * (w * self.npair * lda + first)
        _lib.call("fqehip_spin_block", int(self.complex_op), npull, n,
                  _lib.ptr(fwd), pairs, lda, one_body, _lib.ptr(out),
                  _lib.stream_ptr())
        return out

    def pull_tables(self, graph):
        """(W, Haa, Hbb, beta target words, alpha de-excitation rows) of
        the pull form on the sector of ``graph``, cached per (nalpha,
        nbeta); None where the form does not apply (one-body operators,
        sectors past its limits)."""
        if self.coupling is None:
            return None
        return self._tables.get((graph.nalpha(), graph.nbeta()),
                                self._build_pull, graph)

    def _build_pull(self, graph):
        limits = _lib.Sector(graph.norb(), graph.nalpha(), graph.nbeta(),
                             self.npair, graph.lena(), graph.lenb())
        limits.npull = self.coupling.shape[0]
        if not _lib.call("fqehip_pull_fits_supported", _as_ref(limits),
                         int(self.complex_op)):
            return None
        ta, tb = graph.tables(True), graph.tables(False)
        # restricted operators: one matrix per electron count
        haa, hbb = (
            self._tables.get(("side", alpha if self.spin else None, tab.nele),
                             self._spin_block, tab, alpha)
            for tab, alpha in ((ta, True), (tb, False)))
        return (self.coupling, haa, hbb, tb.pull_table(self.compressed),
                ta.dexc)

    def c_struct(self) -> _lib.Operator:
        return _lib.Operator(int(self.complex_op), _lib.ptr(self.a),
                             _lib.ptr(self.h1))


def _pair_indices(norb: int, compressed: bool):
    """(i, j) of each pair-basis index (representative i >= j when
    compressed, index j + i(i+1)/2)."""
    if compressed:
        return [(i, j) for i in range(norb) for j in range(i + 1)]
    return [(i, j) for i in range(norb) for j in range(norb)]


def _is_pair_symmetric(h1p: numpy.ndarray, v: numpy.ndarray) -> bool:
    return (numpy.array_equal(v, v.transpose(1, 0, 2, 3))
            and numpy.array_equal(v, v.transpose(0, 1, 3, 2))
            and numpy.array_equal(h1p, h1p.T))


def prepare_operator(tensors: Sequence[numpy.ndarray], norb: int,
                     device: torch.device) -> PreparedOperator:
    """Device form of a 1- or 2-tensor spatial operator."""
    if len(tensors) == 1:
        h1 = numpy.asarray(tensors[0], dtype=numpy.complex128)
        if h1.shape != (norb, norb):
            raise ValueError("Inconsistent number of spin-orbitals in "
                             "operators and wavefunction.")
        compressed = numpy.array_equal(h1, h1.T)
        pairs = _pair_indices(norb, compressed)
        vec = numpy.array([h1[i, j] for i, j in pairs], dtype=numpy.complex128)
        d = torch.from_numpy(vec.view(numpy.float64).copy()).to(device)
        return PreparedOperator(norb, compressed, bool(numpy.any(vec.imag)),
                                None, d)
    if len(tensors) != 2:
        raise ValueError("the GPU engine applies 1- and 2-body restricted "
                         "operators")
    h1e, h2e = tensors
    if h1e is None:
        h1e = numpy.zeros((norb, norb))
    h1e = numpy.asarray(h1e)
    h2e = numpy.asarray(h2e)
    assert h1e.shape == (norb, norb)
    assert h2e.shape == (norb, norb, norb, norb)
    v = -numpy.moveaxis(h2e.astype(numpy.complex128), 1, 2)
    h1p = h1e.astype(numpy.complex128) - numpy.einsum("ikkj->ij", v)
    compressed = _is_pair_symmetric(h1p, v)
    complex_op = bool(numpy.any(v.imag) or numpy.any(h1p.imag))
    pairs = _pair_indices(norb, compressed)
    rows = [i * norb + j for i, j in pairs]
    vm = v.reshape(norb * norb, norb * norb)[numpy.ix_(rows, rows)]
    h1row = h1p.reshape(-1)[rows]
    full = numpy.vstack([vm, h1row[None, :]])  # (npair+1) x npair, complex
    a = _real_block_form(full, complex_op)
    w = vm + vm.T
    dev_a, coupling = _upload(a, w, complex_op, device)
    prepared = PreparedOperator(norb, compressed, complex_op, dev_a, None)
    prepared.coupling, prepared.coupling_host = coupling, w
    if not complex_op:
        sq = a[:-1, :]
        prepared.pair_symmetric = bool(numpy.array_equal(sq, sq.T))
    return prepared


def _upload(a: numpy.ndarray, w: numpy.ndarray, complex_op: bool,
            device: torch.device) -> Tuple[torch.Tensor, torch.Tensor]:
    """The GEMM matrix and the coupling (real unless complex_op) on the
    device, in one transfer."""
    dtype = numpy.complex128 if complex_op else numpy.float64
    w = numpy.ascontiguousarray(w if complex_op else w.real, dtype=dtype)
    flat = numpy.concatenate([numpy.asarray(a, dtype=numpy.float64).ravel(),
                              w.view(numpy.float64).ravel()])
    dev = torch.from_numpy(flat).to(device)
    dev_w = dev[a.size:]
    if complex_op:
        dev_w = torch.view_as_complex(dev_w.reshape(-1, 2))
    return dev[:a.size].reshape(a.shape), dev_w.reshape(w.shape)


def _real_block_form(full: numpy.ndarray, complex_op: bool) -> numpy.ndarray:
    """The GEMM matrix of a complex (npair+1) x npair operator: itself when
    real, else the real 2 x 2 block form on planar (re, im) rows."""
    if not complex_op:
        return numpy.ascontiguousarray(full.real)
    m, k = full.shape
    a = numpy.zeros((2 * m, 2 * k))
    a[0::2, 0::2] = full.real
    a[0::2, 1::2] = -full.imag
    a[1::2, 0::2] = full.imag
    a[1::2, 1::2] = full.real
    return a


def prepare_spin_operator(tensors: Sequence[numpy.ndarray], norb: int,
                          device: torch.device) -> PreparedOperator:
    """Device form of a 1- or 2-tensor spin-orbital operator (2 norb
    spin orbitals, alpha first) applied to one (nalpha, nbeta) sector, in
    the reference's dvec form with separate alpha and beta dvecs
    (``src/fqe/fqe_data.py:533-583`` one-body, ``:712-741`` two-body):

        out = sum_ij h1'aa[i,j] Da[i,j] + h1'bb[i,j] Db[i,j]
              + sum_ij E^a_ij Ya[i,j] + E^b_ij Yb[i,j],
        Ya = V'aaaa Da + V'aabb Db,  Yb = V'bbaa Da + V'bbbb Db,

    with V' = -moveaxis(h2e, 1, 2) and h1' = h1e - sum_k V'[i,k,k,j] over
    all 2 norb spin orbitals.  Only the spin-conserving blocks enter, as in
    the reference; the alpha-beta blocks of h1e are not used.  The pair
    basis is the full norb^2 basis of each spin, alpha pairs first: a
    (2 norb^2 + 1) x 2 norb^2 GEMM matrix (the last row h1'), or a pair
    vector for a one-body operator."""
    n = norb
    m = 2 * n
    npair = n * n
    if len(tensors) == 1:
        h1 = numpy.asarray(tensors[0], dtype=numpy.complex128)
        if h1.shape != (m, m):
            raise ValueError("Inconsistent number of spin-orbitals in "
                             "operators and wavefunction.")
        vec = numpy.concatenate([h1[:n, :n].reshape(-1),
                                 h1[n:, n:].reshape(-1)])
        d = torch.from_numpy(vec.view(numpy.float64).copy()).to(device)
        return PreparedOperator(norb, False, bool(numpy.any(vec.imag)), None,
                                d, spin=True)
    if len(tensors) != 2:
        raise ValueError("the GPU engine applies 1- and 2-body spin-orbital "
                         "operators to spin-conserving sectors")
    h1e, h2e = tensors
    if h1e is None:
        h1e = numpy.zeros((m, m))
    h1e = numpy.asarray(h1e)
    h2e = numpy.asarray(h2e)
    assert h1e.shape == (m, m)
    assert h2e.shape == (m, m, m, m)
    v = -numpy.moveaxis(h2e.astype(numpy.complex128), 1, 2)
    h1p = h1e.astype(numpy.complex128) - numpy.einsum("ikkj->ij", v)
    vm = numpy.zeros((2 * npair, 2 * npair), dtype=numpy.complex128)
    for s in range(2):
        for t in range(2):
            vm[s * npair:(s + 1) * npair, t * npair:(t + 1) * npair] = \
                v[s * n:(s + 1) * n, s * n:(s + 1) * n,
                  t * n:(t + 1) * n, t * n:(t + 1) * n].reshape(npair, npair)
    h1row = numpy.concatenate([h1p[:n, :n].reshape(-1),
                               h1p[n:, n:].reshape(-1)])
    full = numpy.vstack([vm, h1row[None, :]])
    complex_op = bool(numpy.any(full.imag))
    w = vm[:npair, npair:] + vm[npair:, :npair].T
    dev_a, coupling = _upload(_real_block_form(full, complex_op), w,
                              complex_op, device)
    prepared = PreparedOperator(norb, False, complex_op, dev_a, None,
                                spin=True)
    prepared.coupling = coupling
    return prepared


def precision_of(dtype: torch.dtype) -> int:
    if dtype == torch.complex128:
        return _lib.C128
    if dtype == torch.complex64:
        return _lib.C64
    raise TypeError(f"unsupported coefficient dtype {dtype}")


def sector_struct(graph, op: PreparedOperator,
                  precision: Optional[int] = None
                  ) -> Tuple[_lib.Sector, tuple]:
    """C descriptor of a sector for the pair basis of ``op``; the second
    element keeps the tables referenced.  For a pair-symmetric operator the
    beta-beta block is attached (split apply): its bfloat16 hi/lo split for
    complex64 (``settings.split``), its FP64 columns for complex128
    (``settings.split_fp64``).  Two-body operators in complex128 get the
    tables of the pull form, unless the digit engine or another kernel is
    asked for (``settings.contraction``, ``split_tile_fp64``)."""
    if op.spin:
        ta = graph.tables(True).spin_pair_table(True)
        tb = graph.tables(False).spin_pair_table(False)
    else:
        ta = graph.tables(True).pair_table(op.compressed)
        tb = graph.tables(False).pair_table(op.compressed)
    keep = [ta, tb]
    fwa = fwb = sla = None
    if settings.fused and not op.complex_op and op.h1 is None and not op.spin:
        fwa, sla = graph.tables(True).fused_tables(op.compressed)
        fwb, _ = graph.tables(False).fused_tables(op.compressed)
        keep += [fwa, fwb, sla]
    nslot = graph.nalpha() * (graph.norb() - graph.nalpha())
    hbb = hbb64 = None
    if fwa is not None and settings.split and precision == _lib.C64:
        hbb = op.beta_block(graph)
    # split kernel limits: gather depth npair + 1 <= 128 (112 for the FP64
    # shared-D-tile variant), at most 64 live pair rows (norb^2/4 + 1)
    kmax = 112 if (settings.contraction == "fp64" and
                   settings.split_tile_fp64 == _lib.TILE_SPLIT_F64_DTILE) else 128
    pull = None
    if (settings.fused and settings.split_fp64 and op.h1 is None
            and precision == _lib.C128
            and (settings.split_tile_fp64 is None
                 or settings.contraction == "ozaki")):
        pull = op.pull_tables(graph)
    if (fwa is not None and settings.split_fp64 and precision == _lib.C128
            and op.npair + 1 <= kmax and graph.norb() ** 2 // 4 + 1 <= 64):
        if pull is not None and op.pair_symmetric:
            hbb64 = pull[2]          # the same matrix
        else:
            blk = op.beta_block(graph)
            hbb64 = blk[4] if blk else None
    s = _lib.Sector(graph.norb(), graph.nalpha(), graph.nbeta(), op.npair,
                    graph.lena(), graph.lenb(), _lib.ptr(ta), _lib.ptr(tb),
                    _lib.ptr(fwa), _lib.ptr(fwb), _lib.ptr(sla), nslot,
                    _lib.ptr(hbb[0]) if hbb else None,
                    _lib.ptr(hbb[1]) if hbb else None,
                    hbb[2] if hbb else 0)
    if hbb:
        keep += [hbb[0], hbb[1]]
        s.tile = int(settings.split_tile)
    if hbb64 is not None:
        keep.append(hbb64)
        s.hbb_f64 = _lib.ptr(hbb64)
        if settings.contraction == "ozaki":
            s.tile = _lib.TILE_OZAKI
            digits = None
            if settings.runs_digits(s.lena, s.lenb):
                digits = op.pull_digits(graph)
            if digits is not None:
                keep += digits
                s.w_oz = _lib.ptr(digits[0])
                if settings.ozaki_beta:
                    s.haa_oz = _lib.ptr(digits[1])
                    s.hbb_oz = _lib.ptr(digits[2])
        elif settings.contraction == "fp64":
            s.tile = int(settings.split_tile_fp64 or 0)
        else:
            raise ValueError(f"settings.contraction={settings.contraction!r}")
    if pull is not None:
        keep += pull
        s.pull_w, s.haa, s.hbb, s.pull_fwd, s.dexc_a = (
            _lib.ptr(t) if t.numel() else None for t in pull)
        s.npull = op.coupling.shape[0]
    return s, tuple(keep)


def workspace(sector: _lib.Sector, precision: int,
              device: torch.device) -> torch.Tensor:
    """Device scratch for one apply (dvec + Y planes); the one-body Taylor
    loop uses it as its second term buffer."""
    nbytes = int(_lib.lib().fqehip_apply_workspace_bytes(precision,
                                                          _as_ref(sector)))
    elem = 8 if precision == _lib.C128 else 4
    n = sector.lena * sector.lenb
    fused = (sector.nslot + 1) * 2 * n * elem
    need = max((2 * sector.npair + 1) * 2 * n * elem, fused)
    if nbytes != need and not (sector.pull_w and nbytes >= 16 * n):
        raise _lib.FqeHipError(f"workspace size {nbytes} != {need}")
    nbytes = max(nbytes, 16 * sector.lena * sector.lenb, 16)
    return torch.empty(nbytes, dtype=torch.uint8, device=device)


def needs_panels(sector: _lib.Sector, op: PreparedOperator,
                 precision: int) -> bool:
    """True for a complex128 two-body apply on the unfused kernels whose
    dvec + Y exceed settings.max_workspace_bytes."""
    if precision != _lib.C128 or op.h1 is not None:
        return False
    import ctypes
    opc = op.c_struct()
    if (_lib.lib().fqehip_pull_supported(precision, ctypes.byref(sector),
                                         ctypes.byref(opc))
            or _lib.lib().fqehip_fused_supported(precision,
                                                 ctypes.byref(sector),
                                                 ctypes.byref(opc))):
        return False
    n = sector.lena * sector.lenb
    return (2 * sector.npair + 1) * 2 * n * 8 > settings.max_workspace_bytes


def _as_ref(struct):
    import ctypes
    return ctypes.byref(struct)


def apply_sector(graph, coeff: torch.Tensor, op: PreparedOperator,
                 out: torch.Tensor, alpha: complex = 1.0, beta: complex = 0.0,
                 cin: Optional[torch.Tensor] = None,
                 acc: Optional[torch.Tensor] = None,
                 partials: Optional[torch.Tensor] = None,
                 done: Optional[torch.Tensor] = None,
                 ws: Optional[torch.Tensor] = None) -> None:
    """out = alpha * H coeff + beta * cin on one sector (device tensors).
    A complex128 sector whose unfused workspace exceeds
    ``settings.max_workspace_bytes`` runs in panels of orbital pairs."""
    prec = precision_of(coeff.dtype)
    s, keep = sector_struct(graph, op, prec)
    if ws is None and op.h1 is None and needs_panels(s, op, prec):
        nbytes = int(settings.max_workspace_bytes)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=coeff.device)
        opc = op.c_struct()
        _lib.call("fqehip_apply_panels", prec, _as_ref(s), _as_ref(opc),
                  _lib.ptr(coeff), float(numpy.real(alpha)),
                  float(numpy.imag(alpha)), float(numpy.real(beta)),
                  float(numpy.imag(beta)), _lib.ptr(cin), _lib.ptr(out),
                  _lib.ptr(acc), _lib.ptr(partials), _lib.ptr(done),
                  _lib.ptr(ws), nbytes, _lib.stream_ptr())
        del keep
        return
    if ws is None and op.h1 is None:
        ws = workspace(s, prec, coeff.device)
    opc = op.c_struct()
    _lib.call("fqehip_apply", prec, _as_ref(s), _as_ref(opc),
              _lib.ptr(coeff), float(numpy.real(alpha)),
              float(numpy.imag(alpha)), float(numpy.real(beta)),
              float(numpy.imag(beta)), _lib.ptr(cin), _lib.ptr(out),
              _lib.ptr(acc), _lib.ptr(partials), _lib.ptr(done),
              _lib.ptr(ws), _lib.stream_ptr())
    del keep


def norm_partials_count(n: int) -> int:
    return int(_lib.lib().fqehip_norm_partials_count(n))


_DOT_WS = {}


def dot128(a: torch.Tensor, b: torch.Tensor) -> complex:
    """<a|b> = sum conj(a) b over complex128 device vectors, FP64 with a
    fixed summation order (fqehip_block_dot)."""
    a = a.reshape(-1)
    b = b.reshape(-1)
    assert a.dtype == torch.complex128 and b.dtype == torch.complex128
    assert a.is_contiguous() and b.is_contiguous() and a.numel() == b.numel()
    dev = a.device
    if dev.index not in _DOT_WS:
        nbytes = int(_lib.call("fqehip_block_dot_workspace_bytes", 1))
        _DOT_WS[dev.index] = (torch.empty(nbytes, dtype=torch.uint8,
                                          device=dev),
                              torch.empty(1, dtype=torch.complex128,
                                          device=dev))
    ws, out = _DOT_WS[dev.index]
    _lib.call("fqehip_block_dot", a.numel(), 1, _lib.ptr(a), a.numel(),
              _lib.ptr(b), _lib.ptr(out), _lib.ptr(ws), _lib.stream_ptr())
    return complex(out.item())


def block_dots(rows: torch.Tensor, x: torch.Tensor) -> numpy.ndarray:
    """[sum_i conj(rows[j, i]) x[i] for j] over complex128 device data
    (fqehip_block_dot, FP64, fixed summation order)."""
    k, n = rows.shape
    assert rows.dtype == torch.complex128 and x.dtype == torch.complex128
    assert rows.is_contiguous() and x.is_contiguous() and x.numel() == n
    ws = torch.empty(max(int(_lib.call("fqehip_block_dot_workspace_bytes",
                                       k)), 16),
                     dtype=torch.uint8, device=rows.device)
    out = torch.empty(k, dtype=torch.complex128, device=rows.device)
    _lib.call("fqehip_block_dot", n, k, _lib.ptr(rows), n, _lib.ptr(x),
              _lib.ptr(out), _lib.ptr(ws), _lib.stream_ptr())
    return out.cpu().numpy()


def gram(a: torch.Tensor, b: torch.Tensor) -> numpy.ndarray:
    """G[p, q] = sum_i conj(a[p, i]) b[q, i] for complex128 device blocks
    a, b of shape [k, n] (fqehip_gram, FP64 matrix cores)."""
    k, n = a.shape
    assert b.shape == (k, n)
    assert a.dtype == torch.complex128 and b.dtype == torch.complex128
    assert a.is_contiguous() and b.is_contiguous()
    ws = torch.empty(max(int(_lib.call("fqehip_gram_workspace_bytes", n, k)),
                         16), dtype=torch.uint8, device=a.device)
    out = torch.empty((k, k), dtype=torch.complex128, device=a.device)
    _lib.call("fqehip_gram", n, k, _lib.ptr(a), _lib.ptr(b), _lib.ptr(out),
              _lib.ptr(ws), _lib.stream_ptr())
    return out.cpu().numpy()


def planar_rows(npair: int, vec: torch.Tensor) -> torch.Tensor:
    """[npair + 1, 2, n] planes for the dvec of a vector, the vector itself
    in the last row (real parts, then imaginary parts)."""
    real = (torch.float64 if vec.dtype == torch.complex128
            else torch.float32)
    d = torch.empty((npair + 1, 2, vec.numel()), dtype=real,
                    device=vec.device)
    d[npair].copy_(torch.view_as_real(vec.reshape(-1)).T)
    return d


def gram_planar(a: torch.Tensor, b: torch.Tensor) -> numpy.ndarray:
    """``gram`` of planar FP64 blocks [k, 2, n] (fqehip_gram_planar); half
    of the products if a and b are the same block."""
    k, _, n = a.shape
    assert b.shape == (k, 2, n)
    assert a.dtype == torch.float64 and b.dtype == torch.float64
    assert a.is_contiguous() and b.is_contiguous()
    ws = torch.empty(max(int(_lib.call("fqehip_gram_workspace_bytes", n, k)),
                         16), dtype=torch.uint8, device=a.device)
    out = torch.empty((k, k), dtype=torch.complex128, device=a.device)
    _lib.call("fqehip_gram_planar", n, k, _lib.ptr(a), _lib.ptr(b),
              _lib.ptr(out), _lib.ptr(ws), _lib.stream_ptr())
    return out.cpu().numpy()


def rdm12(d2: torch.Tensor, d: torch.Tensor, m: int
          ) -> Tuple[numpy.ndarray, numpy.ndarray]:
    """1- and 2-RDM in m orbitals from the planar rows of the bra's and the
    ket's dvec (m^2 pairs, then the vector): rdm1[p, q] = <E_qp bra|ket> and
    rdm2[j, k, i, l] = -<E_ij bra|E_kl ket> + delta_ki rdm1[j, l], both from
    one Gram product."""
    g = gram_planar(d2, d)
    out1 = g[:-1, -1].reshape(m, m).T
    out2 = -g[:-1, :-1].reshape((m,) * 4).transpose(1, 2, 0, 3)
    for i in range(m):
        out2[:, i, i, :] += out1
    return out1.copy(), out2.copy()

