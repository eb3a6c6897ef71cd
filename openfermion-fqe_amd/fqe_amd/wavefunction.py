"""Wavefunction: the sectors of a number- and Sz-conserving CI vector.

Mirrors ``fqe.wavefunction.Wavefunction`` for the apply path (reference
``src/fqe/wavefunction.py:49-118``, ``:241-399``, ``:509-611``,
``:613-812``, ``:961-1054``, ``:1100-1133``): same constructor, ``apply``,
``time_evolve``, ``apply_generated_unitary`` (Taylor), ``norm``,
``normalize``, ``scale``, ``ax_plus_y``, ``set_wfn``, ``get_coeff``,
``expectationValue`` and error behaviour (``TypeError`` for number-
conservation mismatches, ``ValueError`` for sizes, ``RuntimeError`` when
the Taylor series does not converge).
"""

from __future__ import annotations

import copy
import json
import os
import math
from typing import Dict, KeysView, List, Optional, Tuple, Union

import numpy
import torch

from . import _lib
from . import engine
from . import settings
from .fqe_data import FqeData
from .fqe_data_set import FqeDataSet
from .hamiltonians import (Hamiltonian, RestrictedHamiltonian, General,
                           GSOHamiltonian, _SpinOrbitalHamiltonian)
from .util import alpha_beta_electrons, validate_tuple, vdot


def build_hamiltonian(ops, norb: int = 0, conserve_number: bool = True,
                      e_0: complex = 0. + 0.j) -> Hamiltonian:
    """Tuple -> RestrictedHamiltonian (reference
    ``src/fqe/fqe_decorators.py:45-72``)."""
    if isinstance(ops, Hamiltonian):
        return ops
    if isinstance(ops, tuple):
        validate_tuple(ops)
        if norb != 0 and ops[0].shape[0] == norb:
            out = RestrictedHamiltonian(ops, e_0=e_0)
        else:
            out = General(ops, e_0=e_0)
        out._conserve_number = conserve_number
        return out
    raise TypeError('Expected FermionOperator'
                    ' but received {}.'.format(type(ops)))


class Wavefunction:
    """reference ``src/fqe/wavefunction.py:49``"""

    def __init__(self, param: Optional[List[List[int]]] = None,
                 broken: Optional[Union[List[str], str]] = None,
                 dtype=None) -> None:
        self._symmetry_map: Dict[Tuple[int, int], Tuple[int, int]] = {}
        self._conserved: Dict[str, int] = {}
        self._conserve_spin = broken is None or 'spin' not in broken
        self._conserve_number = broken is None or 'number' not in broken
        self._norb = 0
        self._civec: Dict[Tuple[int, int], FqeData] = {}
        self._dtype = numpy.dtype(dtype if dtype is not None
                                  else settings.default_dtype)
        if not self._conserve_spin and not self._conserve_number:
            raise TypeError('Number and spin non-conserving waveunfction is'
                            ' the complete Fock space.')
        if not self._conserve_number:
            raise NotImplementedError(
                "number-broken wavefunctions are outside the GPU engine's "
                "path")
        if param:
            norbs = set(x[2] for x in param)
            if len(norbs) != 1:
                raise ValueError('Number of orbitals is not consistent')
            self._norb = list(norbs)[0]
            for p in param:
                nalpha, nbeta = alpha_beta_electrons(p[0], p[1])
                self._civec[(p[0], p[1])] = FqeData(nalpha, nbeta, self._norb,
                                                    dtype=self._dtype)
            self._conserved['n'] = param[0][0]
            if self._conserve_spin:
                self._conserved['s_z'] = param[0][1]

    # -- containers ------------------------------------------------------------
    def sector(self, key: Tuple[int, int]) -> FqeData:
        return self._civec[key]

    def sectors(self) -> KeysView[Tuple[int, int]]:
        return self._civec.keys()

    def conserve_number(self) -> bool:
        return self._conserve_number

    def conserve_spin(self) -> bool:
        return self._conserve_spin

    def norb(self) -> int:
        return self._norb

    def get_coeff(self, key: Tuple[int, int]) -> numpy.ndarray:
        return self._civec[key].coeff

    def set_wfn(self, strategy: str = 'ones',
                raw_data: Optional[Dict[Tuple[int, int],
                                        numpy.ndarray]] = None) -> None:
        """reference ``src/fqe/wavefunction.py:779-811``"""
        if strategy == 'from_data' and not raw_data:
            raise ValueError('No data provided for set_wfn')
        if strategy == 'from_data':
            for key, data in raw_data.items():
                self._civec[key].set_wfn(strategy='from_data', raw_data=data)
        elif strategy == 'hartree-fock':
            if len(self.sectors()) != 1:
                raise ValueError(("Hartree-Fock wf initialization only works "
                                  "with single sector wavefunctions"))
            for sec in self._civec.values():
                sec.set_wfn(strategy=strategy)
        else:
            for sec in self._civec.values():
                sec.set_wfn(strategy=strategy)
        if strategy == 'random':
            self.normalize()

    def __deepcopy__(self, memodict={}) -> 'Wavefunction':
        new = Wavefunction.__new__(Wavefunction)
        new.__dict__.update({k: copy.copy(v) for k, v in self.__dict__.items()
                             if k != '_civec'})
        new._civec = {k: copy.deepcopy(v) for k, v in self._civec.items()}
        return new

    def _shared_copy(self) -> 'Wavefunction':
        """A copy whose sectors refer to this one's coefficients, for an
        apply that gives each sector new ones."""
        new = Wavefunction.__new__(Wavefunction)
        new.__dict__.update({k: copy.copy(v) for k, v in self.__dict__.items()
                             if k != '_civec'})
        new._civec = {k: v._shared_copy() for k, v in self._civec.items()}
        return new

    # -- vector algebra --------------------------------------------------------
    def norm(self) -> float:
        total = 0.0
        for sec in self._civec.values():
            total += sec.norm() ** 2
        return math.sqrt(total)

    def normalize(self) -> None:
        self.scale(1.0 / self.norm())

    def scale(self, sval: complex) -> None:
        for sec in self._civec.values():
            sec.scale(sval)

    def ax_plus_y(self, sval: complex, wfn: 'Wavefunction') -> None:
        if self._civec.keys() != wfn._civec.keys():
            raise ValueError('inconsistent sectors in Wavefunction.ax_plus_y')
        for key in self._civec:
            self._civec[key].ax_plus_y(sval, wfn._civec[key])

    # -- the hot path ------------------------------------------------------------
    def _check_number(self, hamil: Hamiltonian) -> None:
        if not self._conserve_number or not hamil.conserve_number():
            if self._conserve_number:
                raise TypeError('Number non-conserving hamiltonian passed to'
                                ' number conserving wavefunction')
            if hamil.conserve_number():
                raise TypeError('Number conserving hamiltonian passed to'
                                ' number non-conserving wavefunction')

    def apply(self, hamil) -> 'Wavefunction':
        """H|psi> for a RestrictedHamiltonian (reference
        ``src/fqe/wavefunction.py:314-364``, decorator
        ``src/fqe/fqe_decorators.py:353-370``)."""
        hamil = build_hamiltonian(hamil, norb=self.norb(),
                                  conserve_number=self.conserve_number())
        self._check_number(hamil)
        if isinstance(hamil, _SpinOrbitalHamiltonian):
            return self._apply_spin_orbital(hamil)
        if not isinstance(hamil, RestrictedHamiltonian):
            raise NotImplementedError(
                "the GPU engine applies restricted and spin-orbital "
                "(General, GSOHamiltonian) operators")
        if hamil.dim() != self._norb:
            raise ValueError('Hamiltonian has incorrect size:'
                             ' expected {}'.format(self._norb) +
                             ' provided {}'.format(hamil.dim()))
        return self._apply_array(hamil.tensors(), hamil.e_0(), hamil)

    def _apply_array(self, array, e_0: complex,
                     hamil: Optional[RestrictedHamiltonian] = None
                     ) -> 'Wavefunction':
        """out = H psi + e_0 psi (reference ``src/fqe/wavefunction.py:
        366-399``); the e_0 term is fused into the scatter epilogue."""
        op = _prepared(hamil, array, self._norb)
        # a sector without an array to apply keeps its coefficients
        out = (self._shared_copy() if any(isinstance(x, numpy.ndarray)
                                          for x in array)
               else copy.deepcopy(self))
        beta = e_0 if numpy.abs(e_0) > 1.e-15 else 0.0
        for sec in out._civec.values():
            sec.apply_inplace_scaled(array, alpha=1.0, beta=beta, op=op)
        return out

    def _number_sectors(self) -> Dict[int, FqeDataSet]:
        """Sectors grouped by particle number into FqeDataSets (reference
        ``src/fqe/wavefunction.py:442-471``); every spin sector of each
        number must be present."""
        norb = self.norb()
        out = {}
        for nele in sorted(set(key[0] for key in self._civec)):
            maxalpha = min(norb, nele)
            minalpha = nele - maxalpha
            needed = {(nele, 2 * na - nele)
                      for na in range(minalpha, maxalpha + 1)}
            if set(self._civec.keys()).intersection(needed) != needed:
                raise ValueError('Wave function space is not spin complete.')
            sectors = {(na, nele - na): self._civec[(nele, 2 * na - nele)]
                       for na in range(minalpha, maxalpha + 1)}
            out[nele] = FqeDataSet(nele, norb, sectors)
        return out

    def _apply_spin_orbital(self, hamil) -> 'Wavefunction':
        """H|psi> for spin-orbital tensors (reference
        ``src/fqe/wavefunction.py:349-357``, ``:366-399``): on a
        spin-conserving wavefunction each sector takes the spin-orbital
        apply of its spin-conserving blocks (``FqeData._apply_array_spin1``
        / ``_apply_array_spin12``); on a spin-broken one each particle
        number's FqeDataSet takes the apply; then e_0 psi is added."""
        expected = self._norb * 2
        if hamil.dim() != expected:
            raise ValueError('Hamiltonian has incorrect size:'
                             ' expected {}'.format(expected) +
                             ' provided {}'.format(hamil.dim()))
        if self._conserve_spin:
            if len(hamil.tensors()) > 2:
                raise NotImplementedError(
                    "the GPU engine applies 1- and 1+2-body operators; 3- "
                    "and 4-body operators are outside its path")
            return self._apply_array(hamil.tensors(), hamil.e_0(), hamil)
        out = self._shared_copy()
        beta = hamil.e_0() if numpy.abs(hamil.e_0()) > 1.e-15 else 0.0
        for nsector in out._number_sectors().values():
            nsector.apply_inplace_scaled(hamil.tensors(), beta)
        return out

    def expectationValue(self, ops, brawfn: 'Wavefunction' = None) -> complex:
        """<bra|H|self> (reference ``src/fqe/wavefunction.py:1100-1133``)."""
        if not isinstance(ops, Hamiltonian):
            raise TypeError('Expected an Fqe Hamiltonian or Operator'
                            ' but recieved {}'.format(type(ops)))
        work = self.apply(ops)
        return vdot(brawfn if brawfn else self, work)

    def time_evolve(self, time: float, hamil,
                    inplace: bool = False) -> 'Wavefunction':
        """exp(-i t H) |psi> (reference ``src/fqe/wavefunction.py:961-1054``).

        Non-quadratic restricted Hamiltonians take the Taylor branch, as in
        the reference.  Quadratic ones (h1 only), which the reference
        evolves by an orbital rotation, are evolved here with the same
        Taylor series of the one-body apply.  The e_0 phase is applied
        twice, as the reference does (``:604-605`` and ``:1051-1052``)."""
        hamil = build_hamiltonian(hamil, norb=self.norb(),
                                  conserve_number=self.conserve_number())
        assert isinstance(hamil, Hamiltonian)
        self._check_number(hamil)
        if inplace and not hamil.quadratic():
            raise ValueError("Inplace is not implemented for this case")
        work = self if inplace else copy.deepcopy(self)
        final = work.apply_generated_unitary(time, 'taylor', hamil)
        if numpy.abs(hamil.e_0()) > 1.0e-15:
            final.scale(numpy.exp(-1.j * time * hamil.e_0()))
        return final

    def apply_generated_unitary(self, time: float, algo: str, hamil,
                                accuracy: float = 1.0E-15,
                                expansion: int = 30,
                                spec_lim: Optional[List[float]] = None
                                ) -> 'Wavefunction':
        """Taylor propagation (reference ``src/fqe/wavefunction.py:509-611``):
        psi(t) = sum_k (-i t H)^k psi / k!, stopping when
        ||(-i t H)^k psi|| / k! < accuracy, else RuntimeError after
        expansion-1 terms.  The whole series runs on the device: each term
        is one fused apply whose epilogue scales by -i t / k, adds the term
        to the FP64 sum and reduces its norm; a device flag ends the series
        without host round trips."""
        hamil = build_hamiltonian(hamil, norb=self.norb(),
                                  conserve_number=self.conserve_number())
        assert isinstance(hamil, Hamiltonian)
        if not isinstance(expansion, int):
            raise TypeError(
                "expansion must be an int. You provided {}".format(expansion))
        assert algo in ['taylor', 'chebyshev']
        if isinstance(hamil, _SpinOrbitalHamiltonian):
            if algo != 'taylor':
                raise NotImplementedError(
                    "spin-orbital operators take the Taylor propagator")
            if self._conserve_spin:
                if len(hamil.tensors()) > 2:
                    raise NotImplementedError(
                        "the GPU engine applies 1- and 1+2-body operators")
                # sector by sector, the whole series on the device
                out = _taylor(self, time, hamil, accuracy, expansion)
            else:
                out = _taylor_spin_orbital(self, time, hamil, accuracy,
                                           expansion)
        elif algo == 'chebyshev':
            from .chebyshev import chebyshev_evolve
            out = chebyshev_evolve(self, time, hamil, accuracy, expansion,
                                   spec_lim)
        else:
            out = _taylor(self, time, hamil, accuracy, expansion)
        if numpy.abs(hamil.e_0() * time) > 1.e-15:
            out.scale(numpy.exp(-1.j * time * hamil.e_0()))
        return out

    # -- on-disk format -------------------------------------------------------
    # The reference pickles [symmetry map, conserved, conserve_spin,
    # conserve_number, norb, [key, FqeData]...] (src/fqe/wavefunction.py:
    # 726-765).  Here the same fields go into a versioned numpy .npz with
    # allow_pickle=False: a JSON header ("fqe_amd.wavefunction", version 1)
    # plus one complex array per sector, so reading a file executes nothing
    # from it.
    _FORMAT = "fqe_amd.wavefunction"
    _VERSION = 1

    def save(self, filename: str, path: Optional[str] = None) -> None:
        """Write the wavefunction to path/filename (reference
        ``src/fqe/wavefunction.py:748-765``)."""
        keys = list(self._civec.keys())
        header = {
            "format": self._FORMAT, "version": self._VERSION,
            "norb": self._norb, "conserve_spin": self._conserve_spin,
            "conserve_number": self._conserve_number,
            "conserved": self._conserved,
            "symmetry_map": [[list(k), list(v)]
                             for k, v in self._symmetry_map.items()],
            "dtype": str(self._dtype),
            "sectors": [[int(k[0]), int(k[1])] for k in keys],
        }
        arrays = {f"sector_{i}": numpy.ascontiguousarray(
            self._civec[k].coeff) for i, k in enumerate(keys)}
        full = os.path.join(path if path is not None else os.getcwd(),
                            filename)
        with open(full, "wb") as f:
            numpy.savez(f, header=numpy.frombuffer(
                json.dumps(header).encode(), dtype=numpy.uint8), **arrays)

    def read(self, filename: str, path: Optional[str] = None) -> None:
        """Initialise from a file written by ``save`` (reference
        ``src/fqe/wavefunction.py:726-746``), or by the reference's own
        ``save``: that file is a pickle, which is parsed without running
        anything named in it (``reference_format``)."""
        full = os.path.join(path if path is not None else os.getcwd(),
                            filename)
        with open(full, "rb") as f:
            magic = f.read(2)
        if magic[:1] == b"\x80":
            from .reference_format import read_reference_wavefunction
            with open(full, "rb") as f:
                fields = read_reference_wavefunction(f.read())
            self._norb = fields["norb"]
            self._conserve_spin = fields["conserve_spin"]
            self._conserve_number = fields["conserve_number"]
            self._conserved = dict(fields["conserved"])
            self._symmetry_map = dict(fields["symmetry_map"])
            self._civec = {}
            for (nele, m_s), coeff in fields["sectors"].items():
                nalpha, nbeta = alpha_beta_electrons(nele, m_s)
                self._dtype = numpy.dtype(coeff.dtype)
                sec = FqeData(nalpha, nbeta, self._norb, dtype=self._dtype)
                sec.coeff = coeff
                self._civec[(nele, m_s)] = sec
            return
        with numpy.load(full, allow_pickle=False) as z:
            header = json.loads(bytes(z["header"]).decode())
            if header.get("format") != self._FORMAT:
                raise ValueError(f"{full} is not a {self._FORMAT} file")
            if header.get("version") != self._VERSION:
                raise ValueError(f"unsupported {self._FORMAT} version "
                                 f"{header.get('version')}")
            self._norb = int(header["norb"])
            self._conserve_spin = bool(header["conserve_spin"])
            self._conserve_number = bool(header["conserve_number"])
            self._conserved = dict(header["conserved"])
            self._symmetry_map = {tuple(k): tuple(v)
                                  for k, v in header["symmetry_map"]}
            self._dtype = numpy.dtype(header["dtype"])
            self._civec = {}
            for i, (nele, m_s) in enumerate(header["sectors"]):
                nalpha, nbeta = alpha_beta_electrons(nele, m_s)
                sec = FqeData(nalpha, nbeta, self._norb, dtype=self._dtype)
                sec.coeff = z[f"sector_{i}"]
                self._civec[(nele, m_s)] = sec

    def print_wfn(self, threshold: float = 0.001, fmt: str = 'str') -> None:
        for key, sec in self._civec.items():
            graph = sec.get_fcigraph()
            coeff = sec.coeff
            print('Sector N = {} : S_z = {}'.format(key[0], key[1]))
            for ia in range(sec.lena()):
                for ib in range(sec.lenb()):
                    if numpy.abs(coeff[ia, ib]) > threshold:
                        a = int(graph.string_alpha(ia))
                        b = int(graph.string_beta(ib))
                        print("a'{}'b'{}' {}".format(
                            format(a, 'b').zfill(self._norb),
                            format(b, 'b').zfill(self._norb), coeff[ia, ib]))


def _prepared(hamil: Optional[Hamiltonian], array,
              norb: int) -> engine.PreparedOperator:
    """The device operator of a restricted Hamiltonian, or of spin-orbital
    tensors applied sector by sector (cached on the Hamiltonian)."""
    dev = _lib.device()
    spin = numpy.asarray(array[0]).shape[0] == 2 * norb
    prep = engine.prepare_spin_operator if spin else engine.prepare_operator
    if hamil is None:
        return prep(array, norb, dev)
    key = ("spin" if spin else "op", dev.index)
    if key not in hamil._prepared:
        hamil._prepared[key] = prep(hamil.tensors(), norb, dev)
    return hamil._prepared[key]


def _taylor_spin_orbital(wfn: Wavefunction, time: float, hamil,
                         accuracy: float, expansion: int) -> Wavefunction:
    """The reference's Taylor loop (``src/fqe/wavefunction.py:556-568``)
    over spin-orbital applies: psi(t) = sum_k (-i t H)^k psi / k!, stopping
    once ||(-i t H)^k psi|| / k! < accuracy, RuntimeError after
    expansion - 1 terms."""
    gen = General(hamil.iht(time))
    gen._conserve_number = wfn.conserve_number()
    result = copy.deepcopy(wfn)
    work = copy.deepcopy(wfn)
    for order in range(1, expansion):
        work = work._apply_spin_orbital(gen)
        coeff = 1.0 / math.factorial(order)
        result.ax_plus_y(coeff, work)
        if work.norm() * abs(coeff) < accuracy:
            break
    else:
        raise RuntimeError("maximum taylor expansion limit reached")
    return result


def _taylor(wfn: Wavefunction, time: float, hamil: RestrictedHamiltonian,
            accuracy: float, expansion: int) -> Wavefunction:
    op = _prepared(hamil, hamil.tensors(), wfn.norb())
    dev = _lib.device()
    out = copy.deepcopy(wfn)
    secs = list(out._civec.values())
    if len(secs) == 1:
        return _taylor_single(out, secs[0], op, time, accuracy, expansion)
    # several sectors: one device flag and one norm over all of them, as the
    # reference's loop tests the norm of the whole wavefunction
    terms, results, structs, wss, offs = [], [], [], [], [0]
    for sec in secs:
        c = sec.device_coeff()
        terms.append(c.clone())
        results.append(torch.view_as_real(c.to(torch.complex128).clone()))
        s, keep = engine.sector_struct(sec.get_fcigraph(), op,
                                       engine.precision_of(c.dtype))
        structs.append((s, keep))
        wss.append(engine.workspace(s, engine.precision_of(c.dtype), dev))
        offs.append(offs[-1] + engine.norm_partials_count(c.numel()))
    partials = torch.zeros(max(offs[-1], 1), dtype=torch.float64, device=dev)
    status = torch.zeros(2, dtype=torch.int32, device=dev)
    norm = torch.zeros(1, dtype=torch.float64, device=dev)
    opc = op.c_struct()
    for order in range(1, expansion):
        alpha = -1.0j * time / order
        for k, sec in enumerate(secs):
            prec = engine.precision_of(terms[k].dtype)
            if op.h1 is not None:
                nxt = torch.empty_like(terms[k])
                _lib.call("fqehip_apply1", prec, op.npair, sec.lena(),
                          sec.lenb(), structs[k][0].ptab_a,
                          structs[k][0].ptab_b, _lib.ptr(op.h1),
                          _lib.ptr(terms[k]), 0.0, alpha.imag, 0.0, 0.0, None,
                          _lib.ptr(nxt), _lib.ptr(results[k]),
                          _lib.ptr(partials[offs[k]:]), _lib.ptr(status[1:]),
                          _lib.stream_ptr())
                terms[k] = nxt
            else:
                _lib.call("fqehip_apply", prec, engine._as_ref(structs[k][0]),
                          engine._as_ref(opc), _lib.ptr(terms[k]), 0.0,
                          alpha.imag, 0.0, 0.0, None, _lib.ptr(terms[k]),
                          _lib.ptr(results[k]), _lib.ptr(partials[offs[k]:]),
                          _lib.ptr(status[1:]), _lib.ptr(wss[k]),
                          _lib.stream_ptr())
        _lib.call("fqehip_norm_finalize", _lib.ptr(partials), offs[-1],
                  _lib.ptr(norm), accuracy, order, _lib.ptr(status[1:]),
                  _lib.ptr(status[:1]), _lib.stream_ptr())
    st = status.cpu().numpy()
    if expansion <= 1 or st[1] == 0:
        raise RuntimeError("maximum taylor expansion limit reached")
    for k, sec in enumerate(secs):
        sec.set_device_coeff(torch.view_as_complex(results[k]))
    out._taylor_terms = int(st[0])
    return out


class _TaylorGraph:
    """One recorded Taylor series (fqehip_taylor_graph_create) with the
    buffers its nodes reference."""

    def __init__(self, sec: FqeData, op: engine.PreparedOperator,
                 c: torch.Tensor, time: float, accuracy: float,
                 expansion: int) -> None:
        import ctypes
        dev = c.device
        self.prec = engine.precision_of(c.dtype)
        self.s, self.keep = engine.sector_struct(sec.get_fcigraph(), op,
                                                 self.prec)
        self.ws = engine.workspace(self.s, self.prec, dev)
        self.term = torch.empty_like(c)
        self.result = torch.empty(c.shape, dtype=torch.complex128,
                                  device=dev)
        self.partials = torch.zeros(
            max(engine.norm_partials_count(c.numel()), 1),
            dtype=torch.float64, device=dev)
        self.status = torch.zeros(2, dtype=torch.int32, device=dev)
        self.norm = torch.zeros(1, dtype=torch.float64, device=dev)
        self.opc = op.c_struct()
        handle = ctypes.c_void_p()
        torch.cuda.synchronize()
        _lib.call("fqehip_taylor_graph_create", self.prec,
                  engine._as_ref(self.s), engine._as_ref(self.opc),
                  float(time), float(accuracy), int(expansion),
                  _lib.ptr(self.term), _lib.ptr(self.result),
                  _lib.ptr(self.status), _lib.ptr(self.partials),
                  _lib.ptr(self.norm), _lib.ptr(self.ws),
                  ctypes.byref(handle))
        self.handle = handle

    def run(self, c: torch.Tensor):
        self.term.copy_(c)
        self.result.copy_(c)
        _lib.call("fqehip_taylor_graph_launch", self.handle,
                  _lib.stream_ptr())
        return self.result.clone(), self.status.cpu().numpy()

    def __del__(self):
        try:
            _lib.call("fqehip_taylor_graph_destroy", self.handle)
        except Exception:
            pass


def _taylor_single(out: Wavefunction, sec: FqeData,
                   op: engine.PreparedOperator, time: float, accuracy: float,
                   expansion: int) -> Wavefunction:
    dev = _lib.device()
    c = sec.device_coeff()
    prec = engine.precision_of(c.dtype)
    if settings.taylor_graph:
        g = sec.get_fcigraph()
        key = (g.nalpha(), g.nbeta(), g.norb(), c.dtype, float(time),
               float(accuracy), int(expansion),
               settings.kernel_choice())
        cached = getattr(op, "_taylor_graph", None)
        if cached is None or cached[0] != key:
            op._taylor_graph = None          # free the previous one first
            op._taylor_graph = (key, _TaylorGraph(sec, op, c, time, accuracy,
                                                  expansion))
        result, st = op._taylor_graph[1].run(c)
        if expansion <= 1 or st[1] == 0:
            raise RuntimeError("maximum taylor expansion limit reached")
        sec.set_device_coeff(result)
        out._taylor_terms = int(st[0])
        return out
    term = c.clone()
    result = c.to(torch.complex128).clone()
    s, keep = engine.sector_struct(sec.get_fcigraph(), op, prec)
    ws = engine.workspace(s, prec, dev)
    partials = torch.zeros(max(engine.norm_partials_count(c.numel()), 1),
                           dtype=torch.float64, device=dev)
    status = torch.zeros(2, dtype=torch.int32, device=dev)
    norm = torch.zeros(1, dtype=torch.float64, device=dev)
    opc = op.c_struct()
    _lib.call("fqehip_taylor", prec, engine._as_ref(s), engine._as_ref(opc),
              float(time), float(accuracy), int(expansion), _lib.ptr(term),
              _lib.ptr(result), _lib.ptr(status), _lib.ptr(partials),
              _lib.ptr(norm), _lib.ptr(ws), _lib.stream_ptr())
    st = status.cpu().numpy()
    del keep
    if expansion <= 1 or st[1] == 0:
        raise RuntimeError("maximum taylor expansion limit reached")
    sec.set_device_coeff(result)
    out._taylor_terms = int(st[0])
    return out
