"""Python host side of libfermihip (ctypes), mirroring Fermi.jl's RCCSD / RCCSD(T) interface.

Fermi.jl selects a CC backend by algorithm singleton types (RCCSD.jl:12,76-88;
PerturbativeTriples.jl:1-11).  This module offers the same call shapes on top of the
C ABI in ``include/fermihip.h``:

  * ``RCCSD(moints, alg=RCCSDhip())``               -> MP2 guess + iterations  (RCCSDa.jl:46-90)
  * ``RCCSD(moints, T1, T2, alg=RCCSDhip())``       -> iterations from given amplitudes (RCCSDa.jl:92-245)
  * ``RCCSDpT(ccsd, moints, alg=ijkhip())``         -> (T) correction (ijk.jl:20-150)
  * ``RMP2(moints, alg=RMP2hip())``                 -> DF-MP2 energy (RMP2a.jl:56-144); only
    ``BOV`` and the orbital energies are needed (``BOO``/``BVV`` may be None)
  * ``RHF(S, H, b, ndocc, Vnuc, alg=RHFhip())``      -> DF-RHF SCF (RHFa.jl:14-223)

``moints`` is a :class:`MOIntegrals`, the subset of Fermi's ``IntegralHelper`` cache the path
reads: ``BOO[Q,o,o]``, ``BOV[Q,o,v]``, ``BVV[Q,v,v]``, ``Fii[o]``, ``Faa[v]`` and the
reference energy.  Options use Fermi's key names (Options.jl:62-102).  Errors raise
:class:`FermiException` with the library's message; non-convergence is not an error.

There is no CPU fallback: if ``libfermihip.so`` is missing or no HIP device is present,
every entry point raises.
"""
import ctypes
import os
from dataclasses import dataclass, field

import numpy as np

__all__ = [
    "FermiException", "MOIntegrals", "Options", "RCCSDhip", "ijkhip", "RCCSD", "RCCSDpT", "Context",
    "lib_path", "load_library", "EXPORTED_SYMBOLS", "Mlp", "PRECISIONS", "RMP2", "RMP2hip", "RHF", "RHFhip",
    "ScfOptions", "Basis",
]

HERE = os.path.dirname(os.path.abspath(__file__))
EXPORTED_SYMBOLS = [
    "fh_default_opts", "fh_create", "fh_set_df", "fh_prepare", "fh_t2_guess", "fh_ccsd_energy",
    "fh_ccsd_residual", "fh_ccsd_solve", "fh_mp2_energy", "fh_mp2_energy_noalloc", "fh_set_df_ao", "fh_get_df", "fh_default_scf_opts", "fh_rhf",
    "fh_df_fit", "fh_ao2mo_4index", "fh_set_mo", "fh_triples", "fh_triples_range", "fh_stats", "fh_last_error",
    "fh_destroy", "fh_rhf_conv", "fh_basis_create", "fh_basis_nbf", "fh_basis_destroy", "fh_one_electron",
    "fh_eri_2e4c", "fh_eri_2e3c", "fh_eri_2e2c", "fh_dipole",
    "fh_mlp_create", "fh_mlp_num_params", "fh_mlp_get_params", "fh_mlp_set_params", "fh_mlp_forward",
    "fh_mlp_loss_grad", "fh_mlp_train", "fh_mlp_destroy", "fh_set_t2_model", "fh_load_t2_model",
]


class FermiException(Exception):
    """Mirror of Fermi.Options.FermiException (Options.jl:196-199)."""


class _Opts(ctypes.Structure):
    _fields_ = [
        ("cc_max_iter", ctypes.c_int), ("cc_e_conv", ctypes.c_double), ("cc_max_rms", ctypes.c_double),
        ("cc_diis", ctypes.c_int), ("cc_ndiis", ctypes.c_int), ("diis_start", ctypes.c_int),
        ("cc_diis_relax", ctypes.c_int), ("diis_prec", ctypes.c_int), ("cc_damp_ratio", ctypes.c_double),
        ("precision_override", ctypes.c_int), ("verbose", ctypes.c_int),
        ("precision_mode", ctypes.c_int), ("polish_iters", ctypes.c_int), ("mixed_e_switch", ctypes.c_double),
        ("mixed_rms_switch", ctypes.c_double), ("bf3_e_switch", ctypes.c_double), ("bf3_rms_switch", ctypes.c_double),
        ("max_restarts", ctypes.c_int), ("fault_inject", ctypes.c_int),
    ]


class _Result(ctypes.Structure):
    _fields_ = [
        ("guess_energy", ctypes.c_double), ("correlation", ctypes.c_double), ("e_conv", ctypes.c_double),
        ("t_conv", ctypes.c_double), ("niter", ctypes.c_int), ("converged", ctypes.c_int),
        ("niter_mixed", ctypes.c_int), ("niter_bf3", ctypes.c_int), ("restarts", ctypes.c_int),
    ]


class _ScfOpts(ctypes.Structure):
    _fields_ = [
        ("scf_max_iter", ctypes.c_int), ("scf_e_conv", ctypes.c_double), ("scf_max_rms", ctypes.c_double),
        ("diis", ctypes.c_int), ("ndiis", ctypes.c_int), ("diis_start", ctypes.c_int), ("oda", ctypes.c_int),
        ("oda_cutoff", ctypes.c_double), ("oda_shutoff", ctypes.c_int), ("guess", ctypes.c_int),
    ]


class _ScfResult(ctypes.Structure):
    _fields_ = [("energy", ctypes.c_double), ("e_conv", ctypes.c_double), ("d_rms", ctypes.c_double),
                ("niter", ctypes.c_int), ("converged", ctypes.c_int)]


def ScfOptions(**kw):
    """SCF options with Fermi's key names and defaults (Options.jl:55-89); scf_guess "gwh" | "core"."""
    o = {"scf_max_iter": 50, "scf_e_conv": 1e-10, "scf_max_rms": 1e-9, "diis": True, "ndiis": 8, "diis_start": 3,
         "oda": True, "oda_cutoff": 1e-1, "oda_shutoff": 20, "scf_guess": "gwh"}
    for k in kw:
        if k not in o:
            raise FermiException(f"unknown SCF option {k}")
    o.update(kw)
    if o["scf_guess"] not in ("gwh", "core"):
        raise FermiException(f"scf_guess {o['scf_guess']} is not supported")
    return o


def lib_path():
    return os.environ.get("FERMIHIP_LIB", os.path.join(HERE, "libfermihip.so"))


_LIB = None


def load_library():
    """Load libfermihip.so (built in-tree by build.py).  Raises if it is missing."""
    global _LIB
    if _LIB is not None:
        return _LIB
    p = lib_path()
    if not os.path.exists(p):
        raise FermiException(f"libfermihip.so not found at {p}: run __graft_entry__.build()")
    L = ctypes.CDLL(p)
    dp = ctypes.POINTER(ctypes.c_double)
    L.fh_default_opts.argtypes = [ctypes.POINTER(_Opts)]
    L.fh_default_opts.restype = None
    L.fh_create.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_int]
    L.fh_set_df.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, dp, dp, dp, dp, dp]
    L.fh_prepare.argtypes = [ctypes.c_void_p]
    L.fh_t2_guess.argtypes = [ctypes.c_void_p, ctypes.c_int, dp, dp]
    L.fh_ccsd_energy.argtypes = [ctypes.c_void_p, dp, dp, dp]
    L.fh_ccsd_residual.argtypes = [ctypes.c_void_p, dp, dp, dp, dp]
    L.fh_ccsd_solve.argtypes = [ctypes.c_void_p, ctypes.POINTER(_Opts), dp, dp, ctypes.POINTER(_Result)]
    L.fh_triples.argtypes = [ctypes.c_void_p, ctypes.c_int, dp, dp, dp]
    L.fh_triples_range.argtypes = [ctypes.c_void_p, ctypes.c_int, dp, dp, ctypes.c_longlong, ctypes.c_longlong, dp]
    L.fh_set_mo.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int] + [dp] * 9
    L.fh_mp2_energy.argtypes = [ctypes.c_void_p, dp]
    # device pointers (eps_o, eps_v, Bov, Emp2) as integers
    L.fh_mp2_energy_noalloc.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int] + [ctypes.c_void_p] * 4
    L.fh_set_df_ao.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * 5 + [dp, dp, dp]
    L.fh_get_df.argtypes = [ctypes.c_void_p, dp, dp, dp]
    L.fh_df_fit.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, dp, dp, dp]
    L.fh_ao2mo_4index.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, dp, ctypes.c_int, dp, ctypes.c_int, dp,
                                  ctypes.c_int, dp, dp, dp]
    L.fh_default_scf_opts.argtypes = [ctypes.POINTER(_ScfOpts)]
    L.fh_default_scf_opts.restype = None
    L.fh_rhf.argtypes = [ctypes.c_void_p, ctypes.POINTER(_ScfOpts), ctypes.c_int, ctypes.c_int, ctypes.c_int,
                         ctypes.c_double, dp, dp, dp, dp, dp, ctypes.POINTER(_ScfResult)]
    L.fh_rhf_conv.argtypes = [ctypes.c_void_p, ctypes.POINTER(_ScfOpts), ctypes.c_int, ctypes.c_int, ctypes.c_double,
                              dp, dp, dp, dp, dp, ctypes.POINTER(_ScfResult)]
    ip = ctypes.POINTER(ctypes.c_int)
    L.fh_basis_create.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_int, ip, ip, dp, dp, dp, ctypes.c_int]
    L.fh_basis_nbf.argtypes = [ctypes.c_void_p]
    L.fh_basis_destroy.argtypes = [ctypes.c_void_p]
    L.fh_basis_destroy.restype = None
    L.fh_one_electron.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, dp, dp, dp, dp, dp]
    L.fh_eri_2e4c.argtypes = [ctypes.c_void_p, ctypes.c_void_p, dp]
    L.fh_dipole.argtypes = [ctypes.c_void_p, ctypes.c_void_p, dp, dp, dp, dp]
    L.fh_eri_2e3c.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, dp]
    L.fh_eri_2e2c.argtypes = [ctypes.c_void_p, ctypes.c_void_p, dp]
    L.fh_stats.argtypes = [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_size_t]
    L.fh_last_error.argtypes = []
    L.fh_last_error.restype = ctypes.c_char_p
    L.fh_destroy.argtypes = [ctypes.c_void_p]
    L.fh_destroy.restype = None
    fp = ctypes.POINTER(ctypes.c_float)
    L.fh_mlp_create.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_int, ctypes.c_int, ctypes.c_ulonglong]
    L.fh_mlp_num_params.argtypes = [ctypes.c_void_p]
    L.fh_mlp_num_params.restype = ctypes.c_size_t
    L.fh_mlp_get_params.argtypes = [ctypes.c_void_p, fp]
    L.fh_mlp_set_params.argtypes = [ctypes.c_void_p, fp]
    L.fh_mlp_forward.argtypes = [ctypes.c_void_p, ctypes.c_longlong, fp, fp]
    L.fh_mlp_loss_grad.argtypes = [ctypes.c_void_p, ctypes.c_longlong, fp, fp, dp, fp]
    L.fh_mlp_train.argtypes = [ctypes.c_void_p, ctypes.c_longlong, fp, fp, ctypes.c_int, ctypes.c_int, ctypes.c_float,
                               ctypes.c_ulonglong, dp]
    L.fh_mlp_destroy.argtypes = [ctypes.c_void_p]
    L.fh_mlp_destroy.restype = None
    L.fh_set_t2_model.argtypes = [ctypes.c_void_p, ctypes.c_void_p, fp, fp, ctypes.c_double, dp]
    L.fh_load_t2_model.argtypes = [ctypes.c_void_p, ctypes.c_char_p, dp]
    for name in EXPORTED_SYMBOLS:
        if name not in ("fh_default_opts", "fh_last_error", "fh_destroy", "fh_mlp_destroy", "fh_mlp_num_params",
                        "fh_basis_destroy"):
            getattr(L, name).restype = ctypes.c_int
    _LIB = L
    return L


def _ptr(a):
    if a is None:
        return None
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _fptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


def _samples(X):
    """Sample matrix for the network: [n, 6] row-major float32 (= [6, n] column-major)."""
    X = np.ascontiguousarray(np.asarray(X, dtype=np.float32))
    if X.ndim != 2 or X.shape[1] != 6:
        raise FermiException("network samples must be an [n, 6] array")
    return X


def _colmajor(a):
    """Julia arrays are column-major: hand the library a Fortran-ordered FP64 copy/view."""
    return np.asfortranarray(np.asarray(a, dtype=np.float64))


PRECISIONS = {"double": 0, "mixed": 1, "bf16x3": 2}


def Options(**kw):
    """Fermi option keys read on this path, with the reference defaults (Options.jl:62-102), plus
    the mixed-precision keys of this backend: precision ("double"; "mixed": FP32 contractions then
    FP64 polish; "bf16x3": split-BF16x3 contractions then FP64 polish), polish_iters
    (-1: polish to convergence), mixed_e_switch, mixed_rms_switch, bf3_e_switch, bf3_rms_switch, and the
    failure-handling keys max_restarts (restarts from the last finite amplitudes after a non-finite
    iteration) and fault_inject (iteration whose new T2 gets one NaN; a test hook, 0 = off)."""
    o = dict(cc_max_iter=50, cc_e_conv=1e-10, cc_max_rms=1e-10, cc_diis=True, cc_ndiis=3, diis_start=3,
             cc_diis_relax=3, diis_prec="single", cc_damp_ratio=0.0, precision_override=False, verbose=False,
             precision="double", polish_iters=-1, mixed_e_switch=1e-9, mixed_rms_switch=1e-9, bf3_e_switch=1e-7,
             bf3_rms_switch=1e-8, max_restarts=1, fault_inject=0)
    for k, v in kw.items():
        if k not in o:
            raise FermiException(f"unknown option {k}")
        o[k] = v
    if o["diis_prec"] not in ("single", "double"):
        raise FermiException(f"invalid diis_prec {o['diis_prec']!r} (single|double)")
    if o["precision"] not in PRECISIONS:
        raise FermiException(f"invalid precision {o['precision']!r} (double|mixed|bf16x3)")
    return o


@dataclass
class MOIntegrals:
    """The part of Fermi's IntegralHelper cache read by the CC path (IntegralHelper.jl:50-56)."""
    BOO: np.ndarray
    BOV: np.ndarray
    BVV: np.ndarray
    Fii: np.ndarray
    Faa: np.ndarray
    sd_energy: float = 0.0
    context: "Context" = field(default=None, repr=False)

    @property
    def o(self):
        return self.BOV.shape[1]

    @property
    def v(self):
        return self.BOV.shape[2]

    @property
    def naux(self):
        return self.BOV.shape[0]


class Context:
    """Owns one fh_ctx (device memory of one molecule)."""

    def __init__(self, device=0):
        self.L = load_library()
        h = ctypes.c_void_p()
        self._check(self.L.fh_create(ctypes.byref(h), int(device)))
        self.h = h
        self.device = int(device)
        self.o = self.v = self.naux = 0

    def _check(self, rc):
        if rc != 0:
            raise FermiException(f"libfermihip error {rc}: {self.L.fh_last_error().decode()}")

    def close(self):
        if getattr(self, "h", None):
            self.L.fh_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def set_df(self, eps_o, eps_v, Boo, Bov, Bvv):
        """Hand over the DF tensors (Boo and Bvv may both be None: a context for mp2_energy only)."""
        Q, o, v = Bov.shape
        if (Boo is None) != (Bvv is None):
            raise FermiException("give both BOO and BVV, or neither (DF-MP2 only)")
        if (Boo is not None and (Boo.shape != (Q, o, o) or Bvv.shape != (Q, v, v))) or len(eps_o) != o \
                or len(eps_v) != v:
            raise FermiException("inconsistent DF tensor shapes")
        self._keep = [None if x is None else _colmajor(x) for x in (eps_o, eps_v, Boo, Bov, Bvv)]
        self._check(self.L.fh_set_df(self.h, o, v, Q, *[_ptr(x) for x in self._keep]))
        self._keep = None
        self.o, self.v, self.naux = o, v, Q

    def set_mo(self, eps_o, eps_v, blocks, Fia=None):
        """Hand over the conventional MO blocks (fh_set_mo, the Chonky path of RCCSDa.jl:25-35): blocks is a
        dict with OOOO[i,j,k,l], OOOV[i,j,k,a], OOVV[i,j,a,b], OVOV[i,a,j,b], OVVV[i,a,b,c], VVVV[a,b,c,d];
        Fia[o,v] the occupied-virtual Fock block (None: zero, canonical RHF orbitals)."""
        o, v = len(eps_o), len(eps_v)
        shapes = {"OOOO": (o, o, o, o), "OOOV": (o, o, o, v), "OOVV": (o, o, v, v), "OVOV": (o, v, o, v),
                  "OVVV": (o, v, v, v), "VVVV": (v, v, v, v)}
        for k, sh in shapes.items():
            if k not in blocks or np.shape(blocks[k]) != sh:
                raise FermiException(f"block {k} must have shape {sh}")
        if Fia is not None and np.shape(Fia) != (o, v):
            raise FermiException("Fia must be [o, v]")
        keep = [_colmajor(eps_o), _colmajor(eps_v), None if Fia is None else _colmajor(Fia)] + \
            [_colmajor(blocks[k]) for k in shapes]
        self._check(self.L.fh_set_mo(self.h, o, v, *[_ptr(x) for x in keep]))
        self.o, self.v, self.naux = o, v, 0

    def set_df_ao(self, eps, C, bAO, ndocc, drop_occ=0, drop_vir=0):
        """AO -> MO DF transforms on the device (fh_set_df_ao, DFERI.jl:15-69): bAO[Q,mu,nu] the fitted
        AO tensor, C[mu,p] and eps[p] the RHF orbitals, ndocc doubly occupied orbitals of which the
        first drop_occ are frozen, the last drop_vir virtuals inactive."""
        Q, n, n2 = bAO.shape
        if n2 != n or C.shape != (n, n) or len(eps) != n:
            raise FermiException("inconsistent AO tensor / orbital shapes")
        keep = [_colmajor(x) for x in (eps, C, bAO)]
        self._check(self.L.fh_set_df_ao(self.h, n, Q, int(ndocc), int(drop_occ), int(drop_vir),
                                        *[_ptr(x) for x in keep]))
        self.o, self.v, self.naux = ndocc - drop_occ, n - drop_vir - ndocc, Q

    def df_fit(self, J, Pqp):
        """b[Q,mu,nu] = Pqp[mu,nu,P] J^(-1/2)[P,Q] (fh_df_fit, AtomicIntegrals.jl:31-41)."""
        n, n2, Q = Pqp.shape
        if n2 != n or J.shape != (Q, Q):
            raise FermiException("inconsistent J / Pqp shapes")
        keep = [_colmajor(J), _colmajor(Pqp)]
        b = np.zeros((Q, n, n), order="F")
        self._check(self.L.fh_df_fit(self.h, n, Q, _ptr(keep[0]), _ptr(keep[1]), _ptr(b)))
        return b

    def ao2mo_4index(self, eri, C1, C2, C3, C4):
        """Conventional 4-index transform (fh_ao2mo_4index, Chonky.jl:1-131):
        out[i,j,k,l] = eri[mu,nu,rho,sigma] C1[mu,i] C2[nu,j] C3[rho,k] C4[sigma,l]."""
        n = eri.shape[0]
        if eri.shape != (n, n, n, n) or any(c.shape[0] != n for c in (C1, C2, C3, C4)):
            raise FermiException("inconsistent ERI / coefficient shapes")
        keep = [_colmajor(x) for x in (C1, C2, C3, C4, eri)]
        out = np.zeros((C1.shape[1], C2.shape[1], C3.shape[1], C4.shape[1]), order="F")
        self._check(self.L.fh_ao2mo_4index(self.h, n, C1.shape[1], _ptr(keep[0]), C2.shape[1], _ptr(keep[1]),
                                           C3.shape[1], _ptr(keep[2]), C4.shape[1], _ptr(keep[3]), _ptr(keep[4]),
                                           _ptr(out)))
        return out

    def rhf(self, S, H, b, ndocc, Vnuc=0.0, options=None):
        """DF-RHF SCF (fh_rhf): returns (result dict, eps[nbf], C[nbf,nbf])."""
        Q, n, n2 = b.shape
        if n2 != n or S.shape != (n, n) or H.shape != (n, n):
            raise FermiException("inconsistent S / H / b shapes")
        o = ScfOptions() if options is None else options
        op = _ScfOpts()
        self.L.fh_default_scf_opts(ctypes.byref(op))
        for k in ("scf_max_iter", "scf_e_conv", "scf_max_rms", "ndiis", "diis_start", "oda_cutoff", "oda_shutoff"):
            setattr(op, k, o[k])
        op.diis, op.oda, op.guess = int(bool(o["diis"])), int(bool(o["oda"])), 0 if o["scf_guess"] == "gwh" else 1
        keep = [_colmajor(x) for x in (S, H, b)]
        eps = np.zeros(n)
        C = np.zeros((n, n), order="F")
        res = _ScfResult()
        self._check(self.L.fh_rhf(self.h, ctypes.byref(op), n, Q, int(ndocc), float(Vnuc), *[_ptr(x) for x in keep],
                                  _ptr(eps), _ptr(C), ctypes.byref(res)))
        r = {"energy": res.energy, "e_conv": res.e_conv, "d_rms": res.d_rms, "niter": res.niter,
             "converged": bool(res.converged)}
        return r, eps, C

    def rhf_conv(self, S, H, eri, ndocc, Vnuc=0.0, options=None):
        """RHF with conventional integrals (fh_rhf_conv): returns (result dict, eps[nbf], C[nbf,nbf])."""
        n = S.shape[0]
        if eri.shape != (n, n, n, n) or H.shape != (n, n):
            raise FermiException("inconsistent S / H / eri shapes")
        o = ScfOptions() if options is None else options
        op = _ScfOpts()
        self.L.fh_default_scf_opts(ctypes.byref(op))
        for k in ("scf_max_iter", "scf_e_conv", "scf_max_rms", "ndiis", "diis_start", "oda_cutoff", "oda_shutoff"):
            setattr(op, k, o[k])
        op.diis, op.oda, op.guess = int(bool(o["diis"])), int(bool(o["oda"])), 0 if o["scf_guess"] == "gwh" else 1
        keep = [_colmajor(x) for x in (S, H, eri)]
        eps = np.zeros(n)
        C = np.zeros((n, n), order="F")
        res = _ScfResult()
        self._check(self.L.fh_rhf_conv(self.h, ctypes.byref(op), n, int(ndocc), float(Vnuc), *[_ptr(x) for x in keep],
                                       _ptr(eps), _ptr(C), ctypes.byref(res)))
        r = {"energy": res.energy, "e_conv": res.e_conv, "d_rms": res.d_rms, "niter": res.niter,
             "converged": bool(res.converged)}
        return r, eps, C

    def one_electron(self, basis, atoms):
        """(S, T, V) over a Basis (fh_one_electron); atoms: [(Z, xyz bohr)] or basis.py's atom tuples."""
        n = basis.nbf
        Zs = np.ascontiguousarray([float(a[-2]) for a in atoms])
        X = np.ascontiguousarray(np.array([np.asarray(a[-1], float) for a in atoms]).reshape(-1))
        out = [np.zeros((n, n), order="F") for _ in range(3)]
        self._check(self.L.fh_one_electron(self.h, basis.h, len(atoms), _ptr(Zs), _ptr(X), *[_ptr(x) for x in out]))
        return tuple(out)

    def dipole(self, basis, origin=None):
        """(Dx, Dy, Dz) = <mu| r - origin |nu> (fh_dipole)."""
        n = basis.nbf
        out = [np.zeros((n, n), order="F") for _ in range(3)]
        o = None if origin is None else np.ascontiguousarray(np.asarray(origin, float))
        self._check(self.L.fh_dipole(self.h, basis.h, _ptr(o), *[_ptr(x) for x in out]))
        return tuple(out)

    def eri_2e4c(self, basis):
        n = basis.nbf
        out = np.zeros((n, n, n, n), order="F")
        self._check(self.L.fh_eri_2e4c(self.h, basis.h, _ptr(out)))
        return out

    def eri_2e3c(self, basis, aux):
        out = np.zeros((basis.nbf, basis.nbf, aux.nbf), order="F")
        self._check(self.L.fh_eri_2e3c(self.h, basis.h, aux.h, _ptr(out)))
        return out

    def eri_2e2c(self, aux):
        out = np.zeros((aux.nbf, aux.nbf), order="F")
        self._check(self.L.fh_eri_2e2c(self.h, aux.h, _ptr(out)))
        return out

    def get_df(self):
        """The MO DF tensors held by the context: (BOO[Q,o,o], BOV[Q,o,v], BVV[Q,v,v])."""
        Q, o, v = self.naux, self.o, self.v
        out = [np.zeros(s, order="F") for s in ((Q, o, o), (Q, o, v), (Q, v, v))]
        self._check(self.L.fh_get_df(self.h, *[_ptr(x) for x in out]))
        return tuple(out)

    def prepare(self):
        self._check(self.L.fh_prepare(self.h))

    def mp2_energy(self):
        """DF-MP2 correlation energy (fh_mp2_energy, RMP2a.jl:91-144)."""
        E = ctypes.c_double()
        self._check(self.L.fh_mp2_energy(self.h, ctypes.byref(E)))
        return E.value

    def guess(self, kind=0, copy_out=True):
        """Initial amplitudes (fh_t2_guess): kind 0 MP2, 1 learned (after set_t2_model); add 2 for
        the first-order T1 instead of T1 = 0.  Kept on the device for solve(); returned when copy_out.
        A learned guess that is not available falls back to the MP2 guess (guess_fallback is then True)."""
        T1 = T2 = None
        if copy_out:
            T1 = np.zeros((self.o, self.v), order="F")
            T2 = np.zeros((self.o, self.o, self.v, self.v), order="F")
        rc = self.L.fh_t2_guess(self.h, kind, _ptr(T1), _ptr(T2))
        self.guess_fallback = rc == 1
        if rc != 1:
            self._check(rc)
        return T1, T2

    def set_t2_model(self, model, pair_dist=None):
        """Attach a trained guess network (an Mlp, or a dict/npz with params, x_mean, x_scale,
        y_scale, hidden) for guess(kind=1), with the occupied pair distances [o, o] in bohr."""
        if isinstance(model, Mlp):
            net, xm, xs, ys = model, model.x_mean, model.x_scale, model.y_scale
        else:
            net = Mlp(hidden=int(model["hidden"]), device=self.device)
            net.set_params(np.asarray(model["params"], dtype=np.float32))
            xm, xs, ys = model["x_mean"], model["x_scale"], float(model["y_scale"])
        xm = np.ascontiguousarray(np.asarray(xm, dtype=np.float32))
        xs = np.ascontiguousarray(np.asarray(xs, dtype=np.float32))
        d = None if pair_dist is None else _colmajor(pair_dist)
        if d is not None and d.shape != (self.o, self.o):
            raise FermiException("pair_dist must be [o, o]")
        self._check(self.L.fh_set_t2_model(self.h, net.h, _fptr(xm), _fptr(xs), float(ys), _ptr(d)))

    def load_t2_model(self, path, pair_dist=None):
        """Attach a guess network from a model file (fh_load_t2_model; train_guess.write_model_file)."""
        d = None if pair_dist is None else _colmajor(pair_dist)
        if d is not None and d.shape != (self.o, self.o):
            raise FermiException("pair_dist must be [o, o]")
        self._check(self.L.fh_load_t2_model(self.h, os.fsencode(path), _ptr(d)))

    def energy(self, T1=None, T2=None):
        E = ctypes.c_double()
        if T1 is None:
            self._check(self.L.fh_ccsd_energy(self.h, None, None, ctypes.byref(E)))
        else:
            a, b = _colmajor(T1), _colmajor(T2)
            self._check(self.L.fh_ccsd_energy(self.h, _ptr(a), _ptr(b), ctypes.byref(E)))
        return E.value

    def update_amp(self, T1, T2):
        a, b = _colmajor(T1), _colmajor(T2)
        n1 = np.zeros_like(a, order="F")
        n2 = np.zeros_like(b, order="F")
        self._check(self.L.fh_ccsd_residual(self.h, _ptr(a), _ptr(b), _ptr(n1), _ptr(n2)))
        return n1, n2

    def solve(self, opts=None, T1=None, T2=None, copy_out=True):
        return self._solve(opts, T1, T2, copy_out)

    def _solve(self, opts, T1, T2, copy_out=True, in_place=False):
        opts = Options() if opts is None else opts
        c = _Opts()
        self.L.fh_default_opts(ctypes.byref(c))
        c.cc_max_iter = int(opts["cc_max_iter"]); c.cc_e_conv = float(opts["cc_e_conv"])
        c.cc_max_rms = float(opts["cc_max_rms"]); c.cc_diis = int(bool(opts["cc_diis"]))
        c.cc_ndiis = int(opts["cc_ndiis"]); c.diis_start = int(opts["diis_start"])
        c.cc_diis_relax = int(opts["cc_diis_relax"]); c.diis_prec = 1 if opts["diis_prec"] == "single" else 0
        c.cc_damp_ratio = float(opts["cc_damp_ratio"]); c.precision_override = int(bool(opts["precision_override"]))
        c.verbose = int(bool(opts["verbose"]))
        c.precision_mode = PRECISIONS[opts["precision"]]
        c.polish_iters = int(opts["polish_iters"])
        c.mixed_e_switch = float(opts["mixed_e_switch"])
        c.mixed_rms_switch = float(opts["mixed_rms_switch"])
        c.bf3_e_switch = float(opts["bf3_e_switch"])
        c.bf3_rms_switch = float(opts["bf3_rms_switch"])
        c.max_restarts = int(opts["max_restarts"])
        c.fault_inject = int(opts["fault_inject"])
        r = _Result()
        if T1 is None:
            self._check(self.L.fh_ccsd_solve(self.h, ctypes.byref(c), None, None, ctypes.byref(r)))
            out1 = out2 = None
            if copy_out:
                raise FermiException("copy_out requires starting amplitudes; use T1/T2 arrays")
        else:
            out1, out2 = (T1, T2) if in_place else (_colmajor(T1).copy(order="F"), _colmajor(T2).copy(order="F"))
            self._check(self.L.fh_ccsd_solve(self.h, ctypes.byref(c), _ptr(out1), _ptr(out2), ctypes.byref(r)))
        return r, out1, out2

    def triples(self, T1=None, T2=None, prec_mode=0):
        Et = ctypes.c_double()
        if T1 is None:
            self._check(self.L.fh_triples(self.h, prec_mode, None, None, ctypes.byref(Et)))
        else:
            a, b = _colmajor(T1), _colmajor(T2)
            self._check(self.L.fh_triples(self.h, prec_mode, _ptr(a), _ptr(b), ctypes.byref(Et)))
        return Et.value

    def triples_range(self, first, count, T1=None, T2=None, prec_mode=0):
        """(T) over the triples first .. first+count-1 of the reference's loop order (fh_triples_range)."""
        Et = ctypes.c_double()
        a = b = None
        if T1 is not None:
            a, b = _colmajor(T1), _colmajor(T2)
        self._check(self.L.fh_triples_range(self.h, prec_mode, _ptr(a), _ptr(b), int(first), int(count),
                                            ctypes.byref(Et)))
        return Et.value

    def stats(self):
        import json
        buf = ctypes.create_string_buffer(1 << 20)
        self._check(self.L.fh_stats(self.h, buf, len(buf)))
        return json.loads(buf.value.decode())


class Basis:
    """A Gaussian basis set on the library side (fh_basis_create) from shell dicts (l, center, exps, coefs),
    e.g. fermihip.basis.shells_for(atoms, "cc-pvdz")."""

    def __init__(self, shells, spherical=True):
        from . import basis as _b
        self.L = load_library()
        l, nprim, center, exps, coefs = _b.flatten(shells)
        ip = ctypes.POINTER(ctypes.c_int)
        h = ctypes.c_void_p()
        rc = self.L.fh_basis_create(ctypes.byref(h), len(shells), l.ctypes.data_as(ip), nprim.ctypes.data_as(ip),
                                    _ptr(center), _ptr(exps), _ptr(coefs), int(bool(spherical)))
        if rc != 0:
            raise FermiException(f"libfermihip error {rc}: {self.L.fh_last_error().decode()}")
        self.h = h
        self.nbf = int(self.L.fh_basis_nbf(h))
        self.shells = shells

    def close(self):
        if getattr(self, "h", None):
            self.L.fh_basis_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


# ---------------------------------------------------------------- Fermi-shaped API
class RCCSDhip:
    """Algorithm singleton for the MI355X backend (the role of RCCSDa, RCCSD.jl:85-88)."""


class ijkhip:
    """(T) algorithm singleton for the MI355X backend (the role of ijk, PerturbativeTriples.jl:41-43)."""


@dataclass
class RCCSDResult:
    """Fields of Fermi's RCCSD{T} (RCCSD.jl:61-69)."""
    guessenergy: float
    correlation: float
    energy: float
    T1: np.ndarray
    T2: np.ndarray
    e_conv: float
    t_conv: float
    niter: int
    converged: bool


@dataclass
class RCCSDpTResult:
    """Fields of Fermi's RCCSDpT{T} (PerturbativeTriples.jl:21-25)."""
    CCSD: RCCSDResult
    energy: float
    correction: float


def _ctx_for(moints, device=0):
    if moints.context is None:
        moints.context = Context(device)
        moints.context.set_df(moints.Fii, moints.Faa, moints.BOO, moints.BOV, moints.BVV)
    return moints.context


class RHFhip:
    """RHF algorithm singleton for the MI355X backend (the role of RHFa, RHF.jl:112)."""


@dataclass
class RHFResult:
    """Fields of Fermi's RHF (RHF.jl:69-77), with the orbitals as eps / C."""
    energy: float
    ndocc: int
    nvir: int
    eps: np.ndarray
    C: np.ndarray
    e_conv: float
    d_conv: float
    converged: bool
    niter: int


def RHF(S, H, b, ndocc, Vnuc=0.0, alg=None, options=None, device=0):
    """RHF(ints, ::RHFa) with DF integrals (RHFa.jl:14-223): S = ints["S"], H = ints["T"] + ints["V"],
    b = ints["ERI"] (fitted AO tensor b[Q,mu,nu]), ndocc = Nalpha, Vnuc the nuclear repulsion."""
    if alg is not None and not isinstance(alg, RHFhip):
        raise FermiException(f"invalid algorithm {type(alg).__name__} for the MI355X RHF backend")
    ctx = Context(device)
    try:
        r, eps, C = ctx.rhf(S, H, b, ndocc, Vnuc, options)
    finally:
        ctx.close()
    return RHFResult(r["energy"], int(ndocc), S.shape[0] - int(ndocc), eps, C, r["e_conv"], r["d_rms"],
                     r["converged"], r["niter"])


class RMP2hip:
    """RMP2 algorithm singleton for the MI355X backend (the role of RMP2a, RMP2.jl:69-72)."""


@dataclass
class RMP2Result:
    """Fields of Fermi's RMP2{T} (RMP2.jl:50-53)."""
    correlation: float
    energy: float


def RMP2(moints, alg=None, device=0):
    """RMP2(moints; alg) -> RMP2Result (RMP2a.jl:56-88 with the DF energy of RMP2a.jl:91-144).
    The DF tensors carry the active spaces already (drop_occ / drop_vir applied when BOV was made,
    DFERI.jl:31-51); energy = correlation + moints.sd_energy (RMP2a.jl:80-88)."""
    if alg is not None and not isinstance(alg, RMP2hip):
        raise FermiException(f"invalid algorithm {type(alg).__name__} for the MI355X RMP2 backend")
    ctx = _ctx_for(moints, device)
    Ec = ctx.mp2_energy()
    return RMP2Result(Ec, Ec + moints.sd_energy)


def RCCSD(moints, *args, alg=None, options=None, device=0):
    """RCCSD(moints[, T1, T2]; alg) -> RCCSDResult (RCCSDa.jl:46-245 semantics)."""
    if alg is not None and not isinstance(alg, RCCSDhip):
        raise FermiException(f"invalid algorithm {type(alg).__name__} for the MI355X RCCSD backend")
    ctx = _ctx_for(moints, device)
    opts = Options() if options is None else options
    own = len(args) == 0
    if own:
        T1, T2 = ctx.guess(0)
    elif len(args) == 2:
        T1, T2 = args
        if T1.shape != (moints.o, moints.v) or T2.shape != (moints.o, moints.o, moints.v, moints.v):
            raise FermiException("amplitude shapes do not match the orbital spaces")
    else:
        raise FermiException("invalid arguments for RCCSD method")
    # the guess is on the device, and its arrays are free to take the result
    Eguess = ctx.energy() if own else ctx.energy(T1, T2)
    r, nT1, nT2 = ctx._solve(opts, T1, T2, in_place=own)
    Eref = float(moints.sd_energy)
    return RCCSDResult(Eguess + Eref, r.correlation, r.correlation + Eref, nT1, nT2, r.e_conv, r.t_conv, r.niter,
                       bool(r.converged))


def RCCSDpT(ccsd, moints, alg=None, device=0):
    """RCCSDpT(ccsd, moints; alg) -> RCCSDpTResult (ijk.jl:20-150 semantics)."""
    if alg is not None and not isinstance(alg, ijkhip):
        raise FermiException(f"invalid algorithm {type(alg).__name__} for the MI355X (T) backend")
    ctx = _ctx_for(moints, device)
    Et = ctx.triples(ccsd.T1, ccsd.T2)
    return RCCSDpTResult(ccsd, Et + ccsd.energy, Et)


class Mlp:
    """The learned T2-guess network on the GPU (fh_mlp_*): 6 features -> 3 tanh layers -> 1.
    x_mean, x_scale, y_scale hold the feature/target normalisation used with a context."""

    def __init__(self, hidden=128, device=0, seed=0):
        self.L = load_library()
        self.hidden = int(hidden)
        self.device = int(device)
        h = ctypes.c_void_p()
        self._check(self.L.fh_mlp_create(ctypes.byref(h), self.device, self.hidden, int(seed)))
        self.h = h.value
        self.x_mean = np.zeros(6, np.float32)
        self.x_scale = np.ones(6, np.float32)
        self.y_scale = 1.0

    def _check(self, rc):
        if rc != 0:
            raise FermiException(f"libfermihip error {rc}: {self.L.fh_last_error().decode()}")

    @property
    def num_params(self):
        return int(self.L.fh_mlp_num_params(self.h))

    def get_params(self):
        p = np.zeros(self.num_params, np.float32)
        self._check(self.L.fh_mlp_get_params(self.h, _fptr(p)))
        return p

    def set_params(self, p):
        p = np.ascontiguousarray(np.asarray(p, dtype=np.float32))
        if p.shape != (self.num_params,):
            raise FermiException(f"expected {self.num_params} parameters")
        self._check(self.L.fh_mlp_set_params(self.h, _fptr(p)))

    def forward(self, X):
        X = _samples(X)
        Y = np.zeros(X.shape[0], np.float32)
        self._check(self.L.fh_mlp_forward(self.h, X.shape[0], _fptr(X), _fptr(Y)))
        return Y

    def loss_grad(self, X, T):
        X = _samples(X)
        T = np.ascontiguousarray(np.asarray(T, dtype=np.float32))
        g = np.zeros(self.num_params, np.float32)
        loss = ctypes.c_double()
        self._check(self.L.fh_mlp_loss_grad(self.h, X.shape[0], _fptr(X), _fptr(T), ctypes.byref(loss), _fptr(g)))
        return loss.value, g

    def train(self, X, T, epochs=10, batch=8192, lr=1e-3, seed=0):
        X = _samples(X)
        T = np.ascontiguousarray(np.asarray(T, dtype=np.float32))
        hist = np.zeros(max(epochs, 1))
        self._check(self.L.fh_mlp_train(self.h, X.shape[0], _fptr(X), _fptr(T), int(epochs), int(batch), float(lr),
                                        int(seed), _ptr(hist)))
        return hist[:epochs]

    def state(self):
        return {"params": self.get_params(), "hidden": self.hidden, "x_mean": self.x_mean, "x_scale": self.x_scale,
                "y_scale": self.y_scale}

    def close(self):
        if getattr(self, "h", None):
            self.L.fh_mlp_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass
