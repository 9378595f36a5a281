"""ctypes mirrors of the library's internal launch structures (dslash.h,
qcu_common.h) for tests that look at a kernel's intermediate results.  The
symbols are the C++ ones that libqcu.so exports; test_internals_cpu.py checks
the layouts on the host."""
import ctypes

from qcu_mrhs_amd import _lib

_i, _d, _l, _vp = ctypes.c_int, ctypes.c_double, ctypes.c_long, ctypes.c_void_p
MAX_GROUPS, NUM_SLOTS = 8, 13
ALPHA, OMEGA = 0, 1


class Geom(ctypes.Structure):
    _fields_ = [("L", _i * 4), ("Lxh", _i), ("Vh", _i)]


class Tune(ctypes.Structure):
    _fields_ = [("variant", _i), ("by", _i), ("bz", _i), ("spw", _i)]


class DslashArgs(ctypes.Structure):
    _fields_ = [("out", _vp), ("inp", _vp), ("gauge", _vp), ("xpay", _vp), ("coef", _d), ("g", Geom), ("Nc", _i), ("R", _i),
                ("parity", _i), ("dagger", _i), ("prec", _i), ("tune", Tune), ("keep_order", ctypes.c_bool),
                ("clover", _vp), ("clover_in", _vp)]


class SegTab(ctypes.Structure):
    _fields_ = [("G", _i), ("Rtot", _i), ("Rmax", _i), ("n", _l), ("R", _i * MAX_GROUPS), ("base", _i * MAX_GROUPS),
                ("spw", _i * MAX_GROUPS), ("done", _vp)]


class SegRows(ctypes.Structure):
    _fields_ = [("n", _i * MAX_GROUPS), ("sites", _i * MAX_GROUPS), ("off", _l * MAX_GROUPS), ("total", _l)]


def geom(L):
    return Geom((_i * 4)(*L), L[0] // 2, L[0] * L[1] * L[2] * L[3] // 2)


def args(L, Nc, R, prec, variant=0, **kw):
    return DslashArgs(coef=1.0, g=geom(L), Nc=Nc, R=R, parity=1, dagger=0, prec=prec, tune=Tune(variant=variant), **kw)


def groups(L, Nc, sizes):
    t = SegTab(G=len(sizes), Rtot=sum(sizes), Rmax=max(sizes), n=geom(L).Vh * 4 * Nc)
    for k, R in enumerate(sizes):
        t.R[k], t.base[k], t.spw[k] = R, sum(sizes[:k]), 1
    return t


_A, _G, _T, _W = (ctypes.POINTER(c) for c in (DslashArgs, Geom, SegTab, SegRows))
_SYMBOLS = {
    "dslash_resolve": ("_ZN3qcu14dslash_resolveERKNS_10DslashArgsE", Tune, [_A]),
    "dslash_lane_clover_fused": ("_ZN3qcu24dslash_lane_clover_fusedERKNS_10DslashArgsERKNS_10DslashTuneE", ctypes.c_bool,
                                 [_A, ctypes.POINTER(Tune)]),
    "dslash_dots_partials": ("_ZN3qcu20dslash_dots_partialsERKNS_4GeomEiii", _l, [_G, _i, _i, _i]),
    "dslash_dots_rows": ("_ZN3qcu16dslash_dots_rowsERKNS_4GeomEiiRKNS_6SegTabERNS_7SegRowsE", ctypes.c_bool,
                         [_G, _i, _i, _T, _W]),
    "launch_dslash_dots": ("_ZN3qcu18launch_dslash_dotsERKNS_10DslashArgsENS_8DotsKindEPKvPdlPNS_2CxIdEEP12ihipStream_t",
                           _i, [_A, _i, _vp, _vp, _l, _vp, _vp]),
    "launch_dslash_clover": ("_ZN3qcu20launch_dslash_cloverERKNS_10DslashArgsEP12ihipStream_t", _i, [_A, _vp]),
    "launch_dslash_lane_dots_groups": ("_ZN3qcu30launch_dslash_lane_dots_groupsERKNS_10DslashArgsENS_8DotsKindEPKvRKNS_6SegTab"
                                       "ERKNS_7SegRowsEPdiiP12ihipStream_t", _i, [_A, _i, _vp, _T, _W, _vp, _i, _i, _vp]),
    "launch_dslash_lane_groups": ("_ZN3qcu25launch_dslash_lane_groupsERKNS_10DslashArgsERKNS_6SegTabEiiP12ihipStream_t", _i,
                                  [_A, _T, _i, _i, _vp]),
}


def call(name, *a):
    symbol, res, types = _SYMBOLS[name]
    f = getattr(_lib.load(), symbol)
    f.restype, f.argtypes = res, types
    return f(*[ctypes.byref(v) if isinstance(v, ctypes.Structure) else v for v in a])
