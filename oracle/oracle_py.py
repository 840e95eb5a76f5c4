"""ctypes bindings of the test oracle (TEST INFRASTRUCTURE ONLY).

Loads oracle/libff_oracle.so (the C restatement, ff_oracle.c) and, when it has been built
in this container, oracle/_ref/libfinflo_ref.so (the reference's own Fortran routines
driven by ref_driver.f90).  Only tests/, __graft_entry__.smoke() and bench.py's
cpu_baseline leg import this module; the product package never does.
"""
import ctypes as C
import os

import numpy as np

from finflo_amd.layout import bc_views, wall_views

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "libff_oracle.so")
REFLIB = os.path.join(HERE, "_ref", "libfinflo_ref.so")
REFDIR = "/root/reference"       # the reference's sources, where there are any

_ora = None
_ref = None


def build():
    """Compile the C restatement (and the reference library when the sources exist)."""
    import subprocess
    subprocess.check_call(["make", "-s", "-C", HERE, "all"])
    if os.path.isfile(os.path.join(REFDIR, "charac.f")):
        subprocess.check_call(["make", "-s", "-C", HERE, "ref"])


def oracle():
    global _ora
    if _ora is None:
        if not os.path.exists(LIB):
            raise RuntimeError("oracle library missing: run make -C oracle")
        _ora = C.CDLL(LIB)
        for fn in ("ffo_state", "ffo_turb", "ffo_save_old", "ffo_update"):
            getattr(_ora, fn).argtypes = [C.c_void_p, C.c_void_p]
            getattr(_ora, fn).restype = None
        _ora.ffo_residual.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p]
        _ora.ffo_residual.restype = None
        _ora.ffo_update_level.argtypes = [C.c_void_p, C.c_void_p, C.c_int]
        _ora.ffo_update_level.restype = None
        _ora.ffo_restrict.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
        _ora.ffo_restrict.restype = None
        _ora.ffo_prolong.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
        _ora.ffo_prolong.restype = None
        _ora.ffo_forcing.argtypes = [C.c_void_p, C.c_void_p, C.c_int]
        _ora.ffo_forcing.restype = None
        _ora.ffo_vcycle.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]
        _ora.ffo_vcycle.restype = None
        _ora.ffo_implicit.argtypes = [C.c_void_p, C.c_void_p, C.c_int]
        _ora.ffo_implicit.restype = None
        _ora.ffo_wall_set.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int]
        _ora.ffo_wall_set.restype = None
        _ora.ffo_wall_forces.argtypes = [C.c_int, C.c_int, C.c_void_p]
        _ora.ffo_wall_forces.restype = None
        _ora.ffo_dromax.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p,
                                    C.c_void_p, C.c_void_p]
        _ora.ffo_dromax.restype = None
        _ora.ffo_bc_set.argtypes = [C.c_int, C.c_void_p, C.c_int]
        _ora.ffo_bc_set.restype = None
        _ora.ffo_reflec.argtypes = [C.c_void_p, C.c_void_p, C.c_int]
        _ora.ffo_reflec.restype = None
        _ora.ffo_statim.argtypes = [C.c_void_p, C.c_void_p, C.c_int]
        _ora.ffo_statim.restype = None
        _ora.ffo_ghostext.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_double, C.c_double]
        _ora.ffo_ghostext.restype = None
        _ora.ffo_ddadi_dir.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int]
        _ora.ffo_ddadi_dir.restype = None
        _ora.ffo_inlout.argtypes = [C.c_void_p, C.c_void_p, C.c_int]
        _ora.ffo_inlout.restype = None
        _ora.ffo_bc_cycle.argtypes = [C.c_int, C.c_int]
        _ora.ffo_bc_cycle.restype = None
    return _ora


def have_ref():
    return os.path.exists(REFLIB)


def ref():
    global _ref
    if _ref is None:
        if not have_ref():
            raise RuntimeError("reference library missing: run make -C oracle ref")
        _ref = C.CDLL(REFLIB)
        for fn in ("ref_state", "ref_turb", "ref_implicit", "ref_update"):
            getattr(_ref, fn).argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p]
            getattr(_ref, fn).restype = None
        _ref.ref_residual.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
        _ref.ref_residual.restype = None
        _ref.ref_wall_set.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
        _ref.ref_wall_set.restype = None
        _ref.ref_wall_forces.argtypes = [C.c_int, C.c_int, C.c_void_p]
        _ref.ref_wall_forces.restype = None
        _ref.ref_reflec.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_int,
                                    C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                                    C.c_void_p, C.c_int]
        _ref.ref_reflec.restype = None
        _ref.ref_ddadi_dir.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_int,
                                       C.c_int]
        _ref.ref_ddadi_dir.restype = None
        _ref.ref_bc_set.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p]
        _ref.ref_bc_set.restype = None
        _ref.ref_inlout.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p]
        _ref.ref_inlout.restype = None
    return _ref


class OracleBlock:
    """Runs the C restatement on a finflo_amd.layout.Block in place."""

    def __init__(self, prm, blk, level=1):
        self.prm, self.blk, self.level = prm, blk, level
        self._view = blk.view_struct()
        # the oracle keeps wall and boundary patches per level: a new block starts without
        oracle().ffo_wall_set(level, None, None, 0)
        oracle().ffo_bc_set(level, None, 0)

    def _args(self):
        return C.byref(self.prm), C.byref(self._view)

    def state(self):
        """STATIM(M,N,INN,.TRUE.): the state, then REFLEC over the boundary patches."""
        oracle().ffo_statim(*self._args(), self.level)

    def set_bcs(self, patches):
        """Boundary patches (finflo_amd.layout.BcPatch) of this level."""
        self._bcv = bc_views(patches)
        self._bcp = patches
        oracle().ffo_bc_set(self.level, self._bcv, len(patches))

    def reflec(self):
        oracle().ffo_reflec(*self._args(), self.level)

    def inlout(self):
        """INLET/OUTLET over the INL and OUT patches with the level's cycle count."""
        oracle().ffo_inlout(*self._args(), self.level)

    def bc_cycle(self, icycle=-1):
        """Set the level's cycle count ICYCLE (icycle < 0: add one, as a cycle starts)."""
        oracle().ffo_bc_cycle(self.level, icycle)

    def ghostext(self, alpha=0.0, beta=0.0):
        oracle().ffo_ghostext(*self._args(), self.level, alpha, beta)

    def turb(self):
        oracle().ffo_turb(*self._args())

    def residual(self, m2=1):
        resi = np.zeros(7)
        oracle().ffo_residual(*self._args(), self.level, m2, resi.ctypes.data)
        return resi

    def implicit(self):
        oracle().ffo_implicit(*self._args(), self.level)

    def ddadi_dir(self, direction, phase):
        """One DDADI direction (0 K, 1 I, 2 J) and phase (0 PRED, 1 DIAG, 2 CORR) on the
        current increments (DTL given)."""
        oracle().ffo_ddadi_dir(*self._args(), direction, phase)

    def save_old(self):
        oracle().ffo_save_old(*self._args())

    def update(self):
        oracle().ffo_update_level(*self._args(), self.level)

    def forcing(self, phase):
        """FORCFU (phase 0) or ADDRES (phase 1) on this level."""
        oracle().ffo_forcing(*self._args(), phase)

    def cycle(self):
        self.bc_cycle()
        self.save_old()
        self.state()
        self.turb()
        r = self.residual()
        self.implicit()
        self.update()
        return r

    def set_walls(self, wparams, patches):
        """Solid-wall patches (finflo_amd.layout.WallPatch) of this level; the arrays stay
        owned by the caller and are written in place."""
        self._wp = wparams
        self._wv = wall_views(patches)
        self._wn = len(patches)
        self._wkeep = patches
        oracle().ffo_wall_set(self.level, C.byref(self._wp), self._wv, len(patches))

    def activate(self):
        """Make this block's walls and boundary patches the ones of its level again (the
        oracle keeps one set per level; several blocks of a level take turns)."""
        if getattr(self, "_wv", None) is not None:
            oracle().ffo_wall_set(self.level, C.byref(self._wp), self._wv, self._wn)
        else:
            oracle().ffo_wall_set(self.level, None, None, 0)
        if getattr(self, "_bcv", None) is not None:
            oracle().ffo_bc_set(self.level, self._bcv, len(self._bcp))
        else:
            oracle().ffo_bc_set(self.level, None, 0)

    def forces(self, patch):
        out = np.zeros(19)
        oracle().ffo_wall_forces(self.level, patch, out.ctypes.data)
        return out

    def dromax(self, state, nblock=1, idrxx=6):
        """DROMXX of this block on the running state (DROMAX, IXERR, INERR); returns the
        new state."""
        dm = C.c_double(state[0])
        ix, inn = C.c_int(state[1]), C.c_int(state[2])
        oracle().ffo_dromax(C.byref(self.prm), C.byref(self._view), idrxx, nblock,
                            C.byref(dm), C.byref(ix), C.byref(inn))
        return dm.value, ix.value, inn.value


class OracleHierarchy:
    """The oracle on a block with its multigrid levels (finest first)."""

    def __init__(self, prm, blocks):
        self.prm = prm
        self.levels = [OracleBlock(prm, b, level=m + 1) for m, b in enumerate(blocks)]

    def restrict(self, m):
        """TRANSF/TRANKE from level m to m+1 (1-based levels)."""
        oracle().ffo_restrict(C.byref(self.prm), C.byref(self.levels[m - 1]._view),
                              C.byref(self.levels[m]._view))

    def prolong(self, m):
        """INTERP/INTERT from level m to m-1."""
        oracle().ffo_prolong(C.byref(self.prm), C.byref(self.levels[m - 1]._view),
                             C.byref(self.levels[m - 2]._view))

    def vcycle(self):
        n = len(self.levels)
        arr = (C.c_void_p * n)(*[C.addressof(l._view) for l in self.levels])
        resi = np.zeros(7)
        oracle().ffo_vcycle(C.byref(self.prm), arr, n, resi.ctypes.data)
        return resi


class RefBlock:
    """Runs the reference's Fortran (through ref_driver.f90) on a Block in place."""

    def __init__(self, prm, blk, level=1):
        self.prm, self.blk, self.level = prm, blk, level
        self.pv = prm.dvec()
        # RESIDI takes first order (INTI = 55) on the coarse levels (ns3c.f:2467-2472)
        inter = list(prm.inter) if level == 1 else [55, 55, 55]
        self.iv = np.array([blk.imax, blk.jmax, blk.kmax, prm.iturb, prm.iflux, prm.idiff,
                            inter[0], inter[1], inter[2], level, prm.kover, prm.katol, 1,
                            prm.istres, prm.fullns, prm.turcor, prm.ddadi, 0],
                           dtype=np.int32)
        # the reference driver keeps wall patches per level: a new block starts without any
        if have_ref():
            z = np.zeros(32)
            ref().ref_wall_set(level, 0, z.ctypes.data, z.ctypes.data, z.ctypes.data)
            ref().ref_bc_set(level, 0, z.ctypes.data, z.ctypes.data)

    def _a(self):
        return (self.blk.F.ctypes.data, self.blk.ntot, self.pv.ctypes.data,
                self.iv.ctypes.data)

    def state(self):
        """STATIM: the state, then (REFLEL = .TRUE.) REFLEC over the patches of set_bcs."""
        ref().ref_state(*self._a())
        if getattr(self, "_bcs", None):
            self.reflec(self._bcs)

    def set_bcs(self, patches):
        """REFLEC's patches for STATIM, and the INL/OUT patches for the reference's INLET
        and OUTLET (its ICYCLE restarts at 0; INLET 4 writes BOUNP/BOUNPD into these
        patches' arrays)."""
        from finflo_amd.layout import BOUN_ARRAYS
        self._bcs = list(patches)
        io = [bp for bp in patches if bp.ibc in (3, 5)]
        self._io = io
        n = len(io)
        self._bints = np.zeros((max(n, 1), 8), dtype=np.int32)
        self._bptrs = np.zeros((max(n, 1), len(BOUN_ARRAYS)), dtype=np.uint64)
        self._bkeep = []
        for l, bp in enumerate(io):
            self._bints[l, :7] = [bp.ibc, bp.iface, bp.kx1, bp.kx2, bp.ky1, bp.ky2, bp.inlout]
            for q, name in enumerate(BOUN_ARRAYS):
                a = bp.boun[name]
                if a is None:
                    a = np.zeros(bp.size)
                    self._bkeep.append(a)
                self._bptrs[l, q] = a.ctypes.data
        self.iv[17] = 0
        ref().ref_bc_set(self.level, n, self._bints.ctypes.data, self._bptrs.ctypes.data)

    def inlout(self):
        """The reference's INLET/OUTLET over the INL/OUT patches (directions K, I, J)."""
        ref().ref_inlout(*self._a())

    def bc_cycle(self, icycle):
        self.iv[17] = icycle

    def turb(self):
        ref().ref_turb(*self._a())

    def residual(self, m2=1):
        resi = np.zeros(7)
        self.iv[12] = m2
        ref().ref_residual(*self._a(), resi.ctypes.data)
        return resi

    def implicit(self):
        ref().ref_implicit(*self._a())

    def ddadi_dir(self, direction, phase):
        """The reference's PRED/DIAG/CORR(KE) of one DDADI direction (phase 3: all three)."""
        ref().ref_ddadi_dir(*self._a(), direction, phase)

    def save_old(self):
        b = self.blk
        for new, old in (("TEMP", "TOLD"), ("U", "UOLD"), ("V", "VOLD"), ("W", "WOLD"),
                         ("PDIFF", "POLD"), ("RK", "RKOLD"), ("REPS", "EPSOLD")):
            b[old] = b[new]

    def update(self):
        ref().ref_update(*self._a())

    def cycle(self):
        self.iv[17] += 1
        self.save_old()
        self.state()
        self.turb()
        r = self.residual()
        self.implicit()
        self.update()
        return r

    def set_walls(self, wparams, patches):
        """The same patches for the reference's BOTSKE (ref_wall_set)."""
        from finflo_amd.layout import WALL_ARRAYS
        n = len(patches)
        self._wints = np.zeros((max(n, 1), 8), dtype=np.int32)
        self._wptrs = np.zeros((max(n, 1), len(WALL_ARRAYS)), dtype=np.uint64)
        for l, wp in enumerate(patches):
            self._wints[l, :6] = [wp.iface, wp.kx1, wp.kx2, wp.ky1, wp.ky2, wp.iheat]
            self._wptrs[l] = [wp.a[a].ctypes.data for a in WALL_ARRAYS]
        self._wenv = wparams.dvec()
        ref().ref_wall_set(self.level, n, self._wints.ctypes.data, self._wenv.ctypes.data,
                           self._wptrs.ctypes.data)

    def forces(self, patch):
        out = np.zeros(19)
        ref().ref_wall_forces(self.level, patch, out.ctypes.data)
        return out

    def reflec(self, patches):
        """The reference's REFLEC over the given boundary patches (BcPatch)."""
        n = len(patches)
        ints = np.zeros((max(n, 1), 8), dtype=np.int32)
        tsurf = np.zeros(max(n, 1))
        arrs = {k: [] for k in ("uwall", "vwall", "wwall")}
        for l, bp in enumerate(patches):
            ints[l] = [bp.ibc, bp.iface, bp.kx1, bp.kx2, bp.ky1, bp.ky2, bp.iheat, bp.viscous]
            tsurf[l] = bp.tsurf
            for k in arrs:
                a = getattr(bp, k)
                arrs[k].append(np.zeros(bp.size) if a is None else np.asarray(a, float))
        cat = {k: (np.concatenate(v) if v else np.zeros(1)) for k, v in arrs.items()}
        ref().ref_reflec(*self._a(), n, ints.ctypes.data, tsurf.ctypes.data,
                         cat["uwall"].ctypes.data, cat["vwall"].ctypes.data,
                         cat["wwall"].ctypes.data, len(cat["uwall"]))
