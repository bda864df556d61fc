"""Python bindings of libagbnp3 through its C-ABI (ctypes).

Mirrors the reference API of agbnp3.h (agbnp3_initialize, agbnp3_new,
agbnp3_ener, agbnp3_delete, agbnp3_terminate and the NeighList struct of
nblist.h) with the same argument meaning and AGBNP_OK / AGBNP_ERR returns,
plus the extensions of include/agbnp3_amd.h.  There is no CPU fallback:
loading fails loudly when libagbnp3.so is missing, and agbnp3_initialize
returns AGBNP_ERR when no GPU is visible.
"""
import ctypes
import os

import numpy as np

from . import _paths

AGBNP_OK = 2
AGBNP_ERR = -1
OPT_HB_FIXED = 1
OPT_SPLINE_FIXED = 2
OPT_TIMING = 4
ENERGY_NAMES = ("egb", "evdw", "ecorr_vdw", "ecav", "ecorr_cav", "ehb", "mol_volume")

# exported C symbols, as declared in include/agbnp3.h and include/agbnp3_amd.h
EXPORTED = (
    "agbnp3_initialize", "agbnp3_terminate", "agbnp3_new", "agbnp3_delete", "agbnp3_ener",
    "agbnp_initialize", "agbnp_terminate", "agbnp_delete",
    "agbnp3_set_options", "agbnp3_ener_device", "agbnp3_ener_static", "agbnp3_sync", "agbnp3_stream",
    "agbnp3_natoms",
    "agbnp3_get_int2ext", "agbnp3_get_near_list", "agbnp3_get_tables", "agbnp3_get_internal",
    "agbnp3_get_counts", "agbnp3_get_routes", "agbnp3_kernel_times", "agbnp3_q4_tables",
    "agbnp3_get_tuning", "agbnp3_set_tuning", "agbnp3_tune", "agbnp3_tune_table_save", "agbnp3_tune_table_load",
    "agbnp3_tune_table_clear",
    "agbnp3_batch_new", "agbnp3_batch_delete", "agbnp3_batch_offsets", "agbnp3_batch_set_options",
    "agbnp3_batch_ener_device", "agbnp3_batch_ener", "agbnp3_batch_sync", "agbnp3_batch_stream",
    "agbnp3_batch_graph_capture", "agbnp3_batch_graph_launch", "agbnp3_batch_kernel_times",
    "agbnp3_batch_get_tuning", "agbnp3_batch_set_tuning", "agbnp3_batch_tune",
    "agbnp3_set_nblist_reuse", "agbnp3_batch_set_nblist_reuse", "agbnp3_nblist_rebuilds",
    "agbnp3_sg_new", "agbnp3_sg_delete", "agbnp3_sg_size", "agbnp3_sg_get_params", "agbnp3_sg_set_params",
    "agbnp3_sg_reserve", "agbnp3_batch_sg_collect", "agbnp3_sg_dataset", "agbnp3_sg_fit", "agbnp3_sg_train",
    "agbnp3_sg_set_loss", "agbnp3_sg_train_rows",
    "agbnp3_sg_grads", "agbnp3_sg_infer", "agbnp3_sg_attach", "agbnp3_batch_sg_attach", "agbnp3_sg_stats",
    "agbnp3_batch_sg_stats", "agbnp3_sg_lists", "agbnp3_batch_sg_lists", "agbnp3_sg_modes", "agbnp3_batch_sg_modes",
)
TUNING_PARAMS = ("rows", "desc_chunk", "chain_chunk", "desc_grid", "gb_grid", "chain_grid", "cap", "tree_grid")
NBLIST_EXPORTED = ("nblist_reset_neighbor_list", "nblist_delete_neighbor_list", "nblist_reallocate_neighbor_list")


class NeighVector(ctypes.Structure):
    _fields_ = [("x", ctypes.c_double), ("y", ctypes.c_double), ("z", ctypes.c_double)]


class NeighList(ctypes.Structure):
    """ABI of nblist.h:39-70."""
    _fields_ = [
        ("natoms", ctypes.c_int), ("neighl_size", ctypes.c_int),
        ("nne", ctypes.POINTER(ctypes.c_int)), ("neighl1", ctypes.POINTER(ctypes.c_int)),
        ("neighl", ctypes.POINTER(ctypes.POINTER(ctypes.c_int))),
        ("idx_remap", ctypes.c_int),
        ("int2ext", ctypes.POINTER(ctypes.c_int)), ("ext2int", ctypes.POINTER(ctypes.c_int)),
        ("pbc", ctypes.c_int),
        ("pbc_trans1", ctypes.POINTER(NeighVector)), ("pbc_trans", ctypes.POINTER(ctypes.POINTER(NeighVector))),
        ("data", ctypes.c_int),
        ("data_index1", ctypes.POINTER(ctypes.c_void_p)), ("data_index", ctypes.POINTER(ctypes.c_void_p)),
    ]


_lib = None
_nb = None


def load():
    """Load libagbnp3.so (and libnblist.so); raises if they are not built."""
    global _lib, _nb
    if _lib is None:
        for p in (_paths.LIBNBLIST, _paths.LIBAGBNP3):
            if not os.path.exists(p):
                raise RuntimeError(f"{p} is not built: run `python -c 'import __graft_entry__ as g; g.build()'`")
        _nb = ctypes.CDLL(_paths.LIBNBLIST, mode=ctypes.RTLD_GLOBAL)
        L = ctypes.CDLL(_paths.LIBAGBNP3)
        vp, ci, dp, ip = ctypes.c_void_p, ctypes.c_int, ctypes.c_double, ctypes.c_void_p
        L.agbnp3_initialize.restype = ci
        L.agbnp3_terminate.restype = None
        L.agbnp3_new.restype = ci
        L.agbnp3_new.argtypes = [ctypes.POINTER(ci), ci, vp, vp, vp, vp, vp, dp, dp, vp, vp, vp, vp, ip, vp, ci, ip,
                                 ctypes.POINTER(NeighList), ci]
        L.agbnp3_delete.argtypes = [ci]
        L.agbnp3_ener.restype = ci
        L.agbnp3_ener.argtypes = [ci, ci] + [vp] * 17
        L.agbnp3_set_options.argtypes = [ci, ci]
        L.agbnp3_ener_device.restype = ci
        L.agbnp3_ener_device.argtypes = [ci] + [vp] * 11
        L.agbnp3_ener_static.restype = ci
        L.agbnp3_ener_static.argtypes = [ci] + [vp] * 11
        L.agbnp3_sync.argtypes = [ci]
        L.agbnp3_stream.restype = vp
        L.agbnp3_stream.argtypes = [ci]
        L.agbnp3_natoms.argtypes = [ci, ctypes.POINTER(ci), ctypes.POINTER(ci)]
        L.agbnp3_get_int2ext.argtypes = [ci, vp]
        L.agbnp3_get_near_list.argtypes = [ci, vp, vp, ci]
        L.agbnp3_get_tables.argtypes = [ci, vp, vp, vp]
        L.agbnp3_get_internal.argtypes = [ci, ctypes.c_char_p, vp]
        L.agbnp3_get_counts.argtypes = [ci, vp]
        L.agbnp3_get_routes.argtypes = [ci, vp]
        L.agbnp3_kernel_times.argtypes = [ci, vp, ci, ctypes.c_char_p, ci]
        L.agbnp3_q4_tables.argtypes = [ci, vp, vp, vp, vp]
        L.agbnp3_get_tuning.argtypes = [ci, vp, ci]
        L.agbnp3_set_tuning.argtypes = [ci, vp, ci]
        L.agbnp3_tune.argtypes = [ci, vp, vp, vp, ci, ctypes.c_char_p, ci]
        L.agbnp3_tune_table_save.argtypes = [ctypes.c_char_p]
        L.agbnp3_tune_table_load.argtypes = [ctypes.c_char_p]
        L.agbnp3_batch_new.argtypes = [ctypes.POINTER(ci), ci, vp]
        L.agbnp3_batch_delete.argtypes = [ci]
        L.agbnp3_batch_offsets.argtypes = [ci, ctypes.POINTER(ci), vp]
        L.agbnp3_batch_set_options.argtypes = [ci, ci]
        L.agbnp3_batch_ener_device.argtypes = [ci] + [vp] * 11
        L.agbnp3_batch_ener.argtypes = [ci, vp, vp, vp, vp]
        L.agbnp3_batch_sync.argtypes = [ci]
        L.agbnp3_batch_stream.restype = vp
        L.agbnp3_batch_stream.argtypes = [ci]
        L.agbnp3_batch_graph_capture.argtypes = [ci] + [vp] * 11
        L.agbnp3_batch_graph_launch.argtypes = [ci]
        L.agbnp3_batch_kernel_times.argtypes = [ci, vp, ci, ctypes.c_char_p, ci]
        L.agbnp3_batch_get_tuning.argtypes = [ci, vp, ci]
        L.agbnp3_batch_set_tuning.argtypes = [ci, vp, ci]
        L.agbnp3_batch_tune.argtypes = [ci, vp, vp, vp, ci, ctypes.c_char_p, ci]
        L.agbnp3_set_nblist_reuse.argtypes = [ci, ctypes.c_float, ci]
        L.agbnp3_batch_set_nblist_reuse.argtypes = [ci, ctypes.c_float, ci]
        L.agbnp3_nblist_rebuilds.argtypes = [ci, ctypes.POINTER(ci), ctypes.POINTER(ci)]
        u64, f32 = ctypes.c_ulonglong, ctypes.c_float
        L.agbnp3_sg_new.argtypes = [ctypes.POINTER(ci), u64]
        L.agbnp3_sg_delete.argtypes = [ci]
        L.agbnp3_sg_get_params.argtypes = [ci, vp, ci]
        L.agbnp3_sg_set_params.argtypes = [ci, vp, ci]
        L.agbnp3_sg_reserve.argtypes = [ci, ci]
        L.agbnp3_batch_sg_collect.argtypes = [ci, ci, vp, vp, vp]
        L.agbnp3_sg_dataset.argtypes = [ci, ctypes.POINTER(ci), vp, vp]
        L.agbnp3_sg_fit.argtypes = [ci, f32, u64]
        L.agbnp3_sg_train.argtypes = [ci, ci, ci, f32, f32, u64, vp]
        L.agbnp3_sg_set_loss.argtypes = [ci, f32, f32]
        L.agbnp3_sg_train_rows.argtypes = [ci, vp, vp, vp]
        L.agbnp3_sg_grads.argtypes = [ci, ci, ci, vp, vp]
        L.agbnp3_sg_infer.argtypes = [ci, vp, ci, vp, vp]
        L.agbnp3_sg_attach.argtypes = [ci, ci, ci]
        L.agbnp3_batch_sg_attach.argtypes = [ci, ci, ci]
        L.agbnp3_sg_stats.argtypes = [ci, vp, vp]
        L.agbnp3_batch_sg_stats.argtypes = [ci, vp, vp]
        L.agbnp3_sg_lists.argtypes = [ci, vp, vp]
        L.agbnp3_batch_sg_lists.argtypes = [ci, vp, vp]
        L.agbnp3_sg_modes.argtypes = [ci, vp]
        L.agbnp3_batch_sg_modes.argtypes = [ci, vp]
        _nb.nblist_reallocate_neighbor_list.argtypes = [ctypes.POINTER(NeighList), ci, ci]
        _nb.nblist_reset_neighbor_list.argtypes = [ctypes.POINTER(NeighList)]
        _nb.nblist_delete_neighbor_list.argtypes = [ctypes.POINTER(NeighList)]
        _lib = L
    return _lib


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def make_conntbl(conn_nne, conn_neighl1):
    """A NeighList filled through libnblist, as a caller would build it."""
    load()
    nl = NeighList()
    _nb.nblist_reset_neighbor_list(ctypes.byref(nl))
    n = int(len(conn_nne))
    size = max(int(len(conn_neighl1)), 1)
    if _nb.nblist_reallocate_neighbor_list(ctypes.byref(nl), n, size) != 0:
        raise RuntimeError("nblist_reallocate_neighbor_list failed")
    base = ctypes.addressof(nl.neighl1.contents)
    off = 0
    for i in range(n):
        nl.nne[i] = int(conn_nne[i])
        nl.neighl[i] = ctypes.cast(base + 4 * off, ctypes.POINTER(ctypes.c_int))
        for k in range(int(conn_nne[i])):
            nl.neighl1[off + k] = int(conn_neighl1[off + k])
        off += int(conn_nne[i])
    return nl


# ---------------------------------------------------------- reference API
def agbnp3_initialize():
    return load().agbnp3_initialize()


def agbnp3_terminate():
    load().agbnp3_terminate()


def agbnp3_new(natoms, x, y, z, r, charge, dielectric_in, dielectric_out, igamma, sgamma, ialpha, salpha,
               hbtype, hbcorr, nhydrogen, ihydrogen, conntbl, verbose=0):
    """Returns (rc, tag)."""
    L = load()
    d = [np.ascontiguousarray(a, np.float64) for a in (x, y, z, r, charge, igamma, sgamma, ialpha, salpha, hbcorr)]
    hb = np.ascontiguousarray(hbtype, np.int32)
    ih = np.ascontiguousarray(ihydrogen, np.int32)
    tag = ctypes.c_int(-1)
    rc = L.agbnp3_new(ctypes.byref(tag), int(natoms), _p(d[0]), _p(d[1]), _p(d[2]), _p(d[3]), _p(d[4]),
                      float(dielectric_in), float(dielectric_out), _p(d[5]), _p(d[6]), _p(d[7]), _p(d[8]),
                      _p(hb), _p(d[9]), int(nhydrogen), _p(ih), ctypes.byref(conntbl) if conntbl is not None else None,
                      int(verbose))
    return rc, tag.value


def agbnp3_ener(tag, init, x, y, z):
    """Returns (rc, dict of outputs) with arrays in caller order."""
    L = load()
    x, y, z = (np.ascontiguousarray(a, np.float64) for a in (x, y, z))
    n = x.size
    sp, br, sa = np.zeros(n), np.zeros(n), np.zeros(n)
    g = [np.zeros((n, 3)) for _ in range(4)]
    e = [ctypes.c_double(0.0) for _ in range(7)]
    rc = L.agbnp3_ener(int(tag), int(init), _p(x), _p(y), _p(z), _p(sp), _p(br), ctypes.byref(e[6]), _p(sa),
                       ctypes.byref(e[0]), _p(g[0]), ctypes.byref(e[1]), ctypes.byref(e[2]), _p(g[1]),
                       ctypes.byref(e[3]), ctypes.byref(e[4]), _p(g[2]), ctypes.byref(e[5]), _p(g[3]))
    out = dict(zip(ENERGY_NAMES, (v.value for v in e)))
    out.update(sp=sp, br=br, surf_area=sa, dgbdr=g[0], dvwdr=g[1], decav=g[2], dehb=g[3])
    return rc, out


class HostOutputs:
    """Caller-owned output arrays of agbnp3_ener, allocated once and reused
    (as a C caller's would be): fresh arrays each call would add first-touch
    page faults to every call."""

    def __init__(self, n):
        self.n = n
        self.sp, self.br, self.sa = np.zeros(n), np.zeros(n), np.zeros(n)
        self.g = [np.zeros((n, 3)) for _ in range(4)]
        self.e = [ctypes.c_double(0.0) for _ in range(7)]
        self._args = None

    def args(self):
        if self._args is None:
            e, g = self.e, self.g
            self._args = (_p(self.sp), _p(self.br), ctypes.byref(e[6]), _p(self.sa), ctypes.byref(e[0]), _p(g[0]),
                          ctypes.byref(e[1]), ctypes.byref(e[2]), _p(g[1]), ctypes.byref(e[3]), ctypes.byref(e[4]),
                          _p(g[2]), ctypes.byref(e[5]), _p(g[3]))
        return self._args


def agbnp3_ener_into(tag, x, y, z, outs):
    """agbnp3_ener on contiguous float64 x, y, z into preallocated HostOutputs; returns rc."""
    return load().agbnp3_ener(int(tag), 0, _p(x), _p(y), _p(z), *outs.args())


def agbnp3_delete(tag):
    return load().agbnp3_delete(int(tag))


agbnp_initialize = agbnp3_initialize
agbnp_terminate = agbnp3_terminate
agbnp_delete = agbnp3_delete


def q4_tables(radii):
    """Host-side Q4 tables (no GPU): (y, y2, dx, dxinv) for radius types `radii`."""
    L = load()
    r = np.ascontiguousarray(radii, np.float32)
    nt = r.size
    y = np.zeros(nt * nt * 512, np.float32)
    y2 = np.zeros_like(y)
    dx = np.zeros(2, np.float32)
    if L.agbnp3_q4_tables(nt, _p(r), _p(y), _p(y2), _p(dx)) != AGBNP_OK:
        raise RuntimeError("agbnp3_q4_tables failed")
    return y.reshape(nt * nt, 512), y2.reshape(nt * nt, 512), float(dx[0]), float(dx[1])


# ------------------------------------------------------------ convenience
class Instance:
    """One agbnp3_new() instance built from a synth.System."""

    def __init__(self, s, options=0):
        if agbnp3_initialize() != AGBNP_OK:
            raise RuntimeError("agbnp3_initialize failed (no GPU?)")
        self.sys = s
        self.conn = make_conntbl(s.conn_nne, s.conn_neighl1)
        rc, tag = agbnp3_new(s.natoms, s.x, s.y, s.z, s.r, s.charge, s.eps_in, s.eps_out, s.igamma, s.sgamma,
                             s.ialpha, s.salpha, s.hbtype, s.hbcorr, s.nhydrogen, s.ihydrogen, self.conn)
        if rc != AGBNP_OK:
            raise RuntimeError("agbnp3_new failed")
        self.tag = tag
        self.n = s.natoms
        if options:
            self.set_options(options)

    def set_options(self, options):
        if load().agbnp3_set_options(self.tag, int(options)) != AGBNP_OK:
            raise RuntimeError("agbnp3_set_options failed")

    def ener(self, x=None, y=None, z=None):
        s = self.sys
        rc, out = agbnp3_ener(self.tag, 0, s.x if x is None else x, s.y if y is None else y,
                              s.z if z is None else z)
        if rc != AGBNP_OK:
            raise RuntimeError("agbnp3_ener failed")
        return out

    def delete(self):
        if self.tag is not None:
            agbnp3_delete(self.tag)
            self.tag = None
            _nb.nblist_delete_neighbor_list(ctypes.byref(self.conn))

    def nheavy(self):
        n, nh = ctypes.c_int(), ctypes.c_int()
        load().agbnp3_natoms(self.tag, ctypes.byref(n), ctypes.byref(nh))
        return nh.value

    def int2ext(self):
        out = np.zeros(self.n, np.int32)
        load().agbnp3_get_int2ext(self.tag, _p(out))
        return out

    def near_list(self, cap=256):
        nh = self.nheavy()
        nne = np.zeros(max(nh, 1), np.int32)
        nbr = np.full((max(nh, 1), cap), -1, np.int32)
        load().agbnp3_get_near_list(self.tag, _p(nne), _p(nbr), cap)
        return nne[:nh], nbr[:nh]

    def tables(self):
        L = load()
        nt = L.agbnp3_get_tables(self.tag, None, None, None)
        y = np.zeros(nt * nt * 512, np.float32)
        y2 = np.zeros_like(y)
        radii = np.zeros(nt, np.float32)
        L.agbnp3_get_tables(self.tag, _p(y), _p(y2), _p(radii))
        return y.reshape(nt * nt, 512), y2.reshape(nt * nt, 512), radii

    def internal(self, name):
        out = np.zeros(self.n)
        if load().agbnp3_get_internal(self.tag, name.encode(), _p(out)) != AGBNP_OK:
            raise KeyError(name)
        return out

    def counts(self):
        c = np.zeros(7, np.int64)
        load().agbnp3_get_counts(self.tag, _p(c))
        return dict(kept_overlaps=int(c[0]), evaluated_overlaps=int(c[1]), water_sites=int(c[2]),
                    near_pairs=int(c[3]), max_row=int(c[4]), tree_fallback_volumes=int(c[5]),
                    tree_fallback_derivatives=int(c[6]))

    def routes(self):
        """The sum of agbnp3_get_routes (agbnp3_amd.h) for the last call."""
        r = ctypes.c_int(0)
        if load().agbnp3_get_routes(self.tag, ctypes.byref(r)) != AGBNP_OK:
            raise RuntimeError("agbnp3_get_routes failed")
        return r.value

    def kernel_times(self):
        ms = np.zeros(64, np.float32)
        names = ctypes.create_string_buffer(4096)
        k = load().agbnp3_kernel_times(self.tag, _p(ms), 64, names, 4096)
        return dict(zip(names.value.decode().split(";"), ms[:k].tolist())) if k > 0 else {}

    def stream(self):
        return load().agbnp3_stream(self.tag)

    def ener_device(self, x, y, z, sp, br, sa, dgbdr, dvwdr, decav, dehb, energies):
        """All arguments are device pointers (ints)."""
        return load().agbnp3_ener_device(self.tag, x, y, z, sp, br, sa, dgbdr, dvwdr, decav, dehb, energies)

    def sync(self):
        return load().agbnp3_sync(self.tag)

    def get_tuning(self):
        p = np.zeros(len(TUNING_PARAMS), np.int32)
        if load().agbnp3_get_tuning(self.tag, _p(p), p.size) != AGBNP_OK:
            raise RuntimeError("agbnp3_get_tuning failed")
        return dict(zip(TUNING_PARAMS, p.tolist()))

    def set_tuning(self, **kw):
        t = self.get_tuning()
        t.update(kw)
        p = np.array([t[k] for k in TUNING_PARAMS], np.int32)
        if load().agbnp3_set_tuning(self.tag, _p(p), p.size) != AGBNP_OK:
            raise RuntimeError("agbnp3_set_tuning failed")

    def set_nblist_reuse(self, skin, every=0):
        if load().agbnp3_set_nblist_reuse(self.tag, float(skin), int(every)) != AGBNP_OK:
            raise RuntimeError("agbnp3_set_nblist_reuse failed")

    def sg_attach(self, model, every):
        if load().agbnp3_sg_attach(self.tag, model.id if model is not None else -1, int(every)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_attach failed")

    def sg_stats(self):
        err, mode = np.zeros(1), np.zeros(1, np.int32)
        if load().agbnp3_sg_stats(self.tag, _p(err), _p(mode)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_stats failed")
        return float(err[0]), int(mode[0])

    def sg_modes(self):
        """Calls since sg_attach that were plain, surrogate, and surrogate with
        the plain kernels for out-of-window atoms."""
        c = np.zeros(3, np.int32)
        if load().agbnp3_sg_modes(self.tag, _p(c)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_modes failed")
        return tuple(int(v) for v in c)

    def sg_lists(self):
        """(descriptor neighbour-list builds, overflow flag) since sg_attach."""
        b, o = np.zeros(1, np.int32), np.zeros(1, np.int32)
        if load().agbnp3_sg_lists(self.tag, _p(b), _p(o)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_lists failed")
        return int(b[0]), int(o[0])

    def nblist_rebuilds(self):
        """(calls, candidate rebuilds) since set_nblist_reuse."""
        c, r = ctypes.c_int(), ctypes.c_int()
        if load().agbnp3_nblist_rebuilds(self.tag, ctypes.byref(c), ctypes.byref(r)) != AGBNP_OK:
            raise RuntimeError("agbnp3_nblist_rebuilds failed")
        return c.value, r.value

    def tune(self, x, y, z, reps=3):
        """Autotune on device coordinates (pointers); returns the trial report."""
        rep = ctypes.create_string_buffer(1 << 16)
        if load().agbnp3_tune(self.tag, x, y, z, int(reps), rep, len(rep)) != AGBNP_OK:
            raise RuntimeError("agbnp3_tune failed")
        return rep.value.decode()


class Batch:
    """agbnp3_batch_new() over a list of Instance objects."""

    def __init__(self, instances):
        L = load()
        tags = np.array([i.tag for i in instances], np.int32)
        b = ctypes.c_int(-1)
        if L.agbnp3_batch_new(ctypes.byref(b), tags.size, _p(tags)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_new failed")
        self.id = b.value
        self.nsys = tags.size
        off = np.zeros(self.nsys + 1, np.int32)
        L.agbnp3_batch_offsets(self.id, None, _p(off))
        self.offsets = off
        self.n = int(off[-1])

    def set_options(self, options):
        if load().agbnp3_batch_set_options(self.id, int(options)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_set_options failed")

    def ener(self, x, y, z):
        """Host arrays (concatenated caller order); returns a dict like agbnp3_ener's, energies [nsys, 7]."""
        x, y, z = (np.ascontiguousarray(a, np.float64) for a in (x, y, z))
        n = self.n
        out = np.zeros(15 * n + 7 * self.nsys)
        if load().agbnp3_batch_ener(self.id, _p(x), _p(y), _p(z), _p(out)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_ener failed")
        return dict(sp=out[:n], br=out[n:2 * n], surf_area=out[2 * n:3 * n],
                    dgbdr=out[3 * n:6 * n].reshape(n, 3), dvwdr=out[6 * n:9 * n].reshape(n, 3),
                    decav=out[9 * n:12 * n].reshape(n, 3), dehb=out[12 * n:15 * n].reshape(n, 3),
                    energies=out[15 * n:].reshape(self.nsys, 7))

    def ener_device(self, *ptrs):
        return load().agbnp3_batch_ener_device(self.id, *ptrs)

    def graph_capture(self, *ptrs):
        if load().agbnp3_batch_graph_capture(self.id, *ptrs) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_graph_capture failed")

    def graph_launch(self):
        return load().agbnp3_batch_graph_launch(self.id)

    def sync(self):
        return load().agbnp3_batch_sync(self.id)

    def stream(self):
        return load().agbnp3_batch_stream(self.id)

    def kernel_times(self):
        ms = np.zeros(64, np.float32)
        names = ctypes.create_string_buffer(4096)
        k = load().agbnp3_batch_kernel_times(self.id, _p(ms), 64, names, 4096)
        return dict(zip(names.value.decode().split(";"), ms[:k].tolist())) if k > 0 else {}

    def get_tuning(self):
        p = np.zeros(len(TUNING_PARAMS), np.int32)
        if load().agbnp3_batch_get_tuning(self.id, _p(p), p.size) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_get_tuning failed")
        return dict(zip(TUNING_PARAMS, p.tolist()))

    def set_tuning(self, **kw):
        t = self.get_tuning()
        t.update(kw)
        p = np.array([t[k] for k in TUNING_PARAMS], np.int32)
        if load().agbnp3_batch_set_tuning(self.id, _p(p), p.size) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_set_tuning failed")

    def sg_attach(self, model, every):
        if load().agbnp3_batch_sg_attach(self.id, model.id if model is not None else -1, int(every)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_sg_attach failed")

    def sg_stats(self):
        err, mode = np.zeros(self.nsys), np.zeros(self.nsys, np.int32)
        if load().agbnp3_batch_sg_stats(self.id, _p(err), _p(mode)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_sg_stats failed")
        return err, mode

    def sg_modes(self):
        """Per system: calls since sg_attach in modes 0 (plain), 1 (surrogate), 2 (surrogate with
        the plain kernels for out-of-window atoms), as an [nsys, 3] array."""
        c = np.zeros((self.nsys, 3), np.int32)
        if load().agbnp3_batch_sg_modes(self.id, _p(c)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_sg_modes failed")
        return c

    def sg_lists(self):
        """Per system: (descriptor neighbour-list builds, overflow flags) since sg_attach."""
        b, o = np.zeros(self.nsys, np.int32), np.zeros(self.nsys, np.int32)
        if load().agbnp3_batch_sg_lists(self.id, _p(b), _p(o)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_sg_lists failed")
        return b, o

    def set_nblist_reuse(self, skin, every=0):
        if load().agbnp3_batch_set_nblist_reuse(self.id, float(skin), int(every)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_set_nblist_reuse failed")

    def tune(self, x, y, z, reps=3):
        rep = ctypes.create_string_buffer(1 << 16)
        if load().agbnp3_batch_tune(self.id, x, y, z, int(reps), rep, len(rep)) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_tune failed")
        return rep.value.decode()

    def delete(self):
        if self.id is not None:
            load().agbnp3_batch_delete(self.id)
            self.id = None


class Surrogate:
    """A learned Born-radius model (agbnp3_sg_*)."""

    NFEAT = 66
    NPARAM = 41729      # W1 [66][128], b1, W2 [128][128], b2, W3, b3, w4 [128], b4
    LAYOUT = (("W1", (66, 128)), ("b1", (128,)), ("W2", (128, 128)), ("b2", (128,)), ("W3", (128, 128)),
              ("b3", (128,)), ("w4", (128,)), ("b4", (1,)))

    def __init__(self, seed=0):
        if agbnp3_initialize() != AGBNP_OK:
            raise RuntimeError("agbnp3_initialize failed (no GPU?)")
        m = ctypes.c_int(-1)
        if load().agbnp3_sg_new(ctypes.byref(m), int(seed)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_new failed")
        self.id = m.value

    def delete(self):
        if self.id is not None:
            load().agbnp3_sg_delete(self.id)
            self.id = None

    def get_params(self):
        n = load().agbnp3_sg_size()
        out = np.zeros(n, np.float32)
        if load().agbnp3_sg_get_params(self.id, _p(out), n) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_get_params failed")
        return out

    def set_params(self, flat):
        flat = np.ascontiguousarray(flat, np.float32)
        if load().agbnp3_sg_set_params(self.id, _p(flat), flat.size) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_set_params failed")

    def reserve(self, natoms):
        if load().agbnp3_sg_reserve(self.id, int(natoms)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_reserve failed")

    def collect(self, batch, x, y, z):
        """Plain evaluation of `batch` at device coordinates (pointers), appended to the training set."""
        if load().agbnp3_batch_sg_collect(batch.id, self.id, x, y, z) != AGBNP_OK:
            raise RuntimeError("agbnp3_batch_sg_collect failed")

    def dataset(self):
        c = ctypes.c_int(0)
        load().agbnp3_sg_dataset(self.id, ctypes.byref(c), None, None)
        F = np.zeros((c.value, self.NFEAT), np.float32)
        t = np.zeros(c.value, np.float32)
        if c.value and load().agbnp3_sg_dataset(self.id, None, _p(F), _p(t)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_dataset failed")
        return F, t

    def fit(self, margin=0.05, seed=0):
        if load().agbnp3_sg_fit(self.id, float(margin), int(seed)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_fit failed")

    def set_loss(self, w_abs=1.0, w_diff=1.0):
        if load().agbnp3_sg_set_loss(self.id, float(w_abs), float(w_diff)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_set_loss failed")

    def train_rows(self):
        """(dataset row of each training row, pair-difference scale c)."""
        n = np.zeros(1, np.int32)
        if load().agbnp3_sg_train_rows(self.id, _p(n), None, None) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_train_rows failed")
        rows = np.zeros(int(n[0]), np.int32)
        c = np.zeros(1, np.float32)
        if load().agbnp3_sg_train_rows(self.id, _p(n), _p(rows), _p(c)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_train_rows failed")
        return rows, float(c[0])

    def train(self, epochs, batch=4096, lr=2e-3, decay=0.9, seed=0):
        out = np.zeros(epochs, np.float32)
        if load().agbnp3_sg_train(self.id, int(epochs), int(batch), float(lr), float(decay), int(seed),
                                  _p(out)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_train failed")
        return out

    def grads(self, r0, B):
        g = np.zeros(self.NPARAM, np.float32)
        loss = np.zeros(1, np.float32)
        if load().agbnp3_sg_grads(self.id, int(r0), int(B), _p(g), _p(loss)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_grads failed")
        return float(loss[0]), g

    def infer(self, F):
        F = np.ascontiguousarray(F, np.float32)
        n = F.shape[0]
        s = np.zeros(n, np.float32)
        d = np.zeros((n, 64), np.float32)
        if load().agbnp3_sg_infer(self.id, _p(F), n, _p(s), _p(d)) != AGBNP_OK:
            raise RuntimeError("agbnp3_sg_infer failed")
        return s, d
