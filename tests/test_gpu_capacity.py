"""Inputs beyond the synthetic configurations' shapes.

* More radius types than the descreening kernel keeps in LDS (16): the
  reference builds a table per ordered pair of types for any number of
  types (agbnp3_utils.c:808-838, 840-883); single instances and a batch whose
  union of types passes 16 are checked against the FP64 oracle.
* Hydrogens with vdW coefficients, and heavy atoms that share the
  hydrogens' radius (blocks that mix heavy atoms and hydrogens).
* A neighbour-list row that outgrows the row capacity on the device API
  (agbnp3_ener_device, graph replays): the failed call reports AGBNP_ERR,
  the rows are widened and the next call (or replay) succeeds with the
  results of the host API, which widens within its call.
* Water sites with more heavy-atom candidates than the first free-volume
  launch holds go to a second launch with larger buffers (the reference
  grows its buffers, agbnp3.c:4036-4043); lowering the first launch's
  capacity (AGBNP3_WS_FIRST_CAP) routes most sites there, with results
  bitwise those of the first launch.
"""
import os
import ctypes
import dataclasses

import numpy as np
import pytest

import oracle
from agbnp3_amd import api, hip, synth
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu

OUTS = ("sp", "br", "surf_area", "dgbdr", "dvwdr", "decav", "dehb")


def many_types(seed, n, ntypes):
    """The globular solute with heavy-atom radii spread over `ntypes` distinct
    values (each element's radius plus a multiple of 0.01 A)."""
    s = synth.generate(seed, n)
    r = s.r.copy()
    heavy = np.ones(n, bool)
    heavy[s.ihydrogen] = False
    rng = np.random.default_rng(seed)
    base = np.unique(r[heavy])
    per = int(np.ceil(ntypes / base.size))
    step = rng.integers(0, per, n)
    r[heavy] = r[heavy] + 0.01 * step[heavy]
    return dataclasses.replace(s, r=r)


def ntypes_of(s):
    return np.unique(np.float32(np.asarray(s.r) + 0.5)).size


class DeviceIO:
    def __init__(self, n, nsys=1):
        self.n, self.nsys = n, nsys
        self.xyz = [hip.DeviceArray(8 * n) for _ in range(3)]
        self.out = [hip.DeviceArray(8 * n) for _ in range(3)] + [hip.DeviceArray(24 * n) for _ in range(4)]
        self.e = hip.DeviceArray(56 * nsys)

    def set_xyz(self, x, y, z):
        for a, h in zip(self.xyz, (x, y, z)):
            h = np.ascontiguousarray(h, np.float64)
            hip.check(hip.lib().hipMemcpy(a.ptr, h.ctypes.data_as(ctypes.c_void_p), 8 * self.n, hip.H2D),
                      "hipMemcpy")

    def ptrs(self):
        return [a.addr for a in self.xyz] + [a.addr for a in self.out] + [self.e.addr]

    def result(self):
        n = self.n
        d = {k: a.to_numpy(np.float64, (n,)) for k, a in zip(OUTS[:3], self.out[:3])}
        d.update({k: a.to_numpy(np.float64, (n, 3)) for k, a in zip(OUTS[3:], self.out[3:])})
        e = self.e.to_numpy(np.float64, (self.nsys, 7))
        if self.nsys == 1:
            d.update(zip(api.ENERGY_NAMES, e[0]))
        else:
            d["energies"] = e
        return d

    def free(self):
        for a in self.xyz + self.out + [self.e]:
            a.free()


def test_more_radius_types_than_lds_tables_match_oracle():
    s = many_types(20260101, 1500, 24)
    assert ntypes_of(s) > 16
    inst = api.Instance(s)
    try:
        assert inst.tables()[2].size == ntypes_of(s)
        out = inst.ener()
    finally:
        inst.delete()
    check_against_oracle(out, oracle.Oracle(s).ener(), label="24 radius types")


def test_batch_whose_type_union_passes_16_matches_instances_and_oracle():
    a = many_types(20260102, 900, 11)
    b = dataclasses.replace(many_types(20260103, 1100, 11))
    b = dataclasses.replace(b, r=np.where(b.r > 1.3, b.r + 0.005, b.r))    # disjoint heavy radii
    assert ntypes_of(a) <= 16 and ntypes_of(b) <= 16
    union = np.unique(np.concatenate([np.float32(a.r + 0.5), np.float32(b.r + 0.5)])).size
    assert union > 16
    ia, ib = api.Instance(a), api.Instance(b)
    try:
        ea, eb = ia.ener(), ib.ener()
        batch = api.Batch([ia, ib])
        try:
            out = batch.ener(np.concatenate([a.x, b.x]), np.concatenate([a.y, b.y]), np.concatenate([a.z, b.z]))
        finally:
            batch.delete()
    finally:
        ia.delete()
        ib.delete()
    off = a.natoms
    for k, (e, lo, hi) in enumerate(((ea, 0, off), (eb, off, off + b.natoms))):
        for name in OUTS:
            assert np.array_equal(out[name][lo:hi], e[name]), (k, name)
        assert np.array_equal(out["energies"][k], [e[t] for t in api.ENERGY_NAMES]), k
    check_against_oracle(eb, oracle.Oracle(b).ener(), label="batch member b")


def scaled(s, f):
    c = np.array([s.x.mean(), s.y.mean(), s.z.mean()])
    return c[0] + f * (s.x - c[0]), c[1] + f * (s.y - c[1]), c[2] + f * (s.z - c[2])


def longest_row(s, xyz):
    o = oracle.Oracle(dataclasses.replace(s, x=xyz[0], y=xyz[1], z=xyz[2]))
    o.ener()
    nne, _ = o.near_list()
    return int(nne.max())


def test_device_api_recovers_from_a_row_overflow():
    s = synth.generate(20260104, 2500)
    loose, tight = scaled(s, 1.2), scaled(s, 0.93)
    # preconditions: the loose frame sizes rows for 64, the tight one needs more
    assert longest_row(s, loose) + 8 <= 64 < longest_row(s, tight)
    inst = api.Instance(s)
    io = DeviceIO(s.natoms)
    try:
        inst.ener(*loose)                            # host call: rows sized to 64
        assert inst.get_tuning()["cap"] == 64
        io.set_xyz(*tight)
        assert inst.ener_device(*io.ptrs()) == api.AGBNP_OK
        assert inst.sync() == api.AGBNP_ERR          # the row overflow fails this call
        assert inst.get_tuning()["cap"] == 128
        assert inst.ener_device(*io.ptrs()) == api.AGBNP_OK
        assert inst.sync() == api.AGBNP_OK
        dev = io.result()
        host = inst.ener(*tight)
    finally:
        io.free()
        inst.delete()
    for k in OUTS:
        assert np.array_equal(dev[k], host[k]), k
    for k in api.ENERGY_NAMES:
        assert dev[k] == host[k], k


def test_graph_replay_recovers_from_a_row_overflow():
    sa, sb = synth.generate(20260105, 1800), synth.generate(20260106, 1300)
    la, ta = scaled(sa, 1.2), scaled(sa, 0.93)
    lb, tb = scaled(sb, 1.2), scaled(sb, 0.93)
    assert max(longest_row(sa, la), longest_row(sb, lb)) + 8 <= 64 < longest_row(sa, ta) <= 128
    ia, ib = api.Instance(sa), api.Instance(sb)
    b = api.Batch([ia, ib])
    io = DeviceIO(b.n, 2)
    try:
        loose = [np.concatenate([p, q]) for p, q in zip(la, lb)]
        tight = [np.concatenate([p, q]) for p, q in zip(ta, tb)]
        b.ener(*loose)                               # rows sized for the loose frame
        assert b.get_tuning()["cap"] == 64
        io.set_xyz(*loose)
        b.graph_capture(*io.ptrs())
        assert b.graph_launch() == api.AGBNP_OK and b.sync() == api.AGBNP_OK
        io.set_xyz(*tight)
        assert b.graph_launch() == api.AGBNP_OK
        assert b.sync() == api.AGBNP_ERR            # overflow: rows widened, graph captured again
        assert b.get_tuning()["cap"] == 128
        for _ in range(2):
            assert b.graph_launch() == api.AGBNP_OK
            assert b.sync() == api.AGBNP_OK
            dev = io.result()
            host = b.ener(*tight)
            for k in OUTS:
                assert np.array_equal(dev[k], host[k]), k
            assert np.array_equal(dev["energies"], host["energies"])
    finally:
        io.free()
        b.delete()
        ia.delete()
        ib.delete()


def test_hydrogens_with_vdw_coefficients_match_oracle():
    """Hydrogen rows whose ialpha is non-zero (the chain rule's hydrogen x heavy
    items with vdW terms)."""
    s = synth.generate(20260107, 1600)
    ia = s.ialpha.copy()
    rng = np.random.default_rng(7)
    ia[s.ihydrogen] = rng.uniform(-0.2, -0.05, s.ihydrogen.size)
    s = dataclasses.replace(s, ialpha=ia)
    inst = api.Instance(s)
    try:
        out = inst.ener()
    finally:
        inst.delete()
    check_against_oracle(out, oracle.Oracle(s).ener(), label="H vdW")


def test_heavy_atoms_sharing_the_hydrogen_radius_match_oracle():
    """Heavy atoms with the hydrogens' radius: blocks of that radius type mix
    heavy atoms and hydrogens (the chain rule's general items)."""
    s = synth.generate(20260108, 1600)
    r = s.r.copy()
    heavy = np.setdiff1d(np.arange(s.natoms), s.ihydrogen)
    rh = float(r[s.ihydrogen[0]])
    pick = np.random.default_rng(8).choice(heavy, heavy.size // 5, replace=False)
    r[pick] = rh
    s = dataclasses.replace(s, r=r)
    inst = api.Instance(s)
    try:
        out = inst.ener()
    finally:
        inst.delete()
    check_against_oracle(out, oracle.Oracle(s).ener(), label="mixed blocks")


def test_water_sites_past_the_first_launch_capacity():
    s = synth.generate(20262901, 3000)
    ref = api.Instance(s)
    os.environ["AGBNP3_WS_FIRST_CAP"] = "8"          # read when the instance is built
    try:
        small = api.Instance(s)
    finally:
        del os.environ["AGBNP3_WS_FIRST_CAP"]
    try:
        a, b = small.ener(), ref.ener()
        for name in OUTS + api.ENERGY_NAMES:
            assert np.array_equal(np.asarray(a[name]), np.asarray(b[name])), name
        assert b["ehb"] != 0.0 and np.any(b["dehb"] != 0.0)
    finally:
        small.delete()
        ref.delete()


@pytest.mark.parametrize("natoms,chunk", [(3000, 512), (17001, 0)])
def test_water_sites_listed_for_the_second_launch(natoms, chunk):
    """Where the descreening is the plain kernel's (asked for, or in large calls, whose sites run on the second stream),
    the sites past the first launch's capacity go to a launch of their own."""
    s = synth.generate(20262900 + natoms, natoms)
    insts = [api.Instance(s)]
    os.environ["AGBNP3_WS_FIRST_CAP"] = "8"          # read when the instance is built
    try:
        insts.append(api.Instance(s))
    finally:
        del os.environ["AGBNP3_WS_FIRST_CAP"]
    try:
        for i in insts:
            i.set_tuning(desc_chunk=chunk)
        b, a = (i.ener() for i in insts)
        for name in OUTS + api.ENERGY_NAMES:
            assert np.array_equal(np.asarray(a[name]), np.asarray(b[name])), name
        assert b["ehb"] != 0.0 and np.any(b["dehb"] != 0.0)
    finally:
        for i in insts:
            i.delete()


def test_static_scratch_of_few_heavy_atoms(capfd):
    """A large solute with few heavy atoms and no water sites: the boxes of far columns take nothing from the static
    scratch, or solutes at its limit would no longer fit (161,270,272 bytes without them)."""
    n = 45000
    s = synth.generate(77 + n, n)
    heavy = np.setdiff1d(np.arange(n), s.ihydrogen)
    more = np.random.default_rng(1).permutation(heavy)[int(0.6 * len(heavy)):]
    s = dataclasses.replace(s, ihydrogen=np.sort(np.concatenate([s.ihydrogen, more])).astype(np.int32),
                            hbtype=np.zeros_like(s.hbtype))
    inst = api.Instance(s)
    io = DeviceIO(n)
    try:
        io.set_xyz(s.x, s.y, s.z)
        assert api.load().agbnp3_ener_static(inst.tag, *io.ptrs()) == api.AGBNP_ERR
        assert int(capfd.readouterr().err.split(" needs ")[1].split()[0]) <= 161270272
    finally:
        io.free()
        inst.delete()
