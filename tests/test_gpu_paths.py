"""Calls that a rule on sizes sends another way give the same results.

Bitwise, the two routes of one call against each other: descreening by tiles
(few work items) against the plain kernel; the chain rule by row groups and
the GB pairs by chunks (few work items) against the plain kernels; far columns skipped by boxes against
none skipped.  Against the FP64 oracle: two atoms in one place, which
the GB kernel's off-diagonal tiles meet without the pair mask, water sites
with more than 64 candidate atoms, and overlap terms past the range of the
tree's fast fixed-point conversion.
"""
import dataclasses

import numpy as np
import pytest

import oracle
from agbnp3_amd import api, synth
from test_gpu_parity import G_RMS, check_against_oracle, rms

pytestmark = pytest.mark.gpu

ARRAYS = ("sp", "br", "surf_area", "dgbdr", "dvwdr", "decav", "dehb")


def assert_same(a, b, label):
    for k in api.ENERGY_NAMES:
        assert a[k] == b[k], (label, k, a[k], b[k])
    for k in ARRAYS:
        assert np.array_equal(a[k], b[k]), (label, k)


def merged(a, b, shift):
    """Two solutes as one, the second moved by `shift`."""
    n = a.natoms
    f = {k: np.concatenate([getattr(a, k), getattr(b, k)]) for k in (
        "y", "z", "r", "charge", "igamma", "sgamma", "ialpha", "salpha", "hbtype", "hbcorr", "conn_nne")}
    return dataclasses.replace(
        a, natoms=n + b.natoms, x=np.concatenate([a.x, b.x + shift]),
        ihydrogen=np.concatenate([a.ihydrogen, b.ihydrogen + n]).astype(np.int32),
        conn_neighl1=np.concatenate([a.conn_neighl1, b.conn_neighl1 + n]).astype(np.int32), **f)


@pytest.mark.parametrize("natoms,rows", [(8, 256), (61, 64), (513, 256), (1777, 128), (5000, 256), (9000, 256)])
def test_descreening_by_tiles_equals_the_plain_kernel(natoms, rows):
    # 512 columns per item are what both routes use at these sizes
    s = synth.generate(20260300 + natoms, natoms)
    inst = api.Instance(s)
    try:
        inst.set_tuning(rows=rows)
        tiles = inst.ener()
        inst.set_tuning(rows=rows, desc_chunk=512)
        assert_same(tiles, inst.ener(), natoms)
    finally:
        inst.delete()


@pytest.mark.parametrize("natoms,rows", [(64, 128), (300, 128), (700, 64), (1200, 256), (1500, 128)])
def test_descreening_of_few_tiles_equals_the_plain_kernel(natoms, rows):
    # (64 rows per block there, each wave's columns looked up apart)
    s = synth.generate(20260600 + natoms, natoms)
    inst = api.Instance(s)
    try:
        inst.set_tuning(rows=rows)
        tiles = inst.ener()
        inst.set_tuning(rows=rows, desc_chunk=512)
        assert_same(tiles, inst.ener(), natoms)
    finally:
        inst.delete()


@pytest.mark.parametrize("natoms,mixed,fixed", [(8, False, False), (61, False, True), (300, True, False),
                                                (513, False, False), (1777, True, True), (2000, False, False),
                                                (4100, True, False), (4700, False, True), (6200, False, False)])
def test_chain_rule_by_row_groups_equals_the_plain_kernel(natoms, mixed, fixed):
    """256 columns per item are what both routes use; asked for, they are the plain kernel's.  mixed: hydrogens with
    vdW terms, and some with a heavy atom's radius."""
    s = synth.generate(20260400 + natoms, natoms)
    if mixed:
        r, salpha = s.r.copy(), s.salpha.copy()
        salpha[s.ihydrogen[::2]] = -0.1
        heavy = np.setdiff1d(np.arange(natoms), s.ihydrogen)
        r[s.ihydrogen[::5]] = r[heavy[0]]
        s = dataclasses.replace(s, r=r, salpha=salpha)
    inst = api.Instance(s, api.OPT_HB_FIXED | api.OPT_SPLINE_FIXED if fixed else 0)
    try:
        groups = inst.ener()
        inst.set_tuning(chain_chunk=256)
        assert_same(groups, inst.ener(), natoms)
    finally:
        inst.delete()


@pytest.mark.parametrize("natoms", [8, 61, 64, 130, 257, 513, 700, 2000, 2304])
def test_gb_pairs_by_chunks_equal_the_plain_kernel(natoms):
    """A grid asked for is the plain kernel's; two atoms of different tiles in one place as well."""
    s = synth.generate(20260500 + natoms, natoms)
    h = s.ihydrogen
    x, y, z = s.x.copy(), s.y.copy(), s.z.copy()
    if natoms > 512:
        i, j = int(h[0]), int(h[-1])
        x[j], y[j], z[j] = x[i], y[i], z[i]
    inst = api.Instance(s)
    try:
        chunks = inst.ener(), inst.ener(x, y, z)
        inst.set_tuning(gb_grid=4096)
        assert_same(chunks[0], inst.ener(), natoms)
        assert_same(chunks[1], inst.ener(x, y, z), natoms)
    finally:
        inst.delete()


@pytest.mark.parametrize("shift", [70.0, 92.0, 137.0, 400.0])
def test_far_columns_skipped_by_boxes_change_nothing(shift):
    """An instance created with the two solutes side by side skips nothing;
    one created with them `shift` apart skips what lies past the tables (the
    whole other solute, or its far part)."""
    a, b = synth.generate(20260301, 10007), synth.generate(20260302, 9001)
    apart = merged(a, b, shift)
    near = api.Instance(merged(a, b, 1.0))
    far = api.Instance(apart)
    try:
        ref = near.ener(apart.x, apart.y, apart.z)
        assert_same(far.ener(), ref, shift)
        # and after the coordinates have left those of the creation
        x, y, z = synth.perturb(5, apart.x, apart.y, apart.z, 3.0)
        assert_same(far.ener(x + 30.0, z, y), near.ener(x + 30.0, z, y), shift)
    finally:
        near.delete()
        far.delete()


def test_two_hydrogens_in_one_place_of_different_tiles():
    s = synth.generate(20260303, 900)
    h = s.ihydrogen
    i, j = int(h[3]), int(h[-5])                   # far apart in the internal order: an off-diagonal tile
    x, y, z = s.x.copy(), s.y.copy(), s.z.copy()
    x[j], y[j], z[j] = x[i], y[i], z[i]
    t = s.with_coords(x, y, z)
    inst = api.Instance(t)
    try:
        check_against_oracle(inst.ener(), oracle.Oracle(t).ener(), label="coincident")
    finally:
        inst.delete()


def test_water_sites_with_more_than_64_candidates():
    s = synth.generate(20260310, 600)
    t = s.with_coords(0.75 * s.x, 0.75 * s.y, 0.75 * s.z)   # up to 74 atoms near a site
    inst = api.Instance(t)
    try:
        out, ref = inst.ener(), oracle.Oracle(t).ener()
        assert abs(out["ehb"] - ref["ehb"]) <= 1e-5 * abs(ref["ehb"])
        assert rms(out["dehb"] - ref["dehb"]) <= G_RMS
    finally:
        inst.delete()


@pytest.mark.parametrize("natoms", [61, 700])
def test_overlap_terms_past_the_fast_conversion(natoms):
    """Surface tensions that take some atoms' cavity terms past 2^19, and leave others' below it in the same waves.
    FP32 terms: 1e-5 of the gradients' size, as the energies' bound."""
    s = synth.generate(20260320 + natoms, natoms)
    igamma = s.igamma.copy()
    heavy = np.setdiff1d(np.arange(natoms), s.ihydrogen)
    igamma[heavy[::3]] *= 1e7
    s = dataclasses.replace(s, igamma=igamma)
    inst = api.Instance(s)
    try:
        out, ref = inst.ener(), oracle.Oracle(s).ener()
        assert np.abs(ref["decav"]).max() > 2.0 ** 20
        assert rms(out["decav"] - ref["decav"]) <= 1e-5 * rms(ref["decav"])
        for k in ("dgbdr", "dehb"):
            assert rms(out[k] - ref[k]) <= G_RMS, k
    finally:
        inst.delete()
