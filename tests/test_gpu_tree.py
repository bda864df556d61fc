"""The overlap tree's tiers: a root goes to the next one in both passes or in none, and the last, the depth-first
walk, has the oracle's volumes, areas and derivatives."""
import os

import numpy as np
import pytest

import oracle
from agbnp3_amd import api, synth
from test_gpu_parity import E_REL, G_RMS, GRADS, TERMS, rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms", [300, 613])          # the derivative pass's tiers on one stream and on two
def test_root_that_outgrows_the_derivative_pass_alone_fails_the_call(natoms):
    """Lowered for one instance, the first tier of the derivative pass holds fewer nodes than that of the volumes: its
    larger roots have no tier behind them, and their gradient must not be left out silently."""
    s = synth.generate(20260700 + natoms, natoms)
    ref = api.Instance(s)
    os.environ["AGBNP3_TREE_DERIV_CAP"] = "8"           # read when the instance is built
    try:
        small = api.Instance(s)
    finally:
        del os.environ["AGBNP3_TREE_DERIV_CAP"]
    try:
        out = api.HostOutputs(natoms)
        xyz = [np.ascontiguousarray(a, np.float64) for a in (s.x, s.y, s.z)]
        assert api.agbnp3_ener_into(small.tag, *xyz, out) == api.AGBNP_ERR
        assert api.agbnp3_ener_into(ref.tag, *xyz, out) == api.AGBNP_OK
        c = ref.counts()
        assert c["tree_fallback_volumes"] == c["tree_fallback_derivatives"] == 0
    finally:
        small.delete()
        ref.delete()


@pytest.mark.parametrize("natoms,fixed", [(600, False), (600, True), (2500, False)])
def test_depth_first_walk_matches_oracle(natoms, fixed):
    """Solutes squeezed to half their volume, whose larger trees outgrow the second tier too (15 of 600 atoms' 291).  Their terms are larger,
    and cancel (the molecular volume to less than a tenth): the bounds are the parity tests', of the larger of the
    quantity's size here and at the solute's own coordinates."""
    s = synth.generate(20260310, natoms)
    t = s.with_coords(0.8 * s.x, 0.8 * s.y, 0.8 * s.z)
    own, ref = (oracle.Oracle(u).ener(hb_fixed=fixed, spline_fixed=fixed) for u in (s, t))
    inst = api.Instance(t, api.OPT_HB_FIXED | api.OPT_SPLINE_FIXED if fixed else 0)
    try:
        out, c = inst.ener(), inst.counts()
        assert c["tree_fallback_volumes"] == c["tree_fallback_derivatives"] > 0
    finally:
        inst.delete()
    for k in TERMS:
        assert abs(out[k] - ref[k]) <= E_REL * max(abs(ref[k]), abs(own[k])), (k, out[k], ref[k])
    for k in GRADS:
        assert rms(out[k] - ref[k]) <= G_RMS * max(1.0, rms(ref[k]) / rms(own[k])), (k, rms(out[k] - ref[k]))
    for k in ("sp", "br", "surf_area"):
        assert rms(out[k] - ref[k]) <= 1e-4 * max(1.0, rms(ref[k])), k
