"""The overlap tree's tiers: a root goes to the next one in both passes or in none."""
import os

import numpy as np
import pytest

from agbnp3_amd import api, synth

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
