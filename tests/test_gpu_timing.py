"""Per-kernel times and the autotuner where a change of launch shape changes which kernels a call consists of."""
import ctypes
import re

import numpy as np
import pytest

from agbnp3_amd import api, hip, synth

pytestmark = pytest.mark.gpu


def kernel_times(inst):
    """[(name, ms)] as the library lists them (api's dict would hide a name that is there twice)."""
    ms, names = np.zeros(64, np.float32), ctypes.create_string_buffer(4096)
    k = api.load().agbnp3_kernel_times(inst.tag, ms.ctypes.data_as(ctypes.c_void_p), 64, names, 4096)
    assert k > 0
    return list(zip(names.value.decode().split(";"), ms[:k].tolist()))


def test_kernel_times_after_a_change_of_route():
    """The plain descreening asked for, the water sites are launched apart; back on tiles, the list of kernels holds
    no entry of those calls."""
    inst = api.Instance(synth.generate(20260801, 613), api.OPT_TIMING)
    try:
        for chunk in (0, 512, 0):
            inst.set_tuning(desc_chunk=chunk)
            for _ in range(2):
                inst.ener()
            times = kernel_times(inst)
            names = [n for n, _ in times]
            assert len(set(names)) == len(names) and names[-1] == "final", (chunk, names)
            assert all(t >= 0.0 for _, t in times), (chunk, times)
    finally:
        inst.delete()


def tuned(natoms):
    """(report, tuning) of an autotuner's run on one solute."""
    s = synth.generate(20260800 + natoms, natoms)
    inst = api.Instance(s)
    xyz = [hip.DeviceArray(8 * s.natoms) for _ in range(3)]
    try:
        for a, h in zip(xyz, (s.x, s.y, s.z)):
            h = np.ascontiguousarray(h, np.float64)
            hip.check(hip.lib().hipMemcpy(a.ptr, h.ctypes.data_as(ctypes.c_void_p), h.nbytes, hip.H2D), "hipMemcpy")
        return inst.tune(*(a.addr for a in xyz), reps=5), inst.get_tuning()
    finally:
        for a in xyz:
            a.free()
        inst.delete()
        api.load().agbnp3_tune_table_clear()


def test_autotuner_compares_equal_work():
    """The smallest calls, where the water sites bound the launch that they share with the tiled descreening: what a
    candidate leaves to another kernel counts with it."""
    report, t = tuned(61)
    counted = {int(p): names for p, names in re.findall(r"param (\d+) = .*\((.*)\)", report)}
    assert counted[0] == counted[1] == "descreen ws_free" and counted[4] == "gbpair q2ab", report
    assert t["desc_chunk"] == t["gb_grid"] == 0, report          # 17 us against 28, 19 against 29


def test_autotuner_chooses_among_different_launches_only():
    """3,000 atoms, tiles, chain rule by row groups, 78 GB items: grids of those kernels that are not launched, or
    that no item would go without, are neither tried nor recorded."""
    report, t = tuned(3000)
    tried = [(int(p), int(c)) for p, c in re.findall(r"param (\d+) = (\d+)", report)]
    assert [c for p, c in tried if p == 4] == [0] and not [c for p, c in tried if p == 3], report
    assert t["gb_grid"] == t["desc_grid"] == 0, report
    assert t["chain_chunk"] != 0 or t["chain_grid"] == 0, report
