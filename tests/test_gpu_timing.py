"""Per-kernel times and the autotuner where a change of launch shape changes which kernels a call consists of."""
import ctypes

import numpy as np
import pytest

from agbnp3_amd import api, synth

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
