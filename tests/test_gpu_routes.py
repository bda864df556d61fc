"""The calls of tests/test_gpu_paths.py take the two routes that are compared there."""
import pytest

from agbnp3_amd import api, synth
from test_gpu_paths import merged

pytestmark = pytest.mark.gpu

TILES, FEW, DESC_FAR, GB_CHUNKS, ROW_GROUPS, GROUPED, CHAIN_FAR = (1 << k for k in range(7))


def routes(s, **tuning):
    inst = api.Instance(s)
    try:
        assert inst.routes() == 0
        if tuning:
            inst.set_tuning(**tuning)
        inst.ener()
        return inst.routes()
    finally:
        inst.delete()


@pytest.mark.parametrize("natoms,rows,few", [(8, 256, True), (61, 64, True), (513, 256, True), (1777, 128, True),
                                             (5000, 256, False), (9000, 256, False), (64, 128, True),
                                             (300, 128, True), (700, 64, True), (1200, 256, True), (1500, 128, True)])
def test_descreening(natoms, rows, few):
    s = synth.generate(20260300 + natoms, natoms)
    tiles, plain = routes(s, rows=rows), routes(s, rows=rows, desc_chunk=512)
    assert tiles & (TILES | FEW) == (TILES | FEW if few else TILES)
    assert plain & (TILES | FEW) == 0


@pytest.mark.parametrize("natoms", [8, 61, 300, 513, 1777, 2000, 4100, 4700, 6200])
def test_chain_rule(natoms):
    s = synth.generate(20260400 + natoms, natoms)
    groups, plain = routes(s), routes(s, chain_chunk=256)
    assert groups & (ROW_GROUPS | GROUPED) == ROW_GROUPS
    assert plain & (ROW_GROUPS | GROUPED) == GROUPED


@pytest.mark.parametrize("natoms", [8, 61, 64, 130, 257, 513, 700, 2000, 2304])
def test_gb_pairs(natoms):
    s = synth.generate(20260500 + natoms, natoms)
    chunks, plain = routes(s), routes(s, gb_grid=4096)
    assert chunks & GB_CHUNKS and not plain & GB_CHUNKS


@pytest.mark.parametrize("shift,far", [(1.0, 0), (70.0, DESC_FAR | CHAIN_FAR), (92.0, DESC_FAR | CHAIN_FAR),
                                       (137.0, DESC_FAR | CHAIN_FAR), (400.0, DESC_FAR | CHAIN_FAR)])
def test_far_columns(shift, far):
    s = merged(synth.generate(20260301, 10007), synth.generate(20260302, 9001), shift)
    taken = routes(s)
    assert taken & (DESC_FAR | CHAIN_FAR) == far


def test_calls_past_the_rules():
    """The larger solute of the water sites' second launch (tests/test_gpu_capacity.py)."""
    mask = TILES | GB_CHUNKS | ROW_GROUPS
    taken = routes(synth.generate(20262900 + 17001, 17001)) & mask
    assert taken == 0
