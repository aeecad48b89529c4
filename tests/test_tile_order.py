"""Order in which the step kernels hand tiles to the chip's eight XCDs (CPU only): a permutation
for every tile count; two-phase steps, whose relaxation makes the tiles around a shock cost a
multiple of the others, deal any eighth of the mesh to all XCDs, the others keep one contiguous
range of tiles per XCD."""
import ctypes as C

import numpy as np
import pytest

import ecogen_amd as ea
from ecogen_amd.case import IG_AIR, SG_EPOXY, SG_WATER


def _config(model, nph, dim, precision="fp64"):
    n = (64, 64 if dim > 1 else 1, 64 if dim > 2 else 1)
    eos = {1: [IG_AIR], 2: [SG_WATER, IG_AIR], 3: [SG_WATER, SG_EPOXY, IG_AIR]}[nph]
    return ea.make_config(dict(nx=n[0], ny=n[1], nz=n[2], lx=1., ly=1., lz=1., model=model,
                               eos=[dict(e) for e in eos], order=1, relax_p=True, precision=precision))


def _order(cfg, ntiles):
    L = ea.library()
    return np.array([L.ecg_tile_of_block(C.byref(cfg), ntiles, b) for b in range(ntiles)])


COUNTS = [1, 2, 7, 8, 9, 63, 127, 128, 129, 255, 256, 257, 900, 1892, 3312, 4375, 6144, 6145, 6966]


@pytest.mark.parametrize("ntiles", COUNTS)
@pytest.mark.parametrize("dim", [1, 2, 3])
@pytest.mark.parametrize("model,nph", [("euler", 1), ("pueq", 2), ("ueq", 2), ("ueq", 3)])
def test_order_is_a_permutation(model, nph, dim, ntiles):
    assert np.array_equal(np.sort(_order(_config(model, nph, dim), ntiles)), np.arange(ntiles))


@pytest.mark.parametrize("dim,ntiles", [(2, 1892), (2, 6966), (2, 16384), (3, 3312), (3, 4225), (3, 6144)])
@pytest.mark.parametrize("model", ["pueq", "ueq"])
def test_two_phase_steps_share_any_part_of_the_mesh(model, dim, ntiles):
    """The tiles of any run of a quarter of the mesh lie on all eight XCDs, none with twice its share."""
    tile = _order(_config(model, 2, dim), ntiles)
    xcd = np.empty(ntiles, dtype=int)
    xcd[tile] = np.arange(ntiles) % 8
    part = ntiles // 4
    for lo in range(0, ntiles - part + 1, max(part // 7, 1)):
        share = np.bincount(xcd[lo:lo + part], minlength=8)
        assert share.min() > 0 and share.max() <= 2 * part / 8 + 64, (lo, share)


@pytest.mark.parametrize("cfg", [("euler", 1, 2), ("euler", 1, 3), ("pueq", 3, 2), ("ueq", 3, 3), ("pueq", 2, 1),
                                 ("ueq", 2, 3, "fp32_learned"), ("pueq", 2, 2, "fp32", 16383), ("ueq", 2, 3, "fp64", 6145)])
def test_other_steps_keep_one_range_per_xcd(cfg):
    *cfg, count = cfg if len(cfg) == 5 else (*cfg, 0)
    for ntiles in (count,) if count else (900, 1892, 4375):
        tile = _order(_config(*cfg), ntiles)
        for x in range(8):
            mine = tile[x::8]
            assert np.array_equal(mine, np.arange(mine[0], mine[0] + len(mine)))


def test_blocks_outside_the_launch_are_refused():
    L, cfg = ea.library(), _config("ueq", 2, 2)
    for ntiles, block in ((0, 0), (8, 8), (8, -1)):
        assert L.ecg_tile_of_block(C.byref(cfg), ntiles, block) < 0
