"""The tile kernel against the one-thread-per-pair list kernel over all pairs,
bit for bit, at the edges of its forms: partial blocks, boxes whose row blocks
need one or two images, few, many and no Lennard-Jones atoms (row places),
atoms in other images, lambda dependence, one to eight waves a tile, and row
accumulators that are carried over the tiles of a wave."""

import numpy as np
import pytest
from scipy.spatial import cKDTree

from timemachine_amd.lib import custom_ops

pytestmark = pytest.mark.gpu


def _system(rng, n, side, lj):
    g = int(np.ceil(n ** (1 / 3)))
    sites = np.stack(np.meshgrid(*[np.arange(g)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (sites + rng.uniform(0.2, 0.8, (n, 3))) * (side / g)
    p = np.stack([rng.normal(0, 6, n), rng.uniform(0.1, 0.15, n), rng.uniform(0.3, 0.9, n)], 1)
    p[rng.permutation(n)[int(round(lj * n)):], 2] = 0.0
    return x, p


# tiles up to which a tile is shared by so many waves (tile_split)
FORMS = {8: 576, 4: 1152, 2: 9216, 1: 1 << 30}


@pytest.mark.parametrize("n,side,lj,beta,moving,waves", [
    (63, 2.7, 0.33, 2.0, 0.0, 8), (64, 2.7, 1.0, 2.0, 0.1, 8), (65, 2.62, 0.0, 2.0, 0.0, 8),
    (129, 3.3, 0.5, 2.0, 0.0, 8), (1000, 2.9, 0.33, 2.0, 0.02, 8), (2003, 3.7, 0.33, 2.0, 0.0, 8),
    (2500, 4.1, 0.8, 2.0, 0.01, 8), (3001, 6.3, 0.33, 2.0, 0.0, 8), (900, 3.0, 0.33, 2.7, 0.0, 8),
    (1500, 4.0, 0.33, 3.1, 0.05, 8), (3300, 3.4, 0.33, 2.0, 0.02, 4), (6000, 4.0, 0.33, 2.0, 0.02, 2),
    (26500, 6.45, 0.33, 2.0, 0.0, 2), (29000, 6.6, 0.33, 2.0, 0.01, 1)])
def test_tiles_equal_pair_list(gpu, n, side, lj, beta, moving, waves):
    rng = np.random.default_rng(n)
    x, params = _system(rng, n, side, lj)
    x = x + side * rng.integers(-2, 3, x.shape)  # atoms in any image
    box = np.eye(3) * side
    plane = np.zeros(n, np.int32)
    offset = (rng.random(n) < moving).astype(np.int32)
    tree = cKDTree(np.mod(x, side) % side, boxsize=side)
    pairs = tree.query_pairs(1.21, output_type="ndarray").astype(np.int32)
    tiles = custom_ops.NonbondedAllPairs_f32(None, plane, offset, beta, 1.2)
    plist = custom_ops.NonbondedPairList_f32(None, pairs, np.ones((len(pairs), 2)), plane, offset, beta, 1.2)
    for lam in (0.0, 0.35):  # twice on one object: its partial sums are cleared in between
        a = tiles.execute_fixed_raw(x, params, box, lam)
        b = plist.execute_fixed_raw(x, params, box, lam)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
        for k in (2, 3):
            assert np.sum(a[k], dtype=np.uint64) == np.sum(b[k], dtype=np.uint64)
        # forces alone: the kernel without parameter derivatives
        only = tiles.execute_selective(x, params, box, lam, True, False, False, False)[0]
        np.testing.assert_array_equal(only, a[0].view(np.int64).reshape(n, 3) / 2.0**36)
    assert next(w for w, top in FORMS.items() if tiles.num_tiles() <= top) == waves


@pytest.mark.parametrize("interpolated", [False, True])
def test_row_runs_of_several_tiles(gpu, interpolated):
    """Whole tiles on few waves: each walks 10 to 200 tiles, its row accumulators stay
    over the tiles of a row block, which may begin and end within its range."""
    rng = np.random.default_rng(5)
    n, side = 29000, 6.6
    x, params = _system(rng, n, side, 0.33)
    box = np.eye(3) * side
    plane, offset = np.zeros(n, np.int32), (rng.random(n) < 0.01).astype(np.int32)
    pairs = cKDTree(np.mod(x, side) % side, boxsize=side).query_pairs(1.21, output_type="ndarray").astype(np.int32)
    if interpolated:
        end = params * np.array([0.8, 1.0, 1.0])
        end[::3, 2] = 0.0
        params = np.concatenate([params, end])
    suffix = "_interpolated" if interpolated else ""
    tiles = getattr(custom_ops, "NonbondedAllPairs_f32" + suffix)(None, plane, offset, 2.0, 1.2)
    plist = getattr(custom_ops, "NonbondedPairList_f32" + suffix)(None, pairs, np.ones((len(pairs), 2)), plane, offset,
                                                                  2.0, 1.2)
    want = plist.execute_fixed_raw(x, params, box, 0.35)
    want_dl_dp = None if interpolated else plist.execute_dl_dp(x, params, box, 0.35)
    for grid in (1000, 333, 50):
        tiles.set_tile_grid(grid)
        got = tiles.execute_fixed_raw(x, params, box, 0.35)
        assert tiles.num_tiles() > 9216
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_array_equal(got[1], want[1])
        for k in (2, 3):
            assert np.sum(got[k], dtype=np.uint64) == np.sum(want[k], dtype=np.uint64)
        forces, _, dl, u = tiles.execute_selective(x, params, box, 0.35, True, False, True, True)
        np.testing.assert_array_equal(forces, want[0].view(np.int64).reshape(n, 3) / 2.0**36)
        assert dl == np.sum(want[2], dtype=np.uint64).view(np.int64) / 2.0**36
        assert u == np.sum(want[3], dtype=np.uint64).view(np.int64) / 2.0**36
        if not interpolated:
            np.testing.assert_array_equal(tiles.execute_dl_dp(x, params, box, 0.35), want_dl_dp)
