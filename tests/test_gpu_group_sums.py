"""The sums of the builds, with tiles merged and without: groups of one lane, of a whole wavefront and of lanes that are not next
to each other, tiles that are not full, and values that are not finite or near the largest, which take
the sums lane by lane; filter against the oracle."""
import numpy as np
import pytest
import torch

from conftest import MAX_ABS_TOL, REL_L2_TOL, rel_l2

import oracle
import permutohedral_lattice_amd as pla

pytestmark = pytest.mark.gpu


def positions(kind, h, w, rng):
    y, x = np.meshgrid(np.arange(h), np.arange(w), indexing="ij")
    if kind == "one":              # all points in one simplex
        return np.stack((y, x), -1).reshape(-1, 2) * 1e-4
    if kind == "own":              # next to no two points share a vertex (pd 1: few enough for a tile)
        return (100.0 * (y * w + x)).reshape(-1, 1)
    if kind == "mixed":            # points that share a vertex are spread over the tile
        return np.stack((y / 5.0, x / 5.0, rng.integers(0, 3, (h, w)) * 0.9), -1).reshape(-1, 3)
    return np.concatenate((np.stack((y, x), -1).reshape(-1, 2) / 7.0, rng.uniform(0, 1.5, (h * w, 3))), 1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("vd", [2, 3, 4])
@pytest.mark.parametrize("kind,h,w", [("one", 16, 16), ("own", 12, 16), ("mixed", 17, 23), ("noise", 40, 33),
                                      ("mixed", 8, 9), ("noise", 9, 64)])
def test_sums_of_groups(kind, h, w, vd, dtype):
    rng = np.random.default_rng(100 * vd + h * w)
    pos = np.ascontiguousarray(positions(kind, h, w, rng), dtype=dtype)
    n, pd = pos.shape
    lat = pla.PermutohedralLattice(pd, vd, n, dtype=torch.float32 if dtype == np.float32 else torch.float64)
    lat.set_point_grid((h, w))
    out = torch.empty((n, vd - 1), dtype=lat.dtype, device="cuda")
    large = float(np.finfo(dtype).max) / 4              # (its sums stay in range)
    for extreme in (None, large, np.inf, -np.inf, np.nan):
        val = rng.uniform(0.1, 1, (n, vd - 1)).astype(dtype)
        if extreme is not None:
            val[n // 2, -1] = extreme
        for reverse in (False, True):
            lat.filter(out, torch.from_numpy(val).cuda(), torch.from_numpy(pos).cuda(), reverse)
            assert lat.info(pla.PL_INFO_BUILD_MERGED) == 1
            with np.errstate(all="ignore"):
                want = oracle.Lattice(pd, vd, n, dtype=dtype).filter(val, pos, reverse)
            got = out.cpu().numpy()
            fine = np.isfinite(want)
            assert (np.isfinite(got) == fine).all()
            assert (np.isnan(got) == np.isnan(want)).all()
            scale = large if extreme == large else 1.0
            got, want = got[fine] / scale, want[fine] / scale
            if fine.any():
                assert np.abs(got - want).max() <= MAX_ABS_TOL and rel_l2(got, want) <= REL_L2_TOL
    lat.close()


@pytest.mark.parametrize("vd", [2, 3, 4])
@pytest.mark.parametrize("kind,h,w", [("one", 16, 16), ("own", 16, 16), ("mixed", 17, 23), ("noise", 40, 33),
                                      ("own", 1, 1), ("noise", 9, 7)])
def test_sums_of_groups_without_merging(kind, h, w, vd):
    rng = np.random.default_rng(100 * vd + h * w)
    pos = np.ascontiguousarray(positions(kind, h, w, rng), dtype=np.float32)
    n, pd = pos.shape
    out = torch.empty((n, vd - 1), dtype=torch.float32, device="cuda")
    large = float(np.finfo(np.float32).max) / 4
    for extreme in (None, large, np.inf, np.nan):
        val = rng.uniform(0.1, 1, (n, vd - 1)).astype(np.float32)
        if extreme is not None:
            val[n // 2, -1] = extreme
        pla.filter_static(out, torch.from_numpy(val).cuda(), torch.from_numpy(pos).cuda(), pd, vd)
        with np.errstate(all="ignore"):
            want = oracle.Lattice(pd, vd, n, dtype=np.float32).filter(val, pos, False)
        got = out.cpu().numpy()
        fine = np.isfinite(want)
        assert (np.isfinite(got) == fine).all()
        assert (np.isnan(got) == np.isnan(want)).all()
        scale = large if extreme == large else 1.0
        got, want = got[fine] / scale, want[fine] / scale
        if fine.any():
            assert np.abs(got - want).max() <= MAX_ABS_TOL and rel_l2(got, want) <= REL_L2_TOL
