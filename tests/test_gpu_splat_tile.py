"""Splats of a merged build whose sums meet per workgroup in LDS (pairs sorted by vertex, 5 to 32
channels) and those of the channel counts beside them, which leave a wavefront at a time: filter and a
repeated apply against the oracle, at the edges of the channel blocks and of the tiles."""
import numpy as np
import pytest
import torch

from conftest import MAX_ABS_TOL, REL_L2_TOL, rel_l2
from permutohedral_lattice_amd import synth

import oracle
import permutohedral_lattice_amd as pla

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def check(got, want):
    got = got.cpu().numpy()
    assert np.isfinite(got).all()
    scale = max(1.0, float(np.abs(want).max()))
    assert np.abs(got - want).max() <= MAX_ABS_TOL * scale and rel_l2(got, want) <= REL_L2_TOL


@pytest.mark.parametrize("vd", [2, 3, 4, 5, 6, 15, 16, 17, 22, 31, 32, 33])
@pytest.mark.parametrize("h,w,features", [(16, 16, 3), (17, 23, 3), (40, 33, 0), (31, 64, 6)])
def test_many_channels_on_merged_tiles(h, w, features, vd):
    rng = np.random.default_rng(1000 * vd + h)
    yx = np.stack(np.meshgrid(np.arange(h), np.arange(w), indexing="ij"), -1).reshape(-1, 2) / 6.0
    img = synth.blob_image(h, w, seed=vd).reshape(-1, 3)
    extra = np.concatenate((img, img[:, ::-1]), axis=1)[:, :features] / 0.2
    pos = np.ascontiguousarray(np.concatenate((yx, extra), axis=1), dtype=np.float32)
    n, pd = pos.shape
    for normalize in (1, 0):
        channels = vd - 1 if normalize else vd
        val = rng.uniform(0.1, 1, (n, channels)).astype(np.float32)
        lat = pla.PermutohedralLattice(pd, vd, n)
        lat.set_point_grid((h, w))
        lat.set_option(pla.PL_OPT_NORMALIZE, normalize)
        lat.set_option(pla.PL_OPT_VERTEX_LISTS, 0)      # (an apply splats, it does not gather)
        out = torch.full((n, channels), float("nan"), device="cuda")
        want = {}
        for reverse in (False, True):
            if normalize:
                want[reverse] = oracle.Lattice(pd, vd, n).filter(val, pos, reverse)
            else:                # sums without the division: the normalised ones times the filtered 1
                ones = np.concatenate((val[:, :-1], np.ones((n, 1), np.float32)), axis=1)
                val = ones
                norm = pla.PermutohedralLattice(pd, 2, n)
                norm.set_option(pla.PL_OPT_NORMALIZE, 0)
                two = torch.empty((n, 2), device="cuda")
                norm.filter(two, dev(np.ones((n, 2), np.float32)), dev(pos), reverse)
                mass = two[:, 1:].cpu().numpy()
                want[reverse] = np.concatenate(
                    (oracle.Lattice(pd, vd, n).filter(val[:, :-1].copy(), pos, reverse) * mass, mass), axis=1)
                norm.close()
        for reverse in (False, True):
            lat.filter(out, dev(val), dev(pos), reverse)
            assert lat.info(pla.PL_INFO_BUILD_MERGED) == 1
            check(out, want[reverse])
        lat.build(dev(pos))
        for reverse in (True, False):
            out.fill_(float("nan"))
            lat.apply(out, dev(val), reverse)
            check(out, want[reverse])
        lat.close()
