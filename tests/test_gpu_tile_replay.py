"""What a merging build leaves of its points (places in their workgroup's table of vertices) and the passes
that read it, against the oracle: at the edges of the channel blocks, with tiles whose vertices fit the rows
in LDS and tiles whose do not, in floats and doubles, and where only one of two joint lattices has such
tiles."""
import numpy as np
import pytest
import torch

from conftest import MAX_ABS_TOL, REL_L2_TOL, rel_l2
from permutohedral_lattice_amd import synth
from permutohedral_lattice_amd.crf import MeanField

import oracle
import permutohedral_lattice_amd as pla

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def positions(h, w, features, noise, seed):
    """A grid's coordinates and smooth features with `noise` of a width of noise on them."""
    rng = np.random.default_rng(seed)
    yx = np.stack(np.meshgrid(np.arange(h), np.arange(w), indexing="ij"), -1).reshape(-1, 2) / 6.0
    img = synth.blob_image(h, w, seed=seed).reshape(-1, 3)
    extra = np.concatenate((img, img[:, ::-1]), axis=1)[:, :features] / 0.2
    extra = extra + noise * rng.uniform(-1, 1, extra.shape)
    return np.ascontiguousarray(np.concatenate((yx, extra), axis=1), dtype=np.float32)


def vertices_of_tiles(pos, h, w):
    """Distinct vertices of the workgroups' 16x16 points."""
    pd = pos.shape[1]
    keys = oracle.dump_simplex(pos)["keys"].reshape(h, w, pd + 1, pd)
    return [len(np.unique(keys[y:y + 16, x:x + 16].reshape(-1, pd), axis=0))
            for y in range(0, h, 16) for x in range(0, w, 16)]


def check(got, want):
    got = got.cpu().numpy()
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() <= MAX_ABS_TOL and rel_l2(got, want) <= REL_L2_TOL


@pytest.mark.parametrize("vd", [2, 3, 4, 5, 8, 9, 22, 32, 33, 34, 64, 65, 66, 67])
@pytest.mark.parametrize("h,w,features,noise", [(33, 47, 3, 0.0), (32, 48, 3, 1.1), (20, 30, 5, 0.5), (17, 40, 6, 0.2)])
def test_filter_and_applies(h, w, features, noise, vd):
    pos = positions(h, w, features, noise, 7 * h + features)
    n, pd = pos.shape
    val = np.random.default_rng(vd).uniform(0.1, 1, (n, vd - 1)).astype(np.float32)
    want = {reverse: oracle.Lattice(pd, vd, n).filter(val, pos, reverse) for reverse in (False, True)}
    lat = pla.PermutohedralLattice(pd, vd, n)
    lat.set_point_grid((h, w))
    out = torch.empty((n, vd - 1), device="cuda")
    for reverse in (False, True):
        lat.filter(out.fill_(float("nan")), dev(val), dev(pos), reverse)
        check(out, want[reverse])
    assert lat.info(pla.PL_INFO_BUILD_MERGED) == 1
    for lists in (0, 1):
        lat.set_option(pla.PL_OPT_VERTEX_LISTS, lists)
        lat.build(dev(pos))
        for reverse in (True, False):
            lat.apply(out.fill_(float("nan")), dev(val), reverse)
            check(out, want[reverse])
    vertex, weight = lat.debug_replay()
    keys = lat.debug_keys().cpu().numpy()[vertex.cpu().numpy()]
    simplex = oracle.dump_simplex(pos)
    assert (keys.transpose(1, 0, 2) == simplex["keys"]).all()
    assert (weight.cpu().numpy().T == simplex["barycentric"]).all()
    lat.close()


def test_the_noise_crowds_the_tiles():
    """The inputs above have tiles below and above the rows that fit into the least LDS a slice takes (335 of 21
    channels, 262 of 32: test_crowded_tiles_of_large_images) and none that the merging build cannot take (512)."""
    smooth = vertices_of_tiles(positions(33, 47, 3, 0.0, 7 * 33 + 3), 33, 47)
    noisy = vertices_of_tiles(positions(32, 48, 3, 1.1, 7 * 32 + 3), 32, 48)
    assert max(smooth) < 198 and max(noisy) > 262 and max(noisy) <= 512


@pytest.mark.parametrize("vd", [22, 33, 40])
def test_crowded_tiles_of_large_images(vd):
    """Where the launch fills the GPU a slice has the least rows in LDS: 335 of 21 channels, 262 of 32.  Tiles of
    more gather from memory; against the same lattice built without merging."""
    h, w = 512, 530
    rng = np.random.default_rng(1)
    y, x = np.meshgrid(np.arange(h), np.arange(w), indexing="ij")
    smooth = np.stack([np.sin(x / 50.0), np.cos(y / 40.0), np.sin((x + y) / 70.0)], -1) / 0.42
    # (a few tiles of the most: at 350 of 512 places one in some hundreds looks for its keys too long to be merged)
    crowd = np.where((x < 48) & (y < 48), 1.0, np.where(x < w // 2, 0.85, 0.1))
    noise = crowd[..., None] * rng.uniform(-1, 1, (h, w, 3))
    pos = np.concatenate([np.stack([y, x], -1) / 6.0, smooth + noise], -1).reshape(-1, 5).astype(np.float32)
    used = vertices_of_tiles(pos, h, w)
    assert min(used) < 262 and 335 < max(used) <= 512
    pos, val = dev(pos), dev(rng.uniform(0.1, 1.1, (h * w, vd - 1)).astype(np.float32))
    outs = {}
    for merge in (0, 1):
        lat = pla.PermutohedralLattice(5, vd, h * w)
        lat.set_point_grid((h, w))
        lat.set_option(pla.PL_OPT_MERGE_TILES, merge)
        lat.build(pos)
        assert lat.info(pla.PL_INFO_BUILD_MERGED) == merge
        outs[merge] = [lat.apply(torch.full_like(val, float("nan")), val, reverse) for reverse in (False, True)]
        lat.close()
    for got, want in zip(outs[1], outs[0]):
        # (the same terms in another order)
        assert torch.isfinite(got).all() and float((got - want).abs().max()) <= 2e-5


@pytest.mark.parametrize("vd", [2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("h,w,features,noise", [(33, 47, 3, 0.0), (32, 48, 3, 1.1), (17, 40, 6, 0.2)])
def test_doubles(h, w, features, noise, vd):
    pos = positions(h, w, features, noise, 7 * h + features).astype(np.float64)
    n, pd = pos.shape
    val = np.random.default_rng(vd).uniform(0.1, 1, (n, vd - 1))
    lat = pla.PermutohedralLattice(pd, vd, n, dtype=torch.float64)
    lat.set_point_grid((h, w))
    out = torch.empty((n, vd - 1), device="cuda", dtype=torch.float64)
    for reverse in (False, True):
        want = oracle.Lattice(pd, vd, n, dtype=np.float64).filter(val, pos, reverse)
        lat.filter(out.fill_(float("nan")), dev(val), dev(pos), reverse)
        assert np.abs(out.cpu().numpy() - want).max() <= 1e-12
        lat.build(dev(pos))
        lat.apply(out.fill_(float("nan")), dev(val), reverse)
        assert np.abs(out.cpu().numpy() - want).max() <= 1e-12
    lat.close()


# (0.02: every tile's vertices fit into LDS; 25: of the two lattices 160 to 400, of one at most 350; 300: the
# bilateral lattice is built without merging, the spatial one is not)
@pytest.mark.parametrize("noise,merged", [(0.02, 1), (25.0, 1), (300.0, 0)])
@pytest.mark.parametrize("classes", [4, 5, 21, 31])
def test_joint_messages(noise, merged, classes):
    batch, h, w = 2, 40, 56
    rng = np.random.default_rng(classes)
    guide = np.stack([synth.blob_image(h, w, seed=b) * 255.0 for b in range(batch)])
    guide = (guide + noise * rng.uniform(-1, 1, guide.shape)).astype(np.float32)
    logits = synth.normal_image((batch, h, w, classes), 10)
    upstream = synth.normal_image((batch, h, w, classes), 11)
    mf = MeanField(dev(guide), classes, theta_alpha=80.0, theta_beta=13.0)
    for lat in mf.bilateral:
        assert lat.info(pla.PL_INFO_BUILD_MERGED) == merged
    for lat in mf.spatial:
        assert lat.info(pla.PL_INFO_BUILD_MERGED) == 1
    q = mf.infer(dev(logits), iterations=2).cpu().numpy()
    rev = mf.reverse(dev(upstream)).cpu().numpy()
    want_q, want_rev = oracle.mean_field(logits, guide, 2, upstream=upstream)
    assert np.isfinite(q).all() and np.abs(q.sum(axis=-1) - 1.0).max() <= 1e-5
    assert np.abs(q - want_q).max() <= MAX_ABS_TOL and rel_l2(q, want_q) <= REL_L2_TOL
    assert np.abs(rev - want_rev).max() <= MAX_ABS_TOL * max(1.0, float(np.abs(want_rev).max()))
    assert rel_l2(rev, want_rev) <= REL_L2_TOL
    mf.close()


# Up to four channels a workgroup's rows of sums are listed from 2^19 points on (from four features on).  flat: most of a tile's corners
# name a few vertices (runs over several wavefronts); wild: values that sums of products by 0 and 1 cannot take.
@pytest.mark.parametrize("vd", [2, 3, 4])
@pytest.mark.parametrize("kind", ["image", "flat", "coordinates", "list", "wild"])
def test_rows_of_few_channels(kind, vd):
    gen = torch.Generator(device="cuda").manual_seed(vd)
    h, w = 725, 724
    n = h * w
    assert n >= 1 << 19
    y, x = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"), indexing="ij")
    guide = torch.stack([torch.sin(x / 50.0), torch.cos(y / 40.0), torch.sin((x + y) / 70.0)], -1)
    guide = guide + 0.1 * torch.rand(guide.shape, generator=gen, device="cuda")
    if kind == "flat":
        pos = pla.compute_positions((0.01 * guide).contiguous(), (h, w), 40.0, 1.0)
    elif kind == "coordinates":
        pos = pla.compute_positions(None, (h, w), 8.0)
    else:
        pos = pla.compute_positions(guide.contiguous(), (h, w), 8.0, 0.5)
    if kind == "list":
        pos = pos[:, :4][torch.randperm(n, generator=gen, device="cuda")].contiguous()
    for normalize in (1, 0):
        channels = vd - 1 if normalize else vd
        val = torch.rand((n, channels), generator=gen, device="cuda") + 0.1
        if kind == "wild":
            val[::1000] *= 1e31
        lat = pla.PermutohedralLattice(pos.shape[1], vd, n)
        if kind != "list":
            lat.set_point_grid((h, w))
        lat.set_option(pla.PL_OPT_NORMALIZE, normalize)
        filtered, applied = torch.empty_like(val), torch.empty_like(val)
        want = {reverse: lat.filter(filtered, val, pos, reverse).clone() for reverse in (False, True)}
        lat.build(pos)
        assert lat.info(pla.PL_INFO_BUILD_MERGED) == 1
        for reverse in (False, True):
            lat.apply(applied.fill_(float("nan")), val, reverse)
            # (the same terms in another order: sums of some 10^4 positive floats, 2^-24 an addition on
            # either side and far less on average)
            assert torch.isfinite(applied).all()
            assert float(((applied - want[reverse]).abs() / want[reverse].abs()).max()) <= 1e-4
            assert float((applied - want[reverse]).double().norm() / want[reverse].double().norm()) <= 2e-6
            first = applied.clone()
            lat.apply(applied, val, reverse)
            assert (applied == first).all()     # (one order on every call)
        lat.close()
