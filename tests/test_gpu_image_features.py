"""Features made from the grid in the build against the same features as a positions array: keys and
barycentric weights of every point, bit for bit, over widths that divide by a multiplication and widths
that do not, and grids of every number of extents."""
import numpy as np
import pytest
import torch

import permutohedral_lattice_amd as pla

pytestmark = pytest.mark.gpu


def rows(lat, build):
    build()
    vertex, weight = (x.cpu().numpy() for x in lat.debug_replay())
    keys = lat.debug_keys().cpu().numpy()
    return keys[vertex], weight


@pytest.mark.parametrize("dims", [(5,), (17, 23), (1, 40), (64, 1, 48), (3, 9, 21), (1, 30, 33), (2, 3, 9, 17), (33, 70)])
@pytest.mark.parametrize("channels", [0, 1, 3])
@pytest.mark.parametrize("widths", [(8.0, 0.125), (3.3, 0.07), (0.37, 13.0), (2.0 ** 41, 2.0 ** -41), (1e30, -1.7)])
def test_features_of_the_grid(dims, channels, widths):
    n, pd = int(np.prod(dims)), len(dims) + channels
    rng = np.random.default_rng(n + channels)
    image = rng.uniform(0, 1, (n, channels)).astype(np.float32) if channels else None
    if channels and widths[1] < 1e-6:
        image *= np.float32(widths[1])
    image = torch.from_numpy(image).cuda() if channels else None
    lat = pla.PermutohedralLattice(pd, 2, n)
    got = rows(lat, lambda: lat.build_image(image, dims, *widths))
    positions = pla.compute_positions(image, dims, *widths)
    want = rows(lat, lambda: lat.build(positions))
    assert (got[0] == want[0]).all() and (got[1] == want[1]).all()
    lat.close()


@pytest.mark.parametrize("dims", [(5,), (17, 23), (1, 40), (64, 1, 48), (3, 9, 21), (1, 30, 33), (2, 3, 9, 17), (33, 70), (40, 2)])
@pytest.mark.parametrize("channels", [0, 1, 3])
@pytest.mark.parametrize("widths", [(8.0, 0.125), (3.3, 0.07), (0.37, 13.0), (2.0 ** 41, 0.2)])
def test_features_of_doubles_from_the_grid(dims, channels, widths):
    """The op makes them in the build where the points are a grid of two or three extents: the same filter as
    under the positions array, up to the order of additions (the sums of a vertex are at most some
    hundred terms: 1e-13 of values in [0, 1])."""
    n, pd = int(np.prod(dims)), len(dims) + channels
    rng = np.random.default_rng(n + channels)
    value = torch.from_numpy(rng.uniform(0, 1, (2, n, 2))).cuda()
    image = torch.from_numpy(rng.uniform(0, 1, (2, n, channels))).cuda() if channels else None
    got = pla.lattice_filter(value.view((2,) + dims + (2,)), image.view((2,) + dims + (channels,)) if channels else None,
                             bilateral=channels > 0, theta_alpha=widths[0], theta_beta=widths[1], theta_gamma=widths[0])
    want = torch.empty_like(value)
    for b in range(2):
        # (the op's attributes are floats for every value type)
        positions = pla.compute_positions(image[b] if channels else None, dims, float(np.float32(widths[0])),
                                          float(np.float32(widths[1])), dtype=torch.float64)
        lat = pla.PermutohedralLattice(pd, 3, n, dtype=torch.float64)
        lat.set_point_grid(dims)
        lat.filter(want[b], value[b], positions)
        lat.close()
    assert float((got.view(want.shape) - want).abs().max()) <= 1e-13


@pytest.mark.parametrize("size,quotient", [(2.0 ** -126, 0.0), (2.0 ** -101, 0.0), (2.0 ** -99, 0.0), (1.0, 2.0 ** 14)])
def test_channels_at_the_edges_of_the_rule(size, quotient):
    """Channels below 2^-100 may be an ulp off, which reaches no key and no weight but those as small as they."""
    dims, n = (17, 23), 17 * 23
    rng = np.random.default_rng(5)
    image = (rng.uniform(-1, 1, (n, 1)) * size).astype(np.float32)
    width = size / quotient if quotient else 0.13
    lat = pla.PermutohedralLattice(3, 2, n)
    image = torch.from_numpy(image).cuda()
    got = rows(lat, lambda: lat.build_image(image, dims, 3.3, width))
    want = rows(lat, lambda: lat.build(pla.compute_positions(image, dims, 3.3, width)))
    assert (got[0] == want[0]).all() and float(np.abs(got[1] - want[1]).max()) <= size * 2.0 ** -21 * (size < 1)
    lat.close()


@pytest.mark.parametrize("quotient", [2.0 ** 20, 2.0 ** 79, 2.0 ** 81, 2.0 ** 126])
def test_channels_beyond_every_key_are_refused_either_way(quotient):
    dims, n = (17, 23), 17 * 23
    image = torch.full((n, 1), 0.25, device="cuda")
    image[5] = 1.0
    lat = pla.PermutohedralLattice(3, 2, n)
    for build in (lambda: lat.build_image(image, dims, 3.3, 1.0 / quotient),
                  lambda: lat.build(pla.compute_positions(image, dims, 3.3, 1.0 / quotient))):
        with pytest.raises(pla.PermutohedralError) as e:
            build()
        assert e.value.status == pla.PL_EOVERFLOW
    lat.close()


@pytest.mark.parametrize("dims,channels", [((211, 130), 0), ((130, 211), 2), ((33, 40, 21), 0), ((40, 21, 33), 1)])
@pytest.mark.parametrize("widths", [(0.03, 0.07), (0.0371, 0.11), (0.05, 0.3)])
def test_features_of_doubles_from_the_grid_bit_for_bit(dims, channels, widths):
    """Under widths so small that no two points share a vertex every sum has one term, and the results are
    the same in every bit for as long as the floats are that the embedding makes of the scaled features: an
    ulp of those shows.  (The last bits of the divisions do not: tests/test_rounding.py.)"""
    n, pd = int(np.prod(dims)), len(dims) + channels
    rng = np.random.default_rng(n + channels)
    value = torch.from_numpy(rng.uniform(0, 1, (1, n, 2))).cuda()
    image = torch.from_numpy(rng.uniform(0, 1, (1, n, channels))).cuda() if channels else None
    got = pla.lattice_filter(value.view((1,) + dims + (2,)), image.view((1,) + dims + (channels,)) if channels else None,
                             bilateral=channels > 0, theta_alpha=widths[0], theta_beta=widths[1], theta_gamma=widths[0])
    positions = pla.compute_positions(image[0] if channels else None, dims, float(np.float32(widths[0])),
                                      float(np.float32(widths[1])), dtype=torch.float64)
    lat = pla.PermutohedralLattice(pd, 3, n, dtype=torch.float64)
    lat.set_point_grid(dims)

    def filtered(positions):
        return lat.filter(torch.empty_like(value[0]), value[0], positions)

    want = filtered(positions)
    assert lat.num_vertices == n * (pd + 1)
    assert torch.equal(got.view(want.shape), want) and torch.equal(filtered(positions), want)
    off = filtered(positions * (1.0 + 2.0 ** -22))
    assert float((off != want).any(dim=1).double().mean()) > 0.5
    lat.close()
