"""The images of a batch whose lattices are kept for the gradient: their passes enqueued together, against the
op on one image after the other (no gradient asked for), forward and backward."""
import ctypes as C

import pytest
import torch

import permutohedral_lattice_amd as pla

pytestmark = pytest.mark.gpu


def guide_of(sides, channels, kind, gen):
    """smooth; with noise that leaves few vertices shared; with noise that a merging build cannot take."""
    axes = torch.meshgrid(*(torch.arange(s, device="cuda", dtype=torch.float32) for s in sides), indexing="ij")
    t = sum(a / (17.0 + 5 * i) for i, a in enumerate(axes))
    guide = torch.stack([torch.sin(t * (1 + c)) for c in range(channels)], -1)
    noise = {"smooth": 0.05, "noisy": 0.6, "wild": 40.0}[kind]
    return guide + noise * (torch.rand(guide.shape, generator=gen, device="cuda") - 0.5)


def close(got, want):
    assert torch.isfinite(got).all()
    # (the same terms in another order)
    assert float((got - want).double().norm() / want.double().norm()) <= 2e-6
    assert float((got - want).abs().max()) <= 2e-5 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("channels", [1, 2, 3, 4, 7, 21, 31, 32])
@pytest.mark.parametrize("sides,guide,kinds", [
    ((37, 50), 3, ("smooth", "smooth")),
    ((64, 48), 3, ("smooth", "wild", "noisy", "smooth")),
    ((40, 33), 0, ("smooth",) * 3),
    ((12, 20, 17), 1, ("noisy", "smooth", "smooth", "noisy", "smooth", "smooth")),
    ((33, 40), 1, ("smooth", "noisy", "wild", "smooth", "smooth")),
    ((20, 24), 6, ("smooth", "smooth")),
    ((3, 400), 3, ("smooth", "smooth")),
])
def test_batches(sides, guide, kinds, channels):
    gen = torch.Generator(device="cuda").manual_seed(channels)
    batch = len(kinds)
    ref = torch.stack([guide_of(sides, guide, kind, gen) for kind in kinds]) if guide else None
    thetas = dict(bilateral=guide > 0, theta_alpha=6.0, theta_beta=0.4, theta_gamma=5.0)
    for _ in range(3):      # (the lattices of the first call serve the next, under other inputs)
        x = torch.rand((batch,) + sides + (channels,), generator=gen, device="cuda").requires_grad_(True)
        up = torch.randn(x.shape, generator=gen, device="cuda")
        out = pla.lattice_filter(x, ref, **thetas)
        (grad,) = torch.autograd.grad(out, x, up)
        for b in range(batch):
            one = None if ref is None else ref[b:b + 1]
            with torch.no_grad():
                close(out[b:b + 1], pla.lattice_filter(x[b:b + 1], one, **thetas))
                close(grad[b:b + 1], pla.lattice_filter(up[b:b + 1], one, reverse=True, **thetas))
        if ref is not None:
            ref = ref.flip(0).contiguous()


def test_vertices_numbered_by_the_build_and_by_the_pass_in_one_launch():
    """Of two volumes one has so many rows of sums for vertices of other workgroups that its lattice leaves the
    numbering to the pass in its next build; the other's numbers its vertices."""
    gen = torch.Generator(device="cuda").manual_seed(2)
    sides = (48, 96, 96)
    n = 48 * 96 * 96
    ref = torch.stack([torch.rand((n, 1), generator=gen, device="cuda"),
                       torch.linspace(0.0, 1.0, n, device="cuda").view(n, 1)]).view((2,) + sides + (1,))
    thetas = dict(bilateral=True, theta_alpha=6.0, theta_beta=0.2, theta_gamma=1.0)
    for call in range(4):
        x = torch.rand((2,) + sides + (2,), generator=gen, device="cuda").requires_grad_(True)
        up = torch.randn(x.shape, generator=gen, device="cuda")
        out = pla.lattice_filter(x, ref, **thetas)
        listed = [lat.info(pla.PL_INFO_FOREIGN_ROWS) >= 0 for lat in out.grad_fn.lent.lattices]
        assert all(lat.info(pla.PL_INFO_BUILD_MERGED) == 1 for lat in out.grad_fn.lent.lattices)
        if call:
            assert sorted(listed) == [False, True]
        (grad,) = torch.autograd.grad(out, x, up)
        for b in range(2):
            with torch.no_grad():
                close(out[b:b + 1], pla.lattice_filter(x[b:b + 1], ref[b:b + 1], **thetas))
                close(grad[b:b + 1], pla.lattice_filter(up[b:b + 1], ref[b:b + 1], reverse=True, **thetas))
        del out, grad


def test_applies_behind_one_build_each():
    """Lattices that were built one by one, with and without lists, applied together."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    h, w = 45, 70
    for channels in (3, 21):
        lattices, positions = [], []
        for kind in ("smooth", "noisy", "smooth"):
            pos = pla.compute_positions(guide_of((h, w), 3, kind, gen).contiguous(), (h, w), 6.0, 0.4)
            lat = pla.PermutohedralLattice(5, channels + 1, h * w)
            lat.set_point_grid((h, w))
            lattices.append(lat)
            positions.append(pos)
        x = torch.rand((3, h * w, channels), generator=gen, device="cuda")
        together, alone = torch.empty_like(x), torch.empty_like(x)
        for lists in ((0, 0, 0), (1, 1, 1), (0, 1, 0)):
            for lat, pos, on in zip(lattices, positions, lists):
                lat.set_option(pla.PL_OPT_VERTEX_LISTS, on)
                lat.build(pos)
            for reverse in (False, True, False):
                pla._apply_many(lattices, together.fill_(float("nan")), x, reverse)
                for i, lat in enumerate(lattices):
                    lat.apply(alone[i], x[i], reverse)
                close(together, alone)
        for lat in lattices:
            lat.close()


def test_what_is_refused():
    lib = pla._lib
    a, b = pla.PermutohedralLattice(5, 4, 64), pla.PermutohedralLattice(5, 4, 64)
    other = pla.PermutohedralLattice(5, 3, 64)
    x = torch.rand((2, 64, 3), device="cuda")
    out = torch.empty_like(x)
    ref, dims = torch.rand((2, 64, 3), device="cuda"), (C.c_int * 2)(8, 8)

    def images(*lattices):
        return lib.pl_filter_images(len(lattices), pla._handles(lattices), C.c_void_p(out.data_ptr()),
                                    C.c_void_p(x.data_ptr()), C.c_void_p(ref.data_ptr()), 3, 2, dims, 4.0, 0.5, 0)

    def many(*lattices):
        return lib.pl_apply_many(len(lattices), pla._handles(lattices), C.c_void_p(out.data_ptr()),
                                 C.c_void_p(x.data_ptr()), 0)

    assert images(a, a) == pla.PL_EINVAL and images(a, other) == pla.PL_EINVAL
    assert lib.pl_filter_images(0, None, None, None, None, 3, 2, dims, 4.0, 0.5, 0) == pla.PL_EINVAL
    assert many(a, b) == pla.PL_ESTATE          # not built
    assert images(a, b) == pla.PL_OK and many(a, b) == pla.PL_OK
    assert many(a, a) == pla.PL_EINVAL
    torch.cuda.synchronize()
    for lat in (a, b, other):
        lat.close()


@pytest.mark.parametrize("batch,channels,guide", [(2, 3, 3), (5, 1, 3), (3, 21, 3), (9, 3, 0)])
def test_the_op_on_batches(batch, channels, guide):
    """Together, on streams after an image that a merging build cannot take, and together again (32 calls on)."""
    gen = torch.Generator(device="cuda").manual_seed(batch)
    sides = (29, 52)
    thetas = dict(bilateral=guide > 0, theta_alpha=6.0, theta_beta=0.4, theta_gamma=5.0)
    for call in range(37):
        kinds = ["wild" if call == 1 and b == batch - 1 else "noisy" if b % 3 == 1 else "smooth" for b in range(batch)]
        ref = torch.stack([guide_of(sides, guide, kind, gen) for kind in kinds]) if guide else None
        x = torch.rand((batch,) + sides + (channels,), generator=gen, device="cuda")
        out = pla.lattice_filter(x, ref, **thetas)
        if call in (0, 1, 2, 3, 33, 34, 35, 36):
            for b in range(batch):
                close(out[b:b + 1], pla.lattice_filter(x[b:b + 1], None if ref is None else ref[b:b + 1], **thetas))


def test_noise_meets_a_table_that_is_far_too_small():
    """A build gives up on its table long before every key has seen all of its cells, and the results are
    those of the largest table."""
    h = w = 96
    gen = torch.Generator(device="cuda").manual_seed(1)
    pos = torch.rand((h * w, 5), generator=gen, device="cuda") * 200.0 - 100.0
    val = torch.rand((h * w, 3), generator=gen, device="cuda")
    out, want = torch.empty_like(val), torch.empty_like(val)
    for cells, into in ((4096, out), (131072, want)):
        lat = pla.PermutohedralLattice(5, 4, h * w)
        lat.set_option(pla.PL_OPT_TABLE_CELLS, cells)
        lat.filter(into, val, pos)
        assert lat.num_vertices > 50000
        lat.close()
    close(out, want)
