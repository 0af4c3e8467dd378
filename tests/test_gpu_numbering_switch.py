"""One handle whose builds number their vertices in both ways by turns: in the build itself
(``filter`` on a grid) and in the pass behind it (``build``, and ``filter`` while tiles with too many
distinct keys keep a handle from merging them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(side, beta, seed, blobs):
    import torch
    from permutohedral_lattice_amd import synth
    img = synth.blob_image(side, side, seed) if blobs else synth.uniform_image((side, side, 3), seed)
    pos = synth.bilateral_positions(img, 8.0, beta)
    val = synth.uniform_image((side * side, 3), seed + 1)
    return pos, val, torch.from_numpy(pos).cuda(), torch.from_numpy(val).cuda()


def test_builds_and_filters_by_turns_on_one_handle():
    import oracle
    import torch
    import permutohedral_lattice_amd as pla
    side = 96
    pos, val, d_pos, d_val = _case(side, 0.125, 5, True)
    cpu = oracle.Lattice(5, 4, side * side)
    want = cpu.filter(val, pos, False)
    lat = pla.PermutohedralLattice(5, 4, side * side)
    lat.set_point_grid((side, side))
    out = torch.empty_like(d_val)
    for entry in "bfbffbbfb":
        out.zero_()
        if entry == "b":
            lat.build(d_pos)
            lat.apply(out, d_val)
        else:
            lat.filter(out, d_val, d_pos)
        assert lat.num_vertices == cpu.num_vertices, entry
        assert float(np.abs(out.cpu().numpy() - want).max()) <= 1e-5


def test_a_handle_that_returns_to_merging_again_and_again():
    """A noise image overflows the tiles' tables: plain builds for 32 calls, another try to merge,
    plain builds again."""
    import oracle
    import torch
    import permutohedral_lattice_amd as pla
    side = 64
    pos, val, d_pos, d_val = _case(side, 0.05, 9, False)
    cpu = oracle.Lattice(5, 4, side * side)
    want = cpu.filter(val, pos, False)
    lat = pla.PermutohedralLattice(5, 4, side * side)
    lat.set_point_grid((side, side))
    out = torch.empty_like(d_val)
    for call in range(37):
        out.zero_()
        lat.filter(out, d_val, d_pos)
        # (the try itself overflows and its call is repeated without merging: the second sends the
        # handle back to plain builds for longer than the calls that are left)
        assert lat.info(pla.PL_INFO_BUILD_MERGED) == 0, call
        assert lat.num_vertices == cpu.num_vertices
        assert float(np.abs(out.cpu().numpy() - want).max()) <= 1e-5


def test_the_way_to_number_is_kept_while_the_grid_is_the_same():
    """``filter_image`` sets the grid on every call.  A volume whose tiles share most of their vertices: the
    pass numbers them from the second call on, until another grid (or, after 32 builds, another count)."""
    import torch
    import permutohedral_lattice_amd as pla
    dims = (48, 96, 96)
    n = dims[0] * dims[1] * dims[2]
    gen = torch.Generator("cuda").manual_seed(11)
    guide = torch.rand((n, 1), device="cuda", generator=gen)
    val = torch.rand((n, 1), device="cuda", generator=gen)
    lat = pla.PermutohedralLattice(4, 2, n)
    outs, rows = [], []
    for call in range(36):
        out = torch.empty_like(val)
        lat.filter_image(out, val, guide, dims if call < 35 else (96, 48, 96), 6.0, 0.2)
        rows.append(lat.info(pla.PL_INFO_FOREIGN_ROWS))
        if call < 35:
            outs.append(out)
    assert rows[0] > 0 and rows[1] == -1 and rows[32] == -1     # (-1: numbered by the pass)
    assert rows[33] > 0 and rows[34] == -1 and rows[35] != -1
    for out in outs[1:]:
        assert float((out - outs[0]).abs().max()) <= 2e-6
    lat.close()


def test_the_way_to_number_follows_a_handle_s_inputs():
    """Volumes of one grid by turns, with vertices enough for the numbering pass and with few: a build goes by
    the vertices of the one before it, and the rows are counted anew after 32, 64 and then every 128 builds."""
    import torch
    import permutohedral_lattice_amd as pla
    dims = (48, 96, 96)
    n = dims[0] * dims[1] * dims[2]
    gen = torch.Generator("cuda").manual_seed(12)
    noisy = torch.rand((n, 1), device="cuda", generator=gen)
    smooth = torch.linspace(0.0, 1.0, n, device="cuda").view(n, 1)
    val = torch.rand((n, 1), device="cuda", generator=gen)
    lat = pla.PermutohedralLattice(4, 2, n)
    want = {}
    for _ in range(3):
        for guide in (noisy, smooth):
            for call in range(3):
                out = torch.empty_like(val)
                lat.filter_image(out, val, guide, dims, 6.0, 0.2)
                passed = lat.info(pla.PL_INFO_FOREIGN_ROWS) == -1
                # (the first of the same kind is numbered as the one before it asked for)
                assert passed == ((call > 0) == (guide is noisy))
                assert float((out - want.setdefault(id(guide), out)).abs().max()) <= 2e-6
    rows = []
    for call in range(360):
        lat.filter_image(out, val, noisy, dims, 6.0, 0.2)
        rows.append(lat.info(pla.PL_INFO_FOREIGN_ROWS))
    assert [call for call, r in enumerate(rows) if r != -1] == [0, 33, 98, 227, 356]
    lat.close()
