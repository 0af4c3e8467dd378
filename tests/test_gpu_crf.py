"""The dense-CRF mean-field workload (five iterations of softmax(logits + bilateral(Q) +
spatial(Q)), batch 2, reverse pass on the last iteration) on lattices built once per item,
against the same loop over the CPU oracle with a fresh lattice per message."""
import numpy as np
import pytest
import torch

from conftest import MAX_ABS_TOL, REL_L2_TOL, rel_l2
from permutohedral_lattice_amd import synth
from permutohedral_lattice_amd.crf import MeanField

import oracle

pytestmark = pytest.mark.gpu


def _inputs(batch, h, w, classes, seed):
    guide = np.stack([synth.blob_image(h, w, seed=seed + b) * 255.0 for b in range(batch)])
    logits = synth.normal_image((batch, h, w, classes), seed + 10)
    upstream = synth.normal_image((batch, h, w, classes), seed + 11)
    return guide.astype(np.float32), logits, upstream


@pytest.mark.parametrize("h,w", [(128, 128), (72, 100)])
def test_mean_field_loop_matches_the_oracle(h, w):
    batch, classes = 2, 21
    guide, logits, upstream = _inputs(batch, h, w, classes, 300 + h)
    mf = MeanField(torch.from_numpy(guide).cuda(), classes)
    q = mf.infer(torch.from_numpy(logits).cuda(), iterations=5)
    rev = mf.reverse(torch.from_numpy(upstream).cuda())
    torch.cuda.synchronize()
    q, rev = q.cpu().numpy(), rev.cpu().numpy()
    want_q, want_rev = oracle.mean_field(logits, guide, 5, upstream=upstream)
    # Q is a distribution over the classes: data in [0, 1]
    assert np.isfinite(q).all() and np.abs(q.sum(axis=-1) - 1.0).max() <= 1e-5
    assert np.abs(q - want_q).max() <= MAX_ABS_TOL and rel_l2(q, want_q) <= REL_L2_TOL
    # the reverse pass filters N(0,1) values: tolerance scaled by their range
    scale = float(np.abs(want_rev).max())
    assert np.abs(rev - want_rev).max() <= MAX_ABS_TOL * max(1.0, scale)
    assert rel_l2(rev, want_rev) <= REL_L2_TOL
    mf.close()


def test_mean_field_messages_equal_the_op_called_per_iteration():
    """Lattices built once and applied equal the op called afresh for every message."""
    import permutohedral_lattice_amd as pla
    batch, h, w, classes = 2, 64, 80, 5
    guide, logits, _ = _inputs(batch, h, w, classes, 400)
    d_guide = torch.from_numpy(guide).cuda()
    q = torch.softmax(torch.from_numpy(logits).cuda(), dim=-1)
    mf = MeanField(d_guide, classes)
    got = mf.messages(q).view(batch, h, w, classes)
    want = (pla.lattice_filter(q, d_guide, True, 80.0, 13.0, 3.0)
            + pla.lattice_filter(q, d_guide, False, 80.0, 13.0, 3.0))
    torch.cuda.synchronize()
    assert float((got - want).abs().max()) <= 1e-5
    mf.close()


@pytest.mark.parametrize("classes", [1, 2, 3, 20, 21, 40, 41, 64, 127, 128])
@pytest.mark.parametrize("n", [1, 63, 64, 255, 257, 1031])
def test_mean_field_update_is_the_softmax_of_the_sums(classes, n):
    import permutohedral_lattice_amd as pla
    gen = torch.Generator("cuda").manual_seed(classes * 10000 + n)
    logits, a, b = (3.0 * torch.randn((n, classes), device="cuda", generator=gen) for _ in range(3))
    if n > 2 and classes > 2:
        logits[1, 0] = float("-inf")       # (a class that is ruled out)
        logits[2, 1] = 3.0e38
    assert pla.mean_field_update_supported(logits)
    q = pla.mean_field_update(torch.full_like(logits, float("nan")), logits, a, b)
    want = torch.softmax((logits + (a + b)).double(), dim=-1)
    # in halves of an ulp of 1, 6e-8: the argument's rounding at most 0.37 (d e^-d), e^x 2, the quotient 1,
    # and the sum, of doubles, the terms' own 2.4 and 1 for its rounding: less than 8 for any number of classes
    assert float((q.double() - want).abs().max()) <= 8 * 6e-8
    for which in range(3):                          # in place of each array
        arrays = [t.clone() for t in (logits, a, b)]
        pla.mean_field_update(arrays[which], *arrays)
        assert torch.equal(arrays[which], q)


@pytest.mark.parametrize("classes", [2, 5, 21, 40, 41, 64, 128])
@pytest.mark.parametrize("scale", [1.0, 4.0])
def test_mean_field_update_is_as_precise_as_torch(classes, scale):
    """Its distance from the softmax in 64 bits is that of torch's additions and softmax, whatever the
    number of classes (2 %: what 8192 rows leave to chance where both sum as well as can be)."""
    import permutohedral_lattice_amd as pla
    gen = torch.Generator("cuda").manual_seed(classes)
    logits, a, b = (scale * torch.randn((8192, classes), device="cuda", generator=gen) for _ in range(3))
    sums = logits + (a + b)
    want = torch.softmax(sums.double(), dim=-1)
    q = pla.mean_field_update(torch.empty_like(logits), logits, a, b)
    assert float((q - want).norm()) <= 1.02 * float((torch.softmax(sums, dim=-1) - want).norm())


def test_mean_field_update_leaves_other_calls_to_torch():
    import permutohedral_lattice_amd as pla
    x = torch.zeros((4, 8), device="cuda")
    assert pla.mean_field_update_supported(x)
    assert not pla.mean_field_update_supported(x.double())
    assert not pla.mean_field_update_supported(x.t())
    assert not pla.mean_field_update_supported(x.clone().requires_grad_(True))
    assert not pla.mean_field_update_supported(x.reshape(-1)[1:25].view(3, 8))
    assert not pla.mean_field_update_supported(torch.zeros((2, 129), device="cuda"))
    # autograd into the last softmax, as before
    mf = MeanField(torch.rand((1, 24, 32, 3), device="cuda") * 255.0, 4)
    logits = torch.randn((1, 24, 32, 4), device="cuda", requires_grad=True)
    q = mf.infer(logits, iterations=2)
    (grad,) = torch.autograd.grad(q, logits, torch.ones_like(q))
    assert grad.shape == logits.shape
    with torch.no_grad():
        assert float((mf.infer(logits, iterations=2) - q).abs().max()) <= 1e-6
    mf.close()


def test_messages_put_in_the_place_of_the_class_s():
    """On the object or in a derived class: ``infer`` calls them, and what ``reverse`` gives does not
    change with the next call where they return one tensor again and again."""
    class Scaled(MeanField):
        def messages(self, q, reverse=False):
            self._msg_bi.copy_(super().messages(q, reverse) * 0.5)
            return self._msg_bi

    guide = torch.rand((1, 24, 32, 3), device="cuda") * 255.0
    logits, upstream = (torch.randn((1, 24, 32, 4), device="cuda") for _ in range(2))
    derived, plain = Scaled(guide, 4), MeanField(guide, 4)
    step = torch.softmax(logits, dim=-1)
    for _ in range(2):
        step = torch.softmax(logits + 0.5 * plain.messages(step).view(logits.shape), dim=-1)
    assert float((derived.infer(logits, 2) - step).abs().max()) <= 1e-6
    first = derived.reverse(upstream)
    kept = first.clone()
    derived.reverse(3.0 * upstream)
    assert torch.equal(first, kept)
    own = plain.messages
    plain.messages = lambda q, reverse=False: 0.5 * own(q, reverse)
    assert float((plain.infer(logits, 2) - step).abs().max()) <= 1e-6
    derived.close()
    plain.close()


@pytest.mark.parametrize("shape,guide_channels,classes,batch", [
    ((33, 47), 3, 4, 1), ((64, 80), 1, 5, 3), ((40, 24), 3, 15, 2), ((40, 24), 3, 16, 5), ((24, 33), 3, 31, 1),
    ((9, 17, 20), 1, 21, 2), ((8, 12, 16), 3, 7, 2), ((72, 100), 3, 21, 6),
    ((30, 2), 3, 21, 2)])                       # (a grid too thin for tiles)
def test_lattices_applied_together_equal_them_one_by_one(shape, guide_channels, classes, batch):
    """Every pass of all lattices in one launch, both messages sliced at once: the same sums in the same
    order as an apply each, so equal to an ulp or two of the weighted means."""
    import permutohedral_lattice_amd as pla
    gen = torch.Generator("cuda").manual_seed(batch * 100 + classes)
    guide = torch.rand((batch,) + shape + (guide_channels,), device="cuda", generator=gen) * 255.0
    x = torch.randn((batch,) + shape + (classes,), device="cuda", generator=gen)
    mf = MeanField(guide, classes, 10.0, 60.0, 3.0)
    n = mf.n
    flat = x.view(batch, n, classes)
    for reverse in (False, True):
        together = torch.full_like(flat, float("nan"))
        assert pla.mean_field_messages(mf.bilateral, mf.spatial, together, flat, reverse)
        mf._apply_all(flat, reverse)
        one_by_one = mf._msg_bi + mf._msg_sp
        scale = float(one_by_one.abs().max())
        assert float((together - one_by_one).abs().max()) <= 4 * 1.2e-7 * scale
    q = torch.full_like(flat, float("nan"))
    assert pla.mean_field_infer(mf.bilateral, mf.spatial, q, flat, 3)
    want = torch.softmax(flat, dim=-1)
    for _ in range(3):
        mf._apply_all(want, False)
        want = torch.softmax(flat + (mf._msg_bi + mf._msg_sp), dim=-1)
    # (an error of a few ulps of a logit of size s moves its probability by that many times s ulps)
    assert float((q - want).abs().max()) <= 3 * 8 * 1.2e-7 * float(flat.abs().max() + 2)
    mf.close()


def test_what_cannot_be_applied_together_is_applied_one_by_one():
    import permutohedral_lattice_amd as pla
    gen = torch.Generator("cuda").manual_seed(3)
    guide = torch.rand((2, 40, 56, 3), device="cuda", generator=gen) * 255.0
    for classes, option, together in ((33, None, False), (3, None, False), (21, (pla.PL_OPT_VERTEX_LISTS, 0), False),
                                      (21, (pla.PL_OPT_PAIR_BLUR, 0), False), (21, None, True)):
        x = torch.randn((2, 40, 56, classes), device="cuda", generator=gen)
        mf = MeanField(guide, classes)
        if option:
            mf.spatial[1].set_option(*option)
        out = torch.empty((2, 40 * 56, classes), device="cuda")
        assert pla.mean_field_messages(mf.bilateral, mf.spatial, out, x.view(out.shape)) == together
        got = mf.messages(x).view(x.shape)
        want = pla.lattice_filter(x, guide, True, 80.0, 13.0, 3.0) + pla.lattice_filter(x, guide, False, 80.0, 13.0, 3.0)
        assert float((got - want).abs().max()) <= 1e-4
        mf.close()


def test_lattices_with_different_kinds_of_lists_are_applied_together():
    """Built as for applies of their own, a spatial lattice of few corners a vertex lists its corners."""
    import permutohedral_lattice_amd as pla
    gen = torch.Generator("cuda").manual_seed(4)
    guide = torch.rand((2, 60, 76, 3), device="cuda", generator=gen) * 64.0
    x = torch.randn((2, 60, 76, 21), device="cuda", generator=gen)
    mf = MeanField(guide, 21)
    want = mf.messages(x)
    for lat in mf.bilateral + mf.spatial:
        lat.set_option(pla.PL_OPT_VERTEX_LISTS, 1)
    mf.rebuild(guide)
    out = torch.full((2, 60 * 76, 21), float("nan"), device="cuda")
    assert pla.mean_field_messages(mf.bilateral, mf.spatial, out, x.view(out.shape))
    assert float((out.view(want.shape) - want).abs().max()) <= 1e-4
    mf.close()


def test_lattices_applied_together_from_two_streams():
    """The lattices' own streams, and applies of single lattices on them, stay in order with it."""
    gen = torch.Generator("cuda").manual_seed(5)
    guides = [torch.rand((2, 96, 120, 3), device="cuda", generator=gen) * 255.0 for _ in range(2)]
    x = torch.randn((2, 96, 120, 21), device="cuda", generator=gen)
    mf, want = None, []
    for guide in guides:
        fresh = MeanField(guide, 21)
        want.append((fresh.infer(x, 3), fresh.messages(x, True)))
        torch.cuda.synchronize()
        fresh.close()
    mf = MeanField(guides[0], 21)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for turn in range(6):
        with torch.cuda.stream(streams[turn % 2]):
            streams[turn % 2].wait_stream(streams[1 - turn % 2])
            mf.rebuild(guides[turn % 2])
            q = mf.infer(x, 3)
            mf.bilateral[1].apply(mf._msg_bi[1], x[1].reshape(-1, 21))
            back = mf.messages(x, True).view(x.shape)
        streams[turn % 2].synchronize()
        assert float((q - want[turn % 2][0]).abs().max()) <= 1e-6
        assert float((back - want[turn % 2][1].view(x.shape)).abs().max()) <= 1e-5
    mf.close()


def _one_by_one(mf, x):
    mf._apply_all(x, False)
    out = mf._msg_bi + mf._msg_sp
    torch.cuda.synchronize()
    return out


def test_lattices_on_one_stream_applied_together_from_it_and_another():
    """Calls on another stream, the lattices' own and the other again, nothing built or applied in between
    and no wait by the caller: they share the lattices' value tables alone."""
    gen = torch.Generator("cuda").manual_seed(6)
    guide = torch.rand((2, 96, 120, 3), device="cuda", generator=gen) * 255.0
    own, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(own):
        mf = MeanField(guide, 21, concurrent=False)
    xs = [torch.randn((2, 96, 120, 21), device="cuda", generator=gen) for _ in range(6)]
    torch.cuda.synchronize()
    with torch.cuda.stream(own):
        want = [_one_by_one(mf, x) for x in xs]
    got = []
    for i, x in enumerate(xs):
        with torch.cuda.stream(own if i in (1, 3, 4) else other):
            got.append(mf.messages(x))
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert float((g - w).abs().max()) <= 1e-5
    mf.close()


def test_work_on_a_lattice_s_own_stream_between_calls_that_apply_them_together():
    """An export of the vertex values, and the replay of a captured apply: both only on the lattice's own
    stream, the calls before and behind on the same other one."""
    gen = torch.Generator("cuda").manual_seed(7)
    guide = torch.rand((2, 96, 120, 3), device="cuda", generator=gen) * 255.0
    xs = [torch.randn((2, 96, 120, 21), device="cuda", generator=gen) for _ in range(2)]
    mf = MeanField(guide, 21)
    own, other = mf._streams[2], torch.cuda.Stream()   # (own: of the second image's bilateral lattice)
    lat = mf.bilateral[1]
    want = [_one_by_one(mf, x) for x in xs]
    q = [mf.infer(x, 2) for x in xs]
    torch.cuda.synchronize()
    values = lat.debug_values()
    torch.cuda.synchronize()
    with torch.cuda.stream(other):
        again = mf.infer(xs[1], 2)
        exported = lat.debug_values()
        behind = mf.infer(xs[0], 2)
    torch.cuda.synchronize()
    assert torch.equal(exported, values)
    assert float((again - q[1]).abs().max()) <= 1e-6 and float((behind - q[0]).abs().max()) <= 1e-6
    static_in = xs[0][1].reshape(-1, 21).contiguous()
    static_out, alone = torch.empty_like(static_in), torch.empty_like(static_in)
    torch.cuda.synchronize()
    with torch.cuda.stream(own):
        lat.apply(alone, static_in)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=own):
        lat.apply(static_out, static_in)
    for _ in range(3):
        with torch.cuda.stream(own):
            static_out.zero_()
        got = []
        for i in (1, 0):
            with torch.cuda.stream(other):
                got.append(mf.messages(xs[i]))
            with torch.cuda.stream(own):
                graph.replay()
        with torch.cuda.stream(other):
            got.append(mf.messages(xs[1]))
        torch.cuda.synchronize()
        assert float((static_out - alone).abs().max()) <= 1e-5
        for g, i in zip(got, (1, 0, 1)):
            assert float((g - want[i]).abs().max()) <= 1e-5
    mf.close()


def test_the_number_of_iterations_is_what_range_makes_of_it():
    """A negative count is none, a whole number of any type counts, and a fraction is refused, whether the
    lattices are applied together or one by one."""
    guide = torch.rand((1, 24, 32, 3), device="cuda") * 255.0
    for classes in (5, 3):
        logits = torch.randn((1, 24, 32, classes), device="cuda")
        mf = MeanField(guide, classes)
        for none in (0, -1, np.int64(-3)):
            assert float((mf.infer(logits, none) - torch.softmax(logits, dim=-1)).abs().max()) <= 1e-6
        assert float((mf.infer(logits, np.int32(2)) - mf.infer(logits, 2)).abs().max()) <= 1e-6
        with pytest.raises(TypeError):
            mf.infer(logits, 2.0)
        mf.close()
