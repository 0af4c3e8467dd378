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
