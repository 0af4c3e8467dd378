"""Dense-CRF mean-field message passing on the lattice filter, the use the reference names for
its op (README.md:16 of the reference tree; the reference itself holds no CRF code, so this loop
is this library's own harness around the op's two filters).

Per iteration ``Q <- softmax(logits + bilateral(Q; theta_alpha, theta_beta) + spatial(Q;
theta_gamma))``, where both filters are the ``LatticeFilter`` op's (features and normalisation
as in src/LatticeFilterKernel.cpp:126-142).  The features never change between iterations, so
each batch item builds its two lattices once (``pl_build_image``) and every message is one
``pl_apply``; the reference's op would rebuild them for each of its calls
(src/LatticeFilterKernel.cpp:152-179).  The gradient pass is the reference's rule
(lattice_filter_op_loader.py:32-54): the same two filters with ``reverse=True`` on the upstream
gradient.

The 2 x batch lattices of a step are independent of each other, and at image sizes like 512 x 512
one apply is a chain of short kernels that leaves most of the GPU idle.  They are applied together, every
pass of all of them in one launch on the caller's stream; where that cannot be (see
``pl_mean_field_messages``) every lattice works on a HIP stream of its own (default priority), as the builds
do: a message-passing step waits for its input on the caller's stream, runs the applies of all lattices side
by side, and the caller's stream waits for all of them before it adds the messages up.

torch carries the tensors; the filters, and the softmax over the logits and both messages, are the
HIP library's.
"""
import torch

from . import (PL_OPT_VERTEX_LISTS, PermutohedralLattice, mean_field_infer, mean_field_messages, mean_field_update,
               mean_field_update_supported)


class MeanField:
    """Lattices of one batch of guide images ``[B, H, W, C_ref]`` for ``n_classes`` labels."""

    def __init__(self, guide, n_classes, theta_alpha=80.0, theta_beta=13.0, theta_gamma=3.0,
                 concurrent=True):
        if guide.dim() < 3:
            raise ValueError("guide must be [batch, spatial..., channels]")
        self.batch = int(guide.shape[0])
        self.sdims = [int(s) for s in guide.shape[1:-1]]
        self.n = 1
        for s in self.sdims:
            self.n *= s
        self.n_classes = int(n_classes)
        self.thetas = (float(theta_alpha), float(theta_beta), float(theta_gamma))
        rc, k = int(guide.shape[-1]), len(self.sdims)
        self.concurrent = bool(concurrent)
        self._streams = [torch.cuda.Stream(device=guide.device) if self.concurrent else None
                         for _ in range(2 * self.batch)]
        self.bilateral = [PermutohedralLattice(k + rc, self.n_classes + 1, self.n,
                                               stream=self._streams[2 * b])
                          for b in range(self.batch)]
        self.spatial = [PermutohedralLattice(k, self.n_classes + 1, self.n,
                                             stream=self._streams[2 * b + 1])
                        for b in range(self.batch)]
        for lat in self.bilateral + self.spatial:
            lat.set_option(PL_OPT_VERTEX_LISTS, 2)      # lists for applies in pairs
        shape = (self.batch, self.n, self.n_classes)
        self._msg_bi = torch.empty(shape, dtype=torch.float32, device=guide.device)
        self._msg_sp = torch.empty(shape, dtype=torch.float32, device=guide.device)
        self.rebuild(guide)

    def rebuild(self, guide):
        """Build the lattices again for another batch of guide images of the same shape."""
        self.guide = guide.contiguous()
        rc = int(guide.shape[-1])
        theta_alpha, theta_beta, theta_gamma = self.thetas
        self._side_streams_wait_for_caller()
        # all builds are enqueued, each on its lattice's stream, before the first is waited for: a
        # build is a chain of a dozen short kernels, and 2 x batch of them run side by side
        for b in range(self.batch):
            self.bilateral[b].build_image_begin(self.guide[b].reshape(self.n, rc), self.sdims,
                                                theta_alpha, theta_beta)
            self.spatial[b].build_image_begin(None, self.sdims, theta_gamma)
        for lat in self.bilateral + self.spatial:
            lat.build_end()
        # (a build has ended when its lattice is complete: nothing to wait for here)

    def _side_streams_wait_for_caller(self):
        """What the caller's stream has been given so far is complete before any lattice's stream
        goes on (the guide, the tensor a message is computed from)."""
        if not self.concurrent:
            return
        ready = torch.cuda.Event()
        ready.record(torch.cuda.current_stream())
        for s in self._streams:
            s.wait_event(ready)

    def _caller_waits_for_side_streams(self):
        if not self.concurrent:
            return
        caller = torch.cuda.current_stream()
        for s in self._streams:
            done = torch.cuda.Event()
            done.record(s)
            caller.wait_event(done)

    def _apply_all(self, q, reverse):
        """Both messages of every item, in the lattices' own buffers."""
        q = q.contiguous().view(self.batch, self.n, self.n_classes)
        self._side_streams_wait_for_caller()
        for b in range(self.batch):
            self.bilateral[b].apply(self._msg_bi[b], q[b], reverse)
            self.spatial[b].apply(self._msg_sp[b], q[b], reverse)
        self._caller_waits_for_side_streams()

    def messages(self, q, reverse=False):
        """bilateral(q) + spatial(q) for ``q [B, ..., n_classes]`` (any spatial shape of N points)."""
        if self.batch and q.is_cuda and q.device == self._msg_bi.device:
            flat = q.contiguous().view(self.batch, self.n, self.n_classes)
            total = torch.empty_like(self._msg_bi)
            if mean_field_messages(self.bilateral, self.spatial, total, flat.detach(), reverse):
                return total
        self._apply_all(q, reverse)
        return self._msg_bi + self._msg_sp

    def infer(self, logits, iterations=5):
        """-> Q after ``iterations`` mean-field updates, shaped like ``logits`` (none for a negative count)."""
        iterations = len(range(iterations))
        flat = logits.contiguous().view(self.batch, self.n, self.n_classes)
        own = self._own_messages() and mean_field_update_supported(flat)
        if own and self.batch:
            q = torch.empty_like(flat)
            if mean_field_infer(self.bilateral, self.spatial, q, flat, iterations):
                return q.view(logits.shape)
        q = torch.softmax(flat, dim=-1)
        if not own:
            # (logits that autograd follows into the last softmax, among others)
            for _ in range(iterations):
                q = torch.softmax(flat + self.messages(q), dim=-1)
            return q.view(logits.shape)
        for _ in range(iterations):
            # (q is read by the lattices' streams, and the caller's stream, which writes it anew, has
            # waited for them)
            self._apply_all(q, False)
            mean_field_update(q, flat, self._msg_bi, self._msg_sp)
        return q.view(logits.shape)

    def reverse(self, upstream):
        """The op's registered gradient of one message-passing step with respect to its input:
        both filters with ``reverse=True`` on ``upstream``, summed."""
        total = self.messages(upstream, reverse=True).view(upstream.shape)
        # (messages put in the place of this class's may give the same tensor again on the next call)
        return total if self._own_messages() else total.clone()

    def _own_messages(self):
        """Whether ``messages`` is this class's, neither a derived class's nor put on the object."""
        return getattr(self.messages, "__func__", None) is MeanField.messages

    def close(self):
        for lat in self.bilateral + self.spatial:
            lat.close()
        self.bilateral, self.spatial = [], []
