"""Backward pass (BPTT) through the GLIF3 simulation on the GPU.

bmtk has no gradient code; the definition of the differentiable model is this
package's own and is stated in ``include/bmtk_amd.h`` (``bmtk_glif3_bwd``):
triangular surrogate spike derivative, refractory bookkeeping not
differentiated, everything else the exact transpose of the forward update.
"""
import ctypes as C

import numpy as np
import torch

from . import _lib
from .layout import NASC, NREC
from .ops import _p, _stream


def spike_counts(bits, ne):
    """int32 [ne] spikes per element over all rows of ``bits`` (int64 [n_steps, words])."""
    lib = _lib.load()
    counts = torch.empty(ne, dtype=torch.int32, device=bits.device)
    _lib.check(lib.bmtk_spike_counts(_p(bits, torch.int64), bits.shape[1], bits.shape[0], ne, _p(counts), _stream()))
    return counts


def _plain(counts, n_steps, batch, pop_id, targets):
    """Whether the call is what bmtk_rate_mse takes: its types and layouts on the current device, and nobody who follows the
    operations (gradients by the targets, tracing, transforms, modes)."""
    tensors = (counts, pop_id, targets)
    if any(type(t) is not torch.Tensor or not t.is_cuda or t.get_device() != torch.cuda.current_device() for t in tensors):
        return False
    if any(torch._C._functorch.is_functorch_wrapped_tensor(t) or t.is_conj() or t.is_neg() for t in tensors):
        return False
    if torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack() or torch.autograd.forward_ad._current_level >= 0:
        return False
    return (type(n_steps) is int and n_steps > 0 and type(batch) is int and batch > 0 and counts.dtype == torch.int32 and pop_id.dtype == torch.int64
            and targets.dtype == torch.float32 and not targets.requires_grad and pop_id.dim() == 1 and targets.dim() == 2
            and pop_id.numel() > 0 and counts.numel() == pop_id.numel() * batch and targets.shape[0] == batch and targets.shape[1] > 0
            and counts.is_contiguous() and pop_id.is_contiguous() and targets.is_contiguous())


def rate_mse(counts, n_steps, batch, pop_id, targets):
    """MSE between population rates and targets, and its derivative per spike.

    counts  int32 [n*batch] spikes per element; pop_id int64 [n] population of
    every neuron; targets float [batch, n_pops] in spikes per neuron per step.
    The rate of population p in trial b is mean over its neurons and steps of z.
    Returns (loss, dl_dz_const float32 [n*batch]).

    Two launches and one look at the device; as array operations (every other form of the arguments) it is some 25 launches,
    which a training step of a small network waits for."""
    n = pop_id.numel()
    n_pops = targets.shape[1]
    if _plain(counts, n_steps, batch, pop_id, targets):
        dev = counts.device
        work = torch.zeros(n_pops * (batch + 1) + 1, dtype=torch.int64, device=dev)
        loss, per_spike = torch.empty((), dtype=torch.float32, device=dev), torch.empty(counts.numel(), dtype=torch.float32, device=dev)
        _lib.check(_lib.load().bmtk_rate_mse(_p(counts), n, batch, n_steps, _p(pop_id), n_pops, _p(targets), _p(work), _p(loss), _p(per_spike),
                                             _stream()))
        if work[-1].item():
            raise RuntimeError("pop_id outside 0..{}".format(n_pops - 1))
        return loss, per_spike
    dev = counts.device
    size = torch.bincount(pop_id, minlength=n_pops).to(torch.float32)
    c = counts.view(n, batch).to(torch.float32)
    rate = torch.zeros(n_pops, batch, device=dev).index_add_(0, pop_id, c) / (size.view(-1, 1) * n_steps)
    err = rate.t() - targets
    loss = (err * err).mean()
    # d loss / d z[b, i, t] = 2 err[b, p(i)] / (batch * n_pops) / (size[p(i)] * n_steps)
    g = 2.0 * err / (batch * n_pops) / (size.view(1, -1) * n_steps)
    return loss, g.t()[pop_id].contiguous().view(-1)


class Glif3Bptt:
    """Reverse-time adjoint over a recorded forward run of a ``Glif3Simulator``: of a batch, or of a single trial
    built with ``resident=False``.  (A batch whose simulator leaves ``resident`` at "auto" runs the forward part with
    resident trials where they pay: 1.18 instead of 1.52 ms a step of training at 3,001 neurons x 12 trials x 100 steps.)"""

    # A synapse costs the swept form more once the L2s no longer hold the adjoint ring; the blocked form has a fixed part per
    # row and range, which long rows share among more synapses.  Measured on one MI355X, whole calls of 40 steps, us per step
    # swept / blocked at in-degree 120, 220, 400, 750 (neurons x trials; MB of ring): 9003 x 32 (28) 25/38 34/42 48/51 78/70;
    # 15013 x 32 (46) 45/49 58/58 84/76 131/110; 51978 x 32 (160) 198/170 290/212 452/294 753/446; 20011 x 16 (31) 44/54 64/70 98/99
    # 165/152; 27011 x 16 (41) 63/64 91/87 140/124 244/199; 27011 x 12 (31) 63/65 96/89 156/128 273/203; 15013 x 20 (29) 45/48 63/59
    # 97/81 160/120; 27011 x 8 (21) 43/53 67/76 107/112 186/174; 51978 x 4 (20) 77/81 127/128 212/195 403/350.  The forms cross
    # where the ring times the cube root of the in-degree reaches these marks: lower for batches whose adjoint rows (four
    # bytes a trial) are no whole lines of 64 bytes, so that the swept form's gathers fetch what they do not use.
    BLOCKED_MIN_RING_MB = 31.0          # at in-degree 400, 16 trials
    # 32, 48 and 64 trials, where the blocked form takes two steps per pass: ring times square root of the in-degree.  Swept / blocked as they
    # are now (us per step): 9003 x 32 at in-degree 250 34/36, 400 47/43, 750 76/59; 7000 x 32, 600 47/45; 11000 x 32, 200 34/38;
    # 13000 x 32, 120 35/37; 15000 x 32, 220 52/47; 5000 x 64, 300 42/38; 6500 x 64, 150 39/38; 4000 x 48, 900 64/53
    BLOCKED_MIN_RING_MB_TWO = 25.5
    BLOCKED_MIN_RING_MB_RAGGED = 22.0, 20.0   # other batches up to 16, and above (where it takes two steps per pass)
    # more than 16 trials and two_steps=False, whole lines and others, times the cube root.  Swept / blocked, us per step: 9003 x 32, in-degree 750 75/82;
    # 15000 x 32, 220 55/67, 500 95/94; 20011 x 32, 220 84/84; 30011 x 32, 120 101/110, 400 222/175; 15013 x 20, 220 60/68, 750 161/133; 12000 x 24, 300
    # 60/68; 8000 x 40, 300 58/70; 12000 x 40, 300 104/93
    BLOCKED_MIN_RING_MB_ONE = 50.0, 32.0
    BLOCKED_MIN_RING_MB_FOUR = 17.0     # four trials: a quarter of a line
    # Four trials through a table of more than 150 MB, which does not stay in the memory-side cache beside the rest: launches of
    # their own for the parts (27011 x 4, in-degree 750: 139 against 147 swept; 33123 x 4, 598: 155 against 187 and 169 blocked;
    # 20011 x 4, 750, 120 MB: 106 and 105)
    PLAIN_MIN_TABLE_BYTES = 150e6

    @classmethod
    def blocked_pays(cls, n, batch, ring_slots, nnz, two_steps=True):
        """Whether the blocked form is expected to take less time per step than the swept form.  ``two_steps``: as it will be built."""
        ring_mb = ring_slots * NREC * n * batch * 4e-6
        if batch % 16 == 0 and batch > 16 and two_steps:
            return ring_mb * (nnz / (400.0 * n)) ** 0.5 >= cls.BLOCKED_MIN_RING_MB_TWO
        least = (cls.BLOCKED_MIN_RING_MB_ONE[batch % 16 != 0] if batch > 16 and not two_steps else
                 cls.BLOCKED_MIN_RING_MB if batch % 16 == 0 else cls.BLOCKED_MIN_RING_MB_FOUR if batch <= 4
                 else cls.BLOCKED_MIN_RING_MB_RAGGED[batch > 16])
        return ring_mb * (nnz / (400.0 * n)) ** (1.0 / 3.0) >= least

    @staticmethod
    def target_ranges(n, batch, ring_slots, nnz, two_steps=True):
        """Target ranges of the blocked table.  Two steps per pass (batches above 16): what counts is how long a row's segments are, a
        segment has its fixed part.  us per two steps with 8 / 16 / 24 / 32 ranges: 52000 x 32, in-degree 100 280/291/313/335; 25000 x 40, 120
        212/226/246/270; 12000 x 64, 150 132/135/141/152; 45000 x 40, 200 517/503/530/563; 31000 x 64, 300 490/462/472/489; 20000 x 20, 300
        148/145/149/156; 40000 x 24, 400 390/368/366/372; 30011 x 32, 600 331/314/315/319; 20011 x 20, 700 256/248/244/244; 15000 x 32, 800
        183/182/179/182; 51978 x 32, 1000 888/838/809/812.  Measured up to 200 MB of adjoint ring; larger ones, and one step per pass,
        are left to the share of a ring that an L2 holds."""
        if batch <= 16 or not two_steps or ring_slots * NREC * n * batch * 4 > 200e6:
            from . import ops
            return ops.blocked_table_blocks(n, batch, ring_slots)
        in_degree = nnz / n
        return 8 if in_degree < 175.0 else 16 if in_degree < 600.0 else 24

    @classmethod
    def plain_pays(cls, batch, nnz):
        """Whether a launch per part is expected to take less time than the swept form (where the blocked form does not pay)."""
        return batch <= 4 and 8 * nnz >= cls.PLAIN_MIN_TABLE_BYTES

    def __init__(self, sim, dampening=0.3, blocked=None, n_blocks=None, two_steps=True, swept=None):
        """Three forms of the pass, the same gradients.  ``swept``: one launch per two steps through the plain
        source-major table (its adjoint ring ``lam_ring`` has two slots more than ``sim.L``); ``blocked``: the recurrent
        table regrouped by target range for the transposed propagation; neither: a launch per part and step, any batch.
        None leaves the choice to ``blocked_pays`` and ``plain_pays`` where the batch (a multiple of 4 up to 64) allows it.  ``n_blocks``:
        number of target ranges, a multiple of 8 (None: ``target_ranges``); ``two_steps``: let the blocked form
        take two steps per pass over its table (batches above 16; ``gz`` then holds the partial sums of both)."""
        if sim.res_span or sim.delay_offset:
            raise ValueError("the backward pass needs a simulator built with resident=False (or a batch) and delay_offset 0")
        self.sim, self.dampening = sim, float(dampening)
        self.lib = _lib.load()
        dev, ne = sim.dev, sim.ne
        self.lam_V = torch.zeros(ne, device=dev)
        self.lam_asc = torch.zeros(NASC, ne, device=dev)
        self.lam_y1 = torch.zeros(NREC, ne, device=dev)
        self.lam_y2 = torch.zeros(NREC, ne, device=dev)
        grouped = sim.rec is not None and sim.batch % 4 == 0 and sim.batch <= 64
        can_block = grouped and sim.L * NREC * ne < (1 << 30)
        can_sweep = grouped and ne < (1 << 24) and sim.L + 2 <= 64 and (sim.L + 2) * NREC * ne < (1 << 30)
        if swept and (blocked or not can_sweep):
            raise ValueError("the swept form needs a recurrent table, a batch that is a multiple of 4 up to 64, delays within 61 "
                             "steps and no blocked table")
        if blocked and not can_block:
            raise ValueError("the blocked table needs a recurrent table and a batch that is a multiple of 4 up to 64")
        if blocked is None and not swept:
            blocked = can_block and (swept is False or not can_sweep or self.blocked_pays(sim.n, sim.batch, sim.L, sim.rec.nnz, two_steps))
            swept = not blocked and can_sweep and swept is None and not self.plain_pays(sim.batch, sim.rec.nnz)
        self.swept, blocked = bool(swept), bool(blocked)
        # (the swept form writes the adjoint slots of two steps ahead while others are still read)
        self.lam_ring = torch.zeros(sim.L + (2 if self.swept else 0), NREC, ne, device=dev)
        self.d_rec_w = torch.zeros(sim.rec.nnz, device=dev) if sim.rec is not None else None
        self.blk = None
        if blocked:
            self.n_blocks = int(n_blocks or self.target_ranges(sim.n, sim.batch, sim.L, sim.rec.nnz, two_steps))
            if self.n_blocks % 8:
                raise ValueError("n_blocks must be a multiple of 8")
            self.blk = sim.rec.blocked(sim.n, self.n_blocks)
            self.d_blk_w = torch.zeros(sim.rec.nnz, device=dev)
        # the blocked form takes two steps per pass over its table when gz has room for both steps' partial sums
        self.gz_planes = (16 if two_steps else 8) if blocked else 1
        self.gz = torch.zeros(self.gz_planes * ne, device=dev)
        self.d_inp_w = torch.zeros(sim.inp.nnz, device=dev) if sim.inp is not None and sim.in_ptr is not None else None

    def zero(self):
        # (all in a launch or two: eight small ones were 55 us of a training step, these 15)
        torch._foreach_zero_([t for t in (self.lam_V, self.lam_asc, self.lam_y1, self.lam_y2, self.lam_ring, self.gz, self.d_rec_w, self.d_inp_w)
                              if t is not None])

    def _struct(self, fwd, dl_dz_const, dl_dz, blocked):
        sim, saved, bits = self.sim, fwd["saved"], fwd["bits"]
        if saved is None or bits is None:
            raise ValueError("forward run was made without save_state=True or without spike bits")
        # (resident trials can give up on one another and then leave a record that was never written; no later step of a training
        #  would show it.  A capture cannot look.)
        if sim._pending_check and not torch.cuda.is_current_stream_capturing():
            sim.check()
        n_steps = bits.shape[0]
        a = _lib.Glif3Bwd()
        a.n_neurons, a.batch, a.ring_slots, a.h, a.dampening = sim.n, sim.batch, self.lam_ring.shape[0], sim.h, self.dampening
        a.swept = 1 if self.swept and not blocked else 0
        a.prop, a.prop_stride, a.class_id = _p(sim.prop), sim.prop.shape[1], _p(sim.class_id)
        a.save_v, a.save_flags = _p(saved["v"], torch.float32, n_steps * sim.ne), _p(saved["flags"], torch.uint8)
        a.spike_bits, a.spike_bits_stride = _p(bits, torch.int64), bits.shape[1]
        if sim.rec is not None:
            a.rec_indptr, a.rec_packed = _p(sim.rec.indptr), _p(sim.rec.packed())
            if not blocked:
                a.d_rec_w = _p(self.d_rec_w)
            else:
                a.blk_count, a.blk_indptr, a.blk_packed = self.n_blocks, _p(self.blk[0]), _p(self.blk[1])
                a.gz_planes = self.gz_planes
                a.d_blk_w = _p(self.d_blk_w)
        if self.d_inp_w is not None:
            a.in_ptr, a.in_events = _p(sim.in_ptr), _p(sim.in_events)
            a.inp_indptr, a.inp_packed = _p(sim.inp.indptr), _p(sim.inp.packed())
            a.d_inp_w = _p(self.d_inp_w)
        a.dl_dz = _p(dl_dz, torch.float32, n_steps * sim.ne, "dl_dz")
        a.dl_dz_const = _p(dl_dz_const, torch.float32, sim.ne, "dl_dz_const")
        a.lam_V, a.lam_asc, a.lam_y1, a.lam_y2 = (_p(x) for x in (self.lam_V, self.lam_asc, self.lam_y1, self.lam_y2))
        a.lam_ring, a.gz = _p(self.lam_ring), _p(self.gz)
        return a, saved["step0"], n_steps

    def backward(self, fwd, dl_dz_const=None, dl_dz=None):
        """``fwd`` is what ``sim.run(n, save_state=True)`` returned.  Accumulates
        into ``d_rec_w`` / ``d_inp_w`` (same order as ``sim.rec`` / ``sim.inp``).
        Calls for consecutive chunks must come in reverse time order.  Synchronises once behind runs with resident trials,
        to raise if they gave up (``Glif3Simulator.check``)."""
        a, step0, n_steps = self._struct(fwd, dl_dz_const, dl_dz, self.blk is not None)
        _lib.check(self.lib.bmtk_glif3_simulate_bwd(C.byref(a), step0, n_steps, _stream()))
        if self.blk is not None:  # the blocked kernel accumulates in its table's order: back to the order of sim.rec
            self.d_rec_w.index_add_(0, self.blk[2], self.d_blk_w)
            self.d_blk_w.zero_()

    def backward_stepwise(self, fwd, dl_dz_const=None, dl_dz=None, between=None):
        """The same pass as a loop over the three per-step entry points (transposed propagation through the
        source-major table, state adjoint, weight gradients), calling ``between(k)`` after the state adjoint of
        record row ``k`` -- the place for work of the caller's own on the adjoint state (clipping, a loss that
        depends on it).  Several launches per step where ``backward`` has two: for training loops use ``backward``."""
        from . import ops
        sim = self.sim
        a, step0, n_steps = self._struct(fwd, dl_dz_const, dl_dz, False)
        gz = self.gz[:sim.ne]
        for k in range(n_steps - 1, -1, -1):
            if sim.rec is not None:
                ops.csr_propagate_bwd(sim.rec, self.lam_ring, sim.n, sim.batch, step0 + k, gz=gz)
            else:
                gz.zero_()
            _lib.check(self.lib.bmtk_glif3_step_bwd(C.byref(a), step0, k, 1, _stream()))
            if self.d_rec_w is not None or self.d_inp_w is not None:
                _lib.check(self.lib.bmtk_csr_weight_grad(C.byref(a), step0, k, _stream()))
            if between is not None:
                between(k)
