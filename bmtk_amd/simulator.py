"""Forward GLIF3 simulation on one GPU: the work ``nest.Simulate`` does for a
bmtk PointNet network (bmtk/simulator/pointnet/pointsimulator.py:159-166).

``Glif3Simulator`` owns the device state, the ring buffer and the synapse
tables, validates everything a kernel will index with on the host, and drives
``bmtk_glif3_simulate_fwd``.
"""
import ctypes as C
import math

import numpy as np
import torch

from . import _lib, network as net
from .layout import NPARAM, NPROP, NREC
from .ops import Glif3State, SpikeCompactor, SynapseTable, _dev, _p, _stream, glif3_precompute, n_words, unpack_bits


PULL_MAP_BYTES = 40 * 1024      # activity map of bmtk_csr_propagate_pull: what is left of 80 KB beside its accumulators
PULL_MIN_DENSITY = 0.06         # synaptic events per synapse and step from which "auto" pulls instead of pushing
                                # (the unfused pull form: batches below 8 and above 64)
# What a step of a batched run costs on one MI355X, in picoseconds, fitted to runs of 51,978 neurons x 60 M synapses at
# batches 8, 16, 32 and 0 - 3.2 Hz and of 230,924 neurons x 77 M synapses at batch 8: the fused pull form streams the
# joint table once per two steps (per synapse, divided by how full a row's blocks of 256 are) and adds a little per
# synaptic event; the event-driven form pays per element for its update (less with a class table) and an atomic per event.
# At the smallest sizes either form is a launch or two and its chains of dependent loads (600 neurons x 16: 7.0 us per step
# fused, 5.6 pushed; 3,001 x 12: 8.3 and 9.1; 1,500 x 8: 7.2 and 10.1).
FUSE_PS_PER_STEP = 5.05e6
PUSH_PS_PER_STEP = 4.5e6
FUSE_PS_PER_SYNAPSE = 1.35
FUSE_PS_PER_EVENT = 6.0
PUSH_PS_PER_ELEMENT = 55.0
PUSH_PS_PER_ELEMENT_CLASS_TABLE = 27.0
PUSH_PS_PER_EVENT = 48.0
# The form with resident trials pays a chain of dependent loads per launch and step, a visit per row that fired, little per event.
# Measured at 2 to 3 Hz in calls of 100 to 300 steps, us per step trials / fused / pushed (neurons x trials, in-degree): 51,978 x 32, 1154:
# 40 / 92 / 255; 20,011 x 20, 820: 8.3 / 31 / 55; 230,924 x 8, 335: 48 / 134 / 140; 5,000 x 16, 400: 2.8 / 10.0 / 21; 31,000 x 64, 160:
# 35 / 37 / 83; 60,000 x 64, 130: 70 / 65 / 145; 120,000 x 16, 150: 35 / 51 / 81; 115,000 x 20, 130: 46 / 57 / 91; 12,000 x 64, 130:
# 12.1 / 16.1 / 28; 100,000 x 4, 260: 7.3 / - / 28; 2,000 x 40, 200: 2.7 / 6.7 / 8.7; 3,000 x 4, 200: 2.5 / - / 7.0; 600 x 16, 100:
# 2.2 / - / 4.8; 400,123 x 1, 180: 6.6 / - / 22.  The constants were fitted with a grid barrier per trial and ask for up to a half
# more than lists take; at all of these sizes they pick the faster form still.  What they leave out: a call's own cost (state and
# ring in and out, its events put apart by trial: 31,000 x 64 in calls of 40 steps 59 us a step against 39 fused) and the detour of
# the per-step record (51,978 x 32 6 us a step, 31,000 x 64 7, against 2 and 4 in the fused form).
TRIALS_PS_PER_PASS = 3.0e6
TRIALS_PS_PER_ROW = 6.5e3       # per neuron of ONE trial that fires in a step (and the input events that come with it)
TRIALS_PS_PER_EVENT = 0.8
FUSE_PS_PER_ELEMENT = 10.0
FUSE_LDS_BYTES = 160 * 1024 - 512   # LDS of one workgroup of the fused batched driver (kFuseLdsMax of csrc/simulate_fused.hip)
FUSE_LDS_FIXED = 16 * (2 * NREC * 64 * 8 + 128 * 12)   # ... of it sums and stages (kFuseLdsFixed)
FUSE_BATCHES = range(8, 65)         # lane = trial, at most eight neurons to a wavefront
FUSE_PAD = 64                       # records behind its table (BMTK_FUSE_PAD)
RES_LDS_BYTES = 160 * 1024      # LDS of one gfx950 compute unit
RES_ACT_ENTRIES = 8192          # active-row list of the resident kernel (kActCap of csrc/resident.hip), 4 B each
LIST_MAX = 39                   # neurons of a workgroup's list (kListMax of csrc/fired_lists.hpp)
RES_LDS_EXTRA = RES_ACT_ENTRIES * 4 + 256   # the list plus the kernel's static LDS (rounded up)
# the single-workgroup form: per element the spike offsets and probed potentials of two steps (SOLO_LDS_PER_ELEMENT);
# the items (rows to walk) of two steps and its static LDS (SOLO_LDS_EXTRA)
SOLO_LDS_PER_ELEMENT = 4 * 4
SOLO_LDS_EXTRA = 10240 + 2048
RB_WIDE_SPAN = 1920             # neurons of a workgroup at most with two to a thread
# A launch of resident trials with two neurons to a thread against one.  Sums for the receptors in use only against all four sums of
# one: 51,978 x 32 1.46, 20,011 x 20 1.41, 100,000 x 4 1.52, 120,000 x 16 1.32 (spans of 1472 to 1728 / 832 to 960)
RB_TWO_COST = 1.35
RB_FEW_COST = 1.07              # one to a thread, sums for the receptors in use only (51,978 x 32 1.11, 20,011 x 20 1.07, 230,924 x 8 1.05, 10,000 x 8 1.08, 2,000 x 40 1.07)
# Two to a thread with sums as 32-bit whole numbers.  What counts is where few launches are saved, spans of 1408 to 1536 in the place of
# 1024: five launches to four 128,000 x 10 1.05, four to three 128,000 x 8 1.04, 50,000 x 20 1.16, 62,000 x 16 1.17, 32,000 x 32 1.20, 15,500 x 64 1.21.  Where half of
# them are saved, or more than a third, it may cost more: 51,978 x 32 1.18, 31,000 x 64 1.26, 230,924 x 8 and 20,011 x 20 1.33, 100,000 x 4 1.43, 120,000 x 16 1.51.
# They take less time in as many launches too, no conversion of each weight among other things: 200 steps with sums of 64 / 32 bits
# 5,000 x 16 630 / 614 us, 10,000 x 8 742 / 594, 31,000 x 8 1,091 / 902, 2,000 x 40 620 / 593, 60,000 x 4 1,163 / 975, 4,000 x 64 1,030 / 878; two to a thread 51,978 x 32 5,484 / 4,901, 20,011 x 20 1,212 / 1,060, 100,000 x 4 2,406 / 2,020, 31,000 x 64
# 6,239 / 5,363; in half the launches 230,924 x 8 5,376 / 3,401 (100 steps), 120,000 x 16 12,264 / 9,702
RB_TWO_COST_WHOLE = 1.22
RB_LIST_MIN, RB_LDS_STATIC = 2000, 256   # the form with resident trials: least room (words) for its lists of rows, static LDS
SUM_SHIFT_MAX = 120             # BMTK_SUM_SHIFT_MAX
TRIALS_TABLE_BYTES = 1 << 30    # tables and ring of the form with resident trials at most, or TRIALS_TABLE_RATIO times the synapses' 10 bytes
TRIALS_TABLE_RATIO = 4
TRIALS_MIN_STEPS = 32           # shorter calls are left to the launch-per-step drivers
TRIALS_SAVE_BYTES = 1 << 30     # scratch for the per-step record of a call at most: longer calls go in stretches
RECORD_WAYS = 64                # lists a large spike record is split into (bmtk_glif3_sim.spike_ways)


def resident_span(ne, batch, ring_slots, n_cu, single=True):
    """Elements per workgroup of the resident kernel for a network of ``ne`` elements on ``n_cu`` compute
    units, or 0 when the network does not fit: batch 1, one workgroup per compute unit (rounded down to a
    multiple of 8), at most 1024 elements each, and ring slice + active-row list + static LDS within the
    compute unit's LDS.  ``bmtk_glif3_simulate_fwd`` applies the same bound.  A network of up to 1024 elements
    goes to ONE workgroup when its whole ring fits (``single``): the library then runs the form without a grid
    barrier."""
    cus = n_cu - n_cu % 8
    if batch != 1 or cus <= 0 or ne <= 0:
        return 0
    if single and ne <= 1024:
        whole = -(-ne // 64) * 64
        if (ring_slots * NREC * 4 + SOLO_LDS_PER_ELEMENT) * whole + SOLO_LDS_EXTRA <= RES_LDS_BYTES:
            return whole
    span = -(-(-(-ne // cus)) // 64) * 64
    if span > 1024 or ring_slots * NREC * span * 4 + RES_LDS_EXTRA > RES_LDS_BYTES:
        return 0
    return span


def lists_pay(span, groups, rate_hz, h_ms=1.0):
    """Whether ``groups`` workgroups of ``span`` neurons that fire at ``rate_hz`` are expected to fit what they fire in a step into lists
    (of up to LIST_MAX neurons), which they then exchange in less time than ballots behind a grid barrier.  Measured on one MI355X,
    us per step lists / ballots, and the busiest workgroup of a step: 230,924 neurons at 21, 24, 28, 35, 46, 60 Hz 17.0 / 18.0 (34),
    18.4 / 17.2 (37), 26.3 / 22.4 (43), 29.0 / 23.1 (50), 36.5 / 38.4 (63), 45.4 / 47.0 (79); 120,000 at 45, 57, 71 Hz 15.2 / 15.7 (37),
    22.9 / 18.8 (44), 28.7 / 28.5 (53); 60,000 at 71, 92 Hz 13.0 / 14.2 (30), 17.5 / 17.4 (38); 3,000 at 91 Hz 4.0 / 5.2 (12)."""
    fired = span * float(rate_hz) * 1e-3 * h_ms
    # (the largest of so many Poisson numbers, a little above it)
    return fired + math.sqrt(2.0 * fired * math.log(max(2, groups))) <= LIST_MAX


def resident_trials_plan(n_neurons, batch, ring_slots, n_cu, third=None, sum_bytes=8):
    """How the trials of a batch share ``n_cu`` compute units when each keeps its state in registers and its arrivals of
    the next ring_slots - 1 steps in LDS: dict(span, groups, ways, passes, list, few) -- ``ways`` trials side by side on
    ``groups`` workgroups of ``span`` neurons each, ``passes`` launches, ``list`` places in the list of rows -- or None
    where a single trial does not fit.  ``third``: how many third and fourth receptors the neurons before the i-th use
    (n_neurons + 1 numbers; receptors that no synapse of a neuron ends on have no sums), or None where every neuron is to have all four.
    One trial: only where the network is too large for the resident mode, and with four sums in fp32.  ``sum_bytes`` 4: sums as 32-bit
    whole numbers (``whole_numbers``), four to a neuron.

    A step costs much the same whatever runs beside it: as few launches as possible, if need be with sums only for what is in use
    (``few``) and two neurons to a thread (spans above 1024), which take RB_TWO_COST times as long a step."""
    cus, slots = n_cu - n_cu % 8, ring_slots - 1
    if not 1 <= batch <= 64 or cus <= 0 or n_neurons <= 0 or slots < 1:
        return None

    def places(span, few=False):
        """Words of LDS beside the sums of so many neurons."""
        extra = 2 * span
        if few:
            first = np.arange(0, n_neurons, span)
            extra = int((third[np.minimum(first + span, n_neurons)] - third[first]).max())
        return (RES_LDS_BYTES - RB_LDS_STATIC - slots * (2 * span + extra) * (4 if batch == 1 else sum_bytes)) // 4

    def plan(span, ways, passes, few=False):
        return dict(span=span, groups=-(-n_neurons // span), ways=ways, passes=passes, list=min(RES_ACT_ENTRIES, places(span, few)), few=few)

    if batch == 1:
        # one trial of more neurons than the compute units have threads: two to a thread, sums in fp32
        span = -(-(-(-n_neurons // cus)) // 64) * 64
        return plan(span, 1, 1) if 1024 < span <= RB_WIDE_SPAN and places(span) >= RB_LIST_MIN else None
    best, best_cost = None, None
    # (of equals the first)
    kinds = (((False, 1024, 1.0), (False, RB_WIDE_SPAN, RB_TWO_COST_WHOLE)) if sum_bytes == 4 else
             ((False, 1024, 1.0), (True, 1024, RB_FEW_COST), (True, RB_WIDE_SPAN, RB_TWO_COST))[:1 if third is None else 3])
    for few, most, cost in kinds:
        most = next((span for span in range(most, 0, -64) if places(span, few) >= RB_LIST_MIN), 0)
        if not most or -(-n_neurons // most) > cus:
            continue
        passes = -(-batch // min(batch, cus // -(-n_neurons // most)))
        ways = -(-batch // passes)
        span = -(-(-(-n_neurons // (cus // ways))) // 64) * 64
        if places(span, few) < RB_LIST_MIN:      # (sums dealt out unevenly)
            span = most
        if best is None or passes * cost < best_cost:
            best, best_cost = plan(span, ways, passes, few), passes * cost
    return best


def plan_cost(plan):
    """What the launches of a plan come to, in steps with a neuron to a thread."""
    return plan["passes"] * (1.0 if plan["span"] <= 1024 else RB_TWO_COST if plan.get("few") else RB_TWO_COST_WHOLE)


def fixed_point_shift(tables, n_neurons):
    """How far weights have to be scaled up, as a power of two, for 64-bit fixed point with a lowest bit of 2^-32 to hold every
    one of them exactly, so that no sum has fewer bits than one in fp32: 0 where each weight is a whole multiple of 2^-32 (any
    fp32 number from 2^-9 on is).  None where they do not fit: what could reach a neuron in a step, scaled, has to stay below
    2^30 (a factor of two for ids repeated within a step), and weights have to be finite."""
    tables = [t for t in tables if t.nnz]
    lowest, sizes = 0, []
    for t in tables:
        size = t.weights.abs()
        least, largest = torch.stack(torch.aminmax(size)).tolist()      # (a NaN carries over)
        if not math.isfinite(largest):
            return None
        sizes.append(largest)
        # (from 2^-9 on every number's bits lie above 2^-33)
        for w in size.split(1 << 26) if least < 2.0 ** -9 else ():
            # the power of two that a weight's lowest set bit stands for
            bits = w.contiguous().view(torch.int32)
            exponent, mantissa = bits >> 23, bits & 0x7FFFFF
            mantissa = torch.where(exponent > 0, mantissa | 0x800000, mantissa)
            low_bit = ((mantissa & -mantissa).to(torch.float32).view(torch.int32) >> 23) - 127
            place = torch.where(mantissa != 0, exponent.clamp(min=1) - 150 + low_bit, torch.zeros_like(low_bit))
            lowest = min(lowest, int(place.min()))
    shift = max(0, -32 - lowest)
    if shift > SUM_SHIFT_MAX:
        return None
    limit = 2.0 ** (30 - shift)
    # (all synapses on one neuron; only where that is too much, the synapses of the neuron that has most)
    if (sum(size * t.nnz for size, t in zip(sizes, tables)) >= limit
            and sum(size * int(torch.bincount(t.indices, minlength=n_neurons).max()) for size, t in zip(sizes, tables)) >= limit):
        return None
    return shift


def whole_numbers(rec, inp, n_neurons):
    """Whether the sums of arrivals fit 32-bit whole numbers of a power of two that every weight is a multiple of: (k, how often a step may
    repeat an input id, mark by which the weights are known again) for multiples of 2^-k pA, or None.  A synapse has one delay, so what it brings to a sum comes from the
    events of one step: all synapses of a neuron once, and those of the inputs once more for every time that a step may repeat their id, have
    to come to less than half of what 32 bits hold (the other half is for arrivals under way where ``step`` is set back)."""
    lib, tables = _lib.load(), [t for t in (inp, rec) if t is not None and t.nnz]
    if not tables:
        return 0, 1 << 30, 0
    dev = tables[0].weights.device
    reach, found = torch.zeros(n_neurons, dtype=torch.int64, device=dev), torch.zeros(2, dtype=torch.int64, device=dev)
    of_inputs, mark = found.new_zeros(1), found[1:]     # (the first word: two of 32 bits)
    for t in tables:      # (the inputs first, so that what they come to is known by itself)
        _lib.check(lib.bmtk_csr_weight_reach(t.nnz, _p(t.indices), _p(t.weights), _p(reach), _p(found), _p(mark), _stream()))
        if t is inp:
            of_inputs = reach.max().view(1)
    both, mark, of_inputs, most = torch.cat([found, of_inputs, reach.max().view(1)]).tolist()     # (one look at the device)
    lowest, largest = np.array([both]).view(np.int32).tolist()
    k, of_inputs, most = -lowest, of_inputs / 1024.0, most / 1024.0
    left = 2.0 ** 30 - most * 2.0 ** k
    if largest >= 0x4E800000 or k > 30 or left <= 0.0:      # (2^30 as a float's bits)
        return None
    return k, math.ceil(left / max(1.0, of_inputs * 2.0 ** k)) - 1, mark


def fused_pays(n_neurons, batch, n_synapses, class_table, rate_hz, h_ms=1.0):
    """Whether the fused pull form of the batched driver is expected to take less time per step than pushing the
    spikes as events, for a network of ``n_neurons`` with ``n_synapses`` recurrent and input synapses at ``batch``
    trials and a mean rate of ``rate_hz``."""
    if n_synapses <= 0:
        return False
    events = n_synapses * batch * float(rate_hz) * 1e-3 * h_ms
    row = n_synapses / float(n_neurons)
    blocks_full = row / (256.0 * math.ceil(row / 256.0))
    fused = FUSE_PS_PER_STEP + FUSE_PS_PER_SYNAPSE * n_synapses / blocks_full + FUSE_PS_PER_EVENT * events
    push = ((PUSH_PS_PER_ELEMENT_CLASS_TABLE if class_table else PUSH_PS_PER_ELEMENT) * n_neurons * batch
            + PUSH_PS_PER_EVENT * events + PUSH_PS_PER_STEP)
    return fused < push


def trials_bytes(plan, n_neurons, batch, ring_slots, n_inputs, n_synapses):
    """Device memory that the form with resident trials takes beside the synapse tables: bounds of every workgroup's segment of
    every row, packed records, the ring behind a call."""
    return ((n_neurons + n_inputs) * (plan["groups"] + 1) * 4 + n_synapses * 8 + n_neurons * 4
            + batch * (ring_slots - 1) * NREC * n_neurons * (8 if batch > 1 else 4))


def trials_fit(plan, n_neurons, batch, ring_slots, n_inputs, n_synapses):
    """Whether that memory is in proportion to the synapses'.  With many sources of few synapses (millions of virtual cells) the bounds
    alone, a thousand bytes a source, would be many times the network; the other drivers need none."""
    return (trials_bytes(plan, n_neurons, batch, ring_slots, n_inputs, n_synapses)
            <= max(TRIALS_TABLE_BYTES, TRIALS_TABLE_RATIO * 10 * n_synapses))


def trials_pay(plan, n_neurons, batch, n_synapses, class_table, rate_hz, h_ms, fused):
    """Whether the form with resident trials (``plan``: resident_trials_plan) is expected to take less time per step than
    the driver that would run otherwise, the fused pull form (``fused``) or pushed events."""
    per_trial = n_neurons * float(rate_hz) * 1e-3 * h_ms
    events = n_synapses * batch * float(rate_hz) * 1e-3 * h_ms
    step = TRIALS_PS_PER_PASS + TRIALS_PS_PER_ROW * per_trial
    trials = (plan_cost(plan) if batch > 1 else plan["passes"]) * step + TRIALS_PS_PER_EVENT * events
    if fused:
        other = (FUSE_PS_PER_STEP + FUSE_PS_PER_SYNAPSE * n_synapses + FUSE_PS_PER_EVENT * events
                 + FUSE_PS_PER_ELEMENT * n_neurons * batch)
    else:
        other = ((PUSH_PS_PER_ELEMENT_CLASS_TABLE if class_table else PUSH_PS_PER_ELEMENT) * n_neurons * batch
                 + PUSH_PS_PER_EVENT * events + PUSH_PS_PER_STEP)
    return trials < other


class Glif3Simulator:
    """A population of GLIF3 neurons with recurrent and external synapses.

    par         fp64 [NPARAM, columns] NEST-unit parameters; one column per
                neuron, or per parameter class when ``class_id`` is given
    rec, inp    source-major synapse tables (numpy tuples, see bmtk_amd.network):
                recurrent (rows = neurons) and external (rows = input sources)
    ring_slots  slots of the delay ring buffer; default = largest (residual) delay + 1
    resident    "auto": every ``run`` is one cooperative launch that keeps the state in registers and the ring in
                LDS (the resident kernel) whenever the network fits it -- batch 1, at most 1024 elements per
                compute unit, ring slice within LDS; True: insist on it (ValueError otherwise); False: one launch
                per step, which takes any batch and size (``resident_trials`` then has to be asked for)
    single_workgroup  resident mode: a network of up to 1024 elements whose whole ring fits LDS runs in ONE
                workgroup, without a grid barrier (about 1 us per step instead of 2.5, a third of that where no delay is below some ten
                steps, which it then runs several of between two barriers); False keeps such a network
                on the many-workgroup form
    fired_lists  resident mode with several workgroups: every workgroup publishes the neurons that fired in a step
                as a short list whose words carry the step, and nobody waits at a grid barrier (neurons that a list does
                not hold are read from the ballots), unless at ``expected_rate_hz`` lists would seldom do (``lists_pay``);
                False: ballots behind a grid barrier.  Same results either way.
    expected_rate_hz  what ``fired_lists`` goes by, and "auto" decides ``pull`` / ``fused`` by.  Pushing spikes into the ring costs an atomic per
                synaptic event, pulling a pass over the whole table per step whatever the activity; a synapse
                carries batch * rate * h events per step, and on one MI355X the pass is the cheaper of the two from
                about 0.06 events per synapse and step (measured: 51,978 neurons x 32 trials at 3.2 Hz pull 168 us
                against 340 pushed; 230,924 neurons x 8 and x 16 at 2.8 Hz pushed 132 / 237 us against 321 / 358
                pulled).  Default 3 Hz: batches from 20 at 1 ms steps.  That mark decides the unfused ``pull``;
                ``fused`` is decided by ``fused_pays``, which compares the fitted cost of a step in either form.
    fused       launch-per-step mode, batches of 8 to 64, delay_offset 0: one launch per two steps in which a
                wavefront sums what arrives at a neuron -- over recurrent and input synapses, from a joint
                target-major table and a joint history of spike and input-event bits -- and advances the neuron's
                trials, lane = trial; no arrival sum passes through device memory.  "auto": when ``fused_pays``
                says a step costs less this way than pushed as events (the update's share grows with the batch,
                the table pass does not: 51,978 neurons x 60 M synapses from batch 16 on at any rate, at batch 8
                from about 3.3 Hz); takes any number of sources (above what the activity map in
                LDS holds, one bit of the map stands for 2, 4, ... sources).  False: the pull form as separate
                launches (below).  ``ring`` then holds only the few input ids repeated within a step.
    pull        launch-per-step mode only: sum the recurrent arrivals of a step in one pass over a target-major
                copy of the table from the spike-bit history, instead of pushing them into the ring with global
                atomics as spikes occur -- the faster form for batched runs.  "auto": by ``expected_rate_hz``
                (and delay_offset 0, network small enough for the activity map in LDS).  Recurrent arrivals still ahead at the end
                of a run then live in the history, and ``ring`` holds the input arrivals only.
    resident_trials  batches of 2 to 64, or one trial of more neurons than ``resident`` holds (1024 to a compute unit; here up
                to 1920), with a recurrent table and delay_offset 0: trials side by side, each with its state
                in registers and its ring in LDS for the length of a call, as many at a time as the compute units hold
                (``resident_trials_plan``).  "auto": where resident, fused and pull are "auto" too, the network fits,
                ``trials_pay`` says so and its tables are in proportion to the network (``trials_fit``); where there turns out to be no
                memory for them the other driver runs.  Such a simulator also holds the driver it would have without; a call that asks
                for more than spike bits and, of a batch, the per-step record (``record_cap``, probes; ``save_state`` of a single
                trial or of so many elements that 32 steps of them outgrow TRIALS_SAVE_BYTES), covers fewer than TRIALS_MIN_STEPS
                steps or is captured into a graph, and a look at ``ring``, ``work_bits`` or ``fuse_any``, make it go on with that
                driver for good.  True: insist (ValueError otherwise); False: off.  Sums of a batch's arrivals have 64 bits, or 32 where the
                weights are whole multiples of one power of two that those hold exactly (``whole_numbers``); a call whose
                input events repeat an id in a step more often than these have room for makes it go on with 64-bit sums, or with the
                other driver where those do not fit or pay.
    delay_offset  B steps taken off every delay before the tables are built; spikes and input events are
                then handed to the tables B steps late from a history of spike bits, which gives the same
                arrivals with a ring B slots shorter.  "auto": 0 while the largest delay is at most 63
                steps (what the ring and the packed tables hold), else the smallest delay minus one --
                the case of NEST networks run at a fine resolution (1-2 ms delays at 0.001-0.1 ms steps).
                Also the smallest delay minus one when that is what lets a network of up to 1024 neurons keep its
                whole ring in ONE workgroup's LDS (the resident form without a grid barrier).
                The delay columns may then be any integer type; residual delays must stay within 63.
    """

    def __init__(self, n_neurons, par, h, batch=1, class_id=None, rec=None, inp=None, ring_slots=None,
                 asc_init=None, u_init=None, i_ext=None, device=None, resident="auto", delay_offset="auto",
                 pull="auto", single_workgroup=True, fired_lists=True, fused="auto", fuse_wg_per_cu=0,
                 expected_rate_hz=3.0, resident_trials="auto"):
        self.lib = _lib.load()
        self.dev = device or _dev()
        self.n, self.batch, self.h = int(n_neurons), int(batch), float(h)
        self.ne = self.n * self.batch
        if self.ne >= 2 ** 31:
            raise ValueError("n_neurons*batch must stay below 2^31")
        par = np.ascontiguousarray(par, np.float64)
        if par.shape[0] != NPARAM:
            raise ValueError("par must be [{}, columns]".format(NPARAM))
        if class_id is not None:
            class_id = np.ascontiguousarray(class_id, np.int32)
            if class_id.size != self.n or class_id.min() < 0 or class_id.max() >= par.shape[1]:
                raise ValueError("class_id must map every neuron to a column of par")
        elif par.shape[1] != self.n:
            raise ValueError("par needs one column per neuron when class_id is not given")
        self.prop = glif3_precompute(par, h)
        self.class_id = None if class_id is None else torch.as_tensor(class_id, device=self.dev)
        ends = [x for t in (rec, inp) if t is not None and len(t[3])
                for x in (torch.aminmax(t[3]) if torch.is_tensor(t[3]) else (t[3].min(), t[3].max()))]
        if ends and all(torch.is_tensor(x) for x in ends):
            ends = torch.stack([x.long() for x in ends]).tolist()      # (one look at the device)
        ends = [int(x) for x in ends]
        min_delay, max_delay = (min(ends[::2]), max(ends[1::2])) if ends else (1, 1)
        if min_delay < 1:
            raise ValueError("delays must be at least one step")
        if delay_offset == "auto":
            delay_offset = 0 if max_delay <= 63 else min_delay - 1
            if (delay_offset == 0 and min_delay > 1 and resident and single_workgroup and self.batch == 1
                    and self.n <= 1024 and not ring_slots):
                # a small network whose whole ring only fits ONE workgroup's LDS (the form without a grid barrier)
                # once the part all delays have in common is taken off: bmtk's example networks at dt = 0.1 ms
                # (every delay 2 ms: 21 ring slots for 450 cells are 172 KB, 2 slots 16 KB)
                whole = -(-self.n // 64) * 64

                def fits(slots):
                    return (slots * NREC * 4 + SOLO_LDS_PER_ELEMENT) * whole + SOLO_LDS_EXTRA <= RES_LDS_BYTES
                if not fits(max_delay + 1) and fits(max_delay - min_delay + 2):
                    delay_offset = min_delay - 1
        self.delay_offset = int(delay_offset)
        if not 0 <= self.delay_offset < min_delay:
            raise ValueError("delay_offset must lie in 0..smallest delay - 1")
        # residual delays beyond 63 steps: a wider delay field and a longer ring, which only the launch-per-step
        # driver (without the pull form) handles
        residual = max_delay - self.delay_offset
        self.delay_bits = 6 if residual <= 63 else max(7, int(residual).bit_length())
        if self.delay_bits > 6:
            ring_bytes = (residual + 1) * NREC * self.ne * 4
            if (self.delay_bits > 14 or self.n >= 2 ** (30 - self.delay_bits) or ring_bytes > 8 << 30
                    or resident is True or pull is True):
                raise ValueError("delays span {}..{} steps: after taking off {} the largest still exceeds the 63 steps "
                                 "the ring buffer of the resident and pull forms holds, or what the wide form takes "
                                 "({} ring bytes, {} neurons)".format(min_delay, max_delay, self.delay_offset,
                                                                      ring_bytes, self.n))
            resident = pull = False
        wide = self.delay_bits > 6

        def narrow(t):
            return t is None or t[3].dtype == (torch.uint8 if torch.is_tensor(t[3]) else np.uint8)

        if self.delay_offset or wide or not (narrow(rec) and narrow(inp)):
            def shorten(t):
                if t is None:
                    return None
                d = t[3] - self.delay_offset
                if torch.is_tensor(d):
                    d = d.to(torch.int32 if wide else torch.uint8)
                else:
                    d = d.astype(np.int32 if wide else np.uint8)
                return (t[0], t[1], t[2], d, t[4])
            rec, inp = shorten(rec), shorten(inp)
        self.least_delay = min_delay - self.delay_offset    # ... of the tables' records
        self.L = int(ring_slots) if ring_slots else max_delay - self.delay_offset + 1
        self.rec = self._table(rec, self.n) if rec is not None else None
        self.inp = self._table(inp, None) if inp is not None else None
        for t in (self.rec, self.inp):
            if t is not None:
                t.delay_bits = self.delay_bits
        self.n_inputs = self.inp.n_rows if self.inp is not None else 0
        # A table without a synapse delivers nothing and its arrays have no address to hand over: the kernels are
        # not given it.  Events of input sources that project nowhere are still accepted (and checked).
        if self.rec is not None and self.rec.nnz == 0:
            self.rec = None
        self.inp_without_synapses = self.inp is not None and self.inp.nnz == 0
        if self.inp_without_synapses:
            self.inp = None
        self.state = Glif3State.zeros(self.n, self.batch, asc_init=asc_init, u_init=u_init, device=self.dev)
        self._trials = None     # the form with resident trials (_setup_trials), while it is in use
        self._ring = torch.zeros(self.L, NREC, self.ne, device=self.dev)
        self.i_ext = None if i_ext is None else torch.as_tensor(np.asarray(i_ext, np.float32), device=self.dev)
        if self.i_ext is not None and self.i_ext.numel() != self.ne:
            raise ValueError("i_ext needs one entry per element")
        self.in_ptr = self.in_events = None
        self.in_steps = 0
        self.in_duplicates = False
        self.in_most_repeats, self.in_repeats_of_one = 0, None   # how often one id is repeated in any step, and in each
        self._lists_replaced = False    # since the last run
        self.in_repeat_ptr = self.in_repeat_events = None   # repeated ids of a step, for the pull form of the inputs
        self.step = 0
        self.words = n_words(self.ne)
        # history of spike bits: 2B+3 rows let resident workgroups drift B steps apart, one more lets them look
        # at the grid barrier only where the spikes behind it are needed; B+3 is the least
        self.hist_slots = 2 * self.delay_offset + 4
        if self.hist_slots * (self.words + 1) * 8 > 2 ** 30:
            self.hist_slots = self.delay_offset + 3
        self._work_bits = torch.zeros(self.hist_slots * (self.words + 1), dtype=torch.int64, device=self.dev)
        if self.n >= 2 ** 24:
            raise ValueError("the packed synapse tables index at most 2^24 neurons")
        self.res_sync = torch.zeros(_lib.RES_SYNC_WORDS, dtype=torch.int32, device=self.dev)
        self.res_span = self.res_groups = 0
        self.rec_seg = self.inp_seg = self.res_unified = self.res_fired = None
        self._pending_check = False
        self.probe_ids = self.probe_col = None
        self.probe_every = 1
        self.spin_limit = 0  # resident mode: polls of the grid barrier before giving up (0 = built-in limit)
        self.single_workgroup = bool(single_workgroup)
        self.fired_lists = bool(fired_lists)
        self.expected_rate_hz = float(expected_rate_hz)
        if resident:
            self._setup_resident(required=(resident is True))
        self.pull_table = self.pull_syn = self.pull_work = None
        self.pull_inp_table = self.pull_inp_syn = self.pull_inp_work = self.in_hist = None
        self.fuse_table = self._fuse_any = None
        self.sum_shift = 0      # power of two that the weights of the tables summed in fixed point are scaled by
        self.fuse_wg_per_cu = int(fuse_wg_per_cu)
        can_fuse = ((self.rec is not None or self.inp is not None) and not self.res_span and self.delay_offset == 0
                    and self.delay_bits == 6 and self.batch in FUSE_BATCHES and pull is not False)
        if fused is True and not can_fuse:
            raise ValueError("the fused form needs a synapse table, launch-per-step mode, delay_offset 0, delays "
                             "within 63 steps and a batch of 8 to 64")
        can_pull = (self.rec is not None and not self.res_span and self.delay_offset == 0
                    and self.L * ((self.n + 31) // 32) * 4 <= PULL_MAP_BYTES)
        # the pull form sums in 64-bit fixed point: weights must be finite and below 2^31 in size
        def fixed_point_ok(t):
            w = t.weights
            return not w.numel() or bool(torch.isfinite(w).all() & (w.abs().max() < 2.0 ** 31))
        # events per synapse and step at the expected rate: from PULL_MIN_DENSITY on a pass over the table is cheaper
        dense = self.batch * float(expected_rate_hz) * 1e-3 * self.h >= PULL_MIN_DENSITY
        if can_pull and (pull is True or (pull == "auto" and dense)):
            if not (fixed_point_ok(self.rec) and (self.inp is None or fixed_point_ok(self.inp))):
                if pull is True:
                    raise ValueError("the pull form needs finite weights smaller than 2^31 in size")
                can_pull = False   # the event-driven form propagates IEEE values as they are
        if pull is True and not can_pull:
            raise ValueError("the pull form needs a recurrent table, launch-per-step mode, delay_offset 0 and "
                             "ring_slots * n_neurons / 8 bytes of LDS (at most 40 KB)")
        # What separate launches would have pulled: their history of input events is read from the lists step by step, a
        # call's first step the one before it once more.  The fused form does the same where it takes their place (at
        # batches that do not divide 64), so that lists replaced between two calls mean what they meant there.
        pulls = can_pull and (pull is True or (pull == "auto" and dense))
        inp_pulls = self.inp is not None and self.L * ((self.n_inputs + 31) // 32) * 4 <= PULL_MAP_BYTES
        self.fuse_rereads = pulls and 64 % self.batch != 0 and inp_pulls
        n_syn = sum(t.nnz for t in (self.rec, self.inp) if t is not None)
        if can_fuse and fused and (fused is True or pull is True or
                                   fused_pays(self.n, self.batch, n_syn, self.class_id is not None, expected_rate_hz, self.h)):
            tables = [t for t in (self.rec, self.inp) if t is not None]
            if all(fixed_point_ok(t) for t in tables):
                # Whatever its batches (or separate pull launches in their place) hold in fixed point stays there; where
                # events would be pushed, as fp32, the sums have to be as good.
                shift = fixed_point_shift(tables, self.n)
                if fused is True or shift is not None or 64 % self.batch == 0 or (pulls and (self.inp is None or inp_pulls)):
                    self.sum_shift = shift or 0
                    self._setup_fused()
            elif fused is True:
                raise ValueError("the fused form needs finite weights smaller than 2^31 in size")
        if self.fuse_table is not None:
            pass
        elif pulls:
            self.pull_table = self.rec.transposed(self.n)
            self.pull_syn = torch.zeros(NREC, self.ne, device=self.dev)
            need = self.lib.bmtk_csr_propagate_pull_workspace_bytes(self.L, self.n)
            self.pull_work = torch.zeros(need // 4 + 1, dtype=torch.int32, device=self.dev)
            # the history must hold one row per ring slot, row t % L = spikes of step t
            self.hist_slots = self.L
            self._work_bits = torch.zeros(self.hist_slots * (self.words + 1), dtype=torch.int64, device=self.dev)
            if inp_pulls:
                self.pull_inp_table = self.inp.transposed(self.n)
                self.pull_inp_syn = torch.zeros(NREC, self.ne, device=self.dev)
                need = self.lib.bmtk_csr_propagate_pull_workspace_bytes(self.L, self.n_inputs)
                self.pull_inp_work = torch.zeros(need // 4 + 1, dtype=torch.int32, device=self.dev)
                self.in_hist_stride = n_words(self.n_inputs * self.batch) + 1
                self.in_hist = torch.zeros(self.L * self.in_hist_stride, dtype=torch.int64, device=self.dev)
        self._trials_left, self._pend_from, self._pend_until, self._left_ring, self._kept = False, 0, 0, None, []
        if resident_trials == "auto":
            # (resident=False asks for the launch-per-step drivers, of a batch too)
            wanted = resident == "auto" and fused == "auto" and pull == "auto" and self.pull_table is None
        else:
            wanted = bool(resident_trials)
        plan = used = None
        if wanted and self.rec is not None and not self.res_span and self.delay_offset == 0 and self.delay_bits == 6:
            n_cu = torch.cuda.get_device_properties(self.dev).multi_processor_count
            # (of a batch: what it takes at best, before the tables are looked at)
            plan = resident_trials_plan(self.n, self.batch, self.L, n_cu, np.zeros(self.n + 1, np.int64) if self.batch > 1 else None)
            # 32-bit sums where the weights allow them: 3 to 25 % faster in as many launches (see RB_TWO_COST_WHOLE)
            small = resident_trials_plan(self.n, self.batch, self.L, n_cu, None, 4) if self.batch > 1 else None
            whole = whole_numbers(self.rec, self.inp, self.n) if small and (plan is None or plan_cost(small) <= plan_cost(plan)) else None
            if whole:
                plan = dict(small, whole=whole[0] + 1, room=whole[1], mark=whole[2])
            elif plan and self.batch > 1:
                plan, used = self._fixed_point_plan()
        if plan and not self._trials_possible(plan, resident_trials != "auto"):
            plan = None
        if plan and self.batch > 1 and self.fuse_table is None:     # (one trial: sums in fp32; the fused form: as good as its own)
            shift = fixed_point_shift([t for t in (self.rec, self.inp) if t is not None], self.n)
            if shift is None and not (resident_trials is True and self._trials_weights_ok(fixed_point_ok)):
                plan = None
            self.sum_shift = shift or 0
        if resident_trials is True and plan is None:
            raise ValueError("resident trials need a recurrent table, a batch of 2 to 64 (or more neurons than the resident mode holds), delay_offset 0, no pull table, weights "
                             "that 64-bit fixed point holds and a network whose trial fits the compute units")
        if plan:
            self._trials = dict(plan, seg=None, insisted=resident_trials is True, used=used)

    def _fixed_point_plan(self):
        """The plan of a batch with 64-bit sums, and the receptors in use that it was made from."""
        used = self._receptors_used()
        third = torch.zeros(self.n + 1, dtype=torch.int64, device=self.dev)
        torch.cumsum(self._third_and_fourth(used), 0, out=third[1:])
        n_cu = torch.cuda.get_device_properties(self.dev).multi_processor_count
        return resident_trials_plan(self.n, self.batch, self.L, n_cu, third.cpu().numpy()), used

    def _trials_possible(self, plan, insisted):
        """Whether the tables of a plan can be had and, unless it is asked for, whether it is expected to pay."""
        n_syn = sum(t.nnz for t in (self.rec, self.inp) if t is not None)
        if ((self.n + self.n_inputs) * (plan["groups"] + 1) >= 2 ** 32 or self.n + self.n_inputs >= 2 ** 24
                or n_syn >= 2 ** 31 or self.pull_table is not None):
            return False
        return insisted or (trials_pay(plan, self.n, self.batch, n_syn, self.class_id is not None, self.expected_rate_hz, self.h,
                                       self.fuse_table is not None)
                            and trials_fit(plan, self.n, self.batch, self.L, self.n_inputs, n_syn))

    def _trials_weights_ok(self, fixed_point_ok):
        """Whether weights that 64-bit fixed point does not all hold exactly are good enough for a caller who insists on the form
        with resident trials: large against 2^-32 on average, a neuron's all together small against 2^31."""
        tables = [t for t in (self.rec, self.inp) if t is not None]
        if not all(fixed_point_ok(t) for t in tables):
            return False
        size = sum(t.weights.abs().sum(dtype=torch.float64) for t in tables) / max(1, sum(t.nnz for t in tables))
        most = sum(t.weights.abs().max().double() * torch.bincount(t.indices, minlength=self.n).max() for t in tables if t.nnz)
        return bool((size >= 2.0 ** -8) & (most < 2.0 ** 30))

    def _receptors_used(self):
        """Which receptors some synapse of a neuron ends on, a bit each."""
        used = torch.zeros(self.n, dtype=torch.int32, device=self.dev)
        for t in (self.rec, self.inp):
            if t is not None:
                _lib.check(self.lib.bmtk_csr_receptors_used(t.nnz, _p(t.indices), _p(t.receptors), _p(used), _stream()))
        return used

    @staticmethod
    def _third_and_fourth(used):
        return (sum((used >> r) & 1 for r in range(NREC)) - 2).clamp_(min=0)

    def _setup_trials(self):
        """Tables and buffers of the form with resident trials: recurrent and input rows as one table sorted by target,
        the bounds of every workgroup's segment of every row, the ring behind a call and the ballot history.  False where they cannot be
        had any more: 32-bit sums, weights that somebody has written to since these were chosen, and no room for 64-bit ones."""
        tr, n = self._trials, self.n
        groups = tr["groups"]
        seg = torch.empty(n + self.n_inputs, groups + 1, dtype=torch.int32, device=self.dev)
        packed = torch.empty(self.rec.nnz + (self.inp.nnz if self.inp is not None else 0), 2, dtype=torch.int32, device=self.dev)
        row = at = 0
        for t in (self.rec, self.inp):
            if t is None:
                continue
            own = seg[row:row + t.n_rows]
            try:
                t.segment_offsets(tr["span"], groups, out=own)
            except ValueError:
                t = t.sorted_by_index()
                t.segment_offsets(tr["span"], groups, out=own)
            own += at                                   # (fewer than 2^31 synapses)
            packed[at:at + t.nnz] = t.packed()[:t.nnz]
            row, at = row + t.n_rows, at + t.nnz
        if tr.get("ring") is None:
            tr["ring"] = torch.zeros(self.batch, self.L - 1, NREC, n, device=self.dev, dtype=torch.int64 if self.batch > 1 else torch.float32)
        tr["whole"] = 0 if tr.get("few") else tr.get("whole", 0)
        mark = None
        if tr["whole"]:
            mark = torch.zeros(1, dtype=torch.int64, device=self.dev)
            _lib.check(self.lib.bmtk_csr_pack_whole(at, tr["whole"] - 1, _p(packed), _p(mark), _stream()))
        elif self.sum_shift:
            packed.view(torch.float32)[:, 1] *= 2.0 ** self.sum_shift
        cells, extra = None, 2 * tr["span"]
        if tr.get("few"):           # where a neuron's third sum stands among its workgroup's
            if tr["used"] is None:
                tr["used"] = self._receptors_used()
            own = self._third_and_fourth(tr["used"])
            before = torch.cumsum(own, 0) - own
            begin = torch.arange(groups, device=self.dev) * tr["span"]
            before -= before[begin].repeat_interleave(tr["span"])[:n]
            cells, extra = (tr["used"] | before << NREC).to(torch.int32), int((before + own).max())
        _lib.check(self.lib.bmtk_csr_pack_cells(at, tr["span"], _p(cells), _p(packed), _stream()))
        # lanes to a segment at most: about as many as it holds synapses on average
        segment = int(math.ceil(math.log2(max(1.0, at / float(max(1, row)) / groups))))
        tr.update(seg=seg, packed=packed, cells=cells, extra=extra, max_team_shift=min(6, segment),
                  hist=torch.zeros(tr["ways"], 4, n_words(n) + 1, dtype=torch.int64, device=self.dev))
        if mark is not None and int(mark) != tr["mark"]:     # (looked at with all else under way)
            self._trials_in_fixed_point()
            return not self._trials.get("whole") and self._setup_trials()
        return True

    def _trials_run(self, s, n_steps):
        """Fill ``s`` for a call in the form with resident trials.  Returns what has to live until it is launched."""
        tr = self._trials
        s.rb_span, s.rb_groups, s.rb_ways, s.rb_list = tr["span"], tr["groups"], tr["ways"], tr["list"]
        # as many lanes to a segment as let the workgroup's 896 that pull take the rows of a step in one go (51,978 x 32, 243 rows
        # of 18 synapses: 47 / 40 / 42 us per step with 1 / 2 / 4 lanes; 20,011 x 20, 85 of 33: 10.6 / 9.3 / 9.5 with 4 / 8 / 16;
        # 230,924 x 8, 780 rows of 1.4: one)
        events = self.in_events.numel() / float(max(1, self.in_steps) * self.batch) if self.in_ptr is not None else 0.0
        rows = max(1.0, self.n * self.expected_rate_hz * 1e-3 * self.h + events)
        s.rb_team_shift = max(0, min(tr["max_team_shift"], int(math.log2(max(1.0, 900.0 / rows)))))
        s.rb_late_events = 1 if self.fuse_rereads else 0
        s.rb_cells, s.rb_extra, s.rb_whole = _p(tr["cells"]), tr["extra"], tr["whole"]
        s.rb_seg, s.rb_packed, s.rb_ring, s.rb_hist = _p(tr["seg"]), _p(tr["packed"]), _p(tr["ring"]), _p(tr["hist"])
        s.res_sync, s.res_spin_limit = _p(self.res_sync), int(self.spin_limit)
        if self.inp is None or self.in_ptr is None:
            return None
        # the events of the steps step - 1 .. step + n_steps - 1, apart by trial
        args = (self.batch, self.step - 1, n_steps + 1, s.rb_late_events, _p(self.in_ptr), _p(self.in_events))
        counts = torch.empty(self.batch * (n_steps + 1), dtype=torch.int32, device=self.dev)
        _lib.check(self.lib.bmtk_events_by_trial(*args, _p(counts), None, None, _stream()))
        first = torch.zeros(counts.numel() + 1, dtype=torch.int64, device=self.dev)
        torch.cumsum(counts, 0, out=first[1:])
        sources = torch.empty_like(self.in_events)
        _lib.check(self.lib.bmtk_events_by_trial(*args, None, _p(first), _p(sources), _stream()))
        s.rb_in_ptr, s.rb_in_events = _p(first), _p(sources)
        return first, sources

    def _run_trials(self, n_steps, stretch, bits, saved):
        """A call in the form with resident trials, ``stretch`` steps at a time.  False, and nothing done, if that was the
        constructor's choice and there is no memory for it, or its tables cannot be had any more."""
        scratch = {}
        try:
            if self._trials["seg"] is None and not self._setup_trials():
                return False
            if saved is not None:
                scratch = dict(v=torch.empty(stretch * self.ne, device=self.dev),
                               flags=torch.empty(stretch * self.ne, dtype=torch.uint8, device=self.dev))
        except torch.OutOfMemoryError:
            if self._trials["insisted"]:
                raise
            return False
        for k in range(0, n_steps, stretch):
            steps = min(stretch, n_steps - k)
            s = self._struct(None if bits is None else bits[k:k + steps])
            lists = self._trials_run(s, steps)
            if saved is not None:
                s.save_v, s.save_flags = _p(saved["v"][k:k + steps]), _p(saved["flags"][k:k + steps])
                s.rb_save_v, s.rb_save_flags = _p(scratch["v"]), _p(scratch["flags"])
            _lib.check(self.lib.bmtk_glif3_simulate_fwd(C.byref(s), self.step, steps, _stream()))
            del lists       # (has to live until here)
            self.step += steps
            self._lists_replaced = self._trials_left = False
            self._pending_check = True
        return True

    def _room_for_repeats(self, n_steps):
        """Whether sums of 32 bits, where that is what a batch has, hold the input events of a call of ``n_steps`` steps."""
        tr = self._trials
        if not tr.get("whole") or tr.get("few") or self.in_most_repeats <= tr["room"]:
            return True
        # (some step of the lists repeats an id too often: a call before that step, or behind it, has nothing to do with it)
        most = self.in_repeats_of_one[max(self.step - 1, 0):self.step + n_steps]
        return not most.numel() or int(most.max()) <= tr["room"]

    def _trials_in_fixed_point(self):
        """From 32-bit sums to 64-bit ones, for good, where a plan with those pays as well; what is under way is in rb_ring either way."""
        tr = self._trials
        plan, used = self._fixed_point_plan()
        if plan is None or not self._trials_possible(plan, tr["insisted"]):
            return
        self._let_trials_tables_go(tr)
        self._trials = dict(plan, seg=None, insisted=tr["insisted"], used=used, ring=tr.get("ring"))

    def _let_trials_tables_go(self, tr):
        for key in ("hist", "seg", "packed", "cells"):
            if tr.get(key) is not None:
                self._in_use(tr.pop(key))

    def _leave_trials(self):
        """From the form with resident trials to the driver that takes its place, for good: what is still under way is
        handed over."""
        tr, self._trials = self._trials, None
        if tr is None or tr.get("ring") is None:
            return
        left, slots = tr["ring"], self.L - 1
        self._in_use(left)
        self._let_trials_tables_go(tr)
        if self.fuse_table is not None:
            self._left_ring, self._pend_from, self._pend_until, self._trials_left = left, self.step, self.step + slots, True
            return
        for t in range(self.step, self.step + slots):
            cells = left[:, t % slots]                                            # [batch][4][n]
            if cells.dtype == torch.int64:
                cells = (cells.double() * 2.0 ** -(32 + self.sum_shift)).float()
            self._ring[t % self.L] += cells.permute(1, 2, 0).reshape(NREC, self.ne)
        if torch.cuda.is_current_stream_capturing():
            left.zero_()        # (handed over once, however often the graph is replayed)

    def _in_use(self, t):
        """``t``, which will be let go, is read by launches on the current stream, which need not be the one it was made on, or by a
        graph, with every replay."""
        if torch.cuda.is_current_stream_capturing():
            self._kept.append(t)
        else:
            t.record_stream(torch.cuda.current_stream(t.device))

    # What the launch-per-step drivers keep between calls.  For a caller that looks at it, the form with resident trials gives way
    # to them first.  Pushed events are then handed over in the ring; for the fused form, whose history of spike bits cannot
    # be had from sums, they wait apart (_left_ring) and join its sums in the steps they are due in, unless ``step`` is set back.
    @property
    def ring(self):
        self._leave_trials()
        return self._ring

    @ring.setter
    def ring(self, value):
        self._leave_trials()
        self._ring = value

    @property
    def work_bits(self):
        self._leave_trials()
        return self._work_bits

    @work_bits.setter
    def work_bits(self, value):
        self._leave_trials()
        self._work_bits = value

    @property
    def fuse_any(self):
        self._leave_trials()
        return self._fuse_any

    @fuse_any.setter
    def fuse_any(self, value):
        self._leave_trials()
        self._fuse_any = value

    def _setup_fused(self):
        """Joint target-major table, joint history and activity map of the fused batched driver."""
        n, batch, n_in = self.n, self.batch, self.n_inputs if self.inp is not None else 0
        rows = 64 // batch                   # neurons of a group: one word of a history row
        self.fuse_in_base = -(-n // rows) * rows
        if self.fuse_in_base + n_in + rows >= 2 ** 24:
            return
        self.fuse_table = SynapseTable.joined_by_target(self.rec, self.inp, n, self.fuse_in_base)
        if self.sum_shift:
            self.fuse_table.weights *= 2.0 ** self.sum_shift
        self.fuse_table.pad_packed(FUSE_PAD)
        self.fuse_hist_stride = self.fuse_in_base // rows + -(-n_in // rows) + 1
        self.hist_slots = self.L + 4         # two steps per launch: rows read, written and cleared ahead
        self._ring = torch.zeros(self.L + 2, NREC, self.ne, device=self.dev)   # (its ring: two slots more)
        self._work_bits = torch.zeros(self.hist_slots * self.fuse_hist_stride, dtype=torch.int64, device=self.dev)
        # one bit of the activity map per 2^shift sources: the smallest shift whose map fits the LDS beside the
        # accumulators (where it also fits with a byte per source, the library takes that)
        self.fuse_shift = 0
        while FUSE_LDS_FIXED + self.L * self._fuse_any_words() * 4 > FUSE_LDS_BYTES:
            self.fuse_shift += 1
        self._fuse_any = self._new_fuse_any()

    def set_fuse_shift(self, shift):
        """Fused form: one bit of the activity map per 2^shift sources (the constructor picks the smallest shift
        whose map fits the LDS).  Before the first run only."""
        if self.fuse_table is None or self.step:
            raise ValueError("set_fuse_shift applies to the fused form before its first run")
        old, self.fuse_shift = self.fuse_shift, int(shift)
        if not 0 <= self.fuse_shift <= 16 or FUSE_LDS_FIXED + self.L * self._fuse_any_words() * 4 > FUSE_LDS_BYTES:
            self.fuse_shift = old
            raise ValueError("shift must lie in 0..16 and leave the activity map within the LDS")
        self._fuse_any = self._new_fuse_any()

    def _new_fuse_any(self):
        # the activity map (one row per history row) and, behind it, the map of ring cells that hold something
        # (one row per ring slot, a bit per neuron)
        # (the form with a byte per source keeps two maps, rows padded to whole words of the history)
        byte_words = -(-(self.fuse_hist_stride - 1) * (64 // self.batch) // 4)
        words = max(self.hist_slots * self._fuse_any_words(), 2 * byte_words)
        return torch.zeros(words + (self.L + 2) * (-(-self.n // 32)), dtype=torch.int32, device=self.dev)

    def _fuse_any_words(self):
        groups = -(-(self.fuse_in_base + (self.n_inputs if self.inp is not None else 0)) // (1 << self.fuse_shift))
        return -(-groups // 32)

    def _setup_resident(self, required):
        """Resident mode keeps state in registers and the ring in LDS for a whole
        run; it needs batch 1, at most 1024 elements per compute unit and a ring
        slice that fits in LDS beside the kernel's active-row list."""
        n_cu = torch.cuda.get_device_properties(self.dev).multi_processor_count
        span = resident_span(self.ne, self.batch, self.L, n_cu, single=self.single_workgroup)
        if not span:
            if required:
                raise ValueError("network does not fit resident mode (batch 1, <= 1024 elements per compute unit, "
                                 "ring slice + {} bytes of lists within the {} bytes of LDS)".format(
                                     RES_LDS_EXTRA, RES_LDS_BYTES))
            return
        groups = -(-self.ne // span)
        if groups == 1:
            # (whole rows are read, in any order)
            self.res_span, self.res_groups, self.res_fired = span, groups, None
            return
        if self.rec is not None:
            self.rec = self.rec.sorted_by_index()
            self.rec_seg = self.rec.segment_offsets(span, groups)
        if self.inp is not None:
            self.inp = self.inp.sorted_by_index()
            self.inp_seg = self.inp.segment_offsets(span, groups)
        self.res_unified = None
        if self.rec is not None and self.inp is not None and self.rec.nnz + self.inp.nnz < (1 << 32):
            # One table for both kinds of rows, the input rows behind the recurrent ones: the kernel then needs no
            # choice between two tables per listed row (and fewer of its scarce scalar registers).  The packed
            # records of the two tables become views of the joint array; the input offsets count from its start.
            nr, ni = self.rec.nnz, self.inp.nnz
            packed = torch.empty(max(nr + ni, 1), 2, dtype=torch.int32, device=self.dev)
            packed[:nr] = self.rec.packed()[:nr]
            packed[nr:nr + ni] = self.inp.packed()[:ni]
            self.rec._packed, self.inp._packed = packed[:nr], packed[nr:nr + ni]
            seg = torch.empty(self.n + self.inp.n_rows, groups + 1, dtype=torch.int32, device=self.dev)
            seg[:self.n] = self.rec_seg
            seg[self.n:] = ((self.inp_seg.long() & 0xFFFFFFFF) + nr).to(torch.int32)   # uint32 kept in int32
            self.rec_seg, self.inp_seg = seg[:self.n], seg[self.n:]
            self.res_unified = (packed, seg)
        self.res_span, self.res_groups = span, groups
        # asks for the exchange by lists of fired neurons (bmtk_glif3_sim.res_fired: that it is there is all that is looked at)
        lists = self.fired_lists and lists_pay(span, groups, self.expected_rate_hz, self.h)
        self.res_fired = torch.zeros(1, dtype=torch.int32, device=self.dev) if lists else None

    def check(self):
        """Raise if a resident run since the last check gave up on its grid barrier (synchronises).  The abort
        word is sticky on the device: a run that finds it set gives up at once, so a failure cannot be lost
        between two checks; it is cleared here."""
        if self._pending_check:
            self._pending_check = False
            if int(self.res_sync[1].item()) != 0:
                self.res_sync[1] = 0
                raise RuntimeError("resident simulation aborted: grid barrier timed out; results since the last "
                                   "check are invalid")

    def _table(self, csr, n_rows):
        if torch.is_tensor(csr[0]):
            rows = csr[0].numel() - 1 if n_rows is None else n_rows
            return SynapseTable.from_device(csr, rows, self.n, self.L)
        rows = csr[0].size - 1 if n_rows is None else n_rows
        net.check_csr(csr, rows, self.n, self.L)
        return SynapseTable.from_numpy(csr, self.dev)

    def set_input_events(self, in_ptr, in_events):
        """Per-step event lists: events in_events[in_ptr[t]:in_ptr[t+1]] are
        emitted in step t (their spike stamp is t+1).  Within a step the ids
        (source*batch+trial) must be ascending -- the input-weight gradient kernel
        gives every source's run of events one writer and relies on it.  The same id
        may occur more than once in a step (two spikes of one generator inside one
        resolution step, which NEST delivers both): every occurrence is delivered.
        The pull form of the inputs turns a step's events into bits, which hold an id
        once; the second and later occurrences are then listed apart
        (``in_repeat_ptr`` / ``in_repeat_events``) and delivered as events on top.

        Lists that replace others between two calls should still name the events of the step behind (``step - 1``): the
        separate pull launches read that step once more at the start of a call, and so does the fused form in their
        place (``fuse_rereads``: batches that do not divide 64, from some ``expected_rate_hz`` on).  Lists without them take
        back what those events still had under way there; the other forms have delivered them and look at later steps only."""
        if self.inp is None and not self.inp_without_synapses:
            raise ValueError("no input synapse table")
        n_ids = self.n_inputs * self.batch
        if torch.is_tensor(in_ptr):
            if (not torch.is_tensor(in_events) or in_ptr.dtype != torch.int64 or in_events.dtype != torch.int32
                    or in_ptr.dim() != 1 or in_events.dim() != 1 or not in_ptr.numel()):
                raise ValueError("device input event lists are inconsistent")
            in_ptr, in_events = in_ptr.to(self.dev).contiguous(), in_events.to(self.dev).contiguous()
            look = True
        else:
            in_ptr = np.ascontiguousarray(in_ptr, np.int64)
            in_events = np.ascontiguousarray(in_events, np.int32)
            look = net.check_input_events(in_ptr, in_events, n_ids)
            in_ptr = torch.as_tensor(in_ptr, device=self.dev)
            in_events = torch.as_tensor(in_events, device=self.dev)
        most, longest, repeated = self._look_over_events(in_ptr, in_events, n_ids) if look else (0, None, None)
        self.in_ptr = in_ptr
        self.in_events = in_events if in_events.numel() else in_events.new_zeros(1)
        self.in_steps = in_ptr.numel() - 1
        self._lists_replaced = self.step > 0
        self.in_duplicates, self.in_most_repeats, self.in_repeats_of_one = most > 0, most, longest
        self.in_repeat_ptr, self.in_repeat_events = repeated or (None, None)

    def _look_over_events(self, in_ptr, in_events, n_ids):
        """ValueError for lists that are not what they should be; how often a step repeats an id at most, the same of each step, and the running
        sum of the repeats of the steps with the ids themselves where a form at hand asks for them, or None."""
        steps = in_ptr.numel() - 1
        found = torch.zeros(2 * steps + 3, dtype=torch.int32, device=self.dev)  # ... and behind the three words what each step repeats
        at = _p(found)
        _lib.check(self.lib.bmtk_events_check(steps, _p(in_ptr), in_events.numel(), _p(in_events), n_ids, at + 12, at + 12 + 4 * steps, at, _stream()))
        repeats, longest = found[3:steps + 3], found[steps + 3:]    # (while the device looks)
        bad, count, most = found[:3].tolist()
        if bad & _lib.EVENTS_INCONSISTENT:
            raise ValueError("device input event lists are inconsistent")
        if bad:
            raise ValueError("input events must be ascending within every step")
        if not count or (self.pull_inp_table is None and self.fuse_table is None):
            return most, longest, None
        first = torch.zeros(steps + 1, dtype=torch.int64, device=self.dev)
        torch.cumsum(repeats, 0, out=first[1:])
        again = torch.empty(count, dtype=torch.int32, device=self.dev)
        _lib.check(self.lib.bmtk_events_repeated(steps, _p(in_ptr), _p(in_events), _p(first), _p(again), _stream()))
        return most, longest, (first, again)

    def _struct(self, bits=None, record=None):
        s = _lib.Glif3Sim()
        st = self.state
        s.n_neurons, s.batch, s.ring_slots, s.h = self.n, self.batch, self.L, self.h
        s.V, s.asc, s.y1, s.y2, s.ref = (_p(x) for x in (st.V, st.asc, st.y1, st.y2, st.ref))
        s.prop, s.prop_stride, s.class_id = _p(self.prop), self.prop.shape[1], _p(self.class_id)
        s.ring = _p(self._ring)
        if self.rec is not None:
            s.rec_indptr, s.rec_indices, s.rec_weights, s.rec_delays, s.rec_receptors = self.rec.pointers()
            s.rec_packed = _p(self.rec.packed())
        if self.inp is not None and self.in_ptr is not None:
            s.n_inputs = self.n_inputs
            s.in_ptr, s.in_events = _p(self.in_ptr), _p(self.in_events)
            s.inp_indptr, s.inp_indices, s.inp_weights, s.inp_delays, s.inp_receptors = self.inp.pointers()
            s.inp_packed = _p(self.inp.packed())
        s.i_ext = _p(self.i_ext)
        s.work_bits = _p(self._work_bits)
        s.delay_offset, s.hist_slots, s.delay_bits = self.delay_offset, self.hist_slots, self.delay_bits
        s.sum_shift = self.sum_shift
        if self.pull_table is not None:
            s.pull_indptr, s.pull_packed = _p(self.pull_table.indptr), _p(self.pull_table.packed())
            s.pull_syn, s.pull_work = _p(self.pull_syn), _p(self.pull_work)
            if self.pull_inp_table is not None and self.in_ptr is not None:
                s.pull_inp_indptr, s.pull_inp_packed = _p(self.pull_inp_table.indptr), _p(self.pull_inp_table.packed())
                s.pull_inp_syn, s.pull_inp_work = _p(self.pull_inp_syn), _p(self.pull_inp_work)
                s.in_hist, s.in_hist_stride = _p(self.in_hist), self.in_hist_stride
                if self.in_repeat_ptr is not None:
                    s.in_repeat_ptr, s.in_repeat_events = _p(self.in_repeat_ptr), _p(self.in_repeat_events)
        if not self._pend_from <= self.step < self._pend_until:
            # (all of it has arrived, or the caller began anew with an earlier step)
            self._left_ring, self._pend_until = None, 0
        if self.fuse_table is not None:
            s.n_inputs = self.n_inputs if self.inp is not None else 0   # the history's layout, events or not
            s.fuse_indptr, s.fuse_packed = _p(self.fuse_table.indptr), _p(self.fuse_table.packed())
            s.fuse_any, s.fuse_hist_stride, s.fuse_in_base = _p(self._fuse_any), self.fuse_hist_stride, self.fuse_in_base
            s.fuse_shift, s.fuse_wg_per_cu = self.fuse_shift, self.fuse_wg_per_cu
            s.fuse_max_team = max(1, -(-self.fuse_table.nnz // (256 * -(-self.n // (64 // self.batch)))))
            s.in_again = 1 if self.fuse_rereads and (self._lists_replaced or self._trials_left) else 0
            if self._left_ring is not None:
                s.rb_ring, s.rb_pend_until = _p(self._left_ring), self._pend_until
                self._in_use(self._left_ring)
            if self.in_repeat_ptr is not None:
                s.in_repeat_ptr, s.in_repeat_events = _p(self.in_repeat_ptr), _p(self.in_repeat_events)
        if self.res_span:
            s.res_span, s.res_groups, s.res_sync = self.res_span, self.res_groups, _p(self.res_sync)
            s.res_spin_limit = int(self.spin_limit)
            s.rec_seg, s.inp_seg = _p(self.rec_seg), _p(self.inp_seg)
            s.res_fired = _p(self.res_fired)
            s.res_min_delay = self.least_delay
            s.res_step_events = min(-(-self.in_events.numel() // max(1, self.in_steps)), 1 << 30) if self.in_ptr is not None else 0
            if self.res_unified is not None and s.inp_packed and self.res_groups > 1:
                s.inp_packed = s.rec_packed      # the input offsets count from the start of the joint table
        if bits is not None:
            s.spike_bits, s.spike_bits_stride = _p(bits), bits.shape[1]
        if record is not None:
            s.spike_step, s.spike_elem, s.spike_frac = _p(record["step"]), _p(record["elem"]), _p(record["frac"])
            s.spike_cap, s.spike_count = record["step"].numel(), _p(record["count"])
            s.spike_ways = record.get("ways", 1)
        return s

    def set_probes(self, element_ids, every=1):
        """Record the membrane potential of some elements (what a multimeter connected to them does): after every
        step t with (t + 1) % every == 0, in both modes.  ``run`` then returns ``probe`` = dict(v=[samples,
        len(element_ids)] fp32 of U = V_m - E_L, steps=int64 [samples], the sampled steps).  None switches it off."""
        if element_ids is None:
            self.probe_ids = self.probe_col = None
            return
        ids = np.asarray(element_ids, np.int64).reshape(-1)
        if ids.size == 0 or ids.min() < 0 or ids.max() >= self.ne or np.unique(ids).size != ids.size:
            raise ValueError("probes need distinct element ids in 0..{}".format(self.ne - 1))
        if int(every) < 1:
            raise ValueError("every must be at least 1")
        col = np.full(self.ne, -1, np.int32)
        col[ids] = np.arange(ids.size, dtype=np.int32)
        self.probe_ids, self.probe_every = ids, int(every)
        self.probe_col = torch.as_tensor(col, device=self.dev)

    def run(self, n_steps, spike_bits=True, record_cap=0, save_state=False, record_ways=None):
        """Advance ``n_steps`` steps.  Returns a dict with ``bits`` (int64
        [n_steps, words], spike bits per step) and, when ``record_cap`` > 0,
        the atomic spike record with crossing fractions (read it with ``collect_record``: a large record is
        kept as several lists); ``save_state`` adds the
        per-step record (potentials and flags) the backward pass reads; ``probe``
        holds the potentials asked for with ``set_probes``.  Does not
        synchronise."""
        if self.in_ptr is not None and self.step + n_steps > self.in_steps:
            raise ValueError("input event lists cover {} steps, run would reach {}".format(
                self.in_steps, self.step + n_steps))
        bits = torch.zeros(n_steps, self.words, dtype=torch.int64, device=self.dev) if spike_bits else None
        record = None
        if record_cap:
            # A large record is kept as RECORD_WAYS lists with a counter each (``collect_record`` joins them): the
            # wavefronts of a whole network bumping ONE counter cost the resident kernel 1.5 of 5.5 us per step.
            # No more lists than workgroups (a list nobody appends to is room lost), each of at least 1024 entries.
            # Workgroups are dealt out to the lists in turn, so a list may serve one workgroup more than another:
            # callers size the record with room to spare, as they had to for one list.
            n_wg = self.res_groups if self.res_span else -(-self.ne // 512)
            ways = 1
            while ways * 2 <= min(RECORD_WAYS, n_wg) and record_cap >= ways * 2 * 1024:
                ways *= 2
            if self.res_groups > RECORD_WAYS and self.delay_offset == 0 and record_cap >= 256 * 1024:
                # the resident kernel without slack: with a list per workgroup (at most 256 are launched) a
                # workgroup keeps its count in a register and no wavefront waits for an atomic on device memory
                ways = 256
            if record_ways is not None:      # the caller's choice: a power of two up to 256
                ways = int(record_ways)
                if ways < 1 or ways > 256 or ways & (ways - 1):
                    raise ValueError("record_ways must be a power of two in 1..256")
            record_cap = -(-int(record_cap) // ways) * ways
            # (only the counted entries are ever read: no need to clear a gigabyte of room first)
            record = dict(step=torch.empty(record_cap, dtype=torch.int32, device=self.dev),
                          elem=torch.empty(record_cap, dtype=torch.int32, device=self.dev),
                          frac=torch.empty(record_cap, dtype=torch.float32, device=self.dev),
                          count=torch.zeros(1 if ways == 1 else ways * _lib.RECORD_COUNT_STRIDE, dtype=torch.int64,
                                            device=self.dev), ways=ways)
        use_trials = (self._trials is not None and n_steps >= TRIALS_MIN_STEPS and record is None
                      and self.probe_col is None and not torch.cuda.is_current_stream_capturing())
        stretch = n_steps
        if use_trials and save_state:
            stretch = min(65535, TRIALS_SAVE_BYTES // (5 * self.ne))
            use_trials = self.batch > 1 and stretch >= TRIALS_MIN_STEPS
        if use_trials and not self._room_for_repeats(n_steps):
            self._trials_in_fixed_point()
            use_trials = not self._trials.get("whole")
        if self._trials is not None and n_steps > 0 and not use_trials:
            self._leave_trials()
        saved = None
        if save_state:
            if self.res_span:
                raise ValueError("save_state needs a simulator built with resident=False")
            saved = dict(v=torch.empty(n_steps, self.ne, device=self.dev),
                         flags=torch.empty(n_steps, self.ne, dtype=torch.uint8, device=self.dev), step0=self.step)
        if use_trials:
            if self._run_trials(n_steps, min(stretch, n_steps), bits, saved):
                return dict(bits=bits, record=None, saved=saved, probe=None)
            self._leave_trials()
        s = self._struct(bits, record)
        if saved is not None:
            s.save_v, s.save_flags = _p(saved["v"]), _p(saved["flags"])
        probe = None
        if self.probe_col is not None:
            every = self.probe_every
            first = -(-(self.step + 1) // every) * every - 1  # first step t >= self.step with (t + 1) % every == 0
            steps = torch.arange(first, max(first, self.step + n_steps), every, dtype=torch.int64)  # may be none
            room = torch.empty(max(1, steps.numel()), self.probe_ids.size, device=self.dev)  # a call may sample nothing
            probe = dict(v=room[:steps.numel()], steps=steps)
            s.probe_col, s.probe_v = _p(self.probe_col), room.data_ptr()
            s.probe_stride, s.probe_every = self.probe_ids.size, every
        _lib.check(self.lib.bmtk_glif3_simulate_fwd(C.byref(s), self.step, n_steps, _stream()))
        self.step += n_steps
        self._lists_replaced = self._lists_replaced and n_steps == 0
        self._trials_left = self._trials_left and n_steps == 0
        self._pending_check = self._pending_check or bool(self.res_span)
        return dict(bits=bits, record=record, saved=saved, probe=probe)

    def collect_record(self, record, sort_scale=None):
        """The spike record of a ``run(..., record_cap=...)`` as one list: dict(step int32[], elem int32[], frac
        float32[], count int, overflow bool, ways, way_cap, fullest), unordered within a step.  ``count`` is the
        number of spikes the run produced; ``overflow`` says that some of them found no room (then the lists are
        incomplete).  A record kept as ``ways`` lists overflows as soon as ONE list does -- a workgroup appends to
        its own list of ``way_cap`` = cap / ways entries only, so activity concentrated in the neurons of a few
        workgroups can overflow while ``count`` is far below the record's total size; ``fullest`` is the largest
        count of a single list (``overflow_message`` words it).
        With ``sort_scale`` (the resolution in ms) the list comes back ordered by spike time
        (step + frac) * sort_scale, ties by element -- sorted on the device, where two million spikes take
        milliseconds instead of the second a host sort takes -- and ``time`` (float64, ms) is added.
        Synchronises."""
        self.check()
        ways = record.get("ways", 1)
        cap = record["step"].numel()
        way_cap = cap // ways
        counts = record["count"][::_lib.RECORD_COUNT_STRIDE][:ways] if ways > 1 else record["count"][:1]
        counts = counts.cpu()                                  # the one synchronisation
        stored = torch.clamp(counts, max=way_cap).tolist()
        if ways == 1:
            keep = slice(0, stored[0])
        else:                                                  # the filled part of every list, one after the other
            dev = record["step"].device
            filled = torch.tensor(stored, dtype=torch.int64, device=dev)
            first = torch.arange(ways, dtype=torch.int64, device=dev) * way_cap - (torch.cumsum(filled, 0) - filled)
            keep = torch.arange(sum(stored), dtype=torch.int64, device=dev) + torch.repeat_interleave(first, filled)
        out = dict(step=record["step"][keep], elem=record["elem"][keep], frac=record["frac"][keep],
                   count=int(counts.sum()), overflow=bool((counts > way_cap).any()), ways=ways, way_cap=way_cap,
                   fullest=int(counts.max()))
        if sort_scale is not None:
            t = (out["step"].to(torch.float64) + out["frac"].to(torch.float64)) * float(sort_scale)
            by_elem = torch.argsort(out["elem"], stable=True)
            order = by_elem[torch.argsort(t[by_elem], stable=True)]
            out.update(step=out["step"][order], elem=out["elem"][order], frac=out["frac"][order], time=t[order])
        return out

    @staticmethod
    def overflow_message(rec):
        """What a caller reports when ``collect_record`` came back with ``overflow``: the capacity that ran out is
        that of one list, not of the record."""
        if rec["ways"] == 1:
            return "{} spikes, room for {}".format(rec["count"], rec["way_cap"])
        return ("{} spikes in all; the record is kept as {} lists of {} entries (one per group of workgroups) and "
                "the fullest list was asked to hold {}".format(rec["count"], rec["ways"], rec["way_cap"], rec["fullest"]))

    def to_host(self, *tensors):
        """Device tensors -> NumPy arrays through pinned host memory (torch keeps freed pinned blocks for reuse): a
        spike record of two million entries takes a millisecond or two instead of the five a copy into pageable
        memory takes.  The arrays own their memory.  Synchronises."""
        sizes = [t.numel() * t.element_size() for t in tensors]
        offsets = [0]
        for n in sizes:
            offsets.append(-(-(offsets[-1] + n) // 256) * 256)
        stage = torch.empty(max(offsets[-1], 1), dtype=torch.uint8, pin_memory=True)
        views = []
        for t, n, o in zip(tensors, sizes, offsets):
            v = stage[o:o + n].view(t.dtype).view(t.shape) if n else torch.empty(t.shape, dtype=t.dtype)
            if n:
                v.copy_(t.contiguous(), non_blocking=True)
            views.append(v)
        torch.cuda.synchronize(self.dev)
        return tuple(v.numpy() for v in views)   # (an array keeps its block of pinned memory alive)

    def spikes_from_bits(self, bits, step0=0):
        """Spike bits -> (step int64[], element int64[]) ascending, via the
        compaction kernels (exactly ``numpy.nonzero`` of the raster)."""
        self.check()
        n_steps, words = bits.shape
        per = max(1, (2 ** 31 - 64) // (words * 64))
        steps, elems = [], []
        for k0 in range(0, n_steps, per):
            chunk = bits[k0:k0 + per].contiguous()
            n = chunk.numel() * 64
            comp = SpikeCompactor(n, self.dev)
            ids, count = comp(torch.cat([chunk.reshape(-1), chunk.new_zeros(1)]))
            ids = ids[:int(count.item())].to(torch.int64)
            steps.append(ids // (words * 64) + k0 + step0)
            elems.append(ids % (words * 64))
        return torch.cat(steps), torch.cat(elems)

    def raster(self, bits):
        """uint8 [n_steps, ne] from spike bits."""
        self.check()
        return unpack_bits(bits, self.ne)

    def synaptic_events(self, bits):
        """Number of recurrent synaptic events the spikes in ``bits`` caused
        (sum of the out-degree of every spiking neuron)."""
        if self.rec is None:
            return 0
        _, elems = self.spikes_from_bits(bits)
        deg = (self.rec.indptr[1:] - self.rec.indptr[:-1]).to(torch.int64)
        return int(deg[elems // self.batch].sum().item())
