"""What is measured: the work a program asks of this framework, through the calls such a program makes.

Six kinds of work, one per way of using the package:

script    ``PointSimulator(...).run()``: a whole run script on a network of some hundred cells (bmtk's own examples are
          300 to 450 cells at 0.1 ms), simulator built, spike trains handed over, spikes back in host memory in time order
forward   ``Glif3Simulator.set_input_events`` / ``run``: a stretch of a longer simulation with its own input spikes;
          one trial of networks from a few thousand neurons up to more than stay resident on the chip, or many trials
          of one network at once (``batch``)
train     the same with ``save_state``, a loss on population rates, and ``Glif3Bptt.backward``: one training step
update    ``ops.glif3_step_fwd`` alone: the state update of a caller with a step loop of his own, by class table or
          with parameters per neuron
loop      such a step loop in full: update, compaction of the spikes, event-driven delivery into the ring
deliver   ``ops.csr_propagate_pull2`` alone: two steps' arrivals from the spike history of a batch of trials

Weights of the simulated networks are whole multiples of 1/256 pA, as nsyns * syn_weight of an edge type is a multiple of
the type's weight.  Sums of them are exact in fp32 in any order, so the spikes of a run do not depend on the order in
which an implementation adds: a chaotic network can be compared bit for bit.
"""
import math

import numpy as np
import torch

from bmtk_amd import ops, synthetic, training
from bmtk_amd.layout import PAR
from bmtk_amd.pointnet import PointNetwork, PointSimulator
from bmtk_amd.simulator import Glif3Simulator

IN_RATE_HZ = 5.0
QUANTUM = 1.0 / 256.0   # pA
RATE_HZ = 3.0           # what the networks settle near
SETTLE_STEPS = 200      # steps of every simulation before the first pass: the transient from rest


def listed():
    return [
        # bmtk's example size at NEST's usual resolution, one second of it: latency and set-up count
        dict(name="script_450", kind="script", n=450, k_rec=45, n_in=1000, k_in=110, dt=0.1, steps=10000),
        # a cortical column of moderate size, one trial
        dict(name="forward_10k", kind="forward", n=10007, k_rec=500, n_in=2000, k_in=100, batch=1, classes=37, steps=1000),
        # the V1 model: 230,924 neurons of 111 classes, 17,400 LGN-like inputs, three seconds
        dict(name="forward_v1", kind="forward", n=230924, k_rec=300, n_in=17400, k_in=35, batch=1, classes=111, steps=3000),
        # more neurons than the compute units' registers hold
        dict(name="forward_400k", kind="forward", n=400123, k_rec=150, n_in=30000, k_in=30, batch=1, classes=111, steps=300),
        # 32 trials at once of a network with a thousand synapses per neuron and parameters per neuron
        dict(name="batch32_52k", kind="forward", n=51978, k_rec=1000, n_in=17400, k_in=154, batch=32, classes=0, steps=200),
        # a number of trials as experiments have it, not a power of two
        dict(name="batch20_20k", kind="forward", n=20011, k_rec=700, n_in=5000, k_in=120, batch=20, classes=50, steps=200),
        # a few trials of the V1 model
        dict(name="batch8_v1", kind="forward", n=230924, k_rec=300, n_in=17400, k_in=35, batch=8, classes=111, steps=100),
        # training at the size of the V1 model's core
        dict(name="train_52k", kind="train", n=51978, k_rec=1000, n_in=17400, k_in=154, batch=32, classes=0, steps=40),
        # training of a small network, a batch that is no power of two: launches count
        dict(name="train_3k", kind="train", n=3001, k_rec=200, n_in=1000, k_in=100, batch=12, classes=0, steps=100),
        # the state update alone
        dict(name="update_1m", kind="update", n=1 << 20, batch=1, classes=111),
        # a caller's own step loop, one step
        dict(name="loop_30k", kind="loop", n=30011, k_rec=300, classes=111),
        # delivery alone, 64 trials at 5 Hz
        dict(name="deliver_52k", kind="deliver", n=51978, k_rec=1000, batch=64, rate=5.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("script", "forward", "batched", "train", "update", "loop", "deliver"), (1, 3, 4, 3, 2, 1, 2))[0]
    classes = rng.choice((0, 23, 111, 300))
    if kind == "script":
        n = _log(rng, 150, 900)
        return dict(kind=kind, n=n, k_rec=min(n // 4, rng.randint(20, 80)), n_in=rng.randint(200, 1500), k_in=rng.randint(50, 150),
                    dt=rng.choice((0.1, 0.2, 1.0)), steps=_log(rng, 2000, 10000))
    if kind == "update":
        batch = rng.choice((1, 1, 1, 5, 8, 32, 64))
        return dict(kind=kind, n=max(100, _log(rng, 20000, 4000000) // batch), batch=batch, classes=classes if batch == 1 else 0)
    if kind == "loop":
        n = _log(rng, 5000, 200000)
        return dict(kind=kind, n=n, k_rec=_log(rng, 50, 500), classes=classes)
    if kind == "deliver":
        return dict(kind=kind, n=_log(rng, 5000, 52000), k_rec=_log(rng, 200, 1000), batch=rng.choice((8, 16, 32, 48, 64)),
                    rate=round(math.exp(rng.uniform(math.log(0.3), math.log(20.0))), 2))
    if kind == "forward":
        n = _log(rng, 2000, 400000)
        k = _log(rng, 100, max(101, min(1000, 60000000 // n)))
        return dict(kind=kind, n=n, k_rec=k, n_in=max(500, n // rng.randint(8, 24)), k_in=rng.randint(25, 120 if n < 60000 else 40), batch=1,
                    classes=classes, steps=_log(rng, 200, 1000))
    n = _log(rng, 2000, 120000) if kind == "batched" else _log(rng, 1500, 52000)
    k = _log(rng, 100, max(101, min(1000, 50000000 // n)))
    batch = rng.choice((4, 8, 10, 12, 16, 20, 24, 32, 32, 40, 64) if kind == "batched" else (4, 8, 12, 16, 16, 20, 32, 32))
    while n * batch > 2000000:
        batch = max(4, batch // 2)
    return dict(kind="forward" if kind == "batched" else kind, n=n, k_rec=k, n_in=max(500, n // rng.randint(2, 12)), k_in=rng.randint(25, 150),
                batch=batch, classes=classes, steps=_log(rng, 50, 200) if kind == "batched" else _log(rng, 20, 60))


# ---------------------------------------------------------------------------------------------------------------------
# networks

def _quantized(table):
    indptr, indices, w, d, r = table
    q = torch.round(w.abs() / QUANTUM).clamp_(min=1.0).mul_(QUANTUM)
    return indptr, indices, torch.copysign(q, w), d, r


def _cells(case, seed):
    rng = np.random.default_rng(seed)
    if case["classes"]:
        return synthetic.random_cells(rng, case["classes"]), rng.integers(0, case["classes"], case["n"]).astype(np.int32)
    return synthetic.random_cells(rng, case["n"]), None


def _recurrent_edges(n, k, seed):
    """n * k edges with uniformly random sources and a lognormal spread of in-degrees (sigma 0.5), delays of 1 to 5 steps,
    a fifth of the cells inhibitory.  The weights keep the sum over a neuron's synapses about the same whatever their
    number, so that every network settles at a few spikes per second."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    share = torch.exp(0.5 * torch.randn(n, device="cuda", generator=g, dtype=torch.float64)).cumsum(0)
    tgt = torch.searchsorted(share, torch.rand(n * k, device="cuda", generator=g, dtype=torch.float64) * share[-1]).clamp_(max=n - 1)
    src = torch.randint(0, n, (n * k,), device="cuda", generator=g)
    inh = torch.rand(n, device="cuda", generator=g) < 0.2
    w = torch.exp(torch.randn(n * k, device="cuda", generator=g)) * min(1.0, 200.0 / k)
    w = torch.where(inh[src], -w, w)
    d = torch.randint(1, 6, (n * k,), device="cuda", generator=g, dtype=torch.uint8)
    return src, tgt, w, d, (inh[src].to(torch.uint8) + 2 * inh[tgt].to(torch.uint8))


def _table(n, k, seed):
    t = ops.SynapseTable.from_edges(*_recurrent_edges(n, k, seed), n, n)
    return t.indptr, t.indices, t.weights, t.delays, t.receptors


def _tables(case, seed):
    """Recurrent and input tables, source-major."""
    n, k_in = case["n"], case["k_in"]
    inp = synthetic.device_input_table(case["n_in"], n, n * k_in, seed=seed + 1, w_scale=290.0 / k_in)
    return _quantized(_table(n, case["k_rec"], seed)), _quantized(inp)


class _Simulation:
    """A simulator that has left the transient from rest, and the input spikes of the next stretch."""

    def __init__(self, case, seed):
        par, class_id = _cells(case, seed)
        rec, inp = _tables(case, seed)
        train = case["kind"] == "train"
        self.sim = Glif3Simulator(case["n"], par, 1.0, batch=case["batch"], class_id=class_id, rec=rec, inp=inp,
                                  resident=False if train else "auto")
        self.steps = case["steps"]
        self.in_ptr, self.in_events = ops.poisson_events(case["n_in"], IN_RATE_HZ, 1.0, SETTLE_STEPS, batch=case["batch"], seed=seed)
        self.hand_over()
        self.sim.run(SETTLE_STEPS, spike_bits=False)
        self.in_ptr, self.in_events = ops.poisson_events(case["n_in"], IN_RATE_HZ, 1.0, self.steps, batch=case["batch"], seed=seed + 1)
        if train:
            g = torch.Generator(device="cuda").manual_seed(seed)
            self.pop = torch.randint(0, 17, (case["n"],), device="cuda", generator=g)
            self.targets = torch.rand(case["batch"], 17, device="cuda", generator=g) * 0.01
            self.bptt = training.Glif3Bptt(self.sim, dampening=0.3)

    def hand_over(self):
        """The stretch's own input spikes: lists are indexed by absolute step, the steps behind us have none."""
        behind = self.in_ptr.new_zeros(self.sim.step)
        self.sim.set_input_events(torch.cat([behind, self.in_ptr]), self.in_events)


class _Script:
    """What a run script holds before ``run()``: a network read from its files and one spike train per virtual cell."""

    def __init__(self, case, seed):
        rng = np.random.default_rng(seed)
        n, n_in, dt = case["n"], case["n_in"], case["dt"]
        classes = 5
        par = synthetic.random_cells(rng, classes)
        class_id = rng.integers(0, classes, n).astype(np.int32)
        inh = rng.random(n) < 0.2
        nnz = n * case["k_rec"]
        src, tgt = rng.integers(0, n, nnz), rng.integers(0, n, nnz)
        delay = max(1, int(round(2.0 / dt)))   # 2 ms, as the examples' edge types
        w = np.round(rng.lognormal(0, 1, nnz) / QUANTUM).clip(1) * QUANTUM * np.where(inh[src], -1.0, 1.0)
        rec = (src, tgt, w.astype(np.float32), np.full(nnz, delay), (inh[src] + 2 * inh[tgt]).astype(np.uint8))
        nnz_in = n * case["k_in"]
        w_in = np.round(rng.lognormal(0, 1, nnz_in) * 900.0 / case["k_in"] / QUANTUM).clip(1) * QUANTUM
        inp = (rng.integers(0, n_in, nnz_in), rng.integers(0, n, nnz_in), w_in.astype(np.float32), np.full(nnz_in, delay),
               np.zeros(nnz_in, np.uint8))
        self.network = PointNetwork("cortex", n, par, np.zeros((2, classes)), np.zeros(classes), class_id, np.ones(classes, bool),
                                    rec, inp, {"inputs": 0}, n_in)
        self.room = int(n * case["steps"] * dt * 0.1)   # 100 spikes per second and cell
        self.simulation = PointSimulator(self.network, dt, case["steps"] * dt)
        counts = rng.poisson(IN_RATE_HZ * case["steps"] * dt * 1e-3, n_in)
        ids = np.repeat(np.arange(n_in), counts)
        self.simulation.add_spike_inputs({"inputs": (ids, rng.uniform(dt, (case["steps"] - 1) * dt, ids.size))})


def _prepare_update(case, seed):
    par, class_id = _cells(case, seed)
    n, batch = case["n"], case["batch"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    # states uniform in their physiological ranges, a quarter of the elements refractory
    ne = n * batch
    col = torch.arange(n, device="cuda") if class_id is None else torch.as_tensor(class_id, device="cuda").long()
    col = col.repeat_interleave(batch)
    th = torch.as_tensor(par[PAR["V_TH"]] - par[PAR["E_L"]], device="cuda", dtype=torch.float32)[col]
    ref_steps = torch.as_tensor(np.ceil(par[PAR["T_REF"]]), device="cuda", dtype=torch.int32)[col]
    uniform = lambda *shape: torch.rand(*shape, device="cuda", generator=g)  # noqa: E731
    ref = torch.where(uniform(ne) < 0.25, (uniform(ne) * (ref_steps + 1)).to(torch.int32), torch.zeros_like(ref_steps))
    state = ops.Glif3State(uniform(ne) * th, -300.0 * uniform(2, ne), uniform(4, ne), uniform(4, ne), ref)
    return dict(state=state, prop=ops.glif3_precompute(par, 1.0), batch=batch,
                class_id=None if class_id is None else torch.as_tensor(class_id, device="cuda"),
                i_ext=torch.randn(ne, device="cuda", generator=g) * 50.0,
                z=torch.zeros(ne, dtype=torch.uint8, device="cuda"))


def _prepare_loop(case, seed):
    par, class_id = _cells(case, seed)
    n, L = case["n"], 6
    rec = _table(n, case["k_rec"], seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    col = torch.arange(n, device="cuda") if class_id is None else torch.as_tensor(class_id, device="cuda").long()
    rheobase = torch.as_tensor(par[PAR["G"]] * (par[PAR["V_TH"]] - par[PAR["E_L"]]), device="cuda", dtype=torch.float32)[col]
    s = dict(state=ops.Glif3State.zeros(n), prop=ops.glif3_precompute(par, 1.0), n=n, L=L, k=0,
             class_id=None if class_id is None else torch.as_tensor(class_id, device="cuda"),
             # most cells a little below their rheobase, the others firing at a few Hz
             i_ext=rheobase * (0.7 + 0.4 * torch.rand(n, device="cuda", generator=g)),
             table=ops.SynapseTable.from_device(_quantized(rec), n, n, L), ring=torch.zeros(L, 4, n, device="cuda"),
             zbits=torch.zeros(ops.n_words(n) + 1, dtype=torch.int64, device="cuda"), compact=ops.SpikeCompactor(n))
    for _ in range(SETTLE_STEPS):
        _run_loop(s)
    return s


def _prepare_deliver(case, seed):
    n, batch, L = case["n"], case["batch"], 6
    src, tgt, w, d, r = _recurrent_edges(n, case["k_rec"], seed)
    table = ops.SynapseTable.from_edges(tgt, src, w, d, r, n, n)   # target-major: rows are targets
    g = torch.Generator(device="cuda").manual_seed(seed)
    ne = n * batch
    words = ops.n_words(ne)
    hist = torch.zeros(L, words + 1, dtype=torch.int64, device="cuda")
    for row in hist:
        z = torch.zeros(words * 64, dtype=torch.bool, device="cuda")
        z[:ne] = torch.rand(ne, device="cuda", generator=g) < case["rate"] * 1e-3
        row[:-1] = (z.view(-1, 64).to(torch.int64) << torch.arange(64, device="cuda")).sum(1)
    return dict(table=table, hist=hist, n=n, batch=batch, t=L,
                syn2=torch.zeros(2, 4, ne, device="cuda"))


def prepare(case, seed):
    case, seed = dict(case), int(seed)
    if case["kind"] == "script":
        return case["kind"], _Script(case, seed)
    if case["kind"] == "update":
        return case["kind"], _prepare_update(case, seed)
    if case["kind"] == "loop":
        return case["kind"], _prepare_loop(case, seed)
    if case["kind"] == "deliver":
        return case["kind"], _prepare_deliver(case, seed)
    return case["kind"], _Simulation(case, seed)


# ---------------------------------------------------------------------------------------------------------------------
# passes

def _state(st):
    return dict(V=st.V, asc=st.asc, y1=st.y1, y2=st.y2, ref=st.ref)


def _run_forward(s):
    s.hand_over()
    out = s.sim.run(s.steps)
    return dict(bits=out["bits"], state=_state(s.sim.state))


def _run_train(s):
    s.hand_over()
    fwd = s.sim.run(s.steps, save_state=True)
    counts = training.spike_counts(fwd["bits"], s.sim.ne)
    loss, per_spike = training.rate_mse(counts, s.steps, s.sim.batch, s.pop, s.targets)
    s.bptt.zero()
    s.bptt.backward(fwd, dl_dz_const=per_spike)
    return dict(loss=loss, counts=counts, d_rec_w=s.bptt.d_rec_w, d_inp_w=s.bptt.d_inp_w)


def _run_script(s):
    elems, times = s.simulation.run()["cortex"]
    # in arrays of one length whatever the number of spikes
    if elems.size > s.room:
        raise ValueError("{} spikes".format(elems.size))
    rest = np.full(s.room - elems.size, -1.0)
    return dict(elems=np.concatenate([elems, rest.astype(elems.dtype)]), times=np.concatenate([times, rest]))


def _run_update(s):
    ops.glif3_step_fwd(s["state"], s["prop"], 1.0, batch=s["batch"], class_id=s["class_id"], i_ext=s["i_ext"], z=s["z"])
    return dict(z=s["z"], state=_state(s["state"]))


def _run_loop(s):
    k, L = s["k"], s["L"]
    # the weights that arrive in step k enter y1 with its update; the slot is free again afterwards
    ops.glif3_step_fwd(s["state"], s["prop"], 1.0, class_id=s["class_id"], syn=s["ring"][k % L], clear_syn=True, i_ext=s["i_ext"],
                       zbits=s["zbits"])
    ids, count = s["compact"](s["zbits"])
    ops.csr_propagate_scatter(ids, count, s["table"], s["ring"], s["n"], 1, k)
    s["k"] = k + 1
    return dict(zbits=s["zbits"], count=count, ring=s["ring"], state=_state(s["state"]))


def _run_deliver(s):
    ops.csr_propagate_pull2(s["hist"], s["n"], s["table"], s["syn2"], s["n"], s["batch"], s["t"])
    return s["syn2"]


_RUN = dict(script=_run_script, forward=_run_forward, train=_run_train, update=_run_update, loop=_run_loop, deliver=_run_deliver)


def run(state):
    return _RUN[state[0]](state[1])


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without

STATE_WORDS = 12        # V, 2 after-spike currents, 4 + 4 of the synaptic currents, refractory counter
PARAMETER_WORDS = 29    # propagators of a neuron or class
SYNAPSE_BYTES = 10      # index 4, weight 4, delay 1, receptor 1
FLOPS_PER_UPDATE = 70


def work(case):
    n, batch, steps = case["n"], case.get("batch", 1), case.get("steps", 1)
    ne = n * batch
    columns = case.get("classes", 5) or n
    state = ne * STATE_WORDS * 8 + columns * PARAMETER_WORDS * 4 + (n * 4 if columns != n else 0)
    h = case.get("dt", 1.0) * 1e-3
    if case["kind"] == "update":
        return {"bytes": state + ne * 5, "flops": ne * FLOPS_PER_UPDATE}
    if case["kind"] == "deliver":
        nnz = n * case["k_rec"]
        # either step's arrivals: the synapses whose source fired in some trial, the history, the sums
        active = min(1.0, 2.0 * (1.0 - (1.0 - case["rate"] * h) ** batch))
        return {"bytes": nnz * active * SYNAPSE_BYTES + 6 * ne / 8 + 2 * 16 * ne, "flops": 2 * nnz * batch * case["rate"] * h}
    if case["kind"] == "loop":
        events = n * RATE_HZ * h * case["k_rec"]
        return {"bytes": state + ne * (16 + 4) + ne / 8 + events * (SYNAPSE_BYTES + 8), "flops": ne * FLOPS_PER_UPDATE + events}
    nnz, nnz_in = n * case["k_rec"], n * case["k_in"]
    trials = batch * steps * h   # trial-seconds: a synapse is read at least once if its source fires at all
    used = nnz * (1.0 - math.exp(-RATE_HZ * trials)) + nnz_in * (1.0 - math.exp(-IN_RATE_HZ * trials))
    in_events = case["n_in"] * IN_RATE_HZ * trials
    events = (nnz * RATE_HZ + nnz_in * IN_RATE_HZ) * trials
    bytes_ = state + used * SYNAPSE_BYTES + in_events * 4 + steps * ne / 8
    flops = ne * steps * FLOPS_PER_UPDATE + events
    if case["kind"] == "train":
        # the adjoint of the update, the transposed propagation of every synapse and trial, the gradients
        bytes_ += nnz * SYNAPSE_BYTES + (nnz + nnz_in) * 4
        flops += ne * steps * 2 * FLOPS_PER_UPDATE + 2.0 * nnz * batch * steps + 2 * events
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    if case["kind"] == "train":
        # against the same adjoint in 64 bits, small networks of batch 4 to 32: 5e-7 to 1e-6 and 2e-6 to 4e-6; with the
        # sums of the transposed propagation in another order: 6e-8 and 9e-7
        return {"rel": 4e-6, "max": 2e-5}
    if case["kind"] == "deliver":
        # a handful of fp32 weights per sum, in any order
        return {"rel": 1e-6, "max": 1e-5}
    # exact sums (see the top), and an update whose operations and their order are fixed
    return "exact"
