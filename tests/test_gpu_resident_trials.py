"""The form with resident trials (state in registers, ring in LDS, several trials side by side) against the fp32 oracle."""
import numpy as np
import pytest
import torch

from oracle import glif3_oracle as orc
from bmtk_amd import ops, simulator, synthetic, training
from bmtk_amd.simulator import Glif3Simulator, fixed_point_shift, resident_trials_plan

pytestmark = pytest.mark.gpu
STATE = ("V", "asc", "y1", "y2", "ref")


def _quarter(table):
    indptr, indices, w, d, r = table
    return indptr, indices, (np.round(w * 4.0) / 4.0 + np.sign(w) * 0.25).astype(np.float32), d, r


def _case(n, batch, max_delay, classes=None, n_in=120, steps=150, seed=3, in_rate=60.0, once=(0, 0), small=None):
    cfg = synthetic.small_glif3_network(n=n, n_in=n_in, steps=steps, seed=seed, p_conn=min(0.3, 60.0 / n), in_rate=in_rate,
                                        in_fanout=max(1, min(n, 30)), max_delay=max_delay, n_classes=classes, batch=batch,
                                        w_scale=4.0, in_w_scale=20.0)
    cfg["rec_src"], cfg["inp_src"] = _quarter(cfg["rec_src"]), _quarter(cfg["inp_src"])
    if small is not None:      # the weights of two of the four receptors
        for k in ("rec_src", "inp_src"):
            indptr, indices, w, d, r = cfg[k]
            cfg[k] = indptr, indices, np.where(r >= 2, w * np.float32(small), w).astype(np.float32), d, r
    cfg["i_ext"] = np.random.default_rng(seed).uniform(0.0, 500.0, n * batch).astype(np.float32)
    # every seventh event twice, but for those of the steps once[0] .. once[1] - 1
    times = np.where(np.arange(cfg["in_events"].size) % 7 == 0, 2, 1)
    times[cfg["in_ptr"][once[0]]:cfg["in_ptr"][once[1]]] = 1
    cfg["in_ptr"] = np.concatenate([[0], np.cumsum(times)])[cfg["in_ptr"]].astype(np.int64)
    cfg["in_events"] = np.repeat(cfg["in_events"], times)
    st = orc.new_state(n, batch, np.float32)
    orc.set_threads(orc.max_threads())
    # weights in quarters of a pA: sums are exact in fp32 in any order
    want = orc.simulate(st, orc.precompute(cfg["par"], 1.0), 1.0, steps, batch=batch, class_id=cfg["class_id"],
                        ring=np.zeros((cfg["L"], 4, n * batch), np.float32), rec=cfg["rec_src"], inp=cfg["inp_src"],
                        in_ptr=cfg["in_ptr"], in_events=cfg["in_events"], i_ext=cfg["i_ext"], raster=True)
    assert want["count"] > 0
    return cfg, want["raster"], st


def _sim(cfg, batch, **kw):
    sim = Glif3Simulator(cfg["n"], cfg["par"], 1.0, batch=batch, class_id=cfg["class_id"], rec=cfg["rec_src"], inp=cfg["inp_src"],
                         i_ext=cfg["i_ext"], ring_slots=cfg["L"], resident=False, **kw)
    sim.set_input_events(cfg["in_ptr"], cfg["in_events"])
    return sim


def _same(sim, outs, raster, st):
    sim.check()
    np.testing.assert_array_equal(np.concatenate([sim.raster(o["bits"]).cpu().numpy() for o in outs]), raster)
    got = sim.state.to_numpy()
    for k in STATE:
        np.testing.assert_array_equal(got[k], st[k], err_msg=k)


@pytest.mark.parametrize("n,batch,max_delay,classes", [
    (20, 2, 1, None), (63, 5, 2, None), (64, 64, 4, 3), (65, 3, 6, None), (700, 20, 5, 7), (1025, 33, 4, None), (2100, 8, 12, None),
    (1500, 64, 5, 11)])
def test_equals_the_oracle_over_two_calls(n, batch, max_delay, classes):
    """One neuron to a wavefront's worth and one more, one to several workgroups a trial, a ring of one slot, last launches
    with fewer trials than the others: raster and state bit for bit, arrivals under way between the calls."""
    cfg, raster, st = _case(n, batch, max_delay, classes)
    sim = _sim(cfg, batch, resident_trials=True, fused=batch >= 8)
    outs = [sim.run(50), sim.run(100)]
    assert sim._trials is not None
    _same(sim, outs, raster, st)


PAIRS = ((0, 1), (2, 3), (1, 3), (0, 0), (0, 3), (2, 2), (1, 2))


@pytest.mark.parametrize("n,batch,max_delay,classes,span,four", [
    (65, 3, 6, None, None, 2), (64, 64, 1, 3, None, 0), (1010, 33, 4, None, 1024, 5), (1025, 5, 5, 7, 1088, 3), (1921, 12, 4, None, 1920, 97),
    (1920, 64, 5, 11, 1920, 0), (4100, 16, 3, 5, 1408, 1)])
def test_only_receptors_in_use_have_sums(n, batch, max_delay, classes, span, four):
    """One or two of the four receptors in any combination, every `four`-th neuron with all four, one neuron to a thread and
    two, a last workgroup of one neuron: raster and state bit for bit, over two calls in the form, one with the per-step record and one
    with the driver that takes its place."""
    cfg, _, _ = _case(n, batch, max_delay, classes, steps=200)
    for k in ("rec_src", "inp_src"):
        indptr, indices, w, d, r = cfg[k]
        some = np.asarray(PAIRS, np.uint8)[indices % len(PAIRS), r & 1]
        cfg[k] = indptr, indices, w, d, np.where(indices % four == four - 1, r, some).astype(np.uint8) if four else some
    st = orc.new_state(n, batch, np.float32)
    raster = orc.simulate(st, orc.precompute(cfg["par"], 1.0), 1.0, 200, batch=batch, class_id=cfg["class_id"],
                          ring=np.zeros((cfg["L"], 4, n * batch), np.float32), rec=cfg["rec_src"], inp=cfg["inp_src"],
                          in_ptr=cfg["in_ptr"], in_events=cfg["in_events"], i_ext=cfg["i_ext"], raster=True)["raster"]
    sim = _sim(cfg, batch, resident_trials=True, fused=batch >= 8)
    if span:
        sim._trials.update(span=span, groups=-(-n // span), ways=min(batch, 256 // -(-n // span)), list=400)
    sim._trials["few"] = True
    outs = [sim.run(50), sim.run(60), sim.run(70, save_state=True)]
    assert sim._trials["extra"] > 0 if four else sim._trials["extra"] == 0
    outs.append(sim.run(20))
    assert sim._trials is None
    _same(sim, outs, raster, st)


@pytest.mark.parametrize("how", ["short", "record", "ring"])
@pytest.mark.parametrize("batch,fused", [(6, False), (16, True), (20, True)])
def test_gives_way_to_the_other_drivers_with_arrivals_under_way(batch, fused, how):
    """A short call, one that asks for more than spike bits, a look at the ring: the launch-per-step driver goes on with
    what the calls before left under way, repeated input events included."""
    cfg, raster, st = _case(900, batch, 5, in_rate=150.0)
    sim = _sim(cfg, batch, resident_trials=True, fused=fused, **(dict(expected_rate_hz=40.0) if batch == 20 else {}))
    assert (sim.fuse_table is not None) == fused and sim.in_duplicates and sim.fuse_rereads == (batch == 20)
    outs = [sim.run(70)]
    if how == "ring":
        assert float(sim.ring.abs().sum()) > 0 or fused
        outs += [sim.run(80)]
    elif how == "short":
        outs += [sim.run(1), sim.run(2), sim.run(77)]
    else:
        outs += [sim.run(40, save_state=True), sim.run(40, record_cap=100000)]
    assert sim._trials is None
    _same(sim, outs, raster, st)


@pytest.mark.parametrize("n,batch,classes,stretch", [(63, 2, None, None), (64, 64, 3, None), (65, 5, None, 32), (1025, 20, 7, 40), (2100, 16, None, None)])
def test_per_step_record_equals_the_launch_per_step_drivers(monkeypatch, n, batch, classes, stretch):
    """Potentials and flags in the order [step][neuron][trial], over two calls, in one stretch or several: the bits that the
    other driver records; then that driver goes on."""
    cfg, raster, st = _case(n, batch, 4, classes)
    if stretch:
        monkeypatch.setattr(simulator, "TRIALS_SAVE_BYTES", 5 * n * batch * stretch)
    got = []
    for kw in (dict(resident_trials=True), dict(resident_trials=False)):
        sim = _sim(cfg, batch, fused=batch >= 8, **kw)
        a, b = sim.run(100, save_state=True), sim.run(40, save_state=True)
        assert (sim._trials is not None) == kw["resident_trials"]
        assert a["saved"]["step0"] == 0 and b["saved"]["step0"] == 100
        _same(sim, [a, b, sim.run(10, save_state=True)], raster, st)
        got.append([x[k] for x in (a["saved"], b["saved"]) for k in ("v", "flags")])
    assert got[0][1].any() and int(got[0][1].max()) <= 7
    for x, y in zip(*got):
        assert torch.equal(x, y)


@pytest.mark.parametrize("batch,fused", [(6, False), (12, True), (16, True)])
def test_beginning_anew_leaves_nothing_under_way(batch, fused):
    """State, ring, history and step set back after calls with resident trials: the run from rest once more, without the
    arrivals that were under way."""
    cfg, raster, st = _case(900, batch, 5, in_rate=150.0)
    sim = _sim(cfg, batch, resident_trials=True, fused=fused)
    rest = {k: getattr(sim.state, k).clone() for k in STATE}
    sim.run(70)
    for t in (sim.ring, sim.work_bits) + ((sim.fuse_any,) if fused else ()):
        t.zero_()
    for k in STATE:
        getattr(sim.state, k).copy_(rest[k])
    sim.step = 0
    _same(sim, [sim.run(31), sim.run(119)], raster, st)


def test_input_lists_replaced_between_calls():
    """Lists that say nothing was emitted in the steps behind take the last step's events back at the batches where the
    separate pull launches read them again (20), and leave them alone elsewhere (16)."""
    for batch in (16, 20):
        cfg, _, _ = _case(900, batch, 5, in_rate=150.0)
        results = []
        for kw in (dict(resident_trials=False), dict(resident_trials=True)):
            sim = _sim(cfg, batch, fused=True, expected_rate_hz=40.0, **kw)
            a = sim.run(60)
            ptr = torch.as_tensor(cfg["in_ptr"]).clone()
            events = torch.as_tensor(cfg["in_events"])[int(ptr[60]):]
            sim.set_input_events(np.concatenate([np.zeros(60, np.int64), (ptr[60:] - ptr[60]).numpy()]), events.numpy())
            b = sim.run(90)
            sim.check()
            results.append((torch.cat([a["bits"], b["bits"]]).cpu().numpy(), sim.state.to_numpy()))
        np.testing.assert_array_equal(results[0][0], results[1][0])
        for k in STATE:
            np.testing.assert_array_equal(results[0][1][k], results[1][1][k], err_msg=k)


def test_replaced_lists_mean_what_they_mean_to_separate_pull_launches():
    """At batches that do not divide 64 the fused form takes the place of separate pull launches, which read a call's first step
    from the step before it once more: lists that no longer name that step's events take them back in either form."""
    cfg, _, _ = _case(900, 20, 5, in_rate=150.0)
    results = []
    for kw in (dict(fused=False, pull=True, resident_trials=False), dict(fused=True), dict(fused=True, resident_trials=True)):
        sim = _sim(cfg, 20, expected_rate_hz=40.0, **kw)
        assert (sim.pull_inp_table is None) == kw["fused"] and sim.fuse_rereads
        a = sim.run(60)
        ptr = cfg["in_ptr"]
        sim.set_input_events(np.concatenate([np.zeros(60, np.int64), ptr[60:] - ptr[60]]), cfg["in_events"][ptr[60]:])
        b = sim.run(90)
        sim.check()
        results.append((torch.cat([a["bits"], b["bits"]]), sim.state.to_numpy()))
    for bits, state in results[1:]:
        assert torch.equal(bits, results[0][0])
        for k in STATE:
            np.testing.assert_array_equal(state[k], results[0][1][k], err_msg=k)


@pytest.mark.parametrize("ends,kw", [
    ((60, 84, 150), dict(resident_trials=False, fused=True)), ((60, 84, 150), dict(resident_trials=False, fused=False, pull=False)),
    ((60, 100, 150), dict(resident_trials=True, fused=True)), ((60, 84, 150), dict(resident_trials=True, fused=True)),
    ((60, 84, 150), dict(resident_trials=True, fused=False))])
@pytest.mark.parametrize("batch", [12, 16])
def test_repeated_ids_under_way_outlive_their_lists(batch, ends, kw):
    """Lists with repeated ids up to the last step, then lists without any, then lists with some again, none of which names
    the events of the steps behind it: what the first lists' repeats still had under way arrives when it is due, and only then.
    The oracle's run is one run over all events."""
    cfg, raster, st = _case(900, batch, 5, in_rate=150.0, once=ends[:2])
    ptr, events = cfg["in_ptr"], cfg["in_events"]

    def repeats(a, b):
        return any(np.unique(events[ptr[t]:ptr[t + 1]]).size < ptr[t + 1] - ptr[t] for t in range(a, b))

    assert repeats(ends[0] - 1, ends[0]) and not repeats(*ends[:2]) and repeats(ends[1], ends[2])
    sim = _sim(cfg, batch, **kw)
    assert not sim.fuse_rereads
    outs, at = [], 0
    for end in ends:
        sim.set_input_events(np.concatenate([np.zeros(at, np.int64), ptr[at:end + 1] - ptr[at]]), events[ptr[at]:ptr[end]])
        outs.append(sim.run(end - at))
        at = end
    assert (sim._trials is not None) == (kw["resident_trials"] and ends[1] - ends[0] >= simulator.TRIALS_MIN_STEPS)
    _same(sim, outs, raster, st)


@pytest.mark.parametrize("small", [2.0 ** -12 / 3.0, 2.0 ** -38])
@pytest.mark.parametrize("batch,kw,calls", [
    (12, dict(resident_trials=False, fused=True), (150,)), (16, dict(resident_trials=False, fused=True), (150,)),
    (5, dict(resident_trials=True), (60, 90)), (5, dict(resident_trials=True), (60, 20, 70)), (20, dict(resident_trials=True, fused=True), (60, 20, 70))])
def test_small_weights_keep_their_bits(batch, kw, calls, small):
    """Two receptors of ordinary weights, two of weights a 12,000th (all 24 bits in use) or 2^-38 as large: a weight below 2^-9
    may have bits under 2^-32, one below 2^-32 has no others.  y1 agrees to a few of its last places, receptor by receptor."""
    cfg, raster, st = _case(900, batch, 5, small=small)
    sim = _sim(cfg, batch, **kw)
    outs = [sim.run(n) for n in calls]
    sim.check()
    np.testing.assert_array_equal(np.concatenate([sim.raster(o["bits"]).cpu().numpy() for o in outs]), raster)
    y1 = sim.state.to_numpy()["y1"]
    for r in range(4):
        size = np.abs(st["y1"][r]).max()
        assert size > 0
        # a sum of up to 16 fp32 addends, each addition within half a last place of the sum of their sizes
        np.testing.assert_allclose(y1[r], st["y1"][r], rtol=16 * 2.0 ** -24, atol=16 * 2.0 ** -24 * size, err_msg=str(r))
    assert sim.sum_shift == fixed_point_shift([sim.rec, sim.inp], sim.n) > 0


def test_weights_that_fixed_point_does_not_hold_stay_pushed():
    """2^24 pA beside 2^-40 pA: more than 63 bits.  Left to itself the simulator adds such weights in fp32, as before."""
    for batch in (5, 12):
        cfg, raster, st = _case(900, batch, 5, small=2.0 ** -40)
        auto = dict(i_ext=cfg["i_ext"], ring_slots=cfg["L"], expected_rate_hz=4.0)
        held = Glif3Simulator(cfg["n"], cfg["par"], 1.0, batch=batch, rec=cfg["rec_src"], inp=cfg["inp_src"], **auto)
        assert held._trials is not None and held.sum_shift == 10
        indptr, indices, w, d, r = cfg["rec_src"]
        far = np.where(r == 0, w * np.float32(2.0 ** 24), w)
        sim = Glif3Simulator(cfg["n"], cfg["par"], 1.0, batch=batch, rec=(indptr, indices, far, d, r), inp=cfg["inp_src"], **auto)
        assert sim._trials is None and sim.fuse_table is None


def test_more_rows_in_a_step_than_the_list_holds():
    """Identical neurons driven alike fire together: 5,000 rows in one step against a list of 2,000 places."""
    n, batch, steps = 5000, 4, 60
    rng = np.random.default_rng(21)
    par = synthetic.random_cells(rng, 1)
    cls = np.zeros(n, np.int32)
    src, tgt = rng.integers(0, n, 40000), rng.integers(0, n, 40000)
    rec = _quarter(tuple(t.cpu().numpy() for t in (lambda s: (s.indptr, s.indices, s.weights, s.delays, s.receptors))(
        ops.SynapseTable.from_edges(src, tgt, np.ones(40000, np.float32), rng.integers(1, 6, 40000), rng.integers(0, 4, 40000), n, n))))
    i_ext = np.full(n * batch, 900.0, np.float32)
    st = orc.new_state(n, batch, np.float32)
    want = orc.simulate(st, orc.precompute(par, 1.0), 1.0, steps, batch=batch, class_id=cls, ring=np.zeros((6, 4, n * batch), np.float32),
                        rec=rec, i_ext=i_ext, raster=True)
    assert want["raster"].reshape(steps, n, batch)[:, :, 0].sum(1).max() > 4000
    sim = Glif3Simulator(n, par, 1.0, batch=batch, class_id=cls, rec=rec, i_ext=i_ext, resident=False, resident_trials=True)
    sim._trials["list"] = 2000
    _same(sim, [sim.run(steps)], want["raster"], st)


def _wide_case(n, max_delay, classes, steps, seed):
    """One trial of more neurons than the compute units have threads: sparse, driven by currents and repeated input events."""
    rng = np.random.default_rng(seed)
    par = synthetic.random_cells(rng, classes or n)
    cls = rng.integers(0, classes, n).astype(np.int32) if classes else None
    tables, n_in = [], 500
    for rows, nnz in ((n, 12 * n), (n_in, 2 * n)):
        t = ops.SynapseTable.from_edges(rng.integers(0, rows, nnz), rng.integers(0, n, nnz), rng.normal(0, 20, nnz).astype(np.float32),
                                        rng.integers(1, max_delay + 1, nnz), rng.integers(0, 4, nnz), rows, n)
        tables.append(_quarter(tuple(x.cpu().numpy() for x in (t.indptr, t.indices, t.weights, t.delays, t.receptors))))
    counts = rng.poisson(6.0, steps)
    counts[::5] = 0
    events = np.concatenate([np.sort(rng.integers(0, 40, c)) for c in counts]).astype(np.int32)
    ptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    i_ext = rng.uniform(0.0, 900.0, n).astype(np.float32)
    st = orc.new_state(n, 1, np.float32)
    orc.set_threads(orc.max_threads())
    want = orc.simulate(st, orc.precompute(par, 1.0), 1.0, steps, class_id=cls, ring=np.zeros((max_delay + 1, 4, n), np.float32),
                        rec=tables[0], inp=tables[1], in_ptr=ptr, in_events=events, i_ext=i_ext, raster=True)
    sim = Glif3Simulator(n, par, 1.0, class_id=cls, rec=tables[0], inp=tables[1], i_ext=i_ext, ring_slots=max_delay + 1,
                         resident_trials=True)
    sim.set_input_events(ptr, events)
    return sim, want["raster"], st


@pytest.mark.parametrize("n,max_delay,classes,places", [(262145, 1, 5, None), (300001, 6, None, None), (491520, 5, 111, 2000)])
def test_more_neurons_than_threads(n, max_delay, classes, places):
    """Two neurons to a thread: smallest and largest network, a last workgroup of a few neurons, a list of rows that a step
    outgrows, arrivals under way between two calls.  Sums of quarters are exact in fp32: bit for bit the oracle's."""
    sim, raster, st = _wide_case(n, max_delay, classes, 70, n)
    assert sim._trials is not None and not sim.res_span
    if places:
        assert raster.sum(1).max() > places
        sim._trials["list"] = places
    _same(sim, [sim.run(33), sim.run(37)], raster, st)
    assert sim._trials is not None


@pytest.mark.parametrize("how", ["short", "record", "ring"])
def test_more_neurons_than_threads_give_way(how):
    sim, raster, st = _wide_case(270001, 4, 7, 60, 5)
    outs = [sim.run(35)]
    if how == "ring":
        assert float(sim.ring.abs().sum()) > 0
    outs += [sim.run(3), sim.run(22)] if how == "short" else [sim.run(25, save_state=how == "record", record_cap=10 ** 6)]
    assert sim._trials is None
    _same(sim, outs, raster, st)


@pytest.mark.parametrize("batch,fused", [(6, False), (16, True)])
def test_buffers_given_up_wait_for_the_stream_that_reads_them(batch, fused):
    """Built and first run on the default stream, run and left for the other driver on a second one: the memory of the form's
    tables and of what it handed over is not given out again on the first stream while the second still works."""
    cfg, raster, st = _case(900, batch, 5, in_rate=150.0)
    sim = _sim(cfg, batch, resident_trials=True, fused=fused)
    outs = [sim.run(40)]
    own = torch.cuda.Stream()
    own.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    with torch.cuda.stream(own):
        torch.cuda._sleep(100_000_000)
        outs.append(sim.run(40))
        given_up = [(t.data_ptr(), t.numel() * t.element_size()) for t in (sim._trials[k] for k in ("ring", "hist", "seg", "packed"))]
        outs += [sim.run(20), sim.run(20), sim.run(30)]
        done = torch.cuda.Event()
        done.record()
    assert sim._trials is None and sim._left_ring is None
    others = [torch.empty(size, dtype=torch.uint8, device="cuda") for _, size in given_up for _ in range(4)]
    assert not done.query()
    for at, size in given_up:
        assert all(o.data_ptr() + o.numel() <= at or at + size <= o.data_ptr() for o in others)
    torch.cuda.synchronize()
    _same(sim, outs, raster, st)


@pytest.mark.parametrize("batch,fused", [(6, False), (16, True)])
def test_arrivals_handed_over_under_capture_come_once(batch, fused):
    """A call captured behind one with resident trials goes on with the other driver; what the first had under way arrives in the
    first replay and in no other.  Every replay against the same call made again by a simulator without the form."""
    cfg, _, _ = _case(900, batch, 5, in_rate=150.0)
    first, again = 40, 40           # (a whole number of rounds of the fused form's histories)
    sim, other = _sim(cfg, batch, resident_trials=True, fused=fused), _sim(cfg, batch, resident_trials=False, fused=fused)
    sim.run(first)
    other.run(first)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sim.run(again)
    assert sim._trials is None and sim.step == first + again
    for k in range(4):
        graph.replay()
        other.step = first
        want = other.run(again)
        torch.cuda.synchronize()
        assert torch.equal(out["bits"], want["bits"]), k
        for name in STATE:
            assert torch.equal(getattr(sim.state, name), getattr(other.state, name)), (k, name)


def test_a_barrier_that_gives_up_is_reported():
    cfg, _, _ = _case(700, 4, 5)
    sim = _sim(cfg, 4, resident_trials=True)
    sim.res_sync[1] = 1            # as a workgroup whose wait ran out leaves it
    sim.run(40)
    with pytest.raises(RuntimeError):
        sim.check()


@pytest.mark.parametrize("save", [False, True])
def test_no_memory_for_the_tables(monkeypatch, save):
    """Chosen by the constructor: the call runs with the driver that the simulator holds beside it.  Insisted on: the error."""
    def full(self):
        raise torch.OutOfMemoryError("no memory")

    monkeypatch.setattr(Glif3Simulator, "_setup_trials", full)
    cfg, raster, st = _case(900, 5, 5)
    kw = dict(batch=5, class_id=cfg["class_id"], rec=cfg["rec_src"], inp=cfg["inp_src"], i_ext=cfg["i_ext"], ring_slots=cfg["L"])
    sim = Glif3Simulator(cfg["n"], cfg["par"], 1.0, **kw)
    assert sim._trials is not None
    sim.set_input_events(cfg["in_ptr"], cfg["in_events"])
    outs = [sim.run(50, save_state=save), sim.run(100, save_state=save)]
    assert sim._trials is None and all((o["saved"] is not None) == save for o in outs)
    _same(sim, outs, raster, st)
    sim = _sim(cfg, 5, resident_trials=True)
    with pytest.raises(torch.OutOfMemoryError):
        sim.run(50, save_state=save)


def test_what_does_not_fit_is_refused():
    assert resident_trials_plan(300000, 8, 6, 256) is None and resident_trials_plan(1000, 65, 6, 256) is None
    cfg, _, _ = _case(200, 2, 3)
    with pytest.raises(ValueError):
        Glif3Simulator(cfg["n"], cfg["par"], 1.0, batch=2, inp=cfg["inp_src"], resident=False, resident_trials=True)


def test_resident_false_keeps_the_launches_and_auto_takes_trials_for_training():
    """resident=False is one launch per step (or two), whatever a step would cost otherwise; a training simulator of a batch that
    leaves ``resident`` alone, or asks for them, runs its trials resident, with the same record, and the backward pass takes it."""
    batch = 12
    cfg, _, _ = _case(700, batch, 3)
    want = None
    for kw, trials in ((dict(resident=False), False), (dict(resident_trials=False), False), (dict(), True),
                       (dict(resident=False, resident_trials=True), True)):
        sim = Glif3Simulator(cfg["n"], cfg["par"], 1.0, batch=batch, class_id=cfg["class_id"], rec=cfg["rec_src"], inp=cfg["inp_src"],
                             i_ext=cfg["i_ext"], ring_slots=cfg["L"], **kw)
        sim.set_input_events(cfg["in_ptr"], cfg["in_events"])
        assert (sim._trials is not None) == trials, kw
        out = sim.run(64, save_state=True)
        assert (sim._trials is not None) == trials, kw
        bptt = training.Glif3Bptt(sim)
        bptt.backward(out, dl_dz_const=torch.ones(sim.ne, device="cuda"))
        got = dict(bits=out["bits"], v=out["saved"]["v"], flags=out["saved"]["flags"])
        want = want or dict(got, d_rec_w=bptt.d_rec_w)
        for key in got:
            assert torch.equal(got[key], want[key]), (kw, key)
        assert float(bptt.d_rec_w.abs().max()) > 0.0
        # (the same adjoint; only sums of atomic additions in another order)
        assert float((bptt.d_rec_w - want["d_rec_w"]).norm()) <= 4e-6 * float(want["d_rec_w"].norm())


@pytest.mark.parametrize("stepwise", [False, True])
def test_the_backward_pass_refuses_the_record_of_a_run_that_gave_up(stepwise):
    """The abort word set from the host: the forward run does nothing, its record is whatever the memory held, and the backward pass
    says so instead of taking gradients from it.  The next run is right."""
    batch = 12
    cfg, _, _ = _case(300, batch, 3)
    sim = _sim(cfg, batch, resident_trials=True)
    bptt = training.Glif3Bptt(sim)
    backward = bptt.backward_stepwise if stepwise else bptt.backward
    dl_dz = torch.ones(sim.ne, device="cuda")
    backward(sim.run(40, save_state=True), dl_dz_const=dl_dz)
    bptt.zero()
    sim.res_sync[1] = 1
    with pytest.raises(RuntimeError, match="aborted"):
        backward(sim.run(40, save_state=True), dl_dz_const=dl_dz)
    assert float(bptt.d_rec_w.abs().max()) == 0.0
    backward(sim.run(40, save_state=True), dl_dz_const=dl_dz)
    assert int(sim.res_sync[1].item()) == 0 and bool(torch.isfinite(bptt.d_rec_w).all())


@pytest.mark.parametrize("whole", [True, False])
@pytest.mark.parametrize("n,batch,max_delay,classes,span", [
    (64, 64, 4, 3, None), (700, 20, 5, 7, None), (1025, 33, 1, None, 1024), (1025, 5, 5, 7, 1088), (1921, 12, 4, None, 1920), (4100, 8, 6, 5, 1408)])
def test_sums_of_32_and_of_64_bits(monkeypatch, n, batch, max_delay, classes, span, whole):
    """Weights in quarters of a pA: sums as 32-bit whole numbers of them, or in 64 bits where the weights are taken not to allow that.  One
    neuron to a thread and two, the per-step record, arrivals under way between calls and to the driver that takes its place."""
    cfg, _, _ = _case(n, batch, max_delay, classes, steps=200)
    if not whole:
        monkeypatch.setattr(simulator, "whole_numbers", lambda *a: None)
    st = orc.new_state(n, batch, np.float32)
    raster = orc.simulate(st, orc.precompute(cfg["par"], 1.0), 1.0, 200, batch=batch, class_id=cfg["class_id"],
                          ring=np.zeros((cfg["L"], 4, n * batch), np.float32), rec=cfg["rec_src"], inp=cfg["inp_src"],
                          in_ptr=cfg["in_ptr"], in_events=cfg["in_events"], i_ext=cfg["i_ext"], raster=True)["raster"]
    sim = _sim(cfg, batch, resident_trials=True, fused=batch >= 8)
    assert sim._trials.get("whole", 0) == (3 if whole else 0)      # multiples of 2^-2
    if span:
        sim._trials.update(span=span, groups=-(-n // span), ways=min(batch, 256 // -(-n // span)), list=400, few=not whole and span > 1024)
    outs = [sim.run(50), sim.run(60), sim.run(70, save_state=True)]
    assert sim._trials is not None
    outs.append(sim.run(20))
    assert sim._trials is None
    _same(sim, outs, raster, st)


def test_weights_that_32_bit_sums_take():
    n = 50
    rng = np.random.default_rng(1)

    def table(w, rows=n):
        return ops.SynapseTable.from_edges(rng.integers(0, rows, w.size), rng.integers(0, n, w.size), w.astype(np.float32),
                                           np.ones(w.size, np.int64), np.zeros(w.size, np.int64), rows, n)
    quarters = np.round(rng.normal(0, 20, 400)) / 4
    rec, inp = table(quarters), table(np.full(100, 2.0), 10)
    k, room, _ = simulator.whole_numbers(rec, inp, n)
    of_inputs = np.bincount(inp.indices.cpu().numpy(), minlength=n) * 2.0
    together = of_inputs + np.bincount(rec.indices.cpu().numpy(), np.abs(rec.weights.cpu().numpy()), n)
    assert k == 2 and (together.max() + room * of_inputs.max()) * 4 < 2 ** 30 <= (together.max() + (room + 1) * of_inputs.max()) * 4
    assert simulator.whole_numbers(rec, None, n)[0] == 2 and simulator.whole_numbers(table(np.zeros(3)), None, n)[0] == 0
    assert simulator.whole_numbers(table(np.array([2.0 ** -30])), None, n)[0] == 30
    for bad in ([2.0 ** -31], [np.nan], [np.inf, 1.0], [2.0 ** 31], [2.0 ** 20, 2.0 ** -11], np.full(100000, 2.0 ** 21)):
        assert simulator.whole_numbers(rec, table(np.array(bad)), n) is None
        assert simulator.whole_numbers(table(np.array(bad)), inp, n) is None
    # sums as large as they may come out as they are: every synapse of a neuron at once, either sign
    for sign in (1.0, -1.0):
        w = np.full(3, sign * 2.0 ** 28)
        src, tgt = np.arange(3), np.zeros(3, np.int64)
        one = ops.SynapseTable.from_edges(src, tgt, w.astype(np.float32), np.ones(3, np.int64), np.zeros(3, np.int64), 4, 4)
        tabs = tuple(t.cpu().numpy() for t in (one.indptr, one.indices, one.weights, one.delays, one.receptors))
        par = synthetic.random_cells(np.random.default_rng(2), 4)
        got = {}
        for trials in (True, False):
            sim = Glif3Simulator(4, par, 1.0, batch=2, rec=table_of(4), inp=tabs, resident=False, resident_trials=trials)
            assert not trials or sim._trials["whole"] == 1
            sim.set_input_events(np.concatenate([[0], np.full(40, 3)]).astype(np.int64), np.arange(3, dtype=np.int32) * 2)
            sim.run(40)
            sim.check()
            got[trials] = sim.state.to_numpy()
        for key in STATE:
            np.testing.assert_array_equal(got[True][key], got[False][key], err_msg=key)


def table_of(n):
    """A recurrent table of one synapse that carries nothing."""
    return (np.array([0] + [1] * n, np.int32), np.array([n - 1], np.int32), np.zeros(1, np.float32), np.ones(1, np.uint8), np.zeros(1, np.uint8))


def _heavy(cfg, weight):
    """An input source that never fires (the last), but could bring a neuron ``weight``."""
    indptr, indices, w, d, r = (a.copy() for a in cfg["inp_src"])
    assert indptr[-1] > indptr[-2]
    w[-1] = weight
    cfg["inp_src"] = indptr, indices, w, d, r
    last = cfg["n_in"] - 1
    batch = cfg["i_ext"].size // cfg["n"]
    keep = cfg["in_events"] // batch != last
    cfg["in_ptr"], cfg["in_events"] = np.concatenate([[0], np.cumsum(keep)])[cfg["in_ptr"]].astype(np.int64), cfg["in_events"][keep]


def test_many_repeated_events_leave_32_bit_sums_alone():
    """Hundreds of ids twice in a step: a sum takes one repeat of each where it has room for that of an id that reaches a neuron with all
    its inputs."""
    n, batch = 300, 8
    cfg, _, _ = _case(n, batch, 5, in_rate=400.0)
    _heavy(cfg, 2.0 ** 26)      # 2^28 of 2^30: room for two repeats of an id
    steps = np.repeat(np.arange(150), np.diff(cfg["in_ptr"]))
    repeats = np.bincount(steps[1:][(np.diff(cfg["in_events"]) == 0) & (np.diff(steps) == 0)], minlength=150)
    st = orc.new_state(n, batch, np.float32)
    raster = orc.simulate(st, orc.precompute(cfg["par"], 1.0), 1.0, 150, batch=batch, class_id=cfg["class_id"],
                          ring=np.zeros((cfg["L"], 4, n * batch), np.float32), rec=cfg["rec_src"], inp=cfg["inp_src"],
                          in_ptr=cfg["in_ptr"], in_events=cfg["in_events"], i_ext=cfg["i_ext"], raster=True)["raster"]
    sim = _sim(cfg, batch, resident_trials=True, fused=True)
    assert sim._trials["whole"] == 3 and sim._trials["room"] == 2 and sim.in_most_repeats == 1 and repeats.max() > 40
    outs = [sim.run(60), sim.run(90)]
    assert sim._trials["whole"] == 3
    _same(sim, outs, raster, st)


@pytest.mark.parametrize("n,batch,max_delay,span", [(300, 8, 3, None), (1025, 12, 5, 1088), (2100, 16, 1, None)])
def test_more_repeated_events_than_32_bit_sums_take(n, batch, max_delay, span):
    """A call with a step that repeats an id more often than there is room for: sums of 64 bits from there on, in the same form, with what
    the calls before left under way.  Calls before that step keep 32 bits, lists that hold it or not."""
    cfg, _, _ = _case(n, batch, max_delay, steps=200)
    _heavy(cfg, 2.0 ** 26)
    # an id five times in step 150: four repeats, room for two
    at = cfg["in_ptr"][150]
    assert cfg["in_ptr"][151] > at
    cfg["in_events"] = np.insert(cfg["in_events"], at, np.full(4, cfg["in_events"][at]))
    cfg["in_ptr"][151:] += 4
    st = orc.new_state(n, batch, np.float32)
    raster = orc.simulate(st, orc.precompute(cfg["par"], 1.0), 1.0, 200, batch=batch, class_id=cfg["class_id"],
                          ring=np.zeros((cfg["L"], 4, n * batch), np.float32), rec=cfg["rec_src"], inp=cfg["inp_src"],
                          in_ptr=cfg["in_ptr"], in_events=cfg["in_events"], i_ext=cfg["i_ext"], raster=True)["raster"]
    sim = _sim(cfg, batch, resident_trials=True, fused=True)
    assert sim._trials["whole"] == 3 and sim._trials["room"] == 2 and sim.in_most_repeats >= 4
    if span:
        sim._trials.update(span=span, groups=-(-n // span), ways=min(batch, 256 // -(-n // span)), list=400)
    outs = [sim.run(60), sim.run(90)]
    assert sim._trials["whole"] == 3
    outs.append(sim.run(50))
    assert sim._trials is not None and sim._trials["whole"] == 0
    _same(sim, outs, raster, st)


def test_repeated_events_where_64_bit_sums_do_not_fit(monkeypatch):
    """... then the driver that takes the form's place goes on, also where memory for the other tables is not there."""
    cfg, raster, st = _case(300, 8, 3)
    for how in ("no plan", "no memory"):
        sim = _sim(cfg, 8, resident_trials=True, fused=True)
        outs = [sim.run(60)]
        assert 0 < sim.in_most_repeats <= sim._trials["room"]
        sim._trials["room"] = sim.in_most_repeats - 1
        with monkeypatch.context() as m:
            if how == "no plan":
                m.setattr(simulator, "resident_trials_plan", lambda *a: None)
            else:
                sim._trials["insisted"] = False
                m.setattr(simulator, "trials_pay", lambda *a: True)
                m.setattr(sim, "_setup_trials", _no_memory)
            outs.append(sim.run(90))
        assert sim._trials is None
        _same(sim, outs, raster, st)


@pytest.mark.parametrize("which", ["rec", "inp"])
@pytest.mark.parametrize("scale", [0.3, 2.0 ** 12])
def test_weights_written_to_before_the_first_run(scale, which):
    """Weights that no longer are what 32-bit sums were chosen by, in place, behind the constructor: sums of 64 bits of the new ones."""
    cfg, _, _ = _case(700, 6, 4)
    sim = _sim(cfg, 6, resident_trials=True)
    assert sim._trials["whole"] == 3
    getattr(sim, which).weights.data.mul_(scale)
    key = which + "_src"
    indptr, indices, w, d, r = cfg[key]
    cfg[key] = indptr, indices, w * np.float32(scale), d, r
    new = _sim(cfg, 6, resident_trials=True)
    outs, want = ([s.run(50), s.run(100)] for s in (sim, new))
    assert sim._trials["whole"] == 0
    _same(sim, outs, np.concatenate([new.raster(o["bits"]).cpu().numpy() for o in want]), new.state.to_numpy())


def _no_memory():
    raise torch.OutOfMemoryError("none")
