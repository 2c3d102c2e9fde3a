"""The exchange by lists of fired neurons (sim_resident_lists_kernel) at the edges of what a list holds: 9, 19 and 39 neurons
of a workgroup, more (its ballots), all of them, and more input events in a step than the row list has room for; spans with one
wavefront of neurons, with all wavefronts but the reader's and with all sixteen."""
import numpy as np
import pytest
import torch

from bmtk_amd import simulator, synthetic
from bmtk_amd.layout import PAR

pytestmark = pytest.mark.gpu
N, STEPS = 3000, 70


def _network(seed):
    rng = np.random.default_rng(seed)
    n_in = 6000

    def table(n_src, per_row):
        indptr = np.arange(n_src + 1, dtype=np.int32) * per_row
        idx = rng.integers(0, N, n_src * per_row).astype(np.int32)
        w = (rng.integers(1, 200, idx.size) / 4.0).astype(np.float32)       # sums exact in fp32 in any order
        return (indptr, idx, w, rng.integers(1, 6, idx.size).astype(np.uint8), rng.integers(0, 4, idx.size).astype(np.uint8))

    per_step = rng.integers(0, 40, STEPS)
    per_step[7], per_step[21] = 5000, 300
    events = [np.sort(rng.integers(0, n_in, c)) for c in per_step]
    ptr = np.concatenate([[0], np.cumsum(per_step)]).astype(np.int64)
    return synthetic.random_cells(rng, N), table(N, 40), table(n_in, 7), ptr, np.concatenate(events).astype(np.int32)


def _start(par, span, seed):
    """Potentials above threshold for a chosen number of neurons of every workgroup: they fire in the first step."""
    rng = np.random.default_rng(seed)
    u = np.zeros(N, np.float32)
    counts = [0, 1, 4, 5, 9, 10, 14, 19, 20, 34, 38, 39, 40, 64, span]
    for g, e0 in enumerate(range(0, N, span)):
        mine = min(span, N - e0)
        pick = e0 + rng.permutation(mine)[:min(mine, counts[(g + seed) % len(counts)])]
        u[pick] = (par[PAR["V_TH"]] - par[PAR["E_L"]])[pick] * 3.0
    return u


@pytest.mark.parametrize("form", ["bits", "record", "shared_record", "probes"])
@pytest.mark.parametrize("span", [64, 960, 1024])
def test_lists_at_their_edges_equal_per_step_launches(span, form, monkeypatch):
    for seed in ((0, 5) if span == 64 else (8, 11, 12, 14)):
        par, rec, inp, ptr, events = _network(seed)
        u = _start(par, span, seed)

        def run(resident):
            monkeypatch.setattr(simulator, "resident_span", lambda *a, **k: span)
            sim = simulator.Glif3Simulator(N, par, 1.0, rec=rec, inp=inp, u_init=u, resident=resident)
            assert not resident or (sim.res_groups == -(-N // span) and sim.res_fired is not None)
            sim.set_input_events(ptr, events)
            if form == "probes":
                sim.set_probes(np.arange(0, N, 7), every=2)
            cap, ways = (N * STEPS * 256 if form == "record" else N * STEPS * 2), (256 if form == "record" else 2)
            out = [sim.run(k, record_cap=cap if "record" in form else 0, record_ways=ways if "record" in form else None)
                   for k in (1, 30, STEPS - 31)]
            st = sim.state
            got = dict(bits=torch.cat([o["bits"] for o in out]), V=st.V, y1=st.y1, y2=st.y2, asc=st.asc, ref=st.ref)
            if "record" in form:
                recs = [sim.collect_record(o["record"], sort_scale=1.0) for o in out]
                assert not any(r["overflow"] for r in recs)
                for key in ("step", "elem", "frac"):
                    got[key] = torch.cat([r[key] for r in recs])
            if form == "probes":
                got["probe"] = torch.cat([o["probe"]["v"] for o in out])
            sim.check()
            return got

        want, got = run(False), run(True)
        assert int(want["bits"].ne(0).sum()) > 50
        for key in want:
            assert torch.equal(want[key], got[key]), (seed, key)


@pytest.mark.parametrize("span,places,save", [(64, 2000, False), (64, 64, False), (832, 700, True), (960, 2000, False), (1024, 2000, True),
                                              (1024, 64, False)])
def test_lists_of_trials_side_by_side_at_their_edges(span, places, save, monkeypatch):
    """The same in the form with resident trials, five of them two at a time; `places` 64 leaves the row list no room at all."""
    batch = 5
    par, rec, inp, ptr, events = _network(3)
    rec, inp = [t[:3] + (np.minimum(t[3], 4),) + t[4:] for t in (rec, inp)]
    rng = np.random.default_rng(4)
    by_step = [np.sort(events[a:b] * batch + rng.integers(0, batch, b - a)).astype(np.int32) for a, b in zip(ptr[:-1], ptr[1:])]
    u = np.stack([_start(par, span, seed) for seed in (0, 5, 8, 12, 14)], axis=1).reshape(-1)
    groups = -(-N // span)

    def run(trials):
        monkeypatch.setattr(simulator, "resident_trials_plan", lambda *a: dict(span=span, groups=groups, ways=2, passes=3, list=places))
        sim = simulator.Glif3Simulator(N, par, 1.0, batch=batch, rec=rec, inp=inp, resident=False, resident_trials=trials)
        sim.state.V.copy_(torch.as_tensor(u))
        sim.set_input_events(ptr, np.concatenate(by_step))
        out = [sim.run(k, save_state=save) for k in (33, STEPS - 33)]
        st = sim.state
        got = dict(bits=torch.cat([o["bits"] for o in out]), V=st.V, y1=st.y1, y2=st.y2, asc=st.asc, ref=st.ref)
        if save:
            got.update(v=torch.cat([o["saved"]["v"] for o in out]), flags=torch.cat([o["saved"]["flags"] for o in out]))
        sim.check()
        assert (sim._trials is not None) == trials
        return got

    want, got = run(False), run(True)
    assert int(want["bits"].ne(0).sum()) > 50
    for key in want:
        assert torch.equal(want[key], got[key]), key


def test_a_reader_gives_up_cleanly(monkeypatch):
    """With a limit of one look in vain some reader gives up (workgroups do not start together): every wavefront leaves its loop,
    check() reports the run, and the next one is right."""
    par, rec, inp, ptr, events = _network(1)
    monkeypatch.setattr(simulator, "resident_span", lambda *a, **k: 64)

    def make():
        sim = simulator.Glif3Simulator(N, par, 1.0, rec=rec, inp=inp, resident=True)
        sim.set_input_events(ptr, events)
        return sim
    sim = make()
    sim.spin_limit = 1
    sim.run(40)
    gave_up = int(sim.res_sync[1].item()) != 0
    sim.spin_limit = 0
    sim.run(20)             # finds the word set, if it is, and does nothing
    if gave_up:
        with pytest.raises(RuntimeError, match="barrier"):
            sim.check()
        assert int(sim.res_sync[1].item()) == 0
    want = make()
    want.run(60)
    sim = make()
    sim.run(60)
    sim.check()
    assert torch.equal(want.state.V, sim.state.V)


@pytest.mark.parametrize("batch", [1, 5])
def test_crowded_steps_give_up_cleanly(batch, monkeypatch):
    """The same in steps that all wavefronts work off (39 neurons and more of a workgroup, more events than there is room for): the
    limit holds for the lists' further words too.  The run ends and is reported, or nobody had to wait and it is right."""
    par, rec, inp, ptr, events = _network(1)
    rec, inp = [t[:3] + (np.minimum(t[3], 4),) + t[4:] for t in (rec, inp)]
    ptr, events = np.arange(41, dtype=np.int64) * 3000, np.tile(np.arange(3000, dtype=np.int32) * batch, 40)
    monkeypatch.setattr(simulator, "resident_span", lambda *a, **k: 64)
    monkeypatch.setattr(simulator, "resident_trials_plan", lambda *a: dict(span=64, groups=47, ways=2, passes=3, list=64))
    bits = {}
    for limit in (0, 1):
        sim = simulator.Glif3Simulator(N, par, 1.0, batch=batch, rec=rec, inp=inp, resident=batch == 1, resident_trials=batch > 1)
        sim.state.V.copy_(torch.as_tensor(np.repeat(_start(par, 64, 8), batch)))
        sim.set_input_events(ptr, events)
        sim.spin_limit = limit
        bits[limit] = sim.run(40)["bits"]
        gave_up = int(sim.res_sync[1].item()) != 0
        assert not (gave_up and limit == 0)
        if gave_up:
            with pytest.raises(RuntimeError, match="barrier"):
                sim.check()
        else:
            assert torch.equal(bits[limit], bits[0])


@pytest.mark.parametrize("batch", [1, 5])
def test_scratch_on_any_32_bit_word(batch, monkeypatch):
    """res_sync is scratch of 32-bit words: the lists in it, whose words are of 64 bits, find their own alignment."""
    from bmtk_amd import _lib
    par, rec, inp, ptr, events = _network(2)
    rec, inp = [t[:3] + (np.minimum(t[3], 4),) + t[4:] for t in (rec, inp)]
    monkeypatch.setattr(simulator, "resident_span", lambda *a, **k: 64)
    bits = []
    for words in (0, 1):
        sim = simulator.Glif3Simulator(N, par, 1.0, batch=batch, rec=rec, inp=inp, resident=batch == 1, resident_trials=batch > 1)
        sim.res_sync = torch.zeros(words + _lib.RES_SYNC_WORDS, dtype=torch.int32, device="cuda")[words:]
        assert sim.res_sync.data_ptr() % 8 == 4 * words
        sim.set_input_events(ptr, events * batch)
        bits.append(sim.run(STEPS)["bits"])
        sim.check()
    assert int(bits[0].ne(0).sum()) > 50 and torch.equal(bits[0], bits[1])


@pytest.mark.parametrize("form", ["bits", "two_tables", "trials"])
@pytest.mark.parametrize("n", [4100, 6000, 12300])
def test_volleys_of_any_number_of_workgroups(n, form, monkeypatch):
    """Volleys (the ballots of some workgroups, the lists of others) of 65, 94 and 193 workgroups: 16, 8 and 4 threads share a
    workgroup's words, and rows come in one handing out or several.  Two tables: membrane probes rule out the joint one."""
    span, batch = 64, 3 if form == "trials" else 1
    rng = np.random.default_rng(n)
    indptr = np.arange(n + 1, dtype=np.int32) * 30
    idx = rng.integers(0, n, n * 30).astype(np.int32)
    rec = (indptr, idx, (rng.integers(1, 200, idx.size) / 4.0).astype(np.float32), rng.integers(1, 5, idx.size).astype(np.uint8),
           rng.integers(0, 4, idx.size).astype(np.uint8))
    par = synthetic.random_cells(rng, n)
    u = np.zeros((n, batch), np.float32)
    for b in range(batch):
        for g, e0 in enumerate(range(0, n, span)):
            mine = min(span, n - e0)
            pick = e0 + rng.permutation(mine)[:min(mine, (0, 3, 20, 39, 40, 52, 64)[(g + b) % 7])]
            u[pick, b] = (par[PAR["V_TH"]] - par[PAR["E_L"]])[pick] * 3.0
    i_ext = rng.uniform(0.0, 300.0, n * batch).astype(np.float32)
    groups = -(-n // span)
    monkeypatch.setattr(simulator, "resident_span", lambda *a, **k: span)
    monkeypatch.setattr(simulator, "resident_trials_plan", lambda *a: dict(span=span, groups=groups, ways=1, passes=3, list=2100))
    got = []
    for resident in (False, True):
        sim = simulator.Glif3Simulator(n, par, 1.0, batch=batch, rec=rec, i_ext=i_ext, resident=resident and batch == 1,
                                       resident_trials=resident and batch > 1)
        sim.state.V.copy_(torch.as_tensor(u.reshape(-1)))
        if form == "two_tables":
            sim.set_probes(np.arange(0, n, 11), every=3)
        out = sim.run(40)
        got.append(dict(bits=out["bits"], V=sim.state.V, y1=sim.state.y1, y2=sim.state.y2))
        sim.check()
    assert int(got[0]["bits"][0].ne(0).sum()) > groups // 2
    for key in got[0]:
        assert torch.equal(got[0][key], got[1][key]), key


@pytest.mark.parametrize("batch,places,form", [(1, 0, "bits"), (1, 0, "record"), (1, 0, "probes"), (5, 700, "bits"), (5, 8192, "bits")])
def test_steps_of_many_input_events(batch, places, form, monkeypatch):
    """Around the numbers of events that the reader lists (512), that one turn of the pulling threads takes beside them, that trials'
    rows have room for (half of `places` less 64), and far more of them, on any side of a step with few."""
    par, rec, inp, _, _ = _network(6)
    rec, inp = [t[:3] + (np.minimum(t[3], 4),) + t[4:] for t in (rec, inp)]
    inp = inp[:2] + (inp[2] / 32,) + inp[3:]
    n_in, rng = 6000, np.random.default_rng(8)
    edges = [0, 1, 63, 64, 255, 256, 257, 317, 318, 319, 511, 512, 513, 1023, 1025, 1407, 1408, 1409, 2048, 3297, 3809, 4063, 4064, 4065, 5999]
    per_step = np.array([e for e in edges] + [300, 300, 5000, 300, 2000, 4000, 2000] + list(rng.permutation(edges)))
    ptr = np.concatenate([[0], np.cumsum(per_step)]).astype(np.int64)
    events = np.concatenate([np.sort(rng.choice(n_in, c, replace=False)) for c in per_step]).astype(np.int32)
    monkeypatch.setattr(simulator, "resident_span", lambda *a, **k: 64)
    monkeypatch.setattr(simulator, "resident_trials_plan", lambda *a: dict(span=64, groups=47, ways=2, passes=3, list=places))
    got = []
    for resident in (False, True):
        sim = simulator.Glif3Simulator(N, par, 1.0, batch=batch, rec=rec, inp=inp, resident=resident and batch == 1,
                                       resident_trials=resident and batch > 1)
        sim.state.V.copy_(torch.as_tensor(np.repeat(_start(par, 64, 5), batch)))
        sim.set_input_events(ptr, events * batch + (2 if batch > 1 else 0))
        if form == "probes":
            sim.set_probes(np.arange(0, N, 7), every=2)
        out = sim.run(per_step.size, record_cap=N * per_step.size * 2 if form == "record" else 0)
        got.append(dict(bits=out["bits"], V=sim.state.V, y1=sim.state.y1, y2=sim.state.y2))
        sim.check()
    assert int(got[0]["bits"].ne(0).sum()) > 50
    for key in got[0]:
        assert torch.equal(got[0][key], got[1][key]), key


@pytest.mark.parametrize("rate,lists,ask", [(3.0, True, True), (100.0, True, True), (600.0, False, True), (3.0, False, False)])
def test_the_expected_rate_picks_the_exchange(rate, lists, ask, monkeypatch):
    """Lists unless more neurons of a workgroup are expected to fire in a step than they hold; the same results either way."""
    par, rec, inp, ptr, events = _network(4)
    monkeypatch.setattr(simulator, "resident_span", lambda *a, **k: 64)
    got = []
    for resident in (False, True):
        sim = simulator.Glif3Simulator(N, par, 1.0, rec=rec, inp=inp, u_init=_start(par, 64, 8), resident=resident, expected_rate_hz=rate,
                                       fired_lists=ask, **({} if resident else dict(pull=False)))
        assert not resident or (sim.res_fired is not None) == lists
        sim.set_input_events(ptr, events)
        got.append(sim.run(STEPS)["bits"])
        sim.check()
    assert torch.equal(got[0], got[1])
