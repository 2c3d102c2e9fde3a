"""Input event lists looked over on the device: what is refused, and the repeated ids listed apart."""
import numpy as np
import pytest

from bmtk_amd import synthetic
from bmtk_amd.simulator import Glif3Simulator

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sim():
    cfg = synthetic.small_glif3_network(n=100, n_in=400, steps=10, seed=1)
    return Glif3Simulator(cfg["n"], cfg["par"], cfg["h"], batch=8, rec=cfg["rec_src"], inp=cfg["inp_src"], class_id=cfg["class_id"],
                          resident=False, fused=True)


def _lists(counts, seed, repeats):
    rng = np.random.default_rng(seed)
    by_step = [np.sort(rng.choice(3200, c, replace=False)) for c in counts]
    for ids in by_step if repeats else ():
        if ids.size > 1:
            where = np.unique(np.concatenate([rng.integers(1, ids.size, 3), [ids.size - 1], [k for k in (1, 63, 64, 65, 255, 256, 257) if k < ids.size]]))
            for k in where:
                ids[k] = ids[k - 1]
    return np.concatenate([[0], np.cumsum(counts)]).astype(np.int64), np.concatenate(by_step + [np.zeros(0)]).astype(np.int32)


@pytest.mark.parametrize("counts", [[0], [], [1], [2, 0, 0, 1], [63, 64, 65, 0, 255, 256, 257, 1, 2], [0] * 500 + [1000, 3, 2900], [1] * 40000])
@pytest.mark.parametrize("repeats", [False, True])
@pytest.mark.parametrize("device", [False, True])
def test_repeated_ids_are_listed_apart(sim, counts, repeats, device):
    import torch
    ptr, events = _lists(counts, len(counts), repeats)
    again = np.concatenate([[False], events[1:] == events[:-1]])[:events.size]
    again[ptr[:-1][np.diff(ptr) > 0]] = False
    sim.set_input_events(*((torch.as_tensor(ptr, device="cuda"), torch.as_tensor(events, device="cuda")) if device else (ptr, events)))
    assert sim.in_duplicates == bool(again.any())
    if again.any():
        np.testing.assert_array_equal(sim.in_repeat_events.cpu().numpy(), events[again])
        np.testing.assert_array_equal(sim.in_repeat_ptr.cpu().numpy(), np.concatenate([[0], np.cumsum(again)])[ptr])
    else:
        assert sim.in_repeat_ptr is None and sim.in_repeat_events is None


@pytest.mark.parametrize("before", [0, 1, 5, 63, 200])
@pytest.mark.parametrize("times", [1, 2, 63, 64, 65, 66, 128, 129, 256, 257, 258, 700])
def test_how_often_a_step_repeats_one_id(sim, before, times):
    """An id that occurs `times` times behind `before` others, beside steps that repeat many ids once or twice."""
    import torch
    steps = [np.repeat(np.arange(300), 2), np.concatenate([np.arange(before), np.full(times, 1000), np.arange(1001, 1090)]), np.zeros(0, int),
             np.repeat(np.arange(90), 3), np.arange(90)]
    ptr = np.concatenate([[0], np.cumsum([s.size for s in steps])]).astype(np.int64)
    sim.set_input_events(torch.as_tensor(ptr, device="cuda"), torch.as_tensor(np.concatenate(steps).astype(np.int32), device="cuda"))
    assert sim.in_most_repeats == max(2, times - 1) and sim.in_repeat_events.numel() == 300 + times - 1 + 180


def test_lists_with_faults_are_refused(sim):
    import torch
    ptr, events = _lists([3, 0, 70, 300], 5, True)

    def device(p, e):
        return torch.as_tensor(p, device="cuda"), torch.as_tensor(e, device="cuda")
    sim.set_input_events(*device(ptr, events))
    kept = sim.in_ptr
    for at, value in ((0, 1), (1, 4), (2, -1), (4, 372), (4, 374), (3, 1 << 40)):
        p = ptr.copy()
        p[at] = value
        with pytest.raises(ValueError, match="inconsistent" if at != 1 else "inconsistent|ascending"):
            sim.set_input_events(*device(p, events))
    for at, value in ((0, -1), (372, 3200), (100, -5)):
        e = events.copy()
        e[at] = value
        with pytest.raises(ValueError, match="inconsistent"):
            sim.set_input_events(*device(ptr, e))
    for at in (2, 72, 73 + 64, 372):     # the last of a step, one behind 64 others
        e = events.copy()
        e[at] = e[at - 1] - 1
        with pytest.raises(ValueError, match="ascending"):
            sim.set_input_events(*device(ptr, e))
    for p, e in ((ptr.astype(np.int32), events), (ptr, events.astype(np.int64)), (ptr[:0], events), (ptr[:, None], events)):
        with pytest.raises(ValueError, match="inconsistent"):
            sim.set_input_events(*device(p, e))
    assert sim.in_ptr is kept


def test_tensors_in_host_memory_are_taken_to_the_device(sim):
    """... before the lists at hand give way to them: as arrays are."""
    import torch
    ptr, events = _lists([3, 0, 70, 300, 20, 1, 0, 0, 5, 9], 5, True)
    outs = []
    for make in (lambda a: torch.as_tensor(a, device="cuda"), torch.as_tensor):
        sim.set_input_events(make(ptr), make(events))
        assert sim.in_ptr.is_cuda and sim.in_events.is_cuda
        sim.step = 0
        for t in (sim.state.V, sim.state.asc, sim.state.y1, sim.state.y2, sim.state.ref, sim.ring, sim.work_bits, sim.fuse_any):
            t.zero_()
        outs.append((sim.run(10)["bits"], sim.state.y1.clone()))
    assert float(outs[0][1].abs().sum()) > 0
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("batch", [8, 12, 20, 64])
@pytest.mark.parametrize("repeats", [False, True])
def test_input_words_of_the_fused_form(batch, repeats):
    """Steps with no event, one, a wavefront's load and one more or less, and every id; the first and the last source; several runs of
    64 words: bit for bit what separate launches deliver."""
    import torch
    n_in = 1500
    ids = n_in * batch
    counts = [0, 1, 2, 0, 63, 64, 65, 4095, 4096, 4097, ids, ids - 1, 0, 0, 130, 1, 0, 300, 64, 0]
    cfg = synthetic.small_glif3_network(n=70, n_in=n_in, steps=len(counts), seed=batch, in_fanout=3, batch=batch, in_w_scale=3.0)
    for key in ("rec_src", "inp_src"):
        indptr, indices, w, d, r = cfg[key]
        cfg[key] = (indptr, indices, (np.round(w * 4.0) / 4.0 + np.sign(w) * 0.25).astype(np.float32), d, r)
    rng = np.random.default_rng(batch)
    steps = [np.sort(rng.choice(ids, min(c, ids), replace=False)) for c in counts]
    steps[1][:] = ids - 1
    steps[15][:] = 0
    if repeats:
        for s in steps:
            s[1::5] = s[:-1:5][:s[1::5].size]
    ptr = np.concatenate([[0], np.cumsum([s.size for s in steps])]).astype(np.int64)
    events = np.concatenate(steps).astype(np.int32)
    outs = []
    for fused in (True, False):
        sim = Glif3Simulator(cfg["n"], cfg["par"], cfg["h"], batch=batch, rec=cfg["rec_src"], inp=cfg["inp_src"], class_id=cfg["class_id"],
                             resident=False, pull=True, fused=fused)
        assert (sim.fuse_table is not None) == fused
        sim.set_input_events(ptr, events)
        bits = torch.cat([sim.raster(sim.run(k)["bits"]) for k in (1, 8, 11)])
        outs.append((bits, *(getattr(sim.state, k) for k in ("V", "asc", "y1", "y2", "ref"))))
    assert int(outs[0][0].sum()) > 0
    for a, b in zip(*outs):
        assert torch.equal(a, b)
