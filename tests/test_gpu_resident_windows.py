"""The single-workgroup form by windows: several steps between two barriers where spikes arrive late enough."""
import ctypes

import numpy as np
import pytest

from bmtk_amd import synthetic
from bmtk_amd.simulator import Glif3Simulator

pytestmark = pytest.mark.gpu


def _exact(table, longer):
    """Weights that are whole multiples of 1/4 pA (sums exact in fp32 in any order), delays lengthened."""
    indptr, indices, w, d, r = table
    w = np.where(w < 0, -1.0, 1.0) * np.maximum(1.0, np.round(np.abs(w) * 4.0)) / 4.0
    return indptr, indices, w.astype(np.float32), d.astype(np.int32) + longer, r


# neurons, delays from .. to, delay offset, steps of a window; inputs, their rate, driven neurons, calls; what is left out
CASES = [
    (450, 20, 20, 19, 6, 200, 40.0, 0.0, (1, 149, 250)),       # the ring's room sets the window
    (333, 10, 15, 0, 3, 200, 40.0, 0.0, (1, 149, 250)),        # no offset: delays say how long there is; a longer ring
    (333, 10, 15, 4, 3, 200, 40.0, 0.0, (1, 149, 250)),        # ... part of it an offset
    (70, 41, 42, 40, 8, 200, 40.0, 0.0, (1, 7, 8, 9, 375)),    # calls shorter than a window, and as long
    (65, 30, 32, 10, 8, 200, 40.0, 0.0, (400,)),               # ballots of two words, the second of one neuron
    (1, 6, 6, 0, 2, 200, 40.0, 0.0, (1, 149, 250)),
    (450, 6, 6, 5, 2, 200, 40.0, 0.0, (1, 149, 250)),
    (450, 5, 5, 4, 0, 200, 40.0, 0.0, (1, 149, 250)),          # too soon: single steps
    (512, 63, 64, 62, 6, 200, 40.0, 0.0, (1, 149, 250)),       # the longest offset with its ballots in LDS
    (300, 64, 65, 63, 8, 200, 40.0, 0.0, (1, 149, 250)),       # the shortest with ballots from the history
    (450, 300, 301, 299, 6, 200, 40.0, 0.0, (1, 299, 350)),    # arrivals that no window of the call before delivered
    (961, 12, 12, 11, 3, 200, 40.0, 0.0, (1, 149, 250)),       # every wavefront has neurons
    (1024, 12, 12, 11, 3, 600, 200.0, 0.8, (1, 199, 300)),     # volleys of 800 and 120 events a step: more rows than the lists hold
    (450, 20, 20, 19, 6, 600, 200.0, 0.8, (1, 199, 300)),
    (450, 80, 81, 79, 6, 600, 200.0, 0.8, (1, 199, 300)),      # ... with ballots from the history
    (100, 8, 9, 0, 2, 600, 1000.0, 0.8, (7, 8, 1, 9, 300)),
    (800, 12, 12, 11, 4, 200, 40.0, 0.0, (1, 149, 250)),       # the wavefronts with another role hold no neurons
    (850, 12, 12, 11, 3, 200, 40.0, 0.0, (1, 149, 250)),       # ... one of the three does
    (950, 12, 13, 11, 3, 200, 40.0, 0.0, (1, 149, 250)),       # ... two
    (300, 70, 72, 58, 7, 200, 40.0, 0.0, (1, 149, 250)),       # an offset that leaves the ballots in LDS room for four of twelve further steps
    (150, 70, 72, 58, 8, 200, 40.0, 0.8, (1, 3, 146, 250)),
    (450, 20, 20, 19, 6, 0, 40.0, 0.8, (1, 149, 250), "inputs"),
    (450, 80, 81, 79, 6, 0, 40.0, 0.8, (1, 149, 250), "inputs"),
    (450, 20, 20, 19, 6, 200, 40.0, 0.8, (1, 149, 250), "recurrent"),
    (950, 80, 81, 79, 3, 600, 200.0, 0.8, (1, 149, 250), "recurrent"),
    (450, 20, 20, 19, 6, 200, 40.0, 0.0, (1, 149, 250), "record"),
    (850, 12, 12, 11, 4, 200, 40.0, 0.8, (1, 149, 250), "record"),   # (a longer window in the place of the spike offsets)
    (1024, 80, 81, 79, 3, 600, 200.0, 0.8, (1, 149, 250), "record"),
]


@pytest.mark.parametrize("n,least,most,offset,window,n_in,rate,driven,calls,without", [(*c, None)[:10] for c in CASES])
def test_windows_equal_the_launch_per_step_driver(n, least, most, offset, window, n_in, rate, driven, calls, without):
    """Raster, spike record, probes, state and ring, bit for bit, over several calls; without a table of inputs or recurrent synapses, or without
    record and probes."""
    import torch
    cfg = synthetic.small_glif3_network(n=n, n_in=n_in, steps=sum(calls), seed=31 + n, in_w_scale=8.0, in_fanout=min(n, 60 if not driven else 30),
                                        in_rate=rate, p_conn=min(0.3, 40.0 / n), w_scale=2.0, max_delay=most - least + 1)
    for key in ("rec_src", "inp_src"):
        cfg[key] = _exact(cfg[key], least - 1)
    rng = np.random.default_rng(5)
    i_ext = np.where(np.arange(n) < driven * n, 3000.0, rng.uniform(0.0, 300.0, n)).astype(np.float32) if driven else None
    outs = {}
    for name, kw in (("step", dict(resident=False)), ("one", dict(resident=True))):
        sim = Glif3Simulator(n, cfg["par"], cfg["h"], class_id=cfg["class_id"], rec=None if without == "recurrent" else cfg["rec_src"],
                             inp=None if without == "inputs" else cfg["inp_src"], i_ext=i_ext, delay_offset=offset, ring_slots=most - offset + 1, **kw)
        if without != "inputs":
            # (steps without events behind the last call: the number of a step's events that the choice of a form goes by is small)
            sim.set_input_events(np.concatenate([cfg["in_ptr"], np.full(9 * sum(calls), cfg["in_ptr"][-1])]), cfg["in_events"])
        if without != "record":
            sim.set_probes(np.unique([0, n // 2, n - 1]), every=3)
        if name == "one":
            record = dict(zip(("step", "elem", "frac", "count"), torch.zeros(4, 2, device="cuda")))   # (only their being there counts)
            record = None if without == "record" else record
            assert sim.res_groups == 1 and sim.lib.bmtk_resident_window_steps(ctypes.byref(sim._struct(record=record))) == window
        got = []
        for steps in calls:
            out = sim.run(steps, record_cap=0 if without == "record" else 1 << 19)
            if without == "record":
                got.append([out["bits"]])
                continue
            rec = sim.collect_record(out["record"], sort_scale=1.0)
            assert not rec["overflow"]
            got.append([out["bits"], out["probe"]["v"], torch.stack([rec["time"], rec["elem"].double()], 1)])
        sim.check()
        outs[name] = dict(zip(("bits", "probe", "record"), (torch.cat(g).cpu().numpy() for g in zip(*got))), ring=sim.ring.cpu().numpy(),
                          **sim.state.to_numpy())
    assert np.unpackbits(outs["step"]["bits"].view(np.uint8)).sum() > 2 * n
    for key, want in outs["step"].items():
        np.testing.assert_array_equal(outs["one"][key], want, err_msg=key)
