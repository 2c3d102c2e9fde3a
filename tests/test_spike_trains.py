"""Input spike sources: the reference's seeded Poisson vectors
(bmtk/tests/utils/reports/spike_trains/test_spikes_core.py:8-44) and the
spike_generator rules of bmtk/simulator/pointnet/pointnetwork.py:39-61."""
import json
import os

import numpy as np
import pytest

from bmtk_amd.spike_trains import PoissonSpikeGenerator, bin_spike_times, check_spike_times


@pytest.fixture(scope="module")
def gold(golden_dir):
    return json.load(open(os.path.join(golden_dir, "poisson_seed100.json")))


def _fixed(gold):
    g = gold["fixed"]
    psg = PoissonSpikeGenerator(population="test", seed=g["seed"])
    psg.add(node_ids=range(g["node_ids"]), firing_rate=g["firing_rate"], times=tuple(g["times"]))
    return psg


def test_psg_fixed_matches_reference_vectors(gold):
    g = gold["fixed"]
    psg = _fixed(gold)
    assert psg.populations == ["test"]
    assert psg.node_ids() == list(range(10))
    assert psg.n_spikes() == g["n_spikes"] and psg.n_spikes(population="test") == g["n_spikes"]
    np.testing.assert_allclose(psg.time_range(), g["time_range"])
    assert psg.to_dataframe().shape == (g["n_spikes"], 3)
    np.testing.assert_allclose(psg.get_times(node_id=0), g["node0"], atol=g["atol"])
    np.testing.assert_allclose(psg.get_times(node_id=9, population="test"), g["node9"], atol=g["atol"])


def test_psg_variable_continues_the_global_stream(gold):
    """The reference's second test passes seed=0.0, which does not reseed, so
    its expected trains depend on the stream position the first test left
    behind; reproducing them shows the block-drawing generator consumes
    exactly the draws a draw-by-draw loop would."""
    _fixed(gold)
    g = gold["variable"]
    times = np.linspace(g["t0"], g["t1"], g["n_times"])
    fr = np.exp(-np.power(times - 1.0, 2) / (2 * np.power(.5, 2))) * 5
    psg = PoissonSpikeGenerator(population="test", seed=g["seed"])
    psg.add(node_ids=range(g["node_ids"]), firing_rate=fr, times=times)
    assert psg.n_spikes() == g["n_spikes"]
    np.testing.assert_allclose(psg.time_range(), g["time_range"])
    np.testing.assert_allclose(psg.get_times(node_id=0), g["node0"], atol=g["atol"])
    np.testing.assert_allclose(psg.get_times(node_id=9), g["node9"], atol=g["atol"])


def test_block_drawing_equals_scalar_loop():
    np.random.seed(7)
    want = []
    for _ in range(25):
        c, ts = 0.25, []
        while True:
            c += -np.log(1.0 - np.random.uniform()) / 40.0
            if c > 2.0:
                break
            ts.append(c * 1000.0)
        want.append(ts)
    tail = np.random.uniform()
    psg = PoissonSpikeGenerator(seed=7)
    psg.add(node_ids=range(25), firing_rate=40.0, times=(0.25, 2.0))
    for i in range(25):
        np.testing.assert_allclose(psg.get_times(i), want[i], rtol=1e-14)
    assert np.random.uniform() == tail


def test_argument_errors():
    psg = PoissonSpikeGenerator(seed=1)
    with pytest.raises(ValueError):
        psg.add(node_ids=[0], firing_rate=-1.0)
    with pytest.raises(ValueError):
        psg.add(node_ids=[0], firing_rate=5.0, times=(1.0, 0.5))
    with pytest.raises(ValueError):
        psg.add(node_ids=[0], firing_rate=5.0, tau_ref=-1)
    with pytest.raises(ValueError):
        psg.add(node_ids=[0], firing_rate=[1.0, 2.0], times=[0.0, 1.0, 2.0])
    with pytest.raises(AttributeError):
        PoissonSpikeGenerator(output_units="hours")


def test_spike_time_rules():
    # empty / None are skipped, unsorted is sorted, non-positive raises
    assert check_spike_times(None) is None and check_spike_times([]) is None
    np.testing.assert_array_equal(check_spike_times([3.0, 1.0, 2.0]), [1.0, 2.0, 3.0])
    with pytest.raises(ValueError):
        check_spike_times([1.0, 0.0])
    with pytest.raises(ValueError):
        check_spike_times([-0.1, 2.0])


def test_binning_to_step_events():
    trains = [[1.0, 3.0], None, [3.0, 2.0, 7.6]]
    in_ptr, ev = bin_spike_times(trains, dt=1.0, n_steps=6, batch=2, trial=1)
    # stamp s -> emitted in step s-1; event id = source*batch + trial
    assert in_ptr.tolist() == [0, 1, 2, 4, 4, 4, 4]
    assert ev.tolist() == [1, 5, 1, 5]
    in_ptr, ev = bin_spike_times(trains, dt=1.0, n_steps=10)
    assert in_ptr[-1] == 5 and ev[in_ptr[7]:in_ptr[8]].tolist() == [2]
    # off-grid times are carried to the end of their step; on-grid times stay put
    in_ptr, ev = bin_spike_times([[0.2, 1.0, 1.01]], dt=1.0, n_steps=4)
    assert in_ptr.tolist() == [0, 2, 3, 3, 3]


def test_equals_and_subset_operators(tmp_path):
    """bmtk/tests/utils/reports/spike_trains/test_spikes_core.py:47-78."""
    from bmtk_amd.spike_trains import SpikeTrains
    st1 = SpikeTrains()
    st1.add_spikes(node_ids=0, population="V1", timestamps=[0.1, 0.2, 0.3, 0.4])
    st1.add_spikes(node_ids=1, population="V1", timestamps=[1.0])
    st2 = SpikeTrains()
    st2.add_spikes(node_ids=1, population="V1", timestamps=[1.0])
    st2.add_spikes(node_ids=0, population="V1", timestamps=[0.3, 0.2, 0.1, 0.4])
    assert st1 == st2 and st1 <= st2 and st1 >= st2 and not st1 != st2
    st2 = SpikeTrains()
    st2.add_spikes(node_ids=1, population="V1", timestamps=[1.0])
    st2.add_spikes(node_ids=0, population="V1", timestamps=[0.3, 0.2, 0.1, 0.4, 0.5])
    st2.add_spike(node_id=2, population="V1", timestamp=0.5)
    st2.add_spikes(node_ids=0, population="V2", timestamps=np.linspace(0.0, 1.0, 11))
    assert st1 != st2 and st1 < st2 and st2 > st1 and st1 <= st2 and st2 >= st1
    assert len(st2) == 18 and st2.n_spikes("V2") == 11 and sorted(st2.populations) == ["V1", "V2"]
    # through the two file formats and back
    for name in ("s.h5", "s.csv"):
        path = str(tmp_path / name)
        (st2.to_sonata if name.endswith("h5") else st2.to_csv)(path, sort_order="by_time")
        back = SpikeTrains.load(path)
        assert back == st2 and set(back.node_ids("V1")) == {0, 1, 2}
        assert len(list(back.spikes())) == 18
    assert SpikeTrains.from_sonata(str(tmp_path / "s.h5"), population="V2").populations == ["V2"]
    with pytest.raises(ValueError):
        SpikeTrains.load(str(tmp_path / "s.xyz"))


def test_gamma_generator_draws_and_statistics():
    """GammaSpikeGenerator (spike_trains.py:254-307; the reference holds no vector for it): the trains are exactly
    the running sums of SciPy's gamma draws on the seeded global stream, node by node, cut at tstop; the interval
    CV is 1/sqrt(a); a = 1 has Poisson statistics; bad arguments raise as in the reference."""
    from scipy.stats import gamma
    from bmtk_amd.spike_trains import GammaSpikeGenerator
    g = GammaSpikeGenerator(population="p", seed=77)
    g.add(node_ids=[3, 8], firing_rate=20.0, a=4.0, times=(0.5, 3.0))
    np.random.seed(77)
    for node in (3, 8):
        draws = gamma.rvs(4.0, loc=0, scale=1 / (4.0 * 20.0), size=round(2.5 * 20.0 * 1.5))
        t, want = 0.5, []
        for d in draws:
            t += d
            if t > 3.0:
                break
            want.append(t * 1000.0)
        np.testing.assert_allclose(g.get_times(node, "p"), want, rtol=0, atol=1e-9)
    g = GammaSpikeGenerator(population="p", seed=5)
    g.add(node_ids=range(200), firing_rate=10.0, a=9.0, times=(0.0, 5.0))
    isi = np.concatenate([np.diff(g.get_times(n, "p")) for n in range(200)])
    assert abs(isi.mean() - 100.0) < 2.0 and abs(isi.std() / isi.mean() - 1.0 / 3.0) < 0.02
    g = GammaSpikeGenerator(population="p", seed=6, output_units="s")
    g.add(node_ids=range(200), firing_rate=10.0, a=1.0, times=4.0)
    isi = np.concatenate([np.diff(g.get_times(n, "p")) for n in range(200)])
    assert abs(isi.std() / isi.mean() - 1.0) < 0.05 and g.time_range("p")[1] <= 4.0
    with pytest.raises(Exception, match="stationary"):
        g.add(node_ids=[0], firing_rate=[1.0, 2.0], a=2.0)
    with pytest.raises(ValueError):
        g.add(node_ids=[0], firing_rate=5.0, a=-1.0)
    with pytest.raises(ValueError):
        g.add(node_ids=[0], firing_rate=5.0, a=2.0, times=(2.0, 1.0))


@pytest.mark.parametrize("seed", range(8))
def test_binning_all_trains_at_once_equals_one_by_one(seed):
    rng = np.random.default_rng(seed)
    trains = [None if rng.random() < 0.2 else rng.uniform(0.01, 60, rng.integers(0, 9)) for _ in range(rng.integers(0, 40))]
    trains = [t.tolist() if t is not None and rng.random() < 0.3 else t for t in trains]
    dt, n_steps, batch, trial = float(rng.choice([0.1, 0.25, 1.0])), int(rng.integers(1, 90)), 3, 2
    in_ptr, ev = bin_spike_times(trains, dt, n_steps, batch=batch, trial=trial)
    want = [[] for _ in range(n_steps)]
    for j, st in enumerate(trains):
        st = check_spike_times(st)
        for t in [] if st is None else st:
            step = max(int(np.ceil(t / dt - 1e-6)), 1) - 1
            if step < n_steps:
                want[step].append(j * batch + trial)
    assert in_ptr.dtype == np.int64 and ev.dtype == np.int32 and in_ptr.size == n_steps + 1
    assert [ev[in_ptr[k]:in_ptr[k + 1]].tolist() for k in range(n_steps)] == [sorted(w) for w in want]


def test_the_first_train_that_is_not_valid_is_named():
    with pytest.raises(ValueError, match=r"\[0\. 2\.\]"):
        bin_spike_times([[1.0], [0.0, 2.0], [-1.0]], 1.0, 5)


def test_trains_of_every_form_are_binned_alike():
    """Arrays of several types, lists, tuples, columns and reversed views among the trains: what each gives by itself."""
    x = np.array([0.3, 2.0, 2.0, 7.5])
    forms = [x, None, list(x), x.astype(np.float32), np.array([1, 4]), [], x[:, None], x[::-1], tuple(x), np.zeros(0), np.array([3], np.uint8)]
    ptr, events = bin_spike_times(forms, 0.1, 60)
    alone = [bin_spike_times([None] * j + [np.asarray(f, np.float64).ravel()], 0.1, 60) if f is not None else None for j, f in enumerate(forms)]
    for t in range(60):
        want = sorted(int(e) for a in alone if a is not None for e in a[1][a[0][t]:a[0][t + 1]])
        assert events[ptr[t]:ptr[t + 1]].tolist() == want
    for bad in ([0.0], np.array([1.0, -2.0]), [2.0, 0.0, np.nan], np.zeros(2, np.float32)):
        with pytest.raises(ValueError, match="negative/zero"):
            bin_spike_times([x, None, bad, x], 0.1, 60)
