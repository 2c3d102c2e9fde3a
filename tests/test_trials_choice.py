"""How the trials of a batch are laid out on the compute units, and when that is expected to pay."""
import numpy as np
import pytest

from bmtk_amd.layout import NREC
from bmtk_amd.simulator import RB_LDS_STATIC, RES_LDS_BYTES, lists_pay, resident_trials_plan, trials_bytes, trials_fit, trials_pay


@pytest.mark.parametrize("n,batch,slots", [(1, 2, 2), (64, 64, 6), (65, 3, 6), (5000, 16, 6), (20011, 20, 6), (51978, 32, 6), (230924, 8, 6),
                                           (245000, 2, 6), (2000, 64, 60), (120000, 16, 3)])
def test_plan_holds_every_neuron_and_trial(n, batch, slots):
    p = resident_trials_plan(n, batch, slots, 256)
    assert p["span"] % 64 == 0 and 64 <= p["span"] <= 1024 and p["groups"] == -(-n // p["span"])
    assert 8 * -(-p["ways"] * p["groups"] // 8) <= 256 and p["ways"] <= batch <= p["ways"] * p["passes"]
    assert (slots - 1) * NREC * 8 * p["span"] + 4 * p["list"] + RB_LDS_STATIC <= RES_LDS_BYTES and p["list"] >= 64


@pytest.mark.parametrize("n,batch,slots,share", [(51978, 32, 6, 0.2), (20011, 20, 6, 0.2), (230924, 8, 6, 0.0), (230924, 8, 6, 0.2), (5000, 64, 20, 1.0),
                                                 (120000, 16, 3, 2.0), (64, 2, 2, 2.0)])
def test_plan_with_the_receptors_in_use(n, batch, slots, share):
    """Third and fourth sums in the last neurons only: the workgroup that has most of them counts."""
    extra = np.zeros(n, np.int64)
    extra[n - int(n * share / 2):] = 2
    third = np.concatenate([[0], np.cumsum(extra)])
    p = resident_trials_plan(n, batch, slots, 256, third)
    sums = 2 * p["span"] + max(third[min(k + p["span"], n)] - third[k] for k in range(0, n, p["span"]))
    assert p["span"] % 64 == 0 and 64 <= p["span"] <= 1920 and p["groups"] == -(-n // p["span"])
    assert 8 * -(-p["ways"] * p["groups"] // 8) <= 256 and p["ways"] <= batch <= p["ways"] * p["passes"]
    assert (slots - 1) * 8 * sums + 4 * p["list"] + RB_LDS_STATIC <= RES_LDS_BYTES and p["list"] >= 2000
    old = resident_trials_plan(n, batch, slots, 256)
    assert p["passes"] <= old["passes"]


def test_plan_of_what_does_not_fit():
    for args in ((250000, 8, 6, 256), (1000, 1, 6, 256), (1000, 65, 6, 256), (10000, 8, 63, 64), (1000, 8, 6, 7)):
        assert resident_trials_plan(*args) is None


@pytest.mark.parametrize("n,batch,k,fused,pays", [(51978, 32, 1154, True, True), (230924, 8, 335, False, True), (20011, 20, 820, True, True),
                                                  (31000, 64, 160, True, True), (3000, 4, 200, False, True), (1500, 8, 400, True, True)])
def test_choice_agrees_with_measured_steps(n, batch, k, fused, pays):
    assert trials_pay(resident_trials_plan(n, batch, 6, 256), n, batch, n * k, False, 3.0, 1.0, fused) == pays


def test_many_launches_for_a_long_ring_do_not_pay():
    assert not trials_pay(resident_trials_plan(8000, 64, 60, 256), 8000, 64, 8000 * 100, False, 3.0, 1.0, True)


def test_tables_stay_in_proportion_to_the_network():
    for n, batch, n_in, k in ((230924, 8, 17400, 335), (400123, 1, 30000, 180), (51978, 32, 17400, 1154), (2000, 64, 500, 150), (491520, 1, 60000, 125)):
        assert trials_fit(resident_trials_plan(n, batch, 6, 256), n, batch, 6, n_in, n * k)
    # ten million virtual cells of a few synapses each: 10 GB of segment bounds beside 0.5 GB of synapses
    for n, batch in ((230924, 8), (400123, 1)):
        plan = resident_trials_plan(n, batch, 6, 256)
        assert trials_bytes(plan, n, batch, 6, 10 ** 7, 5 * 10 ** 7) > 9e9
        assert not trials_fit(plan, n, batch, 6, 10 ** 7, 5 * 10 ** 7)


def test_plan_of_one_trial_with_two_neurons_to_a_thread():
    for n, slots, span in ((262145, 6, 1088), (400123, 6, 1600), (491520, 6, 1920), (300001, 7, 1216)):
        p = resident_trials_plan(n, 1, slots, 256)
        assert p["span"] == span and p["groups"] == -(-n // span) <= 256 and p["ways"] == p["passes"] == 1
        assert (slots - 1) * NREC * 4 * span + 4 * p["list"] + RB_LDS_STATIC <= RES_LDS_BYTES and p["list"] >= 2000
    for args in ((262144, 1, 6, 256), (491521, 1, 6, 256), (491520, 1, 7, 256)):
        assert resident_trials_plan(*args) is None


def test_lists_are_exchanged_where_they_were_measured_to_pay():
    """(span, workgroups, Hz): lists against ballots behind a grid barrier, as measured; never ballots at the default rate."""
    for span, groups, rate, lists in ((960, 241, 20.8, True), (960, 241, 24.2, False), (960, 241, 27.8, False), (960, 241, 34.6, False),
                                      (512, 235, 45.1, True), (512, 235, 56.6, False), (256, 235, 70.9, True), (64, 157, 91.0, True),
                                      (64, 47, 91.0, True)):
        assert lists_pay(span, groups, rate) == lists, (span, groups, rate)
    assert all(lists_pay(span, groups, 3.0, h) for span in (64, 512, 1024) for groups in (2, 256) for h in (0.1, 1.0))
    assert lists_pay(64, 5, 0.0)
