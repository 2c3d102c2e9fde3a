"""Which form of the backward pass a network gets, against measured steps of all three."""
import pytest

from bmtk_amd.training import Glif3Bptt

# neurons, trials, in-degree, us per step swept / blocked / a launch per part (one MI355X, calls of 40 steps, ring_slots 6)
MEASURED = [(9003, 32, 120, 25, 38, 43), (9003, 32, 750, 78, 70, 121), (15013, 32, 400, 84, 76, 113), (20011, 32, 220, 89, 73, 100),
            (51978, 32, 220, 290, 212, 270), (51978, 32, 750, 753, 446, 755), (51978, 64, 400, 894, 645, 859), (5011, 20, 750, 46, 50, 90),
            (20011, 20, 120, 68, 59, 78), (20011, 20, 750, 264, 174, 316), (20011, 16, 120, 44, 54, 55), (20011, 16, 750, 165, 152, 195),
            (37003, 16, 220, 149, 117, 153), (15013, 12, 750, 107, 126, 141), (37003, 12, 400, 260, 181, 282), (3001, 12, 200, 10, 40, 22),
            (20011, 8, 400, 72, 92, 84), (51978, 8, 120, 105, 90, 113), (9003, 4, 750, 49, 73, 56), (27011, 4, 750, 147, 168, 139),
            (33123, 4, 598, 187, 169, 155), (51978, 4, 750, 403, 350, 400)]


@pytest.mark.parametrize("n,batch,k,swept,blocked,plain", MEASURED)
def test_choice_is_within_a_tenth_of_the_fastest(n, batch, k, swept, blocked, plain):
    took = blocked if Glif3Bptt.blocked_pays(n, batch, 6, n * k) else plain if Glif3Bptt.plain_pays(batch, n * k) else swept
    assert took <= 1.1 * min(swept, blocked, plain)


def test_a_table_without_synapses_is_no_reason_for_ranges():
    assert not Glif3Bptt.blocked_pays(51978, 32, 6, 0)


# two steps per pass as they are now: neurons, trials, in-degree, us per step swept / blocked
TWO_STEPS = [(7000, 32, 600, 47.3, 45.0), (5000, 64, 300, 41.6, 38.3), (9003, 32, 250, 33.7, 35.5), (11000, 32, 200, 34.1, 37.5), (4000, 48, 900, 64.1, 53.2),
             (9003, 32, 400, 46.6, 42.6), (13000, 32, 120, 35.4, 36.5), (6500, 64, 150, 39.4, 37.6), (9003, 32, 120, 23.4, 29.9), (9003, 32, 750, 75.5, 58.5),
             (15000, 32, 220, 51.9, 47.4), (15000, 32, 500, 92.3, 72.2), (20011, 20, 200, 87.9, 63.0), (20011, 20, 700, 246.6, 136.8), (6000, 64, 500, 69.3, 54.7),
             (12000, 64, 150, 80.4, 65.4)]


@pytest.mark.parametrize("n,batch,k,swept,blocked", TWO_STEPS)
def test_choice_for_two_steps_per_pass(n, batch, k, swept, blocked):
    assert (blocked if Glif3Bptt.blocked_pays(n, batch, 6, n * k) else swept) <= 1.05 * min(swept, blocked)


# one step per pass: neurons, trials, in-degree, us per step swept / blocked
ONE_STEP = [(9003, 32, 400, 45.8, 61.1), (9003, 32, 750, 75.1, 82.3), (7000, 32, 600, 45.8, 60.5), (15000, 32, 220, 55.3, 67.2), (15000, 32, 500, 95.2, 93.7),
            (5000, 64, 300, 41.3, 56.9), (4000, 48, 900, 62.9, 73.2), (30011, 32, 120, 101.0, 110.4), (20011, 32, 220, 83.7, 84.1), (20011, 32, 60, 45.9, 63.8),
            (30011, 32, 400, 222.1, 174.7), (51978, 32, 220, 277.5, 248.6), (40000, 64, 150, 320.3, 337.8), (9003, 20, 400, 53.8, 63.0), (15013, 20, 220, 59.9, 67.7),
            (15013, 20, 750, 161.1, 132.5), (25013, 20, 300, 175.0, 123.1), (12000, 24, 300, 59.5, 67.5), (20000, 24, 300, 127.2, 103.9), (8000, 40, 300, 58.4, 69.6),
            (12000, 40, 300, 103.8, 93.2)]


@pytest.mark.parametrize("n,batch,k,swept,blocked", ONE_STEP)
def test_choice_for_one_step_per_pass(n, batch, k, swept, blocked):
    assert (blocked if Glif3Bptt.blocked_pays(n, batch, 6, n * k, two_steps=False) else swept) <= 1.1 * min(swept, blocked)


# neurons, trials, in-degree, us per two steps with 8 / 16 / 24 target ranges
RANGES = [(52000, 32, 100, 280.4, 291.4, 312.8), (25000, 40, 120, 211.7, 225.7, 246.1), (12000, 64, 150, 132.1, 135.1, 141.0), (45000, 40, 200, 516.5, 503.4, 530.0),
          (31000, 64, 300, 489.9, 461.7, 472.1), (20000, 20, 300, 147.6, 145.1, 148.7), (40000, 24, 400, 389.8, 368.1, 366.3), (30011, 32, 600, 331.4, 314.3, 315.1),
          (20011, 20, 700, 256.3, 248.4, 243.9), (15000, 32, 800, 183.0, 181.8, 179.0), (51978, 32, 1000, 887.8, 837.8, 809.4)]


@pytest.mark.parametrize("n,batch,k,eight,sixteen,more", RANGES)
def test_number_of_target_ranges(n, batch, k, eight, sixteen, more):
    took = {8: eight, 16: sixteen, 24: more}[Glif3Bptt.target_ranges(n, batch, 6, n * k)]
    assert took <= 1.01 * min(eight, sixteen, more)
    from bmtk_amd import ops
    assert Glif3Bptt.target_ranges(n, batch, 6, n * k, two_steps=False) == ops.blocked_table_blocks(n, batch, 6)
    assert Glif3Bptt.target_ranges(4 * n, 64, 6, 4 * n * k) == ops.blocked_table_blocks(4 * n, 64, 6) or 4 * n * 64 * 96 <= 200e6
