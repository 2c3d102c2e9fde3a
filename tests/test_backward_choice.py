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
