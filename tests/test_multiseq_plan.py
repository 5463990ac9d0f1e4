"""The exact MULTISEQ kernel's plans, on the host: every wave's tasks keep to
the x slots that a workgroup stages (eight streams)."""
import ctypes
import random

import pytest

import stratum_amd as K

TYPES = (12, 14, 13, 11, 8, 10, 42)
N_CU, LDS = 256, 163840          # the MI355X


def plan(qtype, N, Kd, B):
    """(LDS bytes or -1, [streams per chunk, chunks, row groups per item, items per chunk, S])."""
    L, p = K.lib(), (ctypes.c_int * 5)()
    L.kqk_mv_plan.restype = ctypes.c_long
    return L.kqk_mv_plan(qtype, N, Kd, B, N_CU, LDS, p), p


# the first two plan chunks of eight and of seven streams in groups of three
@pytest.mark.parametrize("qtype,N,Kd,B", [(14, 815, 16640, 16), (11, 815, 13568, 8)])
def test_slots_of_groups_of_three(qtype, N, Kd, B):
    lds, p = plan(qtype, N, Kd, B)
    assert lds > 0 and p[4] == 3 and p[0] >= 7
    assert K.lib().kqk_mv_slots(p, B) <= 8


def test_slots_over_shapes():
    rng = random.Random(5)
    seen = set()
    for _ in range(4000):
        t, N = rng.choice(TYPES), int(2 ** rng.uniform(0, 15))
        Kd, B = 256 * rng.randint(1, 70), rng.randint(2, 64)
        lds, p = plan(t, N, Kd, B)
        assert lds > 0
        seen.add((p[0], p[4]))
        assert 1 <= K.lib().kqk_mv_slots(p, B) <= 8, (t, N, Kd, B, list(p))
    assert {(7, 3), (8, 3), (8, 4), (8, 2)} <= seen
