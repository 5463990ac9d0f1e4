"""The MULTISEQ kernels' plans, on the host: every wave's tasks keep to the x
slots that a workgroup stages (eight streams), launches to the lanes that HIP
takes."""
import ctypes
import random

import pytest

import stratum_amd as K
from mv_cases import form, plans

TYPES = (12, 14, 13, 11, 8, 10, 42)
N_CU, LDS = 256, 163840          # the MI355X


def plan(qtype, N, Kd, B):
    """(LDS bytes or -1, [streams per chunk, chunks, row groups per item, items per chunk, S])."""
    L, p = K.lib(), (ctypes.c_int * 5)()
    L.kqk_mv_plan.restype = ctypes.c_long
    return L.kqk_mv_plan(qtype, N, Kd, B, N_CU, LDS, p), p


# chunks of eight and of seven streams in groups of three
@pytest.mark.parametrize("qtype,N,Kd,B", [(14, 815, 16640, 16), (11, 815, 13568, 14), (12, 815, 9216, 16)])
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


# the plans of calls that ran slower than one launch of the multi-x kernel: of
# equal costs the one with fewer workgroups on a CU, no S = 4 for one group of
# four streams of Q5_K, not half the waves of a CU's only workgroup idle
@pytest.mark.parametrize("qtype,N,Kd,B,items", [(13, 4096, 4096, 4, 256), (8, 4096, 4096, 2, 256),
                                                (11, 3000, 3072, 2, 188), (13, 17408, 5120, 4, None),
                                                (13, 11007, 4096, 4, None), (8, 2560, 9728, 3, None)])
def test_plans_of_few_streams(qtype, N, Kd, B, items):
    lds, p = plan(qtype, N, Kd, B)
    mc, nmc, ng, nblk, S = p
    assert lds > 0 and nmc == 1
    if items:
        assert nblk == items
    if qtype == 13:
        assert S != 4
    if Kd > 8192:                    # 16 waves, 2 rows a task
        tasks = ng * -(-mc // S)
        cut = S if S * tasks <= 16 else 1
        assert tasks > 16 or 2 * tasks * cut > 16


# very large batches: a plan's grid stays below the 2^32 lanes of a launch, and
# where the whole batch does not fit, a half, a quarter, ... of it does
@pytest.mark.parametrize("qtype,N,Kd,B", [(12, 151936, 8448, 8192), (12, 151936, 1024, 32768),
                                          (14, 151936, 8448, 8192), (10, 32000, 17408, 131072),
                                          (12, 8, 256, 1 << 28)])
def test_plans_of_large_batches(qtype, N, Kd, B):
    lanes = 1024 if Kd > 8192 else 512
    nb = B
    while True:
        lds, p = plan(qtype, N, Kd, nb)
        if lds > 0:
            break
        assert nb > 64
        nb = (nb // 2 + 7) & ~7
    assert (p[3] * p[1] + 7) // 8 * 8 * lanes < 1 << 32
    assert p[0] * p[1] >= nb


# the int8 kernel's most streams a launch: 256 lanes to every 64, 32 or 16 rows
# (one, two or four K-parts) and 16 streams
@pytest.mark.parametrize("N,Kd,rows", [(151936, 12288, 16), (151936, 4096, 32), (151936, 1024, 64),
                                       (32000, 17408, 16), (1, 256, 64), (1 << 26, 256, 64)])
def test_int8_streams_of_a_launch(N, Kd, rows):
    most = K.lib().kqk_mi_streams(N, Kd)
    assert most >= 16 and most % 16 == 0
    wgs = -(-N // rows) * (most // 16)
    assert (wgs + 7) // 8 * 8 * 256 < 1 << 32


def test_gpu_plans_cover_every_form():
    """mv_cases' plans, which the GPU tests launch: every S at every row
    length with no full turn and with one, its left-over tasks in every number
    of pieces."""
    seen = {(H, S) + form(H, S, ng, mc)[::2] for H, S, ng, mc, _ in plans()}
    for H in (1, 2):
        for S in (2, 3, 4):
            cuts = {2: (1, 2), 3: (1, 3), 4: (1, 2, 4)}[S]
            want = {(full, cut) for full in (0, 1) for cut in cuts} | {(1, 0)}
            assert want <= {s[2:] for s in seen if s[:2] == (H, S)}, (H, S)
    for H, S, ng, mc, M in plans():
        assert ng * -(-mc // S) < 2 * {1: 8, 2: 16}[H] and mc <= 8 and mc <= M
