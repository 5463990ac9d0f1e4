"""Exact MULTISEQ (kq_gemv_multix_dev) at the edges of its kernel: row groups
of 8 (at most 128 chunks) and 2 rows, tiles of 16 and 32 chunks, streams in
groups of 2-4 and chunks of 8, one and many workgroups, special x values.
Every stream equals its own single-stream launch bit for bit (the contract:
tolerance none)."""
import ctypes

import numpy as np
import pytest

import stratum_amd as K
from conftest import same_values
from mv_cases import ROWS, SHAPES, plans
from oracle import oracle as O
from stratum_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    K.lib()
    yield
    torch.cuda.synchronize()


# K: one super-block; a tile and a super-block more; the last of 8 phases, the
# first of 32; tiles of 32 with a remainder.  N: below and above a row group.
@pytest.mark.parametrize("qtype", [12, 14, 13, 11, 8, 10, 42])
@pytest.mark.parametrize("N,Kd,B", [(1, 256, 2), (7, 1280, 3), (9, 1024, 5), (129, 8192, 6),
                                    (3, 8448, 4), (65, 10496, 9), (1031, 768, 13),
                                    (2050, 2304, 17)])
def test_multiseq_edges(qtype, N, Kd, B):
    check(qtype, N, Kd, B)


# groups of three with seven and eight streams staged: the last group starts
# before its own streams, at the last three slots
@pytest.mark.parametrize("qtype,N,Kd,B", [(14, 815, 16640, 16), (11, 815, 13568, 14), (12, 815, 9216, 16)])
def test_multiseq_last_group_of_three(qtype, N, Kd, B):
    check(qtype, N, Kd, B)


# the layer shapes whose plans are the forms S = 3 and 4 of long rows, and S = 4
# of Q2_K and type 42
@pytest.mark.parametrize("qtype,N,Kd,B", [(12, 5120, 17408, 3), (12, 5120, 17408, 6)] +
                         [(t, n, k, b) for t in (10, 42) for n, k in ((17408, 5120), (5120, 17408))
                          for b in (8, 16)])
def test_multiseq_layer_shapes(qtype, N, Kd, B):
    check(qtype, N, Kd, B)


@pytest.mark.parametrize("H", [1, 2])
@pytest.mark.parametrize("qtype", [12, 14, 13, 11, 8, 10, 42])
def test_multiseq_every_form(qtype, H):
    """Every form of the kernel, launched with its plan (mv_cases): whole
    items and a last one of two row groups and a row."""
    L, Kd, (W, rpt) = K.lib(), ROWS[H], SHAPES[H]
    L.kqk_mv_plan.restype = ctypes.c_long
    L.kqk_launch_mv.argtypes = [ctypes.c_int, ctypes.POINTER(ctypes.c_int), ctypes.c_long, ctypes.c_void_p,
                                ctypes.c_void_p, ctypes.c_long, ctypes.c_void_p, ctypes.c_long, ctypes.c_int,
                                ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    most = max(ng for h, _, ng, _, _ in plans() if h == H) * rpt + 2 * rpt + 1
    B = max(M for _, _, _, _, M in plans())
    w = torch.from_numpy(synth.tensor(qtype, most, Kd, 4500 + qtype)).cuda()
    x = torch.from_numpy(np.stack([synth.gaussian(synth.rng(4600 + j), Kd) for j in range(B)])).cuda()
    one = torch.empty(B, most, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    for j in range(B):
        K.gemv_dev(qtype, w.data_ptr(), x[j].data_ptr(), one[j].data_ptr(), most, Kd, stream=s)
    xpc = {12: 32, 13: 32, 10: 16, 42: 16}.get(qtype)              # x values of a sum
    for h, S, ng, mc, M in plans():
        if h != H:
            continue
        N = ng * rpt + min(ng, 2) * rpt + 1
        groups = -(-N // rpt)
        p = (ctypes.c_int * 5)(mc, -(-M // mc), ng, -(-groups // ng), S)
        lds = 131072 * H // 2 + (mc * Kd // xpc * 4 if xpc else 0)   # x tiles, x sums
        print(f"multiseq {K.TYPE_NAMES[qtype]} {N}x{Kd} M={M} plan={list(p)}", flush=True)
        assert L.kqk_mv_slots(p, M) <= 8
        got = torch.full((M, N), 7.0, device="cuda")
        assert L.kqk_launch_mv(qtype, p, lds, w.data_ptr(), x.data_ptr(), Kd, got.data_ptr(), N, M, N, Kd, s) == 0
        assert torch.equal(got, one[:M, :N]), (N, M, list(p))


# rows too long for the single-stream launch: up to the x sums that leave room
# for the tiles, and past them (Q4_K / Q5_K 262144, Q2_K / type 42 131072: the
# multi-x kernel); a stream outside its scaled window.  Bound of the parity
# tests.
@pytest.mark.parametrize("qtype,Kd", [(12, 65536), (14, 131072), (12, 262400), (13, 262400), (10, 131328),
                                      (42, 131328)])
def test_multiseq_very_long_rows(port, qtype, Kd):
    N, B = 5, 3
    w = synth.tensor(qtype, N, Kd, 4700 + qtype)
    xs = np.stack([synth.gaussian(synth.rng(4800 + s), Kd) for s in range(B)])
    xs[1, 4097] = np.float32(2.0 ** -60)
    print(f"multiseq {K.TYPE_NAMES[qtype]} {N}x{Kd} B={B}", flush=True)
    dw, dx = torch.from_numpy(w).cuda(), torch.from_numpy(xs).cuda()
    got = torch.full((B, N), 7.0, device="cuda")
    K.gemv_multix_dev(qtype, dw.data_ptr(), dx.data_ptr(), got.data_ptr(), B, N, Kd,
                      stream=torch.cuda.current_stream().cuda_stream)
    for j in range(B):
        assert O.rel_err(got[j].cpu().numpy(), port.gemv(qtype, w, xs[j], N, Kd)).max() <= 1e-5, f"stream {j}"


def check(qtype, N, Kd, B):
    w = synth.tensor(qtype, N, Kd, 4100 + qtype)
    xs = np.stack([synth.gaussian(synth.rng(4200 + s), Kd) for s in range(B)])
    xs[0, 5] = np.float32(1e-42)                 # subnormal
    xs[B - 1, Kd - 3] = np.float32(2.0 ** 70)
    if B > 2:
        xs[1, 0], xs[1, Kd // 2] = np.inf, -np.inf
        xs[2, Kd - 1] = np.nan
    print(f"multiseq {K.TYPE_NAMES[qtype]} {N}x{Kd} B={B}", flush=True)
    s = torch.cuda.current_stream().cuda_stream
    dw, dx = torch.from_numpy(w).cuda(), torch.from_numpy(xs).cuda()
    got = torch.full((B, N), 7.0, device="cuda")
    one = torch.full((B, N), 9.0, device="cuda")
    K.gemv_multix_dev(qtype, dw.data_ptr(), dx.data_ptr(), got.data_ptr(), B, N, Kd, stream=s)
    for j in range(B):
        K.gemv_dev(qtype, dw.data_ptr(), dx[j].data_ptr(), one[j].data_ptr(), N, Kd, stream=s)
    got, one = got.cpu().numpy(), one.cpu().numpy()
    for j in range(B):
        assert same_values(got[j], one[j]), f"stream {j}"


def test_multiseq_past_one_launch():
    """More streams than the lanes of a launch hold go in parts.  Sixteen
    different streams over and over: every one equals its single launch."""
    N, Kd, B = 151936, 256, 32016
    if torch.cuda.mem_get_info()[0] < 30 << 30:
        pytest.skip("needs 20 GB")
    rows = 64
    w = torch.from_numpy(synth.tensor(12, rows, Kd, 4300)).cuda().repeat(N // rows)
    x16 = torch.from_numpy(np.stack([synth.gaussian(synth.rng(4400 + s), Kd) for s in range(16)])).cuda()
    dx, y = x16.repeat(B // 16, 1), torch.empty(B, N, device="cuda")
    one = torch.empty(16, N, device="cuda")
    print(f"multiseq Q4_K {N}x{Kd} B={B}", flush=True)
    s = torch.cuda.current_stream().cuda_stream
    K.gemv_multix_dev(12, w.data_ptr(), dx.data_ptr(), y.data_ptr(), B, N, Kd, stream=s)
    for j in range(16):
        K.gemv_dev(12, w.data_ptr(), x16[j].data_ptr(), one[j].data_ptr(), N, Kd, stream=s)
    for j in range(0, B, 16):
        assert torch.equal(y[j:j + 16], one), f"streams {j} ..."
