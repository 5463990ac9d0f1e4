"""Exact MULTISEQ (kq_gemv_multix_dev) at the edges of its kernel: row groups
of 8 (at most 128 chunks) and 2 rows, tiles of 16 and 32 chunks, streams in
groups of 2-4 and chunks of 8, one and many workgroups, special x values.
Every stream equals its own single-stream launch bit for bit (the contract:
tolerance none)."""
import numpy as np
import pytest

import stratum_amd as K
from conftest import same_values
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
