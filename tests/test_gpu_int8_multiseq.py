"""int8 MULTISEQ of Q4_K / Q6_K (kq_gemv_multix_dev | KQ_INT8_ACT) at the edges
of its kernel: rows below, above and not a multiple of 16 and of a
workgroup's row blocks; one, two and four K-parts with even and odd
super-block counts; streams around the sets of 16; weights at addresses that
are not 16-byte (Q4_K) or 2-byte (Q6_K) aligned.  Every stream equals the
oracle's restatement of the reference's q*_dot_rows2_sdot_multix_pack bit for
bit (the K-parts regroup a binary64 sum, which moves a binary32 result with a
chance of about 1e-8 a value)."""
import numpy as np
import pytest

import stratum_amd as K
from conftest import same_values
from stratum_amd import INT8_ACT, synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    K.lib()
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("qtype", [12, 14])
@pytest.mark.parametrize("N,Kd,B,off", [(1, 256, 2, 0), (15, 256, 15, 2), (65, 2816, 16, 0),
                                        (17, 3072, 17, 0), (33, 3328, 33, 1), (31, 12032, 3, 3),
                                        (16, 12288, 5, 0), (18, 12544, 16, 8)])
def test_int8_multiseq_edges(port, qtype, N, Kd, B, off):
    w = synth.tensor(qtype, N, Kd, 5100 + B)
    xs = np.stack([synth.gaussian(synth.rng(5200 + s), Kd) for s in range(B)])
    xs[0, 256 - 32:256] = 0.0                        # a group of scale 0
    xs[B - 1, 5] = np.float32(2.0 ** 40)
    print(f"int8 multiseq type={qtype} {N}x{Kd} B={B} off={off}", flush=True)
    dw = torch.zeros(w.nbytes + 16, dtype=torch.uint8, device="cuda")[off:off + w.nbytes]
    dw.copy_(torch.from_numpy(w.view(np.uint8).reshape(-1)))
    dx = torch.from_numpy(xs).cuda()
    got = torch.full((B, N), 7.0, device="cuda")
    K.gemv_multix_dev(qtype | INT8_ACT, dw.data_ptr(), dx.data_ptr(), got.data_ptr(), B, N, Kd,
                      stream=torch.cuda.current_stream().cuda_stream)
    want = port.gemv_i8_multix(qtype, w, xs, N, Kd)
    assert same_values(got.cpu().numpy(), want)


def test_int8_multiseq_past_one_launch(port):
    """More streams than the lanes of a launch hold go in parts, the last of
    one stream.  Sixteen different streams over and over: every one equals the
    oracle's."""
    N, Kd, rows = 151936, 12288, 64
    B = K.lib().kqk_mi_streams(N, Kd) + 1
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 25 GB")
    w = synth.tensor(12, rows, Kd, 5300)
    x16 = np.stack([synth.gaussian(synth.rng(5400 + s), Kd) for s in range(16)])
    want = torch.from_numpy(port.gemv_i8_multix(12, w, x16, rows, Kd)).cuda().repeat(1, N // rows)
    dw = torch.from_numpy(w).cuda().repeat(N // rows)
    dx = torch.from_numpy(x16).cuda().repeat(B // 16 + 1, 1)[:B].contiguous()
    y = torch.empty(B, N, device="cuda")
    print(f"int8 multiseq Q4_K {N}x{Kd} B={B}", flush=True)
    K.gemv_multix_dev(12 | INT8_ACT, dw.data_ptr(), dx.data_ptr(), y.data_ptr(), B, N, Kd,
                      stream=torch.cuda.current_stream().cuda_stream)
    for j in range(0, B, 16):
        n = min(16, B - j)
        assert torch.equal(y[j:j + n], want[:n]), f"streams {j} ..."
