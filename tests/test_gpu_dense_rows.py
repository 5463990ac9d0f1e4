"""F16 / F32 rows: a launch of few rows (the router kernel, straight to
registers) gives each row the value a launch of many rows (x staged in LDS)
gives it, bit for bit: both sum one order (contract: no tolerance)."""
import numpy as np
import pytest

import stratum_amd as K
from conftest import same_values
from stratum_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
MANY = 16384        # rows: past eight waves on each CU


# K: one super-block, a part of a block of loads, whole blocks, a remainder
@pytest.mark.parametrize("qtype", [0, 1])
@pytest.mark.parametrize("n,Kd,B", [(1, 256, 1), (5, 768, 1), (128, 2048, 3), (129, 2304, 2),
                                    (60, 8448, 5)])
def test_few_rows_match_many(qtype, n, Kd, B):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    w = torch.from_numpy(synth.tensor(qtype, MANY, Kd, 50 + qtype)).cuda()
    x = torch.from_numpy(np.stack([synth.gaussian(synth.rng(60 + s), Kd) for s in range(B)])).cuda()
    add = torch.from_numpy(synth.gaussian(synth.rng(70), MANY)).cuda()
    few, many = torch.full((B, n), 5.0, device="cuda"), torch.full((MANY,), 6.0, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    K.gemv_multix_dev(qtype, w.data_ptr(), x.data_ptr(), few.data_ptr(), B, n, Kd, stream=s)
    for j in range(B):
        K.gemv_dev(qtype, w.data_ptr(), x[j].data_ptr(), many.data_ptr(), MANY, Kd, stream=s)
        assert same_values(few[j].cpu().numpy(), many[:n].cpu().numpy()), f"stream {j}"
    one = torch.full((n,), 5.0, device="cuda")
    K.gemv_dev(qtype, w.data_ptr(), x[0].data_ptr(), one.data_ptr(), n, Kd, add_ptr=add.data_ptr(), stream=s)
    K.gemv_dev(qtype, w.data_ptr(), x[0].data_ptr(), many.data_ptr(), MANY, Kd, add_ptr=add.data_ptr(), stream=s)
    assert same_values(one.cpu().numpy(), many[:n].cpu().numpy()), "add"


@pytest.mark.parametrize("qtype", [0, 1])
@pytest.mark.parametrize("B", [1, 3])
def test_many_rows_of_long_x(qtype, B):
    """Many rows with x past what the kernel stages in LDS (16384 values: x
    read from memory): 37 rows over and over, each as a launch of few rows
    gives it."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    n, Kd, times = 37, 20480, 112
    w = torch.from_numpy(synth.tensor(qtype, n, Kd, 80 + qtype)).cuda()
    x = torch.from_numpy(np.stack([synth.gaussian(synth.rng(90 + s), Kd) for s in range(B)])).cuda()
    few, many = torch.full((B, n), 5.0, device="cuda"), torch.full((B, n * times), 6.0, device="cuda")
    s, wm = torch.cuda.current_stream().cuda_stream, w.repeat(times)
    K.gemv_multix_dev(qtype, w.data_ptr(), x.data_ptr(), few.data_ptr(), B, n, Kd, stream=s)
    K.gemv_multix_dev(qtype, wm.data_ptr(), x.data_ptr(), many.data_ptr(), B, n * times, Kd, stream=s)
    for j in range(B):
        assert same_values(many[j].cpu().numpy(), few[j].repeat(times).cpu().numpy()), f"stream {j}"
