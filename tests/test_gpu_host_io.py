"""The host-pointer calls on both sides of their pinned buffer's bound (65536
floats a direction): one stream, several, a residual; lengths that
are not whole float4s.  The results are the device entries' bit for bit (the
same kernels: tolerance none), and a NULL vector is refused."""
import ctypes

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
    K.lib().kq_linear_shutdown()


def on_device(w, xs, N, Kd):
    dw, dx = torch.from_numpy(w).cuda(), torch.from_numpy(xs).cuda()
    y = torch.empty(xs.shape[0], N, device="cuda")
    for s in range(xs.shape[0]):
        K.gemv_dev(12, dw.data_ptr(), dx[s].data_ptr(), y[s].data_ptr(), N, Kd,
                   stream=torch.cuda.current_stream().cuda_stream)
    return y.cpu().numpy()


# y: inside, at and past the bound; x: past it for B = 65
@pytest.mark.parametrize("N,Kd,B", [(1, 256, 1), (65536, 256, 1), (65537, 256, 1), (1027, 512, 7),
                                    (32768, 256, 2), (21847, 256, 3), (33, 1024, 65)])
def test_host_vectors(N, Kd, B):
    w = synth.tensor(12, N, Kd, 6100 + B)
    K.WeightRegion(w.view(np.uint8).reshape(-1))
    t = K.make_tensor(12, N, Kd, 0)
    xs = np.stack([synth.gaussian(synth.rng(6200 + s), Kd) for s in range(B)])
    want = on_device(w, xs, N, Kd)
    for _ in range(2):                                  # the buffer again, other contents between
        got = np.stack(K.linear_multix(t, list(xs), N, Kd)) if B > 1 else \
            K.linear_dispatch(t, xs[0], N, Kd)[None]
        assert same_values(got, want)
        add = synth.gaussian(synth.rng(6300), N)
        assert same_values(K.linear_dispatch_add(t, xs[-1], add, N, Kd), add + want[-1])


def test_host_null_vectors():
    w = synth.tensor(12, 8, 256, 6400)
    K.WeightRegion(w.view(np.uint8).reshape(-1))
    t = K.make_tensor(12, 8, 256, 0)
    x, y = np.ones(256, np.float32), np.zeros(8, np.float32)
    L = K.lib()
    assert L.kq_linear_dispatch(ctypes.byref(t), None, K._fptr(y), 8, 256) == -1
    assert L.kq_linear_dispatch(ctypes.byref(t), K._fptr(x), None, 8, 256) == -1
    assert K.linear_dispatch(t, x, 8, 256).any()
