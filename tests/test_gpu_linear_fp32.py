"""apply on the few columns whose quantisation runs inside the vector kernel
(k_linear_fp32): one and two quantisation passes, rows that end inside a
workgroup or a 4-row wave, both weight types, bit for bit against the oracle,
and the error word; and apply where x and y overlap, at every column count."""
import numpy as np
import pytest

import moe_ffn
import oracle as O
import workloads as W
from golden_inputs import q4_1_matrix, q4_matrix

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
DEV = "cuda:0"


@pytest.mark.parametrize("q41,K,M,N", [
    (False, 2048, 2048, 1), (False, 32, 1, 1), (False, 32, 5, 4), (False, 640, 37, 3), (False, 1024, 100, 2),
    (False, 2080, 1000, 1), (False, 2560, 640, 1), (True, 640, 2560, 4), (True, 2560, 200, 1), (True, 2048, 17, 1),
])
def test_apply_few_columns(q41, K, M, N):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    w = q4_1_matrix(K + M + N, K, M) if q41 else q4_matrix(K + M + N, K, M)
    x = W.activations(N, hidden=K, seed=K + N)
    xq = O.quantize_q8(x)
    ref = (O.matrix_gpu_order_q41 if q41 else O.matrix_gpu_order)(w, K, M, xq)
    ref = np.asarray(ref, np.float32).reshape(N, M).view(np.uint32)
    L = moe_ffn.MoeLinear(moe_ffn.TYPE_Q4_1 if q41 else moe_ffn.TYPE_Q4_0, K, M, w, max_columns=N)
    y, err = L.apply(torch.from_numpy(x).to(DEV))
    assert np.array_equal(y.cpu().numpy().view(np.uint32), ref) and int(err.cpu()[0]) == 0
    yn = torch.empty((N, M), dtype=torch.float32, device=DEV)
    e = torch.zeros(1, dtype=torch.int32, device=DEV)
    L.apply_noalloc(torch.from_numpy(x).to(DEV), yn, e)
    assert np.array_equal(yn.cpu().numpy().view(np.uint32), ref) and int(e.cpu()[0]) == 0
    # A nonfinite value poisons its block (as zeros) and raises bit 1.
    x[N - 1, K - 1] = np.inf
    y, err = L.apply(torch.from_numpy(x).to(DEV))
    x[N - 1, K - 32:] = 0.0
    z, _ = L.apply(torch.from_numpy(x).to(DEV))
    assert int(err.cpu()[0]) == 1 and torch.equal(y.view(torch.int32), z.view(torch.int32))
    L.close()


@pytest.mark.parametrize("q41", [False, True])
@pytest.mark.parametrize("K,M,N,shift", [
    (2048, 2048, 1, 0), (512, 512, 4, 0), (512, 16384, 1, 0),   # y starts at x
    (2048, 2048, 1, 1000), (640, 2560, 2, 517), (2048, 512, 1, -300),   # y starts shift floats behind x's first
    (512, 512, 5, 0), (2048, 2048, 40, 0),   # past the fused columns: the vector and the MFMA kernel
])
def test_apply_overlapping_x_and_y(q41, K, M, N, shift):
    """Every output is that of separate buffers: x is read whole before y is
    written (a kernel that quantizes x in each workgroup must not be taken)."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    w = q4_1_matrix(K + M, K, M) if q41 else q4_matrix(K + M, K, M)
    x = W.activations(N, hidden=K, seed=K + M + N)
    ref = (O.matrix_gpu_order_q41 if q41 else O.matrix_gpu_order)(w, K, M, O.quantize_q8(x))
    ref = np.asarray(ref, np.float32).reshape(N, M).view(np.uint32)
    L = moe_ffn.MoeLinear(moe_ffn.TYPE_Q4_1 if q41 else moe_ffn.TYPE_Q4_0, K, M, w, max_columns=N)
    x0, y0 = max(0, -shift), max(0, shift)
    for noalloc in (False, True):
        buf = torch.zeros(N * max(K, M) + abs(shift), dtype=torch.float32, device=DEV)
        xv, yv = buf[x0:x0 + N * K].view(N, K), buf[y0:y0 + N * M].view(N, M)
        xv.copy_(torch.from_numpy(x))
        e = torch.zeros(1, dtype=torch.int32, device=DEV)
        if noalloc:
            L.apply_noalloc(xv, yv, e)
        else:
            L.apply(xv, y=yv, error=e)
        assert np.array_equal(yv.cpu().numpy().view(np.uint32), ref), (K, M, N, shift, noalloc)
        assert int(e.cpu()[0]) == 0
    L.close()
