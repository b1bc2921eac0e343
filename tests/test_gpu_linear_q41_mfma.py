"""The Q4_1 forms of the MFMA linear kernel (csrc/moe_linear_q41.hip): every
fold form, rows and columns that end inside a tile, from canonical input and
from fp32, bit for bit against the oracle's reference order."""
import os

import numpy as np
import pytest

import moe_ffn
import oracle as O
import workloads as W
from golden_inputs import q4_1_matrix

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
DEV = "cuda:0"


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("K,M,N", [
    (32, 1, 40), (640, 2560, 128), (1024, 100, 33), (2048, 264, 65),     # staged leaves, 64 blocks
    (2080, 200, 32), (2560, 640, 40), (3072, 96, 64),                    # 65..96 blocks: the chained second block
    (3104, 64, 32), (8192, 64, 35),                                      # every block chained
])
def test_linear_q41_mfma_bit_exact(K, M, N, monkeypatch):
    monkeypatch.setenv("MOE_LINEAR_MFMA", "1")
    w = q4_1_matrix(K + 2 * M + N, K, M)
    x = W.activations(N, hidden=K, seed=K * 5 + N)
    x[N // 2] = 0.0              # a column of zero blocks
    xq = O.quantize_q8(x)
    ref = np.asarray(O.matrix_gpu_order_q41(w, K, M, xq), np.float32).reshape(N, M)
    L = moe_ffn.MoeLinear(moe_ffn.TYPE_Q4_1, K, M, w, max_columns=N)
    q8 = torch.from_numpy(np.ascontiguousarray(xq).view(np.uint8).reshape(N, -1)).to(DEV)
    y = L.forward_q8(q8, N).cpu().numpy()
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), ("forward_q8", K, M, N)
    ya, err = L.apply(torch.from_numpy(x).to(DEV))
    assert np.array_equal(ya.cpu().numpy().view(np.uint32), ref.view(np.uint32)), ("apply", K, M, N)
    assert int(err.cpu()[0]) == 0
    L.close()
