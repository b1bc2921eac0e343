"""GPU parity of the kernels on fp16 operands (csrc/moe_half.hpp) at the edges
of their tiles: rows of 1..64 blocks (the 64-block form and the one that
zero-fills missing blocks), an odd number of 32-row tiles (an idle second
tile in the last workgroup), and token counts around the 32-token tiles; and
of their inputs: codes of -128, nonfinite heads, rows and activations.
Every comparison is bit for bit: the kernels keep the reference's fp32 order.
"""
import numpy as np
import pytest

import moe_ffn
import oracle as O
import workloads as W

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
DEV = "cuda:0"


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("H,I,columns", [
    (2048, 32, 1), (2048, 96, 33), (2048, 64, 128), (2048, 160, 130),
    (64, 96, 31), (960, 32, 32), (1088, 64, 64), (1984, 160, 97),
])
def test_gate_up_tile_edges(H, I, columns):
    bank = W.q4_bank(2, hidden=H, intermediate=I, seed=H + I + columns)
    L = moe_ffn.MoeLayer(H, I, 2, 1, False, columns, experts_q4=bank)
    x = W.activations(columns, hidden=H, seed=columns)
    x[columns // 2] *= 1e-3
    xq = O.quantize_q8(x)
    n = H // 32 * I * 18
    blob = bank.reshape(2, -1)[1]
    ref = O.expert_forward(blob[:n], blob[n:2 * n], blob[2 * n:], H, I, xq)
    xd = torch.from_numpy(np.ascontiguousarray(xq).view(np.uint8).reshape(columns, -1)).to(DEV)
    got = L.expert_gate_up(1, xd, columns, path=moe_ffn.PATH_MFMA)
    torch.cuda.synchronize()
    assert int(got["error"].cpu()[0]) == 0
    assert np.array_equal(got["middle_q8"].cpu().numpy().reshape(-1),
                          np.ascontiguousarray(ref["middle_q8"]).view(np.uint8).reshape(-1))
    assert np.array_equal(got["middle"].cpu().numpy().view(np.uint32), ref["middle"].view(np.uint32))
    # Without the fp32 middle: the kernel the forward runs.
    mq = torch.empty_like(got["middle_q8"])
    err = torch.zeros(1, dtype=torch.int32, device=DEV)
    st = moe_ffn.library().moe_ffn_expert_gate_up(L.handle, 1, moe_ffn._ptr(xd), columns, None, moe_ffn._ptr(mq), None,
                                                  None, moe_ffn.PATH_MFMA, moe_ffn._ptr(err), moe_ffn._stream(None))
    torch.cuda.synchronize()
    assert st == 0 and torch.equal(mq, got["middle_q8"])
    L.close()


@pytest.mark.parametrize("H", [2048, 1984, 2560, 4096])   # the fp16 forms; int8 for 65..96 blocks and past 96
def test_gate_up_nonfinite_rows(H):
    """Rows whose gate or up is nonfinite make their own middle element 0 and
    raise bit 1, as the reference's per-element sanitisation does; every other
    row of the 32-row block keeps its value, on both kernel paths."""
    I, columns, nb = 64, 40, H // 32
    rows = {3: np.inf, 4: -np.inf, 17: np.nan, 33: np.inf}
    clean = W.q4_bank(1, hidden=H, intermediate=I, seed=H).reshape(3, -1).copy()
    dirty = clean.copy()
    for r, v in rows.items():
        blocks = [m.reshape(I, nb, 18) for m in (clean[0], clean[1])]
        for b in blocks:
            b[r, :, :2] = 0                       # a row of zero blocks: gate = up = 0
        which = dirty[r & 1].reshape(I, nb, 18)   # gate (0) or up (1)
        which[r, nb // 2, :2] = np.array([v], np.float16).view(np.uint8)
    x = W.activations(columns, hidden=H, seed=H + 1)
    xq = O.quantize_q8(x)
    ref = O.expert_forward(clean[0], clean[1], clean[2], H, I, xq)
    xd = torch.from_numpy(np.ascontiguousarray(xq).view(np.uint8).reshape(columns, -1)).to(DEV)
    L = moe_ffn.MoeLayer(H, I, 1, 1, False, columns, experts_q4=dirty.reshape(-1))
    for path in (moe_ffn.PATH_STREAM, moe_ffn.PATH_MFMA):
        got = L.expert_gate_up(0, xd, columns, path=path)
        torch.cuda.synchronize()
        assert int(got["error"].cpu()[0]) == 1, path
        assert np.array_equal(got["middle"].cpu().numpy().view(np.uint32), ref["middle"].view(np.uint32)), path
        assert np.array_equal(got["middle_q8"].cpu().numpy().reshape(-1),
                              np.ascontiguousarray(ref["middle_q8"]).view(np.uint8).reshape(-1)), path
    L.close()


@pytest.mark.parametrize("K,M,N", [
    (1024, 2820, 1000), (2048, 2820, 1000), (1984, 2816, 1001),
    (2048, 2819, 1001), (1056, 2821, 999),   # rows no multiple of 4: stored one value at a time
])
def test_linear_wide_grid_matches_vector(K, M, N, monkeypatch):
    """Grids wide enough for the fp16-operand linear (canonical input, planes,
    and both stagings of the no-allocation call) against the vector kernel,
    which the oracle pins: ragged last rows and columns."""
    w = W.q4_blocks(M * K // 32, np.random.default_rng(K + M)).reshape(-1)
    x = torch.from_numpy(W.activations(N, hidden=K, seed=N)).to(DEV)
    monkeypatch.setenv("MOE_LINEAR_MFMA", "0")
    V = moe_ffn.MoeLinear(moe_ffn.TYPE_Q4_0, K, M, w, max_columns=N)
    monkeypatch.delenv("MOE_LINEAR_MFMA")
    L = moe_ffn.MoeLinear(moe_ffn.TYPE_Q4_0, K, M, w, max_columns=N)
    q8, _ = moe_ffn.quantize_q8_1(x)
    ref = V.forward_q8(q8, N).view(torch.int32)
    assert torch.equal(L.forward_q8(q8, N).view(torch.int32), ref)
    assert torch.equal(L.apply(x)[0].view(torch.int32), ref)
    y = torch.empty((N, M), dtype=torch.float32, device=DEV)
    e = torch.zeros(1, dtype=torch.int32, device=DEV)
    L.apply_noalloc(x, y, e)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int32), ref) and int(e.cpu()[0]) == 0
    V.close()
    L.close()


@pytest.mark.parametrize("M,N,block", [(512, 4096, 36), (512, 5568, 36), (512, 5569, 68)])
def test_linear_workspace_bytes(M, N, block):
    """apply's workspace holds fp16 operand planes only where max_columns can
    reach the kernel that reads them (4 row groups x 175 column tiles do)."""
    w = W.q4_blocks(M * 64, np.random.default_rng(M)).reshape(-1)

    def taken(columns):
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        L = moe_ffn.MoeLinear(moe_ffn.TYPE_Q4_0, 2048, M, w, max_columns=columns)
        torch.cuda.synchronize()
        return before - torch.cuda.mem_get_info()[0], L
    taken(0)[1].close()   # the first one loads code objects
    whole, L = taken(N)
    L.close()
    # The weights (0.6 MB) and the workspace are an allocation each, rounded up
    # to 2 MiB or served from a chunk that is there: within 4 MiB either way,
    # where 36 and 68 bytes a block lie 8 MiB and more apart.
    assert abs(whole - N * 64 * block) <= 4 << 20, (whole, N * 64 * block)


@pytest.mark.parametrize("K", [2048, 1056])
def test_linear_canonical_extremes(K):
    """Canonical blocks as a caller may hand them in: codes of -128, the largest
    and smallest heads, and nonfinite ones, which reach their own column only.
    Bit for bit the vector kernel's values; where those are NaN, NaN."""
    M, N = 2820, 1000
    rng = np.random.default_rng(K)
    w = W.q4_blocks(M * K // 32, rng).reshape(-1)
    q8 = rng.integers(-128, 128, (N, K // 32, 36), dtype=np.int64).astype(np.int8).view(np.uint8)
    heads = rng.standard_normal((N, K // 32, 2)).astype(np.float16)
    heads[1], heads[2], heads[3] = 65504.0, 2.0 ** -24, 0.0
    for i, v in enumerate((np.inf, -np.inf, np.nan)):
        heads[100 + i, K // 64, 0] = v
        heads[110 + i, K // 32 - 1, 1] = v
    q8[..., :4] = heads.view(np.uint8)
    q8[4, :, 4:] = 0x80
    q8[5, :, 4:] = 0x7f
    q8[100:103, :, 4:12] = 0   # an infinite scale times a zero dot
    x = torch.from_numpy(np.ascontiguousarray(q8).reshape(N, -1)).to(DEV)
    L = moe_ffn.MoeLinear(moe_ffn.TYPE_Q4_0, K, M, w)
    got = L.forward_q8(x, N)
    # 8 columns at a time take the vector kernel.
    ref = torch.cat([L.forward_q8(x[c:c + 8].contiguous(), 8) for c in range(0, N, 8)])
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(got), nan)
    assert bool(torch.isfinite(ref[:100]).all()) and not bool(torch.isfinite(ref[100:103]).any())
    assert torch.equal(got[~nan].view(torch.int32), ref[~nan].view(torch.int32))
    L.close()


@pytest.mark.parametrize("H,I", [(2048, 512), (1984, 64), (2560, 640)])
def test_grouped_layer_nonfinite_activations(H, I):
    """A grouped batch whose groups go to MFMA: a block with a nonfinite value
    counts as zeros and raises bit 1; a zeroed block gives the same outputs."""
    E, N = 8, 300
    L = moe_ffn.MoeLayer(H, I, E, 4, True, N, synthetic_seed=H)
    x = W.activations(N, hidden=H, seed=H)
    ids, w = W.routes_uniform(N, experts=E, k=4, seed=1)
    zeroed = x.copy()
    for t, e, v in ((0, 0, np.nan), (17, H - 1, np.inf), (N - 1, 40, -np.inf)):
        x[t, e] = v
        zeroed[t, e // 32 * 32:e // 32 * 32 + 32] = 0.0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    y, err = L.forward(dev(x), dev(ids), dev(w))
    ref, ok = L.forward(dev(zeroed), dev(ids), dev(w))
    assert int(err.cpu()[0]) == 1 and int(ok.cpu()[0]) == 0
    assert L.last_stats()["mfma_items"] > 0
    assert torch.equal(y.view(torch.int32), ref.view(torch.int32))
    L.close()
