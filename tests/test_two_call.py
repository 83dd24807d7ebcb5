"""quantize_lhs + matmul_preq for the types of the f16 matrix-core kernels: the
quantized rows are one image a row, whatever the weight's type, so that they
serve every weight whose type takes the same activation blocks, any leading rows
of them, and stay as they are."""
import numpy as np
import pytest
import torch

Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q2K, Q3K, Q4K, Q5K, Q6K = 2, 3, 6, 7, 8, 10, 11, 12, 13, 14


@pytest.mark.parametrize("k", [256, 4096])
def test_one_layout_for_an_activation(k):
    from xn_amd import _lib

    size = _lib.load().xnq_lhs_workspace_size
    for same in ((Q8_0, Q4_0, Q4_1, Q5_0, Q5_1), (Q2K, Q3K, Q5K)):
        for m in (8, 9, 16, 64, 512):
            assert len({size(dt, m, k) for dt in same}) == 1, (same, m)
            assert 0 <= 16 * size(same[0], m, k) - size(same[0], 16 * m, k) < 16 * 256  # (rounded up to 256 bytes)
    for m in (9, 16, 64):
        assert size(Q5K, m, k) == size(Q6K, m, k)


# (lhs quantized for, rows) -> (weight, rows used): every kernel instance of the row
# images (one and two row tiles, K of whole and of cut stages), lhs of other types
# and longer ones
PAIRS = [
    (Q4K, 16, Q5K, 16, 512, 40), (Q6K, 40, Q2K, 17, 768, 65), (Q4K, 300, Q3K, 300, 256, 1100),
    (Q4K, 300, Q5K, 100, 2304, 33), (Q5K, 64, Q2K, 64, 512, 8200), (Q2K, 64, Q5K, 64, 256, 8200),
    (Q3K, 9, Q3K, 9, 4352, 31), (Q5K, 40, Q6K, 40, 512, 96),
    (Q8_0, 33, Q4_1, 33, 320, 64), (Q5_1, 64, Q4_0, 9, 1056, 31), (Q4_0, 64, Q5_0, 64, 192, 8200),
    (Q8_0, 64, Q5_1, 64, 320, 8200), (Q4_1, 200, Q8_0, 130, 160, 2050), (Q8_0, 512, Q8_0, 512, 512, 1000),
    (Q4_0, 512, Q4_0, 512, 128, 1000), (Q5_1, 65, Q5_1, 65, 4160, 33), (Q8_0, 64, Q4_1, 64, 128, 8200),
]


@pytest.mark.gpu
@pytest.mark.parametrize("ldt,rows,dt,m,k,n", PAIRS)
def test_lhs_of_another_weight(orc, dev, ldt, rows, dt, m, k, n):
    from xn_amd import GgmlDType, QTensor
    from xn_amd.quantized import lhs_workspace, matmul_preq, quantize_lhs

    rng = np.random.default_rng(7 * dt + m + k)
    blocks = orc.from_float(dt, rng.normal(0, 0.02, (n, k)).astype(np.float32))
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    ws = lhs_workspace(GgmlDType(ldt), rows, k, dev)  # the size of what quantize_lhs writes
    quantize_lhs(GgmlDType(ldt), torch.from_numpy(x).to(dev), ws, rows, k)
    before = ws.clone()
    y = torch.full((m, n), float("nan"), device=dev)
    matmul_preq(QTensor.from_gguf_bytes(blocks, (n, k), GgmlDType(dt), dev), m, ws, y)
    got, want = y.cpu().numpy().astype(np.float64), orc.matmul(dt, x[:m], blocks, n).astype(np.float64)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - want) < 2e-6 * np.linalg.norm(want)
    assert torch.equal(ws, before)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,k", [(Q4_1, 320), (Q5_0, 576), (Q8_0, 1056), (Q4_0, 512), (Q5_1, 512), (Q2K, 512), (Q5K, 512)])
@pytest.mark.parametrize("m,n", [(40, 64), (64, 8224)])
def test_nonfinite_rows(orc, dev, dt, k, m, n):
    """Infinities, NaN, overflowing scales and sums reach what they reach on the matvec kernels."""
    from xn_amd import GgmlDType, QTensor
    from xn_amd.quantized import set_route

    rng = np.random.default_rng(900 + dt)
    blocks = orc.from_float(dt, rng.normal(0, 0.02, (n, k)).astype(np.float32))
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    x[3, 7], x[5, 300], x[7, 40], x[9, -5], x[11, 64:96] = np.inf, np.nan, 1e9, -1e9, 3000.0
    x[13] = 0.0
    qt, xt = QTensor.from_gguf_bytes(blocks, (n, k), GgmlDType(dt), dev), torch.from_numpy(x).to(dev)
    got, want = torch.empty((m, n), device=dev), torch.empty((m, n), device=dev)
    qt.matmul_t_split((m, k, n), xt, got)
    try:
        set_route(1)
        qt.matmul_t_split((m, k, n), xt, want)
    finally:
        set_route(0)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
    ok = want.isfinite().all(1)
    assert ok.sum() >= m - 5 and (got[13] == 0).all()
    assert ((got[ok] - want[ok]).double().norm() / want[ok].double().norm()).item() < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [Q4_1, Q8_0, Q2K, Q5K])
def test_workspace_of_the_row_images(orc, dev, dt):
    """matmul_t_ws and a group take a workspace of the row images' size (what
    workspace() gives), and refuse a smaller one."""
    import ctypes

    from xn_amd import GgmlDType, QTensor, XnqError, _lib
    from xn_amd._lib import check

    m, k, n = 40, 512, 96
    rng = np.random.default_rng(930 + dt)
    blocks = [orc.from_float(dt, rng.normal(0, 0.02, (n, k)).astype(np.float32)) for _ in range(2)]
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    qts = [QTensor.from_gguf_bytes(b, (n, k), GgmlDType(dt), dev) for b in blocks]
    want = [orc.matmul(dt, x, b, n).astype(np.float64) for b in blocks]
    xt, ys, ws = torch.from_numpy(x).to(dev), [torch.full((m, n), float("nan"), device=dev) for _ in qts], qts[0].workspace(m)
    assert ws.numel() < qts[0].matmul_t_workspace_size(m)

    def close(y, w):
        return np.linalg.norm(y.cpu().numpy().astype(np.float64) - w) < 2e-6 * np.linalg.norm(w)

    qts[0].matmul_t_ws((m, k, n), xt, ws, ys[0])
    assert close(ys[0], want[0])
    with pytest.raises(XnqError, match="smaller"):
        qts[0].matmul_t_ws((m, k, n), xt, ws[:-256], ys[0])
    hs = (ctypes.c_void_p * 2)(*[q.storage.handle.value for q in qts])
    ds = (ctypes.c_void_p * 2)(*[y.fill_(float("nan")).data_ptr() for y in ys])
    check(_lib.load().xnq_matmul_t_group(hs, 2, m, k, xt.data_ptr(), ds, ws.data_ptr(), ws.numel(),
                                         torch.cuda.current_stream().cuda_stream))
    assert close(ys[0], want[0]) and close(ys[1], want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [Q8_0, Q5_1, Q3K, Q5K])
@pytest.mark.parametrize("n", [96, 65 * 256])  # (a K split and the tile of the f16 image, where it is aligned)
def test_workspace_off_its_alignment(orc, dev, dt, n):
    """Workspace, rows and output at addresses of 4-byte alignment."""
    from xn_amd import GgmlDType, QTensor

    m, k = 130, 512
    rng = np.random.default_rng(960 + dt)
    blocks = orc.from_float(dt, rng.normal(0, 0.02, (n, k)).astype(np.float32))
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    qt = QTensor.from_gguf_bytes(blocks, (n, k), GgmlDType(dt), dev)
    ws = torch.zeros(qt.matmul_t_workspace_size(m) + 260, dtype=torch.uint8, device=dev)
    xt, y = torch.empty(m * k + 1, device=dev), torch.full((m * n + 1,), float("nan"), device=dev)
    xt[1:] = torch.from_numpy(x).to(dev).reshape(-1)
    qt.matmul_t_ws((m, k, n), xt[1:], ws[4:], y[1:])
    got, want = y[1:].view(m, n).cpu().numpy().astype(np.float64), orc.matmul(dt, x, blocks, n).astype(np.float64)
    assert np.linalg.norm(got - want) < 2e-6 * np.linalg.norm(want)
