"""Rounding errors of the f16 matrix-core kernels against 64-bit products of the
same quantized operands (decoded by the independent codecs), next to those of the
matvec kernels on the same weights and rows: zero-mean rows, rows of one sign, and
Q5_K blocks of extreme levels and scales, whose block sums pass 2^24.

The bound is the matvec kernels' own error, or one f32 rounding of each output
(2^-24 of it; 2^-24 / sqrt(3) in the mean of a uniform mantissa), whichever is
larger: 32-bit sums that round off less than that are not told apart."""
import numpy as np
import pytest
import torch

from . import _formats as F

pytestmark = pytest.mark.gpu

Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q2K, Q3K, Q5K = 2, 3, 6, 7, 8, 10, 11, 13
TYPES = [Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q2K, Q3K, Q5K]


def exact(orc, dt, x, blocks, n, dev):
    """64-bit products of x's quantized rows and the weight's blocks."""
    m, k = x.shape
    a = orc.quantize_lhs(dt, x)
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v, dtype=np.float64)).to(dev)  # noqa: E731
    if dt in (Q2K, Q3K, Q5K):
        da, qa, _ = F.decode_q8k(a)
        act = (t(qa) * t(da)[:, None]).view(m, k)
        if dt == Q3K:
            d, sc, q = F.decode_q3k(blocks)
            w = t(q).view(len(d), 16, 16) * t(sc)[:, :, None] * t(d)[:, None, None]
        else:
            d, dmin, sc, mn, q = (F.decode_q2k if dt == Q2K else F.decode_q5k)(blocks)
            subs = sc.shape[1]
            w = t(q).view(len(d), subs, -1) * (t(sc) * t(d)[:, None])[:, :, None] - (t(mn) * t(dmin)[:, None])[:, :, None]
        return act @ w.reshape(n, k).T
    if dt in (Q4_1, Q5_1):
        da, s, qa = F.decode_q8_1(a)
        d, mins, q = (F.decode_q4_1 if dt == Q4_1 else F.decode_q5_1)(blocks)
        y = t(s).view(m, -1) @ t(mins).view(n, -1).T
    else:
        da, qa = F.decode_q8_0(a)
        d, q = {Q4_0: F.decode_q4_0, Q5_0: F.decode_q5_0, Q8_0: F.decode_q8_0}[dt](blocks)
        y = 0.0
    act = (t(qa) * t(da)[:, None]).view(m, k)
    return y + act @ (t(q) * t(d)[:, None]).view(n, k).T


def errors(orc, dev, dt, blocks, x, n):
    from xn_amd import GgmlDType, QTensor
    from xn_amd.quantized import set_route

    m, k = x.shape
    qt = QTensor.from_gguf_bytes(blocks, (n, k), GgmlDType(dt), dev)
    want, xt, y, e = exact(orc, dt, x, blocks, n, dev), torch.from_numpy(x).to(dev), torch.empty((m, n), device=dev), []
    for route in (0, 1):
        try:
            set_route(route)
            qt.matmul_t((m, k, n), xt, y)
        finally:
            set_route(0)
        e.append(((y.double() - want).norm() / want.norm()).item())
    print(f"dt={dt} m={m} k={k} n={n}: {e[0]:.3e} matvec {e[1]:.3e}")
    return e


def check(e):
    assert e[0] <= max(e[1], 2.0 ** -24), f"relative L2 error {e[0]:.3e}, matvec kernels {e[1]:.3e}"


# 16-row (K types: 32-row), 32- and 64-row K-split tiles; 256 x 64 tiles
SHAPES = [(40, 1024, 96, "h16_ksplit16"), (64, 1024, 4096, "h16_ksplit32"), (64, 1024, 8224, "h16_ksplit64"),
          (600, 2048, 4352, "tile")]


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("m,k,n,kernel", SHAPES)
@pytest.mark.parametrize("offset", [0.0, 10.0])
def test_no_larger_than_the_matvec(orc, dev, dt, m, k, n, kernel, offset):
    from xn_amd import GgmlDType, QTensor
    from xn_amd.quantized import matmul_t_kernel

    if dt in (Q2K, Q3K, Q5K):
        kernel = {"h16_ksplit16": "h16_ksplit32", "tile": "h16_super_tile"}.get(kernel, kernel)
    assert matmul_t_kernel(dt, m, n, k) == ("h16_block_tile" if kernel == "tile" else kernel)

    w = torch.empty((n, k), device=dev).normal_(0, 0.02, generator=torch.Generator(device=dev).manual_seed(40 + dt))
    blocks = np.frombuffer(QTensor.quantize_f32(w, dtype=GgmlDType(dt)).data(), np.uint8)
    x = np.random.default_rng(50 + dt).normal(offset, 1.0 if offset == 0.0 else 0.3, (m, k)).astype(np.float32)
    check(errors(orc, dev, dt, blocks, x, n))


def q5k_rows(rng, n, k, levels, scales, d=5e-5):
    """n rows of Q5_K blocks (64 different ones, repeated), as GGUF bytes (n, row bytes)."""
    bits = [int(np.float16(v).view(np.uint16)) for v in (d, 8e-4)]
    b = [F.encode_q5k(*bits, rng.integers(*scales, 8), rng.integers(8, 64, 8), rng.integers(*levels, 256))
         for _ in range(64 * k // 256)]
    return np.tile(np.stack(b).reshape(64, -1), (n // 64, 1))


Q5K_SHAPES = [(9, 64), (64, 4096), (64, 8256), (512, 4352)]


@pytest.mark.parametrize("m,n", Q5K_SHAPES)
@pytest.mark.parametrize("levels,scales", [((0, 32), (24, 64)), ((24, 32), (56, 64)), ((31, 32), (63, 64)), ((0, 2), (56, 64))])
def test_q5k_sums_past_2_24(orc, dev, m, n, levels, scales):
    rng = np.random.default_rng(60 + m)
    k = 512
    x = rng.normal(10, 0.3, (m, k)).astype(np.float32)
    e = errors(orc, dev, Q5K, q5k_rows(rng, n, k, levels, scales).reshape(-1), x, n)
    if levels[1] - levels[0] < 8:
        # A whole block at one end of the levels: the sum of the levels less 16 itself passes
        # 2^24, up to 3.2e7, where each of at most 16 products leaves a rounding of at most 1
        # (0.58 in the mean): 2.3 times d, to a block's 840 (levels 0 and 1) d_a: 1.4e-7.
        e[1] += 1.4e-7
    check(e)


@pytest.mark.parametrize("m,n", Q5K_SHAPES)
def test_q5k_nonfinite_block_scales(orc, dev, m, n):
    """An infinite or NaN d or dmin of a weight block, rows of one sign: what the
    matvec kernels give, in that column alone."""
    from xn_amd import GgmlDType, QTensor
    from xn_amd.quantized import set_route

    rng = np.random.default_rng(80 + m)
    k = 512
    w = q5k_rows(rng, n, k, (1, 32), (24, 64)).copy()
    for row, off, v in ((3, 0, np.inf), (5, 0, -np.inf), (7, 0, np.nan), (9, 2, np.inf), (11, 2, -np.inf), (13, 2, np.nan), (15, 0, 0.0)):
        w[row, off:off + 2] = np.array([v], np.float16).view(np.uint8)
    qt, xt = QTensor.from_gguf_bytes(w.reshape(-1), (n, k), GgmlDType(Q5K), dev), torch.from_numpy(
        rng.normal(10, 0.3, (m, k)).astype(np.float32)).to(dev)
    got, want = torch.empty((m, n), device=dev), torch.empty((m, n), device=dev)
    qt.matmul_t((m, k, n), xt, got)
    try:
        set_route(1)
        qt.matmul_t((m, k, n), xt, want)
    finally:
        set_route(0)
    assert (~want.isfinite()).sum() == 6 * m
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
    ok = want.isfinite()
    assert ((got[ok] - want[ok]).double().norm() / want[ok].double().norm()).item() < 5e-7
