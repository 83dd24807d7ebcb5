"""The f16 matrix-core kernels (k_h16.hip) against the CPU oracle: every type
they take, at the edges of their tiles (16, 32 and 64 rows, 32 and 256 columns),
of their K stages (128 and 256, with the remainders of K), and of the rule
that chooses between them; tiny (f16 subnormal) scales; infinities and NaN in
the activations (and Q3_K's scales) against the matvec kernels; the slabs of matmul_t_noalloc.

The kernels' block sums are exact integers and their sums over K are 32-bit,
so the outputs are held to 32-bit sums of K / 32 terms: relative L2 2e-6
(the oracle itself sums in f32)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q2K, Q3K, Q5K = 2, 3, 6, 7, 8, 10, 11, 13
BLOCK32 = [Q4_0, Q4_1, Q5_0, Q5_1, Q8_0]
SUPER = [Q2K, Q3K, Q5K]


def upload(blocks, n, k, dt, dev):
    from xn_amd import GgmlDType, QTensor

    return QTensor.from_gguf_bytes(blocks, (n, k), GgmlDType(dt), dev)


def run(qt, x, m, k, n, dev):
    dst = torch.full((m, n), float("nan"), dtype=torch.float32, device=dev)
    qt.matmul_t((m, k, n), torch.from_numpy(x).to(dev), dst)
    return dst.cpu().numpy()


def reaches(kernel, dt, m, k, n):
    """The case is on the kernel that its test is about."""
    from xn_amd.quantized import matmul_t_kernel

    assert matmul_t_kernel(dt, m, n, k) == kernel, f"dt={dt} m={m} k={k} n={n}"


def check(orc, dev, dt, m, k, n, seed, wscale=0.02, xscale=1.0, kernel=None):
    if kernel:
        reaches(kernel, dt, m, k, n)
    rng = np.random.default_rng(seed)
    blocks = orc.from_float(dt, (rng.normal(0, wscale, (n, k))).astype(np.float32))
    x = (rng.normal(0, xscale, (m, k))).astype(np.float32)
    got = run(upload(blocks, n, k, dt, dev), x, m, k, n, dev).astype(np.float64)
    want = orc.matmul(dt, x, blocks, n).astype(np.float64)
    assert np.isfinite(got).all()
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert rel < 2e-6, f"dt={dt} m={m} k={k} n={n}: rel {rel}"


# K-split kernel: one and two row tiles, ragged columns, K stages cut short
@pytest.mark.parametrize("dt", BLOCK32)
@pytest.mark.parametrize("m,k,n", [(9, 64, 31), (32, 192, 33), (33, 1088, 65), (17, 4160, 96), (64, 2048, 8200)])
def test_block_types_ksplit(orc, dev, dt, m, k, n):
    check(orc, dev, dt, m, k, n, 100 + dt + m)


# 16-row tiles (K of whole stages): one tile at any N, an odd count of them, ragged rows and columns
@pytest.mark.parametrize("dt", BLOCK32)
@pytest.mark.parametrize("m,k,n", [(9, 128, 31), (16, 640, 8200), (17, 1152, 33), (47, 4224, 67), (125, 2048, 100)])
def test_block_types_16_rows(orc, dev, dt, m, k, n):
    check(orc, dev, dt, m, k, n, 150 + dt + m, kernel="h16_ksplit16")


# 32-row tiles: one row tile (an even and a ragged one), K in whole and in cut stages
@pytest.mark.parametrize("dt", BLOCK32)
@pytest.mark.parametrize("m,k,n", [(64, 64, 4096), (33, 1088, 4065), (64, 512, 4096), (57, 2240, 4070)])
def test_block_types_32_rows(orc, dev, dt, m, k, n):
    check(orc, dev, dt, m, k, n, 170 + dt + m, kernel="h16_ksplit32")


# 64-row tiles: both row tiles full, the second one ragged or missing, K in whole and in cut stages
@pytest.mark.parametrize("dt", BLOCK32)
@pytest.mark.parametrize("m,k,n", [(64, 1088, 8200), (41, 320, 8250), (70, 192, 8200), (96, 512, 8224)])
def test_block_types_64_rows(orc, dev, dt, m, k, n):
    check(orc, dev, dt, m, k, n, 190 + dt + m, kernel="h16_ksplit64")


@pytest.mark.parametrize("dt", SUPER)
@pytest.mark.parametrize("m,k,n,kernel", [(33, 512, 4065, "h16_ksplit32"), (64, 2304, 4096, "h16_ksplit32"),
                                          (41, 512, 8250, "h16_ksplit64"), (70, 2304, 7900, "h16_ksplit64")])
def test_super_types_row_tiles(orc, dev, dt, m, k, n, kernel):
    check(orc, dev, dt, m, k, n, 350 + dt + m, kernel=kernel)


# more 256 x 64 tiles than one round of workgroups
@pytest.mark.parametrize("dt", BLOCK32 + SUPER)
def test_second_round_of_tiles(orc, dev, dt):
    kernel = "h16_super_tile" if dt in SUPER else "h16_block_tile"
    check(orc, dev, dt, 1100, 256 if dt in SUPER else 64, 4608, 370 + dt, kernel=kernel)


@pytest.mark.parametrize("dt", [Q4_0, Q8_0])
@pytest.mark.parametrize("k", [32, 96, 160, 1056])
def test_odd_block_counts(orc, dev, dt, k):
    check(orc, dev, dt, 37, k, 40, 200 + dt + k)


@pytest.mark.parametrize("dt", SUPER)
@pytest.mark.parametrize("m,k,n", [(9, 256, 31), (32, 512, 33), (33, 2304, 65), (17, 4352, 96), (65, 2048, 8200)])
def test_super_types_ksplit(orc, dev, dt, m, k, n):
    check(orc, dev, dt, m, k, n, 300 + dt + m)


# the 256 x 64 tile: full and ragged last tiles, K past its 16-step output sums
@pytest.mark.parametrize("dt,m,k,n", [(dt, 640, 64, 4353) for dt in BLOCK32] + [(dt, 577, 2112, 4608) for dt in BLOCK32]
                         + [(dt, 600, 4160, 4352) for dt in (Q4_0, Q5_1, Q8_0)])
def test_block_types_tile(orc, dev, dt, m, k, n):
    check(orc, dev, dt, m, k, n, 400 + dt + m, kernel="h16_block_tile")


@pytest.mark.parametrize("dt", [Q4_0, Q8_0])
def test_block_types_tile_odd_blocks(orc, dev, dt):
    check(orc, dev, dt, 600, 1056, 4354, 500 + dt, kernel="h16_block_tile")


@pytest.mark.parametrize("dt", SUPER)
@pytest.mark.parametrize("m,k,n", [(512, 256, 4353), (449, 1280, 4352), (520, 4352, 4096)])
def test_super_types_tile(orc, dev, dt, m, k, n):
    check(orc, dev, dt, m, k, n, 600 + dt + m, kernel="h16_super_tile")


# block scales in the f16 subnormal range, on either side
@pytest.mark.parametrize("dt", BLOCK32 + SUPER)
@pytest.mark.parametrize("wscale,xscale", [(2e-5, 1.0), (0.02, 2e-4)])
def test_subnormal_scales(orc, dev, dt, wscale, xscale):
    check(orc, dev, dt, 40, 1024, 64, 700 + dt, wscale, xscale)


def check_nonfinite(got, want, m):
    """NaN and either infinity where the matvec kernels have them; rows without
    them within 32-bit sums."""
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want).all(axis=1)
    assert ok.sum() >= m - 8
    err = np.linalg.norm(got[ok].astype(np.float64) - want[ok]) / np.linalg.norm(want[ok].astype(np.float64))
    assert err < 2e-6


def run_both(orc, dev, dt, m, k, n, x, seed):
    """(matmul_t, the matvec kernels') of random weights on x."""
    from xn_amd.quantized import set_route

    blocks = orc.from_float(dt, np.random.default_rng(seed).normal(0, 0.02, (n, k)).astype(np.float32))
    qt = upload(blocks, n, k, dt, dev)
    got = run(qt, x, m, k, n, dev)
    try:
        set_route(1)
        return got, run(qt, x, m, k, n, dev)
    finally:
        set_route(0)


# (m, n): 16-row tiles, one and two 32-row tiles of the K-split kernel, the 256 x 64 tile
NONFINITE_TILES = [(40, 64), (64, 4096), (64, 8224), (600, 4352)]


@pytest.mark.parametrize("dt", [Q4_1, Q5_1])
@pytest.mark.parametrize("m,n", NONFINITE_TILES)
def test_overflowing_block_sums(orc, dev, dt, m, n):
    """A Q8_1 sum past the f16 range beside a finite scale, alone in its stage of
    four blocks, beside one of the other sign, and from a single large element."""
    k = 320
    x = np.random.default_rng(5850 + dt).normal(0, 1, (m, k)).astype(np.float32)
    x[3, 64:96], x[5, 128:160], x[7, 40], x[9, 288:] = 3000.0, -3000.0, 7e4, 2500.0
    x[11, 0:32], x[11, 96:128] = 3000.0, -3000.0
    reaches({40: "h16_ksplit16", 600: "h16_block_tile"}.get(m, "h16_ksplit32" if n == 4096 else "h16_ksplit64"), dt, m, k, n)
    got, want = run_both(orc, dev, dt, m, k, n, x, 850 + dt)
    assert np.isinf(want[[3, 5, 7, 9]]).any(axis=1).all()
    check_nonfinite(got, want, m)


@pytest.mark.parametrize("dt,k", [(Q8_0, 1056), (Q4_0, 160), (Q4_1, 576), (Q5_0, 576), (Q5_1, 320)])
@pytest.mark.parametrize("m,n", NONFINITE_TILES)
def test_overflowing_scale_in_a_cut_stage(orc, dev, dt, k, m, n):
    """An infinite activation scale in the last block of a K that is not whole
    stages of four blocks: the blocks that fill the stage up add nothing."""
    x = np.random.default_rng(5870 + dt).normal(0, 1, (m, k)).astype(np.float32)
    x[3, -5], x[5, k - 32] = 1e9, -1e9
    few = "h16_ksplit32" if dt in (Q4_0, Q8_0) else "h16_ksplit16"  # (scales of their own: no 16-row tiles of a cut stage)
    reaches({40: few, 600: "h16_block_tile"}.get(m, "h16_ksplit32" if n == 4096 else "h16_ksplit64"), dt, m, k, n)
    got, want = run_both(orc, dev, dt, m, k, n, x, 870 + dt)
    if dt not in (Q4_1, Q5_1):  # (their infinite sum times m meets the infinite product)
        assert np.isinf(want[[3, 5]]).any(axis=1).all()
    check_nonfinite(got, want, m)


@pytest.mark.parametrize("dt", [Q4_0, Q4_1, Q8_0, Q2K, Q5K])
@pytest.mark.parametrize("m,n", [(40, 64), (600, 3840)])
def test_nonfinite_rows(orc, dev, dt, m, n):
    """An infinity, a NaN and an overflowing scale in an activation row reach
    the same outputs as on the matvec kernels, and no other row."""
    from xn_amd.quantized import set_route

    rng = np.random.default_rng(800 + dt)
    k = 512
    blocks = orc.from_float(dt, rng.normal(0, 0.02, (n, k)).astype(np.float32))
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    x[3, 7], x[5, 300], x[20, 40] = np.inf, np.nan, 1e9
    x[8] = 0.0
    few = "h16_ksplit32" if dt in SUPER else "h16_ksplit16"
    reaches(few if m == 40 else "h16_super_tile" if dt in SUPER else "h16_block_tile", dt, m, k, n)
    qt = upload(blocks, n, k, dt, dev)
    got = run(qt, x, m, k, n, dev)
    try:
        set_route(1)
        want = run(qt, x, m, k, n, dev)
    finally:
        set_route(0)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    assert (got[8] == 0).all()
    ok = np.isfinite(want).all(axis=1)
    err = np.linalg.norm(got[ok].astype(np.float64) - want[ok]) / np.linalg.norm(want[ok].astype(np.float64))
    assert err < 2e-6


@pytest.mark.parametrize("m,n,kernel", [(40, 64, "h16_ksplit32"), (64, 8224, "h16_ksplit64"), (512, 4384, "h16_super_tile")])
def test_infinite_q3k_block_scales(orc, dev, m, n, kernel):
    """The reference multiplies eight sums of a super-block by its scale; an infinite one
    leaves NaN unless all eight are of one sign (1 output in 128), as on the matvec kernels."""
    from xn_amd.quantized import set_route

    k = 512
    reaches(kernel, Q3K, m, k, n)
    rng = np.random.default_rng(940)
    blocks = np.frombuffer(bytes(orc.from_float(Q3K, rng.normal(0, 0.02, (n, k)).astype(np.float32))), np.uint8).copy()
    cols = {3: np.inf, 31: -np.inf, 33: np.nan, n - 1: np.inf}
    for c, v in cols.items():
        blocks.reshape(n, k // 256, 110)[c, c % 2, 108:] = np.array([v], np.float16).view(np.uint8)
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    qt, xt = upload(blocks, n, k, Q3K, dev), torch.from_numpy(x).to(dev)
    outs = [torch.empty((m, n), device=dev) for _ in range(3)]
    qt.matmul_t((m, k, n), xt, outs[0])
    qt.matmul_t_split((m, k, n), xt, outs[1])
    try:
        set_route(1)
        qt.matmul_t((m, k, n), xt, outs[2])
    finally:
        set_route(0)
    got, rows, want = (y.cpu().numpy() for y in outs)
    hit = np.isin(np.arange(n), list(cols))
    assert np.isnan(want[:, hit]).mean() > 0.9
    for y in (got, rows):
        assert np.isnan(y[:, hit]).all() and np.isfinite(y[:, ~hit]).all()


@pytest.mark.parametrize("dt", [Q8_0, Q5K])
def test_noalloc_slabs(orc, dev, dt):
    """More rows than the static scratch holds with their f16 copy, but not
    without it: the same outputs as with a workspace."""
    from xn_amd import XnqError

    k, n, m = 4096, 64, 8000
    rng = np.random.default_rng(900 + dt)
    blocks = orc.from_float(dt, rng.normal(0, 0.02, (n, k)).astype(np.float32))
    qt = upload(blocks, n, k, dt, dev)
    assert qt.matmul_t_workspace_size(m) > (64 << 20)
    x = torch.randn((m, k), generator=torch.Generator(device=dev).manual_seed(5), device=dev)
    want = torch.empty((m, n), device=dev)
    got = torch.full((m, n), float("nan"), device=dev)
    qt.matmul_t((m, k, n), x, want)
    qt.matmul_t_noalloc((m, k, n), x, got)
    assert ((got - want).norm() / want.norm()).item() < 1e-6
    # past the rows whose images alone fill it, it refuses as before
    big = torch.zeros((16000, k), device=dev)
    with pytest.raises(XnqError, match="scratch"):
        qt.matmul_t_noalloc((16000, k, n), big, torch.empty((16000, n), device=dev))
