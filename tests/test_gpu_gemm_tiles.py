"""The tile GEMM (prompts) at the edges of its tiles, K slices and K groups:
every tile shape, ragged rows and columns, odd block counts, split and
unsplit, on both combines and under graph replay."""
import numpy as np
import pytest

from parity import check_parity, exact_f64, exact_f64_cond
from rdlquant import synth

pytestmark = pytest.mark.gpu

# smallest (one block, one column), both sides of a 64-row x tile and a 64-column
# weight tile, odd block counts (blocks 2 bytes past a dword, the matrix ending
# inside one), K in 16 / 8 / 4 / 2 slices with a ragged last one, 256 x 128 tiles,
# and rows longer than one workgroup's registers hold (k > 16384)
# (the rows before 257 with k <= 2048 stay on the small-tile kernel)
SHAPES = [(65, 1, 32), (65, 1, 4096), (65, 65, 2080), (129, 63, 4128), (128, 1024, 4096), (80, 4096, 2080),
          (257, 130, 96), (257, 6000, 544), (300, 14400, 96), (513, 4097, 288), (2049, 65, 32), (70, 40, 16416)]


@pytest.mark.parametrize("kind,dtype", [("q4", 2), ("q8", 8)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_tiles(rq, orc, gpu, kind, dtype, m, n, k):
    print(f"case {kind} tiles m={m} n={n} k={k}", flush=True)
    x = synth.activations(m, k, m + n + k)
    w = synth.weights(dtype, n, k, m + n)
    got = getattr(rq, f"matmul_f32_{kind}")(x, w, m, k, n).reshape(m, n)
    rows = np.unique(np.linspace(0, m - 1, 24).astype(int))
    want = orc.matmul(kind, x[rows], w, len(rows), k, n, threads=16)
    check_parity(got[rows].reshape(-1), want, exact_f64(orc, kind, x[rows], w, len(rows), k, n))


# 5 to 64 rows on the tiles: matrices of many strips and of few, ragged, each
# side of 16 and 32 rows; and the x-tile kernel's slices of 16 (many strips; a
# ragged last slice; an odd block count) and of 32 (one round)
@pytest.mark.parametrize("m,n,k", [(5, 24601, 4096), (16, 500, 4224), (17, 510, 544), (31, 4090, 13344), (32, 64, 4096), (33, 4100, 4128),
                                   (64, 1000, 2080), (64, 1, 16384), (16, 8200, 4096), (9, 2050, 14368),
                                   (5, 6150, 2080), (16, 4096, 8192)])
def test_few_rows(rq, orc, gpu, m, n, k):
    print(f"case few rows m={m} n={n} k={k}", flush=True)
    x = synth.activations(m, k, m + n + k)
    w = synth.q4_0_weights(n, k, m + n)
    got = rq.matmul_f32_q4(x, w, m, k, n).reshape(m, n)
    rows = np.unique(np.linspace(0, m - 1, 8).astype(int))
    want = orc.matmul("q4", x[rows], w, len(rows), k, n, threads=16)
    check_parity(got[rows].reshape(-1), want, exact_f64(orc, "q4", x[rows], w, len(rows), k, n))


@pytest.mark.parametrize("kind,dtype,m,k", [("q4", 2, 20, 1024), ("q4", 2, 40, 1024), ("q4", 2, 300, 1024),
                                            ("q8", 8, 40, 4096), ("q8", 8, 300, 4096)])
def test_rows_with_an_infinite_value(rq, orc, gpu, kind, dtype, m, k):
    # +-inf where the weight is not zero, NaN where it is, as in the reference;
    # rows beside it and a row's own finite values keep theirs
    n = 300
    x = synth.activations(m, k, 21 + m)
    x[3, 77], x[5, 900] = np.inf, -np.inf
    w = synth.weights(dtype, n, k, 22)
    got = getattr(rq, f"matmul_f32_{kind}")(x, w, m, k, n).reshape(m, n)
    want = orc.matmul(kind, x[[3, 5]], w, 2, k, n).reshape(2, n)
    assert np.array_equal(got[[3, 5]], want, equal_nan=True)
    assert np.isfinite(np.delete(got, [3, 5], axis=0)).all()


# the formats whose operands or sums are split again, and the small-tile kernel: such
# rows are infinite or NaN throughout (inf - inf, inf times a zero half), others untouched
@pytest.mark.parametrize("kind,dtype,m,k", [("q4_k", 12, 70, 4096), ("q6_k", 14, 70, 4096), ("q4", 2, 100, 1024)])
def test_rows_with_an_infinite_value_elsewhere(rq, gpu, kind, dtype, m, k):
    n = 300
    x = synth.activations(m, k, 23 + m)
    x[3, 77], x[5, 900] = np.inf, -np.inf
    got = getattr(rq, f"matmul_f32_{kind}")(x, synth.weights(dtype, n, k, 24), m, k, n).reshape(m, n)
    assert not np.isfinite(got[[3, 5]]).any()
    assert np.isfinite(np.delete(got, [3, 5], axis=0)).all()


# one 16-row x tile and just past one, both sides of the 128-row weight tiles,
# one super-block a row and 17 (the last slice shorter), odd super-block counts
# (Q6_K rows starting 2 bytes past a dword), the K split, a partial last round
@pytest.mark.parametrize("kind,dtype", [("q4k", 12), ("q6k", 14)])
@pytest.mark.parametrize("m,n,k", [(16, 8192, 256), (32, 1, 4096), (33, 127, 4352), (65, 129, 4096), (128, 2048, 2048),
                                   (130, 8200, 768), (400, 4096, 256)])
def test_super_block_tiles(rq, orc, gpu, kind, dtype, m, n, k):
    print(f"case {kind} tiles m={m} n={n} k={k}", flush=True)
    x = synth.activations(m, k, m + n + k)
    w = synth.weights(dtype, n, k, m + n)
    got = getattr(rq, "matmul_f32_q4_k" if dtype == 12 else "matmul_f32_q6_k")(x, w, m, k, n).reshape(m, n)
    rows = np.unique(np.linspace(0, m - 1, 20).astype(int))
    want = orc.matmul(kind, x[rows], w, len(rows), k, n, threads=16)
    exact, cond = exact_f64_cond(orc, kind, x[rows], w, len(rows), k, n)
    check_parity(got[rows].reshape(-1), want, exact, cond=cond)


@pytest.mark.parametrize("kind,dtype", [("q4k", 12), ("q6k", 14)])
def test_super_block_tiles_extreme_scales(rq, orc, gpu, kind, dtype):
    # d (and dmin) from 2^-24 to 2^10 within a row, scale bytes at both ends.  Each
    # output within 1e-6 sum |w x|: 2^-23 for the x split, as much for Q6_K's
    # dropped lo lo and Q4_K's f16 pairs, and f32 sums of 16 super-blocks
    m, n, k = 40, 130, 4096
    r = np.random.default_rng(7)
    ns = k // 256
    w = synth.weights(dtype, n, k, 8).reshape(n, ns, -1).copy()
    half = lambda: synth.f16_bits(2.0 ** r.integers(-24, 11, size=(n, ns)))[..., None].view(np.uint8).reshape(n, ns, 2)
    if dtype == 12:
        w[..., 0:2], w[..., 2:4] = half(), half()
        w[0, :, 4:16], w[1, :, 4:16] = 0xFF, 0x00
    else:
        w[..., 208:210] = half()
        w[0, :, 192:208], w[1, :, 192:208] = 0x80, 0x00
    x = synth.activations(m, k, 9) * (10.0 ** r.uniform(-6, 4, size=(m, 1))).astype(np.float32)
    got = getattr(rq, "matmul_f32_q4_k" if dtype == 12 else "matmul_f32_q6_k")(x, w.reshape(-1), m, k, n)
    exact, cond = exact_f64_cond(orc, kind, x, w.reshape(-1), m, k, n)
    assert np.all(np.abs(got - exact) <= 1e-6 * cond)
    assert np.all(got.reshape(m, n)[:, 1] == 0.0)


# every tile split, no tile split (Q4_0: the small-tile kernel), whole tiles with a
# split last round; two inputs in turn
# through one workspace, so that a partial of the call before shows
@pytest.mark.parametrize("kind,dtype", [("q4", 2), ("q8", 8), ("q4k", 12), ("q6k", 14)])
@pytest.mark.parametrize("m,n,k", [(128, 1024, 4096), (100, 4096, 1024), (300, 7000, 4096)])
def test_split_tiles_combines_and_replays_agree(rq, orc, gpu, kind, dtype, m, n, k):
    # the XCD-local and the agent-coherent combine and a captured call give the
    # same bits, call after call (the counters return to zero), and each is within
    # 1e-6 sum |w x| of the exact product
    import torch
    print(f"case split tiles {kind} m={m} n={n} k={k}", flush=True)
    raw = synth.weights(dtype, n, k, 5)
    w = rq.Weight.upload(raw, dtype, n, k)
    hosts = [synth.activations(m, k, seed) for seed in (6, 7)]
    xs = [torch.from_numpy(h).to(gpu) for h in hosts]
    rows = np.unique(np.linspace(0, m - 1, 16).astype(int))
    exact = [exact_f64_cond(orc, kind, h.reshape(m, k)[rows], raw, len(rows), k, n) for h in hosts]
    main = torch.cuda.current_stream().cuda_stream

    def product(i):
        y = torch.full((m, n), np.nan, device=gpu)
        w.forward_dev(xs[i].data_ptr(), m, y.data_ptr(), rq.MODE_FLOAT, main)
        return y

    def check(i, y):
        want, cond = exact[i]
        assert np.all(np.abs(y.cpu().numpy()[rows].reshape(-1) - want) <= 1e-6 * cond)
        assert torch.equal(y, first[i])

    local = [product(i % 2) for i in range(6)]
    try:
        rq.set_gemm_combine(rq.COMBINE_COHERENT)
        coherent = [product(i % 2) for i in range(6)]
    finally:
        rq.set_gemm_combine(rq.COMBINE_AUTO)
    first = local[:2]
    for i, (a, b) in enumerate(zip(local, coherent)):
        check(i % 2, a)
        check(i % 2, b)
    g, side, x, y = torch.cuda.CUDAGraph(), torch.cuda.Stream(), xs[0].clone(), torch.empty(m, n, device=gpu)
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=side):
        w.forward_dev(x.data_ptr(), m, y.data_ptr(), rq.MODE_FLOAT, side.cuda_stream)
    for i in (1, 0, 1, 0):
        x.copy_(xs[i])
        y.fill_(np.nan)
        g.replay()
        torch.cuda.synchronize()
        check(i, y)
        check(1 - i, product(1 - i))
    w.free()


# native mode past 64 rows: the smallest product that takes the tiles below 256
# rows, ragged tiles and slices, odd block counts, and both sides of 256 and
# 1024 rows and of k = 16384 (the int8 kernel)
@pytest.mark.parametrize("m,n,k", [(65, 4096, 4096), (65, 4093, 4128), (255, 100, 4096), (256, 1, 32), (300, 257, 544),
                                   (513, 130, 4128), (1024, 64, 2080), (1030, 2049, 96), (257, 33, 16384),
                                   (257, 33, 16416)])
def test_native_tiles(rq, orc, gpu, m, n, k):
    print(f"case native tiles m={m} n={n} k={k}", flush=True)
    x = synth.activations(m, k, m + n + k)
    w = synth.q4_0_weights(n, k, m + n)
    got = rq.matmul_f32_q4_native(x, w, m, k, n).reshape(m, n)
    rows = np.unique(np.linspace(0, m - 1, 12).astype(int))
    want = orc.matmul("q4_native", x[rows], w, len(rows), k, n, 16)
    part = orc.block_dots(x[rows], w, len(rows), k, n).reshape(len(rows), n, k // 32).astype(np.float64)
    sw = w.reshape(n, k // 32, 18)[:, :, 0:2].copy().view(np.float16).astype(np.float64)[..., 0]
    sx = np.stack([orc.quantize_row_q8_0(x[r])[1] for r in rows]).astype(np.float64)
    check_parity(got[rows].reshape(-1), want, (part * sx[:, None, :] * sw[None]).sum(axis=2).reshape(-1))


def test_native_tiles_nan_inf_and_zero_rows(rq, orc, gpu):
    # NaN scores as code 0 and a zero block as scale 0; an overflowing block
    # scale makes every output of its row NaN, as in the reference
    m, n, k = 300, 70, 512
    x = synth.activations(m, k, 95)
    x[2, 5], x[4], x[7, 40], x[9, 300] = np.nan, 0.0, np.inf, 1e9
    x[11] *= 1e-7
    w = synth.q4_0_weights(n, k, 96)
    rows = np.array([0, 2, 4, 7, 9, 11, 12])
    got = rq.matmul_f32_q4_native(x, w, m, k, n).reshape(m, n)
    want = orc.matmul("q4_native", x[rows], w, len(rows), k, n, 4).reshape(len(rows), n)
    assert np.array_equal(np.isnan(got[rows]), np.isnan(want))
    ok = ~np.isnan(want)
    # 2^-22 of a split x element and f32 sums of 16 blocks, over sum |w x| <= 16 x
    # the largest output of a row here
    tol = 1e-6 * 16 * np.abs(np.where(ok, want, 0.0)).max(axis=1, keepdims=True) * np.ones_like(want)
    assert np.all(np.abs(got[rows] - want)[ok] <= tol[ok])
    assert np.isfinite(np.delete(got, [7, 9], axis=0)).all()


def wide_rows(m, k, seed, low):
    """Rows of three kinds in turn: an outlier block (2^10) with every other block
    `low` binades or more below it, an ordinary row, a row of zeros and tiny values."""
    r = np.random.default_rng(seed)
    x = synth.activations(m, k, seed).reshape(m, k // 32, 32)
    x[0::3] *= (2.0 ** -(low - 10.0 + r.integers(0, 8, size=x[0::3].shape[:2])))[..., None]
    x[0::3, 0] *= 2.0 ** (low - 10.0) * 2.0 ** 10
    x[2::3, 1:] *= 1e-30
    x[2::3, 0] = 0.0
    return np.ascontiguousarray(x.reshape(m, k), dtype=np.float32)


def weights_without_block_0(n, k, seed):
    """Q4_0 weights whose first block has the code of zero throughout."""
    w = synth.q4_0_weights(n, k, seed).reshape(n, k // 32, 18).copy()
    w[:, 0, 2:] = 0x88
    return w.reshape(-1)


# A row's other blocks count for all of a result where its largest block meets
# zero weights.  5 to 64 rows on each tile shape, split and unsplit, ragged, and
# (16 x 4096 x 4096) on the x-tile kernel.  Each output within 1e-6 sum |w x|:
# 2^-22 a split element, f32 sums of 33 to 512 blocks whose roundings (2^-24
# each) add up as a random walk
@pytest.mark.parametrize("low", [11, 15, 20, 27, 40])
@pytest.mark.parametrize("m,n,k", [(16, 4096, 4096), (16, 510, 4128), (7, 24600, 4096), (32, 300, 16384), (64, 1000, 2080),
                                   (64, 14336, 4096), (33, 4100, 4128)])
def test_rows_of_wide_range(rq, orc, gpu, m, n, k, low):
    print(f"case wide rows m={m} n={n} k={k} low={low}", flush=True)
    x, w = wide_rows(m, k, m + n + low, low), weights_without_block_0(n, k, n)
    got = rq.matmul_f32_q4(x, w, m, k, n).reshape(m, n)
    rows = np.unique(np.linspace(0, m - 1, 9).astype(int))
    exact, cond = exact_f64_cond(orc, "q4", x[rows], w, len(rows), k, n)
    assert np.all(np.abs(got[rows].reshape(-1) - exact) <= 1e-6 * cond)


# the same in native mode: the int32 dots times both scales, in 64 bits (a
# scale of x below the f16 range is 0, as in the reference)
@pytest.mark.parametrize("low", [11, 20, 24, 30])
@pytest.mark.parametrize("m,n,k", [(65, 4096, 4096), (257, 70, 4128), (513, 1000, 4096), (1030, 2049, 96),
                                   (512, 14336, 2048)])
def test_native_rows_of_wide_range(rq, orc, gpu, m, n, k, low):
    print(f"case native wide rows m={m} n={n} k={k} low={low}", flush=True)
    x, w = wide_rows(m, k, m + n + low, low), weights_without_block_0(n, k, n)
    x[2::3] = x[0:m - 2:3][:len(x[2::3])] * 2.0 ** 9  # (in the f16 scales' range)
    got = rq.matmul_f32_q4_native(x, w, m, k, n).reshape(m, n)
    rows = np.unique(np.linspace(0, m - 1, 9).astype(int))
    part = orc.block_dots(x[rows], w, len(rows), k, n).reshape(len(rows), n, k // 32).astype(np.float64)
    sw = w.reshape(n, k // 32, 18)[:, :, 0:2].copy().view(np.float16).astype(np.float64)[..., 0]
    sx = np.stack([orc.quantize_row_q8_0(x[r])[1] for r in rows]).astype(np.float64)
    terms = part * sx[:, None, :] * sw[None]
    # (within a block the products cancel before the f32 sum: 16 times the block's
    # dot covers that here)
    assert np.all(np.abs(got[rows] - terms.sum(axis=2)) <= 1e-6 * (np.abs(terms).sum(axis=2) * 16 + 1e-30))


def test_wide_row_with_an_infinite_value(rq, orc, gpu):
    m, n, k = 40, 300, 1024
    x, w = wide_rows(m, k, 3, 24), weights_without_block_0(n, k, 4)
    x[3, 77], x[6, 900] = np.inf, -np.inf
    got = rq.matmul_f32_q4(x, w, m, k, n).reshape(m, n)
    want = orc.matmul("q4", x[[3, 6]], w, 2, k, n).reshape(2, n)
    assert np.array_equal(got[[3, 6]], want, equal_nan=True)
    assert np.isfinite(np.delete(got, [3, 6], axis=0)).all()


# K-quant rows keep one power of two a row, so an element of a block 2^low below
# the row's largest is known to 2^(low - 40) of that block's largest (half of 2^-24
# of x' over 2^15-low); the block's sum, for Q4_K's minimums, has to be as good
@pytest.mark.parametrize("kind,dtype", [("q4k", 12), ("q6k", 14)])
@pytest.mark.parametrize("low", [14, 17, 20, 24, 28])
def test_super_block_rows_of_wide_range(rq, orc, gpu, kind, dtype, low):
    print(f"case super block wide rows {kind} low={low}", flush=True)
    m, n, k = 70, 257, 4096
    x = synth.activations(m, k, low).reshape(m, k // 32, 32) * np.float32(2.0 ** -low)
    x[:, 0] *= np.float32(2.0 ** low)
    x = np.ascontiguousarray(x.reshape(m, k))
    w = synth.weights(dtype, n, k, 5).reshape(n, k // 256, -1).copy()
    if dtype == 12:  # the first 32 elements: scale and min 0
        w[:, 0, 4] &= 0xC0
        w[:, 0, 8] &= 0xC0
    else:
        w[:, 0, 192:194] = 0
    w = w.reshape(-1)
    got = getattr(rq, "matmul_f32_q4_k" if dtype == 12 else "matmul_f32_q6_k")(x, w, m, k, n)
    exact, cond = exact_f64_cond(orc, kind, x, w, m, k, n)
    assert np.all(np.abs(got - exact) <= (2.0 ** -22 + 2.0 ** (low - 40)) * cond)


def test_q4_k_minimum_scale_without_minimums(rq, orc, gpu):
    # dmin far above d where every sub-block's minimum is 0 (and the other way round)
    m, n, k = 70, 130, 4096
    r = np.random.default_rng(11)
    w = synth.weights(12, n, k, 12).reshape(n, k // 256, 144).copy()
    small = synth.f16_bits((1.0 + r.random((n, k // 256))) * 2.0 ** -18)[..., None].view(np.uint8).reshape(n, k // 256, 2)
    big = synth.f16_bits((1.0 + r.random((n, k // 256))) * 2.0 ** 12)[..., None].view(np.uint8).reshape(n, k // 256, 2)
    w[..., 0:2], w[..., 2:4] = small, big
    w[..., 4:8] &= 0x3F      # sub-blocks 0-3: scales; 4-7's high bits
    w[..., 8:12] = 0
    w[..., 12:16] &= 0x0F
    half = n // 2            # these rows: d large, scales 0, minimums in use
    w[half:, :, 0:2], w[half:, :, 2:4] = big[half:], small[half:]
    w[half:, :, 8:12] = w[half:, :, 4:8]
    w[half:, :, 4:8] = 0
    w[half:, :, 12:16] <<= 4
    w = w.reshape(-1)
    x = synth.activations(m, k, 13)
    got = rq.matmul_f32_q4_k(x, w, m, k, n)
    exact, cond = exact_f64_cond(orc, "q4k", x, w, m, k, n)
    assert np.all(np.abs(got - exact) <= 1e-6 * cond)
