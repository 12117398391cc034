"""The products' bf16 parts (gemm_x.hpp): the range of values they hold, the
values that are not finite, and the edges of the tiles that split K over
groups of waves."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oxforge
from oxforge import synth

pytestmark = pytest.mark.gpu

U32 = 2.0 ** -24
TILES = ["128x128x32_x", "64x128x32_x8", "64x64x32_x16", "128x128x32_2x2_g", "64x128x32_2x2_g8",
         "64x64x32_2x2_g16", "64x64x16_2x2_g", "32x32x32_d", "32x32x32_2x2_gd"]


@pytest.fixture(scope="module")
def rt():
    with oxforge.Runtime(0) as r:
        yield r


def say(msg):
    print(f"[case] {msg}", flush=True)


def product(rt, A, B, M, N, K, ta=0, tb=0, tile=None):
    dC = rt.empty((M, N))
    if tile:
        rt.gemm_ex_tile(tile, rt.array(A), rt.array(B), dC, M, N, K, trans_a=ta, trans_b=tb)
    else:
        rt.gemm_ex(rt.array(A), rt.array(B), dC, M, N, K, trans_a=ta, trans_b=tb)
    return dC.numpy()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_group_and_guard_edges(rt, tile, ta, tb):
    """K from one slab to every count of slabs per group (with a ragged last
    slab on guarded tiles), one row or column short of the tile and one past
    it: within (K + 8) u of |A| |B| of the f64 product (every order of K
    rounded additions; the parts left out of a product are at most
    (1 + 2^-10) u of it)."""
    bm, bn = (int(x) for x in tile.split("x")[:2])
    guarded = "_g" in tile
    sizes = [(bm, bn)] + ([(bm - 1, bn + 1), (1, 3), (bm + 3, bn - 2)] if guarded else [])
    for M, N in sizes:
        for K in [32, 64, 96, 160, 288, 544] + ([1, 7, 31, 33, 127, 130, 257] if guarded else []):
            say(f"{tile} ta={ta} tb={tb} {M}x{N}x{K}")
            A = synth.uniform((K, M) if ta else (M, K), M + K)
            B = synth.uniform((N, K) if tb else (K, N), N + K)
            a, b = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
            C = product(rt, A, B, M, N, K, ta, tb, tile)
            assert np.all(np.abs(C - a @ b) <= (K + 8) * U32 * (np.abs(a) @ np.abs(b))), (M, N, K)


@pytest.mark.parametrize("tile", TILES)
def test_values_that_are_not_finite(rt, tile):
    """Infinities, NaN and the largest and smallest f32 values in the operands:
    each output is NaN, +inf or -inf where the exact product is, and finite
    and close elsewhere (the lowest f32 value, a usual mask, stays finite)."""
    bm, bn = (int(x) for x in tile.split("x")[:2])
    M, N, K = bm, bn, 288
    say(f"special values {tile}")
    A, B = synth.uniform((M, K), 1), synth.uniform((K, N), 2)
    big = np.finfo(np.float32).max
    A[1, 5], A[2, 40], A[3, 100], A[4, 200] = np.inf, -np.inf, np.nan, big
    A[5, 7], A[5, 250] = np.inf, -np.inf
    A[6, :], A[6, 3] = 0.0, -big
    A[7, :], A[7, 9] = 0.0, np.inf
    B[5, :] = np.where(np.arange(N) % 2, 1.0, -0.5)  # parts of B that are zero
    B[3, 0], B[9, 1], B[64, 2], B[65, 3] = 0.5, 0.0, np.inf, np.nan
    C = product(rt, A, B, M, N, K, tile=tile)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = A.astype(np.float64) @ B.astype(np.float64)
        ref[np.abs(ref) > big] = np.sign(ref[np.abs(ref) > big]) * np.inf
    assert np.array_equal(np.isnan(C), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(np.isinf(C), inf) and np.array_equal(C[inf], ref[inf].astype(np.float32))
    ok = np.isfinite(ref)
    scale = np.abs(np.where(np.isfinite(A), A, 0)).astype(np.float64) @ \
        np.abs(np.where(np.isfinite(B), B, 0)).astype(np.float64)
    assert np.all(np.abs(C[ok] - ref[ok]) <= (K + 8) * U32 * scale[ok])


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("K", [96, 544])
def test_values_whose_parts_are_not_f32(rt, tile, ta, tb, K):
    """Values whose bf16 parts behave otherwise than they do in f32: infinities
    against the smallest values (both ways round), a NaN with its payload in
    the low bits only, a product beyond the f32 range against a sum of the
    other sign, and the largest finite value against zeros and ones.  Each
    output is what f32 multiply-adds give: NaN and infinities as the f64
    product's, the others within (K + 8) u of |A| |B|."""
    M, N = (int(x) for x in tile.split("x")[:2])
    say(f"parts that are not f32: {tile} ta={ta} tb={tb} K={K}")
    A, B = synth.uniform((M, K), 11), synth.uniform((K, N), 12)
    big = np.finfo(np.float32).max
    B[5, :] = np.where(np.arange(N) % 2, 2.0 ** -140, -2.0 ** -149)
    A[1, 5], A[2, 5] = np.inf, -np.inf
    A[3, 20], B[20, 3] = 2.0 ** -149, np.inf
    A[4, 20], B[K - 1, 4] = -2.0 ** -135, -np.inf
    A[5, 9] = np.array([0x7F800001], np.uint32).view(np.float32)[0]
    A[6, :], A[6, 0], A[6, 1] = 0.0, -3e38, 2e19
    B[0, :], B[1, :] = 1.0, 2e19
    A[7, :], A[7, 0] = 0.0, big
    a, b = (A.T.copy() if ta else A), (B.T.copy() if tb else B)
    C = product(rt, a, b, M, N, K, ta, tb, tile)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(C), np.isnan(ref)), np.argwhere(np.isnan(C) != np.isnan(ref))[:4]
    inf = np.isinf(ref)
    assert np.array_equal(np.isinf(C), inf), np.argwhere(np.isinf(C) != inf)[:4]
    assert np.array_equal(C[inf], ref[inf].astype(np.float32))
    ok = np.isfinite(ref)
    scale = np.abs(np.where(np.isfinite(A), A, 0)).astype(np.float64) @ \
        np.abs(np.where(np.isfinite(B), B, 0)).astype(np.float64)
    assert np.all(np.abs(C[ok] - ref[ok]) <= (K + 8) * U32 * scale[ok])


# Mantissas whose parts leave out the most: of a truncated hi, of a rounded one.
WORST = np.array([0x3F80FF80, 0x3F807F80, 0x3F817F80, 0x3FFFFF80, 0x3F80807F, 0xBF80FF80],
                 np.uint32).view(np.float32)


@pytest.mark.parametrize("tile", [t for t in TILES if "_g" in t] + [None])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_short_sums(rt, tile, ta, tb):
    """Sums of up to three products are formed by f32 multiply-adds, K u of
    |A| |B|, one product rounded once; sums of four keep within that bound and
    what the parts leave out.  Among the operands are the mantissas of which
    that is the most."""
    M, N = (int(x) + 1 for x in tile.split("x")[:2]) if tile else (70, 300)
    rng = np.random.default_rng(13)
    for K in (1, 2, 3, 4):
        say(f"short sums {tile} ta={ta} tb={tb} K={K}")
        for worst in (False, True):
            A = rng.choice(WORST, (M, K)) if worst else synth.uniform((M, K), K)
            B = rng.choice(WORST, (K, N)) if worst else synth.uniform((K, N), K + 20)
            C = product(rt, A.T.copy() if ta else A, B.T.copy() if tb else B, M, N, K, ta, tb, tile)
            a, b = A.astype(np.float64), B.astype(np.float64)
            tol = (K * (1 + K * U32) if K < 4 else K + 1) * U32 * (np.abs(a) @ np.abs(b))
            assert K > 1 or np.array_equal(C, A * B)
            assert np.all(np.abs(C - a @ b) <= tol), (K, worst)


@pytest.mark.parametrize("tile", TILES)
def test_sums_of_one_product(rt, tile):
    """One product that is not zero in each sum: what the parts leave out,
    (1 + 2^-10) u of it, and two roundings (of the small parts' sum, below
    2^-7 of it, and of the result)."""
    M, N = (int(x) for x in tile.split("x")[:2])
    rng = np.random.default_rng(14)
    for K in (32, 288):
        say(f"sums of one product {tile} K={K}")
        A, B = np.zeros((M, K), np.float32), rng.choice(WORST, (K, N))
        A[np.arange(M), rng.integers(0, K, M)] = rng.choice(WORST, M)
        C = product(rt, A, B, M, N, K, tile=tile)
        ref = A.astype(np.float64) @ B.astype(np.float64)
        assert np.all(np.abs(C - ref) <= (2 + 2.0 ** -6) * U32 * np.abs(ref)), K


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_smallest_operands(rt, tile, ta, tb):
    """Rows of A and columns of B down to the smallest f32 values, whose parts
    bf16 does not hold, against values of 2^100: within (K + 8) u of |A| |B|
    like any others, and the elements of other rows and columns are bit for
    bit those of a product without them."""
    M, N = (int(x) for x in tile.split("x")[:2])
    for K in (96, 544):
        say(f"smallest operands {tile} ta={ta} tb={tb} K={K}")
        A, B = synth.uniform((M, K), 15), synth.uniform((K, N), 16)
        A[:, ::7] *= np.float32(2.0 ** 100)
        B[3::7, :] *= np.float32(2.0 ** 100)
        flat = lambda X, t: X.T.copy() if t else X  # noqa: E731
        plain = product(rt, flat(A, ta), flat(B, tb), M, N, K, ta, tb, tile)
        rows, cols = {}, {}
        for i, e in enumerate((-149, -148, -140, -134, -133, -126, -118, -111)):
            r, c = (3 * i + 1) % M, (3 * i + 2) % N
            A[r] = np.ldexp(synth.uniform((K,), 30 + i), e).astype(np.float32)
            rows[r] = e
            if i % 2:
                B[:, c] = np.ldexp(synth.uniform((K,), 40 + i), e).astype(np.float32)
                cols[c] = e
        C = product(rt, flat(A, ta), flat(B, tb), M, N, K, ta, tb, tile)
        a, b = A.astype(np.float64), B.astype(np.float64)
        err, scale = np.abs(C - a @ b), np.abs(a) @ np.abs(b)
        # (f32 results under 2^-126 are whole multiples of 2^-149)
        assert np.all(err <= (K + 8) * U32 * scale + K * 2.0 ** -149), float((err / scale).max())
        other = np.ix_([r for r in range(M) if r not in rows], [c for c in range(N) if c not in cols])
        assert np.array_equal(C[other], plain[other])


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("tiles", [("128x128x32_x", "64x128x32_x", "64x64x32_x", "128x128x32_2x2_g",
                                    "64x128x32_2x2_g", "64x64x16_2x2_g", "64x64x32_2x2_gw"),
                                   ("128x128x32_x8", "64x128x32_x8", "128x128x32_2x2_g8",
                                    "64x128x32_2x2_g8"),
                                   ("64x64x32_x16", "64x64x32_2x2_g16"),
                                   ("32x32x32_d", "32x32x32_2x2_gd")])
def test_elements_do_not_depend_on_the_tile(rt, tiles, ta, tb):
    """Operands with every kind of value that the parts do not carry, in some
    rows and columns, among others, and as the small values of otherwise
    ordinary rows (as activations have): tiles of the same number of groups
    give the same bits, whichever elements share a tile."""
    M, N, K = 128, 128, 544
    say(f"elements alone {tiles[0]} ta={ta} tb={tb}")
    rng = np.random.default_rng(17)
    A, B = synth.uniform((M, K), 18), synth.uniform((K, N), 19)
    A[rng.random((M, K)) < 0.02] = 1e-40           # irrelevant to most sums
    A[3], A[70] = np.ldexp(A[3], -120), np.ldexp(A[70], -140)
    A[5], A[6, ::2] = 0.0, 1e-39
    A[5, 9] = 1e-41
    B[:, 33] = np.ldexp(B[:, 33], -130)
    B[::3, 90] = 0.0
    B[9, 90] = 2.0 ** 100
    A[40, 17], A[41, 18], A[42, 19] = np.inf, np.nan, -np.inf
    B[17, 4], B[18, 5], B[100, 6] = 1e-42, 0.0, 3e38
    A[43, 100] = 3e38
    a, b = (A.T.copy() if ta else A), (B.T.copy() if tb else B)
    C = [product(rt, a, b, M, N, K, ta, tb, tile) for tile in tiles]
    for tile, c in zip(tiles, C):
        assert np.array_equal(c.view(np.uint32)[np.isfinite(c)],
                              C[0].view(np.uint32)[np.isfinite(c)]), tile
        assert np.array_equal(c, C[0], equal_nan=True), tile
    with np.errstate(invalid="ignore", over="ignore"):
        a64, b64 = A.astype(np.float64), B.astype(np.float64)
        ref, scale = a64 @ b64, np.abs(a64) @ np.abs(b64)
    ok = np.isfinite(scale) & (scale < 1e38)
    assert np.all(np.abs(C[0][ok] - ref[ok]) <= (K + 8) * U32 * scale[ok] + K * 2.0 ** -149)


@pytest.mark.parametrize("exponent", [-126, -118, -110, -100, -60, 60, 100, 118])
def test_range_of_the_parts(rt, exponent):
    """Operands scaled by 2^exponent against operands of order one: within
    (K + 8) u of |A| |B|, plus what the f32 result loses under its smallest
    value."""
    M, N, K = 128, 128, 288
    say(f"operand scale 2^{exponent}")
    A = np.ldexp(synth.uniform((M, K), 3), exponent).astype(np.float32)
    B = synth.uniform((K, N), 4)
    for a, b in ((A, B), (B.T.copy(), A.T.copy())):
        C = product(rt, a, b, M, N, K)
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        tol = (K + 8) * U32 * (np.abs(a64) @ np.abs(b64)) + K * 2.0 ** -149
        err = np.abs(C - a64 @ b64)
        assert np.all(err <= tol), (exponent, float((err / tol).max()))


@pytest.mark.parametrize("ta,tb,M,N,K", [(0, 0, 2, 3, 2**23 + 5), (0, 1, 3, 2, 2**23 + 5),
                                         (1, 0, 2**23 + 5, 2, 3)])
def test_pitch_beyond_32_bit_offsets(rt, ta, tb, M, N, K):
    """Row pitches above 2^23 floats take the tile with 64-bit addresses: the
    rows on either side of it, and the whole of a short output, within the
    bound of test_group_and_guard_edges."""
    name = rt.gemm_kernel_name(M, N, K, trans_a=bool(ta), trans_b=bool(tb), fused=True)
    say(f"pitch ta={ta} tb={tb} {M}x{N}x{K}: {name}")
    assert name.endswith("_2x2_gw_e")
    A = synth.uniform((K, M) if ta else (M, K), 5)
    B = synth.uniform((N, K) if tb else (K, N), 6)
    C = product(rt, A, B, M, N, K, ta, tb)
    a, b = (A.T if ta else A), (B.T if tb else B).astype(np.float64)
    for r in sorted({0, 1, M // 2, M - 1}):
        row = a[r].astype(np.float64)
        assert np.all(np.abs(C[r] - row @ b) <= (K + 8) * U32 * (np.abs(row) @ np.abs(b))), r


@pytest.mark.parametrize("factors,tile", [("1,50", "128x128x32_x_e"), ("1,1,50,50", "64x128x32_x_e"),
                                          ("1,1,1,1,1,50", "64x128x32_x8_e"),
                                          ("1,1,1,1,1,1,1,50", "64x64x32_x16_e"),
                                          ("1,1,1,1,1,1,1,1,50", "32x32x32_d_e")])
def test_order_of_the_tile_factors(factors, tile):
    """OXFORGE_GEMM_EFF (read once by a process) keeps its documented order:
    128x256, 128x128, 128x64, 64x128, 64x64 and the 64x128 tile of two groups,
    then the later ones."""
    say(f"tile factors {factors}")
    code = ("import oxforge\nwith oxforge.Runtime(0) as rt:\n"
            "    print(rt.gemm_kernel_name(1024, 1024, 1024, fused=True))")
    env = dict(os.environ, OXFORGE_GEMM_EFF=factors,
               PYTHONPATH=os.path.dirname(os.path.dirname(oxforge.__file__)))
    out = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True,
                         timeout=60)
    assert out.returncode == 0, out.stderr
    assert out.stdout.strip().endswith(tile)


def test_named_guarded_tile_takes_any_pitch(rt):
    """The guarded 64 x 64 tile by name at a pitch above 2^23 floats, as the
    plain and the fused product: what the dispatcher gives there."""
    M, N, K = 2, 3, 2**23 + 5
    say(f"named tile at pitch {K}")
    A, B = rt.array(synth.uniform((M, K), 23)), rt.array(synth.uniform((K, N), 24))
    ref, C, E = (rt.empty((M, N)) for _ in range(3))
    rt.gemm(A, B, ref, M, N, K)
    rt.gemm_tile("64x64x16_2x2_g", A, B, C, M, N, K)
    rt.gemm_ex_tile("64x64x16_2x2_g", A, B, E, M, N, K)
    assert np.array_equal(C.numpy(), ref.numpy()) and np.array_equal(E.numpy(), ref.numpy())
    with pytest.raises(oxforge.ForgeError):
        rt.gemm_tile("128x128x32_2x2_g", A, B, C, M, N, K)


@pytest.mark.parametrize("tb,tile", [(0, "128x128x32_2x2_g"), (0, "128x128x32_2x2_g8"),
                                     (1, "128x128x32_2x2_g"), (1, "64x128x32_2x2_g8"), (0, None)])
def test_pitch_up_to_32_bit_offsets(rt, tb, tile):
    """k contiguous at a pitch just under 2^23 floats, whose 128 rows reach
    byte offsets beyond 2^31 from a slab's first value: zeros but for some k
    near the ends and the middle, in rows on either side of that."""
    K = 2**23 - 3
    M, N = (3, 128) if tb else (128, 3)
    say(f"pitch {K} tb={tb} {tile}")
    R, S = (N, M) if tb else (M, N)  # rows of that pitch, and of the other operand
    ks = np.r_[0:9, K // 2:K // 2 + 9, K - 9:K]
    big, small = synth.uniform((R, len(ks)), 21), synth.uniform((len(ks), S), 22)
    dbig, dsmall = rt.empty((R, K)), rt.empty((M, K) if tb else (K, N))
    for d in (dbig, dsmall):
        rt.fill(d, 0.0)
    for i in range(0, len(ks), 9):
        for r in range(R):
            dbig.view(r * K + int(ks[i]), (9,)).upload(np.ascontiguousarray(big[r, i:i + 9]))
        if tb:
            for m in range(M):
                dsmall.view(m * K + int(ks[i]), (9,)).upload(
                    np.ascontiguousarray(small[i:i + 9, m]))
        else:
            dsmall.view(int(ks[i]) * N, (9, N)).upload(np.ascontiguousarray(small[i:i + 9]))
    A, B = (dsmall, dbig) if tb else (dbig, dsmall)
    dC = rt.empty((M, N))
    if tile:
        rt.gemm_ex_tile(tile, A, B, dC, M, N, K, trans_b=tb)
    else:
        rt.gemm_ex(A, B, dC, M, N, K, trans_b=tb)
    C = dC.numpy().T if tb else dC.numpy()
    a, b = big.astype(np.float64), small.astype(np.float64)
    assert np.all(np.abs(C - a @ b) <= (len(ks) + 8) * U32 * (np.abs(a) @ np.abs(b)))
    for d in (dbig, dsmall, dC):
        d.recycle()


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(64, 64, 2048), (1, 70, 2049), (33, 130, 2177), (16, 192, 4095),
                                   (65, 64, 3072)])
def test_sliced_products(rt, ta, tb, M, N, K):
    """Few tiles and a long K: the K slices (whole slabs, a ragged or shorter
    last one) of aligned and guarded products, with the reduction's epilogue,
    within the bound of test_group_and_guard_edges plus one rounding for the
    bias."""
    name = rt.gemm_kernel_name(M, N, K, trans_a=bool(ta), trans_b=bool(tb), fused=True)
    say(f"slices ta={ta} tb={tb} {M}x{N}x{K}: {name}")
    assert "/split" in name
    A = synth.uniform((K, M) if ta else (M, K), 7)
    B = synth.uniform((N, K) if tb else (K, N), 8)
    bias = synth.uniform((N,), 9)
    a, b = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
    dC = rt.empty((M, N))
    rt.gemm_ex(rt.array(A), rt.array(B), dC, M, N, K, trans_a=ta, trans_b=tb, bias=rt.array(bias))
    ref = a @ b + bias
    tol = (K + 8) * U32 * (np.abs(a) @ np.abs(b)) + 2 * U32 * np.abs(ref)
    assert np.all(np.abs(dC.numpy() - ref) <= tol)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(32, 64, 1024), (32, 64, 1056), (64, 32, 1344), (31, 33, 1055),
                                   (40, 70, 1300), (1, 5, 2047), (64, 128, 2048), (33, 65, 2049),
                                   (512, 512, 4096)])
def test_direct_tile_long_k(rt, M, N, K, ta, tb):
    """Products the dispatcher gives the 32x32 tile, K from the slabs a wave
    holds at once onwards, and in slices from 2048: within the bound of
    test_group_and_guard_edges."""
    name = rt.gemm_kernel_name(M, N, K, trans_a=bool(ta), trans_b=bool(tb), fused=True)
    say(f"ta={ta} tb={tb} {M}x{N}x{K}: {name}")
    assert K >= 2048 or "32x32x32" in name
    A = synth.uniform((K, M) if ta else (M, K), M + K)
    B = synth.uniform((N, K) if tb else (K, N), N + K)
    a, b = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
    C = product(rt, A, B, M, N, K, ta, tb)
    assert np.all(np.abs(C - a @ b) <= (K + 8) * U32 * (np.abs(a) @ np.abs(b)))
