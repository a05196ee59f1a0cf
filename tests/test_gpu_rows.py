"""MatMulNBits of up to 64 rows in any float types (k_gemv_rows) on the GPU, at the sizes where its
launch shapes, remainders and operand paths change, and the calls beside it that other kernels take,
against float64 sums over the oracle's weights.

Bound per output, S = sum |a w| of its products: 2^-20 S for the f32 sums (K up to a few thousand in
chunks of 32, each partial sum rounding by 2^-24 of its value) and the weights' own f32 rounding,
plus half a unit in the last place of the dot's and of Y's type (2^-11 f16, 2^-8 bf16)."""

import ctypes
import zlib

import numpy as np
import pytest

from oracle import oracle as o
from synth import nbits_weight
from test_gpu_nbits import as_f64, host_float
from transmuter_amd import PackedWeight
from transmuter_amd._lib import BF16, F16, F32, lib
from transmuter_amd.device import bf16_host
from transmuter_amd.quantized import matmul_nbits

pytestmark = pytest.mark.gpu

HALF_ULP = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def typed(x, dtype):
    h = host_float(x, dtype)
    return bf16_host(h) if dtype == "bf16" else h


def check(ctx, a, a_dtype, w_dtype, k, n, bits, block, zp, bias_dtype=None, seed=0, edit_scales=None):
    rng = np.random.default_rng(seed)
    b, s32, z = nbits_weight(rng, k, n, bits, block, zp=zp, scale_dtype=np.float32)
    scales = typed(s32 if edit_scales is None else edit_scales(s32), w_dtype)
    w = PackedWeight.upload(ctx, b, scales, z, k=k, n=n, bits=bits, block_size=block, weight_dtype=w_dtype)
    bias = None if bias_dtype is None else typed(rng.standard_normal(n), bias_dtype)
    y_t = matmul_nbits(ctx.put(a), w, bias)
    y = as_f64(y_t.numpy(), y_t.dtype)
    dense = o.dequantize_weight(b, as_f64(scales, w_dtype).astype(np.float32), z, k, n, bits, block, w_dtype)
    dense = np.asarray(dense, np.float64)
    af = as_f64(a, a_dtype)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = af @ dense.T
        for row in np.flatnonzero(~np.isfinite(af).all(1)) if np.isfinite(dense).all() else range(len(af)):
            ref[row] = (af[row] * dense).sum(1)  # product by product: a matrix product may skip zeros
    dot_dtype = a_dtype if a_dtype == w_dtype else "f32"
    bound = 2.0 ** -20 * (np.abs(af) @ np.abs(dense).T) + HALF_ULP[dot_dtype] * np.abs(ref)
    if bias is not None:
        ref = ref + as_f64(bias, bias_dtype)
    bound = bound + HALF_ULP[y_t.dtype] * np.abs(ref) + (2.0 ** -24 if "f16" in (dot_dtype, y_t.dtype) else 0)
    w.free()
    return y, ref, bound


def chunk(bits):
    return 512 // bits


# Launch shapes: tiles x 16-row sets against 256, 512, 1024 and 2048 workgroups; up to 8 chunks and more.
SHAPES = [(1, 16, 1), (16, 17, 8), (17, 40, 9), (33, 300, 17), (64, 1024, 33), (1, 4097, 3), (16, 4160, 11), (8, 33000, 2),
          (31, 2064, 9), (48, 2704, 2), (32, 5000, 3), (20, 9000, 2), (30, 16500, 2), (64, 16400, 2), (20, 66000, 1)]
TYPES = [("f16", "f16"), ("bf16", "bf16"), ("f32", "f32")]


@pytest.mark.parametrize("a_dtype,w_dtype", TYPES)
@pytest.mark.parametrize("m,n,chunks", SHAPES)
def test_launch_shapes(ctx, m, n, chunks, a_dtype, w_dtype):
    k = chunks * chunk(4) - 24  # a partial last chunk and block
    print(f"rows m={m} n={n} k={k} {a_dtype}", flush=True)
    rng = np.random.default_rng(m * 1000 + n)
    a = typed(rng.standard_normal((m, k)), a_dtype)
    # (An f32 bias keeps up to 16 rows of f16 from the f16 decode GEMV.)
    bias = "f32" if a_dtype == "f16" and m <= 16 else None
    y, ref, bound = check(ctx, a, a_dtype, w_dtype, k, n, 4, 32, "packed", bias, seed=n)
    assert (np.abs(y - ref) <= bound).all()


# The shapes of several tiles or sets of rows with 2- and 8-bit weights and parameters that change within a
# lane's group.
@pytest.mark.parametrize("a_dtype,w_dtype", TYPES)
@pytest.mark.parametrize("bits,block", [(2, 16), (2, 64), (4, 16), (8, 32)])
@pytest.mark.parametrize("m,n,chunks", [(16, 4160, 9), (16, 33000, 2), (20, 5000, 3), (48, 2704, 2), (30, 16500, 2), (64, 16200, 3),
                                        (24, 5000, 5), (24, 5000, 9), (40, 5000, 9)])
def test_launch_shapes_of_other_weights(ctx, m, n, chunks, bits, block, a_dtype, w_dtype):
    k = chunks * chunk(bits) - 24
    print(f"rows m={m} n={n} k={k} b{bits} bs{block} {a_dtype}", flush=True)
    rng = np.random.default_rng(m * 1000 + n)
    a = typed(rng.standard_normal((m, k)), a_dtype)
    bias = "f32" if a_dtype == "f16" and m <= 16 else None
    y, ref, bound = check(ctx, a, a_dtype, w_dtype, k, n, bits, block, "packed", bias, seed=n)
    assert (np.abs(y - ref) <= bound).all()


# 17 to 64 rows against so many columns that the prefill GEMM takes them, unsplit (from 33 rows on; against
# 65536 columns 17 of 2 bits and 25 of 4; 8 bits from 65536 columns on), and the row counts beside.
@pytest.mark.parametrize("a_dtype", ["f16", "bf16"])
@pytest.mark.parametrize("bits,block,zp", [(2, 64, "packed"), (8, 32, "none"), (8, 128, "packed"), (4, 32, "packed")])
@pytest.mark.parametrize("m,n", [(32, 16400), (33, 16400), (64, 16384), (16, 65550), (17, 65550), (25, 65550), (33, 65550)])
def test_few_rows_of_the_prefill_gemm(ctx, m, n, bits, block, zp, a_dtype):
    k = 2 * chunk(bits) + 40
    print(f"few prefill rows m={m} n={n} k={k} b{bits} bs{block} {zp} {a_dtype}", flush=True)
    rng = np.random.default_rng(m + n)
    a = typed(rng.standard_normal((m, k)), a_dtype)
    y, ref, bound = check(ctx, a, a_dtype, a_dtype, k, n, bits, block, zp, None, seed=n)
    assert (np.abs(y - ref) <= bound).all()


CODE = {"f32": F32, "f16": F16, "bf16": BF16}
NP = {"f32": np.float32, "f16": np.float16, "bf16": np.uint16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def check_rows(ctx, m, k, n, a_dtype, w_dtype, bits, block, zp, lda, ldy, a_off, y_off):
    """One call over rows lda and ldy apart that start a_off and y_off values into their buffers; the rest
    of Y's buffer stays as it was."""
    rng = np.random.default_rng(m * 7919 + k)
    b, s32, z = nbits_weight(rng, k, n, bits, block, zp=zp, scale_dtype=np.float32)
    scales = typed(s32, w_dtype)
    w = PackedWeight.upload(ctx, b, scales, z, k=k, n=n, bits=bits, block_size=block, weight_dtype=w_dtype)
    y_dtype = a_dtype if a_dtype == w_dtype else "f32"
    a = typed(rng.standard_normal(a_off + m * lda), a_dtype)
    a_d, y_d = ctx.put(a), ctx.put(np.full(y_off + m * ldy + 8, 7, NP[y_dtype]))
    a_at = ctypes.c_void_p(a_d.ptr.value + a_off * SIZE[a_dtype])
    y_at = ctypes.c_void_p(y_d.ptr.value + y_off * SIZE[y_dtype])
    ctx.check(lib().tmh_matmul_nbits(ctx.handle, w.handle, a_at, CODE[a_dtype], m, lda, None, 0, y_at, CODE[y_dtype], ldy, None))
    whole = y_d.numpy()
    w.free()
    rows = whole[y_off:y_off + m * ldy].reshape(m, ldy)
    assert (whole[:y_off] == 7).all() and (rows[:, n:] == 7).all() and (whole[y_off + m * ldy:] == 7).all()
    y = as_f64(rows[:, :n], y_dtype)
    af = as_f64(a[a_off:].reshape(m, lda)[:, :k], a_dtype)
    dense = np.asarray(o.dequantize_weight(b, as_f64(scales, w_dtype).astype(np.float32), z, k, n, bits, block, w_dtype), np.float64)
    ref = af @ dense.T
    # Over 64 rows an f32 factor goes through the prefill GEMM as two bf16 parts, 16 bits and a half of it:
    # 2^-17 for each factor and 2^-16 for the product of the low parts, left out.
    part = 2.0 ** -15 if m > 64 and "f32" in (a_dtype, w_dtype) else 2.0 ** -20
    bound = part * (np.abs(af) @ np.abs(dense).T) + 2 * HALF_ULP[y_dtype] * np.abs(ref) + (2.0 ** -24 if y_dtype == "f16" else 0)
    assert (np.abs(y - ref) <= bound).all()


PATHS = TYPES + [("f32", "f16"), ("f16", "f32"), ("bf16", "f32"), ("f16", "bf16")]


@pytest.mark.parametrize("a_dtype,w_dtype", PATHS)
@pytest.mark.parametrize("m,bits,block,zp", [(20, 4, 32, "packed"), (64, 4, 16, "none"), (20, 8, 64, "float"), (3, 2, 64, "packed")])
@pytest.mark.parametrize("y_off", [0, 1, 2])
def test_strides_and_y_off_its_alignment(ctx, m, bits, block, zp, a_dtype, w_dtype, y_off):
    print(f"strides m={m} b{bits} bs{block} {zp} {a_dtype} {w_dtype} y_off={y_off}", flush=True)
    check_rows(ctx, m, 264, 150, a_dtype, w_dtype, bits, block, zp, 280, 150 + (5 if y_off else 6), 0, y_off)


# K no multiple of 8, or rows of A off 16-byte boundaries: the kernels that load value by value.
@pytest.mark.parametrize("a_dtype,w_dtype", PATHS)
@pytest.mark.parametrize("m", [1, 5, 17, 40, 70])
@pytest.mark.parametrize("k,lda,a_off,bits,block,zp", [(77, 77, 0, 4, 16, "packed"), (100, 104, 0, 4, 32, "float"),
                                                       (264, 264, 1, 8, 32, "none"), (300, 301, 2, 2, 64, "packed")])
def test_rows_off_the_vector_loads(ctx, m, k, lda, a_off, bits, block, zp, a_dtype, w_dtype):
    print(f"off the loads m={m} k={k} lda={lda} +{a_off} b{bits} bs{block} {zp} {a_dtype} {w_dtype}", flush=True)
    check_rows(ctx, m, k, 75, a_dtype, w_dtype, bits, block, zp, lda, 75, a_off, 0)


@pytest.mark.parametrize("bits,block", [(2, 16), (2, 64), (4, 16), (4, 64), (4, 256), (8, 16), (8, 32), (8, 128)])
@pytest.mark.parametrize("zp", ["none", "packed", "float"])
@pytest.mark.parametrize("a_dtype,w_dtype", TYPES + [("f32", "f16"), ("f16", "f32"), ("bf16", "f32"), ("f16", "bf16")])
def test_operand_paths(ctx, bits, block, zp, a_dtype, w_dtype):
    case = (bits, block, zp, a_dtype, w_dtype)
    rng = np.random.default_rng(zlib.crc32(repr(case).encode()))
    m, n = int(rng.choice([3, 16, 21, 70])), int(rng.choice([19, 150]))
    k = chunk(bits) * int(rng.integers(1, 12)) + 8 * int(rng.integers(0, 4))
    bias = [None, "f32", w_dtype][int(rng.integers(3))]
    print(f"operand path {case} m={m} n={n} k={k} bias={bias}", flush=True)
    a = typed(rng.standard_normal((m, k)), a_dtype)
    y, ref, bound = check(ctx, a, a_dtype, w_dtype, k, n, bits, block, zp, bias, seed=m)
    if m > 64 and a_dtype != w_dtype or (m > 64 and zp == "float") or (m > 64 and a_dtype == "f32"):
        bound = bound + 2.0 ** -14 * np.abs(ref).max()  # the prefill GEMM keeps 16 bits of each f32 factor
    assert (np.abs(y - ref) <= bound).all()


@pytest.mark.parametrize("a_dtype,w_dtype", [("f32", "f32"), ("f32", "f16"), ("bf16", "bf16"), ("f16", "f16")])
def test_wide_range_infinities_and_nan(ctx, a_dtype, w_dtype):
    """Values over the type's whole range, and rows with an infinity or a NaN: those rows' outputs are
    the float64 sum's (infinite or NaN), and no other row sees them."""
    rng = np.random.default_rng(5)
    m, k, n = 20, 520, 64
    top = 4 if a_dtype == "f16" else 30
    a = rng.standard_normal((m, k)) * 10.0 ** rng.uniform(-top, top, (m, 1))
    a[3, 17], a[4, 40], a[5, 300] = np.inf, -np.inf, np.nan
    a = typed(a, a_dtype)
    y, ref, bound = check(ctx, a, a_dtype, w_dtype, k, n, 4, 32, "none", seed=9)
    special = [3, 4, 5]
    assert not np.isfinite(y[special]).any()
    rest = [i for i in range(m) if i not in special]
    limit = {"f16": 65504.0}.get(a_dtype if a_dtype == w_dtype else "f32", 3.4e38)
    fits = np.abs(ref[rest]) < limit
    assert (np.abs(y[rest] - ref[rest])[fits] <= bound[rest][fits]).all()


# Paths whose factors are cut in parts, and beside them the f16 one.
SPECIAL = [("f32", "f16", 4, 32, "packed"), ("f16", "f32", 4, 32, "none"), ("bf16", "f32", 8, 64, "packed"),
           ("f32", "bf16", 8, 16, "none"), ("f32", "f32", 2, 64, "packed"), ("f32", "f32", 4, 16, "none"),
           ("f16", "f16", 4, 32, "float"), ("bf16", "bf16", 8, 32, "float"), ("f32", "f32", 8, 32, "float"),
           ("f16", "f16", 4, 32, "packed"), ("f32", "f32", 4, 32, "none"), ("f32", "f32", 8, 64, "packed"),
           ("bf16", "bf16", 4, 32, "packed"), ("bf16", "bf16", 2, 64, "none")]


@pytest.mark.parametrize("a_dtype,w_dtype,bits,block,zp", SPECIAL)
@pytest.mark.parametrize("infinite_weights", [False, True])
def test_infinities_as_in_float64(ctx, a_dtype, w_dtype, bits, block, zp, infinite_weights):
    """An infinity or NaN in A, or an infinite weight (an f16 scale times q - zero past 65504; in the wider
    types an infinite scale), gives +inf, -inf or NaN exactly where the float64 sum does, and every
    finite output stays within the bound."""
    print(f"infinities {a_dtype} {w_dtype} b{bits} bs{block} {zp} weights={infinite_weights}", flush=True)
    rng = np.random.default_rng(6)
    m, k, n = 20, 520, 64
    a = np.abs(rng.standard_normal((m, k))) + 0.1
    a[3, 17], a[4, 40], a[5, 300], a[6, 2], a[6, 500] = np.inf, -np.inf, np.nan, np.inf, -np.inf
    a = typed(a, a_dtype)

    def some_infinite(s32):
        s = s32.reshape(n, -1).copy()
        s[5, 1] = s[50, 0] = 60000.0 if w_dtype == "f16" else np.inf
        return s.reshape(s32.shape)

    # (f16 and bf16 operands of one type multiply on their own matrix instructions, whose weights
    # overflow as the type does.)
    y, ref, bound = check(ctx, a, a_dtype, w_dtype, k, n, bits, block, zp, seed=9,
                          edit_scales=some_infinite if infinite_weights else None)
    for kind in (np.isposinf, np.isneginf, np.isnan):
        assert np.array_equal(kind(y), kind(ref)), kind.__name__
    fin = np.isfinite(ref)
    assert fin.sum() > n and (np.abs(y - ref)[fin] <= bound[fin]).all()


@pytest.mark.parametrize("a_dtype,w_dtype,bits,block,zp", [("f32", "f32", 4, 16, "packed"), ("f32", "f32", 2, 64, "none"),
                                                           ("f32", "f32", 4, 32, "float")])
def test_parts_leave_no_bias(ctx, a_dtype, w_dtype, bits, block, zp):
    """Both factors cut in bf16 parts, every product of one sign and significands near 2, where the
    products of the smaller parts are largest: the mean relative error of the outputs is that of the
    rounding of a few f32 sums (each within 2^-24, of either sign), without what a dropped product of
    parts would take from all of them."""
    print(f"parts {a_dtype} {w_dtype} b{bits} bs{block} {zp}", flush=True)
    rng = np.random.default_rng(8)
    m, k, n = 16, 16 if bits == 4 else 64, 512
    near2 = lambda shape: (2.0 - rng.integers(1, 200, shape) * 2.0 ** -23).astype(np.float32)
    b, s32, z = nbits_weight(rng, k, n, bits, block, zp=zp, scale_dtype=np.float32)
    b = np.full_like(b, 0xFF)  # the largest value everywhere
    if zp == "packed":
        z = np.zeros_like(z)
    elif zp == "float":
        z = np.zeros_like(z)
    scales, a = near2(s32.shape), near2((m, k))
    w = PackedWeight.upload(ctx, b, scales, z, k=k, n=n, bits=bits, block_size=block, weight_dtype=w_dtype)
    y = matmul_nbits(ctx.put(a), w).numpy().astype(np.float64)
    w.free()
    dense = np.asarray(o.dequantize_weight(b, scales, z, k, n, bits, block, w_dtype), np.float64)
    ref = a.astype(np.float64) @ dense.T
    rel = (y - ref) / ref
    print(f"mean {rel.mean() * 2.0 ** 24:.4f} max {np.abs(rel).max() * 2.0 ** 24:.3f} units of 2^-24", flush=True)
    assert abs(rel.mean()) <= 2.0 ** -26  # (8192 roundings of either sign average to 2^-30 and less)


@pytest.mark.parametrize("bits,block,zp", [(4, 32, "none"), (4, 128, "packed"), (8, 32, "packed"), (8, 64, "none")])
def test_f32_a_near_the_end_of_its_range(ctx, bits, block, zp):
    """A up to 3e38 against small scales: every output is finite, also where the products of a block
    pass f32's range before its scale."""
    print(f"range b{bits} bs{block} {zp}", flush=True)
    rng = np.random.default_rng(12)
    m, k, n = 20, 520, 80
    a = rng.standard_normal((m, k)) * 10.0 ** rng.uniform(33, 37.8, (m, 1))
    a[7] = 3e38  # one sign: every block's sum is past the range
    a = np.clip(a, -3e38, 3e38).astype(np.float32)
    y, ref, bound = check(ctx, a, "f32", "f32", k, n, bits, block, zp, seed=3, edit_scales=lambda s: s * np.float32(1e-4))
    assert np.isfinite(ref).all() and np.abs(ref).max() < 3e38
    assert (np.abs(y - ref) <= bound).all()


@pytest.mark.parametrize("bits,block,zp", [(4, 32, "packed"), (4, 16, "none"), (8, 64, "none"), (2, 64, "packed")])
@pytest.mark.parametrize("power", [-132, -120, 117])
def test_bf16_scales_at_the_ends_of_the_type(ctx, bits, block, zp, power):
    """bf16 scales of 2^117 to 2^120, and subnormal and nearly subnormal ones, against A at the other
    end of the type."""
    print(f"bf16 scales 2^{power} b{bits} bs{block} {zp}", flush=True)
    rng = np.random.default_rng(13)
    m, k, n = 20, 264, 80
    a = typed(rng.standard_normal((m, k)) * 2.0 ** (100 if power < 0 else -100), "bf16")
    edit = lambda s: (rng.uniform(1, 8, s.shape) * 2.0 ** power).astype(np.float32)
    y, ref, bound = check(ctx, a, "bf16", "bf16", k, n, bits, block, zp, seed=4, edit_scales=edit)
    assert np.isfinite(ref).all()
    print(f"largest error over its bound {(np.abs(y - ref) / bound).max():.3f}", flush=True)
    assert (np.abs(y - ref) <= bound).all()


@pytest.mark.parametrize("bits,block,zp", [(4, 32, "none"), (4, 128, "packed"), (8, 32, "packed"), (8, 64, "none")])
@pytest.mark.parametrize("m,k,n", [(70, 520, 80), (100, 2048, 300)])
def test_prefill_f32_over_a_s_whole_range(ctx, bits, block, zp, m, k, n):
    """The f32 prefill product (over 64 rows, whole-number weights): A up to 3e38 against small scales
    gives finite outputs, A down to 1e-30 the same relative error, and an infinity or a NaN in a row of A
    what the float64 sum gives. A's hi and lo parts hold 16 bits of each value: 2^-16 of every product."""
    print(f"prefill range b{bits} bs{block} {zp} m={m}", flush=True)
    rng = np.random.default_rng(14)
    a = rng.standard_normal((m, k)) * 10.0 ** rng.uniform(-30, 37.8, (m, 1))
    a[7] = 3e38  # one sign: every block's sum is past the range before its scale
    a = np.clip(a, -3e38, 3e38).astype(np.float32)
    a[66] = np.abs(a[66]) + 1.0
    a[66, 3] = np.inf
    a[67, 5] = np.nan
    y, ref, bound = check(ctx, a, "f32", "f32", k, n, bits, block, zp, seed=3, edit_scales=lambda s: s * np.float32(1e-4))
    for kind in (np.isposinf, np.isneginf, np.isnan):
        assert np.array_equal(kind(y), kind(ref)), kind.__name__
    fin = np.isfinite(ref).all(1)
    assert fin.sum() == m - 2 and np.abs(ref[fin]).max() < 3e38
    # bound holds 2^-20 sum |a w|: 16 times that is 2^-16 of every product
    assert (np.abs(y - ref)[fin] <= 16 * bound[fin]).all()


# Over 64 rows without a build of the prefill GEMM: slices of 64 rows in one launch, the rest in a second.
@pytest.mark.parametrize("a_dtype,w_dtype,bits,block,zp", [("bf16", "bf16", 4, 16, "packed"), ("f32", "f32", 4, 16, "none"),
                                                           ("f32", "f16", 2, 32, "packed"), ("f16", "f16", 2, 16, "float")])
@pytest.mark.parametrize("m,n", [(65, 48), (128, 20), (129, 300), (1000, 64)])
def test_slices_of_64_rows(ctx, m, n, a_dtype, w_dtype, bits, block, zp):
    print(f"slices m={m} n={n} {a_dtype} {w_dtype} b{bits} bs{block} {zp}", flush=True)
    rng = np.random.default_rng(m + n)
    k = chunk(bits) + 40
    a = typed(rng.standard_normal((m, k)), a_dtype)
    y, ref, bound = check(ctx, a, a_dtype, w_dtype, k, n, bits, block, zp, "f32" if m == 129 else None, seed=n)
    assert (np.abs(y - ref) <= bound).all()
