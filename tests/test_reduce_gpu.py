"""Parity of the gfx950 reductions with the CPU oracle (a restatement of
avx2::reduce, source/CortexMind/framework/Engine/AVX2/reduce.cpp).

Bars (from the task's parity contract): max and argmax bit-exact; sum and
mean within |gpu - ref| <= 1e-5 * sum|x| per output, because the GPU adds
in a tree and the reference in 8 sequential lanes (both round, differently).
"""
import ctypes

import numpy as np
import pytest

from cortexmind_amd import engine
from cortexmind_amd._lib import E_INVALID, call, lib
from cortexmind_amd.data import SplitMix64, c2_reduce
from cortexmind_amd.device import DeviceArray

from gpu_util import bits_equal, dev, empty

pytestmark = pytest.mark.gpu

SUM_TOL = 1e-5


def gpu_reduce(op, x, sizes, ptr_offset_floats=0):
    """Run one reduction on the device; sizes = (n,) or (outer, dim, inner)."""
    flat = np.ascontiguousarray(x, np.float32).ravel()
    buf = np.concatenate([np.zeros(ptr_offset_floats, np.float32), flat])
    dx = DeviceArray.from_numpy(buf)
    n_out = 1 if len(sizes) == 1 else sizes[0] * sizes[2]
    dz = DeviceArray((n_out,), np.int32 if op in ("argmax", "argmin") else np.float32)
    xp = dx.ptr + 4 * ptr_offset_floats
    if len(sizes) == 1:
        call(f"cxm_reduce_{op}_flat_f32", xp, dz.ptr, sizes[0], None)
    else:
        call(f"cxm_reduce_{op}_f32", xp, dz.ptr, *sizes, None)
    return dz.numpy()


def abs_sums(x, sizes):
    a = np.abs(np.asarray(x, np.float64)).ravel()
    if len(sizes) == 1:
        return np.array([a.sum()])
    o, d, i = sizes
    return a.reshape(o, d, i).sum(axis=1).ravel()


def check(op, x, sizes, orc, **kw):
    got = gpu_reduce(op, x, sizes, **kw)
    ref = orc.reduce_flat(op, x) if len(sizes) == 1 else orc.reduce_axis(op, x, *sizes)
    if op in ("max", "argmax", "min", "argmin"):
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (op, sizes)
    else:
        tol = SUM_TOL * abs_sums(x, sizes)
        if op == "mean":
            tol = tol / sizes[1 if len(sizes) == 3 else 0]
        err = np.abs(got.astype(np.float64) - ref.astype(np.float64))
        assert np.all(err <= tol + 1e-30), (op, sizes, float(np.max(err - tol)))
    return got, ref


# ------------------------------------------------------------- C2 full size

@pytest.fixture(scope="module")
def c2():
    return c2_reduce()


@pytest.mark.parametrize("op", ["sum", "mean", "max", "argmax"])
def test_c2_global(hip, orc, c2, op):
    if op in ("max", "argmax"):
        check(op, c2, (c2.size,), orc)
    else:
        got, _ = check(op, c2, (c2.size,), orc)
        exact = np.sum(c2.astype(np.float64))
        if op == "mean":
            exact /= c2.size
        # the GPU's own error against float64 is well inside the bar too
        assert abs(got[0] - exact) <= SUM_TOL * np.abs(c2.astype(np.float64)).sum() / (
            c2.size if op == "mean" else 1)


@pytest.mark.parametrize("op", ["sum", "mean", "max", "argmax"])
@pytest.mark.parametrize("axis", [0, 1])
def test_c2_axis(hip, orc, c2, op, axis):
    sizes = (1, 4096, 4096) if axis == 0 else (4096, 4096, 1)
    check(op, c2, sizes, orc)


@pytest.mark.parametrize("n", [4096 * 4096, 4096 * 4096 + 3, 1 << 22])
def test_global_sum_exact_integers(hip, n):
    """Full-size global sum and mean of integers in {-1, 0, 1}: every partial
    sum is an integer below 2^24 in magnitude, so each is exact in fp32 and
    the result must equal the exact sum bit for bit.  A lost or doubled
    segment partial (std ~52 for 8192 such terms) cannot hide under this bar,
    where it could under the 1e-5 * sum|x| tolerance of U(-1, 1) data.
    Flat and (1, n, 1) forms; the odd length also runs the scalar tail."""
    r = SplitMix64(0xE1 + n).next_u64(n)
    x = ((r % np.uint64(3)).astype(np.int64) - 1).astype(np.float32)
    exact = int(np.sum(x.astype(np.int64)))
    assert abs(exact) < (1 << 24)
    for sizes in [(n,), (1, n, 1)]:
        got = gpu_reduce("sum", x, sizes)
        assert got[0] == np.float32(exact), (sizes, float(got[0]), exact)
        mean = gpu_reduce("mean", x, sizes)
        # flat: sum / (float)N; axis with one output: the division tail
        want = np.float32(exact) / np.float32(n)
        assert mean[0] == want, (sizes, float(mean[0]), float(want))


@pytest.mark.parametrize("sizes", [(4096, 4096, 1), (1, 4096, 4096), (3, 1000, 257)])
def test_axis_sum_exact_integers(hip, sizes):
    """Row and column sums of integers in {-1, 0, 1}: exact, bit for bit."""
    o, d, i = sizes
    r = SplitMix64(0xE2 + d).next_u64(o * d * i)
    x = ((r % np.uint64(3)).astype(np.int64) - 1).astype(np.float32).reshape(o, d, i)
    exact = x.astype(np.int64).sum(axis=1).ravel().astype(np.float32)
    got = gpu_reduce("sum", x, sizes)
    assert np.array_equal(got, exact), sizes


def test_c2_deterministic(hip, c2):
    a = gpu_reduce("sum", c2, (c2.size,))
    b = gpu_reduce("sum", c2, (c2.size,))
    c = gpu_reduce("sum", c2, (1, 4096, 4096))
    d = gpu_reduce("sum", c2, (1, 4096, 4096))
    assert a.tobytes() == b.tobytes() and c.tobytes() == d.tobytes()


# -------------------------------------------------------------- edge shapes

@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 255, 1023, 1025, 4099, 65537, (1 << 20) + 3])
@pytest.mark.parametrize("op", ["sum", "mean", "max", "argmax"])
def test_flat_ragged(hip, orc, n, op):
    x = SplitMix64(n).normal((n,), 0.0, 3.0)
    check(op, x, (n,), orc)


@pytest.mark.parametrize("op", ["sum", "max", "argmax"])
def test_flat_unaligned_pointer(hip, orc, op):
    x = SplitMix64(77).uniform((10001,), -1, 1)
    check(op, x, (x.size,), orc, ptr_offset_floats=1)


@pytest.mark.parametrize("sizes", [(7, 9, 1), (3, 1025, 1), (64, 131072, 1), (5, 33, 1),
                                   (1, 7, 3), (2, 5, 9), (1, 257, 33), (3, 64, 17),
                                   (2, 100, 1000), (4, 4, 4096), (1, 3000, 260)])
@pytest.mark.parametrize("op", ["sum", "mean", "max", "argmax"])
def test_axis_shapes(hip, orc, sizes, op):
    o, d, i = sizes
    x = SplitMix64(o * 1000003 + d * 101 + i).normal((o, d, i), 0.0, 2.0)
    check(op, x, sizes, orc)


@pytest.mark.parametrize("sizes", [(64, 2048, 1), (32, 8192, 1), (16, 16384, 1), (2, 4096, 2048), (1, 4096, 512)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("op", ["sum", "mean", "max", "argmax"])
def test_whole_row_and_chunk_forms(hip, orc, sizes, op):
    """Shapes that take the straight-line kernels: whole aligned rows of one
    load batch (2048, 8192 and 16384 floats: 4, 16 and -- for argmax's
    256-thread rows -- 4 to 16 float4 a thread) and column chunks of exactly
    256 rows over whole tiles, with two outer slices."""
    o, d, i = sizes
    x = SplitMix64(0x3A11 + o + d + i).uniform((o, d, i), -2.0, 2.0)
    check(op, x, sizes, orc)


def test_argmax_ties_first_index(hip, orc):
    x = np.zeros((6, 40), np.float32)
    x[1, [3, 17, 39]] = 5.0          # repeated maximum -> first one
    x[2, :] = -1.0                   # all equal -> 0
    x[3, [0, 39]] = 2.0
    x[4, 10:] = 7.0
    x[5, :] = -np.inf                # all -inf -> 0
    for sizes in [(6, 40, 1), (1, 6, 40)]:
        check("argmax", x, sizes, orc)
    check("argmax", x.ravel(), (x.size,), orc)


def test_max_minus_inf_semantics(hip, orc):
    # flat and row forms start from -FLT_MAX (reduce.cpp:206); the column
    # form starts from the first slice, so an all -inf column stays -inf
    x = np.full((4, 16), -np.inf, np.float32)
    x[1, 5] = 3.0
    row = gpu_reduce("max", x, (4, 16, 1))
    assert row[0] == np.float32(-np.finfo(np.float32).max) and row[1] == 3.0
    col = gpu_reduce("max", x, (1, 4, 16))
    assert col[0] == -np.inf and col[5] == 3.0
    check("max", x, (4, 16, 1), orc)
    check("max", x, (1, 4, 16), orc)


def test_flat_zero_elements(hip):
    z = DeviceArray((1,), np.float32)
    for op, want in [("sum", 0.0), ("max", -np.finfo(np.float32).max)]:
        call(f"cxm_reduce_{op}_flat_f32", None, z.ptr, 0, None)
        assert z.numpy()[0] == np.float32(want)
    call("cxm_reduce_mean_flat_f32", None, z.ptr, 0, None)
    assert np.isnan(z.numpy()[0])
    assert lib().cxm_reduce_argmax_flat_f32(None, z.ptr, 0, None) == E_INVALID


def test_engine_mirror_names(hip, orc):
    # the reference's call shape: reduce::sum(Xx, Xz, outer, dim, inner)
    x = SplitMix64(5).uniform((3, 50, 8), -1, 1)
    dx = DeviceArray.from_numpy(x)
    dz = DeviceArray((24,), np.float32)
    engine.reduce.max(dx, dz, 3, 50, 8)
    assert np.array_equal(dz.numpy(), orc.reduce_axis("max", x, 3, 50, 8))
    engine.reduce.sum(dx, dz, x.size)
    assert abs(dz.numpy()[0] - np.sum(x.astype(np.float64))) <= SUM_TOL * np.abs(x).sum()


def _wait_limit(polls):
    old = ctypes.c_uint(0)
    call("cxm_exchange_wait_limit", polls, ctypes.byref(old))
    return old.value


@pytest.mark.parametrize("n", [4096 * 4096, (1 << 20) + 3, 1000003])
@pytest.mark.parametrize("op", ["sum", "mean", "max", "min", "norm1", "norm2"])
def test_flat_recompute_is_bit_identical(hip, orc, n, op):
    """Flat reductions with 32-bit partials combine them in one reader
    workgroup that waits for tagged slots; a partial it does not see within
    the wait limit is recomputed from the input with the writer's arithmetic.
    Forcing that for every segment (limit 0) gives the same bits."""
    x = SplitMix64(0xF1A7 + n).uniform((n,), -1.0, 1.0)
    normal = gpu_reduce(op, x, (n,))
    old = _wait_limit(0)
    try:
        forced = gpu_reduce(op, x, (n,))
    finally:
        _wait_limit(old)
    assert normal.tobytes() == forced.tobytes()
    ref = orc.reduce_flat(op, x)
    if op in ("max", "min"):
        assert normal.tobytes() == ref.tobytes()
    else:
        assert abs(float(normal[0]) - float(ref[0])) <= SUM_TOL * max(float(np.abs(x).sum()), 1e-30)


def test_flat_slot_state_across_shapes(hip, orc):
    """Flat reductions of different lengths (different segment counts over
    the same tagged slots), interleaved with row, column and segmented-row
    reductions on the same stream, each checked against the oracle: no call
    reads a partial an earlier call left behind."""
    g = SplitMix64(0x51075)
    seq = [(1 << 24,), (100003,), (3, 50000, 1), (1 << 24,), (5000,), (1, 4096, 4096), ((1 << 22) + 1,),
           (1 << 24,), (777,), (1 << 21,)]
    for sizes in seq:
        x = g.uniform(sizes if len(sizes) > 1 else sizes[0], -1.0, 1.0)
        check("sum", x, sizes, orc)
        check("max", x, sizes, orc)


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("sizes", [((1 << 22) + 3,), (3, 100003, 1), (64, 4097, 1), (2, 5, 1)])
@pytest.mark.parametrize("op", ["sum", "max", "argmax"])
def test_unaligned_ragged_rows(hip, orc, off, sizes, op):
    """Row bases off 16-byte alignment and lengths not a multiple of 4: each
    row's head (before its first aligned float4) and tail are folded in by
    its first segment, the body still takes 128-bit loads."""
    x = SplitMix64(off * 7919 + sum(sizes)).normal(sizes if len(sizes) > 1 else sizes[0], 0.0, 2.0)
    check(op, x, sizes, orc, ptr_offset_floats=off)



@pytest.mark.parametrize("sizes", [(1, 1, 2), (3, 1, 3), (2, 2, 2), (1, 2, 3), (1, 1, 4), (5, 3, 5), (160, 404, 3),
                                   (1, 100003, 10), (1, 5000, 64), (2, 700, 63), (3, 1000, 257), (300, 9, 257),
                                   (1, 4000, 255), (2, 65, 1021), (1, 3000, 1024), (1, 513, 1025), (2, 100, 1031),
                                   (1, 1000, 4099), (1, 37, 4100)])
@pytest.mark.parametrize("off", [0, 1])
def test_columns_of_any_width(hip, orc, sizes, off):
    """The flat column kernel at the edges of its plan (fewer floats than a
    float4, one to three columns, thread counts that are not whole waves,
    several chunks per slice with a ragged last one, both tickets) and the
    column tiles it hands over to, each with rows that are no multiple of 4
    and bases that are only 4-byte aligned."""
    o, d, i = sizes
    x = SplitMix64(0xC015 + 7 * o + 3 * d + i).uniform((o, d, i), -1.0, 1.0)
    if d > 2:
        x[0, :, 0] = x[0, 1, 0]  # ties: the first index wins
        x[o - 1, 0, i - 1] = np.nan
    dx = dev(x, off)
    for op in ("sum", "mean", "max", "min", "argmax", "argmin", "norm1", "norm2", "var"):
        z = empty((o, i), np.int32 if op.startswith("arg") else np.float32)
        getattr(engine.reduce, op)(dx, z, o, d, i)
        got = z.numpy()
        x64 = x.astype(np.float64)
        if op in ("max", "min"):
            assert bits_equal(got, getattr(np, op)(x, axis=1))  # np.max / np.min give NaN for the NaN column
        elif op.startswith("arg"):
            # a NaN in the first row stays the answer (index 0), as does the first of equal values
            assert np.array_equal(got, getattr(np, op)(x, axis=1))
        else:
            ref = {"sum": lambda: x64.sum(axis=1), "mean": lambda: x64.mean(axis=1),
                   "norm1": lambda: np.abs(x64).sum(axis=1), "norm2": lambda: np.sqrt((x64 * x64).sum(axis=1)),
                   "var": lambda: x64.var(axis=1)}[op]()
            size = np.abs(x64).sum(axis=1) / (d if op == "mean" else 1)
            if op in ("norm2", "var"):
                size = ref + 1e-7
            fin = np.isfinite(ref)
            if op != "var":  # (a NaN among the deviations gives a variance of 0)
                assert np.array_equal(fin, np.isfinite(got))
            assert np.all(np.abs(got - ref)[fin] <= 1e-5 * size[fin])


@pytest.mark.parametrize("dim", [1, 2, 3, 4, 5, 15, 16, 17, 31, 33, 63, 64, 65, 127, 129, 255, 257, 511, 513, 1003, 1025,
                                 2047, 2049, 4095, 4097, 10698])
@pytest.mark.parametrize("off", [0, 1])
def test_rows_of_any_length(hip, dim, off):
    """Short rows at the edges of their lanes-per-row and float4-per-lane
    ranges, with a last workgroup partly empty, NaN and ties included."""
    rows = 131
    x = SplitMix64(0x50A7 + dim).uniform((rows, dim), -1.0, 1.0)
    x[3, :] = -np.inf
    x[4, :] = x[4, 0]
    x[5, 0] = np.nan
    dx = dev(x, off)
    for op in ("sum", "mean", "max", "min", "argmax", "argmin", "norm1", "norm2", "var"):
        z = empty((rows,), np.int32 if op.startswith("arg") else np.float32)
        getattr(engine.reduce, op)(dx, z, rows, dim, 1)
        got = z.numpy()
        x64 = x.astype(np.float64)
        if op in ("max", "min"):
            ref = getattr(np, op)(x, axis=1)
            if op == "max":
                ref[3] = -np.finfo(np.float32).max  # the running maximum starts there
            assert bits_equal(got, ref)
        elif op.startswith("arg"):
            assert np.array_equal(got, getattr(np, op)(x, axis=1))
        else:
            with np.errstate(invalid="ignore"):
                ref = {"sum": lambda: x64.sum(axis=1), "mean": lambda: x64.mean(axis=1),
                       "norm1": lambda: np.abs(x64).sum(axis=1), "norm2": lambda: np.sqrt((x64 * x64).sum(axis=1)),
                       "var": lambda: x64.var(axis=1)}[op]()
                size = np.abs(x64).sum(axis=1) / (dim if op == "mean" else 1)
            if op in ("norm2", "var"):
                size = ref + 1e-7
            fin = np.isfinite(ref)
            assert np.all(np.abs(got - ref)[fin] <= 1e-5 * size[fin])
            if op != "var":
                assert np.array_equal(np.isnan(ref), np.isnan(got))


@pytest.mark.parametrize("dim", [33, 34, 65, 67, 129, 130])
def test_short_rows_error(hip, dim):
    """Rows a little longer than a power of two of floats: their last lane's
    few floats are added to one lane's sum, not to the whole row's, so the
    error against 64 bits stays below that of sums of four floats met
    pairwise from the first on, the rest last (fp32, the same inputs)."""
    rows = 40000
    x = SplitMix64(0x5047 + dim).normal((rows, dim), 0.5, 1.0)
    dx, z = DeviceArray.from_numpy(x), DeviceArray((rows,), np.float32)
    engine.reduce.sum(dx, z, rows, dim, 1)
    ref = x.astype(np.float64).sum(axis=1)
    quads = np.zeros((rows, -(-dim // 4) * 4), np.float32)
    quads[:, :dim] = x
    quads = quads.reshape(rows, -1, 4)
    t = (quads[..., 0] + quads[..., 1]) + (quads[..., 2] + quads[..., 3])
    while t.shape[1] > 1:
        n = t.shape[1] // 2 * 2
        t = np.concatenate([t[:, 0:n:2] + t[:, 1:n:2], t[:, n:]], axis=1)

    def error(a):
        return np.sqrt(np.mean((a - ref) ** 2))

    t = t[:, 0]
    assert error(z.numpy()) <= 0.96 * error(t), (error(z.numpy()), error(t))


@pytest.mark.parametrize("outer,dim,inner", [(8, 65, 4095), (37, 74, 1003), (8, 100, 2001), (2, 404, 20001), (2, 74, 20000), (300, 74, 131)])
def test_ragged_column_sums_error(hip, outer, dim, inner):
    """Column sums, above all of slices of no multiple of four floats: no
    further from 64 bits than four interleaved runs of rows added in fp32 (3%
    for the two orders' scatter)."""
    x = SplitMix64(0xC0E + dim).normal((outer, dim, inner), 0.5, 1.0)
    dx, z = DeviceArray.from_numpy(x), DeviceArray((outer, inner), np.float32)
    engine.reduce.sum(dx, z, outer, dim, inner)
    ref = x.astype(np.float64).sum(axis=1)
    runs = [np.zeros((outer, inner), np.float32) for _ in range(4)]
    for r in range(dim):
        runs[r % 4] = runs[r % 4] + x[:, r]
    four = ((runs[0] + runs[1]) + runs[2]) + runs[3]

    def error(a):
        assert a.shape == ref.shape
        return np.sqrt(np.mean((a - ref) ** 2))

    assert error(z.numpy()) <= 1.03 * error(four), (error(z.numpy()), error(four))


def test_more_rows_than_lanes_can_number(hip):
    """2^26 rows of 129 floats, a wave each, would be a grid of 2^32 threads:
    CXM_E_TOO_LARGE from the host, with operands of that size; a few rows
    fewer are reduced (the first and last of them, of zeros but for one
    element, checked)."""
    from cortexmind_amd._lib import E_TOO_LARGE

    rows, dim = 1 << 26, 129
    x, z = DeviceArray((rows * dim,), np.float32), DeviceArray((rows,), np.float32)
    assert lib().cxm_reduce_sum_f32(x.ptr, z.ptr, rows, dim, 1, None) == E_TOO_LARGE
    x.fill_bytes(0)
    one = np.ones(1, np.float32)
    n = rows - 16
    call("cxm_memcpy_h2d", x.ptr + 4 * ((n - 1) * dim + 7), one.ctypes.data, 4, None)
    call("cxm_reduce_sum_f32", x.ptr, z.ptr, n, dim, 1, None)
    got = z.numpy()[:n]
    assert got[-1] == 1.0 and not np.any(got[:-1])


@pytest.mark.parametrize("outer,dim,inner", [(1, 205, 40), (1, 204, 40), (32, 1000, 64), (33, 1000, 64), (2, 1001, 48),
                                             (3, 513, 16), (3, 512, 16), (5, 900, 17), (4, 1000, 9), (2, 993, 20), (1, 40, 33), (7, 62, 33), (1, 31, 66)])
def test_narrow_columns_routes(hip, outer, dim, inner):
    """Narrow columns at the edges of the flat form, the column tiles and the
    flat form's single chunk: sum and variance against float64, the index of
    the maximum exactly (the first of equal ones)."""
    x = SplitMix64(0x2A4 + dim * inner).normal((outer, dim, inner), 0.5, 1.0)
    x[:, dim // 2] = x[:, dim // 3]
    dx = DeviceArray.from_numpy(x)
    z, zi = DeviceArray((outer, inner), np.float32), DeviceArray((outer, inner), np.int32)
    x64 = x.astype(np.float64)
    engine.reduce.sum(dx, z, outer, dim, inner)
    assert np.all(np.abs(z.numpy() - x64.sum(1)) <= 1e-6 * np.abs(x64).sum(1))
    engine.reduce.var(dx, z, outer, dim, inner)
    assert np.allclose(z.numpy(), x64.var(1), rtol=1e-6)
    engine.reduce.argmax(dx, zi, outer, dim, inner)
    assert np.array_equal(zi.numpy(), x.argmax(1))
