"""Matmul on the f16 matrix cores (k_gemm.hip; GpuDispatch::matmul,
gpu.rs:443-455): Q4_K, Q6_K and Q8_0 against x in two f16 parts, at the sizes
where the tiles, splits and dispatch can go wrong.

Tolerance: x is within 2^-23 of each element above 2^-16 of its block's largest
(2^-39 of the largest below), every product exact, and a result
takes one f32 rounding per 16 columns of a super-block and per super-block:
about sqrt(33) * 2^-25 of the summed products' size, which the codes' offset
(mean 7.5 of 0..15) makes up to three times the result's.  2e-6 covers both
with a factor of two; the paths they took before are held to 1e-5.
"""
import numpy as np
import pytest

from test_gpu_matvec import zero_columns

pytestmark = pytest.mark.gpu

TOL = 2e-6
Q8, Q4K, Q6K = 2, 3, 13


def run(gpu, orc, dtype, rows, cols, xs, w, key):
    n = len(xs)
    out = np.full(n * rows, np.nan, np.float32)
    try:
        assert gpu.matmul(key, w, dtype, rows, cols, n, xs, out), gpu.last_error()
    finally:
        gpu.weight_drop(key)
    return out.reshape(n, rows)


@pytest.mark.parametrize("dtype,rows,cols,n", [
    # few-token kernel: one tile (full, one past, one short of it), rows that end inside a 32-row
    # tile and a 256-row block, one super-block per split, more splits than fit evenly
    (Q4K, 4096, 4096, 8), (Q4K, 1025, 4096, 31), (Q4K, 1055, 4096, 32), (Q4K, 4097, 4096, 33),
    (Q4K, 300, 4352, 4), (Q4K, 1, 4352, 5), (Q6K, 4100, 4352, 7), (Q6K, 289, 6912, 32),
    # tiled kernel: 64-token tiles (one full, one token over, ragged), one and several splits
    (Q4K, 14336, 4096, 64), (Q4K, 4099, 14336, 65), (Q6K, 4096, 14336, 127), (Q6K, 2500, 512, 1700),
    # Q8_0: whole and partial last super-blocks (64, 128 and 192 columns of one; an odd block padded)
    (Q8, 4096, 4096, 17), (Q8, 1300, 4160, 33), (Q8, 4099, 1152, 40), (Q8, 4097, 1216, 16), (Q8, 333, 4448, 6),
    # small weights of 4096 and 2048 columns, on both sides of the line
    (Q4K, 100, 4096, 9), (Q8, 100, 4096, 16), (Q8, 512, 3072, 17), (Q8, 300, 2048, 313), (Q4K, 300, 1536, 1751),
    # odd row and token counts whose product is no multiple of four, over several splits
    (Q4K, 4097, 4096, 17), (Q8, 1301, 6400, 19),
    # Q4_K from 3584 columns, on both sides of the line and of its token counts
    (Q4K, 1025, 3328, 16), (Q4K, 300, 3584, 9), (Q4K, 1025, 3584, 16), (Q4K, 1000, 3840, 33), (Q4K, 4097, 3840, 64),
    # whole rounds of 16 tokens in one pass of the integer kernels, and one round past it
    (Q4K, 4096, 1536, 128), (Q4K, 4096, 1536, 144), (Q4K, 2048, 2304, 128), (Q4K, 2048, 2304, 144),
])
def test_matmul_f16_matrix_cores(gpu, orc, dtype, rows, cols, n):
    w = orc.synth(dtype, rows, cols, 201, rows + n)
    xs = orc.normal(n * cols, 1.0, 202, cols + n).reshape(n, cols)
    print(f"gemm dtype {dtype} {rows}x{cols} n={n}", flush=True)
    out = run(gpu, orc, dtype, rows, cols, xs, w, f"gemm.{dtype}.{rows}.{cols}.{n}")
    for t in sorted({0, 1, n // 2, n - 2, n - 1}):
        assert orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t])) < TOL, t
    assert np.all(np.isfinite(out))


@pytest.mark.parametrize("dtype,rows,cols,n", [(Q4K, 4200, 4096, 9), (Q4K, 14400, 4096, 70), (Q6K, 300, 4352, 9),
                                               (Q6K, 1000, 1024, 1300), (Q8, 1100, 4224, 33),
                                               (Q8, 333, 4160, 33), (Q8, 300, 4544, 40), (Q8, 300, 4128, 20),
                                               (Q8, 300, 4256, 20)])
@pytest.mark.parametrize("ratio", [1e4, 1e6, 1e9])
def test_matmul_f16_outliers_under_zero_weights(gpu, orc, dtype, rows, cols, n, ratio):
    """Two elements of every 128 columns `ratio` times the rest, zero weights
    under them: the result is made of the small elements alone, which must
    keep the precision they have without the large ones."""
    zc = np.sort(np.concatenate([np.arange(5, cols, 128), np.arange(97, cols, 128)]))
    w = zero_columns(dtype, orc.synth(dtype, rows, cols, 203, n), rows, cols, zc)
    xs = orc.normal(n * cols, 1.0, 204, n).reshape(n, cols)
    xs[:, zc] *= np.float32(ratio)
    out = run(gpu, orc, dtype, rows, cols, xs, w, f"gemm.outl.{dtype}.{ratio}")
    for t in (0, n // 2, n - 1):
        e = orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t]))
        assert e < TOL, (t, e)


@pytest.mark.parametrize("dtype,rows,cols,n", [(Q4K, 4200, 4096, 9), (Q4K, 14400, 4096, 70), (Q6K, 300, 4352, 9),
                                               (Q8, 1100, 4224, 33)])
def test_matmul_f16_outliers_join(gpu, orc, dtype, rows, cols, n):
    """Elements that the staging takes out (1e7 times the rest) under ordinary
    weights carry the result."""
    w = orc.synth(dtype, rows, cols, 205, n)
    xs = orc.normal(n * cols, 1.0, 206, n).reshape(n, cols)
    for t in range(0, n, 2):
        xs[t, (37 * t + 11) % cols::640] *= np.float32(1e7)
    out = run(gpu, orc, dtype, rows, cols, xs, w, f"gemm.join.{dtype}")
    for t in (0, 1, n - 1):
        e = orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t]))
        assert e < TOL, (t, e)


@pytest.mark.parametrize("dtype,rows,cols,n", [(Q4K, 4200, 4096, 9), (Q4K, 14400, 4096, 70), (Q6K, 300, 4352, 9),
                                               (Q8, 1100, 4224, 33)])
def test_matmul_f16_nonfinite_and_extreme_tokens(gpu, orc, dtype, rows, cols, n):
    """A token with an Inf or a NaN gives non-finite outputs and leaves the
    others alone; tokens of 1e-30, 1e30 and zeros keep their precision."""
    w = orc.synth(dtype, rows, cols, 207, n)
    xs = orc.normal(n * cols, 1.0, 208, n).reshape(n, cols)
    xs[1, 300] = np.inf
    xs[2, cols - 1] = np.nan
    xs[3] *= np.float32(1e-30)
    xs[4] *= np.float32(1e30)
    xs[5] = 0.0
    out = run(gpu, orc, dtype, rows, cols, xs, w, f"gemm.ext.{dtype}")
    assert not np.isfinite(out[1]).any() and not np.isfinite(out[2]).any()
    assert np.all(out[5] == 0.0)
    for t in (0, 3, 4, 6, n - 1):
        assert orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t])) < TOL, t


@pytest.mark.parametrize("dtype,rows,cols,n", [
    (Q4K, 4096, 4352, 6),    # the batched vector kernel
    (Q4K, 14336, 4096, 64),  # the integer kernels, which would stage x in scratch too
    (Q8, 4096, 4096, 64),
])
def test_matmul_captured_before_any_scratch(orc, dtype, rows, cols, n):
    """A capture that comes before any eager call finds no scratch to grow: the
    kernels that need none take it, and the replays give the product."""
    from soso_amd.dispatch import HipGpu
    w = orc.synth(dtype, rows, cols, 209, 1)
    xs = orc.normal(n * cols, 1.0, 210, 1).reshape(n, cols)
    with HipGpu(0) as g:
        assert g.gemma_subir("w", w, dtype, rows, cols), g.last_error()
        xd, yd = g.dev_alloc(xs.nbytes), g.dev_alloc(n * rows * 4)
        g.h2d(xd, xs)
        g.graph_begin()
        ok = g.matmul_dev("w", n, xd, yd)
        gid = g.graph_end()
        assert ok, g.last_error()
        for _ in range(3):
            g.h2d(yd, np.zeros(n * rows, np.float32))
            g.graph_launch(gid)
            g.sync()
            out = g.d2h(yd, (n, rows), np.float32)
            for t in {0, 3, n - 1}:
                assert orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t])) < 1e-5, t
        # an eager call grows the scratch; the graph's replays go on
        assert g.matmul_dev("w", n, xd, yd), g.last_error()
        g.sync()
        eager = g.d2h(yd, (n, rows), np.float32)
        assert orc.rel_l2(eager, out) < 1e-5
        g.graph_launch(gid)
        g.sync()
        assert np.array_equal(g.d2h(yd, (n, rows), np.float32), out)
        g.dev_free(xd)
        g.dev_free(yd)


@pytest.mark.parametrize("rows,cols,n", [(4096, 1024, 128), (4096, 1024, 129), (8192, 4096, 200), (70000, 256, 130)])
def test_matmul_host_long_transfers(gpu, orc, rows, cols, n):
    """Host-buffer calls whose y is one, just over one, several and over sixteen
    2 MiB pieces, x up to two: the device entry's bits."""
    w = orc.synth(Q8, rows, cols, 211, n)
    xs = orc.normal(n * cols, 1.0, 212, n).reshape(n, cols)
    key = f"gemm.host.{rows}.{n}"
    out = np.full((n, rows), np.nan, np.float32)
    xd, yd = gpu.dev_alloc(xs.nbytes), gpu.dev_alloc(out.nbytes)
    try:
        assert gpu.matmul(key, w, Q8, rows, cols, n, xs, out), gpu.last_error()
        gpu.h2d(xd, xs)
        assert gpu.matmul_dev(key, n, xd, yd), gpu.last_error()
        gpu.sync()
        assert np.array_equal(gpu.d2h(yd, (n, rows), np.float32), out)
    finally:
        gpu.weight_drop(key)
        gpu.dev_free(xd)
        gpu.dev_free(yd)


@pytest.mark.parametrize("dtype,rows,cols,n", [(Q4K, 4200, 4096, 9), (Q4K, 14400, 4096, 70), (Q6K, 300, 4352, 9),
                                               (Q6K, 4100, 4352, 130), (Q8, 1100, 4224, 33), (Q8, 333, 4160, 33),
                                               (Q8, 300, 4544, 40), (Q8, 300, 4128, 20), (Q8, 300, 4256, 20)])
def test_matmul_f16_outliers_above_subnormals(gpu, orc, dtype, rows, cols, n):
    """Two elements of ordinary size in every 256, the others subnormal (what a
    SwiGLU that underflows leaves): the large ones are taken out of the scale,
    2^-s of the rest leaves f32's range, and they must still be added."""
    w = orc.synth(dtype, rows, cols, 213, n)
    xs = (orc.normal(n * cols, 1.0, 214, n) * np.float32(1e-42)).reshape(n, cols)
    xs[:, 10::256] = np.float32(1.0)
    xs[:, 200::256] = np.float32(0.5)
    out = run(gpu, orc, dtype, rows, cols, xs, w, f"gemm.subn.{dtype}.{n}")
    for t in (0, 1, n // 2, n - 1):
        e = orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t]))
        assert e < TOL, (t, e)


HALVES = [(Q4K, 4200, 4096, 9), (Q4K, 14400, 4096, 70), (Q6K, 300, 4352, 9), (Q8, 1100, 4224, 33)]


@pytest.mark.parametrize("dtype,rows,cols,n", HALVES)
@pytest.mark.parametrize("ratio", [1e4, 1e6, 1e7, 1e9])
def test_matmul_f16_halves_apart(gpu, orc, dtype, rows, cols, n, ratio):
    """One 128-column half of a super-block `ratio` times the rest throughout,
    zero weights under it: the other half, which shares its scale, must keep
    its precision."""
    nb = cols // 256
    zc = np.array([c for c in range(256 * nb) if (c >> 7) % 2 == (c >> 8) % 2])
    w = zero_columns(dtype, orc.synth(dtype, rows, cols, 215, n), rows, cols, zc)
    xs = orc.normal(n * cols, 1.0, 216, n).reshape(n, cols)
    for t in range(n):
        h = 256 * (t % nb) + 128 * (t % nb % 2)
        xs[t, h:h + 128] *= np.float32(ratio)
    out = run(gpu, orc, dtype, rows, cols, xs, w, f"gemm.half.{dtype}.{ratio}")
    for t in (0, 1, n // 2, n - 1):
        e = orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t]))
        assert e < TOL, (t, e)


@pytest.mark.parametrize("dtype,rows,cols,n", HALVES)
@pytest.mark.parametrize("ratio", [1e5, 1e7, 1e9])
def test_matmul_f16_sparse_halves(gpu, orc, dtype, rows, cols, n, ratio):
    """Halves of one or two elements, one of them `ratio` times the rest of the
    super-block and under a zero weight: beside a full half (t % 3 = 0, 1), and
    two such halves (2)."""
    nb = cols // 256
    zc = np.sort(np.concatenate([np.arange(5, 256 * nb, 256), np.arange(192, 256 * nb, 256)]))
    w = zero_columns(dtype, orc.synth(dtype, rows, cols, 217, n), rows, cols, zc)
    xs = orc.normal(n * cols, 1.0, 218, n).reshape(n, cols)
    for t in range(n):
        b = xs[t, :256 * nb].reshape(nb, 256)
        if t % 3 < 2:
            b[:, :128] = 0.0
            b[:, 5] = ratio
            b[:, 60] = t % 3
        else:
            b[:] = 0.0
            b[:, 3::128] = 7.0
            b[:, 192] = -ratio
    out = run(gpu, orc, dtype, rows, cols, xs, w, f"gemm.sparse.{dtype}.{ratio}")
    for t in (0, 1, 2, n - 1):
        e = orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t]))
        assert e < TOL, (t, e)


@pytest.mark.parametrize("dtype,rows,cols,n", HALVES)
@pytest.mark.parametrize("ratio", [1.0, 1e4, 1e7])
def test_matmul_f16_zero_groups(gpu, orc, dtype, rows, cols, n, ratio):
    """Super-blocks with whole groups of zeros: a zero 32-column group (t % 4 = 0),
    halves of three, two and one 8-column groups, one of whose elements is `ratio`
    times the rest and under a zero weight (1, 2, 3): the rest keeps its precision."""
    nb = cols // 256
    zc = np.arange(5, 256 * nb, 256)
    w = zero_columns(dtype, orc.synth(dtype, rows, cols, 221, n), rows, cols, zc)
    xs = orc.normal(n * cols, 1.0, 222, n).reshape(n, cols)
    for t in range(n):
        b = xs[t, :256 * nb].reshape(nb, 256)
        if t % 4 == 0:
            b[:, 64:96] = 0.0
        else:
            keep = np.zeros(128, bool)
            for c in (0, 40, 96)[:4 - t % 4]:
                keep[c:c + 8] = True
            b[:, :128][:, ~keep] = 0.0
            if t % 4 == 3:
                b[:, 128:] = 0.0
        b[:, 5] *= np.float32(ratio)
    out = run(gpu, orc, dtype, rows, cols, xs, w, f"gemm.zgroup.{dtype}.{ratio}")
    for t in (0, 1, 2, 3, n - 1):
        e = orc.rel_l2(out[t], orc.matvec_f64(dtype, w, rows, cols, xs[t]))
        assert e < TOL, (t, e)
