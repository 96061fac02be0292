"""The Gated DeltaNet block's kernels (k_gdn.hip) where their shapes change: the
token count at which a head moves from one workgroup to eight, the edges of the
32-token chunks, every unrolled conv width and the loop, and blocks cut so that
the pieces run on different kernels.

Tolerance: against the oracle's f32 restatement, whose own sums of 128 terms
are within a few 2^-24 of exact, as these are: 2e-6.
"""
import numpy as np
import pytest

from test_gpu_gdn import make_block

pytestmark = pytest.mark.gpu

D, EPS = 128, 1e-6


@pytest.mark.parametrize("n,n_k,n_v,kernel", [
    (3, 2, 4, 2), (4, 3, 3, 4), (5, 3, 6, 4), (31, 1, 2, 3), (32, 2, 2, 1), (33, 2, 4, 16), (65, 1, 1, 5), (96, 2, 5, 4),
])
def test_gdn_block_shapes(gpu, orc, n, n_k, n_v, kernel):
    print(f"gdn block n={n} n_k={n_k} n_v={n_v} kernel={kernel}", flush=True)
    hist, conv, z, decay, beta, norm, state = make_block(orc, n, n_k, n_v, D, kernel, 700 + n)
    ref_out, ref_state = orc.gdn_block(hist, conv, z, decay, beta, norm, state, n, n_k, n_v, D, kernel, EPS)
    st = state.copy()
    out = gpu.gdn_block(hist, conv, z, decay, beta, norm, st, n, n_k, n_v, D, kernel, EPS)
    assert out is not False, gpu.last_error()
    e_out, e_st = orc.rel_l2(out, ref_out), orc.rel_l2(st, ref_state)
    assert e_out < 2e-6 and e_st < 2e-6, (e_out, e_st)


@pytest.mark.parametrize("cuts", [(1, 40), (4, 9, 40), (33, 37, 40), (3, 8, 11, 15, 40)])
def test_gdn_block_pieces_keep_the_bits(gpu, orc, cuts):
    n, n_k, n_v, kernel = 40, 2, 4, 4
    C = (2 * n_k + n_v) * D
    hist, conv, z, decay, beta, norm, state = make_block(orc, n, n_k, n_v, D, kernel, 750)
    whole_st = state.copy()
    whole = gpu.gdn_block(hist, conv, z, decay, beta, norm, whole_st, n, n_k, n_v, D, kernel, EPS)
    H, st, outs, t0 = hist.reshape(kernel - 1 + n, C), state.copy(), [], 0
    for t1 in cuts:
        outs.append(gpu.gdn_block(H[t0:t1 + kernel - 1].ravel(), conv, z[t0 * n_v * D:t1 * n_v * D],
                                  decay[t0 * n_v:t1 * n_v], beta[t0 * n_v:t1 * n_v], norm, st, t1 - t0, n_k, n_v, D,
                                  kernel, EPS))
        t0 = t1
    assert np.array_equal(np.concatenate(outs), whole) and np.array_equal(st, whole_st)


@pytest.mark.parametrize("n", [2, 37])
def test_gdn_block_dev_pointers_off_by_a_float(gpu, orc, n):
    """Device buffers that start one float past an aligned address."""
    n_k, n_v, kernel = 2, 4, 4
    bufs = make_block(orc, n, n_k, n_v, D, kernel, 770)
    st = bufs[6].copy()
    out = gpu.gdn_block(*bufs[:6], st, n, n_k, n_v, D, kernel, EPS)
    ptrs = []
    try:
        for b in list(bufs) + [out]:
            p = gpu.dev_alloc(b.nbytes + 4)
            gpu.h2d(p + 4, b)
            ptrs.append(p)
        at = [p + 4 for p in ptrs]
        assert gpu.gdn_block_dev(*at, n, n_k, n_v, D, kernel, EPS), gpu.last_error()
        gpu.sync()
        assert np.array_equal(gpu.d2h(at[7], out.shape, np.float32), out)
        assert np.array_equal(gpu.d2h(at[6], st.shape, np.float32), st)
    finally:
        for p in ptrs:
            gpu.dev_free(p)


@pytest.mark.parametrize("n", [1, 4, 5, 33, 70])
def test_gdn_block_dev_out_is_z(gpu, orc, n):
    """The output may take z's buffer: the same bits as with one of its own."""
    n_k, n_v, kernel = 2, 4, 4
    bufs = make_block(orc, n, n_k, n_v, D, kernel, 780 + n)
    st = bufs[6].copy()
    out = gpu.gdn_block(*bufs[:6], st, n, n_k, n_v, D, kernel, EPS)
    ptrs = []
    try:
        for b in bufs:
            ptrs.append(gpu.dev_alloc(b.nbytes))
            gpu.h2d(ptrs[-1], b)
        assert gpu.gdn_block_dev(*ptrs, ptrs[2], n, n_k, n_v, D, kernel, EPS), gpu.last_error()
        gpu.sync()
        assert np.array_equal(gpu.d2h(ptrs[2], out.shape, np.float32), out)
        assert np.array_equal(gpu.d2h(ptrs[6], st.shape, np.float32), st)
    finally:
        for p in ptrs:
            gpu.dev_free(p)
