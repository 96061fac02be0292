"""MoE layers whose experts get enough tokens for the f16 matrix cores
(k_gemm.hip's grouped kernel: over 512 slots, six or more per active expert; of
fewer slots the integer kernel that scans the ranking takes them, some cases here
among them) and the route that serves them, at the edges: expert loads around a
32-slot tile, experts without tokens, row blocks that end early, the
allocation-free entry's bits, non-finite tokens, outliers.

Tolerance: as the matmul's (x within 2^-23, exact products, f32 sums), twice
over for the two products in a row, with the oracle's own f32 sums: 4e-6.
"""
import numpy as np
import pytest

from test_gpu_moe import Layer, moe_dev

pytestmark = pytest.mark.gpu

TOL = 4e-6


def moe_noalloc(gpu, layer, xs):
    n = xs.size // layer.h
    xd, od = gpu.dev_alloc(xs.nbytes), gpu.dev_alloc(xs.nbytes)
    try:
        gpu.h2d(xd, xs)
        assert gpu.moe_ffn_dev_noalloc(layer.name, xd, n, od), gpu.last_error()
        gpu.sync()
        return gpu.d2h(od, (n, layer.h), np.float32)
    finally:
        gpu.dev_free(xd)
        gpu.dev_free(od)


@pytest.mark.parametrize("n_exp,h,ffn,top_k,n", [
    (8, 512, 256, 2, 128),     # 32 slots per expert: about half the experts need a second tile
    (16, 256, 256, 1, 97),     # one super-block per row, one slot per token
    (5, 768, 512, 3, 40),      # three super-blocks
    (128, 256, 256, 8, 300),   # many experts, over 512 slots
    (200, 512, 256, 5, 260),   # more than 128 experts; 4.. slots each on average
    (32, 512, 256, 8, 700),    # two route blocks of at most 4096 slots
    # over 512 slots: 65 per expert, one slot per token and super-block, three
    # super-blocks, row blocks of 128 and 256 that end early, just over the line
    (8, 512, 256, 2, 260), (16, 256, 256, 1, 520), (5, 768, 512, 3, 180), (6, 1280, 768, 3, 171),
])
def test_moe_many_tokens_match_cpu(gpu, orc, n_exp, h, ffn, top_k, n):
    layer = Layer(orc, n_exp, h, ffn, top_k, 310 + n)
    xs = orc.normal(n * h, 1.0, 311, n)
    try:
        layer.upload(gpu)
        print(f"moe gemm {n_exp} experts {h}x{ffn} top-{top_k} n={n}", flush=True)
        out, idx, wgt = moe_dev(gpu, layer, xs)
        for t in sorted({0, 1, 31, 32, n // 2, n - 1}):
            ref, ci, cw = layer.cpu(orc, xs[t * h:(t + 1) * h])
            assert np.array_equal(idx[t], ci), t
            assert orc.rel_l2(wgt[t], cw) < 1e-6
            assert orc.rel_l2(out[t], ref) < TOL, (t, orc.rel_l2(out[t], ref))
        # the allocation-free entry converts x in every workgroup: the same bits
        slots_bytes = n * top_k * (h + ffn) * 4
        if slots_bytes < 7 << 20:
            xd, od = gpu.dev_alloc(xs.nbytes), gpu.dev_alloc(n * h * 4)
            try:
                gpu.h2d(xd, xs)
                assert gpu.moe_ffn_dev_noalloc(layer.name, xd, n, od), gpu.last_error()
                gpu.sync()
                assert np.array_equal(gpu.d2h(od, (n, h), np.float32), out)
            finally:
                gpu.dev_free(xd)
                gpu.dev_free(od)
    finally:
        layer.drop(gpu)


@pytest.mark.parametrize("n", [64, 200])  # 192 slots (the integer kernel), 600 (the f16 one)
def test_moe_many_tokens_outliers_and_nonfinite(gpu, orc, n):
    """Tokens with elements 1e6 times the rest keep to the CPU's result, a NaN
    token's outputs are NaN, and neither touches the others."""
    n_exp, h, ffn, top_k = 6, 512, 256, 3
    layer = Layer(orc, n_exp, h, ffn, top_k, 330)
    xs = orc.normal(n * h, 1.0, 331, n).reshape(n, h)
    clean = xs.copy()
    xs[3, 7] *= np.float32(1e6)
    xs[3, 300] *= np.float32(1e6)
    xs[5, 100] = np.nan
    try:
        layer.upload(gpu)
        base, _, _ = moe_dev(gpu, layer, clean.ravel())
        out, idx, _ = moe_dev(gpu, layer, xs.ravel())
        assert np.isnan(out[5]).all()
        same = [t for t in range(n) if t not in (3, 5)]
        assert np.array_equal(out[same], base[same])
        ref, ci, _ = layer.cpu(orc, xs[3])
        assert np.array_equal(idx[3], ci)
        assert orc.rel_l2(out[3], ref) < TOL, orc.rel_l2(out[3], ref)
        # the allocation-free entry: the same bits
        bare = moe_noalloc(gpu, layer, xs.ravel())
        assert np.isnan(bare[5]).all()
        assert np.array_equal(np.delete(bare, 5, 0), np.delete(out, 5, 0))
    finally:
        layer.drop(gpu)


def test_moe_many_tokens_intermediate_outliers(gpu, orc):
    """Three rows of every expert's gate and up 2^11 times the others, so that
    where their gate is positive the intermediate activations hold elements some
    2^22 times the rest: down must add them, from staged x and without.

    Few elements carry such a result, so a product's error (4e-7 of its terms'
    size) meets gates that cancel to a tenth of that size: 2e-5."""
    n_exp, h, ffn, top_k, n = 6, 512, 256, 3, 200
    layer = Layer(orc, n_exp, h, ffn, top_k, 336)
    for w in layer.gate + layer.up:
        dm = w.reshape(ffn, h // 256, 144)[:, :, :4].view(np.float16)
        dm[..., 0], dm[..., 1] = 2.0 ** -10, 2.0 ** -7
        dm[[7, 40, 200]] *= np.float16(2.0 ** 11)
    xs = orc.normal(n * h, 1.0, 337, n).reshape(n, h)
    try:
        layer.upload(gpu)
        out = moe_dev(gpu, layer, xs.ravel())[0]
        assert np.array_equal(moe_noalloc(gpu, layer, xs.ravel()), out)
        for t in (0, 1, 2, n // 2, n - 1):
            ref, _, _ = layer.cpu(orc, xs[t])
            assert orc.rel_l2(out[t], ref) < 2e-5, (t, orc.rel_l2(out[t], ref))
    finally:
        layer.drop(gpu)


@pytest.mark.parametrize("n_exp,h,top_k,n", [(128, 2048, 8, 160), (17, 68, 3, 163), (256, 260, 64, 64), (1, 64, 1, 200),
                                             (33, 4100, 5, 333)])
def test_router_topk_many_tokens(gpu, orc, n_exp, h, top_k, n):
    """The matrix-core logits at tiles that end early, widths that end inside a
    16-column step, one expert, 256 experts."""
    w = orc.normal(n_exp * h, 0.05, 340, n_exp)
    xs = orc.normal(n * h, 1.0, 341, n)
    idx, wgt = np.full(n * top_k, -1, np.int32), np.zeros(n * top_k, np.float32)
    key = f"router.many.{n_exp}.{h}.{n}"
    assert gpu.router_topk(key, w, xs, n, h, n_exp, top_k, idx, wgt), gpu.last_error()
    # against 64 bits (the oracle's f32 sum of 2048 terms in a row is itself 1e-6 off); a logit here is
    # within about 2^-22 of its terms' size, some 1e-6, and so are the probabilities
    W, X = w.reshape(n_exp, h).astype(np.float64), xs.reshape(n, h).astype(np.float64)
    idx, wgt = idx.reshape(n, top_k), wgt.reshape(n, top_k)
    for t in range(n):
        lg = W @ X[t]
        p = np.exp(lg - lg.max())
        p /= p.sum()
        order = np.argsort(-p, kind="stable")[:top_k]
        assert np.array_equal(idx[t], order) or np.allclose(p[idx[t]], p[order], rtol=1e-5, atol=0), t
        assert len(set(idx[t].tolist())) == top_k
        assert orc.rel_l2(wgt[t], p[order] / p[order].sum()) < 4e-6, t


@pytest.mark.parametrize("n_exp,h,top_k,n", [
    (128, 2048, 8, 520), (256, 260, 16, 160), (33, 4100, 5, 800), (131, 68, 3, 190),  # past ROUTE_LOGITS
    (17, 68, 3, 163),
])
def test_routing_does_not_depend_on_the_call(gpu, orc, n_exp, h, top_k, n):
    """A token's experts and weights have the same bits whether it is routed
    alone, with a few others or with many (also where a call ends in a smaller
    block): a near-tie must not go another way."""
    w = orc.normal(n_exp * h, 0.05, 343, n_exp)
    xs = orc.normal(n * h, 1.0, 344, n).reshape(n, h)

    def route(rows):
        idx, wgt = np.full(len(rows) * top_k, -1, np.int32), np.zeros(len(rows) * top_k, np.float32)
        assert gpu.router_topk(f"router.cut.{n_exp}.{h}", w, np.ascontiguousarray(rows).ravel(), len(rows), h, n_exp, top_k,
                               idx, wgt), gpu.last_error()
        return idx.reshape(-1, top_k), wgt.reshape(-1, top_k)

    many = route(xs)
    for t0, c in ((0, 1), (1, 8), (9, 33), (n - 3, 3), (n // 2, 1)):
        few = route(xs[t0:t0 + c])
        assert np.array_equal(many[0][t0:t0 + c], few[0]), t0
        assert np.array_equal(many[1][t0:t0 + c].view(np.uint32), few[1].view(np.uint32)), t0


def test_moe_many_tokens_outliers_above_subnormals(gpu, orc):
    """Tokens of a few ordinary elements among subnormal ones, 600 slots of six
    experts: the elements taken out must be added though 2^-s of the rest of
    their block leaves f32's range; the allocation-free entry too."""
    n_exp, h, ffn, top_k, n = 6, 512, 256, 3, 200
    layer = Layer(orc, n_exp, h, ffn, top_k, 333)
    xs = (orc.normal(n * h, 1.0, 334, n) * np.float32(1e-42)).reshape(n, h)
    xs[:, 10::256] = orc.normal(n * (h // 256), 1.0, 335, n).reshape(n, -1)
    xs[:, 200::256] = np.float32(3.0)
    try:
        layer.upload(gpu)
        for name, out in (("eager", moe_dev(gpu, layer, xs.ravel())[0]), ("noalloc", moe_noalloc(gpu, layer, xs.ravel()))):
            for t in (0, 1, n // 2, n - 1):
                ref, _, _ = layer.cpu(orc, xs[t])
                assert orc.rel_l2(out[t], ref) < TOL, (name, t, orc.rel_l2(out[t], ref))
    finally:
        layer.drop(gpu)


def test_moe_many_tokens_marks_in_long_rows(gpu, orc):
    """Rows of 68 super-blocks, more than the 64 that marks are kept for: tokens
    with a large element, and with one half 1e6 times the other, in super-blocks on
    either side of that and in one whose place another shares, keep the CPU's result
    and leave the others' bits."""
    n_exp, h, ffn, top_k, n = 2, 17408, 256, 2, 260
    layer = Layer(orc, n_exp, h, ffn, top_k, 338)
    clean = orc.normal(n * h, 1.0, 339, n).reshape(n, h)
    xs = clean.copy()
    marked = (3, 40, 41, 259)
    xs[3, 7] *= np.float32(1e6)                         # super-block 0
    xs[40, 256 * 64 + 128:256 * 65] *= np.float32(1e6)  # 64, which shares 0's place
    xs[41, 256 * 63 + 5] *= np.float32(1e6)
    xs[259, 256 * 67:256 * 67 + 128] *= np.float32(1e6)
    xs[259, 256 * 30 + 200] *= np.float32(1e6)
    try:
        layer.upload(gpu)
        base = moe_dev(gpu, layer, clean.ravel())[0]
        out, idx, _ = moe_dev(gpu, layer, xs.ravel())
        same = [t for t in range(n) if t not in marked]
        assert np.array_equal(out[same], base[same])
        for t in marked:
            ref, ci, _ = layer.cpu(orc, xs[t])
            assert np.array_equal(idx[t], ci), t
            assert orc.rel_l2(out[t], ref) < TOL, (t, orc.rel_l2(out[t], ref))
    finally:
        layer.drop(gpu)
