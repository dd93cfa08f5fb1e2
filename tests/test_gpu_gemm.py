"""GPU parity of the batched-prefill dequant-GEMM (lrs_gemm_dev) against the
CPU oracle's dequant (bit-exact dequant.rs restatement) and float64 products.

precision 1 (bf16 operands, f32 accumulation) is checked
against the exact product of the same bf16-rounded operands (tolerance 1e-5
relative L2: only the f32 summation order differs); precision 3 (f16 hi/lo
activations) against the f32 operands themselves (tolerance 1e-4).
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14


@pytest.fixture(scope="module")
def ctx(lrs):
    c = lrs.Context(0)
    yield c
    c.close()


def bf16(x):
    """Round float32 to the nearest bfloat16 (ties to even), as float32."""
    b = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    b = (b + 0x7FFF + ((b >> 16) & 1)) & 0xFFFF0000
    return b.astype(np.uint32).view(np.float32)


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, Q8_0])
# (64, 256, 4096), (96, 128, 8192) and (512, 384, 4096) split K over
# workgroups (few output tiles, long K); m >= 512 uses the 256-token tile at
# precision 1 (ragged m and n included)
@pytest.mark.parametrize("m,n,k", [(1, 200, 512), (7, 128, 256), (130, 300, 768), (256, 256, 1024),
                                   (64, 256, 4096), (96, 128, 8192), (512, 256, 1024),
                                   (600, 200, 512), (512, 384, 4096), (1000, 136, 2048)])
def test_gemm_matches_oracle(lrs, orc, ctx, t, m, n, k):
    w = orc.gen_weight(t, 31 + m + n, n, k, mode=1)
    deq = orc.dequant(t, w).reshape(n, k)
    a = np.random.default_rng(m * 7 + n).standard_normal((m, k)).astype(np.float32)
    W = lrs.Weight.upload(ctx, t, w, k, n)
    y1 = W.gemm(a, precision=1)
    ref1 = bf16(a).astype(np.float64) @ bf16(deq).astype(np.float64).T
    assert rel_l2(y1, ref1) < 1e-5
    y3 = W.gemm(a, precision=3)
    ref = a.astype(np.float64) @ deq.astype(np.float64).T
    assert rel_l2(y3, ref) < 1e-4
    # plain bf16 is ~2^-9 per operand: far from f32, which is why prefill uses 3
    assert rel_l2(y1, ref) < 1e-2


def test_gemm_row_of_one_hot_activations_is_a_weight_column(lrs, orc, ctx):
    """a = identity rows: y[i] = column i of W (exact for values that bf16
    represents, which the hi/lo activations reach to 2^-22)."""
    k, n = 256, 64
    w = orc.gen_weight(Q4_K, 5, n, k, mode=1)
    deq = orc.dequant(Q4_K, w).reshape(n, k)
    a = np.eye(k, dtype=np.float32)[:40]
    y = lrs.Weight.upload(ctx, Q4_K, w, k, n).gemm(a, precision=3)
    assert np.allclose(y, deq[:, :40].T, rtol=2e-5, atol=0)


def test_gemm_rejects_bad_arguments(lrs, orc, ctx):
    # n_in must be a multiple of 256 (one K-step of the tile), for Q8_0 too
    w = lrs.Weight.upload(ctx, Q8_0, orc.gen_weight(Q8_0, 1, 4, 64), 64, 4)
    with pytest.raises(lrs.ModelError):
        w.gemm(np.zeros((2, 64), np.float32))
    w4 = lrs.Weight.upload(ctx, Q4_K, orc.gen_weight(Q4_K, 1, 4, 256), 256, 4)
    with pytest.raises(lrs.ModelError):
        w4.gemm(np.zeros((2, 256), np.float32), precision=2)


@pytest.mark.parametrize("types,m", [((Q4_K, Q4_K, Q6_K), 512), ((Q4_K, Q4_K, Q6_K), 130),
                                     ((Q5_K, Q6_K), 600), ((Q8_0, Q8_0), 77), ((Q6_K,), 256)])
def test_gemm_group_equals_single_gemms(lrs, orc, ctx, types, m):
    """lrs_gemm_group_dev (the prompt block's q / k / v as one launch, segments
    of ragged width and two types) against the oracle at both precisions and
    against one lrs_gemm_dev call per weight (the same per-tile arithmetic;
    the single calls may split K, so within 1e-6 rather than bit-exact)."""
    k = 1024
    widths = [200, 136, 72][:len(types)]
    ws, deqs = [], []
    for i, (t, n) in enumerate(zip(types, widths)):
        w = orc.gen_weight(t, 71 + i, n, k, mode=1)
        deqs.append(orc.dequant(t, w).reshape(n, k))
        ws.append(lrs.Weight.upload(ctx, t, w, k, n))
    a = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    for prec in (1, 3):
        ys = lrs.gemm_group(ctx, ws, a, precision=prec)
        for y, w, deq in zip(ys, ws, deqs):
            single = w.gemm(a, precision=prec)
            assert rel_l2(y, single) < 1e-6
            if prec == 3:
                ref = a.astype(np.float64) @ deq.astype(np.float64).T
                assert rel_l2(y, ref) < 1e-4
            else:
                ref = bf16(a).astype(np.float64) @ bf16(deq).astype(np.float64).T
                assert rel_l2(y, ref) < 1e-5


def test_gemm_group_rejects_bad_groups(lrs, orc, ctx):
    w4 = lrs.Weight.upload(ctx, Q4_K, orc.gen_weight(Q4_K, 1, 16, 512), 512, 16)
    w6 = lrs.Weight.upload(ctx, Q6_K, orc.gen_weight(Q6_K, 2, 16, 512), 512, 16)
    w8 = lrs.Weight.upload(ctx, Q8_0, orc.gen_weight(Q8_0, 3, 16, 512), 512, 16)
    w4k = lrs.Weight.upload(ctx, Q4_K, orc.gen_weight(Q4_K, 4, 16, 256), 256, 16)
    a = np.zeros((4, 512), np.float32)
    for group in ([w6, w4], [w4, w6, w4], [w4, w8], [w4, w4k], [w4, w4, w4, w4]):
        with pytest.raises(lrs.ModelError):
            lrs.gemm_group(ctx, group, a)


def quantizer_like(t, n, k, seed):
    """GGUF blocks with every scale a quantizer can leave: Q6_K scales of -128
    (products above 2048), Q8_0 scales that differ by 2^12 inside a row, K-quant
    super-blocks with d = 0 (only the minimum counts) and with dmin = 0."""
    rng = np.random.default_rng(seed)
    be, bb = {Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}[t]
    b = rng.integers(0, 256, (n * k // be, bb), dtype=np.uint8)
    nb = b.shape[0]
    f16 = lambda v: np.ascontiguousarray(v, np.float16).view(np.uint8).reshape(nb, 2)
    if t == Q8_0:
        b[:, 0:2] = f16(2.0 ** rng.uniform(-16, -4, nb))
        b[rng.integers(0, nb, max(1, nb // 16)), 0:2] = 0
    elif t == Q6_K:
        b[:, 192] = 128
        b[:, 200] = 127
        b[:, 208:210] = f16(rng.uniform(0.7, 1.3, nb) * 1e-5)
    else:
        d = rng.uniform(0.5, 2.0, nb) * 1e-4
        d[rng.integers(0, nb, max(1, nb // 8))] = 0
        m = rng.uniform(0.5, 2.0, nb) * 1e-3
        m[rng.integers(0, nb, max(1, nb // 8))] = 0
        b[:, 0:2], b[:, 2:4] = f16(d), f16(m)
    return b.reshape(-1)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, Q8_0])
# row tiles of 32 tokens (1, 2 or 4 of them a workgroup) and 256 weight rows,
# K in whole super-blocks (1: nothing to prefetch; 3: an uneven K split): the
# sizes at, below and past each edge
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (2, 255, 256), (32, 257, 768), (33, 16, 512),
                                   (64, 272, 1280), (65, 513, 256), (129, 31, 2816)])
def test_gemm_edges_and_extreme_blocks(lrs, orc, ctx, t, m, n, k):
    """Tile edges, quantizer-like blocks, and activations whose rows differ by
    2^100, with a super-block of zeros and outliers of 2^12."""
    w = quantizer_like(t, n, k, m + n)
    deq = orc.dequant(t, w).reshape(n, k).astype(np.float64)
    rng = np.random.default_rng(n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, 5] *= 4096.0
    a[m // 2] *= np.float32(2.0 ** 50)
    a[m // 3] *= np.float32(2.0 ** -50)
    a[m - 1, :256] = 0.0
    W = lrs.Weight.upload(ctx, t, w, k, n)
    y3, y1 = W.gemm(a, precision=3), W.gemm(a, precision=1)
    ref3 = a.astype(np.float64) @ deq.T
    ref1 = bf16(a).astype(np.float64) @ bf16(deq.astype(np.float32)).astype(np.float64).T
    for r in range(m):
        # the sum's f32 rounding is relative to its terms, which cancel: the
        # bounds are the 22-bit activations' and f32 sums' against their size
        size = np.linalg.norm(np.abs(a[r].astype(np.float64)) @ np.abs(deq).T)
        assert np.linalg.norm(y3[r] - ref3[r]) <= 2e-6 * size
        # bf16 of a fused a * q - b may round the other way at a tie: 2^-9 of
        # a few weights
        assert np.linalg.norm(y1[r] - ref1[r]) <= 1e-5 * size


def zero_column_5(t, w):
    """Quantizer-like blocks whose weight 5 of every 256 is zero: beside an
    activation of any size there, the others' contributions show."""
    bb = {Q8_0: 34 * 8, Q4_K: 144, Q5_K: 176, Q6_K: 210}[t]
    b = w.reshape(-1, bb).copy()
    if t == Q8_0:
        b[:, 2 + 5] = 0
    elif t == Q6_K:
        b[:, 5] &= 0xF0
        b[:, 128 + 5] = (b[:, 128 + 5] & 0xFC) | 2
    else:
        b[:, 8] &= 0xC0  # the first sub-block's minimum
        b[:, {Q4_K: 16, Q5_K: 48}[t] + 5] &= 0xF0
        if t == Q5_K:
            b[:, 16 + 5] &= 0xFE
    return b.reshape(-1)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, Q8_0])
def test_gemm_activations_beside_a_large_one(lrs, orc, ctx, t):
    """One activation of 2^20 in every 256 (of either sign, its weights zero):
    the rest keep what a bf16 hi + lo pair would (2^-17 of themselves).  An
    element's error is at most 2^-40 of the largest's next power of two, 2^-19;
    the f32 sums add 2^-22 of the terms."""
    m, n, k = 33, 48, 768
    w = zero_column_5(t, quantizer_like(t, n, k, 3))
    deq = orc.dequant(t, w).reshape(n, k).astype(np.float64)
    assert not deq[:, 5::256].any()
    rng = np.random.default_rng(8)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, 5::256] = np.float32(2.0 ** 20) * rng.choice([-1, 1], (m, k // 256))
    y = lrs.Weight.upload(ctx, t, w, k, n).gemm(a, precision=3)
    a[:, 5::256] = 0
    ref = a.astype(np.float64) @ deq.T
    # independent roundings: their 2-norm, eight times (a K-quant's two terms,
    # scale times quant and the minimum, are each up to about twice the weight)
    tol = 8 * 2.0 ** -19 / np.sqrt(3) * np.linalg.norm(deq, axis=1) + 2.0 ** -22 * (np.abs(a) @ np.abs(deq).T)
    assert np.all(np.abs(y - ref) <= tol)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, Q8_0])
def test_gemm_super_blocks_of_different_size(lrs, orc, ctx, t):
    """Inside a row, 256-column blocks scaled by 2^20 and 2^-20 in turn: the
    small blocks alone (the others zero) as exact as any, and their scale taken
    into a sum with the large ones."""
    m, n, k = 5, 40, 1024
    w = quantizer_like(t, n, k, 4)
    deq = orc.dequant(t, w).reshape(n, k).astype(np.float64)
    a = np.random.default_rng(9).standard_normal((m, k)).astype(np.float32)
    s = np.repeat([2.0 ** 20, 2.0 ** -20, 2.0 ** 20, 2.0 ** -20], 256).astype(np.float32)
    W = lrs.Weight.upload(ctx, t, w, k, n)
    for keep in (s > 1, s < 1, s > 0):
        x = a * s * keep
        ref = x.astype(np.float64) @ deq.T
        y = W.gemm(x, precision=3)
        size = np.linalg.norm(np.abs(x.astype(np.float64)) @ np.abs(deq).T)
        assert np.linalg.norm(y - ref) <= 2e-6 * size


@pytest.mark.parametrize("t", [Q8_0, Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("n,k,shift", [(1, 256, 0), (17, 768, 0), (5, 512, 1)])
def test_dequant_into_any_float_address_is_exact(lrs, orc, ctx, t, n, k, shift):
    """lrs_weight_dequant_dev at whole and odd row tiles; Q8_0 rows that end
    inside 256 elements; an output that is not 16-byte aligned; nothing written
    past the end."""
    k += 32 if t == Q8_0 else 0
    w = quantizer_like(t, n, k, n)
    W = lrs.Weight.upload(ctx, t, w, k, n)
    out = ctx.alloc(4 * (n * k + 8))
    out.upload(np.full(n * k + 8, 7.0, np.float32))
    lrs.check(lrs.lib.lrs_weight_dequant_dev(ctx.h, W.h, out.ptr + 4 * shift))
    ctx.sync()
    got = out.download(np.float32, n * k + 8)
    ref = orc.dequant(t, w)
    assert np.array_equal(got[shift:shift + n * k].view(np.uint32), ref.view(np.uint32))
    assert np.all(got[:shift] == 7.0) and np.all(got[shift + n * k:] == 7.0)


@pytest.mark.parametrize("t", [Q4_K, Q8_0])
@pytest.mark.parametrize("prec,rows", [(1, 512), (1, 1024), (3, 512), (3, 768)])
def test_gemm_whose_partials_do_not_fit_the_scratch_gives_the_same_bits(lrs, orc, t, prec, rows):
    """Inside a capture the scratch may not grow. Where it holds the packed
    input (made by a call of `rows` tokens) but not the K slices' partial sums
    (2 MB each, at least three), the slices go by in rounds: of one, straight to y
    (512), or of the two that fit.  The same bits as a call whose partials fit,
    single and grouped."""
    n_in, n_out, m = 5120, 1024, 512
    a = np.random.default_rng(5).standard_normal((rows, n_in)).astype(np.float32)
    with lrs.Context(0) as c, lrs.Context(0) as free:
        host = [orc.gen_weight(t, 2 + i, n, n_in, mode=1) for i, n in enumerate((n_out, 256))]
        up = lambda x: [lrs.Weight.upload(x, t, h, n_in, n) for h, n in zip(host, (n_out, 256))]
        ws, wf = up(c), up(free)
        small = lrs.Weight.upload(c, t, orc.gen_weight(t, 1, 16, n_in), n_in, 16)
        small.gemm(a, precision=prec)  # the scratch holds this input
        ab = c.alloc(a.nbytes)
        ab.upload(a)
        ys = [c.alloc(4 * m * n_out), c.alloc(4 * m * n_out), c.alloc(4 * m * 256)]
        wa = (C.c_void_p * 2)(*[w.h for w in ws])
        ya = (C.c_void_p * 2)(ys[1].ptr, ys[2].ptr)

        def calls():
            ws[0].gemm_dev(ab, ys[0], m, prec)
            lrs.check(lrs.lib.lrs_gemm_group_dev(c.h, wa, 2, ab.ptr, ya, m, prec))

        g = c.capture(calls)
        ref = [wf[0].gemm(a[:m], precision=prec)] + lrs.gemm_group(free, wf, a[:m], precision=prec)
        for _ in range(3):
            for y in ys:
                y.upload(np.full(y.nbytes // 4, 7.0, np.float32))
            g.launch()
            c.sync()
            for y, r in zip(ys, ref):
                assert np.array_equal(y.download(np.float32, r.size).reshape(r.shape), r)
        g.close()


@pytest.mark.parametrize("prec", [1, 3])
@pytest.mark.parametrize("m", [1, 3, 33])
def test_short_gemm_first_made_inside_a_capture(lrs, orc, m, prec):
    """Whatever call made the scratch, its first size holds a short GEMM's packed
    input (whole tiles of 32 rows: 3.8 MB for 33 x 13824 at precision 3), so that
    a capture needs no such call before it; the bits of an eager call."""
    n_in, n_out = 13824, 256
    a = np.random.default_rng(m).standard_normal((m, n_in)).astype(np.float32)
    host = orc.gen_weight(Q4_K, 3, n_out, n_in, mode=1)
    with lrs.Context(0) as c:
        w = lrs.Weight.upload(c, Q4_K, host, n_in, n_out)
        w.matvec(a[0])
        ab, yb = c.alloc(a.nbytes), c.alloc(4 * m * n_out)
        ab.upload(a)
        g = c.capture(lambda: w.gemm_dev(ab, yb, m, prec))
        g.launch()
        c.sync()
        got = yb.download(np.float32, m * n_out).reshape(m, n_out)
        g.close()
        assert np.array_equal(got, w.gemm(a, precision=prec))
