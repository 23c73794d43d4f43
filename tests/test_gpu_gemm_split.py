"""The split-product GEMMs (gemm_split.hip): every fp32 operand as three bf16
parts, six products on the bf16 matrix cores.

  - the split itself, restated in numpy: the three parts add up to 2^24 times
    the operand exactly, from the smallest subnormal to 2^103, none of them is
    subnormal, and the products left out are below 2^-24 of the whole;
  - each variant at the edges of its tiles and k steps, componentwise within
    the bound of a sum of K rounded products, (K + 8) 2^-24 sum |a||b|;
  - sums over C's rows with operands of one sign: what the matrix cores' own
    rounding would leave in all rows alike is no more than the fp32 variant's;
  - the same bound for operands down to the smallest subnormals against large
    ones, and for operands and sums beyond what the scaled split holds;
  - infinities, NaN and magnitudes that bf16 rounds to infinity come out as
    fp32 gives them, and padding past N never reaches C;
  - the SwiGLU epilogues agree with the oracle through the decoder's prefill.
"""
import numpy as np
import pytest

SPLIT_TILES = ["128x128", "64x128_k32", "64x64_k32"]
U = 2.0 ** -24


def bf16(x):
    """fp32 rounded to bf16, nearest even (finite values)."""
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)


def test_three_parts_add_up_exactly():
    rng = np.random.default_rng(0)
    x = np.ldexp(rng.uniform(1, 2, 200000), rng.integers(-149, 103, 200000)).astype(np.float32)
    x *= rng.choice(np.float32([-1, 1]), x.size) * np.float32(2.0 ** 24)
    h = bf16(x)
    m = bf16(x - h)
    low = (x - h) - m
    assert np.array_equal(bf16(low), low)            # the last part is a bf16 as it stands
    s = h.astype(np.float64) + m + low
    assert np.array_equal(s, x.astype(np.float64))
    assert all((np.abs(v[v != 0]) >= 2.0 ** -126).all() for v in (h, m, low))
    a, b = slice(0, 100000), slice(100000, 200000)
    H, M, L = [v.astype(np.float64) for v in (h, m, low)]
    left = np.abs(M[a] * L[b]) + np.abs(L[a] * M[b]) + np.abs(L[a] * L[b])
    assert (left <= U * np.abs(s[a] * s[b])).all()


def operands(dev, A, B, ta, tb, fill=0.0):
    """op(A), op(B) on the device, rows padded to 16 bytes with `fill`."""
    out = []
    for x, t in ((A, ta), (B, tb)):
        x = x.T if t else x
        p = np.full((x.shape[0], (x.shape[1] + 3) // 4 * 4), fill, np.float32)
        p[:, :x.shape[1]] = x
        out += [dev.upload(p), p.shape[1]]
    return out


def product(dev, tile, splits, A, B, ta, tb, fill=0.0):
    (M, K), N = A.shape, B.shape[1]
    dA, lda, dB, ldb = operands(dev, A, B, ta, tb, fill)
    dC = dev.upload(np.full((M, N), 7.0, np.float32))
    try:
        dev.force(tile, splits)
        dev.matmul(ta, tb, dA, dB, dC, M, N, K, lda, ldb, N)
        family = "xgemm" if tile in SPLIT_TILES else "gemm"
        assert dev.last_variant() == ("k_%s_%s_%s" % (family, ["nn", "nt", "tn"][2 * ta + tb], tile), splits)
        return dev.download(dC, (M, N))
    finally:
        dev.force(None)
        for p in (dA, dB, dC):
            dev.free(p)


@pytest.fixture(scope="module")
def dev(trlm):
    d = trlm.Device()
    yield d
    d.close()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", SPLIT_TILES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K,splits", [(1, 1, 1, 1), (129, 63, 31, 1), (64, 128, 32, 1), (63, 131, 33, 1),
                                          (130, 257, 65, 1), (257, 66, 447, 1), (128, 128, 4099, 3)])
def test_edges(dev, tile, ta, tb, M, N, K, splits):
    rng = np.random.default_rng(M + 3 * N + 7 * K + ta + 2 * tb)
    A = (rng.standard_normal((M, K)) * np.exp2(rng.integers(-12, 13, (M, 1)))).astype(np.float32)
    B = (rng.standard_normal((K, N)) * np.exp2(rng.integers(-12, 13, (1, N)))).astype(np.float32)
    got = product(dev, tile, splits, A, B, ta, tb)
    want = A.astype(np.float64) @ B.astype(np.float64)
    bound = (K + 8) * U * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))
    assert (np.abs(got - want) <= bound).all(), float((np.abs(got - want) / bound).max())


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K,splits", [(1, 1, 1, 1), (129, 63, 31, 1), (63, 131, 33, 1), (257, 67, 447, 2),
                                          (2051, 4099, 37, 1), (3001, 4001, 131, 1)])
def test_unaligned_edges(dev, M, N, K, ta, tb, splits):
    """Tight odd rows (64x64_u, and 128x128_u for the last shape): every value
    is loaded by itself and none past the last row's end (an odd M or N leaves
    a pair's second row outside)."""
    rng = np.random.default_rng(M + 3 * N + 7 * K + ta + 2 * tb)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    As, Bs = [np.ascontiguousarray(x.T if t else x) for x, t in ((A, ta), (B, tb))]
    dA, dB, dC = dev.upload(As), dev.upload(Bs), dev.upload(np.full((M, N), 7.0, np.float32))
    try:
        dev.force(None, splits)     # a forced split count leaves the 32x32 kernels out
        dev.matmul(ta, tb, dA, dB, dC, M, N, K, As.shape[1], Bs.shape[1], N)
        name = dev.last_variant()[0]
        got = dev.download(dC, (M, N))
    finally:
        dev.force(None)
        for p in (dA, dB, dC):
            dev.free(p)
    if As.shape[1] % 4 or Bs.shape[1] % 4:
        assert name == "k_xgemm_%s_%s_u" % (["nn", "nt", "tn", "tt"][2 * ta + tb],
                                            "128x128" if M == 3001 and not (ta and tb) else "64x64")
    want = A.astype(np.float64) @ B.astype(np.float64)
    bound = (K + 8) * U * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))
    assert (np.abs(got - want) <= bound).all(), (name, float((np.abs(got - want) / np.maximum(bound, 1e-30)).max()))


@pytest.mark.gpu
@pytest.mark.parametrize("tile", SPLIT_TILES)
def test_row_sums_keep_no_common_error(dev, tile):
    """A of one sign against the same B: every row of C sums the same way, so a
    rounding bias would be the same in all rows.  The error of C's column sums
    is at most four times the fp32 variant's (256x128, the same splits)."""
    rng = np.random.default_rng(5)
    M, N, K = 1024, 128, 8192
    A = rng.random((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    want = (A.astype(np.float64) @ B.astype(np.float64)).sum(0)
    err = {}
    for t in (tile, "256x128"):
        got = product(dev, t, 4, A, B, 0, 0).astype(np.float64).sum(0)
        err[t] = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err[tile] <= 4 * err["256x128"] + U, err


@pytest.mark.gpu
@pytest.mark.parametrize("tile", SPLIT_TILES)
@pytest.mark.parametrize("ea,eb", [(-111, 90), (-115, 100), (100, -120), (-126, 103), (103, -126), (-149, 103),
                                   (103, -140), (-60, -60), (110, -100), (-126, 120), (50, 60)])
def test_ends_of_the_range(dev, tile, ea, eb):
    """Operands around 2^ea and 2^eb: 24 bits of each count, down to the
    subnormals (-126 and below; an operand of -149 has its one bit), up to the
    split's 2^104, and past it and past sums of 2^80 (the last three)."""
    rng = np.random.default_rng(1000 + ea + 3 * eb)
    M, N, K = 130, 67, 77
    A = np.ldexp(rng.choice([-1.0, 1.0], (M, K)) * rng.uniform(1, 2, (M, K)), ea).astype(np.float32)
    B = np.ldexp(rng.choice([-1.0, 1.0], (K, N)) * rng.uniform(1, 2, (K, N)), eb).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    bound = (K + 8) * U * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)) + 2.0 ** -149
    for ta, tb in ((0, 0), (0, 1), (1, 0)):
        got = product(dev, tile, 1, A, B, ta, tb)
        assert (np.abs(got - want) <= bound).all(), (ta, tb, float((np.abs(got - want) / bound).max()))


@pytest.mark.gpu
@pytest.mark.parametrize("tile", SPLIT_TILES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
def test_values_without_a_split(dev, tile, ta, tb):
    rng = np.random.default_rng(9)
    M, N, K = 150, 139, 77
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    A[3, 5] = np.inf
    A[140, 0] = -np.inf
    A[70, 76] = np.nan
    A[71] = 0.0
    A[71, 9] = np.float32(3.4e38)          # rounds to infinity in bf16
    B[9] = np.clip(B[9], -0.9, 0.9)
    B[20, 130] = np.inf
    got = product(dev, tile, 1, A, B, ta, tb, fill=np.nan)
    with np.errstate(invalid="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf].astype(np.float32))
    fine = np.isfinite(want)
    bound = (K + 8) * U * (np.abs(np.where(np.isfinite(A), A, 0)).astype(np.float64)
                           @ np.abs(np.where(np.isfinite(B), B, 0)).astype(np.float64))
    assert (np.abs(got[fine] - want[fine]) <= bound[fine]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("F,B,T,kernel", [(32, 1, 33, "k_smallgemm_nn_glu"), (64, 2, 70, "k_smallgemm_nn_glu"),
                                          (320, 3, 129, "k_gemm_nn_64x64_k32_glu"),
                                          (1024, 2, 300, "k_xgemm_nn_64x64_k32_glu"),
                                          (1024, 8, 1024, "k_xgemm_nn_128x128_glu")])
def test_swiglu_epilogue_of_every_kernel(trlm, orc, F, B, T, kernel):
    """The gate/up product with the SwiGLU epilogue, through the decoder's
    prefill (whose engine takes the split products), at sizes where the plan
    takes the 32-, the fp32 64-, the split 64- and the 128-wide tile: the last
    position's logits against the oracle's."""
    V, D, H, L = 150, 64, 2, 1
    assert trlm.gemm_plan(0, 0, B * T, 2 * F, D, glu_F=F) == (kernel, 1)
    model = orc.Model(V, D, H, L, F)
    params = model.init(1337, 1)
    ids = orc.random_tokens(B * T, V, 4242, 13, hi_exclusive=V)
    hm = trlm.HostModel(V, D, H, L, F, params)
    tr = trlm.Trainer(hm, 1, 8)
    dec = trlm.Decoder(tr, B, T + 1)
    try:
        dec.prefill(ids.reshape(B, T))
        got = dec.logits()
    finally:
        dec.destroy()
        tr.destroy()
        hm.close()
    want = model.forward_logits(params, ids, B, T).reshape(B, T, V)[:, -1]
    assert np.abs(got - want).max() <= 1e-4 * np.abs(want).max()


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K,wg", [(1, 1, 1200, 8), (65, 63, 8190, 48), (127, 2050, 777, 198),
                                      (16 * 64, 16 * 64, 1201, 256), (16 * 64 + 1, 16 * 64, 1201, 17 * 16 * 4),
                                      (1000, 4, 8190, 256), (4097, 200, 64, 260)])
def test_lone_workgroups(dev, M, N, K, ta, tb, wg):
    """The plan's own kernel up to and just beyond one 64x64 workgroup per CU
    (256), with and without split-K: fp32 tiles up to it, split products beyond."""
    dev.current()
    rng = np.random.default_rng(M + 3 * N + 7 * K + ta + 2 * tb)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    dA, lda, dB, ldb = operands(dev, A, B, ta, tb)
    dC = dev.upload(np.full((M, N), 7.0, np.float32))
    try:
        dev.matmul(ta, tb, dA, dB, dC, M, N, K, lda, ldb, N)
        name, splits = dev.last_variant()
        got = dev.download(dC, (M, N))
    finally:
        for p in (dA, dB, dC):
            dev.free(p)
    ran = -(-M // 64) * -(-N // 64) * splits
    assert ran == wg, (name, splits)
    assert name == "k_%s_%s_64x64_k32" % ("gemm" if ran <= 256 else "xgemm", ["nn", "nt", "tn"][2 * ta + tb])
    want = A.astype(np.float64) @ B.astype(np.float64)
    bound = (K + 8) * U * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))
    assert (np.abs(got - want) <= bound).all(), (name, float((np.abs(got - want) / bound).max()))
