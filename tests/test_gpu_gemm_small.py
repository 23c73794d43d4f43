"""The small-product GEMMs (gemm_small.hip, k_smallgemm_*): one 32x32 tile
of C per workgroup, k shared out over its four waves.

Each layout, aligned and not, at the edges of its tile and of its 32-deep
blocks (waves without a block, a partial last block), with every epilogue
term, componentwise within (K + 8) 2^-24 sum |a||b| plus the terms' own
rounding; NaN in the rows' padding never reaches C.  Then through the
trainer: RoPE, SwiGLU and the column sums against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.fixture(scope="module")
def dev(trlm):
    d = trlm.Device()
    yield d
    d.close()


def stored(x, trans, pad):
    x = x.T if trans else x
    ld = (x.shape[1] + 3) // 4 * 4 if pad else x.shape[1] + (2 if x.shape[1] % 2 else 1)   # odd: unaligned
    out = np.full((x.shape[0], ld), np.nan, np.float32)
    out[:, :x.shape[1]] = x
    return out


@pytest.mark.parametrize("pad", [True, False])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (3, 70, 31), (32, 32, 32), (33, 31, 33), (65, 97, 127), (64, 160, 128),
                                   (31, 40, 129), (130, 66, 250), (256, 512, 97), (40, 33, 768)])
def test_edges_and_epilogue(dev, M, N, K, ta, tb, pad):
    rng = np.random.default_rng(M + 3 * N + 7 * K + ta + 2 * tb)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    C0, R = [rng.standard_normal((M, N)).astype(np.float32) for _ in range(2)]
    bias = rng.standard_normal(N).astype(np.float32)
    As, Bs = stored(A, ta, pad), stored(B, tb, pad)
    dA, dB, dC, dR, db = [dev.upload(x) for x in (As, Bs, C0, R, bias)]
    try:
        dev.matmul(ta, tb, dA, dB, dC, M, N, K, As.shape[1], Bs.shape[1], N, alpha=0.5, beta=2.0, bias=db, resid=dR,
                   ldr=N)
        name, splits = dev.last_variant()
        got = dev.download(dC, (M, N))
    finally:
        for p in (dA, dB, dC, dR, db):
            dev.free(p)
    assert (name, splits) == ("k_smallgemm_" + ["nn", "nt", "tn"][2 * ta + tb] + ("" if pad else "_u"), 1)
    prod = 0.5 * (A.astype(np.float64) @ B.astype(np.float64))
    want = R + ((prod + 2.0 * C0) + bias)
    mag = 0.5 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))
    bound = (K + 8) * U * mag + 4 * U * (mag + 2 * np.abs(C0) + np.abs(bias) + np.abs(R))
    assert (np.abs(got - want) <= bound).all(), (name, float((np.abs(got - want) / bound).max()))


@pytest.mark.parametrize("D,H,F,B,T", [(32, 2, 32, 1, 5), (96, 3, 96, 3, 41), (128, 2, 160, 1, 128)])
def test_through_the_trainer(trlm, orc, D, H, F, B, T):
    """Forward, loss and every gradient of a model whose layer products are
    all small (RoPE, SwiGLU with F a multiple of 32, bias gradients)."""
    V, L = 70, 2
    assert trlm.gemm_plan(0, 0, B * T, 2 * F, D, fp32=True, glu_F=F) == ("k_smallgemm_nn_glu", 1)
    model = orc.Model(V, D, H, L, F)
    params = model.init(1337, 1)
    toks = orc.random_tokens(3000, V)
    ids, tgt = orc.sample_batch(toks, T, B, 2026)
    want_loss, want_g, _ = model.forward_backward(params, ids, tgt, B, T)
    hm = trlm.HostModel(V, D, H, L, F, params)
    tr = trlm.Trainer(hm, B, T)
    try:
        loss = tr.forward_backward(ids, tgt)
        g = tr.grads()
    finally:
        tr.destroy()
        hm.close()
    assert abs(loss - want_loss) <= 1e-4 * abs(want_loss)
    for gi, wi in zip(model.split(g), model.split(want_g)):
        assert np.abs(gi - wi).max() <= 1e-4 * np.abs(wi).max() + 1e-12
