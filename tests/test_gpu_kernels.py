"""Kernel-level parity of the HIP hot path against the oracle / f64 restatements (GPU).

Tolerances: f32 contractions and reductions 1e-4 norm-wise relative error
(max|a-b| / max|b|); f16 outputs within one f16 ulp of the f64-accumulated value rounded at the same
points; index/tie work bit-exact.
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from anneal_amd import _lib as L
from anneal_amd.backend import Trainer
from anneal_amd.executor import Buffer, ExecItem, Executor

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(99)


def q16(a):
    return np.asarray(a, np.float32).astype(np.float16).astype(np.float32)


def store_operand(X, trans):
    return np.ascontiguousarray(X.T if trans else X)


GEMM_CASES = [
    # dtype, ta, tb, M, N, K, tile
    (L.AH_F32, 0, 0, 64, 128, 784, 0), (L.AH_F32, 0, 1, 64, 128, 10, 0), (L.AH_F32, 1, 1, 10, 128, 64, 0),
    (L.AH_F32, 1, 0, 70, 33, 37, 64), (L.AH_F32, 0, 0, 300, 260, 130, 128), (L.AH_F32, 1, 1, 256, 256, 96, 256),
    (L.AH_F16, 0, 0, 256, 256, 256, 0), (L.AH_F16, 0, 1, 130, 200, 72, 64), (L.AH_F16, 1, 1, 96, 160, 300, 128),
    (L.AH_F16, 1, 0, 512, 512, 128, 256), (L.AH_F16, 0, 0, 33, 17, 24, 64),
]


@pytest.mark.parametrize("case", GEMM_CASES, ids=lambda c: "dt%d_ta%d_tb%d_%dx%dx%d_t%d" % c)
def test_gemm_store_and_bias_relu(dev, case):
    dt, ta, tb, M, N, K, tile = case
    A = RNG.standard_normal((M, K)).astype(np.float32)
    B = RNG.standard_normal((N, K)).astype(np.float32)
    bias = RNG.standard_normal(N).astype(np.float32)
    if dt == L.AH_F16:
        A, B, bias = q16(A), q16(B), q16(bias)
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    As, Bs = store_operand(A, ta), store_operand(B, tb)
    npdt = np.float16 if dt == L.AH_F16 else np.float32
    dA, dB = dev.buffer(As.astype(npdt), dt), dev.buffer(Bs.astype(npdt), dt)
    dbias = dev.buffer(bias.astype(npdt), dt)
    dC = dev.buffer(M * N, dt)
    common = dict(dtype=dt, ta=ta, tb=tb, M=M, N=N, K=K, A=dA, B=dB, lda=As.shape[1], ldb=Bs.shape[1], C_out=dC,
                  ldc=N, tile=tile)
    dev.gemm(epi=L.EPI_STORE, scale=0.5, **common)
    C = dC.read().astype(np.float32).reshape(M, N)
    if dt == L.AH_F32:
        assert O.relerr(C, 0.5 * ref) < 1e-5
    else:
        np.testing.assert_allclose(C, q16(0.5 * ref), rtol=2e-3, atol=2e-3 * np.abs(ref).max())
    dev.gemm(epi=L.EPI_BIAS_RELU, bias=dbias, **common)
    H = dC.read().astype(np.float32).reshape(M, N)
    if dt == L.AH_F32:
        z = ref + bias
        assert O.relerr(H, np.maximum(z, 0)) < 1e-5
    else:
        z = q16(q16(ref) + bias)
        np.testing.assert_allclose(H, np.maximum(z, 0), rtol=2e-3, atol=2e-3 * np.abs(z).max())
    dead = np.signbit(H) & (H == 0)
    assert np.array_equal(dead, z < 0), "ReLU tag (-0 for z<0) mismatch"
    for b in (dA, dB, dbias, dC):
        b.free()


@pytest.mark.parametrize("dt", [L.AH_F32, L.AH_F16])
def test_gemm_mask_colsum_and_sgd(dev, dt):
    M, N, K = 192, 160, 96
    npdt = np.float16 if dt == L.AH_F16 else np.float32
    A = RNG.standard_normal((M, K)).astype(np.float32)
    Bm = RNG.standard_normal((K, N)).astype(np.float32)       # stored [K,N] (tb = 1)
    if dt == L.AH_F16:
        A, Bm = q16(A), q16(Bm)
    Hact = RNG.standard_normal((M, N)).astype(np.float32)
    Hact = np.where(Hact < 0, np.float32(-0.0), Hact).astype(npdt)
    ref = A.astype(np.float64) @ Bm.astype(np.float64)
    masked = np.where(np.signbit(Hact.astype(np.float32)) & (Hact == 0), 0.0, 2.0 * ref)
    dA, dB, dH = dev.buffer(A.astype(npdt), dt), dev.buffer(Bm.astype(npdt), dt), dev.buffer(Hact, dt)
    dC = dev.buffer(M * N, dt)
    cs = dev.buffer(np.zeros(N, np.float32), L.AH_F32)
    dev.gemm(dtype=dt, epi=L.EPI_MASK, ta=0, tb=1, M=M, N=N, K=K, A=dA, B=dB, lda=K, ldb=N, C_out=dC, ldc=N,
             aux=dH, ldaux=N, scale=2.0, colsum=cs)
    C = dC.read().astype(np.float32).reshape(M, N)
    tol = 1e-5 if dt == L.AH_F32 else 2e-3
    assert O.relerr(C, masked) < tol
    assert O.relerr(cs.read(), masked.sum(0)) < 1e-4
    # SGD epilogue: W -= lr * (scale * A^T-contraction); dW[n,k] = sum_m G[m,n] X[m,k]
    G, X = A, RNG.standard_normal((M, 48)).astype(np.float32)
    if dt == L.AH_F16:
        X = q16(X)
    W = RNG.standard_normal((K, 48)).astype(np.float32)
    dG, dX = dev.buffer(G.astype(npdt), dt), dev.buffer(X.astype(npdt), dt)
    dW, dg = dev.buffer(W, L.AH_F32), dev.buffer(K * 48, L.AH_F32)
    dW16 = dev.buffer(K * 48, L.AH_F16)
    dev.gemm(dtype=dt, epi=L.EPI_SGD, ta=1, tb=1, M=K, N=48, K=M, A=dG, B=dX, lda=K, ldb=48, ldc=48, scale=0.25,
             W32=dW, W16=dW16, lr=0.1, gout=dg)
    gref = 0.25 * (G.astype(np.float64).T @ X.astype(np.float64))
    assert O.relerr(dg.read().reshape(K, 48), gref) < (1e-5 if dt == L.AH_F32 else 1e-4)
    Wn = dW.read().reshape(K, 48)
    assert O.relerr(Wn - W, -0.1 * gref) < 1e-4
    np.testing.assert_array_equal(dW16.read(), Wn.astype(np.float16).ravel())


def test_gemm_mse_epilogue(dev):
    M, N, K = 128, 96, 64
    A, B = q16(RNG.standard_normal((M, K))), q16(RNG.standard_normal((N, K)) * 0.2)
    bias, T = q16(RNG.standard_normal(N) * 0.1), q16(RNG.standard_normal((M, N)))
    dA, dB = dev.buffer(A.astype(np.float16), L.AH_F16), dev.buffer(B.astype(np.float16), L.AH_F16)
    db, dT = dev.buffer(bias.astype(np.float16), L.AH_F16), dev.buffer(T.astype(np.float16), L.AH_F16)
    dD = dev.buffer(M * N, L.AH_F16)
    cs, la = dev.buffer(np.zeros(N, np.float32), L.AH_F32), dev.buffer(np.zeros(1, np.float32), L.AH_F32)
    dev.gemm(dtype=L.AH_F16, epi=L.EPI_MSE, ta=0, tb=0, M=M, N=N, K=K, A=dA, B=dB, lda=K, ldb=K, C_out=dD, ldc=N,
             bias=db, aux=dT, ldaux=N, colsum=cs, lossacc=la)
    P = q16(q16(A.astype(np.float64) @ B.astype(np.float64).T) + bias)
    d = q16(P - T)
    got = dD.read().astype(np.float32).reshape(M, N)
    assert np.mean(got == d) > 0.99 and O.relerr(got, d) < 2e-3
    assert O.relerr(cs.read(), d.astype(np.float64).sum(0)) < 1e-3
    assert abs(la.read()[0] - ((P - T).astype(np.float64) ** 2).sum()) < 1e-3 * ((P - T) ** 2).sum()


@pytest.mark.parametrize("B,C", [(64, 10), (7, 512), (4096, 512), (3, 1)])
def test_softmax_ce_kernel(dev, B, C):
    z = (RNG.standard_normal((B, C)) * 3).astype(np.float32)
    z[0, : min(C, 3)] = z[0].max() + 1.0          # a tied maximum
    lab = RNG.integers(0, C, B).astype(np.int32)
    wl, wdz = O.softmax_ce(z, lab)
    dz_, dl_, dd, dloss = dev.buffer(z), dev.buffer(lab, L.AH_I32), dev.buffer(B * C), dev.buffer(1)
    dev.softmax_ce(dz_, dl_, B, C, dd, dloss)
    assert O.relerr(dd.read().reshape(B, C), wdz) < 1e-5
    assert abs(dloss.read()[0] - wl) <= 1e-5 * max(1.0, abs(wl))


@pytest.mark.parametrize("B,C", [(1, 2), (255, 64), (257, 65), (300, 128), (4097, 129), (8200, 256), (5, 513), (9, 1024),
                                 (1, 1025), (700, 2048), (3, 2049), (513, 4097), (2, 8192), (3, 8193)])
def test_softmax_ce_edges(dev, B, C):
    """Edges of the rows' kernels (a wave a row to 1024 logits, a workgroup to 8192, then a wave from memory; several rows
    a wave or workgroup), called twice (the second call reads the workspace the first one left), and the item's row terms.
    dz and the loss are sums of up to C terms in f32 against float64: at most 12 tree levels and 32 terms a lane, each
    rounding 2^-24, over an exponential good to a few ulp: 1e-5 of the largest leaves a factor of 3."""
    rng = np.random.default_rng(B * 8209 + C)
    z = (rng.standard_normal((B, C)) * 3).astype(np.float32)
    z[B // 2, : min(C, 3)] = z[B // 2].max() + 1.0   # a tied maximum
    lab = rng.integers(0, C, B).astype(np.int32)
    lab[0] = C                                       # no such column: no term, no gradient
    x = z.astype(np.float64)
    m = x.max(1, keepdims=True)
    e = np.exp(x - m)
    logp = x - m - np.log(e.sum(1, keepdims=True))
    inside = lab < C
    rows = np.where(inside, logp[np.arange(B), np.minimum(lab, C - 1)], 0.0)
    P = e / e.sum(1, keepdims=True)
    d = P.copy()
    d[np.arange(B)[inside], lab[inside]] -= 1.0      # the max's own gradient is the sum of the others', zero up to rounding
    d[~inside] = 0.0
    dz_, dl_, dd, dloss = dev.buffer(z), dev.buffer(lab, L.AH_I32), dev.buffer(B * C), dev.buffer(1)
    for _ in range(2):
        dev.softmax_ce(dz_, dl_, B, C, dd, dloss)
        got = dd.read().reshape(B, C).astype(np.float64) * B
        assert np.abs(got - d).max() <= 1e-5
        want = -rows.sum() / B
        assert abs(dloss.read()[0] - want) <= 1e-5 * max(1.0, abs(want))
    bufs = [Buffer(12, B * C, [B, C]), Buffer(11, B * C, [B, C]), Buffer(2, B, [B], L.AH_I32), Buffer(13, B, [B])]
    out = Executor(dev).run([ExecItem(f"tmpl:softmax_ce;B={B};C={C}", bufs)], {11: z.ravel(), 2: lab.view(np.float32)})
    assert np.array_equal(out[12].view(np.uint32), dd.read().view(np.uint32).ravel())
    assert np.abs(out[13] - rows).max() <= 1e-5 * max(1.0, np.abs(rows).max())


def test_softmax_ce_long_rows(dev):
    """Rows of more than 8192 logits, more of them than workgroups times waves (each wave then takes several): against the
    item, which computes the same rows one to a wave and no loss (the same bits, and the loss within 1e-5 of the rows' sum);
    and the call takes no longer than the item's kernel by more than a quarter (twice as long with 512 workgroups)."""
    B, C_ = 8200, 8200
    z, lab = RNG.standard_normal((B, C_), dtype=np.float32), RNG.integers(0, C_, B).astype(np.int32)
    bz, bl, bd, bs = dev.buffer(z), dev.buffer(lab, L.AH_I32), dev.buffer(B * C_), dev.buffer(1)
    bd2, br = dev.buffer(B * C_), dev.buffer(B)
    k, one = C.c_void_p(), (C.c_uint32 * 3)(1, 1, 1)
    L.check(dev.lib.ah_module_get(dev.h, f"tmpl:softmax_ce;B={B};C={C_}".encode(), b"kernel", C.byref(k)))
    p = (C.c_void_p * 4)(bd2.ptr, bz.ptr, bl.ptr, br.ptr)

    def ms(call):
        best = 1e9
        for _ in range(5):
            dev.timer_start()
            call()
            best = min(best, dev.timer_stop())
        return best

    item = ms(lambda: L.check(dev.lib.ah_launch(dev.h, k, one, one, p, 4, None, 0)))
    call = ms(lambda: dev.softmax_ce(bz, bl, B, C_, bd, bs))
    assert np.array_equal(bd.read().view(np.uint32), bd2.read().view(np.uint32))
    want = -br.read().astype(np.float64).sum() / B
    assert abs(bs.read()[0] - want) <= 1e-5 * abs(want)
    for b in (bz, bl, bd, bs, bd2, br):
        b.free()
    assert call < 1.25 * item, (call, item)


# The column-strip kernel that holds X on chip, in one part and several (test_chain_three_kernels has the shapes it leaves)
@pytest.mark.parametrize("R,Cc,grow", [(64, 32, False), (257, 260, False), (1024, 512, False), (4096, 256, False),
                                       (8192, 64, False), (8192, 528, False), (4096, 256, True), (8192, 64, True)])
def test_chain_kernel_vs_oracle(dev, R, Cc, grow):
    """grow: half the columns jump by +50 in their second half of rows, far above the maximum of the
    rows the strip kernel's threads take their provisional max from (it then re-bases its sums)."""
    X = RNG.standard_normal((R, Cc)).astype(np.float32)
    if grow:
        X[R // 2:, : Cc // 2] += 50.0
    X[5, :] = X.max() + 0.5                             # every row of Y gets a tie candidate
    X[9, :] = X[5, :]
    g = (1 + 0.02 * RNG.standard_normal(Cc)).astype(np.float32)
    wl, wdX, wdg = O.chain_step(X, g)
    dXb, dgb, dX, dg, dl = dev.buffer(X), dev.buffer(g), dev.buffer(R * Cc), dev.buffer(Cc), dev.buffer(1)
    dev.chain_step(dXb, dgb, R, Cc, dX, dg, dl)
    # Each column's max elements carry the max-path tie share, zero in exact arithmetic and a rounding
    # residue in any f32 evaluation (it depends on how sum e was rounded): those are judged against the
    # float64 closed form, no further from it than the oracle is (plus 1e-4); the rest against the oracle.
    from oracle_np import chain_dX_f64
    got = dX.read().reshape(R, Cc)
    exact = chain_dX_f64(X, g)
    mask = X == X.max(0, keepdims=True)
    den = np.max(np.abs(wdX))
    assert np.max(np.abs(got - wdX)[~mask]) / den < 1e-4
    assert np.max(np.abs(got - exact)[mask]) / den <= np.max(np.abs(wdX - exact)[mask]) / den + 1e-4
    assert O.relerr(dg.read(), wdg) < 1e-5
    assert abs(dl.read()[0] - wl) < 1e-5 * abs(wl)
    for b in (dXb, dgb, dX, dg, dl):
        b.free()


# Row counts around the strip kernel's slots (64 rows), parts (4096 rows, or fewer for few columns) and instances; columns
# that end inside a 32-column strip, one strip, more strips than CUs; 16 parts of 40 slots
@pytest.mark.parametrize("R,Cc", [(1, 4), (64, 36), (65, 32), (513, 64), (1025, 100), (2049, 260), (2881, 8200), (3001, 2052),
                                  (4097, 64), (5000, 132), (8192, 96), (9000, 8), (16384, 32), (40960, 4)])
@pytest.mark.parametrize("spin", [-1, 0])
def test_chain_strip_edges(dev, R, Cc, spin):
    """The chain item against the float64 closed form and, bit for bit, against itself with spin = 0: there a workgroup
    whose strip's other parts have not arrived takes their statistics from X itself. -FLT_MAX entries (a mask) and a
    column of them, where every element ties, and a jump far above the first rows."""
    rng = np.random.default_rng(R + Cc)
    X = rng.standard_normal((R, Cc)).astype(np.float32)
    X[:, 1] = np.float32(-3.4028234663852886e38) if R > 1 else X[:, 1]
    X[: R // 3, 2] = np.float32(-3.4028234663852886e38)
    X[R // 2:, 3] += 100.0
    g = (1 + 0.02 * rng.standard_normal(Cc)).astype(np.float32)
    ex = Executor(dev)

    def run(spin):
        bufs = [Buffer(10, R * Cc, [R, Cc]), Buffer(1, R * Cc, [R, Cc]), Buffer(2, Cc, [Cc]), Buffer(11, Cc, [Cc]), Buffer(12, 1, [1])]
        key = f"tmpl:chain;R={R};Cc={Cc}" + (f";spin={spin}" if spin >= 0 else "")
        return ex.run([ExecItem(key, bufs)], {1: X.ravel(), 2: g})

    out = run(spin)
    x = X.astype(np.float64)
    m = x.max(0)
    e = np.exp(x - m)
    S = e / e.sum(0)
    T = np.sqrt((S * S).mean(0) + 1e-6)
    dg = 1 / T
    gS = g / T - S * (g * S.sum(0) / (R * T**3))
    dX = S * (gS - (gS * S).sum(0))
    got = out[10].reshape(R, Cc)
    # An f32 evaluation forms dX = S (gS - sum gS S) from terms of S g / T that nearly cancel, a few roundings each; at the
    # maxima the tie share adds what is left of g / T - g / T: an ulp of it after each of four roundings.
    assert np.all(np.abs(got - dX) <= 16 * 2.0**-23 * (S * g / T) + 4 * 2.0**-24 * (g / T) * (x == m) + 1e-30)
    assert np.allclose(out[11], dg, rtol=1e-5) and np.allclose(out[12][0], (g * dg).sum(), rtol=1e-5)
    if spin == 0:
        for k, v in run(-1).items():
            np.testing.assert_array_equal(out[k].view(np.uint32), v.view(np.uint32))


@pytest.mark.parametrize("R,Cc,strips", [(8192, 4096, True), (4096, 8192, True), (3000, 8196, True), (16000, 1028, True), (64, 20000, True),
                                         (5000, 4100, False), (7000, 4100, False), (4096, 8196, False), (9000, 3072, False),
                                         (2, 27724, False), (16000, 4096, True)])
def test_chain_route(dev, R, Cc, strips):
    """The strips take what fits on chip in one round of workgroups; a second round of large ones, and few rows of very many
    columns, are the three kernels' (test_chain_three_kernels has their results)."""
    t = Trainer(dev, L.TRAIN_CHAIN, [R, Cc])
    names = t.kernel_names(R)
    t.close()
    assert names == (["chain_resident"] if strips else ["chain_stats", "chain_finalize", "chain_grad"])


# More strips than the counters, one more part than a round holds, a few rows, few and many row chunks; columns that end inside
# a block of 256 and inside a finalize block of 16
@pytest.mark.parametrize("R,Cc", [(46081, 4), (5000, 4100), (4097, 4364), (2, 27724), (33, 33000), (7, 16420)])
def test_chain_three_kernels(dev, R, Cc):
    """Shapes that run chain_stats, chain_finalize and chain_grad, with masked entries (-FLT_MAX and -inf) and ties, against
    the float64 closed form: the bound of test_chain_strip_edges, twice the terms (the op order rounds the factors of dX an
    element at a time)."""
    t = Trainer(dev, L.TRAIN_CHAIN, [R, Cc])
    assert t.kernel_names(R) == ["chain_stats", "chain_finalize", "chain_grad"]
    rng = np.random.default_rng(R + Cc)
    X = rng.standard_normal((R, Cc)).astype(np.float32)
    X[R // 2, ::3] = X[R - 1, ::3]                           # a tie, maybe of the maximum
    X[: R // 2, 1], X[: R // 2, 2] = np.float32(-3.4028234663852886e38), -np.inf
    g = (1 + 0.02 * rng.standard_normal(Cc)).astype(np.float32)
    t.set("X", X)
    t.set("g", g)
    t.step(R)
    got, dg, loss = t.get("dX", R * Cc).reshape(R, Cc), t.get("dg", Cc), t.get("loss", 1)[0]
    t.close()
    x = X.astype(np.float64)
    m = x.max(0)
    S = np.exp(x - m) / np.exp(x - m).sum(0)
    T = np.sqrt((S * S).mean(0) + 1e-6)
    gS = g / T - S * (g * S.sum(0) / (R * T**3))
    dX = S * (gS - (gS * S).sum(0))
    assert np.all(np.abs(got - dX) <= 32 * 2.0**-23 * (S * g / T) + 8 * 2.0**-24 * (g / T) * (x == m) + 1e-30)
    assert np.allclose(dg, 1 / T, rtol=1e-5) and np.allclose(loss, (g / T).sum(), rtol=1e-5)


# One slot (64 rows), a part of 512 rows, several parts, whole strips of one workgroup
@pytest.mark.parametrize("R,Cc", [(1, 4), (64, 36), (1025, 100), (2049, 260), (3001, 2052), (4097, 64), (8192, 96), (9000, 8)])
@pytest.mark.parametrize("spin", [-1, 0])
def test_chain_infinite_entries(dev, R, Cc, spin):
    """Entries of -inf (a mask) leave the chain finite, as exp2(-inf) = 0: a leading block, one row, a third of a column, the
    first row of a thread, all but the last row, and beside -FLT_MAX only; a NaN or +inf makes its own column NaN and the
    loss, no other column. Against the float64 closed form, with the bound of test_chain_strip_edges."""
    rng = np.random.default_rng(R * 3 + Cc)
    X = rng.standard_normal((R, Cc)).astype(np.float32)
    ninf, low = np.float32(-np.inf), np.float32(-3.4028234663852886e38)
    if R > 1:
        X[R // 2, :] = ninf                                  # one row in all columns
        X[:min(512, R - 1), 0] = ninf                        # a whole part where a part has 512 rows
        X[: R // 3, 1] = ninf
        X[:-1, 2] = ninf                                     # the last row alone is left
        X[:, 3] = np.where(np.arange(R) % 3 == 0, low, ninf)  # nothing above -FLT_MAX
    if Cc >= 32:
        X[::64, 5] = ninf                                    # some lanes' first rows
        X[R - 1, 6], X[0, 7] = np.nan, np.inf
    g = (1 + 0.02 * rng.standard_normal(Cc)).astype(np.float32)
    bufs = [Buffer(10, R * Cc, [R, Cc]), Buffer(1, R * Cc, [R, Cc]), Buffer(2, Cc, [Cc]), Buffer(11, Cc, [Cc]), Buffer(12, 1, [1])]
    key = f"tmpl:chain;R={R};Cc={Cc}" + (f";spin={spin}" if spin >= 0 else "")
    out = Executor(dev).run([ExecItem(key, bufs)], {1: X.ravel(), 2: g})
    bad = ~(np.isfinite(X) | (X == ninf)).all(0)
    got, x, g = out[10].reshape(R, Cc), X.astype(np.float64)[:, ~bad], g[~bad]
    m = x.max(0)
    e = np.exp(x - m)
    S = e / e.sum(0)
    T = np.sqrt((S * S).mean(0) + 1e-6)
    dg = 1 / T
    gS = g / T - S * (g * S.sum(0) / (R * T**3))
    dX = S * (gS - (gS * S).sum(0))
    assert np.all(np.abs(got[:, ~bad] - dX) <= 16 * 2.0**-23 * (S * g / T) + 4 * 2.0**-24 * (g / T) * (x == m) + 1e-30)
    assert np.allclose(out[11][~bad], dg, rtol=1e-5)
    if bad.any():
        assert np.isnan(got[:, bad]).all() and np.isnan(out[11][bad]).all() and np.isnan(out[12][0])
    else:
        assert np.allclose(out[12][0], (g * dg).sum(), rtol=1e-5)


@pytest.mark.parametrize("R,Cc", [(1, 4), (64, 36), (1025, 100), (4096, 260), (4097, 64), (8192, 96), (9000, 8)])
@pytest.mark.parametrize("same", ["X", "g", "both"])
def test_chain_in_place(dev, R, Cc, same):
    """dX written over X, dg over g: through both entry points, and through the item's kernel with spin = 0, where a workgroup
    whose strip's other parts have not arrived takes their statistics from X at once. Against the float64 closed form, with
    the bound of test_chain_strip_edges."""
    rng = np.random.default_rng(R + 7 * Cc)
    X, g = rng.standard_normal((R, Cc)).astype(np.float32), (1 + 0.02 * rng.standard_normal(Cc)).astype(np.float32)
    x = X.astype(np.float64)
    m = x.max(0)
    S = np.exp(x - m) / np.exp(x - m).sum(0)
    T = np.sqrt((S * S).mean(0) + 1e-6)
    gS = g / T - S * (g * S.sum(0) / (R * T**3))
    dX = S * (gS - (gS * S).sum(0))
    k = C.c_void_p()
    L.check(dev.lib.ah_module_get(dev.h, f"tmpl:chain;R={R};Cc={Cc};spin=0".encode(), b"kernel", C.byref(k)))
    one = (C.c_uint32 * 3)(1, 1, 1)

    def item(bX, bg, R, Cc, bdX, bdg, bl):
        p = (C.c_void_p * 5)(bdX.ptr, bX.ptr, bg.ptr, bdg.ptr, bl.ptr)
        L.check(dev.lib.ah_launch(dev.h, k, one, one, p, 5, None, 0))

    for call in (dev.chain_step, dev.chain_step_noalloc, item):
        bX, bg, bl = dev.buffer(X), dev.buffer(g), dev.buffer(1)
        bdX = bX if same != "g" else dev.buffer(R * Cc)
        bdg = bg if same != "X" else dev.buffer(Cc)
        call(bX, bg, R, Cc, bdX, bdg, bl)
        dev.sync()
        got = bdX.read().reshape(R, Cc)
        assert np.all(np.abs(got - dX) <= 16 * 2.0**-23 * (S * g / T) + 4 * 2.0**-24 * (g / T) * (x == m) + 1e-30)
        assert np.allclose(bdg.read(), 1 / T, rtol=1e-5) and np.allclose(bl.read()[0], (g / T).sum(), rtol=1e-5)
        for b in {id(b): b for b in (bX, bg, bl, bdX, bdg)}.values():
            b.free()


F16_VARIANTS = list(range(1, 40))   # every gemm16 variant (gemm16_kernel.h Var<V>; 32-39 use 16x16x32 MFMAs)
KGROUP_VARIANTS = (10, 11, 15, 25, 28, 31, 35, 36, 37, 38)   # variants that add two k-halves
VARIANT_SHAPES = [
    # ta, tb, M, N, K: full tiles, ragged edges (scalar epilogue), short K, both layouts
    (0, 0, 512, 512, 192), (0, 1, 520, 300, 128), (1, 1, 264, 520, 64), (1, 0, 256, 256, 320),
    (0, 0, 384, 640, 512), (1, 1, 264, 256, 256),      # K in whole stage pairs: the k-group variants run
]


@pytest.mark.parametrize("variant", F16_VARIANTS)
@pytest.mark.parametrize("shape", VARIANT_SHAPES, ids=lambda s: "ta%d_tb%d_%dx%dx%d" % s)
def test_gemm16_variants_store_mask_sgd(dev, variant, shape):
    """Every f16 kernel variant (tile, wave layout, fetch mode) against an f64 contraction of the
    same f16 operands, through the STORE, MASK+colsum and SGD epilogues."""
    ta, tb, M, N, K = shape
    A = q16(RNG.standard_normal((M, K)))
    B = q16(RNG.standard_normal((N, K)))
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    As, Bs = store_operand(A, ta), store_operand(B, tb)
    dA, dB = dev.buffer(As.astype(np.float16), L.AH_F16), dev.buffer(Bs.astype(np.float16), L.AH_F16)
    dC = dev.buffer(M * N, L.AH_F16)
    common = dict(dtype=L.AH_F16, ta=ta, tb=tb, M=M, N=N, K=K, A=dA, B=dB, lda=As.shape[1], ldb=Bs.shape[1],
                  ldc=N, variant=variant)
    dev.gemm(epi=L.EPI_STORE, scale=1.0, C_out=dC, **common)
    C = dC.read().astype(np.float32).reshape(M, N)
    np.testing.assert_allclose(C, q16(ref), rtol=2e-3, atol=2e-3 * np.abs(ref).max())
    Hact = RNG.standard_normal((M, N)).astype(np.float32)
    Hact = np.where(Hact < 0, np.float32(-0.0), Hact).astype(np.float16)
    dH = dev.buffer(Hact, L.AH_F16)
    cs = dev.buffer(np.zeros(N, np.float32), L.AH_F32)
    dev.gemm(epi=L.EPI_MASK, scale=0.5, C_out=dC, aux=dH, ldaux=N, colsum=cs, **common)
    masked = np.where(np.signbit(Hact.astype(np.float32)) & (Hact == 0), 0.0, 0.5 * ref)
    assert O.relerr(dC.read().astype(np.float32).reshape(M, N), masked) < 2e-3
    assert O.relerr(cs.read(), masked.sum(0)) < 1e-4
    W = RNG.standard_normal((M, N)).astype(np.float32)
    dW, dg, dW16 = dev.buffer(W, L.AH_F32), dev.buffer(M * N, L.AH_F32), dev.buffer(M * N, L.AH_F16)
    dev.gemm(epi=L.EPI_SGD, scale=0.25, W32=dW, W16=dW16, lr=0.1, gout=dg, **common)
    assert O.relerr(dg.read().reshape(M, N), 0.25 * ref) < 1e-5
    Wn = dW.read().reshape(M, N)
    assert O.relerr(Wn - W, -0.025 * ref) < 1e-4
    np.testing.assert_array_equal(dW16.read(), Wn.astype(np.float16).ravel())
    for b in (dA, dB, dC, dH, cs, dW, dg, dW16):
        b.free()


@pytest.mark.parametrize("shape", [(0, 0, 512, 384, 256), (1, 1, 256, 512, 192), (0, 1, 300, 260, 128)],
                         ids=lambda s: "ta%d_tb%d_%dx%dx%d" % s)
def test_gemm16_variants_bit_identical_and_tune(dev, shape):
    """Variants without k-groups accumulate each output over k in the same order, so their results are
    bit-identical; k-group variants add two k-halves (f32 rounding differs, 1e-6 relative). The tuner
    picks one variant, caches it, and variant-0 launches reproduce that variant's result."""
    ta, tb, M, N, K = shape
    A, B = q16(RNG.standard_normal((M, K))), q16(RNG.standard_normal((N, K)))
    As, Bs = store_operand(A, ta), store_operand(B, tb)
    dA, dB = dev.buffer(As.astype(np.float16), L.AH_F16), dev.buffer(Bs.astype(np.float16), L.AH_F16)
    dC = dev.buffer(M * N, L.AH_F32)
    dW = dev.buffer(np.zeros(M * N, np.float32))
    common = dict(dtype=L.AH_F16, ta=ta, tb=tb, M=M, N=N, K=K, A=dA, B=dB, lda=As.shape[1], ldb=Bs.shape[1], ldc=N)
    outs = []
    for v in F16_VARIANTS:
        dW.write(np.zeros(M * N, np.float32))
        dev.gemm(epi=L.EPI_SGD, scale=1.0, W32=dW, lr=-1.0, variant=v, **common)   # W = 0 + acc, exact f32
        outs.append(dW.read())
    for v, o in zip(F16_VARIANTS, outs):
        if v in KGROUP_VARIANTS:
            assert O.relerr(o, outs[0]) < 1e-6, v      # two k-halves added: different f32 rounding
        else:
            np.testing.assert_array_equal(o.view(np.uint32), outs[0].view(np.uint32), err_msg=f"variant {v}")
    best, us = dev.gemm_tune(iterations=2, epi=L.EPI_SGD, scale=1.0, W32=dW, lr=-1.0, **common)
    assert best in F16_VARIANTS and us > 0
    dW.write(np.zeros(M * N, np.float32))
    dev.gemm(epi=L.EPI_SGD, scale=1.0, W32=dW, lr=-1.0, **common)
    np.testing.assert_array_equal(dW.read().view(np.uint32), outs[best - 1].view(np.uint32))
    for b in (dA, dB, dC, dW):
        b.free()


@pytest.mark.parametrize("dt", [L.AH_F32, L.AH_F16])
def test_gemm_dot_path_epilogues(dev, dt):
    """Few outputs with a long K (M*N <= 16384, K >= 256, A and B K-contiguous) take the
    wave-per-output path: bias+ReLU, mask+colsum and SGD epilogues against f64."""
    M, N, K = 24, 40, 300
    npdt = np.float16 if dt == L.AH_F16 else np.float32
    A, B = RNG.standard_normal((M, K)).astype(np.float32), RNG.standard_normal((N, K)).astype(np.float32)
    bias = RNG.standard_normal(N).astype(np.float32)
    if dt == L.AH_F16:
        A, B, bias = q16(A), q16(B), q16(bias)
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    dA, dB, db = dev.buffer(A.astype(npdt), dt), dev.buffer(B.astype(npdt), dt), dev.buffer(bias.astype(npdt), dt)
    dC = dev.buffer(M * N, dt)
    common = dict(dtype=dt, ta=0, tb=0, M=M, N=N, K=K, A=dA, B=dB, lda=K, ldb=K, ldc=N)
    dev.gemm(epi=L.EPI_BIAS_RELU, bias=db, C_out=dC, **common)
    H = dC.read().astype(np.float32).reshape(M, N)
    z = ref + bias if dt == L.AH_F32 else q16(q16(ref) + bias)
    tol = 1e-5 if dt == L.AH_F32 else 2e-3
    assert O.relerr(H, np.maximum(z, 0)) < tol
    assert np.array_equal(np.signbit(H) & (H == 0), z < 0)
    Hact = np.where(RNG.standard_normal((M, N)) < 0, np.float32(-0.0), np.float32(1.0)).astype(npdt)
    dH, cs = dev.buffer(Hact, dt), dev.buffer(np.zeros(N, np.float32))
    dev.gemm(epi=L.EPI_MASK, scale=0.5, aux=dH, ldaux=N, colsum=cs, C_out=dC, **common)
    masked = np.where(np.signbit(Hact.astype(np.float32)), 0.0, 0.5 * ref)
    assert O.relerr(dC.read().astype(np.float32).reshape(M, N), masked) < tol
    assert O.relerr(cs.read(), masked.sum(0)) < 1e-4
    W = RNG.standard_normal((M, N)).astype(np.float32)
    dW, dg = dev.buffer(W), dev.buffer(M * N)
    dev.gemm(epi=L.EPI_SGD, scale=0.25, W32=dW, lr=0.1, gout=dg, **common)
    assert O.relerr(dg.read().reshape(M, N), 0.25 * ref) < 1e-5
    assert O.relerr(dW.read().reshape(M, N) - W, -0.025 * ref) < 1e-4
    for b in (dA, dB, db, dC, dH, cs, dW, dg):
        b.free()


def test_gemm_tune_disk_cache(dev, tmp_path):
    """Tuned choices survive a save/load through the disk cache, and a malformed file is rejected."""
    M, N, K = 256, 256, 128
    A, B = q16(RNG.standard_normal((M, K))), q16(RNG.standard_normal((N, K)))
    dA, dB = dev.buffer(A.astype(np.float16), L.AH_F16), dev.buffer(B.astype(np.float16), L.AH_F16)
    dC = dev.buffer(M * N, L.AH_F16)
    best, _ = dev.gemm_tune(iterations=1, dtype=L.AH_F16, epi=L.EPI_STORE, ta=0, tb=0, M=M, N=N, K=K, A=dA, B=dB,
                            lda=K, ldb=K, C_out=dC, ldc=N)
    path = tmp_path / "tune.txt"
    dev.gemm_tune_cache(str(path), True)
    lines = path.read_text().splitlines()
    assert lines[0].startswith("# anneal_hip gemm variants v1")
    assert f"1/0/0/{M}/{N}/{K} {best}" in lines
    dev.gemm_tune_cache(str(path), False)
    bad = tmp_path / "bad.txt"
    bad.write_text(lines[0] + "\n1/0/0/8/8/8 99\n")
    with pytest.raises(L.AnnealHipError, match="bad line"):
        dev.gemm_tune_cache(str(bad), False)
    for b in (dA, dB, dC):
        b.free()


@pytest.mark.parametrize("splits", [0, 1, 2, 4, 8, 16])
@pytest.mark.parametrize("epi", ["store", "bias_relu", "mask", "grad"])
def test_gemm_f32_split_k(dev, epi, splits):
    """The f32 tiled kernel with K split across workgroups (splits=s fixes the count, 0 lets the shape
    choose: 4 k-groups x 8 splits here): partials folded in split order by the last split to arrive, so
    every launch gives the same bits, and each launch leaves the tiles' arrival counters at zero for the
    next (checked by a second launch on other inputs)."""
    from anneal_amd.executor import Buffer, ExecItem, Executor
    M, N, K, ta, tb = (256, 512, 2048, 0, 0) if epi != "grad" else (512, 256, 2048, 1, 1)
    key = f"tmpl:gemm;dtype=f32;epi={epi};ta={ta};tb={tb};M={M};N={N};K={K};tile=64;splits={splits}"
    if splits == 0:
        key = f"tmpl:gemm;dtype=f32;epi={epi};ta={ta};tb={tb};M={M};N={N};K={K}"
    bufs = [Buffer(10, M * N, [M, N], L.AH_F32), Buffer(1, M * K, [K, M] if ta else [M, K], L.AH_F32),
            Buffer(2, N * K, [K, N] if tb else [N, K], L.AH_F32)]
    if epi in ("bias_relu", "mask"):
        bufs.append(Buffer(3, N if epi == "bias_relu" else M * N, [N] if epi == "bias_relu" else [M, N], L.AH_F32))
    ex = Executor(dev)
    prev = None
    for rep in range(2):
        rng = np.random.default_rng(1000 + rep)
        A = rng.standard_normal((M, K)).astype(np.float32)
        B = rng.standard_normal((N, K)).astype(np.float32)
        ins = {1: store_operand(A, ta).ravel(), 2: store_operand(B, tb).ravel()}
        ref = A.astype(np.float64) @ B.astype(np.float64).T
        if epi == "bias_relu":
            bias = rng.standard_normal(N).astype(np.float32)
            ins[3] = bias
            ref = np.maximum(ref + bias, 0)
        elif epi == "mask":
            H = rng.standard_normal((M, N)).astype(np.float32)
            H = np.where(H < 0, np.float32(-0.0), H).astype(np.float32)
            ins[3] = H.ravel()
            ref = np.where(np.signbit(H) & (H == 0), 0.0, ref)
        got = ex.run([ExecItem(key, bufs)], ins)[10].reshape(M, N)
        assert O.relerr(got, ref) < 1e-5, (epi, splits, rep)
        again = ex.run([ExecItem(key, bufs)], ins)[10].reshape(M, N)
        np.testing.assert_array_equal(again.view(np.uint32), got.view(np.uint32))
        assert prev is None or not np.array_equal(prev, got)
        prev = got


def test_gemm_f32_tune_and_cache(dev, tmp_path):
    """The tuner over the f32 kernel's (tile, k-groups, splits) configurations: it returns an index into
    the 58-entry table (38 register-staged, 5 direct-to-LDS, those 5 with K split 2 / 4 / 8 ways), later
    automatic launches of the shape use
    the winner (against float64), and the choice survives the disk cache, where an index past the table
    is rejected."""
    M, N, K = 256, 512, 2048
    A = RNG.standard_normal((M, K)).astype(np.float32)
    B = RNG.standard_normal((N, K)).astype(np.float32)
    dA, dB = dev.buffer(A), dev.buffer(B)
    dC = dev.buffer(M * N, L.AH_F32)
    common = dict(dtype=L.AH_F32, epi=L.EPI_STORE, ta=0, tb=0, M=M, N=N, K=K, A=dA, B=dB, lda=K, ldb=K, C_out=dC,
                  ldc=N)
    best, us = dev.gemm_tune(iterations=2, **common)
    assert 0 <= best < 58 and us > 0
    dev.gemm(**common)
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    assert O.relerr(dC.read().reshape(M, N), ref) < 1e-5
    path = tmp_path / "tune32.txt"
    dev.gemm_tune_cache(str(path), True)
    lines = path.read_text().splitlines()
    assert f"0/0/0/{M}/{N}/{K} {best}" in lines
    dev.gemm_tune_cache(str(path), False)
    bad = tmp_path / "bad32.txt"
    bad.write_text(lines[0] + f"\n0/0/0/{M}/{N}/{K} 58\n")
    with pytest.raises(L.AnnealHipError, match="bad line"):
        dev.gemm_tune_cache(str(bad), False)
    for b in (dA, dB, dC):
        b.free()


# direct-to-LDS f32 configurations (gemm32d.hip): (tile, k per stage, stages)
DMA_CFGS = [(64, 64, 3), (64, 64, 4), (64, 32, 4), (128, 32, 4), (128, 64, 2)]


@pytest.mark.parametrize("shape", [(200, 300, 1024), (36, 20, 128)])
@pytest.mark.parametrize("dma", range(5))
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("epi", ["store", "bias_relu", "mask", "grad"])
def test_gemm_f32_dma_same_bits_as_register_staged(dev, dma, ta, tb, epi, shape):
    """The direct-to-LDS f32 kernel adds K in the order of the register-staged kernel with one k-group
    and no split, so each of its configurations gives the same bits as that kernel at the same tile, for
    every layout and epilogue, on ragged shapes (M, N not multiples of the tile, down to one tile smaller
    than the tile); both against float64.
    The 128-wide configurations take only the store and bias epilogues and run the automatic choice for
    the others, which must then match that choice's bits."""
    from anneal_amd.executor import Buffer, ExecItem, Executor
    tile = DMA_CFGS[dma][0]
    M, N, K = shape
    common = f"tmpl:gemm;dtype=f32;epi={epi};ta={ta};tb={tb};M={M};N={N};K={K}"
    dma_key = common + f";dma={dma}"
    fallback = tile == 128 and epi in ("mask", "grad")
    ref_key = common if fallback else common + f";tile={tile};kg=1;splits=1"
    bufs = [Buffer(10, M * N, [M, N], L.AH_F32), Buffer(1, M * K, [K, M] if ta else [M, K], L.AH_F32),
            Buffer(2, N * K, [K, N] if tb else [N, K], L.AH_F32)]
    rng = np.random.default_rng(31 + dma)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((N, K)).astype(np.float32)
    ins = {1: store_operand(A, ta).ravel(), 2: store_operand(B, tb).ravel()}
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    if epi in ("bias_relu", "mask"):
        bufs.append(Buffer(3, N if epi == "bias_relu" else M * N, [N] if epi == "bias_relu" else [M, N], L.AH_F32))
    if epi == "bias_relu":
        bias = rng.standard_normal(N).astype(np.float32)
        ins[3] = bias
        ref = np.maximum(ref + bias, 0)
    elif epi == "mask":
        H = rng.standard_normal((M, N)).astype(np.float32)
        H = np.where(H < 0, np.float32(-0.0), H).astype(np.float32)
        ins[3] = H.ravel()
        ref = np.where(np.signbit(H) & (H == 0), 0.0, ref)
    elif epi == "grad":
        ref = -ref   # SGD with lr 1 on a zeroed array: the array becomes -g
    ex = Executor(dev)
    got = ex.run([ExecItem(dma_key, bufs)], ins)[10].reshape(M, N)
    want = ex.run([ExecItem(ref_key, bufs)], ins)[10].reshape(M, N)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    if epi == "grad":
        return   # the grad key's scale and sign are the register-staged kernel's, checked by its own tests
    assert O.relerr(got, ref) < 1e-5


@pytest.mark.parametrize("dma,splits", [(0, 2), (2, 4), (1, 8), (3, 2), (4, 4)])
@pytest.mark.parametrize("epi", ["store", "mask", "grad"])
def test_gemm_f32_dma_split_k_same_bits(dev, dma, splits, epi):
    """The direct-to-LDS kernel splitting K across workgroups folds the partials as the register-staged
    kernel does (split order, the last arriver's own from registers), so dma=i with splits=s gives the bits
    of tile=BM with one k-group and s splits; two launches in a row give the same bits and leave the
    arrival counters at zero (a second launch on other inputs differs)."""
    from anneal_amd.executor import Buffer, ExecItem, Executor
    tile = DMA_CFGS[dma][0]
    M, N, K, ta, tb = (256, 192, 2048, 0, 0) if epi == "store" else (192, 256, 2048, 1, 1)
    if epi == "mask":
        ta, tb = 0, 1
    common = f"tmpl:gemm;dtype=f32;epi={epi};ta={ta};tb={tb};M={M};N={N};K={K}"
    fallback = tile == 128 and epi in ("mask", "grad")
    dma_key = common + f";dma={dma};splits={splits}"
    ref_key = common if fallback else common + f";tile={tile};kg=1;splits={splits}"
    bufs = [Buffer(10, M * N, [M, N], L.AH_F32), Buffer(1, M * K, [K, M] if ta else [M, K], L.AH_F32),
            Buffer(2, N * K, [K, N] if tb else [N, K], L.AH_F32)]
    if epi == "mask":
        bufs.append(Buffer(3, M * N, [M, N], L.AH_F32))
    ex = Executor(dev)
    prev = None
    for rep in range(2):
        rng = np.random.default_rng(50 + rep)
        A = rng.standard_normal((M, K)).astype(np.float32)
        B = rng.standard_normal((N, K)).astype(np.float32)
        ins = {1: store_operand(A, ta).ravel(), 2: store_operand(B, tb).ravel()}
        if epi == "mask":
            H = rng.standard_normal((M, N)).astype(np.float32)
            ins[3] = np.where(H < 0, np.float32(-0.0), H).astype(np.float32).ravel()
        got = ex.run([ExecItem(dma_key, bufs)], ins)[10]
        again = ex.run([ExecItem(dma_key, bufs)], ins)[10]
        want = ex.run([ExecItem(ref_key, bufs)], ins)[10]
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
        np.testing.assert_array_equal(again.view(np.uint32), got.view(np.uint32))
        if epi == "store":
            assert O.relerr(got.reshape(M, N), A.astype(np.float64) @ B.astype(np.float64).T) < 1e-5
        assert prev is None or not np.array_equal(prev, got)
        prev = got


def test_gemm_f32_dma_key_checks(dev):
    """dma=i is a configuration index, and it excludes tile / kg."""
    from anneal_amd.executor import Buffer, ExecItem, Executor
    bufs = [Buffer(10, 64 * 64, [64, 64], L.AH_F32), Buffer(1, 64 * 64, [64, 64], L.AH_F32),
            Buffer(2, 64 * 64, [64, 64], L.AH_F32)]
    ins = {1: np.ones(64 * 64, np.float32), 2: np.ones(64 * 64, np.float32)}
    for bad in ("dma=5", "dma=0;tile=64", "dma=1;kg=2"):
        with pytest.raises(L.AnnealHipError, match="dma|kg"):
            Executor(dev).run([ExecItem(f"tmpl:gemm;dtype=f32;epi=store;ta=0;tb=0;M=64;N=64;K=64;{bad}", bufs)], ins)


@pytest.mark.parametrize("cfg", [(64, 0, 4), (64, 4, 2), (128, 2, 8), (128, 0, 16), (64, 1, 3)])
def test_gemm_f32_split_k_ragged(dev, cfg):
    """Split-K on ragged tiles (M, N and K not multiples of the tile or the 32-wide k chunk), with fixed
    or automatic k-groups; splits=3 runs three splits (groups past K load zeros)."""
    from anneal_amd.executor import Buffer, ExecItem, Executor
    tile, kg, splits = cfg
    M, N, K = 200, 300, 1000
    key = f"tmpl:gemm;dtype=f32;epi=bias_relu;ta=1;tb=0;M={M};N={N};K={K};tile={tile};splits={splits}"
    if kg:
        key += f";kg={kg}"
    rng = np.random.default_rng(7)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((N, K)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    bufs = [Buffer(10, M * N, [M, N], L.AH_F32), Buffer(1, M * K, [K, M], L.AH_F32), Buffer(2, N * K, [N, K], L.AH_F32),
            Buffer(3, N, [N], L.AH_F32)]
    got = Executor(dev).run([ExecItem(key, bufs)], {1: store_operand(A, 1).ravel(), 2: B.ravel(), 3: bias})[10]
    ref = np.maximum(A.astype(np.float64) @ B.astype(np.float64).T + bias, 0)
    assert O.relerr(got.reshape(M, N), ref) < 1e-5


# Sizes around the split f16 kernel's edges: a tile and one more row, column or stage; K that ends inside a stage, inside a
# 32-wide k-step, at one row (the weight gradient of one sample); outputs of one tile with K split many ways; 256-wide tiles.
SPLIT_SHAPES = [(0, 0, 1, 64, 64), (0, 0, 3, 70, 2048), (0, 0, 32, 1000, 4104), (0, 0, 65, 129, 520), (0, 0, 200, 257, 72),
                (0, 0, 999, 1000, 2056), (0, 0, 2100, 2056, 1000), (0, 1, 1, 64, 64), (0, 1, 33, 72, 2000), (0, 1, 130, 264, 136),
                (0, 1, 1100, 520, 1000), (0, 1, 2100, 3080, 264), (1, 1, 64, 64, 1), (1, 1, 72, 136, 33), (1, 1, 264, 136, 4100),
                (1, 1, 1000, 520, 77), (1, 1, 2056, 3080, 130)]


@pytest.mark.parametrize("shape", SPLIT_SHAPES, ids=lambda s: "ta%d_tb%d_%dx%dx%d" % s)
def test_gemm16_split_kernel_edges(dev, shape):
    """Every epilogue of the untuned f16 contraction against float64 at sizes that are no multiple of a tile. The f32 sums
    of K products are within (K + 16) * 2^-24 of the sum of their magnitudes; f16 results add a rounding each (2^-11 of the
    value, twice with a bias). Memory past the output stays as it was, and a repeat gives the same bits (the partials of a
    split K are added in split order)."""
    ta, tb, M, N, K = shape
    rng = np.random.default_rng(M + N + K)
    A, B = (q16(rng.standard_normal(s)) for s in ((M, K), (N, K)))
    bias, aux, W = q16(rng.standard_normal(N)), q16(rng.standard_normal((M, N))), rng.standard_normal((M, N)).astype(np.float32)
    aux = np.where(aux < 0, np.float32(-0.0), aux)
    ref, mag = A.astype(np.float64) @ B.astype(np.float64).T, np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64).T
    acc = (K + 16) * 2.0**-24 * mag
    half = lambda v: v.astype(np.float16)   # noqa: E731
    As, Bs = store_operand(A, ta), store_operand(B, tb)
    pad = 64
    bufs = dict(A=dev.buffer(half(As), L.AH_F16), B=dev.buffer(half(Bs), L.AH_F16))
    dC = dev.buffer(np.full(M * N + pad, 7, np.float16), L.AH_F16)
    dbias, daux = dev.buffer(half(bias), L.AH_F16), dev.buffer(half(aux), L.AH_F16)
    kw = dict(dtype=L.AH_F16, ta=ta, tb=tb, M=M, N=N, K=K, lda=As.shape[1], ldb=Bs.shape[1], ldc=N, **bufs)

    def f16_out(**e):
        dev.gemm(C_out=dC, **kw, **e)
        one = dC.read()
        dev.gemm(C_out=dC, **kw, **e)
        two = dC.read()
        np.testing.assert_array_equal(one.view(np.uint16), two.view(np.uint16))
        assert np.all(one[M * N:] == 7)
        return one[:M * N].astype(np.float64).reshape(M, N)

    tiny = 2.0**-24   # half the smallest f16 step
    C = f16_out(epi=L.EPI_STORE, scale=0.5)
    assert np.all(np.abs(C - 0.5 * ref) <= 0.5 * acc + 2.0**-11 * np.abs(C) + 2 * tiny)
    z = ref + bias
    C = f16_out(epi=L.EPI_BIAS_RELU, bias=dbias)
    slack = acc + 2.0**-11 * (np.abs(ref) + np.abs(z)) * 1.01 + 4 * tiny
    assert np.all(np.abs(C - np.maximum(z, 0)) <= slack)
    sure = np.abs(z) > slack
    assert np.array_equal((np.signbit(C) & (C == 0))[sure], (z < 0)[sure])
    dead = np.signbit(aux) & (aux == 0)
    C = f16_out(epi=L.EPI_MASK, aux=daux, ldaux=N, scale=1.0)
    assert np.all(np.abs(C - np.where(dead, 0.0, ref)) <= acc + 2.0**-11 * np.abs(C) + 2 * tiny)
    dW, dg, dW16 = dev.buffer(W), dev.buffer(np.full(M * N + pad, 7, np.float32)), dev.buffer(M * N, L.AH_F16)
    dev.gemm(epi=L.EPI_SGD, scale=0.25, lr=0.5, W32=dW, W16=dW16, gout=dg, **kw)
    g, Wn = dg.read(), dW.read().reshape(M, N)
    assert np.all(g[M * N:] == 7)
    g = g[:M * N].reshape(M, N)
    assert np.all(np.abs(g - 0.25 * ref) <= 0.25 * acc + 2.0**-24 * np.abs(g))
    assert np.all(np.abs(Wn - (W - 0.5 * g.astype(np.float64))) <= 2.0**-23 * (np.abs(Wn) + np.abs(g)))
    np.testing.assert_array_equal(dW16.read(), Wn.astype(np.float16).ravel())
    for b in (*bufs.values(), dC, dbias, daux, dW, dg, dW16):
        b.free()


def test_gemm16_split_kernel_unaligned_output(dev):
    """A row stride that 16-byte accesses do not divide (ldc 77) and an operand with a padded stride."""
    M, N, K, ldc, lda = 70, 75, 200, 77, 208
    rng = np.random.default_rng(3)
    A, B = q16(rng.standard_normal((M, lda))), q16(rng.standard_normal((N, K)))
    dA, dB = dev.buffer(A.astype(np.float16), L.AH_F16), dev.buffer(B.astype(np.float16), L.AH_F16)
    dC = dev.buffer(np.full(M * ldc, 7, np.float16), L.AH_F16)
    dev.gemm(dtype=L.AH_F16, epi=L.EPI_STORE, ta=0, tb=0, M=M, N=N, K=K, A=dA, B=dB, lda=lda, ldb=K, C_out=dC, ldc=ldc)
    C = dC.read().astype(np.float64).reshape(M, ldc)
    ref = A[:, :K].astype(np.float64) @ B.astype(np.float64).T
    assert np.all(np.abs(C[:, :N] - ref) <= 2.0**-11 * np.abs(ref) + 1e-3) and np.all(C[:, N:] == 7)
    for b in (dA, dB, dC):
        b.free()


def gemm16_bits(dev, M, N, K, ta=0, tb=0, variant=0, rows=None, store=False):
    """The f32 bits of the sums (an SGD step of 1 from zero weights) on fixed operands, or of the first `rows` rows of A; with
    store, the f16 bits of a scaled store instead."""
    rng = np.random.default_rng(M * 31 + N * 7 + K)
    As, Bs = store_operand(q16(rng.standard_normal((M, K))), ta), store_operand(q16(rng.standard_normal((N, K))), tb)
    dA, dB, dW = dev.buffer(As.astype(np.float16), L.AH_F16), dev.buffer(Bs.astype(np.float16), L.AH_F16), dev.buffer(np.zeros(M * N, np.float32))
    m = rows or M
    if store:
        dC = dev.buffer(M * N, L.AH_F16)
        dev.gemm(dtype=L.AH_F16, epi=L.EPI_STORE, ta=ta, tb=tb, M=m, N=N, K=K, A=dA, B=dB, lda=As.shape[1], ldb=Bs.shape[1], ldc=N,
                 scale=1.0 / 3, C_out=dC, variant=variant)
        out = dC.read().view(np.uint16).reshape(M, N)[:m].copy()
        for b in (dA, dB, dW, dC):
            b.free()
        return out
    dev.gemm(dtype=L.AH_F16, epi=L.EPI_SGD, ta=ta, tb=tb, M=m, N=N, K=K, A=dA, B=dB, lda=As.shape[1], ldb=Bs.shape[1], ldc=N,
             scale=1.0, W32=dW, lr=-1.0, variant=variant)
    out = dW.read().view(np.uint32).reshape(M, N)[:m].copy()
    for b in (dA, dB, dW):
        b.free()
    return out


@pytest.mark.parametrize("M,N,K", [(3, 1000, 2048), (8, 320, 6544), (8, 64, 4096), (27, 64, 296), (16, 512, 4096), (64, 64, 8192)])
def test_gemm16_few_outputs_take_the_dot_kernel(dev, M, N, K):
    """Up to 2^25 products of at most 16384 outputs: a wave an output, as for one row (the split kernel took twice the time),
    and so the bits of one row alone."""
    C = gemm16_bits(dev, M, N, K)
    np.testing.assert_array_equal(C[:1], gemm16_bits(dev, M, N, K, rows=1))
    np.testing.assert_array_equal(C[:2], gemm16_bits(dev, M, N, K, rows=2))


@pytest.mark.parametrize("shape", [(0, 0, 1024, 1024, 128), (0, 1, 1024, 1024, 128), (1, 1, 1024, 1152, 128), (0, 0, 1024, 1024, 512)],
                         ids=lambda s: "ta%d_tb%d_%dx%dx%d" % s)
def test_gemm16_short_k_keeps_one_k_group(dev, shape):
    """Whole tiles and a short K: variant 1's sums (one run over K), not those of two k-groups."""
    ta, tb, M, N, K = shape
    np.testing.assert_array_equal(gemm16_bits(dev, M, N, K, ta, tb), gemm16_bits(dev, M, N, K, ta, tb, variant=1))


@pytest.mark.parametrize("M,N,K,variant", [(2100, 2056, 1024, 1), (1500, 2304, 704, 1), (1031, 3080, 1152, 35), (1100, 2312, 768, 35),
                                           (4000, 3600, 320, 3)])
def test_gemm16_ragged_nt_takes_whole_tiles(dev, M, N, K, variant):
    """Ragged outputs of many tiles, both operands along K: the sums of the whole-tile variant of that size (the split kernel adds
    the k-steps of its wave sets, which shows where two k-groups are the variant)."""
    C = gemm16_bits(dev, M, N, K, store=True)
    np.testing.assert_array_equal(C, gemm16_bits(dev, M, N, K, variant=variant, store=True))


@pytest.mark.parametrize("shape", [(0, 1, 2440, 2056, 1152), (1, 1, 2440, 2056, 1152), (0, 1, 2000, 2056, 192), (1, 1, 2000, 2056, 192)],
                         ids=lambda s: "ta%d_tb%d_%dx%dx%d" % s)
def test_gemm16_ragged_stores_take_whole_tiles(dev, shape):
    """The same for a plain store in the other layouts, up to their line in K and tiles."""
    ta, tb, M, N, K = shape
    np.testing.assert_array_equal(gemm16_bits(dev, M, N, K, ta, tb, store=True), gemm16_bits(dev, M, N, K, ta, tb, variant=1, store=True))


@pytest.mark.parametrize("shape", [(0, 0, 905, 5120, 1088), (0, 0, 6709, 6656, 320), (0, 1, 3904, 1280, 256)],
                         ids=lambda s: "ta%d_tb%d_%dx%dx%d" % s)
def test_gemm16_ragged_stores_are_no_slower_than_whole_tiles(dev, shape):
    """An open ragged store takes no longer than the whole-tile kernel its size had before the split one (1.22 to 1.25 times as
    long where the split kernel took it)."""
    ta, tb, M, N, K = shape
    kw = dict(dtype=L.AH_F16, epi=L.EPI_STORE, ta=ta, tb=tb, M=M, N=N, K=K, A=dev.buffer(M * K, L.AH_F16), B=dev.buffer(N * K, L.AH_F16),
              lda=K, ldb=N if tb else K, C_out=dev.buffer(M * N, L.AH_F16), ldc=N)

    def us(variant):
        best = 1e9
        for _ in range(6):
            dev.timer_start()
            for _ in range(30):
                dev.gemm(variant=variant, **kw)
            best = min(best, dev.timer_stop() / 30 * 1e3)
        return best

    whole = us(3 if M * N > 224 * 65536 else 1)
    assert us(0) < 1.1 * whole
    for k in ("A", "B", "C_out"):
        kw[k].free()


@pytest.mark.parametrize("M,N,K", [(256, 5696, 32), (1044, 1088, 56), (2100, 1500, 104), (1153, 1024, 8)])
def test_gemm16_short_ragged_k(dev, M, N, K):
    """A short K that 64 does not divide, 65 to 192 tiles: the register-staged kernel's bits (which a fixed variant runs here, as
    no whole-tile variant takes such a K), and float64 within the bound of the split kernel's test."""
    C = gemm16_bits(dev, M, N, K, store=True)
    np.testing.assert_array_equal(C, gemm16_bits(dev, M, N, K, variant=1, store=True))
    rng = np.random.default_rng(M * 31 + N * 7 + K)
    A, B = q16(rng.standard_normal((M, K))).astype(np.float64), q16(rng.standard_normal((N, K))).astype(np.float64)
    got = C.view(np.float16).astype(np.float64)
    acc = (K + 16) * 2.0**-24 * (np.abs(A) @ np.abs(B).T)
    assert np.all(np.abs(got - (A @ B.T) / 3) <= acc / 3 + 2.0**-11 * np.abs(got) * 1.01 + 2.0**-23)


@pytest.mark.parametrize("shape", [(0, 0, 32, 4096, 4096), (0, 0, 999, 1000, 2056), (0, 1, 72, 2048, 1024), (8, 64, 4096)],
                         ids=lambda s: "x".join(map(str, s)))
def test_gemm16_tune_keeps_the_faster_automatic_choice(dev, shape, tmp_path):
    """Where the split or the dot kernel is the fastest, tuning finds it (variant 0), drops an older choice of the shape, and
    later calls run it: the same bits as before."""
    ta, tb, M, N, K = shape if len(shape) == 5 else (0, 0) + shape
    path = tmp_path / "tune.txt"
    dev.gemm_tune_cache(str(path), True)
    head = path.read_text().splitlines()[0]
    A, Bm = q16(RNG.standard_normal((M, K))), q16(RNG.standard_normal((N, K)))
    Bs = store_operand(Bm, tb)
    dA, dB, dW = dev.buffer(A.astype(np.float16), L.AH_F16), dev.buffer(Bs.astype(np.float16), L.AH_F16), dev.buffer(M * N)
    kw = dict(dtype=L.AH_F16, epi=L.EPI_SGD, ta=ta, tb=tb, M=M, N=N, K=K, A=dA, B=dB, lda=K, ldb=Bs.shape[1], ldc=N, scale=1.0,
              W32=dW, lr=-1.0)

    def bits():
        dW.write(np.zeros(M * N, np.float32))
        dev.gemm(**kw)
        return dW.read().view(np.uint32)

    want, key = bits(), f"1/{ta}/{tb}/{M}/{N}/{K}"
    path.write_text(f"{head}\n{key} 1\n")
    dev.gemm_tune_cache(str(path), False)
    best, us = dev.gemm_tune(iterations=3, **kw)
    assert best == 0 and us > 0
    np.testing.assert_array_equal(bits(), want)
    dev.gemm_tune_cache(str(path), True)
    assert not any(line.startswith(key + " ") for line in path.read_text().splitlines())
    for b in (dA, dB, dW):
        b.free()
