"""MUL_MAT at more than 8 columns on F16 / F32 weights (the MFMA GEMM) on MI355X, against the product in double precision.

The bound: every product is exact (fp16 x fp16) or rounded once (fp32), and the fp32 sums are chains of at most 16
additions of MFMA results (each itself up to 16 products), K / 128 + 8 sums of those, and 8 group and split sums, so
|error| <= (2 * 16 + K / 128 + 32) * 2^-24 * sum |w x|.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng


def data(mx, t, N, K, M, seed):
    g = RNG(seed)
    w = (g.standard_normal((N, K)) * 0.05).astype(np.float32)
    x = g.standard_normal((M, K)).astype(np.float32)
    if t == mx.F16:
        return w.astype(np.float16), x, w.astype(np.float16).astype(np.float64), x.astype(np.float16).astype(np.float64)
    return w, x, w.astype(np.float64), x.astype(np.float64)


def check(y, w64, x64):
    K = w64.shape[1]
    bound = (64 + K / 128) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T) + 1e-38
    assert np.all(np.abs(y.astype(np.float64) - x64 @ w64.T) <= bound)


def upload(mx, be, t, ne, w):
    return be.tensor(t, ne, w.view(np.uint16) if t == mx.F16 else w)


# M, N at tile edges (16, 32, 64, 128) and one past them; K at and around a slice (64 halves, 32 floats), a stage of
# several slices, odd tails (8 halves, 4 floats) and the K-split rule (K >= 4096)
SHAPES = [(9, 1, 8), (9, 33, 64), (16, 32, 72), (17, 31, 136), (31, 130, 264), (32, 64, 1056), (33, 129, 520),
          (64, 257, 2048), (65, 100, 2056), (28, 64, 4608), (40, 300, 4104), (133, 200, 6144), (128, 128, 64),
          (129, 1000, 96), (130, 2500, 128), (200, 8200, 192), (512, 8192, 72), (65, 16500, 200)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("tname", ["F16", "F32"])
def test_product(mx, be, tname, M, N, K):
    t = getattr(mx, tname)
    w, x, w64, x64 = data(mx, t, N, K, M, 7 * M + N + K)
    W, X, Y = upload(mx, be, t, (K, N), w), be.tensor(mx.F32, (K, M), x), be.tensor(mx.F32, (N, M))
    be.mul_mat(W, X, Y)
    be.sync()
    check(Y.numpy().reshape(M, N), w64, x64)


@pytest.mark.parametrize("tname", ["F16", "F32"])
@pytest.mark.parametrize("M", [20, 300])
def test_group_and_strided_rows(mx, be, tname, M):
    """Weights of different widths in one launch; rows of src1 and dst with gaps; the gaps of dst stay as they were."""
    t, K, Ns, gap = getattr(mx, tname), 328, (70, 200, 33), 16
    g = RNG(M)
    xf = g.standard_normal((M, K + gap)).astype(np.float32)
    Xf = be.tensor(mx.F32, (K + gap, M), xf)
    X = Xf.view((K, M), (4, (K + gap) * 4))
    Ws, ys, refs = [], [], []
    for i, N in enumerate(Ns):
        w, _, w64, _ = data(mx, t, N, K, 1, 50 + i)
        Ws.append(upload(mx, be, t, (K, N), w))
        refs.append(w64)
        ys.append(be.tensor(mx.F32, (N + 4, M), np.full((M, N + 4), 7.0, np.float32)))
    be.mul_mat_group(Ws, X, [y.view((N, M), (4, (N + 4) * 4)) for y, N in zip(ys, Ns)])
    be.sync()
    x = xf[:, :K]
    x64 = (x.astype(np.float16) if t == mx.F16 else x).astype(np.float64)
    for y, N, w64 in zip(ys, Ns, refs):
        got = y.numpy().reshape(M, N + 4)
        check(got[:, :N], w64, x64)
        assert np.all(got[:, N:] == 7.0)


@pytest.mark.parametrize("tname", ["F16", "F32"])
def test_batches(mx, be, tname):
    """Broadcast weights over batch slices: dst[:, :, i2, i3] = W[:, :, i2 / r2, i3 / r3] x src1[:, :, i2, i3]."""
    t, K, N, M = getattr(mx, tname), 104, 50, 40
    w, x, w64, x64 = data(mx, t, 2 * N, K, M * 4, 3)
    W, X = upload(mx, be, t, (K, N, 2), w), be.tensor(mx.F32, (K, M, 4), x)
    Y = be.tensor(mx.F32, (N, M, 4))
    be.mul_mat(W, X, Y)
    be.sync()
    y = Y.numpy().reshape(4, M, N)
    for i in range(4):
        check(y[i], w64[(i // 2) * N:(i // 2 + 1) * N], x64[i * M:(i + 1) * M])


@pytest.mark.parametrize("tname", ["F16", "F32"])
@pytest.mark.parametrize("M,N,K,slices,r", [
    (9, 33, 64, (24, 3), (2, 3)),        # a tile or two a slice, both axes, broadcast along both
    (40, 200, 4608, (5, 1), (5, 1)),     # K split: one matrix to every slice
    (130, 260, 4104, (3, 2), (1, 2)),    # K split or the fp16 pass
    (300, 400, 136, (40, 1), (1, 1)),    # the fp16 pass over every slice
    (2100, 8, 4096, (4, 1), (2, 1)),     # fp16 rows of 17 MB a slice: more than a launch's scratch holds
])
def test_slices_share_launches(mx, tname, M, N, K, slices, r):
    """However many slices a product has, it takes a few launches (counted in a recording): slices with gaps between them,
    against double precision; the gaps stay as they were."""
    be = mx.Backend(0)
    t, (n2, n3), (r2, r3) = getattr(mx, tname), slices, r
    m2, m3 = n2 // r2, n3 // r3
    w, x, w64, x64 = data(mx, t, N * m2 * m3, K, M * n2 * n3, N + K)
    W = upload(mx, be, t, (K, N, m2, m3), w)
    xg = np.zeros((n3, n2, M + 3, K), np.float32)  # three rows between slices
    xg[:, :, :M] = x.reshape(n3, n2, M, K)
    yg = np.full((n3, n2, M + 2, N + 4), 7.0, np.float32)
    Xb, Yb = be.tensor(mx.F32, (K, M + 3, n2, n3), xg), be.tensor(mx.F32, (N + 4, M + 2, n2, n3), yg)
    X = Xb.view((K, M, n2, n3), (4, 4 * K, 4 * K * (M + 3), 4 * K * (M + 3) * n2))
    Y = Yb.view((N, M, n2, n3), (4, 4 * (N + 4), 4 * (N + 4) * (M + 2), 4 * (N + 4) * (M + 2) * n2))
    be.mul_mat(W, X, Y)
    be.sync()
    got = Yb.numpy()
    for i3 in range(n3):
        for i2 in range(n2):
            z, m = i3 * n2 + i2, (i3 // r3) * m2 + i2 // r2
            check(got[i3, i2, :M, :N], w64[m * N:(m + 1) * N], x64[z * M:(z + 1) * M])
    assert np.all(got[:, :, M:] == 7.0) and np.all(got[:, :, :, N:] == 7.0)
    be.graph_begin()
    be.mul_mat(W, X, Y)
    g = be.graph_end()
    assert be.graph_nodes(g) <= 6  # pass, product, reduce; twice where the scratch holds some of the slices
    Yb.set(yg)
    be.graph_launch(g)
    be.sync()
    assert np.array_equal(Yb.numpy(), got)
    be.graph_free(g)
    del W, X, Y, Xb, Yb
    be.close()


@pytest.mark.parametrize("tname", ["F16", "F32"])
def test_more_rows_than_a_grid_has(mx, be, tname):
    """2^24 rows and some: a grid of one workgroup of 256 to a row is refused (2^32 threads). Small integers: exact."""
    M, N, K = (1 << 24) + 40, 2, 8
    g = RNG(8)
    w = g.integers(-8, 8, (N, K)).astype(np.float16 if tname == "F16" else np.float32)
    x = g.integers(-8, 8, (M, K)).astype(np.float32)
    W, X, Y = upload(mx, be, getattr(mx, tname), (K, N), w), be.tensor(mx.F32, (K, M), x), be.tensor(mx.F32, (N, M))
    be.mul_mat(W, X, Y)
    be.sync()
    assert np.array_equal(Y.numpy().reshape(M, N), x @ w.astype(np.float32).T)


@pytest.mark.parametrize("side", ["weights", "activations"])
def test_subnormal_halves(mx, be, side):
    """fp16 subnormals count in full: times small integers every sum is a multiple of 2^-24 below 2^-9, exact in fp32."""
    K, N, M = 64, 40, 48
    g = RNG(5)
    sub = lambda n: g.integers(-60, 60, (n, K)) * 2.0 ** -24  # noqa: E731
    w = (sub(N) if side == "weights" else g.integers(-8, 8, (N, K))).astype(np.float16)
    x = (sub(M) if side == "activations" else g.integers(-8, 8, (M, K))).astype(np.float32)
    W, X, Y = upload(mx, be, mx.F16, (K, N), w), be.tensor(mx.F32, (K, M), x), be.tensor(mx.F32, (N, M))
    be.mul_mat(W, X, Y)
    be.sync()
    assert np.array_equal(Y.numpy().reshape(M, N), (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32))


def test_infinities(mx, be):
    """An infinity or NaN reaches its own row or column only."""
    K, N, M = 72, 40, 48
    w, x, _, _ = data(mx, mx.F16, N, K, M, 6)
    Y = be.tensor(mx.F32, (N, M))
    x[3, 5] = np.inf
    w[7, 9] = np.nan
    W, X = upload(mx, be, mx.F16, (K, N), w), be.tensor(mx.F32, (K, M), x)
    be.mul_mat(W, X, Y)
    be.sync()
    bad = ~np.isfinite(Y.numpy().reshape(M, N))
    bad[3] = bad[:, 7] = False
    assert not bad.any()


def test_recorded_before_and_after_the_buffer_grows(mx):
    """Recorded with no eager run before it (no scratch to be had then: the mat-vec computes it), and recorded with
    scratch that a larger product replaces later: every replay gives the eager result's values to the bound."""
    be = mx.Backend(0)
    K, N, M = 512, 4096, 256  # 128 x 128 and 64 x 128 tiles: the fp16 rows are in scratch
    w, x, w64, x64 = data(mx, mx.F16, N, K, M, 9)
    W, X, Y = upload(mx, be, mx.F16, (K, N), w), be.tensor(mx.F32, (K, M), x), be.tensor(mx.F32, (N, M))
    graphs = []
    for _ in range(2):
        be.graph_begin()
        be.mul_mat(W, X, Y)
        graphs.append(be.graph_end())
        be.mul_mat(W, X, Y)  # now there is scratch
        be.sync()
    assert be.graph_nodes(graphs[0]) > be.graph_nodes(graphs[1])
    big = be.tensor(mx.F32, (K, 4 * M), np.concatenate([x] * 4))
    be.mul_mat(W, big, be.tensor(mx.F32, (N, 4 * M)))
    for _ in range(3):
        for g in graphs:
            Y.set(np.zeros((M, N), np.float32))
            be.graph_launch(g)
            be.sync()
            check(Y.numpy().reshape(M, N), w64, x64)
    for g in graphs:
        be.graph_free(g)
    del W, X, Y, big
    be.close()
