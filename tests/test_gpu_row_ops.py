"""The wide forms of the row ops (RMS_NORM, ADD / MUL, SWIGLU, q/k norm + RoPE + KV stores over many rows) on MI355X:
each gives what the general form gives for the same rows, which operands off 16-byte alignment (or fewer rows) still take.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_view(mx, be, x, gap, off):
    """x [rows, n] on the device in rows n + gap floats apart, starting `off` floats into the buffer."""
    rows, n = x.shape
    buf = np.full(rows * (n + gap) + off + 8, 3.0, np.float32)
    for r in range(rows):
        buf[off + r * (n + gap):off + r * (n + gap) + n] = x[r]
    return be.tensor(mx.F32, (buf.size,), buf).view((n, rows), (4, (n + gap) * 4), 4 * off)


def read(mx, be, v, rows, n, gap, off):
    b = v.base_tensor.get_bytes().view(np.float32)
    return np.stack([b[off + r * (n + gap):off + r * (n + gap) + n] for r in range(rows)]), b


# (gap, offset) in floats: 16-byte rows, and rows or bases off them
WIDE, OFF = [(0, 0), (8, 4)], [(1, 0), (0, 1), (4, 2)]


@pytest.mark.parametrize("rows,n", [(1, 4), (3, 1020), (2, 1024), (5, 1028), (7, 2052), (600, 2048), (3, 8192)])
@pytest.mark.parametrize("op", ["add", "mul", "swiglu"])
def test_elementwise(mx, be, op, rows, n):
    g = np.random.default_rng(rows + n)
    a, b = (g.standard_normal((rows, n)).astype(np.float32) * 3 for _ in range(2))
    a[0, :4] = [0, -0.0, 88, -104]
    got = []
    for gap, off in WIDE + OFF:
        A, B = rows_view(mx, be, a, gap, off), rows_view(mx, be, b, 4, 4 if off % 4 == 0 else 0)
        Y = rows_view(mx, be, np.zeros_like(a), gap, off)
        getattr(be, op)(A, B, Y)
        be.sync()
        y, buf = read(mx, be, Y, rows, n, gap, off)
        assert np.count_nonzero(buf == 3.0) >= rows * gap + off  # nothing between the rows was written
        got.append(y)
    if op != "swiglu":
        assert np.array_equal(got[0], a + b if op == "add" else a * b)
    for y in got[1:]:
        assert np.array_equal(y.view(np.uint32), got[0].view(np.uint32))


@pytest.mark.parametrize("b_ne", [(12, 1, 1, 1), (12, 6, 1, 1), (12, 6, 4, 2), (1, 6, 4, 2), (12, 1, 4, 1), (4, 6, 4, 2)])
@pytest.mark.parametrize("permuted", [False, True])
def test_repeats(mx, be, b_ne, permuted):
    """b repeated along any axes over a [12, 6, 4, 2], a contiguous or with its axes 1 and 2 exchanged."""
    g = np.random.default_rng(7)
    a = g.standard_normal((2, 4, 6, 12)).astype(np.float32)
    b = g.standard_normal(b_ne[::-1]).astype(np.float32)
    want = a * np.tile(b, [x // y for x, y in zip(a.shape, b.shape)])
    if permuted:  # memory [ne3, ne1, ne2, ne0]
        A = be.tensor(mx.F32, (12, 4, 6, 2), np.ascontiguousarray(a.transpose(0, 2, 1, 3)))
        A = A.view((12, 6, 4, 2), (4, 4 * 48, 48, 4 * 288))
    else:
        A = be.tensor(mx.F32, (12, 6, 4, 2), a)
    Y = be.tensor(mx.F32, (12, 6, 4, 2))
    be.mul(A, be.tensor(mx.F32, b_ne, b), Y)
    be.sync()
    assert np.array_equal(Y.numpy(), want)


@pytest.mark.parametrize("rows,n", [(1, 1024), (5, 1020), (3, 1028), (300, 2048), (2, 2052), (4, 4096), (3, 4100), (2, 8192),
                                    (2, 8196)])
@pytest.mark.parametrize("weight", [False, True])
def test_rms_norm(mx, be, rows, n, weight):
    """Both forms sum the squares in double and round the mean to float: the result is the reference's to 2 ulp."""
    g = np.random.default_rng(n)
    x = g.standard_normal((rows, n)).astype(np.float32)
    x[0] *= 1e-3
    w = g.standard_normal(n).astype(np.float32) if weight else None
    sq = (x * x).astype(np.float64).sum(1, keepdims=True)
    scale = (np.float32(1) / np.sqrt((sq / n).astype(np.float32) + np.float32(1e-6))).astype(np.float32)
    want = (x * scale) * (w if weight else np.float32(1))
    W = be.tensor(mx.F32, (n,), w) if weight else None
    for gap, off in WIDE + OFF:
        X, Y = rows_view(mx, be, x, gap, off), rows_view(mx, be, np.zeros_like(x), gap, off)
        be.rms_norm(X, Y, 1e-6, W)
        be.sync()
        y, _ = read(mx, be, Y, rows, n, gap, off)
        assert np.all(np.abs(y - want) <= 2 * np.spacing(np.abs(want)))


@pytest.mark.parametrize("nq,nkv,rows", [(16, 8, 256), (16, 8, 97), (5, 3, 400), (2, 1, 3000), (16, 8, 512)])
def test_qk_norm_rope_kv_rows(mx, be, nq, nkv, rows):
    """Many rows in one call give the bits of one call per 32 rows; a position outside the caches stores nothing there."""
    g = np.random.default_rng(rows)
    d, cap = 128, rows + 40
    q, k, v = (g.standard_normal((rows, n * d)).astype(np.float32) for n in (nq, nkv, nkv))
    pos = g.permutation(cap)[:rows].astype(np.int32)
    pos[rows // 2] = cap + 3
    nw = [be.tensor(mx.F32, (d,), 1 + 0.1 * g.standard_normal(d).astype(np.float32)) for _ in range(2)]
    T = [be.tensor(mx.F32, (x.shape[1], rows), x) for x in (q, k, v)]
    P = be.tensor(mx.I32, (rows,), pos)
    results = []
    for step in (rows, 32):
        out = be.tensor(mx.F32, (nq * d, rows), np.zeros((rows, nq * d), np.float32))
        kc, vc = (be.tensor(mx.F16, (nkv * d, cap), np.zeros((cap, nkv * d), np.uint16)) for _ in range(2))
        errors = 0
        for r0 in range(0, rows, step):
            n = min(step, rows - r0)
            heads = lambda t, h: t.view((d, h, n), (4, 4 * d, 4 * d * h), r0 * 4 * d * h)  # noqa: E731
            be.qk_norm_rope_kv(heads(T[0], nq), heads(T[1], nkv), heads(T[2], nkv), *nw, P.view((n,), (4,), 4 * r0),
                               heads(out, nq), kc, vc, 1e-6, 1e6)
            try:
                be.sync()
            except mx.MxError as e:
                assert e.code == mx.INVALID
                errors += 1
        assert errors == 1
        results.append([t.get_bytes() for t in (out, kc, vc)])
    for a, b in zip(*results):
        assert np.array_equal(a, b)


def test_norm_of_more_rows_than_a_grid_has(mx, be):
    """2^24 rows of 1024 floats (64 GiB, in place): a workgroup of 256 to a row would be a grid of 2^32 threads, which is
    refused. The first rows, the last ones and some between."""
    n, rows = 1024, 1 << 24
    try:
        X = be.tensor(mx.F32, (n, rows))
    except mx.MxError as e:
        pytest.skip(f"no 64 GiB on the device: {e}")
    at = [0, 1, 2, 3, (1 << 22) + 5, (1 << 23) - 1, rows - 2, rows - 1]
    x = np.random.default_rng(4).standard_normal((len(at), n)).astype(np.float32)
    for r, v in zip(at, x):
        X.set(v, 4 * n * r)
    be.rms_norm(X, X, 1e-6)
    be.sync()
    got = np.stack([X.get_bytes(4 * n * r, 4 * n).view(np.float32) for r in at])
    x64 = x.astype(np.float64)
    want = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-6)
    assert np.all(np.abs(got - want) <= 2.0 ** -22 * np.abs(want))
    X.free()
