"""FLASH_ATTN_EXT of several query rows (the matrix-core kernel) on MI355X, against attention in double precision.

The bound: a score is an fp32 sum of D exact products, scaled and masked with a rounding each, so it is off by at most
ds = 2^-24 (D + 4) scale sum|q k| + 2^-22 max|s|; a probability's relative error is at most 2 ds (itself and the
denominator) plus a few roundings (its exponential, its two fp16 parts, the fp32 sums), under 2^-18 for the lengths here.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def case(rows, n_kv, heads, kv, D, seed, past=None):
    """q [rows, heads, D] f32, k / v [n_kv, kv, D] f16; a causal mask when past is given (row i sees past + i)."""
    g = np.random.default_rng(seed)
    q = g.standard_normal((rows, heads, D)).astype(np.float32) * 2
    k, v = (g.standard_normal((n_kv, kv, D)).astype(np.float16) for _ in range(2))
    mask = None
    if past is not None:
        mask = np.where(np.arange(n_kv)[None] <= past + np.arange(rows)[:, None], 0, -np.inf).astype(np.float16)
    return q, k, v, mask


def exact(q, k, v, mask, scale):
    rows, heads, D = q.shape
    kv = k.shape[1]
    q = q.astype(np.float16).astype(np.float64)
    out, bound = np.zeros((rows, heads, D)), np.zeros((rows, heads, 1))
    for h in range(heads):
        kk, vv = k[:, h // (heads // kv)].astype(np.float64), v[:, h // (heads // kv)].astype(np.float64)
        s = q[:, h] @ kk.T * scale + (0 if mask is None else mask[:, :k.shape[0]].astype(np.float64))
        m = s.max(1, keepdims=True)
        p = np.exp(s - np.where(np.isfinite(m), m, 0))
        l = p.sum(1, keepdims=True)
        out[:, h] = np.where(l > 0, p @ vv / np.where(l > 0, l, 1), 0)
        ds = 2.0 ** -24 * (D + 4) * abs(scale) * (np.abs(q[:, h]) @ np.abs(kk).T).max() + \
            2.0 ** -22 * np.abs(s[np.isfinite(s)]).max(initial=0)
        bound[:, h] = (2 * ds + 2.0 ** -18) * np.abs(vv).max()
    return out, bound


def device(mx, be, q, k, v, mask, scale, cap=0, mask_pad=0, q_gap=0):
    """The call as the decoder makes it: q as a view [D, rows, heads], the caches as views of [kv D, cap] rows."""
    rows, heads, D = q.shape
    n_kv, kv = k.shape[0], k.shape[1]
    cap = max(cap, n_kv)
    qp = np.zeros((rows, heads * D + q_gap), np.float32)
    qp[:, :heads * D] = q.reshape(rows, -1)
    Q = be.tensor(mx.F32, (heads * D + q_gap, rows), qp)
    caches = []
    for x in (k, v):
        c = np.full((cap, kv * D), np.float16(np.nan))  # nothing past the positions may be read into a result
        c[:n_kv] = x.reshape(n_kv, -1)
        caches.append(be.tensor(mx.F16, (kv * D, cap), c.view(np.uint16)))
    M = None
    if mask is not None:
        mp = np.zeros((rows, n_kv + mask_pad), np.float16)
        mp[:, :n_kv] = mask
        M = be.tensor(mx.F16, (n_kv + mask_pad, rows), mp.view(np.uint16))
    Y = be.tensor(mx.F32, (D, heads, rows), np.full((rows, heads, D), 7.0, np.float32))
    qv = Q.view((D, rows, heads), (4, (heads * D + q_gap) * 4, D * 4))
    views = [c.view((D, n_kv, kv), (2, kv * D * 2, D * 2)) for c in caches]
    be.flash_attn_ext(qv, views[0], views[1], M, Y, scale)
    be.sync()
    return Y.numpy().reshape(rows, heads, D)


# pairs (rows x heads per kv head) around 32, positions around a step (32), a turn of the eight waves (256) and splits
SHAPES = [(2, 1, 2, 2), (2, 31, 4, 2), (3, 32, 2, 1), (5, 33, 6, 2), (16, 64, 4, 2), (17, 100, 4, 2), (33, 257, 2, 2),
          (4, 1000, 16, 2), (31, 255, 3, 1), (32, 256, 8, 1), (65, 512, 16, 8), (5, 3010, 16, 8), (130, 700, 32, 8),
          (300, 320, 16, 8), (9, 5000, 2, 1)]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("rows,n_kv,heads,kv", SHAPES)
def test_causal(mx, be, rows, n_kv, heads, kv, D):
    past = max(0, n_kv - rows)
    q, k, v, mask = case(rows, n_kv, heads, kv, D, rows + n_kv, past)
    want, bound = exact(q, k, v, mask, D ** -0.5)
    for pad in (0, (-n_kv) % 8, (-n_kv) % 8 + 64):  # mask rows in 16-byte steps (the matrix cores) or not (row by row)
        got = device(mx, be, q, k, v, mask, D ** -0.5, cap=n_kv + 40, mask_pad=pad)
        assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("scale", [0.1, -0.3, 0.0])
@pytest.mark.parametrize("q_gap", [0, 4, 1])
def test_no_mask(mx, be, scale, q_gap):
    """Scales of either sign; q rows at other strides, 16-byte aligned or not."""
    q, k, v, _ = case(20, 333, 4, 2, 128, 4)
    want, bound = exact(q, k, v, None, scale)
    assert np.all(np.abs(device(mx, be, q, k, v, None, scale, cap=500, q_gap=q_gap) - want) <= bound)


def test_masks(mx, be):
    """Finite mask values (fp16's lowest among them), rows with nothing visible (zeros), scores far apart."""
    rows, n_kv = 40, 600
    q, k, v, mask = case(rows, n_kv, 4, 2, 128, 8, 0)
    g = np.random.default_rng(1)
    mask = g.choice(np.array([0, -np.inf, -65504, -3.5, 2.25], np.float16), (rows, n_kv))
    mask[3] = -np.inf
    mask[5] = -65504
    mask[:, 64:400] = -np.inf  # whole steps hidden
    mask[7, 100] = 0
    q[9] *= 40
    want, bound = exact(q, k, v, mask, 0.25)
    got = device(mx, be, q, k, v, mask, 0.25)
    assert np.all(np.abs(got - want) <= bound) and np.all(got[3] == 0)


def test_growing_scores(mx, be):
    """Scores that grow along the positions: the running reference moves at almost every step."""
    q, k, v, _ = case(40, 2048, 2, 1, 128, 9)
    k = (k.astype(np.float32) * 0.05 + q[:, 0].mean(0) * np.linspace(0, 3, 2048)[:, None, None]).astype(np.float16)
    q = np.abs(q)
    want, bound = exact(q, k, v, None, 0.5)
    assert np.all(np.abs(device(mx, be, q, k, v, None, 0.5) - want) <= bound)


def test_not_a_number(mx, be):
    """A NaN in q reaches its own row only; one in a key that every row hides reaches nothing."""
    rows, n_kv = 24, 320
    q, k, v, mask = case(rows, n_kv, 2, 1, 128, 3, 200)
    k[310] = v[300] = np.float16(np.nan)  # row i sees 200 + i: hidden, in steps that hold other hidden positions only
    mask[:, 224:] = -np.inf
    want, bound = exact(q, np.nan_to_num(k), np.nan_to_num(v), mask, 0.1)
    assert np.all(np.abs(device(mx, be, q, k, v, mask, 0.1) - want) <= bound)
    q[5, 1, 17] = np.nan
    got = device(mx, be, q, k, v, mask, 0.1)
    assert np.isnan(got[5, 1]).all() and np.isfinite(np.delete(got, 5, 0)).all() and np.isfinite(got[5, 0]).all()


@pytest.mark.parametrize("heads,kv,D", [(2, 1, 128), (16, 8, 128), (6, 2, 128), (4, 2, 64), (3, 3, 64)])
@pytest.mark.parametrize("odd", ["nan", "inf", "-inf", "both", "key"])
def test_hidden_odd_values(mx, be, heads, kv, D, odd):
    """Infinities and NaN reach the rows that see their position and no other: positions that some rows of a workgroup see
    (causal; 77 hidden from the first rows), and one that no row sees in a step with positions that some do."""
    rows, n_kv, past = 70, 400, 220
    q, k, v, mask = case(rows, n_kv, heads, kv, D, 5, past)
    mask[:9, 77] = -np.inf
    want, bound = exact(q, k, v, mask, D ** -0.5)
    at = [77, past + 3, past + 40, past + rows + 5]
    for i, j in enumerate(at):
        (k if odd == "key" else v)[j, :, ::3] = np.nan if odd == "key" else (np.inf, -np.inf)[i % 2] if odd == "both" else float(odd)
    for i in range(rows):  # what the odd values that a row sees add to the sums of its others
        for j in at:
            if mask[i, j] == 0:
                with np.errstate(invalid="ignore"):
                    want[i] += np.nan if odd == "key" else np.where(np.isfinite(v[j]), 0, v[j]).repeat(heads // kv, 0)
    got = device(mx, be, q, k, v, mask, D ** -0.5, cap=n_kv + 8)
    inf = np.isinf(want)  # (NaN where the merge of splits multiplies it by a split's weight of 0)
    assert np.isnan(got[np.isnan(want)]).all() and np.all(np.isnan(got[inf]) | (got[inf] == want[inf]))
    ok = np.isfinite(want)  # (channels without odd values are whole in every row)
    assert ok[:3].all() and np.all(np.abs(got[ok] - want[ok]) <= np.broadcast_to(bound, want.shape)[ok])


@pytest.mark.parametrize("odd", ["nan", "inf", "key"])
@pytest.mark.parametrize("rows,n_kv", [(4, 500), (7, 300), (20, 60)])
@pytest.mark.parametrize("heads,kv", [(3, 3), (4, 2), (8, 2)])
def test_hidden_odd_values_few_rows(mx, be, heads, kv, rows, n_kv, odd):
    """The same where a few rows go to the one-row kernel; a row that sees nothing but a NaN score is NaN."""
    past = n_kv - rows - 8
    q, k, v, mask = case(rows, n_kv, heads, kv, 128, 6, past)
    mask[0, 17] = -np.inf
    want, bound = exact(q, k, v, mask, 0.1)
    at = [17, past + rows - 1, past + rows + 3]  # hidden from the first row, from all but the last, from all
    for j in at:
        (k if odd == "key" else v)[j, :, ::3] = np.nan if odd == "key" else float(odd)
    got = device(mx, be, q, k, v, mask, 0.1, cap=n_kv + 8)
    assert np.all(np.abs(got[0] - want[0]) <= np.broadcast_to(bound, want.shape)[0])
    if odd == "key":
        assert np.isnan(got[1:]).all()
        mask[2] = -np.inf
        mask[2, 17] = 0
        assert np.isnan(device(mx, be, q, k, v, mask, 0.1)[2]).all()
    else:
        assert not np.isfinite(got[1:, :, ::3]).any()
        assert np.all(np.abs(got - want) <= bound, where=(np.arange(128) % 3 != 0))


# either side of the lines between the kernels: one chunk of 64, two, three, eight (64-position chunks of 512 and 256 in all)
@pytest.mark.parametrize("rows,n_kv,heads,kv", [(64, 64, 16, 8), (65, 64, 16, 8), (64, 64, 16, 16), (65, 64, 16, 16),
                                                (32, 128, 16, 8), (8, 256, 16, 8), (9, 256, 16, 8), (8, 449, 16, 8),
                                                (9, 449, 16, 8), (6, 300, 32, 8), (7, 300, 32, 8), (128, 192, 2, 2)])
def test_kernel_lines(mx, be, rows, n_kv, heads, kv):
    q, k, v, mask = case(rows, n_kv, heads, kv, 128, rows, n_kv - rows)
    want, bound = exact(q, k, v, mask, 0.088)
    assert np.all(np.abs(device(mx, be, q, k, v, mask, 0.088, mask_pad=(-n_kv) % 8) - want) <= bound)


def test_few_rows_recorded_without_scratch(mx):
    """A call that the one-row kernel would take in splits, recorded with no eager run before it: no scratch to be had, so
    the matrix cores take it in one."""
    be = mx.Backend(0)
    rows, n_kv, heads, kv, D = 3, 250, 4, 2, 128
    q, k, v, _ = case(rows, n_kv, heads, kv, D, 2)
    want, bound = exact(q, k, v, None, 0.09)
    K, V = (be.tensor(mx.F16, (kv * D, n_kv), x.reshape(n_kv, -1).view(np.uint16)) for x in (k, v))
    Q, Y = be.tensor(mx.F32, (heads * D, rows), q.reshape(rows, -1)), be.tensor(mx.F32, (D, heads, rows))
    views = [c.view((D, n_kv, kv), (2, kv * D * 2, D * 2)) for c in (K, V)]
    be.graph_begin()
    be.flash_attn_ext(Q.view((D, rows, heads), (4, heads * D * 4, D * 4)), views[0], views[1], None, Y, 0.09)
    g = be.graph_end()
    for _ in range(3):
        Y.set(np.zeros((rows, heads, D), np.float32))
        be.graph_launch(g)
        be.sync()
        assert np.all(np.abs(Y.numpy().reshape(rows, heads, D) - want) <= bound)
    be.graph_free(g)
    del Q, K, V, Y, views
    be.close()


@pytest.mark.parametrize("heads,kv,D", [(8, 1, 128), (12, 4, 128), (8, 1, 64), (16, 16, 64)])
def test_weights_in_full(mx, be, heads, kv, D):
    """Scores that are exact in fp32 (one product each), so that the error is the weights' own and that of their sums. A
    weight is off by half a unit of its exponent where that is below 2 (2^-24), of its exponential (2^-24) and of its two
    fp16 parts (2^-24 of most of them), the sum, the division and the product by 2^-25 each: root mean square about
    1.2 * 2^-24 = 7.3e-8 of a result of one to some ten weights. Exponents of 4 to 8 (units of 2^-21) would add 1.2e-7."""
    g = np.random.default_rng(D)
    rows = 72
    q, k, v, mask = case(rows, rows, heads, kv, D, 1, 0)
    q[:] = 0
    np.put_along_axis(q, g.integers(0, D, (rows, heads, 1)), 8 * g.uniform(1, 2, (rows, heads, 1)).astype(np.float16), 2)
    k = g.uniform(-0.5, 0.5, k.shape).astype(np.float16)
    want, _ = exact(q, k, v, mask, 0.125)
    got = device(mx, be, q, k, v, mask, 0.125)
    assert np.square(got[:48] - want[:48]).sum() <= (1e-7) ** 2 * np.square(want[:48]).sum()


def test_recorded(mx):
    """Recorded with no eager run before it (splits need scratch: the row kernel takes it), then after one; replayed."""
    be = mx.Backend(0)
    rows, n_kv, heads, kv, D = 5, 1500, 4, 2, 128
    q, k, v, _ = case(rows, n_kv, heads, kv, D, 2)
    want, bound = exact(q, k, v, None, 0.09)
    K, V = (be.tensor(mx.F16, (kv * D, n_kv), x.reshape(n_kv, -1).view(np.uint16)) for x in (k, v))
    Q, Y = be.tensor(mx.F32, (heads * D, rows), q.reshape(rows, -1)), be.tensor(mx.F32, (D, heads, rows))
    qv = Q.view((D, rows, heads), (4, heads * D * 4, D * 4))
    kvw = [c.view((D, n_kv, kv), (2, kv * D * 2, D * 2)) for c in (K, V)]
    one = Q.view((D, 1, heads), (4, heads * D * 4, D * 4))  # sizes the row kernel's scratch, as a decode step does
    big = be.tensor(mx.F32, (1 << 20,))
    be.argmax(be.tensor(mx.F32, (1 << 20, 4)), be.tensor(mx.I32, (4,)))
    be.flash_attn_ext(one, kvw[0], kvw[1], None, be.tensor(mx.F32, (D, heads, 1)), 0.09)
    be.sync()
    graphs = []
    for _ in range(2):
        be.graph_begin()
        be.flash_attn_ext(qv, kvw[0], kvw[1], None, Y, 0.09)
        graphs.append(be.graph_end())
        be.flash_attn_ext(qv, kvw[0], kvw[1], None, Y, 0.09)
        be.sync()
    for _ in range(3):
        for g in graphs:
            Y.set(np.zeros((rows, heads, D), np.float32))
            be.graph_launch(g)
            be.sync()
            assert np.all(np.abs(Y.numpy().reshape(rows, heads, D) - want) <= bound)
    for g in graphs:
        be.graph_free(g)
    del Q, K, V, Y, big, qv, kvw, one
    be.close()
