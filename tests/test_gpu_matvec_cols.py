"""Products of 1 to 8 columns on quantized weights (the mat-vec: four waves and one set of rows a workgroup, or, from two
columns on, eight waves that go on to further rows), and the quantizers' divisions, on MI355X against the oracle.

The bound of a product: the kernels sum the oracle's exact block integers, K / 32 scaled terms in fp32 in another order
(at most 192 here), so about sqrt(192) * 2^-24 = 8e-7 of a row's largest output; 2e-5 would still show a lost term. Behind
a norm or a GLU an activation that differs in its last bit may round to the next quant: one in 127 * 32 of a block's sum
of squares, at most a few blocks a row, 2e-4.
"""
import numpy as np
import pytest

import oracle as O
from helpers import rel_err

pytestmark = pytest.mark.gpu

NAMES = {O.TYPE_Q8_0: "q8_0", O.TYPE_Q4_K: "q4_K", O.TYPE_Q5_K: "q5_K", O.TYPE_Q6_K: "q6_K"}
TYPES = pytest.mark.parametrize("t", list(NAMES), ids=lambda t: NAMES[t])


def weights(t, N, K, seed):
    return O.quantize_chunk(t, O.fill_normal(seed, N, K, 0.0, 0.05))


# rows at and around a workgroup's (8 waves x 1, 2 or 4 row groups), at the launch cap (512 workgroups, 32 rows each at
# 256 elements, and one row more; one pass and two), K at one super-block, the four-wave rule (1024) and past the
# preloaded pieces (2048 elements each)
@TYPES
@pytest.mark.parametrize("M", [1, 2, 3, 4, 7, 8])
@pytest.mark.parametrize("N,K", [(1, 256), (7, 1024), (8, 1280), (9, 4352), (33, 768), (129, 2304), (16385, 256), (8193, 512)])
def test_columns(mx, be, t, M, N, K):
    w, x = weights(t, N, K, 11 + N + K), O.fill_normal(13 + M, M, K)
    W, X, Y = be.tensor(t, (K, N), w), be.tensor(mx.F32, (K, M), x), be.tensor(mx.F32, (N, M))
    be.mul_mat(W, X, Y)
    be.sync()
    assert rel_err(Y.numpy().reshape(M, N), O.mul_mat(t, w, x)) <= 2e-5


# either side of the lines between the two shapes: 16,384 rows up to K = 1024 and past it; Q5_K (16 rows a workgroup, 4 at
# K = 4096) half a chip of workgroups, a chip, two, with M <= 4
@pytest.mark.parametrize("t", [O.TYPE_Q4_K, O.TYPE_Q5_K, O.TYPE_Q6_K], ids=lambda t: NAMES[t])
@pytest.mark.parametrize("fused", [False, True], ids=["plain", "residual"])
@pytest.mark.parametrize("M", [2, 4, 6])
@pytest.mark.parametrize("N,K", [(16383, 256), (16384, 512), (2049, 256), (4097, 256), (8193, 256), (1030, 4096)])
def test_shape_of_a_workgroup(mx, be, t, fused, M, N, K):
    w, x, r = weights(t, N, K, 5 + N), O.fill_normal(7 + M, M, K), O.fill_normal(3, M, N)
    W, X, Y = be.tensor(t, (K, N), w), be.tensor(mx.F32, (K, M), x), be.tensor(mx.F32, (N, M), r)
    if fused:
        be.mul_mat_fused([W], X, [Y], residual=[Y])
    else:
        be.mul_mat(W, X, Y)
    be.sync()
    assert rel_err(Y.numpy().reshape(M, N) - (r if fused else 0), O.mul_mat(t, w, x)) <= 2e-5


@TYPES
@pytest.mark.parametrize("M", [1, 2, 5, 8])
@pytest.mark.parametrize("Ns,K", [((70, 9, 1), 1024), ((4100, 8300), 512), ((2048, 1024, 1024), 2304)])
def test_group_behind_a_norm(mx, be, t, M, Ns, K):
    """Narrower problems of a group end early; the norm's sum over four and eight waves; residuals in place."""
    ws = [weights(t, n, K, 17 + i) for i, n in enumerate(Ns)]
    x, nw = O.fill_normal(19 + M, M, K) * np.float32(3), O.fill_normal(23, 1, K, 1.0, 0.1)[0]
    r = [O.fill_normal(29 + i, M, n) for i, n in enumerate(Ns)]
    W = [be.tensor(t, (K, n), w) for n, w in zip(Ns, ws)]
    R = [be.tensor(mx.F32, (n, M), v) for n, v in zip(Ns, r)]
    be.mul_mat_fused(W, be.tensor(mx.F32, (K, M), x), R, norm_w=be.tensor(mx.F32, (K,), nw), eps=1e-6, residual=R)
    be.sync()
    h = O.binary("mul", O.rms_norm(x, 1e-6), nw)
    for n, w, v, y in zip(Ns, ws, r, R):
        assert rel_err(y.numpy().reshape(M, n) - v, O.mul_mat(t, w, h)) <= 2e-4


@TYPES
@pytest.mark.parametrize("M", [2, 6])
def test_glu(mx, be, t, M):
    K, N = 3072, 1030
    w, g, u = weights(t, N, K, 31), O.fill_normal(37, M, K), O.fill_normal(41, M, K)
    W, G, U, Y = be.tensor(t, (K, N), w), be.tensor(mx.F32, (K, M), g), be.tensor(mx.F32, (K, M), u), be.tensor(mx.F32, (N, M))
    be.mul_mat_fused([W], G, [Y], glu_b=U)
    be.sync()
    assert rel_err(Y.numpy().reshape(M, N), O.mul_mat(t, w, O.swiglu(g, u))) <= 2e-4


@pytest.mark.parametrize("qt", [O.TYPE_Q8_0, O.TYPE_Q8_1, O.TYPE_Q8_K])
@pytest.mark.parametrize("rounding", [O.ROUND_REF, O.ROUND_X86])
def test_quantizers_over_all_exponents(mx, be, qt, rounding):
    """Bit for bit from the smallest block maxima whose reciprocal is finite to 2^127, one exponent a row."""
    if qt == O.TYPE_Q8_K and rounding == O.ROUND_X86:
        pytest.skip("Q8_K has a single rounding")
    K, es = 512, np.arange(-117, 127)
    base = O.fill_normal(43, len(es), K)
    base /= np.abs(base).max(axis=1, keepdims=True) * np.float32(1.01)  # the largest below 1
    x = np.ldexp(base, es[:, None] + 1).astype(np.float32)
    assert np.all(np.isfinite(x))
    out = be.quantize_act(qt, rounding, be.tensor(mx.F32, (K, len(es)), x), K, len(es))
    be.sync()
    got = out.get_bytes()[: O.row_size(qt, K) * len(es)].reshape(len(es), -1)
    want = O.quantize_rows(qt, x, rounding)
    assert np.array_equal(got, want), f"rows differing: {es[(got != want).any(axis=1)]}"


def q8_blocks(x, rounding):
    """Blocks [n, 32] as the device quantizes them, with IEEE divisions: d (fp16) and codes. Casts to int saturate, NaN is 0
    (the C source leaves those to the machine)."""
    f = np.float32
    with np.errstate(all="ignore"):
        a = np.abs(x).max(1, keepdims=True)
        d = a / f(127)
        if rounding == O.ROUND_X86:
            q = np.rint(x * np.where(a != 0, f(127) / a, f(0)))
        else:
            v = x * np.where(d != 0, f(1) / d, f(0))  # roundf: half away from zero, exact in double
            q = np.where(np.isfinite(v), np.copysign(np.floor(np.abs(v).astype(np.float64) + 0.5), v), v)
        q = np.nan_to_num(q.astype(np.float64), nan=0, posinf=2.0 ** 31 - 1, neginf=-2.0 ** 31)
        return d[:, 0].astype(np.float16), np.clip(q, -2.0 ** 31, 2.0 ** 31 - 1).astype(np.int64).astype(np.int8)


def q8_device(mx, be, x, rounding):
    out = be.quantize_act(O.TYPE_Q8_0, rounding, be.tensor(mx.F32, (x.size,), x), x.size, 1)
    be.sync()
    b = out.get_bytes()[:34 * len(x)].reshape(-1, 34)
    return b[:, :2].copy().view(np.float16)[:, 0], b[:, 2:].view(np.int8)


ROUNDINGS = pytest.mark.parametrize("rounding", [O.ROUND_REF, O.ROUND_X86], ids=["ref", "x86"])


@ROUNDINGS
def test_q8_0_over_every_mantissa(mx, be, rounding):
    """A block for each float of [1, 2) as its largest, the others near the halves between codes: there the last bit of the
    reciprocal shows."""
    n = 1 << 20
    half = (np.arange(32) * 4 % 127 + 0.5).astype(np.float32) / np.float32(127) * np.where(np.arange(32) % 2, -1, 1).astype(np.float32)
    half[0] = 1
    for part in range(8):
        v = (np.arange(n, dtype=np.uint32) + np.uint32(0x3F800000 + part * n)).view(np.float32)
        x = v[:, None] * half
        d, q = q8_device(mx, be, x, rounding)
        want_d, want_q = q8_blocks(x, rounding)
        assert np.array_equal(d.view(np.uint16), want_d.view(np.uint16)) and np.array_equal(q, want_q)


@ROUNDINGS
def test_q8_0_at_the_ends(mx, be, rounding):
    """Zero blocks, subnormal maxima (whose reciprocal overflows, and past that), mantissas of all ones and of one bit at
    every exponent, the largest float, infinities."""
    g = np.random.default_rng(3)
    e = np.arange(0, 255, dtype=np.uint32) << 23
    top = np.concatenate([np.arange(1, 300, dtype=np.uint32), 1 << np.arange(23, dtype=np.uint32), e, e + 1, e + 0x7FFFFF, e + 0x400000,
                          np.array([0, 0x7F7FFFFF, 0x7F800000, 0x7F800000], np.uint32)]).view(np.float32)
    x = (g.uniform(-1, 1, (len(top), 32)) * np.where(np.isfinite(top), top, 1)[:, None]).astype(np.float32)
    x[np.arange(len(top)), g.integers(0, 32, len(top))] = top * g.choice([-1, 1], len(top)).astype(np.float32)
    x[0] *= -0.0
    d, q = q8_device(mx, be, x, rounding)
    want_d, want_q = q8_blocks(x, rounding)
    assert np.array_equal(d.view(np.uint16), want_d.view(np.uint16))
    assert np.array_equal(q, want_q), top[(q != want_q).any(1)]


def test_q8_k_over_every_mantissa(mx, be):
    """d = 1 / (-127 / largest) of Q8_K blocks, fp32, for each float of [1, 2) and, at every exponent, a few mantissas. The
    blocks overlap: rows of 256 floats, 16 bytes apart, of values that descend, each block's first its largest."""
    def check(v):  # descending
        x = np.zeros(4 * len(v) + 256, np.float32)
        x[:4 * len(v):4] = v
        X = be.tensor(mx.F32, (x.size,), x)
        X.desc.nb[1] = 16
        out = be.quantize_act(O.TYPE_Q8_K, O.ROUND_REF, X, 256, len(v))
        be.sync()
        d = out.get_bytes()[:292 * len(v)].reshape(-1, 292)[:, :4].copy().view(np.float32)[:, 0]
        with np.errstate(all="ignore"):
            want = np.float32(1) / (np.float32(-127) / v)
        assert np.array_equal(d.view(np.uint32), want.view(np.uint32)), v[d.view(np.uint32) != want.view(np.uint32)]

    for top in range(0x3FFFFFFF, 0x3F7FFFFF, -65535):  # (rows are grid.y)
        check(np.arange(top, max(top - 65535, 0x3F7FFFFF), -1, dtype=np.uint32).view(np.float32))
    m = np.array([0, 1, 2, 3, 0x2AAAAA, 0x3FFFFF, 0x400000, 0x555555, 0x7FFFFD, 0x7FFFFE, 0x7FFFFF], np.uint32)
    all_e = np.sort(np.concatenate([(np.arange(0, 255, dtype=np.uint32)[:, None] << np.uint32(23) | m).ravel(), [0x7F800000]]))
    check(all_e[1:][::-1].astype(np.uint32).view(np.float32).copy())
