"""The int8 Q8_0 GEMM at the edges of its ring, tiles and splits on MI355X against the oracle: exact block integers, summed
in fp32 in another order over at most K / 32 = 128 blocks, about 1e-6 of a row's largest output; 2e-5 shows a lost term.
"""
import numpy as np
import pytest

import oracle as O
from helpers import rel_err

pytestmark = pytest.mark.gpu


# stages 1 .. 7 (around the ring's three and two), M and N at and one past 32 and 64, one row, more than a tile; the last
# two take the 64 x 128 tile, a split K and a ragged group
@pytest.mark.parametrize("K", [128, 256, 384, 512, 640, 896])
@pytest.mark.parametrize("M,Ns", [(9, (1,)), (32, (33, 64)), (65, (65, 127, 1)), (200, (129,)), (64, (65536, 33))])
def test_stages_and_tiles(mx, be, K, M, Ns):
    product(mx, be, K, M, Ns)


@pytest.mark.parametrize("K,M,Ns", [(4096, 33, (70, 130)), (4224, 100, (256,)), (2176, 513, (8200,))])
def test_splits(mx, be, K, M, Ns):
    product(mx, be, K, M, Ns)


def product(mx, be, K, M, Ns):
    ws = [O.quantize_chunk(O.TYPE_Q8_0, O.fill_normal(51 + i, n, K, 0.0, 0.05)) for i, n in enumerate(Ns)]
    x = O.fill_normal(53 + M, M, K)
    W = [be.tensor(O.TYPE_Q8_0, (K, n), w) for n, w in zip(Ns, ws)]
    Y = [be.tensor(mx.F32, (n, M)) for n in Ns]
    be.mul_mat_group(W, be.tensor(mx.F32, (K, M), x), Y)
    be.sync()
    for n, w, y in zip(Ns, ws, Y):
        assert rel_err(y.numpy().reshape(M, n), O.mul_mat(O.TYPE_Q8_0, w, x)) <= 2e-5
