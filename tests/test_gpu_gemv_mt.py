"""The multi-token row-major Q8_0 / Q6_K GEMV (and Q4_K / Q5_K at eight tokens)
at the edges of its tiles and stages: rows around 16, rows whose stages start
off a 16-byte boundary, matrices ending inside one, a last stage of 1 to 7
blocks, fewer stages than waves, strided tokens and outputs.  Bit-exact with
the oracle in every dot order.
"""
import numpy as np
import pytest

import quantr_amd as Q
from conftest import bits
from oracle import ORDER_AVX2, ORDER_AVX512, ORDER_SEQ
from quantr_amd import synth

pytestmark = pytest.mark.gpu

Q8_SHAPES = [(1, 32), (15, 64), (16, 256), (17, 288), (33, 608), (83, 2144), (4100, 96),
             (256, 2144), (257, 2144)]  # the last two: a line of the route (as many rows as CUs)
K_SHAPES = [(1, 256), (17, 512), (333, 768), (40, 1792), (4099, 2304),
            (8176, 768), (8177, 768), (256, 5632), (257, 5632)]  # lines of the route
CASES = ([(Q.TYPE_Q8_0, o, n, d) for o in (ORDER_SEQ, ORDER_AVX2, ORDER_AVX512) for n, d in Q8_SHAPES]
         + [(Q.TYPE_Q6_K, ORDER_SEQ, n, d) for n, d in K_SHAPES]
         + [(t, ORDER_SEQ, n, d) for t in (Q.TYPE_Q4_K, Q.TYPE_Q5_K) for n, d in K_SHAPES[:3]])


@pytest.mark.parametrize("nt", [2, 3, 4, 8])
@pytest.mark.parametrize("qtype,order,n,d", CASES)
def test_multi_token_edges(dev, oracle, qtype, order, n, d, nt):
    if nt == 8 and d > 2144:
        d = 2048 if qtype != Q.TYPE_Q8_0 else d
    W = synth.weights(4000 + n + d, n, d, qtype)
    xs, ys = d + 4, n + 3  # strides beyond the sizes
    X = synth.normal(4100 + nt, (nt, xs))
    X[:, d:] = np.nan
    if d >= 96:
        X[0, 32:64] = 0.0  # a block without a scale
    wb, xb = dev.upload(W), dev.upload(X)
    yb = dev.upload(np.full((nt, ys), 7.0, np.float32))
    dev.gemv(qtype, wb.ptr, xb.ptr, yb.ptr, n, d, nt, xstride=xs, ystride=ys, order=order)
    got = dev.download(yb, (nt, ys), np.float32)
    want = oracle.matmul_q_fused(np.ascontiguousarray(X[:, :d]), W, qtype, n, d, threads=8,
                                 order=order).reshape(nt, n)
    assert (bits(got[:, :n]) == bits(want)).all()
    assert (got[:, n:] == 7.0).all()
