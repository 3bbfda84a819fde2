"""The tiled and row-major GEMV of several tokens on the sides of the lines
between a row of workgroups per token, per two tokens, and all tokens per
workgroup (short and long rows, few and many tiles, a last workgroup without
tiles), with strided tokens and outputs.  Bit-exact with the oracle.
"""
import numpy as np
import pytest

import quantr_amd as Q
from conftest import bits
from quantr_amd import synth

pytestmark = pytest.mark.gpu

SHAPES = [(8192, 2048), (8200, 2048), (8, 512), (16008, 512), (32008, 512), (1032, 4608),
          (5640, 4608)]


@pytest.mark.parametrize("layout", ["tiled", "rows"])
@pytest.mark.parametrize("n,D", SHAPES)
@pytest.mark.parametrize("qtype", [Q.TYPE_Q8_0, Q.TYPE_Q4_K, Q.TYPE_Q5_K, Q.TYPE_Q6_K])
def test_token_rows(dev, oracle, qtype, n, D, layout):
    W = synth.weights(700 + qtype, n, D, qtype)
    xs, ys = D + 4, n + 3
    X = synth.normal(701, (8, xs))
    X[:, D:] = np.nan
    want = oracle.matmul_q_fused(np.ascontiguousarray(X[:, :D]), W, qtype, n, D, threads=16)
    wb, xb, t = dev.upload(W), dev.upload(X), qtype
    if layout == "tiled":
        tb = dev.alloc(W.nbytes)
        dev.tile(qtype, wb.ptr, tb.ptr, n, D)
        wb, t = tb, qtype | Q.TILED
    for nt in (2, 3, 4, 8):
        if nt == 8 and layout == "rows" and D > 2048:
            continue  # past the call's limit on the tokens' length
        yb = dev.upload(np.full((nt, ys), 7.0, np.float32))
        dev.gemv(t, wb.ptr, xb.ptr, yb.ptr, n, D, nt, xstride=xs, ystride=ys)
        got = dev.download(yb, (nt, ys), np.float32)
        assert (bits(got[:, :n]) == bits(want.reshape(8, n)[:nt])).all(), nt
        assert (got[:, n:] == 7.0).all(), nt
