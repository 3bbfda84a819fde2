"""The tiled and row-major GEMV of several tokens on both sides of the line
between a row of workgroups per token (or two) and all tokens per workgroup:
1024 and 1025 tiles of 8 rows, with strided tokens and outputs.  Bit-exact with
the oracle.
"""
import numpy as np
import pytest

import quantr_amd as Q
from conftest import bits
from quantr_amd import synth

pytestmark = pytest.mark.gpu

D = 2048


@pytest.mark.parametrize("layout", ["tiled", "rows"])
@pytest.mark.parametrize("n", [8192, 8200])
@pytest.mark.parametrize("qtype", [Q.TYPE_Q8_0, Q.TYPE_Q4_K, Q.TYPE_Q5_K, Q.TYPE_Q6_K])
def test_token_rows(dev, oracle, qtype, n, layout):
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
        yb = dev.upload(np.full((nt, ys), 7.0, np.float32))
        dev.gemv(t, wb.ptr, xb.ptr, yb.ptr, n, D, nt, xstride=xs, ystride=ys)
        got = dev.download(yb, (nt, ys), np.float32)
        assert (bits(got[:, :n]) == bits(want.reshape(8, n)[:nt])).all(), nt
        assert (got[:, n:] == 7.0).all(), nt
