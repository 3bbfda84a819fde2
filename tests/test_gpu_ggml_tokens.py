"""The llama.cpp-layout GEMV of several tokens on both sides of its split: each
token its own row of workgroups (few tiles), two, or several tokens per workgroup
and two rows of four (many tiles), with strided tokens and outputs.  Bit-exact
with the oracle.
"""
import numpy as np
import pytest

import ggml_blocks as GB
import quantr_amd as Q
from conftest import bits
from quantr_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [2, 3, 4, 8])
@pytest.mark.parametrize("n,d", [(65, 768), (24601, 2048), (50001, 512)])
@pytest.mark.parametrize("qtype", [GB.Q4_K, GB.Q5_K, GB.Q6_K])
def test_ggml_tokens(dev, oracle, qtype, n, d, nt):
    W = GB.random_rows(90 + qtype, qtype, n, d)
    xs, ys = d + 8, n + 3  # strides beyond the sizes
    X = synth.normal(600 + nt, (nt, xs))
    X[:, d:] = np.nan
    wb, xb = dev.upload(W), dev.upload(X)
    yb = dev.upload(np.full((nt, ys), 7.0, np.float32))
    dev.gemv(qtype | Q.GGML, wb.ptr, xb.ptr, yb.ptr, n, d, nt, xstride=xs, ystride=ys)
    got = dev.download(yb, (nt, ys), np.float32)
    want = oracle.ggml_matmul(np.ascontiguousarray(X[:, :d]), W, qtype, n, d)
    assert (bits(got[:, :n]) == bits(want.reshape(nt, n))).all()
    assert (got[:, n:] == 7.0).all()
