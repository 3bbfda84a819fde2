"""The fp32 terms of the int8 MFMA products at the edges of their fused form:
block sums whose product with a min needs more than 24 bits, and block scales
that are not finite, beside ordinary blocks.  Bit-exact with the oracle (the
sum of a row that meets a NaN has no bits to compare, only to be NaN too).
"""
import numpy as np
import pytest

import quantr_amd as Q
from conftest import bits
from oracle import ORDER_SEQ, Oracle
from quantr_amd import synth

pytestmark = pytest.mark.gpu

N, D, T = 83, 768, 37  # rows past a 64-row block, three stages, pairs past two 16-pair tiles


def make(kind, qtype):
    W = synth.weights(300 + qtype, N, D, qtype)
    x = synth.normal(310, (T, D))
    be, bb = synth.BLOCK_ELEMS[qtype], synth.BLOCK_BYTES[qtype]
    blk = W.reshape(N, D // be, bb)
    rng = np.random.default_rng(5)
    if kind == "bsum":
        # whole blocks at +amax / -amax: block sums of +-4064, and near the
        # largest that stays exact (2732)
        x[::3, :256] = 1.0
        x[1::3, 256:512] = -0.25
        x[2::3] = np.where(np.arange(D) % 32 < 27, 1.0, -0.9).astype(np.float32)
        if qtype in (Q.TYPE_Q4_K, Q.TYPE_Q5_K):  # mins of 3 times an odd half
            blk[..., 2] |= 1
            blk[..., 2] |= 0xFE
            blk[..., 4:12] |= 0xC0
    elif kind == "nonfinite":
        at = 0 if qtype in (Q.TYPE_Q8_0, Q.TYPE_Q4_K, Q.TYPE_Q5_K) else 208
        for r, h in ((3, 0x7C00), (17, 0xFC00), (40, 0x7E01), (82, 0x7C00)):
            blk[r, rng.integers(D // be), at:at + 2] = np.frombuffer(np.uint16(h).tobytes(), np.uint8)
        if qtype in (Q.TYPE_Q4_K, Q.TYPE_Q5_K):
            blk[50, 1, 2:4] = np.frombuffer(np.uint16(0x7C00).tobytes(), np.uint8)
        # a half's largest and subnormal scales stay on the fused form
        blk[5, 0, at:at + 2] = np.frombuffer(np.uint16(0x7BFF).tobytes(), np.uint8)
        blk[6, 0, at:at + 2] = np.frombuffer(np.uint16(0x83FF).tobytes(), np.uint8)
    return blk.reshape(W.shape), x


@pytest.mark.parametrize("kind", ["plain", "bsum", "nonfinite"])
@pytest.mark.parametrize("qtype", [Q.TYPE_Q8_0, Q.TYPE_Q4_K, Q.TYPE_Q5_K, Q.TYPE_Q6_K])
@pytest.mark.parametrize("nt", [3, 16, T], ids=["skinny", "one_tile", "tiles"])
def test_term_edges(dev, oracle, kind, qtype, nt):
    W, x = make(kind, qtype)
    x = x[:nt]
    wb, xb, yb = dev.upload(W), dev.upload(x), dev.alloc(nt * N * 4)
    dev.gemv_rows(qtype, wb.ptr, xb.ptr, yb.ptr, N, D, nt)
    got = dev.download(yb, (nt, N), np.float32)
    with np.errstate(invalid="ignore"):
        want = oracle.matmul_q_fused(x, W, qtype, N, D, threads=4)
    nan = np.isnan(want)
    assert (np.isnan(got) == nan).all()
    assert (bits(got)[~nan] == bits(want)[~nan]).all()
    if kind != "nonfinite":
        assert not nan.any()


E, K, HIDDEN = 8, 2, 288  # gate/up: 16 rows of each matrix per wave, a last tile half full


@pytest.mark.parametrize("kind", ["bsum", "nonfinite"])
@pytest.mark.parametrize("ut,dt", [(Q.TYPE_Q4_K, Q.TYPE_Q8_0), (Q.TYPE_Q5_K, Q.TYPE_Q8_0),
                                   (Q.TYPE_Q6_K, Q.TYPE_Q8_0), (Q.TYPE_Q8_0, Q.TYPE_Q8_0)])
@pytest.mark.parametrize("nt", [16, 80], ids=["items16", "items32"])
def test_term_edges_moe(dev, oracle, kind, ut, dt, nt):
    """The same edges in the gate/up product (two matrices, their outputs as the down
    product's records) and in the routed down product, with 16- and 32-pair items:
    in each expert some rows take the fused form and some do not."""
    rng = np.random.default_rng(7)
    be, bb = synth.BLOCK_ELEMS[ut], synth.BLOCK_BYTES[ut]
    up = synth.weights(320 + ut, E * HIDDEN, D, ut).reshape(E, HIDDEN, D // be, bb)
    gate = synth.weights(330 + ut, E * HIDDEN, D, ut).reshape(E, HIDDEN, D // be, bb)
    down = synth.weights(340 + dt, E * D, HIDDEN, dt).reshape(E, D, -1)
    router = synth.normal(350, (E, D), 0.05)
    x, xb = synth.normal(351, (nt, D)), synth.normal(352, (nt, D))
    if kind == "bsum":
        xb[::3, :256] = 1.0
        xb[1::3, 256:512] = -0.25
        xb[2::6] = np.where(np.arange(D) % 32 < 27, 1.0, -0.9).astype(np.float32)
        if ut in (Q.TYPE_Q4_K, Q.TYPE_Q5_K):  # mins of 3 times an odd half
            for w in (up, gate):
                w[..., 2] = 0xFF
                w[..., 4:12] |= 0xC0
    else:
        at = 208 if ut == Q.TYPE_Q6_K else 0
        for e in range(0, E, 2):
            for w, r, h in ((up, 3, 0x7C00), (gate, 19, 0xFC00), (up, 287, 0x7E01)):
                w[e, r, rng.integers(D // be), at:at + 2] = np.frombuffer(np.uint16(h).tobytes(),
                                                                          np.uint8)
        down[1, 5, 34:36] = np.frombuffer(np.uint16(0x7C00).tobytes(), np.uint8)
        down[3, 700, 0:2] = np.frombuffer(np.uint16(0xFE00).tobytes(), np.uint8)
    bufs = [dev.upload(a) for a in (router, up, gate, down)]
    L = Q.MoeLayer(D, HIDDEN, E, K, *[b.ptr for b in bufs], ut, ut, dt)
    xd, xbd = dev.upload(x), dev.upload(xb)
    dev.set_moe_path(Q.MOE_PATH_MFMA)
    try:
        dev.moe_forward(L, xd.ptr, xbd.ptr, nt, ORDER_SEQ)
        got = dev.download(xd, (nt, D), np.float32)
    finally:
        dev.set_moe_path(Q.MOE_PATH_AUTO)
    keep = []
    OL = Oracle.make_layer(keep, D, HIDDEN, E, K, router, up, ut, gate, ut, down, dt)
    with np.errstate(all="ignore"):
        want, _, _ = oracle.moe_forward(x, xb, OL, order=ORDER_SEQ, dot_order=ORDER_SEQ)
    nan = np.isnan(want)
    assert (np.isnan(got) == nan).all()
    assert (bits(got)[~nan] == bits(want)[~nan]).all()
    assert (~nan).any() and nan.any() == (kind == "nonfinite")
