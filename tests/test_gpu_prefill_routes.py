"""The prefill attention's routes, on both sides of each line between them: one
workgroup per head and token, or softmax and values as two launches (few and many
tokens; extents up to 16384), the softmax's 4, 2 or 1 rows per workgroup (extents
4096 and 8192), one, two or four query heads per thread (by tokens, head_dim 64 to
256 and the query heads of a kv head).  Two chunks of one prompt take the two sides.
Bit-exact with the oracle's token-by-token decode.
"""
import numpy as np
import pytest

import inputs as I
import quantr_amd as Q
from conftest import assert_bits_equal
from oracle import ORDER_AVX2, ORDER_AVX512
from test_gpu_prefill import make_decoder, prefill

pytestmark = pytest.mark.gpu


def _model(heads, kv_heads, hd, seq_len):
    m = I.qwen3_small_model(n_layers=1, seq_len=seq_len)
    m.update(n_heads=heads, n_kv_heads=kv_heads, head_dim=hd)
    dim, wt = m["dim"], m["wtype"]
    m["layers"][0].update(wq=I._rows(9601, wt[0], heads * hd, dim),
                          wk=I._rows(9602, wt[1], kv_heads * hd, dim),
                          wv=I._rows(9603, wt[2], kv_heads * hd, dim),
                          wo=I._rows(9604, wt[3], dim, heads * hd))
    return m


def _run(dev, oracle, m, kv_type, page, pos0, chunks):
    """The chunks' tokens from position pos0 of a cache of random rows."""
    kvd, n = m["n_kv_heads"] * m["head_dim"], sum(chunks)
    rng = np.random.default_rng(61)
    toks = rng.integers(0, m["vocab"], size=n).astype(np.int32)
    rs = oracle.kv_row_bytes(kv_type, kvd)
    kc = np.zeros((1, m["seq_len"], rs), np.uint8)
    vc = np.zeros_like(kc)
    d = make_decoder(dev, m, kv_type, ORDER_AVX2, page=page)
    if pos0:
        kv = rng.standard_normal((2, pos0, kvd)).astype(np.float32)
        kc[0, :pos0], vc[0, :pos0] = oracle.kv_rows(kv[0], kv_type), oracle.kv_rows(kv[1], kv_type)
        kb, vb = dev.upload(kv[0]), dev.upload(kv[1])
        d.kv_write(0, 0, pos0, kb.ptr, vb.ptr)
    print("prefill routes hd %d heads %d/%d kv %d pos %d chunks %s" % (
        m["head_dim"], m["n_heads"], m["n_kv_heads"], kv_type, pos0, chunks), flush=True)
    got, x, at = [], None, 0
    for c in chunks:
        lg, x = prefill(dev, d, m, toks[at:at + c], pos0=pos0 + at, chunk=c)
        got.append(lg)
        at += c
    d.close()
    want, xs = oracle.forward_cached(m, kc.reshape(-1), vc.reshape(-1), [int(t) for t in toks], pos0,
                                     ORDER_AVX2, kv_type)
    assert_bits_equal(np.concatenate(got), want, "prefill logits")
    assert_bits_equal(x, xs[-1], "prefill residual")


# (heads, kv heads, head_dim, cache, chunks): at 256 CUs the first chunk lies
# past a line of the route, the second on it
ROUTES = [
    (8, 1, 128, Q.KV_Q8_0, (65, 64)),    # two launches (two heads per thread) / per head
    (8, 1, 128, Q.KV_F16, (65, 64)),
    (8, 1, 192, Q.KV_Q8_0, (65, 64)),    # four heads per thread / per head
    (8, 1, 256, Q.KV_F16, (65, 64)),
    (8, 2, 256, Q.KV_Q8_0, (33, 32)),    # 4:1, two heads per thread / per head
    (8, 2, 192, Q.KV_F16, (33, 32)),
    (32, 4, 64, Q.KV_Q8_0, (129, 128)),  # two heads per thread / one
    (32, 4, 64, Q.KV_F16, (512, 3)),     # four heads per thread / one
    (8, 2, 64, Q.KV_Q8_0, (7, 2)),       # 4:1, one head per thread, two tokens a workgroup
    (16, 4, 64, Q.KV_F16, (258, 256)),   # 4:1, two heads per thread / one
    (16, 4, 128, Q.KV_F16, (129, 128)),
    (16, 4, 64, Q.KV_F32, (129, 128)),   # fp32 rows: two launches / per head
    (32, 4, 128, Q.KV_F32, (129, 128)),
    (32, 4, 192, Q.KV_F32, (129, 1)),
]


@pytest.mark.parametrize("heads,kv_heads,hd,kv_type,chunks", ROUTES,
                         ids=["%d_%d_hd%d_kv%d_%d" % (r[:4] + r[4][:1]) for r in ROUTES])
def test_prefill_routes(dev, oracle, heads, kv_heads, hd, kv_type, chunks):
    m = _model(heads, kv_heads, hd, sum(chunks) + 8)
    _run(dev, oracle, m, kv_type, 16, 0, chunks)


@pytest.mark.parametrize("kv_type", [Q.KV_Q8_0, Q.KV_F16], ids=["q8", "f16"])
@pytest.mark.parametrize("extent", [4096, 8192, 16384])
def test_prefill_extent_lines(dev, oracle, extent, kv_type):
    """Chunks ending at the extent and one position past it: the softmax's rows per
    workgroup change (4096, 8192), or the two launches end (16384)."""
    m = _model(8, 1, 64, extent + 16)
    _run(dev, oracle, m, kv_type, 256, extent - 3, (3, 1, 2))


def test_prefill_wide_lane_order_rows(dev, oracle):
    """A k projection of as many rows as CUs, 8192 wide, Q8_0 in the AVX-512 order:
    three tokens of it are more than the general GEMV's LDS holds."""
    m = I.qwen3_small_model(n_layers=1, seq_len=16)
    dim, H, hd, E, hidden = 8192, 2, 128, 2, 256
    m.update(dim=dim, n_heads=H, n_kv_heads=H, head_dim=hd, E=E, K=1, hidden=hidden)
    wt = m["wtype"]
    m["tok_embd"] = I._rows(9701, m["tok_type"], m["vocab"], dim)
    m["wcls"] = I._rows(9702, m["wcls_type"], m["vocab"], dim)
    m["rms_final"] = (1.0 + I.activations(9703, 1, dim, std=0.1)[0]).astype(np.float32)
    m["layers"] = [dict(
        rms_att=(1.0 + I.activations(9704, 1, dim, std=0.1)[0]).astype(np.float32),
        rms_ffn=(1.0 + I.activations(9705, 1, dim, std=0.1)[0]).astype(np.float32),
        wq=I._rows(9706, wt[0], H * hd, dim), wk=I._rows(9707, wt[1], H * hd, dim),
        wv=I._rows(9708, wt[2], H * hd, dim), wo=I._rows(9709, wt[3], dim, H * hd),
        router=I.activations(9710, E, dim, std=0.05),
        up=I.blocks(9711, m["up_type"], E * hidden * (dim // 256)),
        gate=I.blocks(9712, m["up_type"], E * hidden * (dim // 256)),
        down=I.blocks(9713, m["down_type"], E * dim * (hidden // 256)))]
    toks = np.array([3, 7, 11], np.int32)
    print("prefill routes wide rows", flush=True)
    d = make_decoder(dev, m, Q.KV_F32, ORDER_AVX512, page=16)
    lg, x = prefill(dev, d, m, toks)
    d.close()
    kvb = oracle.kv_row_bytes(Q.KV_F32, H * hd)
    kc, vc = np.zeros((2, m["seq_len"], kvb), np.uint8)
    want, xs = oracle.forward_cached(m, kc.reshape(-1), vc.reshape(-1), [int(t) for t in toks], 0,
                                     ORDER_AVX512, Q.KV_F32)
    assert_bits_equal(lg, want, "prefill logits")
    assert_bits_equal(x, xs[-1], "prefill residual")
