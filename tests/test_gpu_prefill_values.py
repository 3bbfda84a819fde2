"""The prefill attention at the edges of its split: token groups that do not
divide the chunk, position groups of 32 cut short, few tokens (a workgroup per
head and token, or one head per thread) and many (four heads per thread), each
cache type and pages smaller than a position group.  Bit-exact with the oracle's
token-by-token decode.
"""
import numpy as np
import pytest

import inputs as I
import quantr_amd as Q
from conftest import assert_bits_equal
from oracle import ORDER_AVX2
from test_gpu_prefill import make_decoder, oracle_prompt, prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_type,page,n_kv,tokens,chunk", [
    (Q.KV_Q8_0, 64, 1, 37, 37), (Q.KV_F16, 16, 1, 33, 5), (Q.KV_F32, 32, 2, 65, 32),
    (Q.KV_Q8_0, 16, 2, 31, 31), (Q.KV_Q8_0, 256, 1, 1030, 1024)],
    ids=["q8_37", "f16_chunks5", "f32_gqa4", "q8_gqa4_31", "q8_wide_1030"])
def test_prefill_value_edges(dev, oracle, kv_type, page, n_kv, tokens, chunk):
    m = I.qwen3_small_model(n_layers=1, seq_len=max(64, tokens + 2), n_kv_heads=n_kv)
    toks = np.random.default_rng(53).integers(0, m["vocab"], size=tokens).astype(np.int32)
    want_lg, want_xs, _, _ = oracle_prompt(oracle, m, toks, kv_type, ORDER_AVX2)
    d = make_decoder(dev, m, kv_type, ORDER_AVX2, page=page)
    lg, x = prefill(dev, d, m, toks, chunk=chunk)
    d.close()
    assert_bits_equal(lg, want_lg, "prefill logits")
    assert_bits_equal(x, want_xs[-1], "prefill residual")
