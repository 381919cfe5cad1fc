"""GPU parity of the prefill router's tiles (32 x 32, 64 x 32, 64 x 64 tokens by experts) against the CPU oracle, at counts of
tokens and experts that are no whole tiles, with activation rows of up to 512 values and wider ones."""
import numpy as np
import pytest

import picoforge_amd as pf
from picoforge_amd import abi

from helpers import assert_parity, forward_with, make_layer_inputs

pytestmark = pytest.mark.gpu

# (experts, inner width, tokens): one tile size each, the widest row a wave keeps, and the shortest hidden row for eight waves
CASES = [(70, 256, 401), (500, 768, 701), (1000, 256, 801)]


@pytest.mark.parametrize("e,i,tokens", CASES)
def test_router_tiles(product, oracle, e, i, tokens):
    print(f"case router tiles e={e} i={i} tokens={tokens}", flush=True)
    cfg = abi.moe_config(256, e, 4, i, i)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, tokens, seed=e + tokens)
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, tokens) as layer:
        _, y, ids, w = layer.forward(x)
        assert_parity(y, ids, w, *want[:3], label=f"e={e} T={tokens}")
        np.testing.assert_array_equal(y, layer.forward(x)[1], err_msg="not deterministic")
