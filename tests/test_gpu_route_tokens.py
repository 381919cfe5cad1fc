"""GPU parity of the routing of chunks and of the general path (pf_k_route_tokens): several tokens of a workgroup whose best logits
are too close, at one, two, three and sixteen tokens a workgroup."""
import numpy as np
import pytest

import picoforge_amd as pf
from picoforge_amd import abi

from helpers import assert_parity, forward_with, make_layer_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [33, 257, 600, 3841])
@pytest.mark.parametrize("clones", [2, 20])
def test_flagged_tokens_of_a_workgroup(product, oracle, tokens, clones):
    """Router rows in groups of `clones` that differ by an ulp in a place: nearly every token is routed again, two clones with
    the candidates of several tokens side by side in the chain's lanes, twenty with more candidates than lanes."""
    print(f"case route tokens {tokens}, groups of {clones}", flush=True)
    cfg = abi.moe_config(256, 64, 6, 256, 256)
    weights, few = make_layer_inputs(cfg, abi.GGUF_Q4_K, 97, seed=tokens + clones)
    router = weights.raw[0].view(np.float32).reshape(64, 256)
    for e in range(64):
        router[e] = router[e - e % clones]
        router[e, 3 * e] = np.nextafter(router[e, 3 * e], np.float32(10))
    want = forward_with(oracle, cfg, weights, few)
    row = np.arange(tokens) % 97
    want = [a[row] for a in want]
    with pf.MoeLayer(product, cfg, weights, tokens) as layer:
        layer.force_grouped()
        _, y, ids, w = layer.forward(few[row])
        assert_parity(y, ids, w, *want, label="chunk")
        assert layer.serial_order_reroutes() > tokens // 2
        if tokens <= 600:
            layer.force_general()
            _, y, ids, w = layer.forward(few[row])
            assert_parity(y, ids, w, *want, label="general kernels")
