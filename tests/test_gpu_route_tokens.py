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


@pytest.mark.parametrize("clones", [2, 20])
def test_every_rerouting_routes_alike(product, oracle, clones):
    """The same flagged tokens one by one (pf_route_fix_block, inside the decode kernels), sixteen at a time (pf_fix_token, in a launch of
    its own), in a chunk and on the general kernels (pf_k_route_tokens): the candidates' order, the doubt about it and the long way are
    written more than once, and a token's routes are the reference's by every one of them."""
    print(f"case re-routings alike, groups of {clones}", flush=True)
    cfg = abi.moe_config(512, 64, 6, 256, 256)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, 64, seed=7 + clones)
    router = weights.raw[0].view(np.float32).reshape(64, 512)
    for e in range(64):
        router[e] = router[e - e % clones]
        router[e, 7 * e] = np.nextafter(router[e, 7 * e], np.float32(10))
    _, ids, w = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, 64) as layer:
        routed, before = {}, 0
        for name, step in (("one by one", 1), ("sixteen", 16), ("chunk", 64), ("general", 64)):
            layer.force_grouped(name == "chunk")
            layer.force_general(name == "general")
            parts = [layer.forward(x[t:t + step])[2:] for t in range(0, 64, step)]
            routed[name] = [np.concatenate(p) for p in zip(*parts)]
            again = layer.serial_order_reroutes() - before
            before += again
            print(f"  {name}: {again} re-routed", flush=True)
            assert again > 32, "the case must be full of near ties"
    for name, (i, v) in routed.items():
        np.testing.assert_array_equal(i, ids, err_msg=name)
        np.testing.assert_allclose(v, w, rtol=2e-6, err_msg=name)
