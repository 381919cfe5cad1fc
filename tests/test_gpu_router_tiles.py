"""GPU parity of the prefill router's tiles (32 x 32, 32 x 64, 64 x 64 tokens by experts) against the CPU oracle, at counts of
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


@pytest.mark.parametrize("e,i,tokens", CASES)
def test_router_logits(product, e, i, tokens):
    """The logits themselves against 64 bits, on rows of very different sizes.  Bound: every product keeps 2^-23 of itself (the three
    products of parts that are left out), a logit is six products' sums a 16-column step of a wave's eighth of the row, at most twelve
    steps' roundings here, and seven more additions, each off by at most 2^-23 of the sum of the magnitudes."""
    hidden = 256
    cfg = abi.moe_config(hidden, e, 4, i, i)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, tokens, seed=e + tokens)
    scale = np.exp2(np.random.default_rng(e).integers(-60, 61, tokens)).astype(np.float32)
    scale[[0, tokens - 1]] = 1.0, 2.0 ** 100
    x = np.ascontiguousarray(x * scale[:, None])
    x[1, 7] = np.finfo(np.float32).max   # rounded to eight bits it would be infinite
    router = weights.raw[0].view(np.float32).reshape(e, hidden).astype(np.float64)
    want, size = x.astype(np.float64) @ router.T, np.abs(x.astype(np.float64)) @ np.abs(router.T)
    hip = product.hip
    with pf.MoeLayer(product, cfg, weights, tokens) as layer:
        moe, work = layer.device_handles()
        assert hip.moe_kernel_family(moe, work, tokens) == 2
        d_x, d_y = hip.to_device(x), hip.to_device(np.zeros_like(x))
        try:
            print(f"router logits e={e} tokens={tokens}", flush=True)
            hip.work_limit_kernels(work, 1)   # the first stage alone
            hip.check(hip.moe_forward_device(moe, work, d_x, hidden, d_y, hidden, tokens, None), "forward")
            hip.check(hip.synchronize(), "wait")
            got = hip.from_device(hip.work_logits(work), (tokens, e), np.float32)
        finally:
            hip.work_limit_kernels(work, 0)
            hip.free(d_x)
            hip.free(d_y)
    error = np.abs(got - want) / size
    print(f"largest error {error.max():.2e} of the magnitudes' sum", flush=True)
    assert error.max() <= (1 + 12 + 7) * 2.0 ** -23


@pytest.mark.parametrize("e,tokens", [(480, 600), (160, 1700), (480, 1700)])
def test_odd_number_of_expert_tiles(product, oracle, e, tokens):
    """Workgroups of two tiles of 32 experts with one tile left for the last of them."""
    print(f"case router tiles, odd e={e} tokens={tokens}", flush=True)
    cfg = abi.moe_config(256, e, 4, 256, 256)
    weights, few = make_layer_inputs(cfg, abi.GGUF_Q4_K, 97, seed=e)
    row = np.arange(tokens) % 97
    want = [a[row] for a in forward_with(oracle, cfg, weights, few)[:3]]
    with pf.MoeLayer(product, cfg, weights, tokens) as layer:
        layer.force_grouped()
        _, y, ids, w = layer.forward(few[row])
        assert_parity(y, ids, w, *want, label=f"e={e} T={tokens}")


def test_products_of_two_values(product):
    """Logits of one product each: what the parts that are not multiplied leave out.  Bound: with |m| <= 2^-8 and |l| <= 2^-17 of a value
    m l + l m + l l is at most 2^-24 (1 + 2^-10) of the product, the last sum is off by at most 2^-23, the five before it, of at most 2^-7
    of the product, together by less than 2^-27: 2^-24 + 2^-23 + 2^-26 covers them."""
    hidden, e, tokens = 256, 64, 96
    cfg = abi.moe_config(hidden, e, 4, 256, 256)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, tokens, seed=11)
    gen = np.random.default_rng(11)

    def values(n):   # any bits; just under a step of the upper eight; just under half of one
        any_bits = gen.integers(0x3f800000, 0x40000000, n)
        step = 0x3f800000 + (gen.integers(0, 8, n) << 16) + 0xff80 + gen.integers(0, 128, n)
        half = 0x3f800000 + (gen.integers(0, 8, n) << 16) + 0x7f80 + gen.integers(0, 128, n)
        bits = np.choose(np.arange(n) % 3, [any_bits, step, half]).astype(np.uint32)
        bits[0], bits[1] = 0x3f80ffff, 0x3f80ff80
        return bits.view(np.float32) * gen.choice([-1.0, 1.0], n).astype(np.float32)

    router = weights.raw[0].view(np.float32).reshape(e, hidden)
    x[:] = 0.0
    x[:, 37] = values(tokens) * np.exp2(gen.integers(-60, 61, tokens)).astype(np.float32)
    x[2:6, 37] = np.array([0x7f7fffff, 0xff7fffff, 0x7f7f8000, 0x7f7f7fff], np.uint32).view(np.float32)   # on either side of rounding to infinity
    router[:, 37] = values(e) * np.exp2(gen.integers(-12, -2, e)).astype(np.float32)
    want, hip = x[:, 37:38].astype(np.float64) * router[:, 37].astype(np.float64), product.hip
    with pf.MoeLayer(product, cfg, weights, tokens) as layer:
        layer.force_grouped()
        moe, work = layer.device_handles()
        d_x, d_y = hip.to_device(x), hip.to_device(np.zeros_like(x))
        try:
            print("router products of two values", flush=True)
            hip.work_limit_kernels(work, 1)
            hip.check(hip.moe_forward_device(moe, work, d_x, hidden, d_y, hidden, tokens, None), "forward")
            hip.check(hip.synchronize(), "wait")
            got = hip.from_device(hip.work_logits(work), (tokens, e), np.float32)
        finally:
            hip.work_limit_kernels(work, 0)
            hip.free(d_x)
            hip.free(d_y)
    error = np.abs(got / want - 1.0)
    print(f"largest error {error.max() * 2.0 ** 23:.3f} times 2^-23", flush=True)
    assert error.max() <= 2.0 ** -24 + 2.0 ** -23 + 2.0 ** -26
