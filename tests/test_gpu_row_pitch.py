"""Activation rows far apart: every kernel family takes them as it takes dense rows, with the same bits."""
import ctypes as C

import numpy as np
import pytest

import picoforge_amd as pf
from picoforge_amd import abi

from helpers import make_layer_inputs

pytestmark = pytest.mark.gpu

FAR = 1 << 27   # floats from a row to the next: eight rows are more than 32 bits of bytes


@pytest.mark.parametrize("fmt,tokens,family", [(abi.GGUF_Q4_K, 3, 1), ("q2", 11, 3), (abi.GGUF_Q4_K, 9, 2)])
def test_rows_far_apart(product, fmt, tokens, family):
    print(f"case rows far apart, {fmt} tokens={tokens} family={family}", flush=True)
    hidden, hip = 512, product.hip
    cfg = abi.moe_config(hidden, 32, 6, 256, 256)
    weights, x = make_layer_inputs(cfg, fmt, tokens, seed=tokens)
    with pf.MoeLayer(product, cfg, weights, tokens) as layer:
        if family == 2:
            layer.force_grouped()
        moe, work = layer.device_handles()
        assert hip.moe_kernel_family(moe, work, tokens) == family
        d_x, d_y, far = hip.to_device(x), hip.to_device(np.zeros_like(x)), C.c_void_p()
        hip.check(hip.malloc(C.byref(far), 4 * ((tokens - 1) * FAR + hidden)), "malloc")
        try:
            for t in range(tokens):
                hip.check(hip.memcpy_h2d(C.c_void_p(far.value + 4 * FAR * t), x[t].ctypes.data, 4 * hidden), "h2d")
            got = []
            for rows, pitch in ((d_x, hidden), (far, FAR)):
                hip.check(hip.moe_forward_device(moe, work, rows, pitch, d_y, hidden, tokens, None), "forward")
                hip.check(hip.synchronize(), "wait")
                got.append(hip.from_device(d_y, x.shape, np.float32))
        finally:
            for p in (d_x, d_y, far):
                hip.free(p)
    np.testing.assert_array_equal(got[0], got[1])


def test_rows_far_apart_of_a_layer_that_the_general_kernels_do_not_take(product):
    """(ten activation rows of 1792 values are more than those kernels' LDS)"""
    print("case rows far apart, wide layer", flush=True)
    hidden, hip = 512, product.hip
    cfg = abi.moe_config(hidden, 16, 10, 1792, 512)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, 1, seed=5)
    with pf.MoeLayer(product, cfg, weights, 1) as layer:
        moe, work = layer.device_handles()
        assert hip.moe_kernel_family(moe, work, 1) == 1
        d_x, d_y = hip.to_device(x), hip.to_device(np.zeros_like(x))
        try:
            hip.check(hip.moe_forward_device(moe, work, d_x, FAR, d_y, hidden, 1, None), "forward")
            hip.check(hip.synchronize(), "wait")
            assert np.isfinite(hip.from_device(d_y, x.shape, np.float32)).all()
        finally:
            hip.free(d_x)
            hip.free(d_y)
