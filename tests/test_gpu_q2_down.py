"""GPU parity of the grouped product's Q2_K down projection (GemmBlock<PF_Q2_K> in pf_moe_prefill.hip): rows that end in half a
256-block or in a whole one, of one block to four and, beyond 1024 values, on the plain kernel; rows stored wider than they are used."""
import numpy as np
import pytest

import picoforge_amd as pf
from picoforge_amd import abi

from helpers import assert_parity, forward_with
from test_gpu_grouped import ROWS, steered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,i,physical,s", [
    (256, 128, 256, 128), (768, 256, 256, 384), (512, 384, 512, 128), (512, 384, 1024, 1024), (2560, 640, 768, 640), (256, 896, 1024, 128),
    (256, 1024, 1024, 256), (256, 1152, 1280, 256), (256, 640, 768, 1152),
])
def test_widths_of_down_rows(product, oracle, h, i, physical, s):
    print(f"case q2 down h={h} i={i} stored {physical} s={s}", flush=True)
    cfg = abi.moe_config(h, len(ROWS), 1, i, s, down_physical=physical)
    weights, x, expert = steered(cfg, "q2", seed=h + i + s)
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, len(x)) as layer:
        layer.force_grouped()
        _, y, ids, w = layer.forward(x)
        assert_parity(y, ids, w, *want, label=f"q2 down {i}")
        np.testing.assert_array_equal(y, layer.forward(x)[1], err_msg="not deterministic")
