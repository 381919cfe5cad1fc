"""GPU parity of the grouped product (pf_moe_prefill.hip) at the row counts where its tiles change: an expert's last tile of 16
rows or fewer, of 17 to 32, and several tiles; every weight order it reads, rows of one and of several 256-blocks."""
import numpy as np
import pytest

import picoforge_amd as pf
from picoforge_amd import abi

from helpers import assert_parity, forward_with, make_layer_inputs

pytestmark = pytest.mark.gpu

ROWS = [1, 15, 16, 17, 0, 31, 32, 33, 48, 65]   # of the experts, in turn


def steered(cfg, fmt, seed):
    """A layer whose router sends ROWS[e] tokens to expert e."""
    expert = np.repeat(np.arange(len(ROWS)), ROWS)
    np.random.default_rng(seed).shuffle(expert)
    weights, x = make_layer_inputs(cfg, fmt, len(expert), seed=seed)
    router = weights.raw[0].view(np.float32).reshape(cfg.experts, cfg.hidden_size)
    router *= 0.01
    x[:, :cfg.experts] = 0.0
    for e in range(cfg.experts):
        router[e, e] = 5.0
    x[np.arange(len(expert)), expert] = 2.0
    return weights, x, expert


@pytest.mark.parametrize("copy", ["1", "0"])
@pytest.mark.parametrize("h,i,s,physical,fmt", [
    (256, 256, 512, None, abi.GGUF_Q4_K), (768, 512, 256, None, abi.GGUF_Q4_K), (256, 256, 512, None, abi.GGUF_IQ2_XXS),
    (768, 512, 256, None, abi.GGUF_IQ2_XXS), (512, 384, 128, 512, "q2"), (512, 384, 128, None, "q4"), (2560, 640, 640, 768, "q2"),
    (2560, 640, 640, None, "q4"), (256, 128, 128, None, "q4"), (512, 256, 512, None, "q4"), (256, 512, 128, None, "q4"), (256, 768, 128, None, "q4"),
])
def test_row_counts_around_the_tiles(product, oracle, monkeypatch, h, i, s, physical, fmt, copy):
    print(f"case grouped rows {fmt} h={h} i={i} s={s} tile-ordered copies {copy}", flush=True)
    monkeypatch.setenv("PF_MOE_PREFILL_COPY", copy)
    cfg = abi.moe_config(h, len(ROWS), 1, i, s, down_physical=physical)
    weights, x, expert = steered(cfg, fmt, seed=h + i + s)
    want = forward_with(oracle, cfg, weights, x)
    np.testing.assert_array_equal(want[1][:, 0], expert)
    with pf.MoeLayer(product, cfg, weights, len(x)) as layer:
        layer.force_grouped()
        assert product.hip.moe_kernel_family(*layer.device_handles(), len(x)) == 2
        _, y, ids, w = layer.forward(x)
        assert_parity(y, ids, w, *want, label=f"{fmt}")
        np.testing.assert_array_equal(y, layer.forward(x)[1], err_msg="not deterministic")


@pytest.mark.parametrize("tokens,e,k", [(4096, 16, 8), (2049, 300, 7), (1023, 40, 3), (131, 9, 2)])
def test_pairs_that_one_workgroup_groups(product, tokens, e, k):
    """Up to 32768 pairs (128 KB of LDS), at every remainder of four, beside rows that do not fill the last workgroup; an expert
    that every token has."""
    print(f"case grouped, {tokens} tokens of {k} pairs, {e} experts", flush=True)
    cfg = abi.moe_config(256, e, k, 256, 256)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, tokens, seed=tokens + e)
    x[:, 0] = 1.0
    weights.raw[0].view(np.float32).reshape(e, 256)[e // 2, 0] = 9.0
    x[::7] *= 1e-3
    with pf.MoeLayer(product, cfg, weights, len(x)) as layer:
        layer.force_grouped()
        _, y, ids, w = layer.forward(x)
        np.testing.assert_array_equal(y, layer.forward(x)[1], err_msg="not deterministic")
        layer.force_general()
        _, yg, idsg, wg = layer.forward(x)
    assert (ids == e // 2).any(axis=1).mean() > 0.8
    assert_parity(y, ids, w, yg, idsg, wg, label="grouped product against general kernels")


def test_more_pairs_than_one_workgroup_groups(product):
    """Beyond 32768 pairs the row tiles come from the kernels that count, scan and place one after the other."""
    print("case grouped, 4100 tokens of 8 pairs", flush=True)
    cfg = abi.moe_config(256, 16, 8, 256, 256)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, 4100, seed=71)
    with pf.MoeLayer(product, cfg, weights, len(x)) as layer:
        assert product.hip.moe_kernel_family(*layer.device_handles(), len(x)) == 2
        _, y, ids, w = layer.forward(x)
        layer.force_general()
        _, yg, idsg, wg = layer.forward(x)
    assert_parity(y, ids, w, yg, idsg, wg, label="grouped product against general kernels")
