"""GPU parity of the kernels for a few rows per expert (pf_moe_batch.hip) against the CPU oracle: batches that give an
expert one row, one chunk of eight, ragged chunks and several 32-row tiles, in every format combination, at widths that
are whole 256-blocks and at widths whose last piece is short."""
import numpy as np
import pytest

import picoforge_amd as pf
from picoforge_amd import abi

from helpers import assert_parity, forward_with, make_layer_inputs

pytestmark = pytest.mark.gpu

# (h, e, k, i, s, down stored, expert type, batches): the batch sizes are on both sides of a chunk (8 rows), of a row tile
# (32) and of a router tile (16 tokens by 16 experts)
CASES = [
    (512, 32, 6, 256, 256, None, abi.GGUF_Q4_K, (33, 48, 177)), (512, 32, 6, 256, 256, None, abi.GGUF_IQ2_XXS, (33, 48, 177)),
    (2560, 40, 3, 512, 256, None, abi.GGUF_Q4_K, (35, 113)), (2048, 200, 10, 512, 512, None, abi.GGUF_IQ2_XXS, (47, 97)),
    (512, 32, 6, 256, 256, None, "q2", (11, 16, 17, 177)), (512, 32, 6, 256, 256, None, "q4", (17, 31, 177)),
    (1280, 24, 4, 320, 320, 512, "q2", (12, 33, 160)), (768, 24, 3, 384, 448, None, "q4", (18, 33, 160)),
    (2560, 90, 10, 640, 640, 768, "q2", (13, 65)), (2560, 90, 10, 640, 640, None, "q4", (19, 65)),
]


@pytest.mark.parametrize("h,e,k,i,s,physical,fmt,batches", CASES)
def test_batches_of_a_few_rows_per_expert(product, oracle, h, e, k, i, s, physical, fmt, batches):
    print(f"case batch {fmt} h={h} e={e} k={k} i={i} s={s} down stored {physical or i} wide", flush=True)
    cfg = abi.moe_config(h, e, k, i, s, down_physical=physical)
    most = max(batches)
    weights, x = make_layer_inputs(cfg, fmt, most, seed=h + e + i)
    x[5:10] = x[4]                                # tokens that share every expert
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, most) as layer:
        for tokens in batches:
            print(f"  tokens={tokens}", flush=True)
            _, y, ids, w = layer.forward(x[:tokens])
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"{fmt} T={tokens}")
        np.testing.assert_array_equal(y, layer.forward(x[:tokens])[1], err_msg="not deterministic")


@pytest.mark.parametrize("router", [0.0, 1e-19])
def test_activations_whose_squares_overflow(product, oracle, router):
    """A finite activation of 2e19 that the router and the experts all but ignore: its square is infinite, the logits, the
    routes and the outputs are ordinary.  router: the magnitude of the router's weights in its column (0: inf * 0 in the
    sums of squares; 1e-19: an infinite sum, products of about two)."""
    cfg = abi.moe_config(512, 32, 6, 256, 256)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, 65, seed=23)
    rows = weights.raw[0].view(np.float32).reshape(cfg.experts, cfg.hidden_size)
    rows[:, 0] = router * np.linspace(-1.0, 1.0, cfg.experts, dtype=np.float32)
    weights.raw[7].view(np.float32)[0] = 0.0
    for j in (1, 2, 4, 5):
        weights.raw[j].reshape(-1, cfg.hidden_size // 256, 144)[:, 0] = 0   # the first 256 columns of gate and up
    x[::3, 0] = 2e19
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, 65) as layer:
        for tokens in (33, 65):
            print(f"case squares overflow, router {router}, {tokens} tokens", flush=True)
            _, y, ids, w = layer.forward(x[:tokens])
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"T={tokens}")


@pytest.mark.parametrize("h,i,physical,fmt,copy", [
    (512, 256, 256, "q2", "1"), (512, 384, 512, "q2", "1"), (768, 640, 768, "q2", "1"), (512, 896, 1024, "q2", "1"),   # three blocks a row fit the copy in LDS
    (512, 256, None, "q4", "1"), (512, 384, None, "q4", "1"), (512, 512, None, "q4", "1"), (768, 640, None, "q4", "1"),
    (512, 768, None, "q4", "1"), (768, 640, None, "q4", "0"),   # no tile-ordered copy: rows
])
def test_down_rows_by_tile_and_by_row(product, oracle, monkeypatch, h, i, physical, fmt, copy):
    """The orders of the profiles' down weights, at two to five units of 128 columns and one to four blocks a row."""
    print(f"case batch down {fmt} h={h} i={i} down stored {physical or i} wide, tile-ordered copies {copy}", flush=True)
    monkeypatch.setenv("PF_MOE_PREFILL_COPY", copy)
    cfg = abi.moe_config(h, 24, 3, i, i, down_physical=physical)
    weights, x = make_layer_inputs(cfg, fmt, 40, seed=h + i)
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, 40) as layer:
        for tokens in (17, 40):
            assert product.hip.moe_kernel_family(*layer.device_handles(), tokens) == 3
            _, y, ids, w = layer.forward(x[:tokens])
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"{fmt} T={tokens}")


# (experts, top-k, format, last batch of the decode kernels, last of the kernels for a few rows per expert)
LINES = [(16, 4, abi.GGUF_Q4_K, 32, 250), (64, 8, abi.GGUF_Q4_K, 29, 128), (128, 8, abi.GGUF_IQ2_XXS, 28, 247), (64, 8, "q2", 10, 139),
         (128, 8, "q4", 16, 158)]


@pytest.mark.parametrize("e,k,fmt,pair_to,batch_to", LINES)
def test_batches_on_both_sides_of_the_lines_between_the_kernels(product, oracle, e, k, fmt, pair_to, batch_to):
    """The lines go by pairs and experts; a token more on either side of one is another kernel family's and the same block."""
    print(f"case lines {fmt} e={e} k={k}", flush=True)
    cfg = abi.moe_config(512, e, k, 256, 256)
    weights, x = make_layer_inputs(cfg, fmt, batch_to + 1, seed=e + k)
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, batch_to + 1) as layer:
        for tokens, family in ((pair_to, 1), (pair_to + 1, 3), (batch_to, 3), (batch_to + 1, 2)):
            assert product.hip.moe_kernel_family(*layer.device_handles(), tokens) == family, tokens
            _, y, ids, w = layer.forward(x[:tokens])
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"{fmt} T={tokens}")


@pytest.mark.parametrize("h,i,s,k,copy", [
    (512, 256, 256, 6, "1"), (768, 384, 384, 1, "1"), (512, 512, 640, 14, "1"), (512, 256, 256, 15, "1"), (2560, 640, 640, 10, "1"), (1024, 768, 256, 4, "1"),   # 768: no copy
    (2048, 256, 256, 14, "1"), (2048, 384, 640, 12, "1"), (2048, 512, 512, 10, "1"),   # the largest on the block-scaled product
    (2560, 640, 640, 10, "0"),
])
def test_short_batches_of_the_q4_profile(product, oracle, monkeypatch, h, i, s, k, copy):
    """The decode kernels' down projections of MXFP4 rows: on the block-scaled matrix instruction where the layer keeps the
    tile order, from the work on where that pays; two to five units of 128 columns, one to fifteen slots."""
    print(f"case short q4 batches h={h} i={i} s={s} k={k} tile-ordered copies {copy}", flush=True)
    monkeypatch.setenv("PF_MOE_PREFILL_COPY", copy)
    cfg = abi.moe_config(h, 32, k, i, s)
    weights, x = make_layer_inputs(cfg, "q4", 16, seed=h + i + k)
    x[3] = 0.0
    x[4, : h // 2] *= 1e-4
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, 16) as layer:
        for tokens in (1, 2, 3, 4, 5, 16):
            assert product.hip.moe_kernel_family(*layer.device_handles(), tokens) == (1 if copy == "1" or tokens <= 4 else 3)
            print(f"  tokens={tokens}", flush=True)
            _, y, ids, w = layer.forward(x[:tokens])
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"T={tokens}")
        np.testing.assert_array_equal(y, layer.forward(x)[1], err_msg="not deterministic")


@pytest.mark.parametrize("h,e,k,fmt", [(512, 70, 6, abi.GGUF_Q4_K), (2560, 33, 4, abi.GGUF_Q4_K), (768, 100, 5, abi.GGUF_IQ2_XXS), (2048, 512, 3, abi.GGUF_IQ2_XXS),
                                       (512, 300, 6, abi.GGUF_Q4_K), (2560, 257, 4, abi.GGUF_Q4_K), (768, 500, 5, abi.GGUF_IQ2_XXS)])   # 32, 32, 17 tokens on
def test_decode_kernels_on_either_side_of_the_matrix_router(product, oracle, h, e, k, fmt):
    """Up to 16 tokens or 8192 logits the decode kernels' own router, beyond them tiles of 16 tokens and experts, whose images they read."""
    print(f"case decode router {fmt} h={h} e={e} k={k}", flush=True)
    cfg = abi.moe_config(h, e, k, 256, 256)
    weights, x = make_layer_inputs(cfg, fmt, 32, seed=h + e)
    x[3] = 0.0
    x[20] *= 1e-4
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, 32) as layer:
        for tokens in (16, 17, 25, 32):
            assert product.hip.moe_kernel_family(*layer.device_handles(), tokens) == 1
            _, y, ids, w = layer.forward(x[:tokens])
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"T={tokens}")


ROWS = [1, 24, 7, 8, 9, 0, 16, 17, 33, 25, 32, 65]


def steered(cfg, fmt, rows, seed):
    """A layer whose router sends rows[e] tokens to expert e."""
    expert = np.repeat(np.arange(len(rows)), rows)
    np.random.default_rng(seed).shuffle(expert)
    weights, x = make_layer_inputs(cfg, fmt, len(expert), seed=seed)
    router = weights.raw[0].view(np.float32).reshape(cfg.experts, cfg.hidden_size)
    router *= 0.01
    x[:, :cfg.experts] = 0.0
    router[np.arange(cfg.experts), np.arange(cfg.experts)] = 5.0
    x[np.arange(len(expert)), expert] = 2.0
    return weights, x, expert


@pytest.mark.parametrize("h,i,s,physical,fmt", [
    (512, 256, 512, None, abi.GGUF_Q4_K), (512, 256, 256, None, abi.GGUF_IQ2_XXS), (512, 384, 256, 512, "q2"), (512, 384, 256, None, "q4")])
def test_experts_of_every_row_count(product, oracle, h, i, s, physical, fmt):
    """Experts of no row up to three row tiles in one batch: the item list's classes (up to 8, 16, 24 rows, more) with an expert on
    either side of each, and a shared expert of eight tiles ahead of them."""
    print(f"case few rows, every row count, {fmt} h={h} i={i} s={s}", flush=True)
    cfg = abi.moe_config(h, len(ROWS), 1, i, s, down_physical=physical)
    weights, x, expert = steered(cfg, fmt, ROWS, seed=h + i + s)
    want = forward_with(oracle, cfg, weights, x)
    np.testing.assert_array_equal(want[1][:, 0], expert)
    with pf.MoeLayer(product, cfg, weights, len(x)) as layer:
        assert product.hip.moe_kernel_family(*layer.device_handles(), len(x)) == 3
        _, y, ids, w = layer.forward(x)
        assert_parity(y, ids, w, *want, label=f"{fmt}")
        np.testing.assert_array_equal(y, layer.forward(x)[1], err_msg="not deterministic")


@pytest.mark.parametrize("h,i,s,physical,fmt", [
    (512, 256, 512, None, abi.GGUF_Q4_K), (512, 256, 256, None, abi.GGUF_IQ2_XXS), (512, 384, 256, 512, "q2"), (512, 256, 256, None, "q4"), (512, 384, 512, None, "q4")])
def test_shared_rows_behind_the_routed_ones(product, oracle, h, i, s, physical, fmt):
    """Few experts of many rows, whose launches take the shared expert's chunks last (from 96 tokens on), on both sides of that line."""
    print(f"case shared rows last, {fmt} h={h} i={i} s={s}", flush=True)
    cfg = abi.moe_config(h, 8, 2, i, s, down_physical=physical)
    weights, x = make_layer_inputs(cfg, fmt, 131, seed=h + i + s)
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, len(x)) as layer:
        for tokens in (95, 96, 131):
            assert product.hip.moe_kernel_family(*layer.device_handles(), tokens) == 3
            _, y, ids, w = layer.forward(x[:tokens])
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"{fmt} T={tokens}")
        np.testing.assert_array_equal(y, layer.forward(x[:tokens])[1], err_msg="not deterministic")


# (hidden, inner width, experts, top-k, format, last batch of the decode kernels): the three classes of widths
WIDTH_LINES = [(2048, 512, 16, 4, abi.GGUF_Q4_K, 28), (2048, 512, 64, 8, abi.GGUF_Q4_K, 16), (1024, 512, 64, 8, abi.GGUF_Q4_K, 21),
               (1024, 256, 128, 8, abi.GGUF_Q4_K, 32), (2048, 512, 24, 4, abi.GGUF_IQ2_XXS, 17), (512, 512, 256, 8, abi.GGUF_IQ2_XXS, 20),
               (1024, 256, 200, 10, abi.GGUF_IQ2_XXS, 23)]


@pytest.mark.parametrize("h,i,e,k,fmt,pair_to", WIDTH_LINES)
def test_first_line_goes_by_the_work_of_a_pair(product, oracle, h, i, e, k, fmt, pair_to):
    print(f"case first line {fmt} h={h} i={i} e={e} k={k}", flush=True)
    cfg = abi.moe_config(h, e, k, i, i)
    weights, x = make_layer_inputs(cfg, fmt, 33, seed=h + e)
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, 33) as layer:
        for tokens, family in ((pair_to, 1), (pair_to + 1, 3)):
            assert product.hip.moe_kernel_family(*layer.device_handles(), tokens) == family, tokens
            _, y, ids, w = layer.forward(x[:tokens])
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"{fmt} T={tokens}")
