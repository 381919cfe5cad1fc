"""Host-pointer forwards on both sides of each way rows travel: the page-locked block (up to 64 tokens), the ring of pieces by
one thread, and by the crew (from 1 MB); a value that is not finite in the last row is found before anything is written."""
import threading

import numpy as np
import pytest

import picoforge_amd as pf
from picoforge_amd import abi

from helpers import assert_parity, forward_with, make_layer_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,batches", [(512, (1, 64, 65, 257, 512, 513, 700)), (2560, (64, 104, 105, 460))])
def test_rows_through_block_ring_and_crew(product, oracle, hidden, batches):
    cfg = abi.moe_config(hidden, 16, 3, 256, 256)
    most = max(batches)
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, most, seed=hidden)
    want = forward_with(oracle, cfg, weights, x)
    with pf.MoeLayer(product, cfg, weights, most) as layer:
        for tokens in batches:
            print(f"case hidden={hidden} tokens={tokens}", flush=True)
            for bad in (np.nan, -np.inf):
                spoilt = x[:tokens].copy()
                spoilt[-1, -1] = bad
                st, y, ids, w = layer.forward(spoilt, check=False)
                assert st == abi.QW4_NONFINITE and b"nonfinite input" in bytes(layer.err.detail)
                assert (y == -99.0).all() and (w == -99.0).all() and (ids == 0xFFFFFFFF).all()
            _, y, ids, w = layer.forward(x[:tokens])   # the workspace is as usable as before
            assert_parity(y, ids, w, want[0][:tokens], want[1][:tokens], want[2][:tokens], label=f"T={tokens}")
            _, y2, _, _ = layer.forward(x[:tokens], want_routes=False)
            np.testing.assert_array_equal(y, y2)


def test_pieces_that_start_off_a_16_byte_boundary(product, oracle):
    """Rows of 132 bytes (33 F32 columns, the general kernels): the second piece of the ring starts 12 bytes off a 16-byte
    boundary of the device rows, and its 4 rows are a multiple of 16 bytes long."""
    cfg = abi.moe_config(33, 8, 2, 32, 32)
    tokens = 512 * 1024 // 132 + 4
    weights, x = make_layer_inputs(cfg, abi.GGUF_F32, tokens, seed=33, std=0.1)
    want = forward_with(oracle, cfg, weights, x)
    assert_parity(*forward_with(product, cfg, weights, x), *want, label=f"hidden 33, {tokens} tokens")


def test_two_workspaces_at_once(product):
    """Two threads, each with a layer and a workspace of its own, on batches that are worth the crew: whoever finds it at work
    for the other copies alone, and every call's rows are what the call gives by itself."""
    cfg = abi.moe_config(512, 16, 3, 256, 256)
    layers, inputs, alone, wrong = [], [], [], []
    for seed in (5, 6):
        weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, 900, seed=seed)
        layers.append(pf.MoeLayer(product, cfg, weights, 900))
        inputs.append((x, x[:600]))
        alone.append([layers[-1].forward(rows)[1:] for rows in inputs[-1]])

    def calls(which):
        try:
            for turn in range(12):
                got = layers[which].forward(inputs[which][turn % 2])[1:]
                if not all(np.array_equal(a, b) for a, b in zip(got, alone[which][turn % 2])):
                    wrong.append((which, turn))
        except Exception as e:   # a thread's error would be lost
            wrong.append((which, repr(e)))

    threads = [threading.Thread(target=calls, args=(which,)) for which in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for layer in layers:
        layer.close()
    assert not wrong, wrong


@pytest.mark.parametrize("hidden,k", [(256, 1), (768, 3), (2560, 5)])
def test_pieces_of_every_length_call_after_call(product, hidden, k):
    """Last pieces of less than a kernel's 16 KB, of a whole number of them and of more, slots taken again within a call and by
    the next one; ids and weights of a longer batch at every remainder of four."""
    step = 512 * 1024 // (4 * hidden)
    cfg = abi.moe_config(hidden, 12, k, 256, 256)
    most = 9 * step + 3
    weights, x = make_layer_inputs(cfg, abi.GGUF_Q4_K, most, seed=hidden + k)
    with pf.MoeLayer(product, cfg, weights, most) as layer:
        layer.force_general()
        _, y, ids, w = layer.forward(x[:300])
        for tokens in (65, 66, 67, 68, step, step + 1, 2 * step - 1, 8 * step + 4, most, 65, 9 * step):
            print(f"case pieces hidden={hidden} tokens={tokens}", flush=True)
            _, yt, idst, wt = layer.forward(x[:tokens])
            n = min(tokens, 300)
            np.testing.assert_array_equal(yt[:n], y[:n])
            np.testing.assert_array_equal(idst[:n], ids[:n])
            np.testing.assert_array_equal(wt[:n], w[:n])
            _, again, _, _ = layer.forward(x[:tokens])
            np.testing.assert_array_equal(yt, again)
