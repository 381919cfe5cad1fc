"""The measured work of the MoE feed-forward block: what a program that runs a model through it has it do.

A case is one pass of a token batch through a few layers, each with weights of its own, by one of the four ways a
program calls the block:

  device    pf_hip_moe_forward_device: activations stay in device memory, the call only enqueues
  hc        pf_hip_moe_forward_hc_device: the same between the hyper-connection read and add of four residual streams
  host      qwen4_moe_forward: the drop-in call of a forward loop that keeps its activations in host memory
  streamed  pf_moe_forward_streamed: the routed experts of a model larger than device memory come from a file

Several layers for short batches because a token meets every layer of a model in turn: each layer's experts then come
from memory, not from a cache that the pass before left warm.  Shapes: the measured layer (hidden 2048, 512 experts,
top-10, intermediate and shared 512) and the widths of real checkpoints (hidden 2560, intermediate and shared 640).
Formats: Q4_K or IQ2_XXS throughout, and the two checkpoint profiles ("q2": IQ2_XXS gate and up, Q2_K down, "q4": Q4_K
gate and up, MXFP4 down; shared expert Q8_0 in both).
"""
import ctypes as C
import math
import os

import numpy as np
import torch

import picoforge_amd as pf
from picoforge_amd import abi, workloads

EXPERTS, TOP_K, STREAMS = 512, 10, 4
ROUTER_STD, ZIPF_TEMPERATURE = 0.02, 0.18   # as the benchmark draws its routers
FORMATS = {"q4k": abi.GGUF_Q4_K, "iq2xxs": abi.GGUF_IQ2_XXS, "q2": "q2", "q4": "q4"}
ROUTED_BLOCKS = 16381   # distinct blocks that the routed tensors of a state are filled with


def case(name, entry, fmt, shape, layers, tokens, calls=1, rho=0.0, zipf=0.0, slots=0):
    """rho: correlation of neighbouring tokens (0.85: neighbours share about half of their experts); zipf: exponent of
    the experts' popularity (0: all alike); slots: experts that a streamed layer's pool holds; calls: consecutive
    batches that a streamed pass consists of."""
    hidden, inter = {"measured": (2048, 512), "checkpoint": (2560, 640)}[shape]
    physical = 768 if fmt == "q2" and inter == 640 else inter   # Q2_K rows are stored in whole blocks of 256
    c = {"entry": entry, "format": fmt, "hidden": hidden, "inter": inter, "down_physical": physical, "layers": layers,
         "tokens": tokens, "calls": calls, "rho": rho, "zipf": zipf, "slots": slots}
    return dict(c, name=name) if name else c


def listed():
    return [
        # generation for one user: a token through consecutive layers, activations resident
        case("decode_q4k", "device", "q4k", "measured", 4, 1),
        # the same as a checkpoint's forward loop runs it, between its hyper-connection steps
        case("decode_hc_q2_checkpoint", "hc", "q2", "checkpoint", 4, 1),
        # the same from a loop that keeps its activations on the host, the experts in the smallest format
        case("decode_host_iq2xxs", "host", "iq2xxs", "measured", 4, 1),
        # a draft of four tokens verified at once
        case("verify4_q4k", "device", "q4k", "measured", 4, 4, rho=0.85),
        # a few users' tokens at once, host activations, an odd count
        case("batch13_host_q4_checkpoint", "host", "q4", "checkpoint", 2, 13),
        # many users' tokens at once
        case("batch32_q4k", "device", "q4k", "measured", 2, 32),
        # the short rest of a prompt, or more users: a ragged count, skewed experts
        case("batch101_q2_checkpoint", "device", "q2", "checkpoint", 1, 101, zipf=1.1),
        # a prompt's chunk at the benchmark's size
        case("prefill1024_q4k", "device", "q4k", "measured", 1, 1024, zipf=1.1),
        # the largest chunk, as a checkpoint's forward loop runs it
        case("prefill2048_hc_q4_checkpoint", "hc", "q4", "checkpoint", 1, 2048, zipf=1.1),
        # a prompt of no round length, host activations
        case("prefill777_host_iq2xxs", "host", "iq2xxs", "measured", 1, 777, zipf=1.1),
        # generation with streamed experts: 64 tokens, nearly three experts of a token's ten not in the pool
        case("streamed_decode_q4k", "streamed", "q4k", "measured", 1, 1, calls=64, zipf=1.1, slots=320),
        # a prompt's pieces with streamed experts
        case("streamed_prompt_q2_checkpoint", "streamed", "q2", "checkpoint", 1, 24, calls=4, zipf=1.1, slots=384),
    ]


def log_int(rng, low, high):
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng):
    fmt, shape = rng.choice(sorted(FORMATS)), rng.choice(["measured", "checkpoint"])
    if fmt in ("q4k", "iq2xxs"):
        shape = "measured"   # rows of 640 values are no whole blocks of these two formats
    kind = rng.choice(["short", "short", "batch", "chunk", "streamed"])
    if kind == "streamed":
        tokens = log_int(rng, 1, 24)
        return case(None, "streamed", fmt, shape, 1, tokens, calls=max(2, 64 // tokens), zipf=round(rng.uniform(0.8, 1.2), 2),
                    slots=rng.choice([320, 352, 384]))
    entry = rng.choice(["device", "device", "hc", "host"])
    if kind == "short":   # one user, a verified draft, a few users
        tokens = log_int(rng, 1, 16)
        rho = round(rng.uniform(0.7, 0.9), 2) if tokens <= 8 and rng.random() < 0.5 else 0.0
        return case(None, entry, fmt, shape, 4 if tokens <= 4 else 2, tokens, rho=rho)
    if kind == "batch":
        tokens = log_int(rng, 17, 256)
        zipf = rng.choice([0.0, round(rng.uniform(0.8, 1.2), 2)])
        return case(None, entry, fmt, shape, 2 if tokens <= 40 else 1, tokens, zipf=zipf)
    return case(None, entry, fmt, shape, 1, log_int(rng, 257, 1024 if entry == "host" else 2048), zipf=round(rng.uniform(0.8, 1.2), 2))


def config(c):
    return abi.moe_config(c["hidden"], EXPERTS, TOP_K, c["inter"], c["inter"], c["down_physical"])


def quantised(synth, gtype, blocks, seed):
    """N(0, 0.02) weights; IQ2_XXS: blocks drawn evenly."""
    if gtype == abi.GGUF_Q4_K:
        return synth.q4k_normal(blocks, seed, 0.02)
    if gtype == abi.GGUF_IQ2_XXS:
        return synth.iq2xxs_uniform(blocks, seed)
    return synth.quantised_normal(gtype, blocks * abi.BLOCK[gtype][0], seed, 0.02)


class RoutedBytes:
    """Routed tensors of one format: some blocks, repeated over the tensor; every tensor starts at another of them."""

    def __init__(self, synth, gtype, blocks, seed):
        few = quantised(synth, gtype, ROUTED_BLOCKS, seed)
        self.block_bytes, self.cut = abi.BLOCK[gtype][1], 0
        self.bytes = np.empty((blocks // ROUTED_BLOCKS + 2) * len(few), np.uint8)
        for at in range(0, len(self.bytes), len(few)):
            self.bytes[at:at + len(few)] = few

    def tensor(self, blocks):
        self.cut = (self.cut + 7919) % ROUTED_BLOCKS
        return self.bytes[self.cut * self.block_bytes:(self.cut + blocks) * self.block_bytes]


def layer_weights(c, cfg, seed):
    """The eight tensors of every layer, as a model file holds them."""
    synth, fmt = pf.Synth(), FORMATS[c["format"]]
    gate, down, shared = pf.LayerWeights.PROFILE.get(fmt, (fmt,) * 3)
    types = [abi.GGUF_F32, gate, gate, down, shared, shared, shared, abi.GGUF_F32]
    h, i, e = cfg.hidden_size, cfg.intermediate, cfg.experts
    count = [h * e, h * i * e, h * i * e, cfg.down_physical * h * e, h * i, h * i, i * h, h]
    blocks = [n // abi.BLOCK[t][0] for n, t in zip(count, types)]
    routed = {}
    for j in (1, 2, 3):
        if types[j] not in routed:
            routed[types[j]] = RoutedBytes(synth, types[j], max(blocks[a] for a in (1, 2, 3) if types[a] == types[j]), seed + j)
    out = []
    for layer in range(c["layers"]):
        raw = []
        for j in range(8):
            stream = seed + 1000 * (layer + 1) + j
            if j in (0, 7):
                raw.append(synth.normal((count[j],), stream, ROUTER_STD).view(np.uint8))
            elif j <= 3:
                raw.append(routed[types[j]].tensor(blocks[j]))
            else:
                raw.append(quantised(synth, types[j], blocks[j], stream))
        weights = pf.LayerWeights(cfg, raw, types)
        if c["zipf"]:
            workloads.zipf_router(weights, stream, s=c["zipf"], temperature=ZIPF_TEMPERATURE)
        out.append(weights)
    return out


def activations(c, rows, seed):
    """RMS-normalised rows; with skewed experts, coordinate 0 is the router bias's input."""
    x = pf.Synth().normal((rows, c["hidden"]), seed)
    if c["rho"]:
        for t in range(1, rows):
            x[t] = c["rho"] * x[t - 1] + math.sqrt(1 - c["rho"] ** 2) * x[t]
    x = pf.rms_normalise(x)
    if c["zipf"]:
        x[:, 0] = 1.0
    return x


def checked(status, what):
    if status != 0:
        raise RuntimeError("%s: status %d" % (what, status))


class State:
    """A program's layers and workspaces, and what it has in hand before the call."""

    def __init__(self, c, seed):
        self.case, self.api, self.layers, self.pool, self.fd = c, pf.load_product(), [], None, -1
        cfg, rows = config(c), c["tokens"] * c["calls"]
        weights = layer_weights(c, cfg, seed)
        for l, w in enumerate(weights):
            handle = self.streamed_layer(cfg, w) if c["entry"] == "streamed" else None
            self.layers.append(pf.MoeLayer(self.api, cfg, w, c["tokens"], handle=handle))
        x = [activations(c, rows, seed + 77 + l) for l in range(c["layers"])]
        getattr(self, "hold_" + ("host" if c["entry"] == "streamed" else c["entry"]))(c, x, seed)

    def streamed_layer(self, cfg, w):
        """The routed tensors in a file in memory behind a pool, the rest of the layer resident."""
        self.fd, at, offsets = os.memfd_create("experts"), 0, []
        for j in (1, 2, 3):
            offsets.append(at)
            os.truncate(self.fd, at + w.raw[j].size)
            done = 0
            while done < w.raw[j].size:
                done += os.pwrite(self.fd, w.raw[j][done:done + (1 << 28)], at + done)
            at += w.raw[j].size
        h, i = cfg.hidden_size, cfg.intermediate
        sizes = (C.c_size_t * 3)(*(w.raw[j].size // cfg.experts for j in (1, 2, 3)))
        table = (abi.QW4ExpertLayer * 1)(abi.QW4ExpertLayer((C.c_uint64 * 3)(*offsets)))
        self.pool = self.api.pool_create(self.fd, table, 1, cfg.experts, sizes, self.case["slots"])
        if not self.pool:
            raise RuntimeError("no expert pool")
        checked(self.api.pool_set_formats(self.pool, (C.c_uint32 * 3)(*w.types[1:4]), (C.c_size_t * 3)(h, h, cfg.down_physical),
                                          (C.c_size_t * 3)(i, i, h)), "pool formats")
        err, handle, struct = abi.Qwen4Error(), C.c_void_p(), w.without_routed_bytes()
        checked(self.api.create_streamed(C.byref(cfg), C.byref(struct), C.byref(handle), C.byref(err)), "streamed layer")
        return handle

    def hold_device(self, c, x, seed):
        self.handles = [layer.device_handles() for layer in self.layers]
        self.x = [torch.from_numpy(a).cuda() for a in x]
        self.y = [torch.empty_like(a) for a in self.x]

    def hold_hc(self, c, x, seed):
        """Streams as the loop's normalisation leaves them, gate logits, injection weights and the residual of four
        streams that every layer adds into."""
        self.handles = [layer.device_handles() for layer in self.layers]
        gen = torch.Generator("cuda").manual_seed(seed)
        shape = (c["tokens"], STREAMS, c["hidden"])
        self.normed, self.gates, self.inject = [], [], []
        for a in x:
            rows = torch.from_numpy(a).cuda()[:, None, :]
            noise = torch.randn(shape, device="cuda", generator=gen)
            if c["zipf"]:
                noise[:, :, 0] = 0.0
            self.normed.append((2.0 * rows + 0.5 * noise).contiguous())   # the gates halve it
            gates = torch.randn(shape, device="cuda", generator=gen)
            if c["zipf"]:
                gates[:, :, 0] = 0.0
            self.gates.append(gates)
            self.inject.append(0.5 * torch.rand(shape[:2], device="cuda", generator=gen))
        self.residual = torch.randn(shape, device="cuda", generator=gen)

    def hold_host(self, c, x, seed):
        self.rows = []
        for a in x:
            y = np.empty_like(a)
            ids, weights = np.empty((len(a), TOP_K), np.uint32), np.empty((len(a), TOP_K), np.float32)
            calls = []
            for first in range(0, len(a), c["tokens"]):
                part = slice(first, first + c["tokens"])
                calls.append((abi.f32_view(a[part]), abi.f32_view(y[part]),
                              abi.Qwen4MoeRoutes(abi.u32_view(ids[part]), abi.f32_view(weights[part]))))
            self.rows.append((a, y, ids, weights, calls))

    def close(self):
        for layer in self.layers:
            layer.close()
        if self.pool:
            self.api.pool_destroy(self.pool)
        if self.fd >= 0:
            os.close(self.fd)
        self.layers, self.pool, self.fd = [], None, -1

    def __del__(self):
        self.close()


def prepare(c, seed):
    return State(c, int(seed) * 100003 + 17)


def run_device(s):
    hip, n, h = s.api.hip, s.case["tokens"], s.case["hidden"]
    stream = torch.cuda.current_stream().cuda_stream
    for (moe, work), x, y in zip(s.handles, s.x, s.y):
        checked(hip.moe_forward_device(moe, work, x.data_ptr(), h, y.data_ptr(), h, n, stream), "forward")
    return s.y


def run_hc(s):
    hip, n, h = s.api.hip, s.case["tokens"], s.case["hidden"]
    stream, cube = torch.cuda.current_stream().cuda_stream, STREAMS * h
    for (moe, work), normed, gates, inject in zip(s.handles, s.normed, s.gates, s.inject):
        checked(hip.moe_forward_hc_device(moe, work, normed.data_ptr(), cube, h, gates.data_ptr(), cube, h,
                                          s.residual.data_ptr(), cube, h, inject.data_ptr(), STREAMS, n, stream), "forward")
    return s.residual


def run_host(s):
    for layer, (_, _, _, _, calls) in zip(s.layers, s.rows):
        for x, y, routes in calls:
            checked(s.api.forward(layer.handle, x, y, C.byref(routes), layer.work, C.byref(layer.err)), "forward")
    return [(y, ids.view(np.int32), weights) for _, y, ids, weights, _ in s.rows]


def run_streamed(s):
    layer, (_, y, ids, weights, calls) = s.layers[0], s.rows[0]
    for x, out, routes in calls:
        checked(s.api.forward_streamed(layer.handle, s.pool, 0, x, out, C.byref(routes), layer.work, C.byref(layer.err)), "forward")
    return y, ids.view(np.int32), weights


def run(state):
    return {"device": run_device, "hc": run_hc, "host": run_host, "streamed": run_streamed}[state.case["entry"]](state)


def distinct_experts(c):
    """Expected number of experts that a batch meets.  An expert's logit is normal around its bias; it is met by a token
    when it is over the bar that TOP_K experts reach on average.  (A correlated neighbour brings a part of its own.)"""
    draws = c["tokens"] if not c["rho"] else 1 + (c["tokens"] - 1) * (1 - c["rho"] ** 4)
    spread = ROUTER_STD * math.sqrt(c["hidden"])
    bias = [-c["zipf"] * ZIPF_TEMPERATURE * math.log(rank) for rank in range(1, EXPERTS + 1)]
    low, high = -10.0, 10.0
    for _ in range(40):
        bar = (low + high) / 2
        share = [0.5 * math.erfc((bar - b) / (spread * math.sqrt(2))) for b in bias]
        low, high = (bar, high) if sum(share) > TOP_K else (low, bar)
    return sum(1.0 - (1.0 - p) ** draws for p in share)


def work(c):
    """Every met expert, the shared expert and the routers read once a batch, activations in and out once."""
    cfg, t, h = config(c), c["tokens"], c["hidden"]
    b = workloads.layer_bytes(FORMATS[c["format"]], cfg)
    weights = distinct_experts(c) * (b["gate_up"] + b["down"]) + b["shared_gate_up"] + b["shared_down"] + b["routers"]
    rows = t * 4 * (h * (4 * STREAMS if c["entry"] == "hc" else 2))   # hc: two cubes in, the residual in and out
    flops = 2 * t * ((TOP_K + 1) * 3 * h * c["inter"] + (EXPERTS + 1) * h)
    passes = c["layers"] * c["calls"]
    return {"bytes": passes * (weights + rows), "flops": passes * flops}


def tolerance(c):
    """Quantised weights are exact in every product and sums are 32-bit; ids are exact."""
    return {"rel": 1e-5}
