"""Workloads the speed of this library is measured on.

Each case is one call sequence that a program using the library makes: a decode step's MLP
layers launched one after another (`layers`), the same with part of each layer's groups handed
over through the ready queue (`queue`), a stack of dependent layers in one launch (`chain`), and
a decode step whose groups are staged from pinned host memory (`stream`). A stack has its own
weights for every layer, as a model has, so a layer's weights come from HBM wherever the whole
stack is larger than the 256 MB Infinity Cache.

Weights are uniform INT4 with per-128-column fp16 scales U(lo, hi), activations N(0, 1) in fp16
(bf16 on the batched path, batch 5 .. 32): the distributions of bench.py and the tests.
"""
import math

import numpy as np
import torch

from leanstream_amd.backend import MODE_PROGRESSIVE, NativeBackend, ReadyQueue
from leanstream_amd.streaming import StreamingDecode
from leanstream_amd.synth import LayerConfig, StreamConfig

DEV = "cuda"
WIDTHS = (256, 512, 1024, 2048, 4096, 8192)   # the widths the kernels are built for
MAX_BYTES = 850e6                              # of one pass: the largest listed case


def _case(name, kind, width, groups, active, batch=1, group=64, layers=1, queued=0, lo=0.005, hi=0.02):
    c = dict(kind=kind, width=width, groups=groups, active=active, batch=batch, group=group, layers=layers,
             queued=queued, lo=lo, hi=hi)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one small layer, 16 of 64 groups: the smallest call, where latency counts
        _case("layer_d1024_b1", "layers", 1024, 64, 16),
        # one decode step's layers, 8B-model shape, 30 % of the groups active
        _case("stack_d4096_b1", "layers", 4096, 192, 58, layers=12),
        # the same at a 70B-model shape, one sequence and four
        _case("stack_d8192_b1", "layers", 8192, 448, 90, layers=4, lo=0.003, hi=0.015),
        _case("stack_d8192_b4", "layers", 8192, 448, 90, batch=4, layers=4, lo=0.003, hi=0.015),
        # the 8B production pack: groups of two neurons, 20 % active
        _case("stack_d4096_g2_b1", "layers", 4096, 7168, 1434, group=2, layers=15),
        # ragged: 48-neuron groups, an odd count of them, three sequences
        _case("layer_d2048_g48_b3", "layers", 2048, 171, 53, batch=3, group=48),
        # half of each layer's groups resident, half staged and handed over through the ready queue
        _case("queue_d4096_b1", "queue", 4096, 192, 58, layers=12, queued=29),
        # batched decode on the matrix cores: every group, 32 sequences
        _case("dense_d4096_b32", "layers", 4096, 224, 224, batch=32, layers=4),
        # few sequences, a smaller model
        _case("dense_d2048_b7", "layers", 2048, 128, 128, batch=7, layers=8),
        # 70B-model shape, 16 sequences, 20 % of the groups
        _case("dense_d8192_b16", "layers", 8192, 448, 90, batch=16, layers=4, lo=0.003, hi=0.015),
        # a whole decode step's dependent layers (hidden state and RMSNorm between them), one launch
        _case("chain_d4096", "chain", 4096, 192, 58, layers=36),
        # a decode step whose active groups are all staged from pinned host memory
        _case("stream_d1024", "stream", 1024, 64, 16, layers=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layers", "layers", "layers", "batch", "dense", "dense", "dense", "queue", "chain", "stream"])
    group, batch, queued, layers = 64, 1, 0, 1
    if kind == "chain":
        width = rng.choice([1024, 4096])
        active = _log(rng, 8, 72)
        layers = rng.randint(4, 36)
    elif kind == "stream":
        width = rng.choice([512, 1024, 2048])
        active = _log(rng, 8, 32)
        layers = rng.randint(3, 16)
    else:
        width = rng.choice(WIDTHS[1:] if kind == "dense" else WIDTHS)
        active = _log(rng, 9, 240 if width <= 4096 else 110)
        if kind == "batch":
            batch = rng.randint(2, 4)
            group = rng.choice([64, 64, 64, 48, 32])
        elif kind == "dense":
            batch = rng.randint(5, 32)
        elif kind == "layers":
            group = rng.choice([64, 64, 64, 64, 2, 8, 24, 96])
            if group < 64:
                active = min(2000, active * 64 // group)
        elif kind == "queue":
            queued = rng.randint(1, active)
        layers = rng.randint(1, 12)
    groups = active + rng.randint(0, 3 * active)
    c = _case(None, kind if kind in ("queue", "chain", "stream") else "layers", width, groups, active, batch, group,
              layers, queued)
    while c["layers"] > 1 and work(c)["bytes"] > MAX_BYTES:
        c["layers"] -= 1
    return c


# ---------------------------------------------------------------------------- inputs
def _geometry(case):
    G, d = case["group"], case["width"]
    return G, d, G * 3 * d // 2, G * 3 * (d // 128)   # neurons, width, bytes and scales of a group


def _gen(seed, what, device=DEV):
    return torch.Generator(device=device).manual_seed(1000003 * int(seed) + what)


def _inputs(case, seed):
    """Packed weights, scales, x and the active groups of every layer, on the GPU."""
    G, d, gb, sw = _geometry(case)
    L, n = case["layers"], case["groups"]
    cache = torch.randint(0, 256, (L * n * gb,), dtype=torch.uint8, device=DEV, generator=_gen(seed, 1))
    scales = torch.rand(L * n * sw, device=DEV, generator=_gen(seed, 2))
    scales = (case["lo"] + (case["hi"] - case["lo"]) * scales).half()
    x = torch.randn(case["batch"], d, device=DEV, generator=_gen(seed, 3))
    x = x.to(torch.bfloat16 if case["batch"] > 4 else torch.float16)
    g = _gen(seed, 4, "cpu")
    active = torch.stack([torch.randperm(n, generator=g)[: case["active"]] for _ in range(L)])
    # RMSNorm weights of a chain: small, so that layers of random weights keep the stream bounded
    norm = (0.05 + 0.1 * torch.rand(L, d, device=DEV, generator=_gen(seed, 5))).half()
    return cache, scales, x, active, norm


def _rows(case, active, layer):
    """ExecDesc rows: logical id, scale row, slot, destination row, source kind (0: cache arena)."""
    k = case["active"]
    rows = np.zeros((k, 5), dtype=np.uint32)
    rows[:, 0] = active
    rows[:, 1] = rows[:, 2] = layer * case["groups"] + np.asarray(active)
    rows[:, 3] = np.arange(k)
    return rows


class _State:
    """A bound backend, its weights, descriptors and output rows."""

    def __init__(self, case, seed):
        self.case = case
        self.cache, self.scales, self.x, active, self.norm = _inputs(case, seed)
        G, d, _, _ = _geometry(case)
        L, n, k, q = case["layers"], case["groups"], case["active"], case["queued"]
        rows = np.stack([_rows(case, active[l].numpy(), l) for l in range(L)])
        self.core_count = k - q
        self.queue_rows = np.ascontiguousarray(rows[:, k - q:])
        self.core = torch.from_numpy(np.ascontiguousarray(rows[:, : k - q]).astype(np.int32)).cuda()
        self.y = torch.empty(L, case["batch"], d, dtype=torch.float16, device=DEV)
        self.queues = [ReadyQueue(max(1, q)) for _ in range(L if q else 1)]
        self.backend = NativeBackend()
        self.backend.bind(d, G, k, self.cache, self.scales, physical_groups=L * n, cache_groups=L * n,
                          queue_capacity=max(1, q), batch=case["batch"])
        self.epoch = 1
        if not q:   # no streamed groups: an empty queue, sealed once
            self.queues[0].reset(1)
            self.queues[0].seal(0)
        if case["kind"] == "chain":
            self.hidden = torch.empty(L, d, dtype=torch.float16, device=DEV)
            layers = []
            for l in range(L):
                b = dict(core=self.core[l], core_count=k, cache=self.cache, cache_groups=L * n, scales=self.scales,
                         physical_groups=L * n, output=self.y[l, 0], hidden=self.hidden[l], epoch=1, norm_eps=1e-5)
                if l:
                    b["norm_weight"] = self.norm[l]
                else:
                    b["input"] = self.x
                layers.append(b)
            self.blocks = self.backend.chain_blocks(layers)
        torch.cuda.synchronize()

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.backend.close()
            for q in self.queues:
                q.close()
        except Exception:
            pass


class _Stream:
    """A streaming decoder over a pinned host store with this seed's weights and ranks."""

    def __init__(self, case, seed):
        cache, scales, x, active, _ = _inputs(case, seed)
        G, d, _, _ = _geometry(case)
        n, k = case["groups"], case["active"]
        cfg = LayerConfig("stream", d, n * G, k / n, group_size=G, scale_lo=case["lo"], scale_hi=case["hi"])
        self.sd = StreamingDecode(StreamConfig("stream", cfg, layers=case["layers"], arrival_mean_ns=0.0),
                                  arrivals=False)
        assert cfg.active == k
        self.sd.host.copy_(cache)
        self.sd.scales.copy_(scales)
        self.sd.x.copy_(x.reshape(-1))
        # group g of layer l has its bytes and scales at row l * n + g, and is ranked as drawn
        rows = self.sd.layouts
        rows["physical"] = np.arange(len(rows))
        rows["offset"] = np.arange(len(rows), dtype=np.uint64) * cfg.group_bytes
        self.sd.rank_words[:] = active.numpy()
        torch.cuda.synchronize()

    def __del__(self):
        try:
            self.sd.close()
        except Exception:
            pass


def prepare(case, seed):
    return _Stream(case, seed) if case["kind"] == "stream" else _State(case, seed)


# ---------------------------------------------------------------------------- one pass
def run(state):
    if isinstance(state, _Stream):
        state.sd.run()
        return state.sd.y
    s, case = state, state.case
    stream = torch.cuda.current_stream().cuda_stream
    if case["kind"] == "chain":
        s.backend.enqueue_chain(s.blocks, stream)
        return s.y, s.hidden
    if case["kind"] == "queue":
        # a queue is reused only once the launch that consumed it has finished
        while not s.backend.complete():
            pass
        s.epoch = s.epoch % 1000000 + 1
        for l in range(case["layers"]):
            q = s.queues[l]
            q.reset(s.epoch)
            q.write_descriptors(s.queue_rows[l])
            q.seal(case["queued"])
            q.publish_all()
            s.backend.enqueue(l, 0, s.epoch, s.x, s.y[l], stream, s.core[l] if s.core_count else None, s.core_count,
                              q, MODE_PROGRESSIVE)
        return s.y
    core, step = s.core.data_ptr(), 20 * s.core_count
    y, row = s.y.data_ptr(), 2 * s.y[0].numel()
    for l in range(case["layers"]):
        s.backend.enqueue(l, 0, 1, s.x, y + l * row, stream, core + l * step, s.core_count, s.queues[0],
                          MODE_PROGRESSIVE)
    return s.y


# ---------------------------------------------------------------------------- what a pass needs
def work(case):
    G, d, gb, sw = _geometry(case)
    k, L, B = case["active"], case["layers"], case["batch"]
    # each active group's weights and scales once; x in (once for the stack) and y out, 16 bits
    rows = 2 * L + (2 * (L - 1) if case["kind"] == "chain" else 0)   # chain: hidden states, norm weights
    return {"bytes": L * k * (gb + 2 * sw) + 2 * B * d * (1 + L) + 2 * d * (rows - 2 * L),
            "flops": 2 * 3 * d * k * G * L * B}


def tolerance(case):
    # fp16 outputs (rounding: 2.8e-4 of the value) of fp32 sums over h values rounded to fp16 at
    # four places, where a sum taken in another order moves a few of them by one unit in the last
    # place. In a chain every layer's input is the previous layer's fp16 hidden state.
    if case["kind"] == "chain":
        return {"rel": 5e-3}
    return {"rel": 1.5e-3}


# ---------------------------------------------------------------------------- 64-bit reference
def _layer64(case, cache, scales, groups, x):
    """silu(x Wg) * (x Wu) Wd over the groups in 64 bits; x [batch, d] float64. The weights are the
    format's: fp16(q * scale), q the signed nibbles, low nibble first."""
    G, d, gb, sw = _geometry(case)
    y = torch.zeros_like(x)
    for part in torch.as_tensor(groups, device=DEV).split(max(1, (1 << 25) // (G * d))):
        m = len(part)
        b = cache.view(-1, gb)[part].view(m * G * 3, d // 2)
        q = torch.stack([b & 15, b >> 4], dim=-1).view(m * G * 3, d // 128, 128).to(torch.int16)
        q = torch.where(q > 7, q - 16, q).half()
        w = (q * scales.view(-1, sw)[part].view(m * G * 3, d // 128, 1)).view(m * G, 3, d)
        gate, up, down = (w[:, i].double().contiguous() for i in range(3))
        g = x @ gate.t().contiguous()
        h = g / (1 + torch.exp(-g)) * (x @ up.t().contiguous())
        y += h @ down
    return y


def exact(case, seed):
    cache, scales, x, active, norm = _inputs(case, seed)
    n, L = case["groups"], case["layers"]
    x = x.double()
    if case["kind"] == "chain":
        ys, hs, res = [], [], x
        for l in range(L):
            if l:
                inv = 1 / torch.sqrt((res * res).mean(dim=-1, keepdim=True) + 1e-5)
                x = res * inv * norm[l].double()
            y = _layer64(case, cache, scales, l * n + active[l], x)
            res = res + y
            ys.append(y)
            hs.append(res[0])
        return torch.stack(ys), torch.stack(hs)
    out = torch.stack([_layer64(case, cache, scales, l * n + active[l], x) for l in range(L)])
    return out.reshape(L, -1) if case["kind"] == "stream" else out
