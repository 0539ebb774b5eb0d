"""The performance cases of this framework, through its public entry points.

Four kinds of work, each over its real range of sizes:

  decode   one launch of a block's compressed weights into its workspace
           (DeviceStore, prepare_batch, decode_batch): what the runtime's
           hook does before every block of a forward
  product  the fused decode and matrix-vector product of the Linears that
           share one input (prepare_matvec, matvec): one-token steps with
           matvec_tokens
  stack    a whole forward of a transformer stack with the runtime attached:
           a prefill run eagerly, or a one-token step replayed from a HIP
           graph, whose blocks are decoded on the fly
  load     the storage archive of a checkpoint decoded on the CPU
           (NeuralZipCompressor.decode)

Weights are N(0, std^2) with 0.1 % of the entries std * Student-t(3), the
statistics the repository's benchmark uses; every tensor of a set takes the
next std of its list, so that larger sets span several codebooks. They are
made from the seed on the GPU.
"""
import gc
import math

import torch
from torch import nn

from neuralzip_amd import _native
from neuralzip_amd.compressor import NeuralZipCompressor
from neuralzip_amd.dtypes import DTYPES
from neuralzip_amd.gpu import decoder as gpu_decoder
from neuralzip_amd.gpu.inference import NeuralZipRuntime, export_model_for_gpu, export_tensors_for_gpu
from neuralzip_amd.setup import NeuralZipSetup

DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
STDS = (0.005, 0.01, 0.02, 0.05, 0.1)
# Bits of the coded byte per element for such weights: the entropy of the
# exponent (bf16, fp32), or of fp16's high byte (sign, exponent and two
# mantissa bits).
CODED_BITS = {"bf16": 2.55, "fp16": 5.5, "fp32": 2.55}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # The smallest call: two odd Linears with a few fragments (the
        # repository's smoke model); launch and latency count.
        dict(name="decode-smoke-bf16", kind="decode", dtype="bf16", shapes="257x513 513x17", one_std=True,
             chunk=16384),
        # One block of the Qwen2-0.5B shape: an ordinary small block.
        dict(name="decode-qwen-block-bf16", kind="decode", dtype="bf16", one_std=True, chunk=262144,
             shapes="896x896 128x896 128x896 896x896 4864x896 4864x896 896x4864"),
        # Eight tensors of Llama-3-8B layer shapes, five stds and so several
        # codebooks: the repository's headline workload and the largest call.
        dict(name="decode-8b-layers-bf16", kind="decode", dtype="bf16", one_std=False, chunk=262144,
             shapes="4096x4096 4096x14336 14336x4096 1024x4096 1024x4096 4096x4096 14336x4096 4096x14336"),
        # The attention weights of a Llama-3-8B layer in fp16, whose coded
        # byte takes more than twice the bits.
        dict(name="decode-8b-attention-fp16", kind="decode", dtype="fp16", one_std=True, chunk=262144,
             shapes="4096x4096 1024x4096 1024x4096 4096x4096"),
        # An MLP kept in fp32 (Qwen2-0.5B shape): three raw byte lanes.
        dict(name="decode-qwen-mlp-fp32", kind="decode", dtype="fp32", one_std=True, chunk=262144,
             shapes="4864x896 4864x896 896x4864"),
        # One-token products of a Llama-3-8B layer: q/k/v together (small),
        # gate/up together (large), down in fp16, and q/k/v with biases for
        # four rows at once.
        dict(name="product-8b-qkv-bf16", kind="product", dtype="bf16", cols=4096, rows="4096 1024 1024", batch=1,
             bias=False),
        dict(name="product-8b-gate-up-bf16", kind="product", dtype="bf16", cols=4096, rows="14336 14336", batch=1,
             bias=False),
        dict(name="product-8b-down-fp16", kind="product", dtype="fp16", cols=14336, rows="4096", batch=1, bias=False),
        dict(name="product-8b-qkv-bf16-b4", kind="product", dtype="bf16", cols=4096, rows="4096 1024 1024", batch=4,
             bias=True),
        # A prompt of 128 tokens through two Llama-3-8B layers and a head,
        # eager: each block decoded on the side stream while the one before
        # it computes.
        dict(name="prefill-8b-2-layers", kind="stack", dtype="bf16", hidden=4096, ffn=14336, heads=32, kv_heads=8,
             layers=2, vocab=32000, tokens=128, cache=128, graph=False),
        # One-token steps of four such layers, replayed from a HIP graph with
        # the decodes captured in it: the serving loop.
        dict(name="step-8b-4-layers-graph", kind="stack", dtype="bf16", hidden=4096, ffn=14336, heads=32, kv_heads=8,
             layers=4, vocab=32000, tokens=1, cache=256, graph=True),
        # Loading a checkpoint: the attention weights of a layer from their
        # storage archive, on the host's cores.
        dict(name="load-8b-attention-bf16", kind="load", dtype="bf16",
             shapes="4096x4096 1024x4096 1024x4096 4096x4096", one_std=True, chunk=262144),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choices(("decode", "product", "stack", "load"), (8, 8, 2, 1))[0]
    dtype = rng.choices(("bf16", "fp16", "fp32"), (4, 2, 2))[0]
    if kind in ("decode", "load"):
        most = {"decode": 120_000_000, "load": 30_000_000}[kind] // (2 if dtype == "fp32" else 1)
        total = _log_uniform(rng, 100_000, most)
        parts = rng.randint(1, 7)
        shapes = []
        for _ in range(parts):
            n = max(64, total // parts)
            cols = min(max(8, _log_uniform(rng, 16, 16384)), n)
            shapes.append("%dx%d" % (max(1, n // cols), cols))
        return dict(kind=kind, dtype=dtype, shapes=" ".join(shapes), one_std=rng.random() < 0.5,
                    chunk=rng.choice((65536, 262144, 262144, 1 << 20)))
    if kind == "product":
        # rows of at least one tile, in whole 16-byte vectors
        cols = 8 * _log_uniform(rng, 256, 2048)
        total = _log_uniform(rng, 64, 100_000_000 // cols)
        parts = rng.randint(1, 4)
        rows = [max(1, int(total * rng.uniform(0.3, 1.0) / parts)) for _ in range(parts)]
        return dict(kind=kind, dtype=dtype, cols=cols, rows=" ".join(map(str, rows)), batch=rng.randint(1, 4),
                    bias=rng.random() < 0.5)
    hidden = 128 * rng.randint(4, 24)
    graph = rng.random() < 0.5
    tokens = 1 if graph else _log_uniform(rng, 2, 256)
    return dict(kind=kind, dtype="bf16", hidden=hidden, ffn=64 * _log_uniform(rng, 16, 160), heads=hidden // 64,
                kv_heads=hidden // 128, layers=rng.randint(2, 4), vocab=_log_uniform(rng, 1000, 32000), tokens=tokens,
                cache=tokens + rng.randint(0, 100), graph=graph)


# ------------------------------------------------------------------ inputs

def _shapes(case):
    return [tuple(map(int, s.split("x"))) for s in case["shapes"].split()]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _weight(shape, std, dtype, g):
    """N(0, std^2) with 0.1 % of the entries std * Student-t(3)."""
    w = torch.randn(shape, generator=g, device="cuda").mul_(std)
    flat = w.view(-1)
    n = flat.numel() // 1000
    if n:
        # one place in every thousand
        at = torch.arange(n, device="cuda") * 1000 + torch.randint(0, 1000, (n,), generator=g, device="cuda")
        z = torch.randn((4, n), generator=g, device="cuda")
        flat[at] = std * z[0] / (z[1:].square().sum(0) / 3).sqrt()
    return w.to(dtype)


def _tensors(case, seed):
    g, dtype = _generator(seed), DTYPE[case["dtype"]]
    return {"layers.%d.weight" % i: _weight(shape, 0.02 if case["one_std"] else STDS[i % len(STDS)], dtype, g)
            for i, shape in enumerate(_shapes(case))}


def _product_tensors(case, seed):
    g, dtype = _generator(seed), DTYPE[case["dtype"]]
    rows = [int(r) for r in case["rows"].split()]
    weights = [_weight((r, case["cols"]), 0.02, dtype, g) for r in rows]
    x = torch.randn((case["batch"], case["cols"]), generator=g, device="cuda").to(dtype)
    biases = [torch.randn(r, generator=g, device="cuda").mul_(0.1).to(dtype) for r in rows] if case["bias"] else None
    return weights, x, biases


def _store(tensors, setup):
    """The packed device store of {name: tensor}, each tensor's fragments and
    workspace offset, and the workspace's elements."""
    exported = export_tensors_for_gpu(tensors, setup)
    entries, members, offsets, offset, frag = [], {}, {}, 0, 0
    for layout, ids, _, _, name in exported.tensors:
        entries.append((layout, ids, offset))
        members[name], offsets[name] = list(range(frag, frag + layout.n_fragments)), offset
        frag += layout.n_fragments
        offset = (offset + tensors[name].numel() + 127) // 128 * 128
    store = gpu_decoder.DeviceStore(exported.codebooks, entries, torch.device("cuda", torch.cuda.current_device()))
    return store, members, offsets, offset


def _prepare_decode(case, seed):
    tensors = _tensors(case, seed)
    dtype = DTYPE[case["dtype"]]
    setup = NeuralZipSetup(cluster_js_threshold=0.05, chunk_size=case["chunk"]).build(tensors)
    store, members, offsets, size = _store(tensors, setup)
    workspace = torch.zeros(max(size, 1), dtype=dtype, device="cuda")
    views = {name: workspace[offset:offset + tensors[name].numel()].view(tensors[name].shape)
             for name, offset in offsets.items()}
    kinds = {}
    for f in (f for fs in members.values() for f in fs):
        kinds.setdefault(int(store.descs[f]["kind"]) == _native.KIND_LONG, []).append(f)
    decoder = gpu_decoder.default_decoder()
    batches = [decoder.prepare_batch(store, fs, DTYPES[dtype], workspace) for _, fs in sorted(kinds.items())]
    return dict(kind="decode", decoder=decoder, batches=batches, views=views, store=store)


def _prepare_product(case, seed):
    weights, x, biases = _product_tensors(case, seed)
    dtype = DTYPE[case["dtype"]]
    tensors = {"layers.%d.weight" % i: w for i, w in enumerate(weights)}
    setup = NeuralZipSetup(cluster_js_threshold=0.05).build(tensors)
    store, members, offsets, _ = _store(tensors, setup)
    decoder = gpu_decoder.default_decoder()
    weights = [(members[name], offsets[name], w.shape[0]) for name, w in tensors.items()]
    plan = decoder.prepare_matvec(store, weights, DTYPES[dtype], case["cols"])
    partials = torch.empty(2 * plan.n_tiles * case["batch"], dtype=torch.float32, device="cuda")
    return dict(kind="product", decoder=decoder, plan=plan, x=x, biases=biases, partials=partials)


class _Block(nn.Module):
    """A pre-norm attention and gated-MLP layer with a static KV cache."""

    def __init__(self, c):
        super().__init__()
        h, head = c["hidden"], c["hidden"] // c["heads"]
        self.c, self.head = c, head
        kv = c["kv_heads"] * head
        self.q, self.k, self.v, self.o = (nn.Linear(h, n, bias=False) for n in (h, kv, kv, h))
        self.gate, self.up = nn.Linear(h, c["ffn"], bias=False), nn.Linear(h, c["ffn"], bias=False)
        self.down = nn.Linear(c["ffn"], h, bias=False)

    def forward(self, x, keys, values, mask):
        c, t = self.c, x.shape[0]
        h = _norm(x)
        first = c["cache"] - c["tokens"]     # earlier tokens' keys and values are in the cache
        keys[first:] = self.k(h).view(t, c["kv_heads"], self.head)
        values[first:] = self.v(h).view(t, c["kv_heads"], self.head)
        q = self.q(h).view(t, c["heads"], self.head)
        x = x + self.o(_attention(q, keys, values, mask, c).to(x.dtype))
        h = _norm(x)
        return x + self.down(nn.functional.silu(self.gate(h)) * self.up(h))


class _Stack(nn.Module):
    def __init__(self, c):
        super().__init__()
        self.layers = nn.ModuleList([_Block(c) for _ in range(c["layers"])])
        self.head = nn.Linear(c["hidden"], c["vocab"], bias=False)

    def forward(self, x, caches, mask):
        for layer, (keys, values) in zip(self.layers, caches):
            x = layer(x, keys, values, mask)
        return self.head(_norm(x))


def _norm(x):
    wide = x if x.dtype == torch.float64 else x.float()
    return (wide * torch.rsqrt(wide.square().mean(-1, keepdim=True) + 1e-5)).to(x.dtype)


def _attention(q, keys, values, mask, c):
    """Grouped-query attention in fp32 (fp64 for fp64 inputs): (tokens, hidden)."""
    wide = torch.float64 if q.dtype == torch.float64 else torch.float32
    repeat = c["heads"] // c["kv_heads"]
    k = keys.to(wide).repeat_interleave(repeat, 1).permute(1, 2, 0).contiguous()
    v = values.to(wide).repeat_interleave(repeat, 1).transpose(0, 1).contiguous()
    scores = torch.matmul(q.to(wide).transpose(0, 1).contiguous(), k) / math.sqrt(q.shape[-1]) + mask.to(wide)
    return torch.matmul(scores.softmax(-1), v).transpose(0, 1).reshape(q.shape[0], -1)


def _stack_inputs(case, seed):
    g, dtype = _generator(seed), DTYPE[case["dtype"]]
    with torch.device("meta"):
        model = _Stack(case)
    model = model.to(dtype).to_empty(device="cuda").requires_grad_(False).eval()
    for p in model.parameters():
        p.copy_(_weight(p.shape, 0.02, dtype, g))
    x = torch.randn((case["tokens"], case["hidden"]), generator=g, device="cuda").to(dtype)
    shape = (case["cache"], case["kv_heads"], case["hidden"] // case["heads"])
    caches = [tuple(torch.randn(shape, generator=g, device="cuda").to(dtype) for _ in range(2))
              for _ in range(case["layers"])]
    at = torch.arange(case["cache"], device="cuda")
    mask = torch.where(at[None, :] > at[case["cache"] - case["tokens"]:, None], -torch.inf, 0.0)
    return model, x, caches, mask


def _prepare_stack(case, seed):
    model, x, caches, mask = _stack_inputs(case, seed)
    setup = NeuralZipSetup(cluster_js_threshold=0.05).build(model)
    runtime = NeuralZipRuntime.attach(model, export_model_for_gpu(model, setup))
    state = dict(kind="stack", model=model, x=x, caches=caches, mask=mask, graph=None)
    if not case["graph"]:
        return state
    state["input"] = torch.zeros_like(x)
    gc.collect()     # nothing of an earlier capture is freed while this one runs
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                model(state["input"], caches, mask)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with runtime.graph_capture(), torch.cuda.graph(state["graph"]):
            state["logits"] = model(state["input"], caches, mask)
    torch.cuda.synchronize()
    return state


def _prepare_load(case, seed):
    tensors = _tensors(case, seed)
    setup = NeuralZipSetup(cluster_js_threshold=0.05, chunk_size=case["chunk"]).build(tensors)
    blob, metadata, _, _ = NeuralZipCompressor(setup).encode(tensors.items())
    return dict(kind="load", blob=blob, metadata=metadata)


def prepare(case, seed):
    return {"decode": _prepare_decode, "product": _prepare_product, "stack": _prepare_stack,
            "load": _prepare_load}[case["kind"]](case, seed)


# ------------------------------------------------------------------ one pass

def run(state):
    kind = state["kind"]
    if kind == "decode":
        for batch in state["batches"]:
            state["decoder"].decode_batch(batch)
        return state["views"]
    if kind == "product":
        return list(state["decoder"].matvec(state["plan"], state["x"], state["biases"], state["partials"]))
    if kind == "load":
        return NeuralZipCompressor().decode(state["blob"], state["metadata"])
    with torch.no_grad():
        if state["graph"] is None:
            return state["model"](state["x"], state["caches"], state["mask"])
        state["input"].copy_(state["x"])     # the step's token
        state["graph"].replay()
        return state["logits"]


# ------------------------------------------------------------------ what a pass needs

def _coded_bytes(elements, dtype):
    """The compressed form: raw byte lanes and the coded lane's bits."""
    return elements * (DTYPE[dtype].itemsize - 1 + CODED_BITS[dtype] / 8)


def work(case):
    size = DTYPE[case["dtype"]].itemsize
    if case["kind"] in ("decode", "load"):
        n = sum(math.prod(s) for s in _shapes(case))
        return {"bytes": _coded_bytes(n, case["dtype"]) + n * size, "flops": 0}
    if case["kind"] == "product":
        rows = sum(int(r) for r in case["rows"].split())
        n = rows * case["cols"]
        vectors = case["batch"] * (case["cols"] + rows) + (rows if case["bias"] else 0)
        return {"bytes": _coded_bytes(n, case["dtype"]) + vectors * size, "flops": 2 * n * case["batch"]}
    h, kv = case["hidden"], case["kv_heads"] * (case["hidden"] // case["heads"])
    n = case["layers"] * (2 * h * h + 2 * kv * h + 3 * h * case["ffn"]) + h * case["vocab"]
    t = case["tokens"]
    attention = 4 * case["layers"] * t * case["cache"] * h
    # the compressed weights once, the decoded words once each way, the cache and the token rows
    moved = _coded_bytes(n, "bf16") + 4 * n + 4 * case["layers"] * case["cache"] * kv + 2 * t * (h + case["vocab"])
    return {"bytes": moved, "flops": 2 * n * t + attention}


def tolerance(case):
    if case["kind"] in ("decode", "load"):
        return "exact"     # decoded weights are the original words
    if case["kind"] == "product":
        # fp32 sums rounded once to the weight's dtype
        return {"rel": {"bf16": 6e-3, "fp16": 8e-4, "fp32": 2e-6}[case["dtype"]]}
    return {"rel": 2e-2}   # bf16 activations through every layer


def exact(case, seed):
    if case["kind"] == "decode":
        return {name: t.double() for name, t in _tensors(case, seed).items()}
    if case["kind"] == "load":
        return {name: t.double().cpu() for name, t in _tensors(case, seed).items()}
    if case["kind"] == "product":
        weights, x, biases = _product_tensors(case, seed)
        ys = [x.double() @ w.double().t() for w in weights]
        return [y + b.double() for y, b in zip(ys, biases)] if biases else ys
    with torch.no_grad():
        model, x, caches, mask = _stack_inputs(case, seed)
        return model.double()(x.double(), [(k.double(), v.double()) for k, v in caches], mask.double())
