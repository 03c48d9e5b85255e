"""The workloads whose speed this repository is measured by: the MoE half of MiMo-V2.6-Flash decoder layers from one
decoded token to a whole prompt chunk, a small configuration where call overhead counts, and the MXFP4 codec that
converts a checkpoint.

`listed()` holds the named cases and `draw` makes others of the same ranges; `prepare` builds a case's inputs on the
GPU from a seed, `run` is one pass through the public entry points, `work` what such a pass cannot do without,
`tolerance` how far a correct result may be off, and `exact` the same pass in 64 bits by plain torch.
"""
import functools
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mimo-on-a-mac_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

EPS = 1e-5
WEIGHT_STD = 0.02        # expert and router weights, as the reference's test pools
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)

# hidden, intermediate, experts, routes per row
MIMO = (4096, 2048, 256, 8)
SMALL = ((256, 512, 8, 2), (512, 1024, 16, 3), (1024, 512, 32, 4), (2048, 1024, 64, 6))


def _layer(op, rows, dims=MIMO, layers=1, skew=0.0, shared=0.0, graph=False):
    H, I, E, k = dims
    return {"op": op, "rows": rows, "hidden": H, "inter": I, "experts": E, "top_k": k, "layers": layers, "skew": skew,
            "shared": shared, "graph": graph}


def _codec(op, rows, cols):
    return {"op": op, "rows": rows, "cols": cols}


def listed():
    # skew 0.22: expert popularity as measured on MiMo's middle layers (top experts chosen 6-7 times as often as the
    # average); shared 0.8: consecutive rows of one sequence choose about 2.5 of their 8 experts alike
    return [
        # a small model's block on a few rows: the call's own latency, nothing to stream
        dict(_layer("block", 4, dims=SMALL[0]), name="small_block_4"),
        # one decoded token through one layer, called from Python as an engine without graphs does
        dict(_layer("layer", 1), name="layer_decode_1"),
        # one decoded token through a run of layers in a captured graph, as a serving loop replays them
        dict(_layer("layer", 1, layers=6, skew=0.22, graph=True), name="graph_decode_1"),
        # four rows per step (a small batch, or a speculative verify) through the same
        dict(_layer("layer", 4, layers=6, skew=0.22, shared=0.8, graph=True), name="graph_decode_4"),
        # the widest verify step
        dict(_layer("layer", 8, skew=0.22, shared=0.8), name="layer_decode_8"),
        # a short follow-up turn
        dict(_layer("layer", 24, skew=0.22), name="layer_prefill_24"),
        # a prompt of ragged length
        dict(_layer("layer", 137, skew=0.22), name="layer_prefill_137"),
        # chunks of a prompt, with near-uniform and with measured-like popularity
        dict(_layer("layer", 512), name="layer_prefill_512"),
        dict(_layer("layer", 2048, skew=0.22), name="layer_prefill_2048"),
        # a whole prompt in one chunk, off every multiple of a tile
        dict(_layer("layer", 6250, skew=0.22), name="layer_prefill_6250"),
        # checkpoint conversion: gate rows of 32 experts to MXFP4, and down rows back
        dict(_codec("quantize", 65536, 4096), name="quantize_65536"),
        dict(_codec("dequantize", 65536, 2048), name="dequantize_65536"),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.random()
    skew = round(rng.uniform(0.0, 0.3), 2)
    if kind < 0.3:
        graph = rng.random() < 0.5
        return _layer("layer", rng.randint(1, 8), layers=rng.randint(2, 6) if graph else 1, skew=skew,
                      shared=round(rng.uniform(0.0, 0.9), 2), graph=graph)
    if kind < 0.75:
        return _layer("layer", spread(9, 6250), skew=skew)
    if kind < 0.88:
        return _layer("block", spread(1, 1024), dims=rng.choice(SMALL), skew=skew)
    return _codec("quantize" if rng.random() < 0.5 else "dequantize", spread(1024, 65536),
                  rng.choice((256, 1024, 2048, 4096)))


# ------------------------------------------------------------------ inputs (torch alone, from the seed)
def _generator(seed, part):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + part) % (1 << 62))


def _weight_rows(rows, cols, g):
    """Codes [rows, cols / 8] int32 and scales [rows, cols / 32] uint8: MXFP4 of N(0, WEIGHT_STD) values."""
    v = (torch.randn(rows, cols // 32, 32, generator=g, device="cuda") * WEIGHT_STD).to(torch.bfloat16).float()
    e = torch.frexp(v.abs().amax(-1)).exponent - 3          # floor(log2(amax)) - 2
    y = torch.ldexp(v, -e[..., None])
    m = y.abs()
    grid = torch.tensor(E2M1, device="cuda")
    code = torch.bucketize(m, (grid[1:] + grid[:-1]) / 2).int() + torch.where(y < 0, 8, 0).int()
    code = code.reshape(rows, cols // 8, 8)
    word = torch.zeros(rows, cols // 8, dtype=torch.int32, device="cuda")
    for j in range(8):
        word |= code[..., j] << (4 * j)
    return word, (e + 127).to(torch.uint8)


def _pool(slots, out, cols, g):
    """A projection's pool: every weight row one of 8192 quantised rows, drawn anew for each slot and output."""
    word, scale = _weight_rows(8192, cols, g)
    at = torch.randint(8192, (slots * out,), generator=g, device="cuda")
    return (word.index_select(0, at).view(slots, out, cols // 8),
            scale.index_select(0, at).view(slots, out, cols // 32))


def _layer_inputs(case, seed, part):
    """One layer's tensors: bank, router weight and bias, norm weight, rows."""
    H, I, E = case["hidden"], case["inter"], case["experts"]
    g = _generator(seed, part)
    bank = {}
    for name, (out, cols) in {"gate": (I, H), "up": (I, H), "down": (H, I)}.items():
        bank[name + "_w"], bank[name + "_s"] = _pool(E, out, cols, g)
    W = (torch.randn(E, H, generator=g, device="cuda") * WEIGHT_STD).to(torch.bfloat16)
    rank = torch.randperm(E, generator=g, device="cuda").float()
    bias = -case["skew"] * torch.log(rank + 1.0) / math.log(E)
    norm = (1.0 + 0.1 * torch.randn(H, generator=g, device="cuda")).to(torch.bfloat16)
    a = case["shared"]
    x = (a * torch.randn(1, H, generator=g, device="cuda")
         + math.sqrt(1.0 - a * a) * torch.randn(case["rows"], H, generator=g, device="cuda")).to(torch.bfloat16)
    return bank, W, bias, norm, x


def _codec_inputs(case, seed):
    g = _generator(seed, 0)
    if case["op"] == "quantize":
        return ((torch.randn(case["rows"], case["cols"], generator=g, device="cuda") * WEIGHT_STD).to(torch.bfloat16),)
    word, scale = _weight_rows(min(case["rows"], 8192), case["cols"], g)
    at = torch.randint(word.shape[0], (case["rows"],), generator=g, device="cuda")
    return word.index_select(0, at), scale.index_select(0, at)


# ------------------------------------------------------------------ the framework
def _make(case, seed, part):
    from mimo_stream import MoEBlock, MoELayer, Router
    bank, W, bias, norm, x = _layer_inputs(case, seed, part)
    router = Router(case["hidden"], case["experts"], case["top_k"])
    router.weight.copy_(W)
    router.e_score_correction_bias.copy_(bias)
    block = MoEBlock(router, bank)
    return (MoELayer(block, norm, EPS) if case["op"] == "layer" else block), x


def prepare(case, seed):
    if case["op"] in ("quantize", "dequantize"):
        return {"op": case["op"], "inputs": _codec_inputs(case, seed)}
    pairs = [_make(case, seed, n) for n in range(case["layers"])]
    state = {"op": case["op"], "pairs": pairs}
    if case["graph"]:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            for call, x in pairs:
                call(x)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            state["outputs"] = [call(x) for call, x in pairs]
        state["graph"] = graph
    return state


def run(state):
    if state["op"] == "quantize":
        from mimo_stream.kernels import quantize_mxfp4
        return quantize_mxfp4(*state["inputs"])
    if state["op"] == "dequantize":
        from mimo_stream.kernels import dequantize_mxfp4
        return dequantize_mxfp4(*state["inputs"])
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    return [call(x) for call, x in state["pairs"]]


# ------------------------------------------------------------------ what a pass needs
@functools.lru_cache(maxsize=None)
def _distinct_experts(rows, E, k, skew, shared, spread):
    """Experts that at least one row chooses, for routes drawn as prepare() draws them."""
    g = torch.Generator().manual_seed(1)
    logits = shared * torch.randn(1, E, generator=g) + math.sqrt(1.0 - shared * shared) * torch.randn(rows, E, generator=g)
    bias = -skew * torch.log(torch.arange(E) + 1.0) / math.log(E)
    return torch.unique((torch.sigmoid(spread * logits) + bias).topk(k).indices).numel()


def work(case):
    rows = case["rows"]
    if case["op"] in ("quantize", "dequantize"):
        n = rows * case["cols"]
        return {"bytes": n * (2 if case["op"] == "quantize" else 4) + n // 2 + n // 32, "flops": 0}
    H, I, E, k = case["hidden"], case["inter"], case["experts"], case["top_k"]
    U = _distinct_experts(rows, E, k, case["skew"], case["shared"], WEIGHT_STD * math.sqrt(H))
    expert = 3 * H * I // 2 + 3 * H * I // 32
    size = U * expert + 2 * E * H + 4 * rows * H
    flops = 2 * rows * E * H + 6 * rows * k * H * I
    return {"bytes": case["layers"] * size, "flops": case["layers"] * flops}


def tolerance(case):
    if case["op"] in ("quantize", "dequantize"):
        return "exact"
    return {"rel": 1e-2, "max": 5e-2}


# ------------------------------------------------------------------ 64 bits
def _dequantize64(word, scale):
    shift = torch.arange(0, 32, 4, device=word.device, dtype=torch.int32)
    code = (word[..., None] >> shift) & 15
    grid = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=word.device)
    v = grid[code.long()].reshape(*scale.shape, 32)
    return torch.ldexp(v, scale.to(torch.int32)[..., None] - 127).reshape(*word.shape[:-1], word.shape[-1] * 8)


def _exact_layer(case, seed, part):
    bank, W, bias, norm, x = _layer_inputs(case, seed, part)
    k = case["top_k"]
    r = x
    if case["op"] == "layer":     # the norm's two bf16 roundings are part of the layer: the router reads its bf16 rows
        x64 = x.double()
        unit = (x64 / torch.sqrt(x64.square().mean(-1, keepdim=True) + EPS)).to(torch.bfloat16)
        r = (norm.double() * unit.double()).to(torch.bfloat16)
    r = r.double()
    score = torch.sigmoid(r @ W.double().T)
    inds = (score + bias.double()).topk(k).indices
    w = score.gather(1, inds)
    w = w / w.sum(-1, keepdim=True)
    y = torch.zeros_like(r)
    for e in torch.unique(inds).tolist():
        row, j = (inds == e).nonzero(as_tuple=True)
        rows = r[row]
        gate, up, down = (_dequantize64(bank[p + "_w"][e], bank[p + "_s"][e]) for p in ("gate", "up", "down"))
        a = rows @ gate.T
        y.index_add_(0, row, ((a * torch.sigmoid(a) * (rows @ up.T)) @ down.T) * w[row, j][:, None])
    return x.double() + y if case["op"] == "layer" else y


def exact(case, seed):
    if case["op"] == "quantize":
        return None                      # codes and scales: whole numbers
    if case["op"] == "dequantize":
        return _dequantize64(*_codec_inputs(case, seed))
    return [_exact_layer(case, seed, part) for part in range(case["layers"])]
