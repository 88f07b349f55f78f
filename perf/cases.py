"""The work that a serving process has the EXL3 linear path do, as timed cases.

A vLLM worker calls the quantized layers in four ways, and each kind here is one of them:

* ``linear``  one linear module (its fused shards) called eagerly through its linear method;
* ``block``   the four linear modules of one decoder layer (qkv_proj, o_proj, gate_up_proj,
              down_proj), each on activations of its own, since attention, norms and the
              activation function run between them.  Decode batches and prompt chunks up to 512 rows are replayed from
              a HIP graph, captured once per batch size as decode serving does; other
              prompt chunks run eagerly;
* ``head``    the end of a step: the quantized lm_head's logits, their top k, and the int8
              embedding rows of the next step's tokens.

Shapes are those of the 27B-shaped stack that the benchmark uses (5120 wide, q 6144, k/v
1024, MLP 17408, vocabulary 151936, 2..5 bits per weight, a 6-bit head) and generic smaller
ones.  A drawn case takes any widths (multiples of 128), bits, rows and types in between.
Activations are normal with a few large channels; weights are uniform trellis words with
+-1 input signs and output scales around 1/sqrt(inputs).
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "orcasaq2-kernel_amd"))

import orcasaq2  # noqa: E402,F401
from orcasaq2 import _native  # noqa: E402
from orcasaq2.config import Exl3Config, Exl3LinearMethod  # noqa: E402
from orcasaq2.heads import Exl3EmbeddingMethod  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
SHAPE_27B = dict(hidden=5120, q=6144, kv=1024, inter=17408)
SHAPE_SMALL = dict(hidden=2048, q=2048, kv=512, inter=6144)
MAX_GRAPH_ROWS = 512
SHARD_NAMES = {"qkv": ("q", "k", "v"), "gate_up": (0, 1), "linear": ("q", "k", "v")}


def _block(name, rows, bits, dtype, graph, shape, mcg=False):
    """bits: one digit per tensor, in the order q k v o gate up down."""
    return dict(name=name, kind="block", rows=rows, bits=bits, dtype=dtype, graph=graph, mcg=mcg, **shape)


def listed():
    return [
        # an eager single-sequence call of the smallest fused layer: latency and host path
        dict(name="qkv_1", kind="linear", rows=1, ic=5120, ocs="6144,1024,1024", bits="455", dtype="fp16",
             graph=False, mcg=False),
        # one decode token of one sequence
        _block("block_1", 1, "4553354", "bf16", True, SHAPE_27B),
        # speculative decoding (a drafted token block) or four sequences
        _block("block_4", 4, "3454235", "fp16", True, SHAPE_27B),
        # sixteen sequences
        _block("block_16", 16, "4553344", "bf16", True, SHAPE_27B),
        # a small model serving 24 sequences
        _block("small_24", 24, "4444444", "fp16", True, SHAPE_SMALL),
        # a larger decode batch
        _block("block_48", 48, "4553344", "bf16", True, SHAPE_27B),
        # a short prompt of odd length, not captured
        _block("block_131", 131, "5335243", "fp16", False, SHAPE_27B, mcg=True),
        # chunked prefill in graphs
        _block("block_512", 512, "3454234", "bf16", True, SHAPE_27B),
        # the usual prefill token budget
        _block("block_2048", 2048, "4553344", "bf16", False, SHAPE_27B),
        # a long prompt chunk
        _block("block_4096", 4096, "4353325", "fp16", False, SHAPE_27B),
        # sampling from the top 20 for one sequence; greedy decoding for sixteen
        dict(name="head_1", kind="head", rows=1, hidden=5120, vocab=151936, bits="6", topk=20, dtype="bf16",
             graph=True, mcg=False),
        dict(name="head_16", kind="head", rows=16, hidden=5120, vocab=151936, bits="6", topk=1, dtype="fp16",
             graph=True, mcg=False),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    return 128 * _log_uniform(rng, lo // 128, hi // 128)


def draw(rng):
    kind = rng.choices(("block", "linear", "head"), (5, 3, 2))[0]
    dtype = rng.choice(("fp16", "bf16"))
    mcg = rng.random() < 0.25
    if kind == "head":
        return dict(kind=kind, rows=_log_uniform(rng, 1, 64), hidden=_width(rng, 1024, 5120),
                    vocab=_width(rng, 32000, 151936), bits=str(rng.randint(4, 6)), topk=rng.choice((1, 1, 5, 20, 50)),
                    dtype=dtype, graph=rng.random() < 0.5, mcg=mcg)
    rows = _log_uniform(rng, 1, 4096)
    graph = rows <= MAX_GRAPH_ROWS and rng.random() < 0.7
    if kind == "linear":
        n = rng.choice((1, 1, 2, 3))
        ocs = [_width(rng, 512, 17408 // n) for _ in range(n)]
        return dict(kind=kind, rows=rows, ic=_width(rng, 512, 17408), ocs=",".join(map(str, ocs)),
                    bits="".join(str(rng.randint(2, 6)) for _ in range(n)), dtype=dtype, graph=graph, mcg=mcg)
    hidden = _width(rng, 1024, 5120)
    return dict(kind=kind, rows=rows, hidden=hidden, q=_width(rng, 1024, 6144), kv=_width(rng, 256, 1024),
                inter=_width(rng, 2 * hidden, 17408), bits="".join(str(rng.randint(2, 5)) for _ in range(7)),
                dtype=dtype, graph=graph, mcg=mcg)


# ---------------------------------------------------------------- the modules of a case

def _modules(case):
    """[(name, inputs, [outputs of each shard], [bits of each shard])] of a case."""
    b = [int(c) for c in case["bits"]]
    if case["kind"] == "linear":
        return [("linear", case["ic"], [int(n) for n in case["ocs"].split(",")], b)]
    if case["kind"] == "head":
        return [("lm_head", case["hidden"], [case["vocab"]], b)]
    h, q, kv, inter = case["hidden"], case["q"], case["kv"], case["inter"]
    return [("qkv", h, [q, kv, kv], b[0:3]), ("o", q, [h], b[3:4]), ("gate_up", h, [inter, inter], b[4:6]),
            ("down", inter, [h], b[6:7])]


def _inputs(case, seed):
    """Everything random of a case, from its seed: the modules' tensors and activations, the
    embedding table, its scales and the next tokens."""
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    rows, dtype = case["rows"], DTYPES[case["dtype"]]

    def sign(n):
        return (torch.randint(0, 2, (n,), generator=gen, device=dev) * 2 - 1).half()

    mods = []
    for name, ic, ocs, bits in _modules(case):
        shards = []
        for oc, k in zip(ocs, bits):
            words = torch.randint(-2 ** 31, 2 ** 31, (ic // 16, oc // 16, 8 * k), generator=gen, device=dev,
                                  dtype=torch.int32)
            svh = (torch.randn(oc, generator=gen, device=dev).abs() * 0.8 / math.sqrt(ic)).half() * sign(oc)
            shards.append(dict(trellis=words.view(torch.int16), suh=sign(ic), svh=svh, k=k))
        x = torch.randn(rows, ic, generator=gen, device=dev)
        x[:, torch.randint(0, ic, (4,), generator=gen, device=dev)] *= 10.0
        mods.append(dict(name=name, shards=shards, x=x.to(dtype)))
    out = dict(mods=mods)
    if case["kind"] == "head":
        vocab, hidden = case["vocab"], case["hidden"]
        out["table"] = torch.randint(-128, 128, (vocab, hidden), generator=gen, device=dev, dtype=torch.int8)
        out["scales"] = (torch.rand(vocab, 1, generator=gen, device=dev) * 0.02 + 0.001).to(dtype)
        out["ids"] = torch.randint(0, vocab, (rows,), generator=gen, device=dev)
    return out


# ---------------------------------------------------------------- what a program holds, and its call

def prepare(case, seed):
    got = _inputs(case, seed)
    cfg = Exl3Config.from_config({"bits": 4.0, "codebook": "mcg" if case["mcg"] else "3inst", "head_bits": 6})
    calls = []
    for m in got["mods"]:
        layer, method = torch.nn.Module(), Exl3LinearMethod(cfg, m["name"])
        ic, ocs = m["x"].shape[1], [s["svh"].numel() for s in m["shards"]]
        method.create_weights(layer, ic, ocs, ic, sum(ocs), m["x"].dtype)
        for i, s in enumerate(m["shards"]):
            sid = SHARD_NAMES[m["name"]][i] if m["name"] in SHARD_NAMES else None
            for tensor in ("trellis", "suh", "svh"):
                getattr(layer, tensor).weight_loader(getattr(layer, tensor), s[tensor], sid)
            if case["mcg"]:
                layer.mcg.weight_loader(layer.mcg, torch.ones(1), sid)
        method.process_weights_after_loading(layer)
        calls.append((m["name"], method, layer, m["x"]))
    embed = None
    if case["kind"] == "head":
        embed = (Exl3EmbeddingMethod(), torch.nn.Module())
        embed[0].create_weights(embed[1], case["hidden"], [case["vocab"]], case["hidden"], case["vocab"],
                                DTYPES[case["dtype"]])
        embed[1].qweight.weight_loader(embed[1].qweight, got["table"])
        embed[1].scales.weight_loader(embed[1].scales, got["scales"])
        embed[0].process_weights_after_loading(embed[1])
    state = dict(calls=calls, embed=embed, ids=got.get("ids"), topk=case.get("topk"), graph=None)
    if case["graph"]:
        # as a serving engine captures a batch size: one eager pass, then the capture
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.no_grad():
            with torch.cuda.stream(stream):
                _call(state)
            torch.cuda.current_stream().wait_stream(stream)
            with torch.cuda.graph(graph, stream=stream):
                state["out"] = _call(state)
        state["graph"] = graph
    return state


def _call(state):
    if state["embed"] is None:
        return {name: method.apply(layer, x) for name, method, layer, x in state["calls"]}
    (_, method, layer, x), = state["calls"]
    logits = method.apply_fp16(layer, x)
    values, columns = _native.topk(logits, state["topk"])
    method, layer = state["embed"]
    return dict(logits=logits, values=values, columns=columns, embedding=method.embedding(layer, state["ids"]))


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    with torch.no_grad():
        return _call(state)


# ---------------------------------------------------------------- what a case cannot do without

def work(case):
    rows, nbytes, flops = case["rows"], 0, 0
    for _, ic, ocs, bits in _modules(case):
        nbytes += rows * ic * 2
        for oc, k in zip(ocs, bits):
            nbytes += ic * oc * k // 8 + 2 * (ic + oc) + rows * oc * 2
            flops += 2 * rows * ic * oc
    if case["kind"] == "head":
        nbytes += rows * (case["hidden"] * 3 + 10 + 10 * case["topk"])
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Against the 64-bit result an fp16 output is 3.3e-4 off (activations, weights and outputs
    each rounded to 11 bits) and a bf16 one 1.7e-3 (8 bits); four times that.  The columns of
    equal or nearly equal logits trade places."""
    t = {"rel": 1.4e-3, "max": 0.02} if case["dtype"] == "fp16" or case["kind"] == "head" else {"rel": 7e-3, "max": 0.04}
    if case["kind"] == "head":
        t["differ"] = 0.5
    return t


# ---------------------------------------------------------------- the 64-bit result

_H128 = None


def _hadamard(x):
    """Blocks of 128 along the last dimension times the Sylvester matrix / sqrt(128)."""
    global _H128
    if _H128 is None or _H128.device != x.device:
        h = torch.ones(1, 1, dtype=torch.float64)
        for _ in range(7):
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        _H128 = (h / math.sqrt(128)).to(x.device)
    return (x.reshape(*x.shape[:-1], -1, 128) @ _H128).reshape(x.shape)


def _decode(trellis, k, mcg):
    """The fp16 weights (inputs, outputs) of trellis tiles (rows of tiles, columns of tiles, 16 k int16):
    position t of a tile is the 16 stream bits that end at bit (t + 1) k."""
    dev = trellis.device
    ti, tn, _ = trellis.shape
    words = trellis.contiguous().view(torch.int32).to(torch.int64) & 0xFFFFFFFF
    pos = torch.arange(256, device=dev)
    start = ((pos + 1) * k - 16) % (256 * k)
    at, off = start // 32, start % 32
    state = (((words[..., at] << 32) | words[..., (at + 1) % (8 * k)]) >> (48 - off)) & 0xFFFF
    x = state * 0xCBAC1FED if mcg else state * 89226354 + 64248484
    x = ((x & 0xFFFFFFFF) & 0x8FFF8FFF) ^ 0x3B603B60
    lo, hi = ((v & 0xFFFF).to(torch.int16).view(torch.float16).float() for v in (x, x >> 16))
    j, i = pos // 8, pos % 8
    row = 2 * (j % 4) + torch.tensor([0, 1, 8, 9], device=dev)[i % 4]
    col = j // 4 + 8 * (i // 4)
    tile = torch.empty(ti, tn, 256, dtype=torch.float16, device=dev)
    tile[..., row * 16 + col] = (lo + hi).half()
    return tile.reshape(ti, tn, 16, 16).permute(0, 2, 1, 3).reshape(ti * 16, tn * 16)


def exact(case, seed):
    got = _inputs(case, seed)
    out = {}
    for m in got["mods"]:
        # the path takes its activations in fp16
        x = m["x"].half().double()
        parts = []
        for s in m["shards"]:
            xh = _hadamard(x * s["suh"].double())
            step = max(8, (1 << 26) // x.shape[1] // 128 * 8)
            y = torch.cat([xh @ _decode(s["trellis"][:, c:c + step], s["k"], case["mcg"]).double()
                           for c in range(0, s["trellis"].shape[1], step)], 1)
            parts.append(_hadamard(y) * s["svh"].double())
        out[m["name"]] = torch.cat(parts, 1)
    if case["kind"] != "head":
        return out
    logits = out["lm_head"]
    ids = got["ids"]
    return dict(logits=logits, values=logits.sort(1, descending=True)[0][:, :case["topk"]].contiguous(), columns=None,
                embedding=got["table"][ids].double() * got["scales"][ids].double())
