"""Timing cases of the MoE layer: what a program that uses this package calls, at the sizes it calls it with.

Six paths, each through the public entry point a user's program reaches it by:

``layer``     forward of ``MixMOETransformerMLP`` without gradients, the whole layer as one call (prefill, encoders)
``staged``    the same module with ``fused=False``: gate, routing, the two expert products and the combine one call
              after the other, in the reference's own order of calls (decode and short prompts)
``train``     forward and backward of the same module, returning the output and every gradient
``segments``  ``ops.moe_ffn_segments``: one GPU's share of an expert-parallel layer, an inbound buffer of rows
              addressed by (start, length, expert) triples
``blocks``    ``mix_moe_hip.MixMOE.forward``: the reference's extension object with its 64-row block arrays and
              its transposed [E, K, N] weights
``gate``      gate, counts and positions alone (``AsyncExpertAssignment.process_data``), with an fp32 router

``listed()`` are fixed cases, ``draw()`` makes more of the same ranges.  The model sizes are the repository's own
(``ccfuser_amd/workloads.py``: 256/1024, 1024/4096, 4096/14336, 2048/8192, 768/3072) and generic widths.
"""
import math

import torch

from ccfuser_amd import mix_moe_hip, ops
from ccfuser_amd.mix_moe import MixMOETransformerMLP
from ccfuser_amd.mix_moe.gates import NaiveGate
from ccfuser_amd.mix_moe.transformer import AsyncExpertAssignment

_POPULAR = 3                 # spare expert slots of MixMOETransformerMLP's parameters (its default)
_BLOCK = 64                  # rows of a block of the reference's block arrays


def _case(name, kind, tokens, d, f, experts, top_k, capacity=0.0, skew=0.0, sources=0):
    """``capacity``: capacity factor, 0 = no limit.  ``skew``: exponent of the experts' Zipf loads, 0 = even.
    ``sources``: source ranks of an inbound buffer."""
    c = {"kind": kind, "tokens": tokens, "d": d, "f": f, "experts": experts, "top_k": top_k,
         "capacity": capacity, "skew": skew, "sources": sources}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one sequence being decoded: a single token, two experts, launches and weight bytes only
        _case("decode_1", "staged", 1, 4096, 14336, 8, 2),
        # a decoding batch: a few dozen rows per expert, every expert's weights read once
        _case("decode_128", "staged", 128, 4096, 14336, 8, 2),
        # a short prompt of odd length: under a tile of rows per expert
        _case("prefill_333", "staged", 333, 4096, 14336, 8, 2),
        # the repository's benchmark: a full prefill batch
        _case("prefill_4096", "layer", 4096, 4096, 14336, 8, 2),
        # a toy layer: five short kernels, host work and launches count
        _case("small_512", "layer", 512, 256, 1024, 4, 1),
        # GShard-like encoder layer, overflow beyond the capacity dropped
        _case("capacity_8192", "layer", 8192, 1024, 4096, 8, 2, capacity=1.25),
        # switch layer with many small experts and loads from thousands of rows to none
        _case("skewed_32768", "layer", 32768, 768, 3072, 32, 1, skew=1.5),
        # the rows that eight ranks sent to this GPU's eight experts
        _case("segments_16384", "segments", 16384, 2048, 8192, 8, 1, skew=1.2, sources=8),
        # the reference's own kernel shapes through its extension interface
        _case("blocks_8192", "blocks", 8192, 1024, 4096, 16, 2),
        # one training step of a GPT-2 / BERT sized layer on an odd number of tokens
        _case("train_1999", "train", 1999, 768, 3072, 8, 2),
        # one training step at the benchmark's shape
        _case("train_4096", "train", 4096, 4096, 14336, 8, 2),
        # router kept in fp32, ahead of the experts
        _case("gate_fp32_8192", "gate", 8192, 2048, 8192, 64, 2),
    ]


_MODELS = ((256, 1024), (1024, 4096), (4096, 14336), (2048, 8192), (768, 3072))
_MAX_FORWARD_FLOPS = 4.0 * 2 * 4096 * 4096 * 14336          # the largest forward listed
_MAX_WEIGHTS = 8 * 4096 * 14336                             # elements of one expert matrix over all experts


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("layer", "staged", "train", "segments", "blocks", "gate"), (8, 6, 6, 3, 3, 2))[0]
    if rng.random() < 0.5:
        d, f = rng.choice(_MODELS)
    else:                                                   # any multiple of 64
        d = 64 * _log_int(rng, 4, 64)
        f = 4 * d if kind == "staged" else 64 * int(round(d * rng.uniform(3.0, 4.0) / 64))
    experts = rng.choice((4, 8, 8, 16, 32))
    while experts * d * f > _MAX_WEIGHTS:
        experts //= 2
    top_k = rng.choice((1, 2, 2))
    capacity = skew = 0.0
    sources = 0

    def batch(rows_lo, rows_hi, most=32768):                # tokens that give an expert that many rows on average
        lo = -(-rows_lo * experts // top_k)
        return min(_log_int(rng, lo, max(lo, rows_hi * experts // top_k)), most)

    if kind == "layer":
        tokens = batch(128, 4096)
        capacity = rng.choice((0.0, 0.0, 1.25))
        skew = rng.choice((0.0, 0.0, 1.5))
    elif kind == "staged":                                  # one sequence, or a batch of them
        tokens = 1 if rng.random() < 0.3 else batch(32, 256)
    elif kind == "train":
        tokens = batch(64, 1024)
        capacity = rng.choice((0.0, 0.0, 1.25))
    elif kind == "segments":
        top_k = 1
        tokens = batch(128, 2048)
        skew, sources = rng.choice((0.0, 1.2)), rng.choice((2, 4, 8))
    elif kind == "blocks":
        top_k = 2
        tokens = batch(16, 1024, 16384)
    else:
        tokens = _log_int(rng, 1, 32768)
        experts = rng.choice((8, 16, 32, 64))
    while kind != "gate" and 4.0 * tokens * top_k * d * f > _MAX_FORWARD_FLOPS:
        tokens = (tokens + 1) // 2
    return _case(None, kind, tokens, d, f, experts, top_k, capacity, skew, sources)


# ---------------------------------------------------------------- inputs
def _zipf(experts, skew):
    """Shares of the experts' loads, largest first."""
    w = [r ** -skew for r in range(1, experts + 1)]
    return [v / sum(w) for v in w]


class _Maker:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(self, *shape, std=1.0, dtype=torch.float16):
        t = torch.empty(*shape, dtype=dtype, device="cuda")
        return t.normal_(0.0, std, generator=self.gen)

    def fill(self, param, std=0.02):
        with torch.no_grad():
            param.normal_(0.0, std, generator=self.gen)

    def gate_bias(self, gate, d, skew):
        """A bias that gives the experts Zipf loads: the logits' noise is about 0.02 sqrt(d) wide, a Gumbel
        variable's pi / sqrt(6), and a Gumbel argmax follows the softmax of the bias."""
        self.fill(gate.bias)
        if skew:
            E = gate.bias.numel()
            rank = torch.randperm(E, generator=self.gen, device="cuda").float() + 1.0
            ratio = 0.02 * math.sqrt(d) / (math.pi / math.sqrt(6.0))
            with torch.no_grad():
                gate.bias.add_((-skew * ratio * rank.log()).to(gate.bias.dtype))


def _module(case, mk):
    d, f, E = case["d"], case["f"], case["experts"]
    with torch.device("cuda"):
        mlp = MixMOETransformerMLP("naive", {"num_local_expert": E, "hidden_size": f}, d, 0, 1,
                                   total_batch_size=case["tokens"], top_k=case["top_k"],
                                   capacity_factor=case["capacity"] or None, fused=case["kind"] != "staged").half()
    mk.fill(mlp.gate.gate.weight)
    mk.gate_bias(mlp.gate.gate, d, case["skew"])
    for lin in (mlp.experts.htoh4, mlp.experts.h4toh):
        mk.fill(lin.weight)
        mk.fill(lin.bias)
    return mlp


def _segments(case, mk):
    """Per source rank one contiguous span of rows, grouped by local expert."""
    R, E, S = case["tokens"], case["experts"], case["sources"]
    share = torch.tensor(_zipf(E, case["skew"]))
    share = share[torch.randperm(E, generator=mk.gen, device="cuda").cpu()].cuda()
    expert = torch.multinomial(share, R, replacement=True, generator=mk.gen).cpu()
    cuts = torch.rand(S - 1, generator=mk.gen, device="cuda").mul_(R).long().sort().values.cpu().tolist()
    start, length, owner = [], [], []
    for lo, hi in zip([0] + cuts, cuts + [R]):
        at = lo
        for e, n in enumerate(torch.bincount(expert[lo:hi], minlength=E).tolist()):
            if n:
                start.append(at)
                length.append(n)
                owner.append(e)
                at += n
    return [torch.tensor(v, dtype=torch.int32, device="cuda") for v in (start, length, owner)]


def prepare(case, seed):
    mk = _Maker(seed)
    T, d, f, E, k = (case[n] for n in ("tokens", "d", "f", "experts", "top_k"))
    kind = case["kind"]
    st = {"kind": kind, "E": E}
    if kind in ("layer", "staged", "train"):
        st["mlp"] = _module(case, mk)
        st["x"] = mk.randn(T, d)
        if kind == "train":
            st["x"].requires_grad_(True)
            st["grad"] = mk.randn(T, d, std=0.1)
        else:
            st["mlp"].requires_grad_(False)
    elif kind == "segments":
        st["args"] = [mk.randn(T, d), *_segments(case, mk), mk.randn(E, f, d, std=0.02), mk.randn(E, f, std=0.02),
                      mk.randn(E, d, f, std=0.02), mk.randn(E, d, std=0.02)]
    elif kind == "blocks":
        # a router's choice per token, then the arrays the reference's planner hands to the extension
        idx = torch.rand(T, E, generator=mk.gen, device="cuda").topk(k, dim=-1).indices
        r = ops.route(idx.reshape(-1), E, k)
        plan = ops.plan_blocks(r["counts"], T * k)
        total, remote = plan["block_nums"].tolist()
        st["args"] = [mk.randn(T, d), r["pos"], plan["expert_ids"][:total], plan["ranks"][:total],
                      plan["lens"][:total], plan["start_addrs"][:total], total, remote]
        # weights as the reference passes them: [E, K, N]
        st["moe"] = mix_moe_hip.MixMOE(1, T, E, k, d, f, _BLOCK, mk.randn(E, d, f, std=0.02),
                                       mk.randn(E, f, d, std=0.02), mk.randn(E, f, std=0.02), mk.randn(E, d, std=0.02))
    else:
        with torch.device("cuda"):
            st["gate"] = NaiveGate(d, E, 1, k)
        mk.fill(st["gate"].gate.weight)
        mk.gate_bias(st["gate"].gate, d, case["skew"])
        st["gate"].requires_grad_(False)
        st["assign"] = AsyncExpertAssignment(0, 1, 0, E, T)
        st["x"] = mk.randn(T, d, dtype=torch.float32)
    return st


def run(state):
    kind = state["kind"]
    if kind in ("layer", "staged"):
        return state["mlp"](state["x"])
    if kind == "train":
        mlp, x = state["mlp"], state["x"]
        mlp.zero_grad(set_to_none=True)
        x.grad = None
        out = mlp(x)
        out.backward(state["grad"])
        grads = {n: p.grad for n, p in mlp.named_parameters()}
        return {"out": out.detach(), "x": x.grad, **grads}
    if kind == "segments":
        return ops.moe_ffn_segments(*state["args"])
    if kind == "blocks":
        return state["moe"].forward(*state["args"])
    pos, score, infos = state["assign"].process_data(state["gate"], state["x"], state["E"], 1)
    return {"pos": pos, "score": score, "counts": infos["counts"], "offsets": infos["offsets"],
            "inv_pos": infos["inv_pos"]}


# ------------------------------------------------------------ work, error
def work(case):
    """Inputs and touched weights read once, outputs written once; the products of the routed rows."""
    T, d, f, E, k = (case[n] for n in ("tokens", "d", "f", "experts", "top_k"))
    kind = case["kind"]
    share = _zipf(E, case["skew"])
    rows = T * k
    if case["capacity"]:
        cap = math.ceil(case["capacity"] * rows / E)
        rows = sum(min(rows * s, cap) for s in share)
    gate_flops = 2.0 * T * d * E
    if kind == "gate":
        n = T * k
        return {"bytes": 4.0 * (T * d + E * d) + n * (8 + 4 + 4) + 8.0 * E, "flops": gate_flops}
    touched = sum(1.0 - (1.0 - min(k * s, 1.0)) ** T for s in share)        # experts that get a row
    weights = 2.0 * touched * (2 * d * f + d + f)
    flops = 4.0 * rows * d * f
    if kind == "train":
        grads = 2.0 * (E + _POPULAR) * (2 * d * f + d + f) + 2.0 * (E * d + E)
        return {"bytes": 4 * 2.0 * T * d + 2.0 * E * d + weights + grads, "flops": 3.0 * (flops + gate_flops)}
    rows_out = rows if kind == "blocks" else T
    nbytes = 2.0 * (T * d + rows_out * d) + weights
    if kind in ("layer", "staged"):
        return {"bytes": nbytes + 2.0 * E * d, "flops": flops + gate_flops}
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """fp16 results of fp32 sums, with the activation rounded to fp16 between the two products.  Against the same
    path in float64 with the same choice of experts, over 1 to 8192 tokens and widths of 256 to 4096, outputs are
    off by 2.9e-4 .. 4.5e-4, gradients, which pass through up to four roundings, by 2.0e-4 .. 5.8e-4, and the fp32
    router's scores by 1.6e-7 (its whole numbers follow from sums in a fixed order and are exact)."""
    if case["kind"] == "gate":
        return {"rel": 1e-6}
    return {"rel": 2.5e-3 if case["kind"] == "train" else 2e-3}
