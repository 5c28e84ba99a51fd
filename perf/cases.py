"""The work that perf measurements of this framework time: GGUF linear layers of a 27B decoder
(hidden 5120, 17408 in the FFN), built and called through GGUFLinearMethod as a vLLM model does.

A case is one projection ("part" q / qkv / o / gate_up / down / head) or the four of a whole decoder
layer ("layer"), in one of three mixes of weight types:
  iq3   IQ3_S everywhere, IQ4_XS for down (the layer sweep of bench.py)
  k     a K-quant file: Q4_K, with Q6_K for v and down
  rco   a low-bit file: Q2_K q beside IQ3_S k and v, IQ3_XXS o, IQ2_S gate beside IQ2_XXS up,
        IQ2_XS down (the types that the golden rows of tests/golden/dequant name for them)
and a number of activation rows m: 1..8 when tokens are decoded, 9..48 when drafts of several
sequences are verified, more when a prompt is read. "graph" says that the passes are replays of a
captured graph, as a server decodes; prompts run eagerly. Weights are random codes with scales
that give values of about 0.02; activations are N(0, 1) with a few channels of 20 times that.
"""

import base64
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "vllm-gsqrco-exl3_amd"))

from vllm_gguf_plugin.quantization.linear import GGUFLinearMethod  # noqa: E402

# ggml type ids and bytes per block of 256 values
TYPES = {"Q2_K": (10, 84), "Q4_K": (12, 144), "Q6_K": (14, 210), "IQ2_XXS": (16, 66), "IQ2_XS": (17, 74),
         "IQ3_XXS": (18, 98), "IQ3_S": (21, 110), "IQ2_S": (22, 82), "IQ4_XS": (23, 136)}
# byte offsets of the fp16 block scales, each with the scale of weights of about 0.02
SCALES = {"Q2_K": ((80, 1.4e-3), (82, 1.9e-3)), "Q4_K": ((0, 1.3e-4), (2, 9e-4)), "Q6_K": ((208, 1.5e-5),),
          "IQ2_XXS": ((0, 3.6e-4),), "IQ2_XS": ((0, 3.6e-4),), "IQ3_XXS": ((0, 1.5e-4),), "IQ3_S": ((0, 1.4e-4),),
          "IQ2_S": ((0, 3.6e-4),), "IQ4_XS": ((0, 1.6e-5),)}
MIXES = {
    "iq3": {"q": "IQ3_S", "k": "IQ3_S", "v": "IQ3_S", "o": "IQ3_S", "gate": "IQ3_S", "up": "IQ3_S", "down": "IQ4_XS",
            "head": "Q6_K"},
    "k": {"q": "Q4_K", "k": "Q4_K", "v": "Q6_K", "o": "Q4_K", "gate": "Q4_K", "up": "Q4_K", "down": "Q6_K",
          "head": "Q6_K"},
    "rco": {"q": "Q2_K", "k": "IQ3_S", "v": "IQ3_S", "o": "IQ3_XXS", "gate": "IQ2_S", "up": "IQ2_XXS",
            "down": "IQ2_XS", "head": "Q4_K"},
}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(part, mix, m, dtype="bf16", graph=False, hidden=5120, ffn=17408, q=6144, kv=1024, vocab=151936):
    return {"part": part, "mix": mix, "m": m, "dtype": dtype, "graph": graph, "hidden": hidden, "ffn": ffn, "q": q,
            "kv": kv, "vocab": vocab}


def listed():
    return [
        # the smallest call: one token through one 4096 x 4096 Q4_K projection in fp32 (the CPU
        # baseline's size in bench.py), called eagerly: launches and the host's share
        dict(_case("q", "k", 1, "fp32", hidden=4096, q=4096), name="q4096-m1"),
        # one token through a decoder layer, as a server decodes one sequence
        dict(_case("layer", "iq3", 1, graph=True), name="layer-iq3-m1"),
        # four rows: one sequence with three drafted tokens, on the low-bit file
        dict(_case("layer", "rco", 4, graph=True, q=12288), name="layer-rco-m4"),
        # logits of four rows: the largest weight of the model
        dict(_case("head", "iq3", 4, graph=True), name="head-m4"),
        # four sequences' drafts verified together
        dict(_case("layer", "iq3", 16, graph=True), name="layer-iq3-m16"),
        # a ragged verify batch, fp16 activations, K-quants
        dict(_case("layer", "k", 37, "fp16", graph=True), name="layer-k-m37"),
        # the same on the low-bit file
        dict(_case("layer", "rco", 24, graph=True, q=12288), name="layer-rco-m24"),
        # a short prompt
        dict(_case("layer", "iq3", 100), name="layer-iq3-m100"),
        # a prompt of ordinary length, and the usual chunk of a longer one, on each file
        dict(_case("layer", "k", 509, "fp16"), name="layer-k-m509"),
        dict(_case("layer", "iq3", 512), name="layer-iq3-m512"),
        dict(_case("layer", "rco", 1024, q=12288), name="layer-rco-m1024"),
        # the largest: a 2048-token chunk, a prompt-reading server's full batch
        dict(_case("layer", "iq3", 2048), name="layer-iq3-m2048"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    mix = rng.choice(["iq3", "k", "rco"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    hidden = 512 * rng.randint(5, 10)
    ffn = 512 * rng.randint(11, 34)
    q = 128 * rng.randint(16, 48)  # o reads q columns: whole 512s
    kv = 128 * rng.randint(1, 8)
    kind = rng.random()
    if kind < 0.1:  # logits of a few rows, over vocabularies that are no multiple of anything
        return _case("head", mix, rng.randint(1, 8), dtype, True, hidden, ffn, vocab=rng.randint(32000, 151936))
    part = rng.choice(["layer", "layer", "qkv", "o", "gate_up", "down"])
    # a low-bit layer costs about twice the others' time at a given m
    m = (rng.randint(1, 8) if kind < 0.35 else rng.randint(9, 48) if kind < 0.6
         else _log(rng, 49, 1024 if mix == "rco" else 2048))
    return _case(part, mix, m, dtype, m <= 48, hidden, ffn, q - q % 512 if part in ("layer", "o") else q, kv)


# ------------------------------------------------------------------------------ shapes
def _projections(case):
    """[(shards [(weight type, rows)], shard ids, k)] of the case's products."""
    t = MIXES[case["mix"]]
    h, f, q, kv = case["hidden"], case["ffn"], case["q"], case["kv"]
    # o reads the attention's output: q's columns, or half of them where q carries a gate (12288)
    attn = q // 2 if q > 6144 else q
    every = {
        "q": ([(t["q"], q)], [None], h),
        "qkv": ([(t["q"], q), (t["k"], kv), (t["v"], kv)], ["q", "k", "v"], h),
        "o": ([(t["o"], h)], [None], attn),
        "gate_up": ([(t["gate"], f), (t["up"], f)], [0, 1], h),
        "down": ([(t["down"], h)], [None], f),
        "head": ([(t["head"], case["vocab"])], [None], h),
    }
    return [every[p] for p in (("qkv", "o", "gate_up", "down") if case["part"] == "layer" else (case["part"],))]


def _raw(gen, name, rows, k):
    """Random GGUF blocks of one tensor, uint8 [rows, row bytes]."""
    w = torch.randint(0, 256, (rows, k // 256, TYPES[name][1]), dtype=torch.uint8, device="cuda", generator=gen)
    for at, s in SCALES[name]:
        d = (s * (0.5 + torch.rand(rows, k // 256, device="cuda", generator=gen))).half()
        w[:, :, at:at + 2] = d.view(torch.uint8).view(rows, k // 256, 2)
    return w.view(rows, -1)


def _x(gen, case, k):
    x = torch.randn(case["m"], k, device="cuda", generator=gen)
    x[:, torch.randperm(k, device="cuda", generator=gen)[:k // 256]] *= 20
    return x.to(DTYPES[case["dtype"]])


def _inputs(case, seed):
    """[(raw tensors, x)] of the case's products: one seed, one set."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    for shards, ids, k in _projections(case):
        yield [(name, _raw(gen, name, rows, k)) for name, rows in shards], ids, _x(gen, case, k)


# ------------------------------------------------------------------------------ the measured pass
def prepare(case, seed):
    layers = []
    for shards, ids, x in _inputs(case, seed):
        layer, method = torch.nn.Module(), GGUFLinearMethod()
        sizes = [raw.shape[0] for _, raw in shards]
        with torch.device("cuda"):
            method.create_weights(layer, x.shape[1], sizes, x.shape[1], sum(sizes), x.dtype)
        for (name, raw), sid in zip(shards, ids):
            layer.weight.weight_loader(layer.weight, raw, sid)
            layer.weight_type.weight_loader(layer.weight_type, torch.tensor(TYPES[name][0]), sid)
        method.process_weights_after_loading(layer)
        layers.append((method, layer, x))
    state = {"layers": layers, "graph": None}
    if case["graph"]:
        _apply(state)  # before the capture, as servers warm up
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = _apply(state)
    return state


def _apply(state):
    return [method.apply(layer, x) for method, layer, x in state["layers"]]


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return _apply(state)


def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    nbytes = flops = 0
    for shards, _, k in _projections(case):
        rows = sum(r for _, r in shards)
        nbytes += sum(r * (k // 256) * TYPES[t][1] for t, r in shards) + case["m"] * (k + rows) * es
        flops += 2 * case["m"] * rows * k
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Sums in another order move fp32 results by 4e-7 of their norm, fp16 ones by 2e-5 and bf16 ones by
    # 4e-5 (a last bit that falls the other way here and there). The k and rco mixes hold formats of
    # which an implementation may keep a product in fp32 or round it to fp16 (Q6_K's sub-scale times
    # quant, Q2_K's block scale times sub-scale, 2^-12): 1.4e-4, 2.6e-4 and 7e-4.
    tight = case["mix"] == "iq3" and case["part"] != "head"
    rel = {"fp32": 2e-6, "fp16": 1e-4, "bf16": 2e-4} if tight else {"fp32": 6e-4, "fp16": 1e-3, "bf16": 3e-3}
    return {"rel": rel[case["dtype"]]}


# ------------------------------------------------------------------------------ 64-bit results
# The codebooks of the IQ types: the points of a small lattice that each uses, as a bitmap over the
# lattice codes (digits of the entry's bytes, byte 0 the least significant); members in ascending
# order of code are the table.
LATTICE = {"IQ2_XXS": (8, (8, 25, 43)), "IQ2_XS": (8, (8, 25, 43)), "IQ2_S": (8, (8, 25, 43)),
           "IQ3_XXS": (4, (4, 12, 20, 28, 36, 44, 52, 62)), "IQ3_S": (4, (1, 3, 5, 7, 9, 11, 13, 15))}
MEMBERS = {
    "IQ2_XXS": (
        "VRUUVRBEQUEABBREABAAAAAEQAAUAEAAAAAABAAAUBBAQREAARQEQFAEQAAQAAAFEAAAUAAAAQAAQAAAQRQEQBQUAAAEAAAEAAAEAAAAAAAA"
        "BBAAAAAAAAAAABQEEBAAQAAEEQAEARAAQEAAAQAAAAAAAQQAAAAAABAEQARAAAAEAAAAABAAAAAQAAAAQAAQAAAAAAAAAAAFAQAEAABAAAAA"
        "EQAAAAAAAAAAAQAAAABAAAAAAAAUBAAAAQABBQAAAAAAEBAAAAAAAFAAAAAAAAAAAABAQQAAAUAAAAAAQAAAAAQAQAAAAAAAAAAAAAAAQAAA"
        "QAAEAAAAAAAEAAAAAAAAAAAAAAAAAAAAAQAAAAAAUBBEQRAQARQEABAAQAAAAAREAABAQAAAQEAAAQAAQBAAAQAAABAAEAAABBAAAAAAAAAA"
        "AQAAAAAAAAAAABQEABABAAAAAAAEAAAAABABBAAAAAAAAAQAAAAEABBEUAAAAAAEAQAAAQAABAAAAAAAAQAAAAAAAABAAAAAAAAAAAAAQAEA"
        "AAEAAAAAAAAAAAQAAAAAAQAAAAAEEAQAAAAEAAAAAAAAQAAAAAAAAAAEAAAAAAAAAAAAQQAAAQAAAQAAQAAAAABAAAAAAAAAQAAAABAAAAAA"
        "EQAAAAAAAAAAAAAUAAAAAAAEAAAAAAAAAAAAAAAAAAAAAAEAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAQEEAAAQAAEAAAAAEQAAEAAAAAAAA"
        "AAQAAAAAAAAAABREABAAQAAAAAAEAAAABAAAABAAAAQAQAAAAQAAAEAAAAAAAAAAAAAAAQAAAAAAAAAAAAABAAAAAAAAAAAEARAEAAAAAAAB"
        "AEAAAAAAQAAAAAAAAAABAAAAAAAEAEAAAQAAAAAAAAAAAAABAAAAAAAAAAAAAAAAAAAAAAAAAAAAEAAAAAAAAQAAAAAAAAAAAAAAAAAAAAAA"
        "BAAAABAAAAQAAAABAAAAAAAAAAAEAAAAAAAAAAAAAAAEAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAEAAAAAAAEAAAAAAAAAAAA"
        "AAAAAAAAAAAAAAA="),
    "IQ2_XS": (
        "VVVVUVVFQRVFAVRVVVBFQRAFAQBUURBAQQQAAQEAUFVFQRUVARQEAFBFQQAFAQQEAABAQQAQBQAAQAAAQFUFERQEARAAQEAFAQAEAABAEAAA"
        "AQAEAQAAAAAQAVRVUVBFQUAFAQBUURBAQQAAAVAAUBEAQAAAAQAAAFBFQQBFARAEAABAQQAAAQAAAAAAQAAEAAABAAAAAAAFBQAEQAAABAAA"
        "EQAAAAAABAAAAAAAAABAAAAAAABVVRBAQQAAAQAEUBAAQBAAEAAAABAAAAEAAAAEAABEQQBAAQAAAAAAQAAAAAQQAAAAEAABAAEAAAAAAAAQ"
        "QQEEAAABABAABAAAAAAAABAAAQAAARAAAAAARAEAUFVFQVUFERQEAFBFQQAFAQBEAEBAQQFAAQAAAAAAQBVFARQEABAAAQAFARAEAAAAAEAA"
        "AQEAQBAAAAAAABQEABABAQEAAAAEEAAAQQBAAAAAQAAAAAAAAAAAAFBFQRAFAQAEAABAQQQABQAAAAAAQAAAABAAAAAAAEAFAQQEABBAAAAB"
        "QQAAAAAAQBAAAAAAEAAAABAAAAQEQABAQAAAAAABAAAQQAEAAAAAAAAAAAAAAABAAABAQQAAARAQAAEAUAAAAAAAAAAAAAAAABAABAAAAAEA"
        "AUAAAAAAAAAAAAAEABABAAAAABAAAAAAAAAAAAAAEAAAAAAAAAEAAAAAAAQAAAAAAAAABAAAABAQAAAAQBUFARUEAFAAAFAVAQAEEAQAAAAA"
        "AQAEAAAAQAEAQRRUABAAQABAAAAEAAAAAQAAAABAAAAEAAAAAAEAABAEAAQAAAEUAAAEBAAAAAAAAAAAAAAABAAAABAEBBAFAQAEAAEAAQAA"
        "AQAQAAAAAQAAAAAAAAAABABAAABEAAAAQRAAAAAAAAAAEAAAAAAUAAAAAAABAAAAAAAAAAAAAAQAAAAABAAAAAABAAAAAAAAEAAAABAAAAAA"
        "RQEEBAAAAAAAAQAAAABAEAAAAEAUAQAQAAAAAQAEAAAAQAAAAABAAAAAAAAAAAAAAAAAAAAAAABAAAAEAEAARQAAAAAAQBAEAAAAAAAABQAA"
        "AAAABQAAAAABAAE="),
    "IQ2_S": (
        "VVVVUVVFVRUFEVVVUVBFVRQFFRRUURBQVQQAEREQUFVFVVVVFVRFUVBVVRRVVRRUURBAVQQAURQEUBAAQBVVEVVVURABAUAFVQREURBAQAAA"
        "ARQQBRAAAABAAFRVUVFFVRUVURRUVVVFVRUFVRQAUBRBQQQFABQEAFBFVRRVVRRUURBAVRUFVRQEUBAAQBQFARQEABAAAEBVUQRUURBAAQAA"
        "VRQEUBAAEAAABBAEABAABAAAAABUURVRQQUEAREAVFBBQAUFARQEABAQAFEEAQAABQBEVRQFVRQEUBAAQBQFARQEABEAAAAFAQAEAAQAAAAA"
        "ERQAUBAAAEAAABUEAAAAAAAAEAAABEAAAAAEQAEAUFVVRVVVFRREUVBFVQVVVRRUURBAQRUEURQEUAAAQFVVVVRVUVBFQQBVVRRUURBQQQAA"
        "VRQEUBAAQAAAEBRVUVBFQQAEAQBUURBAQQAAAUAAUBAAQAAAAAAAAFBFVRVVVRRUUQBAVRUFVRQEUBAAQBQFARQEABQAAABVVRRUURBAQQAA"
        "VRQEUBAAQAAAABQEABEAAAAAAABUURBAQUAAAQAAUBAAQAAAAAAAABAAEAAAAABAAABERRUFURQEQBAAQBUFARQEABAAEAAEAQAEAAEAAAAB"
        "URQEUBAAQAAAABQEABAQABAABAAEAAAAAAAAABAAUBAAAAAAEAAAARAAAEAAAAAAAAAAAAAABAAAAABAQBVFERRUERBBAQBFVRRUUQBAQQBA"
        "ERUAUBAAAAAAAFRVEVBFQQAFAQBUURBAQQAAAQEAUBAAUAAAAAAAABBBAQAFAQAAAEBAAQAAAQBAAAAAAAAABAAABUAAAAFFVRBUURBAQQAA"
        "ERQAUBAQAAAAABQEABAAAAAAAEBUURBAQQAAAUAAUBAAQAAAAAAAERAAAAAQABAAAABAQQAQAQAAAAAAUAAAAAARAAAAAAAAAAAAAAAAQAAA"
        "EREQVBAAAAAABAEAABAAAAQAAAAQBEAUAAAARAEAURAAQAAAAAABQBAAEAAAAAAAAAAAAAAAAAQAAAAAAEAAQAAAAAAAAAEAAAAAQAAABAAA"
        "QAEUAQAAABAAAAE="),
    "IQ3_XXS": (
        "FYoFAgQAACgKBSIFAhAAARUCBYoAggAgggUgAAAAAAEACACAEIAAKIIAAAQABAAAAAAAIAAAEAAAUQAACAACAAoFChWAAQAABQIFAAAAAAAK"
        "BQIBAAAABAUAAQJAAEAAIgAAAAABAAAAABEAQAAAAiAAAAAAAAAAAAAEAAEAAAAFCkUCBAAAACoFAgEAAIgBBYIFgAEgAAACEQAAAAAAEQAA"
        "ACAACAAACACAAAIAABAAAAAAAAAAAApAAAAgAAAAAgUKAAABIAQFAAECUAAAAAoBIAAABAAEAAIACAAAAAAAAAABgAAABEEABAAAIAAAABAA"
        "QAAACAAAAAAIAAABABCAAKAAiAAAAAAAAAAAABAAAAGAAQBBAIAAAAAgAAAAEAAAAAACEAAAACAACAAAAQAAAAAAAAAAIAUAAQAAAAAABAAA"
        "AgAAAUEAQAAAIAAAABAABAAAAAQEAAAAAAgAAAABiAAAAAAEBAAAAgAAAAAAAAAAAAEAAAAAEAAEAAAAAAAQAFAAEAAAAAIAAAACAACAAAAA"
        "ABAAAAAAQQAAAAAAAAAAEAAAACAAAAAABAAAAAAACAAAAAAIAAIAAAAAAKgBAAQABAAAAABAAAEAAAAABAAAIAQAAAEgAAgAAAEAAAACAAIA"
        "AAAFABAAAAAAAAAAAAEAAAAAAAAAAAAAAAA="),
    "IQ3_S": (
        "p1cjCKUKBZIXI4kiEAAiBKNJIhGkCgAJCCIFShAFgCIBiBIECQIAARQARQiiAEAIQAoAAgAEAAIVAEUIABEAABerBVIAUAIESxECCQIFAEEB"
        "pBEECSABBJIJghECAAQBKBQACkQRAAACCQIFAAIAAAAAkQBQAAAACgUCIAIABAGrVYoFKgWAKQWJJBIEAgAAkgAKgQKIABIlAhQKBAFAAIIA"
        "CSQCAAAkEAIEgAEIAAGFAAIAACACACACQAEIAQAABKoEKpQCCAIqEAoAAQABRAEEARQAAQAAAhGKAYogAAgIQgQCAAQRAAIFIAQQQAAIAEAA"
        "AAIAAAAKAAUgAAAAABEEkQQCAQABhAoEIQgiAAAKIQIIAYAEARAKBSIAAAAABQAQgAEAAAKgAAIAAAAEAAAIABAAAAEAACEAAQgCAAAEEQQA"
        "kQRAECoEAgQAAAAEAQIIQQAIAACEAYAAEAIgCBIAAQRAAAAAAARAAAAKAAAAAAAABAAAABQABAAAAAAAACoACgAAAQABAIEAAAAQAAAEABAE"
        "IAQBARACAAEAAAAAACAACAAEAAkAABAAAAEAIAAAAAEAAAAACgAAAAAAAJEABUABEAQABAIQACgAAAASQQIBAAIAAAQAACQACAAAIggBAAAB"
        "AAAAAAQABAAAAAQAAAIAAAAAAQAAAAAAAAA="),
}
KVALUES = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _grid(name):
    n, levels = LATTICE[name]
    bits = np.unpackbits(np.frombuffer(base64.b64decode(MEMBERS[name]), np.uint8), bitorder="little")
    codes = np.flatnonzero(bits)
    digits = codes[:, None] // len(levels) ** np.arange(n) % len(levels)
    return torch.tensor(np.array(levels)[digits], dtype=torch.float64, device="cuda")


def _f16(b, at):
    return b[..., at:at + 2].contiguous().view(torch.float16).double()


def _signs(bits):
    """[..., n] sign bytes -> [..., n, 8]: bit j negates value j."""
    return 1.0 - 2.0 * ((bits.unsqueeze(-1) >> torch.arange(8, device="cuda")) & 1).double()


def _ksigns(i):
    """7 sign bits and an eighth that makes the parity even."""
    p = i ^ (i >> 4)
    p = p ^ (p >> 2)
    return i | (((p ^ (p >> 1)) & 1) << 7)


def _u32(b, at, n):
    v = b[..., at:at + 4 * n].reshape(*b.shape[:-1], n, 4).long()
    return v[..., 0] | v[..., 1] << 8 | v[..., 2] << 16 | v[..., 3] << 24


def _dequantise(name, raw):
    """GGUF rows -> float64 [rows, k]."""
    rows = raw.shape[0]
    b = raw.view(rows, -1, TYPES[name][1])
    nb = b.shape[1]
    u = b.int()  # the bytes as numbers
    nib = lambda v: torch.stack([v & 15, v >> 4], -1)  # noqa: E731
    g7 = 7 * torch.arange(4, device="cuda")
    if name == "Q4_K":
        s = u[..., 4:16]
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | (s[..., :4] >> 6) << 4], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | (s[..., 4:8] >> 6) << 4], -1)
        q = u[..., 16:].reshape(rows, nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 3).reshape(rows, nb, 8, 32)
        w = (_f16(b, 0) * sc).unsqueeze(-1) * q - (_f16(b, 2) * mn).unsqueeze(-1)
    elif name == "Q2_K":
        q = u[..., 16:80].reshape(rows, nb, 2, 1, 32)
        q = ((q >> (2 * torch.arange(4, device="cuda").view(4, 1))) & 3).reshape(rows, nb, 16, 16)
        s = u[..., :16]
        w = (_f16(b, 80) * (s & 15)).unsqueeze(-1) * q - (_f16(b, 82) * (s >> 4)).unsqueeze(-1)
    elif name == "Q6_K":
        lo = u[..., :128].reshape(rows, nb, 2, 2, 32)
        lo = torch.cat([lo & 15, lo >> 4], 3)
        hi = u[..., 128:192].reshape(rows, nb, 2, 1, 32) >> (2 * torch.arange(4, device="cuda").view(4, 1))
        q = ((lo | (hi & 3) << 4) - 32).reshape(rows, nb, 16, 16)
        w = (_f16(b, 208) * b[..., 192:208].contiguous().view(torch.int8)).unsqueeze(-1) * q
    elif name == "IQ4_XS":
        ls = nib(u[..., 4:8]).reshape(rows, nb, 8)
        ls = ls | (((u[..., 2:3] | u[..., 3:4] << 8) >> (2 * torch.arange(8, device="cuda"))) & 3) << 4
        q = u[..., 8:].reshape(rows, nb, 8, 1, 16)
        q = torch.tensor(KVALUES, dtype=torch.float64, device="cuda")[torch.cat([q & 15, q >> 4], 3).long()]
        w = (_f16(b, 0) * (ls - 32)).unsqueeze(-1) * q.reshape(rows, nb, 8, 32)
    elif name == "IQ3_S":
        qh = (u[..., 66:74].unsqueeze(-1) >> torch.arange(8, device="cuda")) & 1
        v = _grid(name)[(u[..., 2:66] | qh.reshape(rows, nb, 64) << 8).long()].reshape(rows, nb, 8, 32)
        sg = _signs(u[..., 74:106]).reshape(rows, nb, 8, 32)
        w = (_f16(b, 0) * (1 + 2 * nib(u[..., 106:110]).reshape(rows, nb, 8))).unsqueeze(-1) * v * sg
    elif name == "IQ3_XXS":
        aux = _u32(b, 66, 8)
        v = _grid(name)[u[..., 2:66].long()].reshape(rows, nb, 8, 32)
        sg = _signs(_ksigns((aux.unsqueeze(-1) >> g7) & 127)).reshape(rows, nb, 8, 32)
        w = (_f16(b, 0) * (2 * (aux >> 28) + 1) / 4).unsqueeze(-1) * v * sg
    elif name == "IQ2_XXS":
        v = _grid(name)[u[..., 2:66].reshape(rows, nb, 8, 8)[..., :4].long()].reshape(rows, nb, 8, 32)
        aux = _u32(b, 2, 16)[..., 1::2]
        sg = _signs(_ksigns((aux.unsqueeze(-1) >> g7) & 127)).reshape(rows, nb, 8, 32)
        w = (_f16(b, 0) * (2 * (aux >> 28) + 1) / 8).unsqueeze(-1) * v * sg
    else:
        if name == "IQ2_XS":
            i = u[..., 2:66:2] | u[..., 3:66:2] << 8
            v, sg, at = _grid(name)[(i & 511).long()], _signs(_ksigns(i >> 9)), 66
        else:  # IQ2_S
            qh = (u[..., 66:74].unsqueeze(-1) >> (2 * torch.arange(4, device="cuda"))) & 3
            v, sg, at = _grid(name)[(u[..., 2:34] | qh.reshape(rows, nb, 32) << 8).long()], _signs(u[..., 34:66]), 74
        ls = 2 * nib(u[..., at:at + 8]).reshape(rows, nb, 16) + 1
        w = (_f16(b, 0) * ls / 8).unsqueeze(-1) * (v * sg).reshape(rows, nb, 16, 16)
    return w.reshape(rows, -1)


def exact(case, seed):
    """The products of the dequantised weights with the activations as they were given, in float64 (4096
    weight rows at a time, so that the expanded codes fit beside the weights)."""
    out = []
    for shards, _, x in _inputs(case, seed):
        xd = x.double()
        out.append(torch.cat([xd @ _dequantise(name, raw[i:i + 4096]).T
                              for name, raw in shards for i in range(0, raw.shape[0], 4096)], 1))
    return out
