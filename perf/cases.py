"""The work that users of this package have it do, as cases that can be timed.

A case is a dict of plain values:
    op        "forward"  attention without gradients (prefill, scoring, decode: the query length says which)
              "train"    forward, then the gradients of q, k and v for a given gradient of the output
    entry     "flax"     flax_attention on [B, H, L, D] tensors with a BlockMask
              "pallas"   flax_attention_pallas on [B, L, H, D] tensors (bhln=False, what a model's projections give)
    dtype     "f16" | "bf16" | "f32", always in the entry point's default numerics
    B, Hq, Hkv, Lq, Lkv, D
    score     "none" | "alibi" | "checkerboard" | "softcap" | "bias" (a plain function that adds a learned
              relative-position table)
    mask      "none" | "causal" (aligned to the last key) | "window" (causal sliding window and four sink keys)
              | "documents" (a plain function: causal inside packed documents, other documents for every sequence)
    window, docs      parameters of the last two, 0 elsewhere
    fresh     True: the block mask is made anew in every call, as where each batch or chunk brings another mask
What changes with every batch or optimizer step is read from its source in every call: the document ids from the tokens,
the float32 bias table from the half-precision weight.
"""
import math
import random

import torch

import flaxattention_amd as fa
from flaxattention_amd.masks import causal_mask, generate_attention_sink, offset_causal_mask
from flaxattention_amd.mods import generate_alibi_bias, generate_checkerboard, generate_tanh_softcap

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
SINK = 3          # generate_attention_sink keeps keys 0 .. SINK: four of them
BIAS_SPAN = 128   # the learned table covers distances -BIAS_SPAN .. BIAS_SPAN
END = 0           # the token that ends a document


def _case(name, op, dtype, B, Hq, Hkv, Lq, Lkv, D, score="none", mask="none", entry="flax", window=0, docs=0, fresh=False):
    return dict(name=name, op=op, entry=entry, dtype=dtype, B=B, Hq=Hq, Hkv=Hkv, Lq=Lq, Lkv=Lkv, D=D, score=score, mask=mask,
                window=window, docs=docs, fresh=fresh)


def listed():
    return [
        # the smallest call: one short sequence in float32, a forward of a few microseconds (latency and launches)
        _case("forward_small_f32", "forward", "f32", 1, 4, 4, 256, 256, 64, mask="causal"),
        # a training step on short sequences: fine-tuning batches, the sizes of the tests
        _case("train_short_bf16", "train", "bf16", 2, 8, 8, 512, 512, 64, mask="causal"),
        # the headline of the benchmark: half precision, a multiplicative score_mod, nothing masked
        _case("train_dense_f16", "train", "f16", 8, 8, 8, 2048, 2048, 64, score="checkerboard"),
        # the benchmark's bfloat16 training step: ALiBi under a causal block mask
        _case("train_alibi_bf16", "train", "bf16", 8, 8, 8, 2048, 2048, 64, score="alibi", mask="causal"),
        # a decoder block of current size: grouped heads, 128 wide, one long sequence in the layout of its projections
        _case("train_grouped_bf16", "train", "bf16", 1, 32, 8, 4096, 4096, 128, mask="causal", entry="pallas"),
        # packed documents, a ragged length, another mask with every batch
        _case("train_documents_bf16", "train", "bf16", 2, 8, 8, 3000, 3000, 64, mask="documents", docs=9, fresh=True),
        # a learned relative-position bias, written as a plain function, in an encoder that reads short sequences
        _case("train_bias_f16", "train", "f16", 8, 12, 12, 384, 384, 64, score="bias"),
        # wide heads
        _case("train_wide_f16", "train", "f16", 2, 8, 8, 2048, 2048, 256, mask="causal"),
        # long-context prefill: sliding window, sink keys and a soft-capped score (the benchmark's sparse forward)
        _case("forward_window_bf16", "forward", "bf16", 4, 16, 16, 8192, 8192, 128, score="softcap", mask="window", window=1024),
        # one chunk of a long prompt against the cache of the earlier ones; its mask is new with every chunk
        _case("forward_chunk_bf16", "forward", "bf16", 1, 32, 8, 512, 16384, 128, mask="causal", fresh=True),
        # decode with a full cache (the benchmark's): one query row per head, ALiBi
        _case("decode_f16", "forward", "f16", 8, 8, 8, 1, 16384, 64, score="alibi", mask="causal"),
        # decode of a batch with grouped heads and a cache of odd length
        _case("decode_grouped_bf16", "forward", "bf16", 16, 32, 8, 1, 6001, 128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


MOST_FLOPS = 4.5e11     # of a drawn case in 16 bits: below the largest listed one
MOST_FLOPS_F32 = 4e10   # float32 runs at a sixteenth of the rate
MOST_BYTES = 1 << 30
MOST_GRID = 1 << 25     # positions at which a mask or a bias written as a plain function is evaluated


def draw(rng):
    kind = rng.choice(["train", "train", "train", "forward", "forward", "chunk", "decode", "decode"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "f32"])
    D = rng.choice([64, 64, 128, 128, 96, 256]) if dtype != "f32" else rng.choice([64, 128])
    Hkv, G = rng.choice([2, 4, 8, 12, 16]), rng.choice([1, 1, 2, 4])
    score = rng.choice(["none", "none", "alibi", "checkerboard", "softcap"])
    mask, entry, window, docs, fresh = "none", "flax", 0, 0, False
    if kind in ("train", "forward"):
        B, L = _log(rng, 1, 16), _log(rng, 128, 8192)
        Lq = Lkv = L if rng.random() < 0.5 else max(128, L // 128 * 128)
        mask = rng.choice(["causal", "causal", "causal", "none", "window", "documents"])
        if mask == "window":
            window = _log(rng, 64, 1024)
        if mask == "documents":
            docs, fresh = rng.randint(2, 12), True
        elif rng.random() < 0.3:
            entry = "pallas"
        elif score == "none" and G == 1 and L <= 1024 and rng.random() < 0.5:
            score = "bias"
    elif kind == "chunk":
        B, Lkv = _log(rng, 1, 4), _log(rng, 2048, 32768)
        Lq, mask, fresh = min(_log(rng, 96, 1024), Lkv), "causal", True
    else:
        B, Lkv = _log(rng, 1, 32), _log(rng, 512, 32768)
        Lq, mask = rng.choice([1, 1, 1, 2, 4, 8]), rng.choice(["none", "causal"])
        dtype = rng.choice(["bf16", "f16"])
    case = _case("", "train" if kind == "train" else "forward", dtype, B, Hkv * G, Hkv, Lq, Lkv, D, score, mask, entry, window,
                 docs, fresh)
    del case["name"]
    while case["B"] > 1 and _too_much(case):
        case["B"] = max(1, case["B"] // 2)
    while case["Hkv"] > 1 and _too_much(case):
        case["Hkv"] //= 2
        case["Hq"] = case["Hkv"] * G
    while _too_much(case):
        case["Lq"], case["Lkv"] = max(1, case["Lq"] // 2), max(128, case["Lkv"] // 2)
    return case


def _too_much(case):
    w = work(case)
    grid = case["Lq"] * case["Lkv"] * (case["B"] if case["mask"] == "documents" else case["Hq"] if case["score"] == "bias" else 0)
    return grid > MOST_GRID or w["flops"] > (MOST_FLOPS_F32 if case["dtype"] == "f32" else MOST_FLOPS) or w["bytes"] > MOST_BYTES


def _document_lengths(case):
    """Lengths that differ by up to a factor of ten or so and fill the sequence."""
    rng = random.Random(1000 * case["docs"] + case["Lq"])
    cuts = sorted(rng.sample(range(1, case["Lq"]), case["docs"] - 1)) if case["docs"] > 1 else []
    return [b - a for a, b in zip([0] + cuts, cuts + [case["Lq"]])]


def _mask_mod(case, tokens):
    if case["mask"] == "causal":
        offset = case["Lkv"] - case["Lq"]
        return offset_causal_mask(offset) if offset else causal_mask
    if case["mask"] == "window":
        return generate_attention_sink(case["window"], SINK)
    if case["mask"] == "documents":
        ends = tokens == END
        doc_ids = ends.cumsum(1) - ends.to(torch.int64)   # a document's last token belongs to it

        def packed(b, h, q_idx, kv_idx):
            return (doc_ids[b, q_idx] == doc_ids[b, kv_idx]) & (q_idx >= kv_idx)
        return packed
    return None


def _score_mod(case, weight):
    if case["score"] == "alibi":
        return generate_alibi_bias(case["Hq"], -1.0)
    if case["score"] == "checkerboard":
        return generate_checkerboard(0.5, 2.0)
    if case["score"] == "softcap":
        return generate_tanh_softcap(50.0)
    if case["score"] == "bias":
        table = weight.to(torch.float32)

        def relative(score, b, h, q_idx, kv_idx):
            return score + table[h, (kv_idx - q_idx).clamp(-BIAS_SPAN, BIAS_SPAN) + BIAS_SPAN]
        return relative
    return None


def _block_mask(case, mask_mod):
    per_sequence = case["B"] if case["mask"] == "documents" else None
    return fa.create_block_mask(mask_mod, per_sequence, None, case["Lq"], case["Lkv"])


def prepare(case, seed):
    dev, dtype = torch.device("cuda", torch.cuda.current_device()), DTYPES[case["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(seed)
    B, Hq, Hkv, Lq, Lkv, D = (case[n] for n in ("B", "Hq", "Hkv", "Lq", "Lkv", "D"))

    def normal(H, L):
        shape = (B, L, H, D) if case["entry"] == "pallas" else (B, H, L, D)
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32).to(dtype)
    state = {"case": case, "q": normal(Hq, Lq), "k": normal(Hkv, Lkv), "v": normal(Hkv, Lkv)}
    if case["op"] == "train":
        state["d_out"] = normal(Hq, Lq)
        for n in ("q", "k", "v"):
            state[n].requires_grad_(True)
    if case["mask"] == "documents":
        rng, rows = random.Random(seed), []
        for _ in range(B):   # every sequence packs documents of the same lengths, in an order of its own
            lengths = _document_lengths(case)
            rng.shuffle(lengths)
            rows.append([t for n in lengths for t in [1] * (n - 1) + [END]])
        state["tokens"] = torch.tensor(rows, dtype=torch.int32, device=dev)
    elif not case["fresh"]:
        state["mask_mod"] = _mask_mod(case, None)
        if case["entry"] == "flax" and state["mask_mod"] is not None:
            state["block_mask"] = _block_mask(case, state["mask_mod"])
    if case["score"] == "bias":
        state["weight"] = (0.5 * torch.randn((Hq, 2 * BIAS_SPAN + 1), generator=gen, device=dev)).to(dtype)
    else:
        state["score_mod"] = _score_mod(case, None)
    return state


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    gqa = case["Hq"] != case["Hkv"]
    score_mod = _score_mod(case, state["weight"]) if case["score"] == "bias" else state["score_mod"]
    if case["entry"] == "pallas":
        out = fa.flax_attention_pallas(q, k, v, score_mod=score_mod, mask_mod=state["mask_mod"], bhln=False,
                                       enable_gqa=gqa)
    else:
        block_mask = _block_mask(case, _mask_mod(case, state.get("tokens"))) if case["fresh"] else state.get("block_mask")
        out = fa.flax_attention(q, k, v, score_mod=score_mod, block_mask=block_mask, enable_gqa=gqa)
    if case["op"] == "forward":
        return out
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["d_out"])
    return out.detach(), dq, dk, dv


def _visible(case):
    """Visible (query, key) pairs of one head of one sequence, and the keys that some row sees."""
    Lq, Lkv = case["Lq"], case["Lkv"]
    if case["mask"] == "causal":
        first = Lkv - Lq + 1   # keys the first row sees
        return Lq * (first + Lkv) // 2, Lkv
    if case["mask"] == "window":
        pairs = 0
        for i in range(Lq):
            near = min(i + 1, case["window"] + 1)
            pairs += near + min(SINK + 1, i + 1 - near)
        return pairs, Lkv
    if case["mask"] == "documents":
        return sum(n * (n + 1) // 2 for n in _document_lengths(case)), Lkv
    return Lq * Lkv, Lkv


def work(case):
    pairs, keys = _visible(case)
    size = 4 if case["dtype"] == "f32" else 2
    rows_q, rows_kv = case["B"] * case["Hq"] * case["Lq"], case["B"] * case["Hkv"] * keys
    nbytes = (2 * rows_q + 2 * rows_kv) * case["D"] * size           # q, k, v and the output
    flops = 4 * case["D"] * pairs * case["B"] * case["Hq"]           # two products
    if case["op"] == "train":
        nbytes *= 2                                                  # and their gradients
        flops = flops * 7 // 2                                       # and five products more
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Of outputs and gradients, about four times what was measured against the same formulas in 64 bits (f32 up to 2.6e-6,
    # f16 3e-4 .. 1.2e-3, bf16 2.9e-3 .. 4.7e-3; a checkerboard doubles the scores and their rounding): scores,
    # probabilities and results are rounded to the input type.
    return {"rel": {"f32": 1e-5, "f16": 4e-3, "bf16": 1.5e-2}[case["dtype"]]}
