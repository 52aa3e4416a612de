"""HIP block-mask builder vs the CPU oracle: bit-exact integer outputs."""
import numpy as np
import pytest
import torch

import flaxattention_amd as fa
from flaxattention_amd.masks import causal_mask, generate_attention_sink, generate_sliding_window, offset_causal_mask
from flaxattention_amd.core.common import MaskMod, INT_MAX, INT_MIN
from oracle import (o_attention_sink, o_causal_mask, o_full_masked, o_noop_mask, o_offset_causal, o_sink_window_lt,
                    o_sliding_window, ref_create_block_mask)

pytestmark = pytest.mark.gpu

FIELDS = ["kv_num_blocks", "kv_indices", "full_kv_num_blocks", "full_kv_indices",
          "q_num_blocks", "q_indices", "full_q_num_blocks", "full_q_indices"]


def check(bm, ref):
    for f in FIELDS:
        got = getattr(bm, f).cpu().numpy()
        assert got.dtype == np.int32
        assert got.shape == ref[f].shape, (f, got.shape, ref[f].shape)
        assert np.array_equal(got, ref[f]), f
    assert bm.BLOCK_SIZE == ref["BLOCK_SIZE"]
    assert bm.used_block_size == ref["used_block_size"]


def sink_lt(window, sink):
    # benchmark-config spelling: kv_idx < sink always visible
    return generate_attention_sink(window, sink - 1)


CASES = [
    ("causal_c1", causal_mask, o_causal_mask, 1, 4, 256, 256, 128),
    ("causal_c3", causal_mask, o_causal_mask, 2, 3, 2048, 2048, 128),
    ("causal_bs64", causal_mask, o_causal_mask, 1, 2, 512, 512, 64),
    ("causal_ragged", causal_mask, o_causal_mask, 1, 1, 300, 500, 128),
    ("causal_rect_blocks", causal_mask, o_causal_mask, 1, 2, 384, 512, (128, 64)),
    ("window", generate_sliding_window(10), o_sliding_window(10), 1, 1, 1024, 1024, 128),
    ("sink_ref", generate_attention_sink(300, 4), o_attention_sink(300, 4), 1, 2, 2048, 2048, 128),
    ("sink_c4", sink_lt(1024, 4), o_sink_window_lt(1024, 4), 1, 1, 8192, 8192, 128),
    ("noop", fa.noop_mask, o_noop_mask, 1, 1, 256, 384, 128),
    ("short_q", causal_mask, o_causal_mask, 4, 8, 64, 64, 128),
    ("decode_q1", offset_causal_mask(16383), o_offset_causal(16383), 1, 1, 1, 16384, 128),
    ("decode_q16", offset_causal_mask(16384 - 16), o_offset_causal(16384 - 16), 1, 1, 16, 16384, 128),
    ("decode_q64", offset_causal_mask(16384 - 64), o_offset_causal(16384 - 64), 2, 2, 64, 16384, 128),
]


@pytest.mark.parametrize("name,mask,omask,B,H,Q,KV,bs", CASES, ids=[c[0] for c in CASES])
def test_builder_matches_oracle(name, mask, omask, B, H, Q, KV, bs, dev):
    print(f"case {name} B{B} H{H} Q{Q} KV{KV} bs{bs}", flush=True)
    bm = fa.create_block_mask(mask, B, H, Q, KV, BLOCK_SIZE=bs, device=dev)
    ref = ref_create_block_mask(omask, B, H, Q, KV, BLOCK_SIZE=bs)
    check(bm, ref)


def test_fully_masked(dev):
    def fullmask(b, h, q_idx, kv_idx):
        return False
    bm = fa.create_block_mask(fullmask, 4, 8, 64, 64, device=dev)
    ref = ref_create_block_mask(o_full_masked, 4, 8, 64, 64)
    check(bm, ref)
    assert bm.sparsity() == 100.0


def test_python_callable_recognised_as_band(dev):
    def my_causal(b, h, q_idx, kv_idx):
        return q_idx >= kv_idx
    bm = fa.create_block_mask(my_causal, 1, 1, 512, 512, device=dev)
    assert bm.spec.bits is None and (bm.spec.lo, bm.spec.sink) == (0, -1)
    check(bm, ref_create_block_mask(o_causal_mask, 1, 1, 512, 512))


def test_python_callable_bitmap(dev):
    # depends on b and h, not a band: goes through the packed bitmap
    def weird(b, h, q_idx, kv_idx):
        return ((q_idx * 7 + kv_idx * 3 + h) % 11 < 6) & (kv_idx <= q_idx + 200 * b)
    bm = fa.create_block_mask(weird, 2, 3, 384, 640, device=dev)
    assert bm.spec.bits is not None
    check(bm, ref_create_block_mask(weird, 2, 3, 384, 640))

    def doc_mask(b, h, q_idx, kv_idx):  # document mask: block-diagonal, many full/empty tiles
        return (q_idx // 256) == (kv_idx // 256)
    bm = fa.create_block_mask(doc_mask, 1, 1, 1024, 1024, device=dev)
    check(bm, ref_create_block_mask(doc_mask, 1, 1, 1024, 1024))


def test_score_mod_as_mask(dev):
    # blockmask.py:307-315: a five-argument mod masks where it returns -inf
    def smod(score, b, h, q_idx, kv_idx):
        return torch.where(q_idx >= kv_idx, score, torch.full_like(score, -float("inf")))
    bm = fa.create_block_mask(smod, 1, 2, 256, 256, device=dev)
    check(bm, ref_create_block_mask(o_causal_mask, 1, 2, 256, 256))


def test_create_mask_matches_oracle(dev):
    """The public dense-mask helper (flaxattention/core/blockmask.py:277-322): a tagged mask, an untagged callable that
    looks at batch and head, a five-argument score_mod (masked where it returns -inf), and B = H = None."""
    from oracle import ref_create_mask

    def doc(b, h, q_idx, kv_idx):
        return ((q_idx // 40) == (kv_idx // 40)) & ((h + b) % 2 == 0)

    def as_score(score, b, h, q_idx, kv_idx):
        return torch.where(q_idx >= kv_idx, score, float("-inf"))
    for got_fn, want_fn, B, H in ((causal_mask, o_causal_mask, 2, 3), (doc, doc, 2, 3), (as_score, as_score, 1, 2),
                                  (generate_sliding_window(10), o_sliding_window(10), None, None)):
        got = fa.create_mask(got_fn, B, H, 100, 130, device=dev)
        want = ref_create_mask(want_fn, B, H, 100, 130)
        assert got.dtype == torch.bool and tuple(got.shape) == want.shape
        assert np.array_equal(got.cpu().numpy(), want)
    with pytest.raises(AssertionError):   # neither four nor five positional arguments (flaxattention/core/common.py:33)
        fa.create_mask(lambda a, b: a, 1, 1, 8, 8, device=dev)


def test_sparsity_and_repr(dev):
    bm = fa.create_block_mask(causal_mask, 1, 1, 2048, 2048, device=dev)
    assert abs(bm.sparsity() - 100 * (1 - 136 / 256)) < 1e-9
    assert "BlockMask(" in repr(bm) and "causal_mask" in repr(bm)
    assert bm.shape == (1, 1, 2048, 2048)
    t = bm.as_tuple()
    assert len(t) == 11 and t[8] == 128 and t[9] == 128 and t[10] is causal_mask


def test_from_kv_blocks_transposes(dev):
    bm = fa.create_block_mask(generate_sliding_window(200), 1, 2, 1024, 1024, device=dev)
    bm2 = fa.BlockMask.from_kv_blocks(bm.kv_num_blocks, bm.kv_indices, bm.full_kv_num_blocks, bm.full_kv_indices,
                                      mask_mod=bm.mask_mod)
    for f in ["q_num_blocks", "q_indices", "full_q_num_blocks", "full_q_indices"]:
        assert torch.equal(getattr(bm, f), getattr(bm2, f)), f


@pytest.mark.parametrize("seed", range(12))
def test_band_closed_form_matches_brute_force(dev, seed):
    """Band masks are classified per tile from its corners; the oracle evaluates every
    (q, kv) pair.  Random band parameters, including unbounded sides, sinks and offsets."""
    import random
    from flaxattention_amd.core.common import INT_MAX
    rnd = random.Random(50 + seed)
    Q, KV = rnd.choice([(256, 384), (300, 200), (512, 512), (64, 1000)])
    lo = rnd.choice([INT_MIN, 0, -17, 5, 130])
    hi = rnd.choice([INT_MAX, 10, 128, 333, max(lo, 0) + 40])
    sink = rnd.choice([-1, 0, 3, 127, 200])
    off = rnd.choice([0, 0, KV - Q, 13])
    bs = rnd.choice([128, 64, (128, 64)])
    print(f"band lo={lo} hi={hi} sink={sink} off={off} Q{Q} KV{KV} bs{bs}", flush=True)
    mask = MaskMod(lo, hi, sink, off, name="band")

    def omask(b, h, q_idx, kv_idx):
        d = q_idx + off - kv_idx
        return (d >= lo) & ((d <= hi) | (kv_idx <= sink))
    bm = fa.create_block_mask(mask, 1, 2, Q, KV, BLOCK_SIZE=bs, device=dev)
    check(bm, ref_create_block_mask(omask, 1, 2, Q, KV, BLOCK_SIZE=bs))


def test_head_and_batch_dependent_callable_at_config4_size(dev):
    """An untagged callable that depends on the batch and the head index, at [4,16,8192,8192]: the dense mask would be
    4.3 GB of booleans; it is evaluated in slabs and packed straight into bitmap words, so that building the block
    mask stays below 1 GiB of device memory, and the lists are the oracle's bit for bit."""
    import flaxattention_amd as fa
    B, H, L = 4, 16, 8192

    def mask(b, h, q_idx, kv_idx):
        return (q_idx >= kv_idx) & (((q_idx - kv_idx) <= 256 * (h + 1) + 64 * b) | (kv_idx < 4))
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats(dev)
    base = torch.cuda.memory_allocated(dev)
    bm = fa.create_block_mask(mask, B, H, L, L, device=dev)
    torch.cuda.synchronize()
    peak = torch.cuda.max_memory_allocated(dev) - base
    print(f"  peak device memory while building: {peak / 2 ** 20:.0f} MiB", flush=True)
    assert peak < 2 ** 30
    assert bm.spec.bits is not None and tuple(bm.spec.bits.shape) == (B, H, L, L // 32)
    for b0, h0 in ((0, 0), (3, 15), (2, 5)):
        ref = ref_create_block_mask(lambda b, h, q, kv: mask(b + b0, h + h0, q, kv), 1, 1, L, L)
        for f in ("kv_num_blocks", "kv_indices", "full_kv_num_blocks", "full_kv_indices", "q_num_blocks", "q_indices",
                  "full_q_num_blocks", "full_q_indices"):
            assert (getattr(bm, f)[b0, h0].cpu().numpy() == ref[f][0, 0]).all(), (f, b0, h0)


@pytest.mark.parametrize("shape", [(1, 1, 128, 128), (2, 3, 128, 384), (1, 2, 384, 128), (3, 1, 256, 640)])
def test_packed_bitmap_equals_torch_formulas(dev, shape):
    """The packing kernel (words along the keys, words along the queries, 32 x 32 classes) against the torch formulas on
    the CPU, bit for bit: slabs of rows, non-contiguous and broadcast inputs, all-set / all-clear / mixed blocks."""
    from flaxattention_amd.core.common import _pack_slab, block_classes, pack_bits
    nb, nh, Q, KV = shape
    print("case pack", shape, flush=True)
    g = torch.Generator().manual_seed(Q + KV)
    m = torch.rand(shape, generator=g) < 0.3
    m[..., :64, :96] = True
    m[..., 32:64, 32:64] = False
    m[..., 96:, 64:96] = False
    forms = {"contiguous": m.to(dev), "transposed": m.transpose(2, 3).contiguous().to(dev).transpose(2, 3),
             "every other": torch.stack([m, ~m], -1).reshape(nb, nh, Q, 2 * KV).to(dev)[..., ::2],
             "rows broadcast": m[:, :, :1].to(dev).expand(shape), "maps broadcast": m[:1, :1].to(dev).expand(shape)}
    for name, md in forms.items():
        want = md.cpu().reshape(nb * nh, Q, KV)
        for step in (Q, 128):
            bits = torch.full((nb * nh + 1, Q, KV // 32), -7, dtype=torch.int32, device=dev)
            bits_t = torch.full((nb * nh + 1, KV, Q // 32), -7, dtype=torch.int32, device=dev)
            blk = torch.full((nb * nh + 1, Q // 32, KV // 32), -7, dtype=torch.int8, device=dev)
            for q0 in range(0, Q, step):
                _pack_slab(md[:, :, q0:q0 + step], q0, 1, bits, bits_t, blk)
            assert torch.equal(bits[1:].cpu(), pack_bits(want)), name
            assert torch.equal(bits_t[1:].cpu(), pack_bits(want.transpose(1, 2).contiguous())), name
            assert torch.equal(blk[1:].cpu(), block_classes(want)), name
            assert all(bool((t[0] == -7).all()) for t in (bits, bits_t, blk)), name   # nothing written ahead of its map


@pytest.mark.parametrize("Q,KV", [(128, 128), (256, 384), (384, 128)])
def test_band_fit_of_packed_bitmaps(dev, Q, KV):
    """The fit on the device finds exactly the bands, on every entry: each verdict against the entries themselves."""
    from flaxattention_amd.core.common import INT_MAX, INT_MIN, MaskMod, _fit_bitmaps, pack_bits
    print("case fit", Q, KV, flush=True)
    q, kv = torch.arange(Q, dtype=torch.int32).reshape(Q, 1), torch.arange(KV, dtype=torch.int32).reshape(1, KV)
    zero = torch.zeros((), dtype=torch.int32)
    bands = [(lo, hi, sink) for lo in (INT_MIN, -KV + 1, -5, 0, 31, Q - 1, Q, INT_MAX)
             for hi, sink in ((INT_MAX, -1), (Q - 1, -1), (Q - 2, 0), (40, -1), (40, 3), (33, 32), (0, 64), (-3, 5))]
    dense = lambda m: torch.broadcast_to(m(zero, zero, q, kv), (Q, KV))
    for b in bands:
        m = dense(MaskMod(*b))
        same, got = _fit_bitmaps(pack_bits(m)[None].to(dev))
        assert same and got is not None and torch.equal(dense(got), m), b
    m = dense(MaskMod(0, 40, 3))
    words = pack_bits(m)
    for r, c in ((0, 0), (Q - 1, KV - 1), (Q // 2, 0), (Q // 2, KV - 1), (Q - 1, 7)):   # one entry off: no band any more
        off = m.clone()
        off[r, c] = ~off[r, c]
        same, got = _fit_bitmaps(pack_bits(off)[None].to(dev))
        assert same and (got is None or torch.equal(dense(got), off)), (r, c)
        assert _fit_bitmaps(torch.stack([words, words, pack_bits(off)]).to(dev)) == (False, None), (r, c)
    same, got = _fit_bitmaps(torch.stack([words, words]).to(dev))
    assert same and torch.equal(dense(got), m)
    g = torch.Generator().manual_seed(Q)
    assert _fit_bitmaps(pack_bits(torch.rand(Q, KV, generator=g) < 0.5)[None].to(dev)) == (True, None)


@pytest.mark.parametrize("bs", [32, 64, 128, (64, 96), (96, 32), (160, 128), (48, 80), 256, (512, 32), (32, 512), (64, 1024)], ids=str)
@pytest.mark.parametrize("B,H,Q,KV", [(2, 1, 700, 700), (1, 3, 130, 1000), (2, 2, 33, 31)])
def test_lists_of_bitmaps_at_any_block_size(dev, B, H, Q, KV, bs):
    """Tiles made of up to 16 whole 32 x 32 blocks are told by the blocks' classes, others by counting bits; empty, full and mixed tiles,
    maps that differ by batch and head, lengths that end inside a tile."""
    print("case bitmap lists", B, H, Q, KV, bs, flush=True)
    gen = torch.Generator().manual_seed(Q + KV)
    doc = torch.randint(0, 3, (B, H, 64), generator=gen).repeat_interleave(29, dim=2)   # 29 positions a piece

    def mask(b, h, q, kv):
        table = doc.to(q.device)   # (positions past the lengths are padding: a captured table is read at the last one there)
        return table[b, h, q.clamp(max=Q - 1)] >= table[b, h, kv.clamp(max=KV - 1)]
    check(fa.create_block_mask(mask, B, H, Q, KV, BLOCK_SIZE=bs, device=dev), ref_create_block_mask(mask, B, H, Q, KV, BLOCK_SIZE=bs))


@pytest.mark.parametrize("B,H", [(1, 1), (2, 8), (3, 6), (4, 16)])
@pytest.mark.parametrize("bs", [64, 128, 256])
def test_lists_of_a_map_that_all_heads_share(dev, B, H, bs):
    """One bitmap for every (batch, head): up to 16 of them read its classes themselves, more order flags that were made once."""
    print("case shared map", B, H, bs, flush=True)
    ids = torch.randint(0, 3, (40,), generator=torch.Generator().manual_seed(bs)).repeat_interleave(29)

    def mask(b, h, q, kv):
        table = ids.to(q.device)
        return table[q.clamp(max=999)] >= table[kv.clamp(max=899)]   # (past the lengths: padding, read at the last position)
    check(fa.create_block_mask(mask, B, H, 1000, 900, BLOCK_SIZE=bs, device=dev), ref_create_block_mask(mask, B, H, 1000, 900, BLOCK_SIZE=bs))


@pytest.mark.parametrize("B,H", [(16, 16), (1, 257), (16, 32)])
@pytest.mark.parametrize("lo,hi,sink,off", [(0, INT_MAX, -1, 0), (0, 60, 40, 3), (5, 4, 70, 0), (-300, -90, -1, 0)])
@pytest.mark.parametrize("bs", [32, (48, 80)], ids=str)
def test_lists_of_a_band_that_many_heads_share(dev, B, H, lo, hi, sink, off, bs):
    """A band for more than 256 (batch, head): flags made once by a thread a tile, the same lists for all as for a single one."""
    print("case shared band", B, H, lo, hi, sink, off, bs, flush=True)
    mask = MaskMod(lo, hi, sink, off, name="band")
    one = fa.create_block_mask(mask, 1, 1, 600, 700, BLOCK_SIZE=bs, device=dev)
    all_heads = fa.create_block_mask(mask, B, H, 600, 700, BLOCK_SIZE=bs, device=dev)

    def omask(b, h, q_idx, kv_idx):
        d = q_idx + off - kv_idx
        return (d >= lo) & ((d <= hi) | (kv_idx <= sink))
    check(one, ref_create_block_mask(omask, 1, 1, 600, 700, BLOCK_SIZE=bs))
    for name in ("kv_num_blocks", "kv_indices", "full_kv_num_blocks", "full_kv_indices", "q_num_blocks", "q_indices",
                 "full_q_num_blocks", "full_q_indices"):
        a, b = getattr(all_heads, name), getattr(one, name)
        assert torch.equal(a, b.expand_as(a)), name


@pytest.mark.parametrize("bs", [32, 128, (48, 80), (128, 1), (1, 64)], ids=str)
@pytest.mark.parametrize("lo,hi,sink,off", [(5, 4, -1, 0), (5, 4, 70, 0), (5, 4, 79, 3), (0, -1, 127, 0), (2**31 - 1, 2**31 - 1, -1, 0), (-300, -90, -1, 0),
                                            (-300, -90, 31, -7), (INT_MIN, -1, 40, 0), (0, 0, -1, 0), (INT_MIN, 2**31 - 1, -1, 0), (0, 63, 1000, 50)])
def test_band_edges_against_brute_force(dev, lo, hi, sink, off, bs):
    """Empty bands with and without sinks (inside a tile, on its last key), bands ahead of the diagonal, unbounded sides, a band of
    one key, tiles of one row or one key."""
    print("case band edges", lo, hi, sink, off, bs, flush=True)

    def omask(b, h, q_idx, kv_idx):
        d = q_idx + off - kv_idx
        return (d >= lo) & ((d <= hi) | (kv_idx <= sink))
    check(fa.create_block_mask(MaskMod(lo, hi, sink, off, name="band"), 1, 1, 200, 330, BLOCK_SIZE=bs, device=dev),
          ref_create_block_mask(omask, 1, 1, 200, 330, BLOCK_SIZE=bs))
