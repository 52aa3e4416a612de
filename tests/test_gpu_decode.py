"""Split-KV decode kernel vs the CPU oracle, and vs the prefill kernel."""
import math

import pytest
import torch

import flaxattention_amd as fa
from flaxattention_amd.masks import generate_sliding_window, offset_causal_mask
from flaxattention_amd.mods import generate_alibi_bias, generate_tanh_softcap
from oracle import (max_abs, o_alibi_config, o_offset_causal, o_tanh_softcap, ref_attention, rel_l2, seeded_qkv)

pytestmark = pytest.mark.gpu


def run_decode(dev, dtype, B, Hq, Hkv, Lq, Lkv, D, splits, score=None, oscore=None, mask=None, omask=None, numerics=None):
    """numerics None: the default (fp16 "fast", bf16 "parity"), held to the stated 1e-3; "fast" on bf16 is the one
    explicitly named case with the widened bound."""
    print(f"decode case {dtype} B{B} Hq{Hq} Hkv{Hkv} Lq{Lq} Lkv{Lkv} D{D} splits{splits} numerics {numerics}", flush=True)
    opts = {"decode_splits": splits}
    if numerics is not None:
        opts["numerics"] = numerics
    q, k, v = seeded_qkv(B, Hq, Hkv, Lq, Lkv, D, dtype)
    bm = fa.create_block_mask(mask, B, Hq, Lq, Lkv, device=dev) if mask is not None else None
    out, lse = fa.flax_attention(q.to(dev), k.to(dev), v.to(dev), score_mod=score, block_mask=bm,
                                 enable_gqa=Hq != Hkv, return_lse=True, kernel_options=opts)
    want, want_lse = ref_attention(q, k, v, oscore, omask, strict=True, return_lse=True)
    a, r = max_abs(out.cpu(), want), rel_l2(out.cpu(), want)
    print(f"  O: max-abs {a:.3e} rel-L2 {r:.3e}", flush=True)
    assert a <= 2e-2 and r <= (6e-3 if (dtype == torch.bfloat16 and numerics == "fast") else 1e-3)
    dead = torch.isneginf(want_lse)
    assert torch.equal(torch.isneginf(lse.cpu()), dead)
    assert max_abs(lse.cpu()[~dead], want_lse[~dead]) <= 2e-2
    return out


@pytest.mark.parametrize("Lq", [1, 16, 64])
@pytest.mark.parametrize("splits", [1, 5, 16])
def test_decode_alibi_offset_causal(dev, Lq, splits):
    # benchmark configuration 5 at reduced KV length
    Lkv = 2048
    run_decode(dev, torch.float16, 2, 8, 8, Lq, Lkv, 64, splits, generate_alibi_bias(8, -1.0), o_alibi_config(8),
               offset_causal_mask(Lkv - Lq), o_offset_causal(Lkv - Lq))


def test_decode_gqa_packs_heads(dev):
    for numerics in (None, "fast"):
        run_decode(dev, torch.bfloat16, 2, 8, 2, 4, 1000, 128, 4, generate_tanh_softcap(30.0), o_tanh_softcap(30.0),
                   offset_causal_mask(996), o_offset_causal(996), numerics=numerics)
    run_decode(dev, torch.float16, 1, 16, 2, 8, 777, 64, 3)       # 64 columns, no mask, ragged KV


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("Lq,D,splits", [(1, 64, 8), (16, 64, 3), (64, 64, 5), (3, 128, 4), (40, 128, 2)])
def test_decode_parity_numerics(dev, dtype, Lq, D, splits):
    """Two-pass decode (merged log-sum-exp, then the normalised rounded P) against the strict oracle at 1e-3."""
    Lkv = 1500
    run_decode(dev, dtype, 2, 4, 4, Lq, Lkv, D, splits, generate_alibi_bias(4, -1.0), o_alibi_config(4),
               offset_causal_mask(Lkv - Lq), o_offset_causal(Lkv - Lq), numerics="parity")


@pytest.mark.parametrize("dtype,numerics", [(torch.float16, None), (torch.bfloat16, None), (torch.bfloat16, "fast"),
                                            (torch.float16, "parity")], ids=["f16", "bf16", "bf16-fast", "f16-parity"])
@pytest.mark.parametrize("Lq,G,splits", [(1, 1, 8), (7, 4, 3), (32, 1, 5), (2, 16, 1)])
@pytest.mark.parametrize("D", [192, 256])
def test_decode_wide_heads(dev, dtype, numerics, Lq, G, splits, D):
    """D = 192 / 256: one column block (at most 32 columns); ALiBi + offset-causal with a ragged KV length, GQA packing."""
    Lkv, Hkv = 1237, 2
    run_decode(dev, dtype, 2, Hkv * G, Hkv, Lq, Lkv, D, splits, generate_alibi_bias(Hkv * G, -1.0), o_alibi_config(Hkv * G),
               offset_causal_mask(Lkv - Lq), o_offset_causal(Lkv - Lq), numerics=numerics)


@pytest.mark.parametrize("D", [192, 256])
def test_decode_wide_heads_choice_and_chunks(dev, D):
    """D = 192 / 256 are routed to the decode kernel up to 32 columns per call; longer queries go there in chunks of 32
    rows on request; the library refuses more than 32 columns in one call and the results agree with the forward
    kernel."""
    from flaxattention_amd.core.attention import _make_plan
    from flaxattention_amd import _lib
    B, H, Lq, Lkv = 1, 2, 80, 4096
    q, k, v = seeded_qkv(B, H, H, Lq, Lkv, D, torch.float16)
    mask, omask = offset_causal_mask(Lkv - Lq), o_offset_causal(Lkv - Lq)
    bm = fa.create_block_mask(mask, B, H, Lq, Lkv, device=dev)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    assert _make_plan(qd[:, :, :32], kd, vd, None, None, None, 0.0625, None).decode_splits < 0
    assert _make_plan(qd, kd, vd, None, bm, None, 0.0625, None).decode_splits == 0         # 80 rows: the forward kernel
    assert _make_plan(qd, kd, vd, None, bm, None, 0.0625, {"decode": True}).decode_splits < 0   # on request: three calls
    out, lse = fa.flax_attention(qd, kd, vd, score_mod=generate_alibi_bias(H, -1.0), block_mask=bm, return_lse=True,
                                 kernel_options={"decode": True})
    want, want_lse = ref_attention(q, k, v, o_alibi_config(H), omask, strict=True, return_lse=True)
    a, r = max_abs(out.cpu(), want), rel_l2(out.cpu(), want)
    print(f"  chunked decode at D={D} O: max-abs {a:.3e} rel-L2 {r:.3e}", flush=True)
    assert a <= 2e-2 and r <= 1e-3
    assert max_abs(lse.cpu(), want_lse) <= 2e-2
    ref = fa.flax_attention(qd, kd, vd, score_mod=generate_alibi_bias(H, -1.0), block_mask=bm, kernel_options={"decode": False})
    assert max_abs(out.cpu(), ref.cpu()) <= 2e-3
    # 33 query heads on one KV head are 33 columns in one call: refused by the library with a message, nothing launched
    q33 = torch.randn(1, 33, 1, D, device=dev, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="at most 32"):
        fa.flax_attention(q33, kd[:, :1], vd[:, :1], enable_gqa=True, kernel_options={"decode_splits": 4})
    # left to itself the front-end takes the forward kernel for that shape
    assert _make_plan(q33, kd[:, :1], vd[:, :1], None, None, None, 0.0625, None).decode_splits == 0


def test_decode_window_uses_tile_lists(dev):
    # only the last 300 keys are visible: most tiles are skipped through the lists
    Lkv, Lq, W = 4096, 2, 300
    from oracle import o_and_masks
    def owin(b, h, q_idx, kv_idx):
        return (q_idx + (Lkv - Lq) - kv_idx <= W) & (q_idx + (Lkv - Lq) >= kv_idx)
    from flaxattention_amd.core.common import MaskMod
    mask = MaskMod(lo=0, hi=W, sink=-1, q_offset=Lkv - Lq, name="decode_window")
    run_decode(dev, torch.float16, 1, 4, 4, Lq, Lkv, 64, 8, mask=mask, omask=owin)


def test_decode_independent_of_split_count(dev):
    q, k, v = (t.to(dev) for t in seeded_qkv(1, 4, 4, 1, 4096, 64, torch.float16))
    outs = [fa.flax_attention(q, k, v, kernel_options={"decode_splits": s}) for s in (1, 2, 7, 32)]
    for o in outs[1:]:
        assert max_abs(o.cpu(), outs[0].cpu()) <= 2e-3


def test_decode_matches_prefill_kernel(dev):
    q, k, v = (t.to(dev) for t in seeded_qkv(2, 8, 8, 16, 4096, 64, torch.float16))
    m = offset_causal_mask(4096 - 16)
    bm = fa.create_block_mask(m, 1, 1, 16, 4096, device=dev)
    a = fa.flax_attention(q, k, v, score_mod=generate_alibi_bias(8, -1.0), block_mask=bm, kernel_options={"decode_splits": 16})
    b = fa.flax_attention(q, k, v, score_mod=generate_alibi_bias(8, -1.0), block_mask=bm, kernel_options={"decode_splits": 0, "decode": False})
    assert max_abs(a.cpu(), b.cpu()) <= 4e-3


def test_decode_is_chosen_automatically(dev):
    """Short queries against a long KV cache take the decode kernel without being asked;
    {"decode": False} keeps the forward kernel; both agree, and the gradient path is unaffected."""
    from flaxattention_amd.core.attention import _make_plan
    q, k, v = (t.to(dev) for t in seeded_qkv(2, 4, 4, 4, 1024, 64, torch.float16))
    assert _make_plan(q, k, v, None, None, None, 0.125, None).decode_splits < 0
    assert _make_plan(q, k, v, None, None, None, 0.125, {"decode": False}).decode_splits == 0
    assert _make_plan(q, k[:, :, :256], v[:, :, :256], None, None, None, 0.125, None).decode_splits == 0
    assert _make_plan(q.float(), k.float(), v.float(), None, None, None, 0.125, None).decode_splits == 0
    qg = q.clone().requires_grad_(True)
    a = fa.flax_attention(qg, k, v, score_mod=generate_alibi_bias(4))
    b = fa.flax_attention(q, k, v, score_mod=generate_alibi_bias(4), kernel_options={"decode": False})
    assert max_abs(a.detach().cpu(), b.cpu()) <= 2e-3
    a.sum().backward()
    assert torch.isfinite(qg.grad).all() and qg.grad.abs().max() > 0


def test_decode_in_chunks_of_64_rows(dev):
    """On request ({"decode": True}) queries of more than 64 rows run as several decode calls, each seeing its
    row offset in score_mod, mask_mod and the tile lists (ALiBi + offset-causal, ragged last chunk)."""
    from flaxattention_amd.core.attention import _make_plan
    B, H, Lq, Lkv, D = 1, 2, 160, 4096, 64
    q, k, v = seeded_qkv(B, H, H, Lq, Lkv, D, torch.float16)
    mask, omask = offset_causal_mask(Lkv - Lq), o_offset_causal(Lkv - Lq)
    bm = fa.create_block_mask(mask, B, H, Lq, Lkv, device=dev)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    assert _make_plan(qd, kd, vd, None, bm, None, 0.125, None).decode_splits == 0         # by default: the forward kernel
    assert _make_plan(qd, kd, vd, None, bm, None, 0.125, {"decode": True}).decode_splits < 0
    out, lse = fa.flax_attention(qd, kd, vd, score_mod=generate_alibi_bias(H, -1.0), block_mask=bm, return_lse=True,
                                 kernel_options={"decode": True})
    want, want_lse = ref_attention(q, k, v, o_alibi_config(H), omask, strict=True, return_lse=True)
    a, r = max_abs(out.cpu(), want), rel_l2(out.cpu(), want)
    print(f"  chunked decode O: max-abs {a:.3e} rel-L2 {r:.3e}", flush=True)
    assert a <= 2e-2 and r <= 1e-3
    assert max_abs(lse.cpu(), want_lse) <= 2e-2
    ref = fa.flax_attention(qd, kd, vd, score_mod=generate_alibi_bias(H, -1.0), block_mask=bm, kernel_options={"decode": False})
    assert max_abs(out.cpu(), ref.cpu()) <= 2e-3


def test_decode_in_chunks_with_gqa_packing(dev):
    """{"decode": True} with several query heads per KV head: a call takes 64 / G rows, so the chunks start at row
    offsets that are multiples of 16 here (sink + window band mask, ALiBi, bf16 in its default numerics)."""
    from flaxattention_amd.core.common import MaskMod
    B, Hq, Hkv, Lq, Lkv, D = 2, 8, 2, 82, 2047, 128
    q, k, v = seeded_qkv(B, Hq, Hkv, Lq, Lkv, D, torch.bfloat16)
    off = Lkv - Lq
    mask = MaskMod(lo=0, hi=700, sink=4, q_offset=off, name="decode_sink_window")
    def omask(b, h, q_idx, kv_idx):
        d = q_idx + off - kv_idx
        return ((d >= 0) & (d <= 700)) | ((kv_idx <= 4) & (d >= 0))   # MaskMod: keys 0 .. sink stay visible
    bm = fa.create_block_mask(mask, B, Hq, Lq, Lkv, device=dev)
    out, lse = fa.flax_attention(q.to(dev), k.to(dev), v.to(dev), score_mod=generate_alibi_bias(Hq, -1.0), block_mask=bm,
                                 enable_gqa=True, return_lse=True, kernel_options={"decode": True})
    want, want_lse = ref_attention(q, k, v, o_alibi_config(Hq), omask, strict=True, return_lse=True)
    a, r = max_abs(out.cpu(), want), rel_l2(out.cpu(), want)
    print(f"  chunked decode with GQA O: max-abs {a:.3e} rel-L2 {r:.3e}", flush=True)
    assert a <= 2e-2 and r <= 1e-3
    assert max_abs(lse.cpu(), want_lse) <= 2e-2


@pytest.mark.parametrize("Lq", [1, 200])
def test_calls_replay_from_a_captured_graph(dev, Lq):
    """Nothing on the path synchronises, allocates outside the caller's allocator or records a memset, so a serving
    loop can capture a call (here one decode call, and a 200-row query served as four decode calls) in a HIP graph
    and replay it.  Every replay, with eager work of the same kind between the replays, gives the eager call's bits."""
    print(f"case graph capture q_len {Lq}", flush=True)
    B, H, Lkv, D = 2, 8, 4096, 64
    g0 = torch.Generator(device="cpu").manual_seed(0)
    mk = lambda *s: torch.randn(*s, generator=g0, dtype=torch.float32).to(torch.float16).to(dev)
    K, V, q_static = mk(B, H, Lkv, D), mk(B, H, Lkv, D), mk(B, H, Lq, D)
    bm = fa.create_block_mask(offset_causal_mask(Lkv - Lq), 1, 1, Lq, Lkv, device=dev)
    call = lambda q: fa.flax_attention(q, K, V, score_mod=generate_alibi_bias(H, -1.0), block_mask=bm, return_lse=True)
    side = torch.cuda.Stream()   # default priority; warm-up off the default stream as graph capture asks
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            call(q_static)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out_static, lse_static = call(q_static)
    for i in range(4):
        q_new = mk(B, H, Lq, D)
        q_static.copy_(q_new)
        graph.replay()
        eager, eager_lse = call(q_new)
        torch.cuda.synchronize()
        assert torch.equal(out_static, eager) and torch.equal(lse_static, eager_lse), f"replay {i} differs from the eager call"


@pytest.mark.parametrize("Lq", [1, 64])
def test_decode_kv_cache_beyond_2_31_elements(dev, Lq):
    """A KV cache of more than 2^31 elements per tensor (more than 2^32 bytes): the rows of its last (batch, head) pair
    lie beyond what 32 bits address.  The pairs of a call are independent, so the last pair's output must equal,
    bit for bit, a decode call on that pair's slice of the cache alone."""
    B, H, Lkv, D = 33, 16, 65536, 64
    assert B * H * Lkv * D > 2 ** 31
    g = torch.Generator(device=dev).manual_seed(9)
    mk = lambda *s: torch.randn(s, generator=g, dtype=torch.float16, device=dev)
    K, V, q = mk(B, H, Lkv, D), mk(B, H, Lkv, D), mk(B, H, Lq, D)
    bm = fa.create_block_mask(offset_causal_mask(Lkv - Lq), 1, 1, Lq, Lkv, device=dev)
    opts = {"decode_splits": 4}
    out, lse = fa.flax_attention(q, K, V, score_mod=generate_alibi_bias(H, -1.0), block_mask=bm, return_lse=True,
                                 kernel_options=opts)
    b, h = B - 1, H - 1
    # head H-1 of H has the ALiBi slope 2^-8, and so has head 0 of 1
    out1, lse1 = fa.flax_attention(q[b:b + 1, h:h + 1].clone(), K[b:b + 1, h:h + 1].clone(), V[b:b + 1, h:h + 1].clone(),
                                   score_mod=generate_alibi_bias(1, -1.0), block_mask=bm, return_lse=True, kernel_options=opts)
    torch.cuda.synchronize()
    assert torch.equal(out[b:b + 1, h:h + 1], out1) and torch.equal(lse[b:b + 1, h:h + 1], lse1)


@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lkv,D,mask", [
    (1, 64, 8, 4, 33000, 128, "none"),      # 32 columns: the widest call that keeps its scores at D = 128
    (32, 64, 16, 4, 8200, 64, "causal"),    # 16 columns, the widest at D = 64; the last step ragged
    (40, 32, 8, 2, 6200, 192, "window"),
    (48, 32, 16, 1, 12001, 256, "window")])
def test_parity_decode_with_and_without_kept_scores(dev, B, Hq, Hkv, Lq, Lkv, D, mask):
    """The parity numerics keep their rounded scores between the two passes where the workspace has room: beyond
    the 16 MiB of flexattn_decode_static the same call reads K twice instead.  Outputs and log-sum-exps are the same bits."""
    from flaxattention_amd import _lib
    from flaxattention_amd.core.attention import _Plan
    from flaxattention_amd.core.common import IDENTITY, MaskMod
    print("case kept scores", B, Hq, Hkv, Lq, Lkv, D, mask, flush=True)
    g = torch.Generator(device=dev).manual_seed(3)
    mk = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    q, k, v = mk(B, Hq, Lq, D), mk(B, Hkv, Lkv, D), mk(B, Hkv, Lkv, D)
    m = {"none": MaskMod(), "causal": MaskMod(0, q_offset=Lkv - Lq), "window": MaskMod(0, 700, 3, Lkv - Lq)}[mask]
    got = []
    L, s = _lib.lib(), torch.cuda.current_stream().cuda_stream
    for static in (False, True):
        o, lse = torch.empty_like(q), torch.empty((B, Hq, Lq), device=dev)
        plan = _Plan(q, k, v, IDENTITY, m, None, D ** -0.5, _lib.FLAG_PARITY | _lib.FLAG_ROUND_S, True)
        p = plan.params(q, k, v, o)
        nbytes = L.flexattn_decode_workspace_bytes(p, 0)
        assert nbytes > 16 << 20
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        args = (p, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), 0)
        _lib.check(L.flexattn_decode_static(*args, s) if static else L.flexattn_decode(*args, ws.data_ptr(), s), "decode")
        torch.cuda.synchronize()
        got.append((o, lse))
    assert torch.isfinite(got[0][0].float()).all() and torch.isfinite(got[0][1]).all()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    # and against the same formulas in float64 for one (batch, head): P rounds to 8 bits, so 2^-8 relative
    qs, ks, vs = q[-1, -1].double(), k[-1, -1].double(), v[-1, -1].double()
    i = torch.arange(Lq, device=dev).reshape(-1, 1)
    x = (qs @ ks.T) * D ** -0.5
    x = x.masked_fill(~m(None, None, i, torch.arange(Lkv, device=dev).reshape(1, -1)), -float("inf")) if mask != "none" else x
    want = torch.softmax(x, -1) @ vs
    assert ((got[0][0][-1, -1].double() - want).norm() / want.norm()).item() < 2 ** -6


@pytest.mark.parametrize("B,H,Lq,Lkv,D,mask,splits", [
    (16, 32, 4, 8200, 64, "lengths", 0),   # 34 MB of scores: the static variant reads K twice, for the same bits
    (2, 3, 1, 8200, 128, "lengths", 0), (12, 8, 16, 2080, 64, "sink", 6), (1, 5, 32, 4097, 128, "sink", 0),
    (3, 2, 2, 1025, 256, "lengths", 0), (2, 2, 1, 1056, 192, "sink", 3), (2, 3, 1, 640, 128, "lengths", 0)])
def test_kept_scores_of_a_listed_tile_that_ends_past_the_last_key(dev, B, H, Lq, Lkv, D, mask, splits):
    """Steps that come from tile lists are halves of 64-key tiles, so the last one may hold no key at all: its scores have
    no slot.  Nothing is written past the workspace or into a neighbour's scores, every (batch, head) against float64."""
    from flaxattention_amd import _lib
    from flaxattention_amd.core.attention import _make_plan
    from flaxattention_amd.core.common import MaskMod
    print("case kept scores, listed tail", B, H, Lq, Lkv, D, mask, flush=True)
    g = torch.Generator(device=dev).manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    q, k, v = mk(B, H, Lq, D), mk(B, H, Lkv, D), mk(B, H, Lkv, D)
    lens = torch.tensor([Lkv - 3 * b for b in range(B)], device=dev)
    mod = (lambda b, h, q_idx, kv_idx: kv_idx < lens[b]) if mask == "lengths" else MaskMod(0, 700, 3, Lkv - Lq)
    bm = fa.create_block_mask(mod, B, None, Lq, Lkv, device=dev)
    plan = _make_plan(q, k, v, None, bm, None, D ** -0.5, None)
    assert plan.decode_splits != 0 and plan.lists is not None and plan.flags & _lib.FLAG_PARITY
    o, lse = torch.empty_like(q), torch.empty((B, H, Lq), device=dev)
    L, s = _lib.lib(), torch.cuda.current_stream().cuda_stream
    p = plan.params(q, k, v, o)
    nbytes = L.flexattn_decode_workspace_bytes(p, splits)
    assert nbytes > B * H * ((Lkv + 31) // 32) * Lq * 64     # the scores are kept
    ws = torch.full((nbytes + (1 << 20),), 0x5A, dtype=torch.uint8, device=dev)
    args = (p, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), splits)
    _lib.check(L.flexattn_decode(*args, ws.data_ptr(), s), "decode")
    torch.cuda.synchronize()
    assert bool((ws[nbytes:] == 0x5A).all())
    i = torch.arange(Lq, device=dev).reshape(-1, 1)
    kv = torch.arange(Lkv, device=dev).reshape(1, -1)
    for b in range(B):
        vis = torch.broadcast_to(mod(b, None, i, kv), (Lq, Lkv))
        x = ((q[b].double() @ k[b].double().transpose(-1, -2)) * D ** -0.5).masked_fill(~vis, -float("inf"))
        want = torch.softmax(x, -1) @ v[b].double()
        rel = (o[b].double() - want).norm(dim=(1, 2)) / want.norm(dim=(1, 2))
        assert rel.max().item() < 2 ** -6, b     # scores and P round to 8 bits: 2^-8 relative
        # (the scores are rounded: 2^-9 of up to 5, and the log-sum-exp averages them)
        assert (lse[b].double() * math.log(2) - torch.logsumexp(x, -1)).abs().max().item() < 1e-2, b
    if nbytes > 16 << 20:
        o2, lse2 = torch.empty_like(o), torch.empty_like(lse)
        args = (p, q.data_ptr(), k.data_ptr(), v.data_ptr(), o2.data_ptr(), lse2.data_ptr(), splits)
        _lib.check(L.flexattn_decode_static(*args, s), "decode_static")
        torch.cuda.synchronize()
        assert torch.equal(o, o2) and torch.equal(lse, lse2)


def test_parity_decode_beyond_the_bound_of_kept_scores(dev):
    """A call whose scores would take more than the stated bound reads K twice: the same bits as its batch elements in
    calls that keep theirs."""
    from flaxattention_amd import _lib
    from flaxattention_amd.core.attention import _make_plan
    B, G, Hkv, Lkv, D, part = 40, 32, 16, 8300, 128, 8
    print("case beyond the bound", flush=True)
    g = torch.Generator(device=dev).manual_seed(6)
    mk = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    q, k, v = mk(B, G * Hkv, 1, D), mk(B, Hkv, Lkv, D), mk(B, Hkv, Lkv, D)
    kept = []
    for n in (B, part):
        plan = _make_plan(q[:n], k[:n], v[:n], None, None, None, D ** -0.5, None)
        p = plan.params(q[:n], k[:n], v[:n], q[:n])
        kept.append(_lib.lib().flexattn_decode_workspace_bytes(p, 2) - (n * G * Hkv * 2 * (D + 2) * 4 + 255) // 256 * 256)
    assert kept == [0, part * Hkv * ((Lkv + 31) // 32) * G * 64]
    opts = {"decode_splits": 2}
    out, lse = fa.flax_attention(q, k, v, enable_gqa=True, return_lse=True, kernel_options=opts)
    for b in range(0, B, part):
        o, l = fa.flax_attention(q[b:b + part], k[b:b + part], v[b:b + part], enable_gqa=True, return_lse=True, kernel_options=opts)
        assert torch.equal(o, out[b:b + part]) and torch.equal(l, lse[b:b + part]), b
