// Fused flash-attention backward for gfx950 (fp16 / bf16, D = Dv in {64, 128}; dQ also at 192 / 256): checks and dispatch.  The kernels are
// in bwd_mfma.cuh, instantiated per (dtype, head size) by bwd_mfma_inst.hip.
#include <cmath>

#include "bwd_mfma.cuh"

using namespace flex;
void flex_set_error(const char* fmt, ...);
int flex_cu_count();
bool flex_mfma_shape_ok(const FlexAttnParams& p);
int flex_mfma_bwd_f16_64(const FlexAttnParams& p, const BwdArgs& a);
int flex_mfma_bwd_f16_128(const FlexAttnParams& p, const BwdArgs& a);
int flex_mfma_bwd_bf16_64(const FlexAttnParams& p, const BwdArgs& a);
int flex_mfma_bwd_bf16_128(const FlexAttnParams& p, const BwdArgs& a);
int flex_mfma_bwd_f16_192(const FlexAttnParams& p, const BwdArgs& a);   // dQ kernels only
int flex_mfma_bwd_bf16_192(const FlexAttnParams& p, const BwdArgs& a);  // dQ kernels only
int flex_mfma_bwd_f16_256(const FlexAttnParams& p, const BwdArgs& a);   // dQ kernels only
int flex_mfma_bwd_bf16_256(const FlexAttnParams& p, const BwdArgs& a);  // dQ kernels only

// 192- and 256-wide heads: the dQ kernel (and its row sweep) is instantiated, the dK/dV kernel is not.  A backward call
// at those sizes is served by flex_mfma_bwd with FLEX_BWD_ONLY_DQ set and the dK/dV kernel of the simple family.
bool flex_mfma_dq_wide_supported(const FlexAttnParams& p) {
  if (p.D != p.Dv || (p.D != 192 && p.D != 256) || (p.flags & FLEX_UNROUNDED)) return false;
  FlexAttnParams as128 = p;  // everything but the head size is checked as for 128
  as128.D = as128.Dv = 128;
  if (!flex_mfma_shape_ok(as128)) return false;
  const FlexTileLists& t = p.tiles_bwd;
  return !t.kv_num || (t.q_block == kBM && t.kv_block == kListBN);
}

bool flex_mfma_bwd_supported(const FlexAttnParams& p) {
  if (!flex_mfma_shape_ok(p)) return false;
  // the dK/dV kernel needs the transposed lists whenever lists are given
  const FlexTileLists& t = p.tiles_bwd;
  if (t.kv_num && (t.q_block != kBM || t.kv_block != kListBN)) return false;
  if (t.kv_num && (!t.q_num || !t.q_idx || !t.full_q_num || !t.full_q_idx)) return false;
  return true;
}

// How many workgroups share a key tile of a dK/dV kernel of which the chip holds `slots` at once: n.g over the query heads
// of the group times n.t over each head's list of query tiles.  A key tile's workgroup visits up to `visits` query tiles
// of visit_us each; under a mask the work of the tiles differs (causal: the heaviest is twice the mean), so with no more
// tiles than slots the heaviest one is the call.  dK/dV as calls of their own, merge included, undivided -> in two parts: bf16
// [1,32->8,4096,128] causal, 256 tiles on 256 slots, 598 -> 346 us; f16 [2,8,2048,256] causal 203 -> 156 us, bf16
// 262 -> 197 us.  What adding the partial sums costs: a launch, and their bytes twice (at the copy rate 27 us for twice 256
// slots at D = 128, 54 us at 256; about half of it hidden).  Taken where it promises a fifth and 30 us
// (less is lost again on the second launch where the host sets the pace: bf16 [1,4,881,64] causal 131 -> 145 us).
DkvParts flex_dkv_parts(const FlexAttnParams& p, double slots, double visit_us) {
  if (p.flags & (FLEX_UNROUNDED | FLEX_NO_SPLIT)) return {1, 1};
  const double tiles = (double)((p.Lkv + kListBN - 1) / kListBN) * p.Hkv * p.B;
  const int G = p.Hq / p.Hkv, nqt = (p.Lq + kBM - 1) / kBM;
  // what a tile's list holds is on the device: bitmaps (documents) count as a quarter full, a window without sink keys
  // by its width (bf16 [2,8,3000,64], 9 documents: in two parts 30 + 11 us against 33 us, so not split)
  double listed = nqt;
  if (p.mask.kind == FLEX_MASK_BITS) listed = fmax(1.0, 0.25 * nqt);
  else if (p.mask.hi != INT32_MAX && p.mask.sink < 0 && p.mask.lo != INT32_MIN)
    listed = fmin(nqt, fmax(0.0, (double)p.mask.hi - p.mask.lo) / kBM + 2);
  const double visits = G * listed, part_us = 2. * kListBN * 2 * p.D * sizeof(float) / 5e6;
  const bool uneven = p.tiles_bwd.kv_num || !mask_hides_nothing(p.mask);
  auto cost = [&](int parts) {
    const double rounds = ceil(tiles * parts / slots);
    const double run = uneven ? fmax(visits / parts, 0.5 * visits * tiles / slots) : visits / parts * rounds;
    return run * visit_us + (parts > 1 ? 4 + tiles * parts * part_us : 0);
  };
  DkvParts best = {1, 1};
  double least = fmin(0.8 * cost(1), cost(1) - 30);
  for (int parts = 2; parts <= 16 && parts <= visits && tiles * parts <= 2 * slots; parts++) {
    int g = parts < G ? parts : G;
    while (G % g || parts % g) g--;   // whole heads first, stretches of the lists for the rest
    if (parts / g > nqt || cost(parts) >= least) continue;
    least = cost(parts);
    best = {g, parts / g};
  }
  return best;
}
static size_t partial_bytes(const FlexAttnParams& p, int64_t parts) {
  const int64_t tiles = (int64_t)((p.Lkv + kListBN - 1) / kListBN) * p.Hkv * p.B;
  return parts < 2 ? 0 : (size_t)parts * tiles * kListBN * 2 * p.D * sizeof(float) + kPartialAlign;
}
// bytes of the partial sums of this very call, with its mask and lists
size_t flex_dkv_partial_bytes_of(const FlexAttnParams& p, double slots, double visit_us) {
  const DkvParts n = flex_dkv_parts(p, slots, visit_us);
  return partial_bytes(p, (int64_t)n.g * n.t);
}
// and for the most parts any mask and lists can get: a workspace may be sized by the shape alone
size_t flex_dkv_partial_bytes(const FlexAttnParams& p, double slots, double visit_us) {
  if (p.flags & (FLEX_UNROUNDED | FLEX_NO_SPLIT)) return 0;
  const int64_t tiles = (int64_t)((p.Lkv + kListBN - 1) / kListBN) * p.Hkv * p.B;
  const int64_t visits = (int64_t)(p.Hq / p.Hkv) * ((p.Lq + kBM - 1) / kBM);
  int64_t parts = (int64_t)(2 * slots) / tiles;
  if (parts > 16) parts = 16;
  if (parts > visits) parts = visits;
  // (a call that cannot save 30 us is never divided; even tiles take more rounds than `visits` only beyond the slots)
  if (parts < 2 || (double)visits * visit_us * fmax(1.0, ceil(tiles / slots)) <= 30) return 0;
  return partial_bytes(p, parts);
}

// two workgroups share a compute unit at D = 64, one has it at D = 128 (and 192 / 256 go to the simple kernel)
static double dkv_slots(const FlexAttnParams& p) { return flex_cu_count() * (p.D == 64 ? 2. : 1.); }
constexpr double kVisitUs = 5.;
static DkvParts dkv_parts(const FlexAttnParams& p) {
  if (p.D != 64 && p.D != 128) return {1, 1};
  return flex_dkv_parts(p, dkv_slots(p), kVisitUs);
}

// beside delta, which the caller accounts for: the partial sums of a divided dK/dV call (any_mask: of any call of the shape)
size_t flex_mfma_bwd_workspace(const FlexAttnParams& p, bool any_mask) {
  if (p.D != 64 && p.D != 128) return 0;
  return (any_mask ? flex_dkv_partial_bytes : flex_dkv_partial_bytes_of)(p, dkv_slots(p), kVisitUs);
}

int flex_mfma_bwd(const FlexAttnParams& p, const void* q, const void* k, const void* v, const void* o, const float* lse2,
                  const void* d_o, void* dq, void* dk, void* dv, void* workspace, hipStream_t s) {
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o | (uintptr_t)d_o | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) & 15) {
    flex_set_error("fused backward needs 16-byte aligned tensors");
    return 1;
  }
  const DkvParts n = dkv_parts(p);
  const BwdArgs a = {q, k, v, o, d_o, lse2, dq, dk, dv, (float*)workspace, dkv_partial_start(workspace, p), n.g, n.t, s};
  int rc;
  if (p.D >= 192 && !(p.flags & FLEX_BWD_ONLY_DQ)) {
    flex_set_error("fused backward: only the dQ kernel exists for 192- and 256-wide heads");
    return 1;
  }
  if (p.dtype == FLEX_F16)
    rc = p.D == 64 ? flex_mfma_bwd_f16_64(p, a) : p.D == 128 ? flex_mfma_bwd_f16_128(p, a) : p.D == 192 ? flex_mfma_bwd_f16_192(p, a) : flex_mfma_bwd_f16_256(p, a);
  else
    rc = p.D == 64 ? flex_mfma_bwd_bf16_64(p, a) : p.D == 128 ? flex_mfma_bwd_bf16_128(p, a) : p.D == 192 ? flex_mfma_bwd_bf16_192(p, a) : flex_mfma_bwd_bf16_256(p, a);
  if (rc == 1) flex_set_error("fused backward: unsupported score_mod kind %d", p.score.kind);
  if (rc == 2) flex_set_error("fused backward: could not raise the dynamic LDS limit");
  return rc;
}
