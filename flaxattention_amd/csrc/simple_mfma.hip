// Simple matrix-core kernels (float32 at D 64 / 128, fp16 / bf16 at D 192 / 256): checks and dispatch.  The kernels
// are in simple_mfma.cuh, instantiated per (dtype, head size) by simple_mfma_inst.hip.
#include <cmath>

#include "simple_mfma.cuh"

using namespace flex;
void flex_set_error(const char* fmt, ...);
int flex_cu_count();
DkvParts flex_dkv_parts(const FlexAttnParams& p, double slots, double visit_us);
size_t flex_dkv_partial_bytes(const FlexAttnParams& p, double slots, double visit_us);
size_t flex_dkv_partial_bytes_of(const FlexAttnParams& p, double slots, double visit_us);
int flex_simple_f32_64(const FlexAttnParams& p, const SimpleArgs& a);
int flex_simple_f32_128(const FlexAttnParams& p, const SimpleArgs& a);
int flex_simple_f16_192(const FlexAttnParams& p, const SimpleArgs& a);
int flex_simple_f16_256(const FlexAttnParams& p, const SimpleArgs& a);
int flex_simple_bf16_192(const FlexAttnParams& p, const SimpleArgs& a);
int flex_simple_bf16_256(const FlexAttnParams& p, const SimpleArgs& a);

// the (dtype, head size) pairs these kernels are instantiated for
bool flex_simple_shape(int dtype, int D, int Dv) {
  if (D != Dv) return false;
  if (dtype == FLEX_F32) return D == 64 || D == 128;
  if (dtype == FLEX_F16 || dtype == FLEX_BF16) return D == 192 || D == 256;
  return false;
}

static bool strides_ok(const int64_t* s, int epc) { return s[0] % epc == 0 && s[1] % epc == 0 && s[2] % epc == 0; }
static bool lists_ok(const FlexTileLists& t, int kv_block) {
  return !t.kv_num || (t.q_block == kSimpleQTile && t.kv_block == kv_block);
}

// which: 0 = forward, 1 = backward
bool flex_simple_supported(const FlexAttnParams& p, int which) {
  if (!flex_simple_shape(p.dtype, p.D, p.Dv)) return false;
  if (p.flags & FLEX_UNROUNDED) {
    if (p.dtype != FLEX_F32) return false;  // high / low parts are not built here; float32 rounds nothing anyway
  }
  if (p.score.kind == FLEX_SCORE_AFFINE && !p.score.mul && !p.score.add) return false;
  const int epc = p.dtype == FLEX_F32 ? 4 : 8;  // rows are read in 16-byte chunks
  if (!strides_ok(p.q_stride, epc) || !strides_ok(p.k_stride, epc) || !strides_ok(p.v_stride, epc) || !strides_ok(p.o_stride, epc))
    return false;
  if ((int64_t)((p.Lq + kSimpleQTile - 1) / kSimpleQTile) * p.Hq * p.B > 0x7fffffff) return false;
  return which == 0 ? lists_ok(p.tiles, 64) : lists_ok(p.tiles_bwd, kSimpleKvTile);
}

static int dispatch(const FlexAttnParams& p, const SimpleArgs& a) {
  int rc = 1;
  if (p.dtype == FLEX_F32) rc = p.D == 64 ? flex_simple_f32_64(p, a) : flex_simple_f32_128(p, a);
  else if (p.dtype == FLEX_F16) rc = p.D == 192 ? flex_simple_f16_192(p, a) : flex_simple_f16_256(p, a);
  else rc = p.D == 192 ? flex_simple_bf16_192(p, a) : flex_simple_bf16_256(p, a);
  if (rc) flex_set_error("simple matrix-core kernels: unsupported score_mod kind %d", p.score.kind);
  return rc;
}

// Shares of the key steps a forward call is split into (1 = none): calls whose query tiles alone would leave most
// compute units without a workgroup -- few rows against a long key sequence -- are split until there is about one
// workgroup per compute unit, with at least 16 steps of 32 keys each.
static int splits_over_keys(const FlexAttnParams& p) {
  const int64_t wgs = (int64_t)((p.Lq + kSimpleQTile - 1) / kSimpleQTile) * p.Hq * p.B;
  const int cus = flex_cu_count();
  if (wgs > cus / 2) return 1;
  const int steps = (p.Lkv + kSimpleStep - 1) / kSimpleStep;
  int s = (int)(cus / wgs);
  if (s > steps / 16) s = steps / 16;
  if (s > 64) s = 64;  // the merge kernel takes one split per lane
  return s < 2 ? 1 : s;
}
// Float32 forwards of few query tiles: 32 rows per workgroup with the key steps divided over its waves
// (simple_fwd_short_kernel) instead of 128 rows.  Four times the workgroups with a quarter of the chain, so it wins while those
// fit the chip about twice, and loses beyond, where it only reads K and V four times as often.  us, 128 rows / 32 rows,
// D = 64 and 128: 8 tiles [1,4,256] causal 27 / 17 and 43 / 19; 16 tiles [1,4,512] 48 / 19 and 80 / 31; 128 tiles [4,8,512]
// dense 48 / 35 and 82 / 63; 192 tiles [8,8,384] dense 37 / 40; 256 tiles [8,16,256] causal 28 / 32.
// More tiles than that only where they are uneven (causal, the heaviest twice the mean) and the mean chain they are cut to
// outweighs four times the workgroups: 192 tiles [8,8,384] 38 / 30 and 63 / 53, 256 tiles [4,8,1024] 92 / 73 and 157 / 133, [8,8,512]
// 49 / 46 and 82 / 81, but 240 tiles [1,80,384] 39 / 39 and 64 / 68.  A window's tiles are even: 256 tiles [1,8,4096] window
// 1000 106 / 130 and 180 / 236, four sinks and window 100 35 / 52 and 55 / 86; 192 tiles [1,12,2048] window 300 47 / 43 and
// 76 / 72, window 64 24 / 22 and 38 / 34, sinks and window 100 34 / 37 and 54 / 60.
// Against the split over workgroups above, by their chains: causal 32 tiles [1,4,1024] 52 / 33, 128 tiles [2,8,1024] 60 / 39 and
// 91 / 68; but 96 tiles [1,6,2048 against 33 keys] at D = 128 17.5 / 20.5; dense 96 tiles [1,6,2048] 97 / 115 and 163 / 221, three packed documents there 53 / 38 and 81 / 64 (as a bitmap, which
// counts as dense); window 64, 96 tiles [1,3,4096] 23 / 18 and 32 / 24, window 300 35 / 31 and 50 / 52, window 1000 65 / 70 and
// 102 / 129.
static bool short_rows(const FlexAttnParams& p) {
  if (p.dtype != FLEX_F32 || (p.flags & FLEX_NO_SPLIT)) return false;
  const int64_t wgs = (int64_t)((p.Lq + kSimpleQTile - 1) / kSimpleQTile) * p.Hq * p.B;
  const int cus = flex_cu_count(), steps = (p.Lkv + kSimpleStep - 1) / kSimpleStep, splits = splits_over_keys(p);
  const bool window = p.mask.kind == FLEX_MASK_BAND && p.mask.hi != INT32_MAX;
  const bool causal = p.mask.kind == FLEX_MASK_BAND && p.mask.lo != INT32_MIN && p.Lq > p.Lkv / 2;
  const double fill = (double)wgs / cus;
  if (causal && !window && wgs > cus / 2) return wgs <= cus && steps >= 12 && steps * (1 - 0.5 * fill) > 7.5 * fill;
  if (causal && !window && splits > 1) return 1.1 * fmax(1, 2 * fill) * steps / 4 <= (double)steps / splits;
  // even tiles, and calls of so few keys that the split above leaves them whole: the steps a 128-row tile lists (a bitmap may
  // list all of them) against the visits of a wave of 32 rows, in as many rounds as four times the workgroups take; a visit
  // costs more than a step of the tile does
  const double visit = p.D == 64 ? 1.25 : 1.4;
  double listed = steps, mine = steps;
  if (window && (splits > 1 || wgs > cus / 2)) {
    const double width = p.mask.lo == INT32_MIN ? p.Lkv : fmin(p.Lkv, (double)p.mask.hi - p.mask.lo);
    const bool sinks = p.mask.sink >= 0;
    listed = fmin(steps, (width + 128) / 32 + 1 + 2 * sinks);
    mine = fmin(steps, (width + 32) / 32 + 1 + sinks);
  }
  if (wgs > cus / 2)   // (a wave's share of a window with sinks is uneven: the sinks' step comes on top of it)
    return causal && fill <= 0.75 && p.mask.sink < 0 && ceil(4 * fill) * (ceil(mine / 4) * visit + 0.65) <= listed;
  return ceil(4 * fill) * ceil(mine / 4) * visit <= listed / splits + 0.5;
}
// any_mask: the most any mask gets (a workspace is sized by the shape alone)
int flex_simple_fwd_splits(const FlexAttnParams& p, bool any_mask) {
  if (p.flags & FLEX_NO_SPLIT) return 1;
  return !any_mask && short_rows(p) ? 1 : splits_over_keys(p);
}

// bytes of the partial (O, m, l) of a split forward
size_t flex_simple_fwd_partial_bytes(const FlexAttnParams& p, int splits) {
  if (splits <= 1) return 0;
  return ((size_t)p.B * p.Hq * p.Lq * splits * (p.D + 2) * sizeof(float) + 255) / 256 * 256;
}

// partials: nullptr for one pass over all keys, else flex_simple_fwd_partial_bytes(p, splits) bytes
int flex_simple_fwd(const FlexAttnParams& p, const void* q, const void* k, const void* v, void* o, float* lse2, int splits,
                    void* partials, hipStream_t s) {
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) & 15) {
    flex_set_error("matrix-core forward needs 16-byte aligned tensors");
    return 1;
  }
  if ((p.flags & FLEX_PARITY) && p.dtype != FLEX_F32 && !lse2) {
    flex_set_error("matrix-core forward: the parity numerics need a log-sum-exp buffer (lse2 or workspace)");
    return 1;
  }
  SimpleArgs a = {};
  a.q = q; a.k = k; a.v = v; a.out = o; a.lse2_out = lse2; a.s = s; a.bwd = false;
  a.splits = 1;
  a.short_rows = short_rows(p);
  if (splits > 1 && partials) {
    if ((uintptr_t)partials & 15) {
      flex_set_error("matrix-core forward needs a 16-byte aligned workspace");
      return 1;
    }
    a.splits = splits;
    a.o_part = (float*)partials;
    a.ml_part = a.o_part + (size_t)p.B * p.Hq * p.Lq * splits * p.D;
  }
  return dispatch(p, a);
}

// The dK/dV kernel divided over the queries as the tuned one is (flex_dkv_parts).  A visit of a 128-row query tile takes about
// 13 us at D = 192 / 256 in 16 bits and 18 / 36 us at D = 64 / 128 in float32; one workgroup per compute unit.
static double simple_visit_us(const FlexAttnParams& p) { return p.dtype != FLEX_F32 ? 13. : p.D == 64 ? 18. : 36.; }
static DkvParts simple_dkv_parts(const FlexAttnParams& p) { return flex_dkv_parts(p, flex_cu_count(), simple_visit_us(p)); }
size_t flex_simple_bwd_workspace(const FlexAttnParams& p, bool any_mask) {
  return (any_mask ? flex_dkv_partial_bytes : flex_dkv_partial_bytes_of)(p, flex_cu_count(), simple_visit_us(p));
}

int flex_simple_bwd(const FlexAttnParams& p, const void* q, const void* k, const void* v, const void* o, const float* lse2,
                    const void* d_o, void* dq, void* dk, void* dv, void* workspace, hipStream_t s) {
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o | (uintptr_t)d_o | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) & 15) {
    flex_set_error("matrix-core backward needs 16-byte aligned tensors");
    return 1;
  }
  SimpleArgs a = {};
  a.q = q; a.k = k; a.v = v; a.o = o; a.d_o = d_o; a.lse2_in = lse2;
  a.dq = dq; a.dk = dk; a.dv = dv; a.delta = (float*)workspace; a.s = s; a.bwd = true;
  a.parts = simple_dkv_parts(p);
  if (a.parts.g * a.parts.t > 1) a.dkv_partial = dkv_partial_start(workspace, p);
  return dispatch(p, a);
}
