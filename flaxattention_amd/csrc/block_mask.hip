// Block-mask builder for gfx950.
//
// Replaces the dense [B,H,Q,KV] boolean mask + reshape/sum + argsort pipeline of
// flaxattention/core/blockmask.py:277-322, 335-369, 57-64: the mask functor is
// evaluated per tile in registers, each tile is classified empty / partial /
// full, and the per-row ordered index lists are produced by a wave-level
// stable partition (selected ids ascending, then the rest ascending -- the
// order a stable descending argsort of a 0/1 row gives).  The dense mask is
// never materialised.  All outputs are integers and bit-exact.
#include <climits>

#include "flex_common.cuh"

namespace flex {

constexpr int kClassifyThreads = 256;

// Bitmaps whose classes the ordering kernel does not work out itself (tile_source).  One workgroup per tile.  flags:
// [B*H, nq, nkv] int8 for partial and full (one set where the map is the same for all (b, h)).
__global__ __launch_bounds__(kClassifyThreads) void classify_tiles_kernel(
    FlexMask mask, int H, int nq, int nkv, int qb, int kvb, int8_t* __restrict__ partial,
    int8_t* __restrict__ full) {
  const int ki = blockIdx.x, qi = blockIdx.y, bh = blockIdx.z;
  const int b = bh / H, h = bh % H;
  MaskEval visible(mask, b, h);
  const int q0 = qi * qb, kv0 = ki * kvb;
  const long long total = (long long)qb * kvb;
  unsigned long long cnt = 0;
  if (mask.kind == FLEX_MASK_BITS && (kvb % 32) == 0) {
    // word-at-a-time: every aligned 32-bit word of a row lies inside the tile
    const int words = kvb / 32;
    const long long nwords = (long long)qb * words;
    for (long long t = threadIdx.x; t < nwords; t += kClassifyThreads) {
      int r = (int)(t / words), w = (int)(t % words);
      uint32_t bits = visible.bits_bh[(int64_t)(q0 + r) * visible.stride_q + (kv0 >> 5) + w];
      cnt += __popc(bits);
    }
  } else {
    for (long long t = threadIdx.x; t < total; t += kClassifyThreads) {
      int r = (int)(t / kvb), c = (int)(t % kvb);
      cnt += visible(q0 + r, kv0 + c) ? 1u : 0u;
    }
  }
  // workgroup reduction
  for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
  __shared__ unsigned long long wsum[kClassifyThreads / 64];
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long s = 0;
    for (int w = 0; w < kClassifyThreads / 64; w++) s += wsum[w];
    size_t at = ((size_t)bh * nq + qi) * nkv + ki;
    full[at] = (s == (unsigned long long)total) ? 1 : 0;
    partial[at] = (s > 0 && s < (unsigned long long)total) ? 1 : 0;
  }
}

// What the ordering kernel selects tiles by: flags that classify_tiles_kernel left (kFlags), or, where a tile's class takes a
// few operations, the class itself, in the same launch.
//   kBand    with d = q + q_offset - kv a key is visible iff d >= lo && (d <= hi || kv <= sink): a tile is full iff its first row
//            sees its last key and its last row's gap (sink, q + q_offset - hi) misses it, and empty iff every row ends ahead
//            of the tile or has the gap over all of it
//   kClasses a bitmap that carries the classes of its 32 x 32 blocks, tiles made of a few whole blocks
// Lists of a band of 512 rows against 16384 keys in tiles of 128 x 128: classify + order 4.7 + 4.6 us, in one launch 4.6; documents
// [2,3000 x 3000] 6.2 + 2.8 -> 7.0.  bf16 [1,32->8,512 of 16384,128] forward with a fresh mask (two sets of lists): 249.4 -> 244.3.
enum { kFlags = 0, kBand = 1, kClasses = 2 };
// A lane reads a tile's block classes one after the other, twice a list (to count, to write) and for every (b, h): so only where a
// tile has at most 16 of them, and where a map that all (b, h) share is not gone through more than 16 times over.  Lists of
// documents [2,3072,3072], flags / classes: 8 blocks a tile 6.8 / 5.1 us, 16 6.5 / 5.5, 32 6.5 / 9.6, 64 6.8 / 12.1, 1024
// 33.6 / 97.4; of one shared map [2048,2048] at 128 x 128 for 16 (b, h) 6.8 / 5.6, for 64 6.8 / 8.5, for 256 7.7 / 22.6.
// A band costs a lane some thirty operations a tile, for every (b, h): above 256 of them flags are made once, a thread per tile.
// Causal lists, flags / corners: 256 (b, h) of [8192 x 8192] in 64 x 64 51.4 / 53.1 us, in 128 x 128 19.2 / 20.9, of [32768 x 32768] in
// 128 x 128 171.5 / 155, small grids 10.5 / 7.9; 512 (b, h) of [2048 x 2048] in 64 x 64 16.6 / 20.7, of [8192 x 8192] in 128 x 128
// 32.0 / 38.0, in 256 x 256 16.2 / 20.1 (flags by a workgroup a tile, as before the corners: 16.9, 33.6 and 16.6).
static int tile_source(const FlexMask& mask, int B, int H, int qb, int kvb) {
  if (mask.kind == FLEX_MASK_BAND) return (long long)B * H <= 256 ? kBand : kFlags;
  const bool shared = mask.bits_stride_b == 0 && mask.bits_stride_h == 0;
  const bool few = qb % 32 == 0 && kvb % 32 == 0 && (long long)(qb / 32) * (kvb / 32) <= 16 && (!shared || (long long)B * H <= 16);
  return mask.blk && few ? kClasses : kFlags;
}
struct TileSource {
  FlexMask mask;
  int qb, kvb, H;
  // 0 some keys visible, 1 all, 2 none
  __device__ __forceinline__ int band(int qi, int ki) const {
    const long long first = (long long)qi * qb + mask.q_offset, last = first + qb - 1;
    const long long kv0 = (long long)ki * kvb, kv_end = kv0 + kvb - 1;
    const long long below = min(last - mask.hi - 1, kv_end);   // last key of the last row's gap inside the tile
    if (first - mask.lo >= kv_end && below < max((long long)mask.sink + 1, kv0)) return 1;
    // rows ahead of `ends` see no key of the tile; from `gone` on the gap covers it (an empty band: for all rows)
    const long long ends = kv0 + mask.lo, gone = mask.hi < mask.lo ? first : kv_end + mask.hi + 1;
    return last < ends || (mask.sink < kv0 && gone <= max(first, ends)) ? 2 : 0;
  }
  __device__ __forceinline__ int classes(const int8_t* blk, int qi, int ki) const {
    const int rows = qb >> 5, cols = kvb >> 5;
    bool all = true, none = true;
    for (int r = 0; r < rows; r++)
      for (int c = 0; c < cols; c++) {
        const int x = blk[(int64_t)(qi * rows + r) * mask.blk_stride_q + ki * cols + c];
        all &= x == 1;
        none &= x == 2;
      }
    return all ? 1 : none ? 2 : 0;
  }
};

// The flags of a band that many (b, h) order: a thread per tile, one set for all of them.
__global__ __launch_bounds__(kClassifyThreads) void classify_band_kernel(TileSource src, int nq, int nkv, int8_t* __restrict__ partial,
                                                                         int8_t* __restrict__ full) {
  const long long at = (long long)blockIdx.x * kClassifyThreads + threadIdx.x;
  if (at >= (long long)nq * nkv) return;
  const int c = src.band((int)(at / nkv), (int)(at % nkv));
  partial[at] = c == 0;
  full[at] = c == 1;
}

// The four ordered lists of a block mask (partial / full, by query block / by key block) come from one
// launch: blockIdx.y names the list.
struct OrderJob {
  const int8_t* flags;
  int32_t* num;
  int32_t* idx;
  int nrows, ncols, row_stride, col_stride;
  bool by_key, full;   // which axis the rows run along, which class is listed
};
struct OrderJobs { OrderJob job[4]; };

// One wave per output row.  Selects column c in [0, ncols) of row r by flags[bh][r*row_stride + c*col_stride] or by the
// tile's class and writes num[bh][r] and idx[bh][r][0..ncols).
template <int SOURCE>
__global__ __launch_bounds__(256) void order_rows_kernel(OrderJobs jobs, TileSource src, long long mat_stride, long long n_bh) {
  const OrderJob& jb = jobs.job[blockIdx.y];
  if (!jb.num && !jb.idx) return;
  const int nrows = jb.nrows, ncols = jb.ncols;
  const int lane = threadIdx.x & 63;
  const long long row = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= n_bh * nrows) return;
  const long long bh = row / nrows;
  const int r = (int)(row % nrows);
  const int8_t* f = SOURCE == kFlags ? jb.flags + bh * mat_stride + (long long)r * jb.row_stride
                                     : src.mask.blk + (bh / src.H) * src.mask.blk_stride_b + (bh % src.H) * src.mask.blk_stride_h;
  const int col_stride = jb.col_stride;
  auto selected = [&](int c) {
    if (c >= ncols) return false;
    if constexpr (SOURCE == kFlags) {
      return f[(long long)c * col_stride] != 0;
    } else {
      const int qi = jb.by_key ? c : r, ki = jb.by_key ? r : c;
      return (SOURCE == kBand ? src.band(qi, ki) : src.classes(f, qi, ki)) == (jb.full ? 1 : 0);
    }
  };
  int count = 0;
  for (int c0 = 0; c0 < ncols; c0 += 64) count += __popcll(__ballot(selected(c0 + lane)));
  if (jb.num && lane == 0) jb.num[row] = count;
  if (!jb.idx) return;
  int32_t* out = jb.idx + row * ncols;
  int before_sel = 0, before_uns = 0;
  const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int c0 = 0; c0 < ncols; c0 += 64) {
    int c = c0 + lane;
    bool in = c < ncols;
    bool sel = selected(c);
    unsigned long long ms = __ballot(sel), mu = __ballot(in && !sel);
    if (sel) out[before_sel + __popcll(ms & lt)] = c;
    else if (in) out[count + before_uns + __popcll(mu & lt)] = c;
    before_sel += __popcll(ms);
    before_uns += __popcll(mu);
  }
}

// ---- lowering of a mask given as evaluated booleans ----
// A callable's mask arrives as one byte per position (any strides, 0 where it broadcasts) and leaves as what the
// attention kernels read: words packed along the keys, words packed along the queries, and the class of every 32 x 32
// block.  Bound by the read of the bytes: every byte is loaded once and serves all three outputs (a wave takes 32
// rows x 64 keys; a row's 64 bytes become two words through one ballot, a lane collects its own key's column and the
// columns' words give the classes).  It stands for some twenty elementwise and reduction launches per slab (two of
// them reductions over innermost extents of 8 and 32, 38 us each at 3072 x 3072): [2,1,3072,3072] with both packings
// and classes 10.4 us (18.9 MB read) against 0.42 ms of device time.
constexpr int kPackRows = 32, kPackCols = 64;

__global__ __launch_bounds__(256) void pack_mask_kernel(const uint8_t* __restrict__ mask, int64_t sb, int64_t sh, int64_t sq,
                                                        int64_t skv, int nh, int q_lo, int Qp, int KVp,
                                                        uint32_t* __restrict__ bits, uint32_t* __restrict__ bits_t,
                                                        int8_t* __restrict__ blk) {
  const int lane = threadIdx.x & 63;
  const int kv0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * kPackCols;
  if (kv0 >= KVp) return;
  const int r0 = blockIdx.y * kPackRows, map = blockIdx.z;
  const uint8_t* src = mask + (map / nh) * sb + (map % nh) * sh + (int64_t)r0 * sq + (int64_t)(kv0 + lane) * skv;
  uint8_t seen[kPackRows];
#pragma unroll
  for (int r = 0; r < kPackRows; r++) seen[r] = src[(int64_t)r * sq];
  uint32_t column = 0;           // this lane's key, bit r = row r0 + r
  unsigned long long row = 0;    // lane r: the 64 keys of row r0 + r
#pragma unroll
  for (int r = 0; r < kPackRows; r++) {
    const unsigned long long ballot = __ballot(seen[r] != 0);
    column |= (seen[r] != 0 ? 1u : 0u) << r;
    if (lane == r) row = ballot;
  }
  const int W = KVp >> 5, Wq = Qp >> 5, qb = (q_lo + r0) >> 5;
  if (lane < kPackRows)
    *(unsigned long long*)(bits + ((int64_t)map * Qp + q_lo + r0 + lane) * W + (kv0 >> 5)) = row;
  if (bits_t) bits_t[((int64_t)map * KVp + kv0 + lane) * Wq + qb] = column;
  const unsigned long long all = __ballot(column == 0xffffffffu), none = __ballot(column == 0);
  if ((lane & 31) == 0) {
    const uint32_t a = (uint32_t)(all >> lane), n = (uint32_t)(none >> lane);
    blk[((int64_t)map * Wq + qb) * W + ((kv0 + lane) >> 5)] = a == 0xffffffffu ? 1 : n == 0xffffffffu ? 2 : 0;
  }
}

// Band fit of packed maps: d = q - kv;  visible = (d >= lo) && (d <= hi || kv <= sink).  Three sweeps over the words, a
// word at a time, each sweep's minima read by the next one on the device, so that the host waits once, for the verdict
// (fitting and checking on the host's side of the stream took up to six waits):
//   fit[0] lowest d of a visible entry (INT_MAX: none)   fit[1] 1 where some map differs from the first
//   fit[2] lowest d, fit[3] lowest kv of a hidden entry with d >= lo (INT_MAX: none)
//   fit[4] / fit[5] 1 where the band with sink = fit[3] - 1 / without sink fails to reproduce the first map
__device__ __forceinline__ uint32_t bits_up_to(long long last, int kv0) {   // bits of the keys kv0 .. last
  const long long n = last - kv0 + 1;
  return n >= 32 ? 0xffffffffu : n <= 0 ? 0u : (1u << n) - 1u;
}

__device__ __forceinline__ int fit_lo(const int32_t* fit, int KVp) {
  return fit[0] <= -(KVp - 1) ? INT_MIN : fit[0];   // hides nothing ahead of the row
}

// At most kFitBlocks workgroups, each ending in one atomic (or, for a flag, plain stores of the same 1): one per wave of
// 1024 workgroups queued up on the one address and took 70 to 88 us a sweep at [2,3072,3072], against 17 us this way.
constexpr int kFitThreads = 512, kFitBlocks = 256;

__device__ __forceinline__ void block_min_to(int v, int32_t* out) {
  __shared__ int wave_min[kFitThreads / 64];
  for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
  __syncthreads();   // (an earlier use has been read)
  if ((threadIdx.x & 63) == 0) wave_min[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kFitThreads / 64; w++) v = min(v, wave_min[w]);
    if (v != INT_MAX) atomicMin(out, v);
  }
}

__global__ void fit_init_kernel(int32_t* fit) {
  const int i = threadIdx.x;
  if (i < 6) fit[i] = (i == 0 || i == 2 || i == 3) ? INT_MAX : 0;
}

__global__ __launch_bounds__(kFitThreads) void fit_visible_kernel(const uint32_t* __restrict__ bits, long long words, int W,
                                                                  long long n_maps, int32_t* fit) {
  int lo = INT_MAX;
  bool differs = false;
  for (long long i = (long long)blockIdx.x * kFitThreads + threadIdx.x; i < words; i += (long long)gridDim.x * kFitThreads) {
    const uint32_t w = bits[i];
    const int q = (int)(i / W), kv0 = (int)(i % W) * 32;
    if (w) lo = min(lo, q - (kv0 + 31 - __clz((int)w)));
    for (long long m = 1; m < n_maps; m++) differs |= bits[m * words + i] != w;
  }
  block_min_to(lo, fit);
  if (differs) fit[1] = 1;
}

// (the sweeps below have nothing to answer once the maps are known to differ)
__global__ __launch_bounds__(kFitThreads) void fit_hidden_kernel(const uint32_t* __restrict__ bits, long long words, int W, int32_t* fit) {
  if (fit[1]) return;
  const long long lo = fit_lo(fit, W * 32);
  int d_min = INT_MAX, kv_min = INT_MAX;
  for (long long i = (long long)blockIdx.x * kFitThreads + threadIdx.x; i < words; i += (long long)gridDim.x * kFitThreads) {
    const int q = (int)(i / W), kv0 = (int)(i % W) * 32;
    const uint32_t hidden = ~bits[i] & bits_up_to(q - lo, kv0);
    if (hidden) {
      d_min = min(d_min, q - (kv0 + 31 - __clz((int)hidden)));
      kv_min = min(kv_min, kv0 + __ffs((int)hidden) - 1);
    }
  }
  block_min_to(d_min, fit + 2);
  block_min_to(kv_min, fit + 3);
}

__global__ __launch_bounds__(kFitThreads) void fit_check_kernel(const uint32_t* __restrict__ bits, long long words, int W, int32_t* fit) {
  if (fit[1]) return;
  const long long lo = fit_lo(fit, W * 32);
  const bool gap = fit[2] != INT_MAX;
  const long long hi = gap ? (long long)fit[2] - 1 : INT_MAX, sink = gap ? fit[3] - 1 : -1;
  bool bad_sink = false, bad_plain = false;
  for (long long i = (long long)blockIdx.x * kFitThreads + threadIdx.x; i < words; i += (long long)gridDim.x * kFitThreads) {
    const int q = (int)(i / W), kv0 = (int)(i % W) * 32;
    const uint32_t w = bits[i], ahead = bits_up_to(q - lo, kv0), near = ~bits_up_to(q - hi - 1, kv0);
    bad_sink |= (ahead & (near | bits_up_to(sink, kv0))) != w;
    bad_plain |= (ahead & near) != w;
  }
  if (bad_sink) fit[4] = 1;
  if (bad_plain) fit[5] = 1;
}

}  // namespace flex

using namespace flex;

extern "C" size_t flexattn_block_mask_workspace_bytes(int32_t B, int32_t H, int32_t nq, int32_t nkv) {
  size_t n = (size_t)B * H * nq * nkv;
  return 2 * ((n + 255) / 256 * 256);
}
extern "C" size_t flexattn_block_mask_workspace_needed(const FlexMask* mask, int32_t B, int32_t H, int32_t nq, int32_t nkv, int32_t qb,
                                                       int32_t kvb) {
  return mask && tile_source(*mask, B, H, qb, kvb) == kFlags ? flexattn_block_mask_workspace_bytes(B, H, nq, nkv) : 0;
}

void flex_set_error(const char* fmt, ...);

extern "C" int flexattn_block_mask_build(const FlexMask* mask, int32_t B, int32_t H, int32_t nq,
                                         int32_t nkv, int32_t qb, int32_t kvb, int32_t* kv_num,
                                         int32_t* kv_idx, int32_t* full_kv_num, int32_t* full_kv_idx,
                                         int32_t* q_num, int32_t* q_idx, int32_t* full_q_num,
                                         int32_t* full_q_idx, void* workspace,
                                         flexattn_stream_t stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (!mask || !workspace) { flex_set_error("block_mask_build: null mask or workspace"); return 1; }
  if (B <= 0 || H <= 0 || nq <= 0 || nkv <= 0 || qb <= 0 || kvb <= 0) {
    flex_set_error("block_mask_build: non-positive size B=%d H=%d nq=%d nkv=%d qb=%d kvb=%d", B, H, nq, nkv, qb, kvb);
    return 1;
  }
  if ((long long)B * H > 65535 || nq > 65535) {
    flex_set_error("block_mask_build: grid too large (B*H=%lld, nq=%d; limit 65535)", (long long)B * H, nq);
    return 1;
  }
  if (mask->kind == FLEX_MASK_BITS && !mask->bits) { flex_set_error("block_mask_build: bitmap mask without bits"); return 1; }
  if (mask->kind != FLEX_MASK_BITS && mask->kind != FLEX_MASK_BAND) { flex_set_error("block_mask_build: unknown mask kind %d", mask->kind); return 1; }
  size_t n = (size_t)B * H * nq * nkv;
  int8_t* partial = (int8_t*)workspace;
  int8_t* full = partial + (n + 255) / 256 * 256;
  const int source = tile_source(*mask, B, H, qb, kvb);
  // (a band, or a bitmap broadcast over batch and head, does not look at (b, h): its tiles are classified once and every
  // (b, h) orders the same flags)
  const bool uniform = mask->kind == FLEX_MASK_BAND || (mask->bits_stride_b == 0 && mask->bits_stride_h == 0);
  const TileSource src = {*mask, qb, kvb, H};
  if (source == kFlags && mask->kind == FLEX_MASK_BAND)
    hipLaunchKernelGGL(classify_band_kernel, dim3((unsigned)(((long long)nq * nkv + kClassifyThreads - 1) / kClassifyThreads)),
                       dim3(kClassifyThreads), 0, stream, src, nq, nkv, partial, full);
  else if (source == kFlags)
    hipLaunchKernelGGL(classify_tiles_kernel, dim3(nkv, nq, uniform ? 1 : B * H), dim3(kClassifyThreads), 0, stream, *mask, H, nq,
                       nkv, qb, kvb, partial, full);
  const long long mat = uniform ? 0 : (long long)nq * nkv;
  OrderJobs jobs;
  auto job = [&](int at, const int8_t* flags, bool transposed, int32_t* num, int32_t* idx) {
    OrderJob& j = jobs.job[at];
    j.flags = flags; j.num = num; j.idx = idx;
    j.nrows = transposed ? nkv : nq; j.ncols = transposed ? nq : nkv;
    j.row_stride = transposed ? 1 : nkv; j.col_stride = transposed ? nkv : 1;
    j.by_key = transposed; j.full = flags == full;
  };
  job(0, partial, false, kv_num, kv_idx);
  job(1, full, false, full_kv_num, full_kv_idx);
  job(2, partial, true, q_num, q_idx);
  job(3, full, true, full_q_num, full_q_idx);
  const bool by_kv = kv_num || kv_idx || full_kv_num || full_kv_idx, by_q = q_num || q_idx || full_q_num || full_q_idx;
  if (by_kv || by_q) {
    const int waves = 4;
    const long long most_rows = (long long)B * H * (by_q ? (by_kv ? (nq > nkv ? nq : nkv) : nkv) : nq);
    const dim3 grid((unsigned)((most_rows + waves - 1) / waves), 4);
    if (source == kBand) hipLaunchKernelGGL(order_rows_kernel<kBand>, grid, dim3(64 * waves), 0, stream, jobs, src, mat, (long long)B * H);
    else if (source == kClasses) hipLaunchKernelGGL(order_rows_kernel<kClasses>, grid, dim3(64 * waves), 0, stream, jobs, src, mat, (long long)B * H);
    else hipLaunchKernelGGL(order_rows_kernel<kFlags>, grid, dim3(64 * waves), 0, stream, jobs, src, mat, (long long)B * H);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { flex_set_error("block_mask_build: launch failed: %s", hipGetErrorString(e)); return 2; }
  return 0;
}

extern "C" int flexattn_pack_mask(const uint8_t* mask, const int64_t* strides, int32_t nb, int32_t nh, int32_t q_lo,
                                  int32_t rows, int32_t Qp, int32_t KVp, int32_t* bits, int32_t* bits_t, int8_t* blk,
                                  flexattn_stream_t stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (!mask || !strides || !bits || !blk) { flex_set_error("pack_mask: null argument"); return 1; }
  if (nb <= 0 || nh <= 0 || rows <= 0 || q_lo < 0 || Qp <= 0 || KVp <= 0 || Qp % 128 || KVp % 128 || q_lo % 32 || rows % 32 ||
      (long long)q_lo + rows > Qp) {
    flex_set_error("pack_mask: bad extents nb=%d nh=%d q_lo=%d rows=%d Qp=%d KVp=%d", nb, nh, q_lo, rows, Qp, KVp);
    return 1;
  }
  const int most_rows = 65535 * kPackRows;   // blockIdx.y
  if ((long long)nb * nh > 65535 || rows > most_rows) {
    flex_set_error("pack_mask: grid too large (nb*nh=%lld, rows=%d)", (long long)nb * nh, rows);
    return 1;
  }
  const int cols = 4 * kPackCols;
  hipLaunchKernelGGL(pack_mask_kernel, dim3((KVp + cols - 1) / cols, rows / kPackRows, nb * nh), dim3(256), 0, stream, mask,
                     strides[0], strides[1], strides[2], strides[3], nh, q_lo, Qp, KVp, (uint32_t*)bits, (uint32_t*)bits_t, blk);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { flex_set_error("pack_mask: launch failed: %s", hipGetErrorString(e)); return 2; }
  return 0;
}

extern "C" int flexattn_bitmap_fit(const int32_t* bits, int32_t n_maps, int32_t Qp, int32_t KVp, int32_t* fit,
                                   flexattn_stream_t stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (!bits || !fit) { flex_set_error("bitmap_fit: null argument"); return 1; }
  if (n_maps <= 0 || Qp <= 0 || KVp <= 0 || KVp % 32) {
    flex_set_error("bitmap_fit: bad extents n_maps=%d Qp=%d KVp=%d", n_maps, Qp, KVp);
    return 1;
  }
  const int W = KVp / 32;
  const long long words = (long long)Qp * W;
  const long long want = (words + kFitThreads - 1) / kFitThreads;
  const unsigned blocks = (unsigned)(want < kFitBlocks ? want : kFitBlocks);
  const uint32_t* w = (const uint32_t*)bits;
  hipLaunchKernelGGL(fit_init_kernel, dim3(1), dim3(64), 0, stream, fit);
  hipLaunchKernelGGL(fit_visible_kernel, dim3(blocks), dim3(kFitThreads), 0, stream, w, words, W, (long long)n_maps, fit);
  hipLaunchKernelGGL(fit_hidden_kernel, dim3(blocks), dim3(kFitThreads), 0, stream, w, words, W, fit);
  hipLaunchKernelGGL(fit_check_kernel, dim3(blocks), dim3(kFitThreads), 0, stream, w, words, W, fit);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { flex_set_error("bitmap_fit: launch failed: %s", hipGetErrorString(e)); return 2; }
  return 0;
}
