// gs_sort.hip — global binning: one key per (Gaussian, covered tile),
// ordered by (tile, depth, Gaussian id), the total order the reference's
// per-tile bitonic sort produces (shaders.js:418-500, tie-break :454).
//
// Three strategies, identical output: tile segments (the default, below the
// radix passes in this file), and two radix strategies:
//  * depth-then-tile (also the fallback for views above kMaxSegTiles tiles):
//    stable LSD radix sort of the n Gaussians by
//    depth bits (emitted in id order, so ties keep id order), then keys are
//    emitted in that order and stably sorted by tile id only
//    (ceil(tileBits/8) passes). Sorting Gaussians instead of keys moves the
//    32 depth bits off the long key array. The first depth pass drops the
//    culled Gaussians (key 0xffffffff, which would sort last and emit no
//    keys) and counts the rest on the device, so the later passes, the count
//    and the emission run over the visible Gaussians only.
//  * global64: keys (tile << 32 | depth bits) emitted in id order and sorted
//    by a stable LSD radix sort over all 32 + tileBits bits.
//
// Every radix pass (8-bit digit) is reduce-then-scan, with no inter-block
// waiting, over a fixed grid of G blocks, each owning a contiguous chunk
// processed in rounds of 2048 keys (8 per thread, wave-striped so every
// load is coalesced):
//   hist    per-wave digit counts in LDS; each wave groups its 64 keys by
//           digit with 8 ballots, and one lane per group adds the group size;
//           the block's 256 counts go to a digit-major table hist[d][block]
//   scan    one block per digit: exclusive scan of the digit's row (a
//           contiguous row) and the digit total
//   scatter digit bases from an in-block scan of the 256 totals;
//           wave-local stable ranks from the same ballot groups, one
//           block-wide digit prefix per round, keys staged in LDS in
//           (digit, position) order, then written out in digit runs by
//           consecutive threads
// Key counts that only exist on the device (the emitted key total) are read
// from device memory by every kernel; the grids are fixed. No pass uses
// global atomics.
#include "gs_kernels.h"
#include "gs_bands.h"

namespace gs {

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

__device__ __forceinline__ uint64_t lanemask_lt() {
  return (1ull << lane_id()) - 1ull;
}

// mask of active lanes whose 8-bit digit equals this lane's
__device__ __forceinline__ uint64_t match_digit8(uint32_t d, uint64_t active) {
  uint64_t m = active;
#pragma unroll
  for (int b = 0; b < 8; b++) {
    const bool bit = (d >> b) & 1u;
    const uint64_t bal = wave_ballot(bit);
    m &= bit ? bal : ~bal;
  }
  return m;
}

constexpr int kItems = 8;
constexpr int kRound = kBlock * kItems;   // keys per block round

// block b's contiguous chunk [lo, hi) of N elements split over G blocks,
// rounded to `align` elements
__device__ __forceinline__ void chunk_range(uint32_t N, int G, uint32_t align, uint32_t& lo, uint32_t& hi) {
  const uint32_t per = (uint32_t)(((uint64_t)N + G - 1) / G);
  const uint32_t chunk = (per + align - 1u) / align * align;
  const uint64_t l = (uint64_t)blockIdx.x * chunk;
  lo = (uint32_t)(l < N ? l : N);
  const uint64_t h = (uint64_t)lo + chunk;
  hi = (uint32_t)(h < N ? h : N);
}

__global__ void k_fill_u32(uint32_t* p, int64_t count, uint32_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) p[i] = v;
}

template <typename KeyT>
__device__ __forceinline__ uint32_t digit_of(KeyT k, int shift) {
  return (uint32_t)(k >> shift) & 0xffu;
}

// kFilter: keys equal to ~0 (culled Gaussians) are left out
template <typename KeyT, bool kFilter>
__global__ __launch_bounds__(kBlock) void k_radix_hist(const KeyT* __restrict__ keys,
                                                       const uint32_t* __restrict__ dN, int shift,
                                                       int G, uint32_t* __restrict__ hist) {
  __shared__ uint32_t wc[4][256];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  wc[0][tid] = wc[1][tid] = wc[2][tid] = wc[3][tid] = 0;
  __syncthreads();
  uint32_t lo, hi;
  chunk_range(*dN, G, kRound, lo, hi);
  for (uint32_t r = lo; r < hi; r += kRound) {
    const uint32_t base = r + (uint32_t)w * 64u * kItems;
    uint32_t d[kItems];
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const uint32_t idx = base + (uint32_t)i * 64u + lane;
      d[i] = 0x100u;
      if (idx < hi) {
        const KeyT k = keys[idx];
        if (!kFilter || k != (KeyT)~(KeyT)0) d[i] = digit_of(k, shift);
      }
    }
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const bool ok = d[i] < 0x100u;
      const uint64_t act = wave_ballot(ok);
      if (!kFilter && act == 0ull) break;   // unfiltered, only the chunk's tail is empty
      if (act == 0ull) continue;
      const uint64_t m = match_digit8(d[i] & 0xffu, act);
      // one lane per digit group: distinct addresses within an instruction
      if (ok && (m & lanemask_lt()) == 0ull) atomicAdd(&wc[w][d[i]], (uint32_t)__popcll(m));
    }
  }
  __syncthreads();
  hist[(int64_t)tid * G + blockIdx.x] = wc[0][tid] + wc[1][tid] + wc[2][tid] + wc[3][tid];
}

// one block per digit: exclusive scan of hist[d][0..G) in place, and the
// digit's total into totals[d] (the scatter adds the digit bases)
__global__ __launch_bounds__(kBlock) void k_radix_scan(uint32_t* __restrict__ hist, int G,
                                                       uint32_t* __restrict__ totals) {
  __shared__ uint32_t wsum[kBlock / 64];
  const int d = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  uint32_t carry = 0u;
  uint32_t* row = hist + (int64_t)d * G;
  for (int b0 = 0; b0 < G; b0 += kBlock) {
    const int b = b0 + tid;
    const uint32_t v = b < G ? row[b] : 0u;
    const uint32_t x = wave_incl_scan(v);
    __syncthreads();
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    uint32_t wpre = 0;
    for (int k = 0; k < w; k++) wpre += wsum[k];
    if (b < G) row[b] = carry + wpre + x - v;
    carry += wsum[0] + wsum[1] + wsum[2] + wsum[3];
  }
  if (tid == 0) totals[d] = carry;
}

// kFilter: keys equal to ~0 are dropped, and block 0 stores the number of
// keys kept in *nOut
template <typename KeyT, bool kWriteKeys, bool kFilter>
__global__ __launch_bounds__(kBlock) void k_radix_scatter(const KeyT* __restrict__ keysIn,
                                                          const uint32_t* __restrict__ valsIn,
                                                          const uint32_t* __restrict__ dN,
                                                          int shift, int G,
                                                          const uint32_t* __restrict__ scan,
                                                          KeyT* __restrict__ keysOut,
                                                          uint32_t* __restrict__ valsOut,
                                                          const uint32_t* __restrict__ totals,
                                                          uint32_t* __restrict__ nOut) {
  __shared__ uint32_t wc[4][256];
  __shared__ uint32_t wpre[4][256];
  __shared__ uint32_t gbase[256];
  __shared__ uint32_t lstart[256];
  __shared__ uint32_t wsum[4];
  __shared__ KeyT sk[kRound];
  __shared__ uint32_t sv[kRound];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  uint32_t lo, hi;
  chunk_range(*dN, G, kRound, lo, hi);
  {
    // digit bases: exclusive scan of the digit totals
    const uint32_t t = totals[tid];
    const uint32_t x = wave_incl_scan(t);
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    uint32_t wp = 0;
    for (int k = 0; k < w; k++) wp += wsum[k];
    gbase[tid] = wp + x - t + scan[(int64_t)tid * G + blockIdx.x];
    if (kFilter && blockIdx.x == 0 && tid == 0) *nOut = wsum[0] + wsum[1] + wsum[2] + wsum[3];
  }
  wc[0][tid] = wc[1][tid] = wc[2][tid] = wc[3][tid] = 0;
  __syncthreads();
  for (uint32_t r = lo; r < hi; r += kRound) {
    // 1. load, then rank within the wave (stable: item-major, then lane)
    const uint32_t base = r + (uint32_t)w * 64u * kItems;
    KeyT key[kItems];
    uint32_t val[kItems], rank[kItems];
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const uint32_t idx = base + (uint32_t)i * 64u + lane;
      bool ok = idx < hi;
      key[i] = ok ? keysIn[idx] : (KeyT)0;
      if (kFilter) ok = ok && key[i] != (KeyT)~(KeyT)0;
      val[i] = ok ? (valsIn ? valsIn[idx] : idx) : 0u;
      rank[i] = ok ? 0u : 0xffffffffu;
    }
    // ranks: all groups' counter updates are issued back to back (the LDS
    // applies one wave's operations in order), then each lane fetches its
    // group leader's pre-add count
    uint64_t mm[kItems];
    uint32_t old[kItems];
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const bool ok = rank[i] == 0u;
      mm[i] = match_digit8(digit_of(key[i], shift), wave_ballot(ok)) ;
      old[i] = 0u;
      if (ok && (mm[i] & lanemask_lt()) == 0ull)
        old[i] = atomicAdd(&wc[w][digit_of(key[i], shift)], (uint32_t)__popcll(mm[i]));
    }
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const bool ok = rank[i] == 0u;
      const int leader = mm[i] ? (int)__builtin_ctzll(mm[i]) : 0;
      const uint32_t b = (uint32_t)__shfl((int)old[i], leader);
      if (ok) rank[i] = b + (uint32_t)__popcll(mm[i] & lanemask_lt());
    }
    __syncthreads();
    // 2. per digit: wave prefixes, round total, local start (block scan)
    const uint32_t c0 = wc[0][tid], c1 = wc[1][tid], c2 = wc[2][tid], c3 = wc[3][tid];
    const uint32_t tot = c0 + c1 + c2 + c3;
    wpre[0][tid] = 0u;
    wpre[1][tid] = c0;
    wpre[2][tid] = c0 + c1;
    wpre[3][tid] = c0 + c1 + c2;
    wc[0][tid] = wc[1][tid] = wc[2][tid] = wc[3][tid] = 0;
    const uint32_t x = wave_incl_scan(tot);
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    uint32_t wp = 0;
    for (int k = 0; k < w; k++) wp += wsum[k];
    const uint32_t myStart = wp + x - tot;
    lstart[tid] = myStart;
    const uint32_t kept = wsum[0] + wsum[1] + wsum[2] + wsum[3];   // keys of this round staged below
    __syncthreads();
    // 3. stage in local (digit, rank) order
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      if (rank[i] != 0xffffffffu) {
        const uint32_t d = digit_of(key[i], shift);
        const uint32_t p = lstart[d] + wpre[w][d] + rank[i];
        sk[p] = key[i];
        sv[p] = val[i];
      }
    }
    __syncthreads();
    // 4. write out: consecutive threads write consecutive slots of a digit run
    for (uint32_t j = tid; j < kept; j += kBlock) {
      const KeyT k = sk[j];
      const uint32_t d = digit_of(k, shift);
      const uint32_t g = gbase[d] + (j - lstart[d]);
      if (kWriteKeys) keysOut[g] = k;
      valsOut[g] = sv[j];
    }
    __syncthreads();
    gbase[tid] += tot;
  }
}

// ---- emission offsets: exclusive scan of cnt[] in sorted order ----

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t& total, uint32_t* wsum) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint32_t x = wave_incl_scan(v);
  __syncthreads();
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  uint32_t pre = 0;
  for (int k = 0; k < w; k++) pre += wsum[k];
  total = wsum[0] + wsum[1] + wsum[2] + wsum[3];
  return pre + x - v;
}

// One block per 256 Gaussians in (depth) order `order` (nullptr: id
// order): gathers each one's key count and tile rectangle once, stores them
// in sort order for the emission pass, and writes the block's key total and
// visible count.
__global__ __launch_bounds__(kBlock) void k_count_partials(const uint32_t* __restrict__ order,
                                                           const uint32_t* __restrict__ cnt,
                                                           const uint2* __restrict__ rect,
                                                           const uint32_t* __restrict__ depthKey,
                                                           const uint32_t* __restrict__ dN,
                                                           uint32_t* __restrict__ cntS,
                                                           uint2* __restrict__ rectS,
                                                           uint32_t* __restrict__ dkS,
                                                           uint64_t* __restrict__ partials,
                                                           uint32_t* __restrict__ vpartials) {
  __shared__ uint32_t wsum[4];
  __shared__ uint32_t wvis[4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint32_t N = *dN;
  const uint32_t r = blockIdx.x * kBlock + tid;
  uint32_t c = 0;
  if (r < N) {
    const uint32_t id = order ? order[r] : r;
    c = cnt[id];
    cntS[r] = c;
    rectS[r] = c ? rect[id] : make_uint2(0, 0);
    if (dkS) dkS[r] = c ? depthKey[id] : 0u;
  }
  uint32_t acc = c, vis = c != 0u;
  for (int o = 32; o > 0; o >>= 1) {
    acc += __shfl_xor(acc, o);
    vis += __shfl_xor(vis, o);
  }
  if (lane == 0) { wsum[w] = acc; wvis[w] = vis; }
  __syncthreads();
  if (tid == 0) {
    partials[blockIdx.x] = (uint64_t)wsum[0] + wsum[1] + wsum[2] + wsum[3];
    vpartials[blockIdx.x] = wvis[0] + wvis[1] + wvis[2] + wvis[3];
  }
}

// single block: exclusive scan of the G partials; numKeys = min(total, cap)
__global__ __launch_bounds__(1024) void k_count_top(uint64_t* __restrict__ partials,
                                                    const uint32_t* __restrict__ vpartials, int G,
                                                    uint64_t cap, uint32_t* __restrict__ numKeys,
                                                    uint64_t* __restrict__ totalKeys,
                                                    uint32_t* __restrict__ numVisible,
                                                    double* __restrict__ stats) {
  __shared__ uint64_t wsum[16];
  __shared__ uint32_t wvis[16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int per = (G + 1023) / 1024;
  uint64_t mine = 0;
  uint32_t vis = 0;
  for (int k = 0; k < per; k++) {
    const int b = tid * per + k;
    if (b < G) { mine += partials[b]; vis += vpartials[b]; }
  }
  for (int o = 32; o > 0; o >>= 1) vis += __shfl_xor(vis, o);
  if (lane == 0) wvis[w] = vis;
  const uint64_t x = wave_incl_scan(mine);
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  uint64_t pre = 0;
  for (int k = 0; k < w; k++) pre += wsum[k];
  uint64_t run = pre + x - mine;
  for (int k = 0; k < per; k++) {
    const int b = tid * per + k;
    if (b < G) {
      const uint64_t v = partials[b];
      partials[b] = run;
      run += v;
    }
  }
  if (tid == 0) {
    uint32_t v = 0;
    for (int k = 0; k < 16; k++) v += wvis[k];
    *numVisible = v;
  }
  if (tid == 1023) {
    const uint64_t total = pre + x;
    *totalKeys = total;
    *numKeys = (uint32_t)(total < cap ? total : cap);
    if (total > cap) stats[kStatDropped] += (double)(total - cap);
  }
}

// Emits one key per covered tile, cooperatively: for every round of 256
// Gaussians (in sort order) the block scans their key counts, then each
// thread produces the keys at consecutive output positions, finding its
// Gaussian by binary search over the round's offsets in LDS. Writes are
// coalesced and the work per thread is balanced whatever the splat sizes.
// kGlobal64: Gaussians in id order, key = (tile << 32) | depth bits.
// Otherwise Gaussians in depth order, key = tile. Keys past the budget `cap`
// are dropped (counted by k_count_top).

// Cover-test constants of Gaussian i's raster record (gs_project.hip): the
// conic and mean from its first float4, C and the cover level L from its
// second (L in the high half of w as an fp16 upper bound when the record
// holds 16-bit colours).
__device__ __forceinline__ gs_cover_splat record_cover(const float4* __restrict__ rec, int recFmt, size_t i) {
  const size_t rs = (size_t)rec_stride(recFmt);
  const float4 g0 = rec[rs * i + 0];
  const float4 g1 = rec[rs * i + 1];
  const float L = recFmt == 0 ? g1.z : gs_h2f(__float_as_uint(g1.w) >> 16);
  return gs_cover_prepare(g0.x, g0.y, g0.z, g0.w, g1.x, L);
}

template <bool kGlobal64>
__global__ __launch_bounds__(kBlock) void k_emit(const uint32_t* __restrict__ order,
                                                 const uint32_t* __restrict__ cntS,
                                                 const uint2* __restrict__ rectS,
                                                 const uint32_t* __restrict__ dkS,
                                                 const uint32_t* __restrict__ dN,
                                                 const uint64_t* __restrict__ partials, int tilesX, int tileSize,
                                                 uint64_t cap, const float4* __restrict__ rec, int recFmt,
                                                 void* __restrict__ keysOut,
                                                 uint32_t* __restrict__ valsOut) {
  __shared__ uint32_t wsum[4];
  __shared__ uint32_t sOff[kBlock];
  __shared__ uint2 sRect[kBlock];
  __shared__ uint32_t sId[kBlock];
  __shared__ uint32_t sDk[kBlock];
  __shared__ gs_cover_splat sG[kBlock];
  const int tid = threadIdx.x;
  const uint32_t N = *dN;
  const uint32_t r = blockIdx.x * kBlock + tid;
  const bool ok = r < N;
  const uint32_t c = ok ? cntS[r] : 0u;
  uint32_t tot;
  const uint32_t ex = block_excl_scan(c, tot, wsum);
  sOff[tid] = ex;
  sRect[tid] = ok ? rectS[r] : make_uint2(0, 0);
  const uint32_t gidr = ok ? (kGlobal64 ? r : order[r]) : 0u;
  sId[tid] = gidr;
  if (kGlobal64) sDk[tid] = ok ? dkS[r] : 0u;
  if (c != 0u) sG[tid] = record_cover(rec, recFmt, gidr);
  __syncthreads();
  const uint64_t run = partials[blockIdx.x];
  for (uint32_t q = tid; q < tot; q += kBlock) {
    int g = 0;
#pragma unroll
    for (int step = kBlock / 2; step > 0; step >>= 1)
      if (sOff[g + step] <= q) g += step;
    const uint64_t pos = run + q;
    if (pos < cap) {
      const uint2 rc = sRect[g];
      const uint32_t tx0 = rc.x & 0xffffu, tx1 = rc.x >> 16, ty0 = rc.y & 0xffffu;
      const uint32_t wdt = tx1 - tx0 + 1u;
      const uint32_t li = q - sOff[g];
      const uint32_t dy = li / wdt;
      const uint32_t tx = tx0 + (li - dy * wdt), ty = ty0 + dy;
      const uint32_t tile = ty * (uint32_t)tilesX + tx;
      if (kGlobal64) ((uint64_t*)keysOut)[pos] = ((uint64_t)tile << 32) | sDk[g];
      else ((uint32_t*)keysOut)[pos] = tile;
      const gs_cover_splat sg = sG[g];
      const uint32_t mask = gs_cover_tile_mask(&sg, (int)tx, (int)ty, tileSize);
      valsOut[pos] = sId[g] | (mask << kMaskShift);
    }
  }
}

// Tile ranges from the sorted keys: ranges[t] = (first key, one past the
// last). A tile with no keys gets (o, o), o = number of keys of lower tiles,
// as the reference's exclusive scan gives it (shaders.js:366-371); the
// threads at key boundaries fill the empty tiles in between, and the thread
// holding the last key fills the tiles after it.
template <typename KeyT>
__global__ void k_tile_ranges(const KeyT* __restrict__ keys, const uint32_t* __restrict__ dN,
                              int shift, int numTiles, uint2* __restrict__ ranges) {
  const uint32_t N = *dN;
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < N; k += gridDim.x * blockDim.x) {
    const uint32_t t = (uint32_t)(keys[k] >> shift);
    const uint32_t tp = k == 0 ? 0xffffffffu : (uint32_t)(keys[k - 1] >> shift);
    if (tp != t) {
      ranges[t].x = k;
      for (uint32_t e = tp + 1u; e < t; e++) ranges[e] = make_uint2(k, k);  // tp + 1 wraps to 0 for k = 0
    }
    if (k == N - 1) {
      ranges[t].y = N;
      for (uint32_t e = t + 1u; e < (uint32_t)numTiles; e++) ranges[e] = make_uint2(N, N);
    } else if ((uint32_t)(keys[k + 1] >> shift) != t) {
      ranges[t].y = k + 1;
    }
  }
}

// Raster launch order: tiles by descending key count (a 256-bucket
// pseudo-logarithmic counting sort; order within a bucket is arbitrary).
// Launching the heaviest tiles first keeps the last partial wave of
// workgroups short. The order changes no result: tiles are independent and
// the fixed-point gradient sums are integer.
__device__ __forceinline__ uint32_t tile_bucket(uint2 r) {
  const uint32_t c = r.y - r.x;
  if (c < 16u) return c;
  const int e = 31 - (int)__builtin_clz(c);
  return min(255u, (uint32_t)(e - 3) * 16u + ((c >> (e - 4)) & 15u));
}

__global__ __launch_bounds__(1024) void k_tile_order(const uint2* __restrict__ ranges, int numTiles,
                                                     uint32_t* __restrict__ order) {
  __shared__ uint32_t cnt[256];
  const int tid = threadIdx.x;
  if (tid < 256) cnt[tid] = 0u;
  __syncthreads();
  for (int t = tid; t < numTiles; t += 1024) atomicAdd(&cnt[tile_bucket(ranges[t])], 1u);
  __syncthreads();
  if (tid == 0) {   // exclusive offsets, highest bucket first
    uint32_t run = 0;
    for (int b = 255; b >= 0; b--) {
      const uint32_t c = cnt[b];
      cnt[b] = run;
      run += c;
    }
  }
  __syncthreads();
  for (int t = tid; t < numTiles; t += 1024) order[atomicAdd(&cnt[tile_bucket(ranges[t])], 1u)] = (uint32_t)t;
}

// ---- host launchers ----

void launch_fill_u32(hipStream_t st, uint32_t* p, int64_t count, uint32_t v) {
  if (count <= 0) return;
  k_fill_u32<<<(unsigned)((count + 255) / 256), 256, 0, st>>>(p, count, v);
}

// ---- tile segments (default strategy) ----
//
// The reference's own structure (shaders.js:318-500): per-tile key counts, a
// scan that lays out one segment per tile under the entry budget, a scatter
// of every (Gaussian, tile) key into its tile's segment, and a sort of each
// segment. Keys are u64 (depth bits << 32 | id << 4 | block mask): within a
// tile no two keys share an id, so sorting by the whole word orders a
// segment by (depth, id), the reference's order (shaders.js:454), whatever
// order the scatter left it in.
//
// No global atomics: blocks of Gaussians (up to 256, of equal cost) count
// their keys per tile in an LDS histogram and write it as one row of a
// [block][tile] table; a column scan turns the table into each block's offset
// inside every tile's segment (and the tile totals); the scatter then places
// keys with LDS counters only, dense views in bands of tile rows. A segment
// of up to 1024 keys sorts in one block: 256-key runs by single waves (bitonic
// through lane exchanges), then up to two LDS merge levels; longer segments
// are split into buckets that sort that way.

constexpr int kSegThreads = 1024;     // threads of the count and scatter blocks
// per-tile LDS arrays (histogram, counters, scan input) are sized to the
// view's tile count at launch, so that small views fit more blocks per CU
extern __shared__ __align__(16) uint32_t seg_dyn[];
constexpr uint32_t kShSort = 2048;    // shaders.js:33 SHARED_SORT: longer segments count pow2-padded
constexpr int kScanChunk = 64;        // tiles per scan thread (shaders.js:325)

__device__ __forceinline__ uint64_t seg_key(uint32_t depth, uint32_t id, uint32_t mask) {
  return ((uint64_t)depth << 32) | ((uint64_t)id << 4) | (uint64_t)mask;
}
__device__ __forceinline__ uint32_t seg_val(uint64_t k) {
  return (uint32_t)((k >> 4) & kIdMask) | ((uint32_t)(k & 0xfu) << kMaskShift);
}

// the binning job of this block: the single view's (by value), or view v
// of the batched array
template <bool kJobs>
__device__ __forceinline__ SegJob seg_job(const SegJob& arg, const SegJob* __restrict__ jobs, int v) {
  if constexpr (kJobs) return global_job(jobs[v]);
  else return arg;
}

// exclusive scan over a block of kT threads (kT / 64 waves)
template <int kT>
__device__ __forceinline__ uint32_t block_excl_scan_t(uint32_t v, uint32_t& total, uint32_t* wsum) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint32_t x = wave_incl_scan(v);
  __syncthreads();
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  uint32_t pre = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < kT / 64; k++) {
    const uint32_t ws = wsum[k];
    pre += k < w ? ws : 0u;
    tot += ws;
  }
  total = tot;
  return pre + x - v;
}

// Gaussians [lo, hi) of a segment block, one round of kSegThreads at a time,
// for one band of bandRows tile rows after the other (one band: all rows).
// Per round the Gaussians with keys are packed to the front of the LDS
// arrays, their keys are spread over the threads, and f(g, tile, tx, ty) runs
// once per key, g the packed index. A wave's 64 keys find their Gaussians
// from one 64-bit word that marks where a Gaussian's keys start and from the
// owner of the word's first key: a popcount each, where a table of every
// key's owner took a store per key and a round of more keys than the table a
// ten-step search per key. The words cover kSegWindow keys at a time. The
// tile comes from an f32 reciprocal of the rectangle's width (an integer
// division costs more than the cover test's line). With both, the count pass
// of 92.6M keys (1920x1080, 1M Gaussians) took 259 -> 102 us, of 8 views of
// 2.9M keys 161 -> 128. `prep` stages per-Gaussian data: prep.load issues its
// global reads, prep.store puts them in LDS.
//
// The loads are pipelined one round ahead (a block holds only 16 waves per
// CU, too few to hide a load's latency otherwise): the next round's counts
// and rectangles are issued at the start of a round, its per-Gaussian data
// before this round's keys, and the first round's before `init` (the
// block's per-tile setup).
constexpr uint32_t kSegWords = kSegThreads;          // one per thread to clear
constexpr uint32_t kSegWindow = 64u * kSegWords;

struct SegBands {
  int tilesY, rows;  // rows >= tilesY: one band, whatever the view's rows
};

struct SegRound {
  uint4* rc;         // kSegThreads: tx0 | width << 16, ty0, first key, 1 / width (f32 bits)
  uint64_t* starts;  // kSegWords: bit k of word w: a Gaussian's first key is 64 w + k
  uint32_t* owner;   // kSegWords: packed index of the Gaussian that key 64 w belongs to
  uint2* wsum;       // kSegThreads / 64: keys, Gaussians with keys
};

template <typename Prep, typename Init, typename F>
__device__ __forceinline__ void seg_rounds(int64_t lo, int64_t hi, const uint32_t* __restrict__ cnt,
                                           const uint2* __restrict__ rect, int tilesX, SegBands bands, const SegRound& sr,
                                           const Prep& prep, Init init, F f) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  uint32_t* starts32 = (uint32_t*)sr.starts;
  int64_t i = lo + tid;
  uint32_t c = i < hi ? cnt[i] : 0u;
  uint2 rc = i < hi ? rect[i] : make_uint2(0, 0);   // read whatever c is: no dependent load
  typename Prep::State ps = prep.load(i, c);
  init();
  if (lo >= hi) return;
  for (int band = 0; band < bands.tilesY; band += bands.rows) {
    for (int64_t r0 = lo; r0 < hi; r0 += kSegThreads) {
      const bool wrap = r0 + kSegThreads >= hi;
      const int64_t in = !wrap ? i + kSegThreads : (band + bands.rows < bands.tilesY ? lo + tid : hi);
      const uint32_t cn = in < hi ? cnt[in] : 0u;
      const uint2 rn = in < hi ? rect[in] : make_uint2(0, 0);
      const uint32_t tx0 = rc.x & 0xffffu, wdt = (rc.x >> 16) - tx0 + 1u;
      uint32_t ty0 = rc.y & 0xffffu;
      if (bands.rows < bands.tilesY && c) {   // the rows of this band
        const uint32_t ty1 = min(rc.y >> 16, (uint32_t)(band + bands.rows - 1));
        ty0 = max(ty0, (uint32_t)band);
        c = ty1 >= ty0 ? (ty1 - ty0 + 1u) * wdt : 0u;
      }
      const uint32_t x = wave_incl_scan(c);
      const uint64_t has = wave_ballot(c != 0u);
      __syncthreads();   // the previous round's reads are done
      if (lane == 63) sr.wsum[w] = make_uint2(x, (uint32_t)__popcll(has));
      sr.starts[tid] = 0ull;
      __syncthreads();
      uint32_t ex = x - c, ci = __builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0u));
      uint32_t tot = 0;
#pragma unroll
      for (int k = 0; k < kSegThreads / 64; k++) {
        const uint2 ws = sr.wsum[k];
        ex += k < w ? ws.x : 0u;
        ci += k < w ? ws.y : 0u;
        tot += ws.x;
      }
      if (c) sr.rc[ci] = make_uint4(tx0 | (wdt << 16), ty0, ex, __float_as_uint(__builtin_amdgcn_rcpf((float)wdt)));
      prep.store(ci, i, c, ps);
      for (uint32_t w0 = 0; w0 == 0u || w0 < tot; w0 += kSegWindow) {
        const uint32_t w1 = tot - w0 < kSegWindow ? tot : w0 + kSegWindow;
        if (w0) {
          __syncthreads();
          sr.starts[tid] = 0ull;
          __syncthreads();
        }
        if (c && ex < w1 && ex + c > w0) {
          if (ex >= w0) atomicOr(&starts32[(ex - w0) >> 5], 1u << ((ex - w0) & 31u));
          const uint32_t a = ex > w0 ? ex - w0 : 0u, e = (ex + c < w1 ? ex + c : w1) - w0;
          for (uint32_t k = (a + 63u) >> 6; 64u * k < e; k++) sr.owner[k] = ci;
        }
        __syncthreads();
        if (w0 == 0u) ps = prep.load(in, cn);
        for (uint32_t q = w0 + tid; q < w1; q += kSegThreads) {
          const uint32_t word = (uint32_t)__builtin_amdgcn_readfirstlane((int)((q - w0) >> 6));
          const uint64_t m = sr.starts[word] >> 1;   // keys 64 word + 1 .. of lane l's key: bits below l
          const uint32_t g = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((uint32_t)m, sr.owner[word]));
          const uint4 r = sr.rc[g];
          const uint32_t li = q - r.z, wd = r.x >> 16;
          // li / wd for li < 2^14 (a splat covers at most kMaxSegTiles tiles):
          // (li + 1/2) / wd is at least 1 / (2 wd) from a whole number, the
          // product's error, two ulp, below 2^-8 / wd
          const uint32_t dy = (uint32_t)(((float)li + 0.5f) * __uint_as_float(r.w));
          const uint32_t tx = (r.x & 0xffffu) + (li - __umul24(dy, wd)), ty = r.y + dy;
          f(g, __umul24(ty, (uint32_t)tilesX) + tx, tx, ty);
        }
      }
      i = in;
      c = cn;
      rc = rn;
    }
  }
  __syncthreads();
}

// count pass: no per-Gaussian data beyond the count; tallies the Gaussians
// with keys
struct CountPrep {
  uint32_t* vis;
  struct State {};
  __device__ State load(int64_t, uint32_t) const { return {}; }
  __device__ void store(uint32_t, int64_t, uint32_t c, const State&) const { *vis += c != 0u; }
};

// Row b of the [block][tile] table: the keys of Gaussians [b G, (b+1) G) per
// tile; visPart[b]: how many of them have keys.
// This block's Gaussians: the chunks of kSegChunk Gaussians whose cost
// prefix p (over the chunks before them) satisfies b K <= p nb < (b + 1) K,
// K the total, so each of the nb blocks takes about K / nb of the cost. A
// chunk costs its keys plus one per Gaussian: a round of Gaussians costs
// its loads, scan and barriers even when they have no keys, so key shares
// alone would hand a block a long run of off-view Gaussians. The first
// block starts at 0 and the last ends at n, and block b's end is block
// b + 1's start by the same formula: the blocks partition [0, n) whatever
// the chunk sums hold (they only set the balance). Returns [lo, hi).
// Logical index of this count/scatter block. Workgroups are dispatched
// round-robin over MI355X's 8 XCDs, so logical blocks 0..nb/8-1 run on the
// first XCD, the next nb/8 on the second, and so on: each tile segment's
// runs from neighbouring logical blocks (adjacent in memory) are written
// from one XCD. Measured ~0.5-1% faster than the identity order at the same
// state. Any bijection partitions the work the same way.
__device__ __forceinline__ int seg_logical_block(int nb) {
  const int i = (int)blockIdx.x;
  return nb % 8 == 0 ? (i % 8) * (nb / 8) + i / 8 : i;
}

__device__ __forceinline__ int2 seg_block_chunks(int64_t n, const uint32_t* __restrict__ chunkKeys, int nb,
                                                 uint64_t* ws64, uint32_t (*wsc)[kSegThreads / 64]) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t nChunks = (n + kSegChunk - 1) / kSegChunk;
  const int64_t m = (nChunks + kSegThreads - 1) / kSegThreads;   // chunks per thread, in order
  const int64_t c0 = (int64_t)tid * m, c1 = c0 + m < nChunks ? c0 + m : nChunks;
  uint64_t part = 0;
  for (int64_t c = c0; c < c1; c++) part += chunkKeys[c] + (uint64_t)kSegChunk;
  const uint64_t x = wave_incl_scan(part);
  if (lane == 63) ws64[w] = x;
  __syncthreads();
  uint64_t pre = 0, total = 0;
  for (int k = 0; k < kSegThreads / 64; k++) {
    const uint64_t v = ws64[k];
    if (k < w) pre += v;
    total += v;
  }
  pre += x - part;
  const uint64_t b = (uint64_t)seg_logical_block(nb);
  const uint64_t tLo = b * total, tHi = (b + 1) * total;
  uint32_t nLo = 0, nHi = 0;          // chunks with prefix * nb below each bound
  for (int64_t c = c0; c < c1; c++) {
    const uint64_t pn = pre * (uint64_t)nb;
    nLo += pn < tLo;
    nHi += pn < tHi;
    pre += chunkKeys[c] + (uint64_t)kSegChunk;
  }
  for (int o = 32; o > 0; o >>= 1) {
    nLo += (uint32_t)__shfl_xor((int)nLo, o);
    nHi += (uint32_t)__shfl_xor((int)nHi, o);
  }
  if (lane == 0) { wsc[0][w] = nLo; wsc[1][w] = nHi; }
  __syncthreads();
  uint32_t sLo = 0, sHi = 0;
  for (int k = 0; k < kSegThreads / 64; k++) { sLo += wsc[0][k]; sHi += wsc[1][k]; }
  __syncthreads();   // ws64 and wsc are free again
  const int64_t lo = (int64_t)sLo * kSegChunk;
  const int64_t hi = b == (uint64_t)(nb - 1) ? n : (int64_t)sHi * kSegChunk;
  return make_int2((int)(lo < n ? lo : n), (int)(hi < n ? hi : n));
}

template <bool kJobs>
__global__ __launch_bounds__(kSegThreads) void k_seg_count(SegJob arg, const SegJob* __restrict__ jobs) {
  const SegJob j = seg_job<kJobs>(arg, jobs, blockIdx.y);
  if (kJobs && j.skip) return;
  const int64_t n = j.n;
  const int nb = j.nb, tilesX = j.tilesX, numTiles = j.numTiles;
  const uint32_t* __restrict__ cnt = j.cnt;
  const uint2* __restrict__ rect = j.rect;
  const uint32_t* __restrict__ chunkKeys = j.chunkKeys;
  uint32_t* __restrict__ blockStart = j.blockStart;
  uint32_t* __restrict__ table = j.table;
  uint32_t* __restrict__ visPart = j.visPart;
  uint32_t* hist = seg_dyn;   // numTiles
  __shared__ uint4 sRc[kSegThreads];
  __shared__ uint64_t starts[kSegWords];
  __shared__ uint32_t owner[kSegWords];
  __shared__ uint2 wsum[kSegThreads / 64];
  __shared__ uint64_t ws64[kSegThreads / 64];
  __shared__ uint32_t wsc[2][kSegThreads / 64];
  const int tid = threadIdx.x;
  const int2 r = seg_block_chunks(n, chunkKeys, nb, ws64, wsc);
  const int lb = seg_logical_block(nb);
  const int64_t lo = r.x, hi = r.y;
  if (tid == 0) {
    blockStart[lb] = (uint32_t)lo;
    if (lb == nb - 1) blockStart[nb] = (uint32_t)hi;
  }
  uint32_t vis = 0;
  const SegRound sr{sRc, starts, owner, wsum};
  seg_rounds(lo, hi, cnt, rect, tilesX, {1, 1}, sr, CountPrep{&vis},
             [&]() { for (int t = tid; t < numTiles; t += kSegThreads) hist[t] = 0u; },
             [&](uint32_t, uint32_t tile, uint32_t, uint32_t) { atomicAdd(&hist[tile], 1u); });
  uint32_t tot;
  block_excl_scan_t<kSegThreads>(vis, tot, wsc[0]);
  if (tid == 0) visPart[lb] = tot;
  __syncthreads();
  uint32_t* row = table + (int64_t)lb * numTiles;
  for (int t = tid; t < numTiles; t += kSegThreads) row[t] = hist[t];
}

// Column scan of the table: table[b][t] becomes the exclusive prefix over
// blocks, tileCnt[t] the column total. Blocks of 256 threads handle 16
// tiles, 16 threads per tile (a wave reads 16 consecutive tiles of 4 rows),
// each thread a sixteenth of the rows.
template <bool kJobs>
__global__ __launch_bounds__(kBlock) void k_seg_colscan(SegJob arg, const SegJob* __restrict__ jobs) {
  const SegJob j = seg_job<kJobs>(arg, jobs, blockIdx.y);
  if (kJobs && j.skip) return;
  uint32_t* __restrict__ table = j.table;
  const int nb = j.nb, numTiles = j.numTiles;
  uint32_t* __restrict__ tileCnt = j.tileCnt;
  __shared__ uint32_t part[16][16];
  const int tl = threadIdx.x & 15, q = threadIdx.x >> 4;
  const int t = blockIdx.x * 16 + tl;
  const int per = (nb + 15) / 16;
  const int b0 = q * per, b1 = b0 + per < nb ? b0 + per : nb;
  // a thread's rows stay in registers: one batch of independent loads
  constexpr int kRegRows = (int)(kSegBlocks / 16);
  static_assert(kSegBlocks % 16 == 0, "sixteenths of the rows");
  uint32_t v[kRegRows];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < kRegRows; k++) {
    const int b = b0 + k;
    v[k] = (t < numTiles && b < b1) ? table[(int64_t)b * numTiles + t] : 0u;
    sum += v[k];
  }
  part[q][tl] = sum;
  __syncthreads();
  if (t >= numTiles) return;
  uint32_t run = 0;
  for (int k = 0; k < q; k++) run += part[k][tl];
#pragma unroll
  for (int k = 0; k < kRegRows; k++) {
    const int b = b0 + k;
    if (b < b1) {
      table[(int64_t)b * numTiles + t] = run;
      run += v[k];
    }
  }
  if (q == 15) tileCnt[t] = run;
}

__device__ __forceinline__ uint32_t seg_padded(uint32_t c) {
  // shaders.js:329-332: segments over SHARED_SORT take a power-of-two slot
  return c <= kShSort ? c : 1u << (32 - __clz((int)(c - 1u)));
}

// Single block of 1024 threads: the reference's budgeted segment scan
// (shaders.js:321-370), the raster launch order and the visible count.
//
// The reference's thread li owns the chunk of tiles [64 li, 64 li + 64). The
// chunk starts at the unbudgeted exclusive prefix of the padded sizes of
// the chunks before it; within the chunk, a tile whose padded size would
// take the running total past the budget is dropped (and counted, as the
// reference counts it, even when empty). Here 64 / kPer threads share a
// chunk, kPer tiles each, held in registers: a chunk whose unbudgeted end
// stays within the budget drops nothing, so each of its threads starts at its
// unbudgeted prefix; a chunk that may overflow is walked in order by its
// first thread, which leaves each tile's kept count in LDS. Kept tiles get
// compact, unpadded segments: ranges[t] = (start, start + count). Then the
// tiles are ordered by descending key count for the raster launch (as
// k_tile_order).
//
// Nothing else runs beside this block, so its latency is what it costs: kPer
// is the least power of two that covers the view (1 up to 1024 tiles, 16 at
// kMaxSegTiles), the scans stay on the VALU, and a tile's place in its bucket
// comes with the count: 6.9 -> 3.5 us at 64x64, 7.5 -> 4.6 at 320x240, 13.0
// -> 10.2 at 1600x900 against 16 tiles per thread read through LDS.
constexpr int kScanThreads = 1024;

template <bool kJobs, int kPer>
__global__ __launch_bounds__(kScanThreads) void k_seg_scan(SegJob arg, const SegJob* __restrict__ jobs) {
  const SegJob j = seg_job<kJobs>(arg, jobs, blockIdx.y);
  if (kJobs && j.skip) return;
  const uint32_t* __restrict__ tileCnt = j.tileCnt;
  const int numTiles = j.numTiles, nb = j.nb;
  const uint64_t cap = j.cap;
  uint2* __restrict__ ranges = j.ranges;
  uint32_t* __restrict__ order = j.tileOrder;
  uint32_t* __restrict__ chunkKeys = j.chunkKeys;
  constexpr int kWaves = kScanThreads / 64;
  constexpr int kShare = kScanChunk / kPer;   // threads per chunk
  uint32_t* sc = seg_dyn;                     // numTiles: kept counts of overflowing chunks
  __shared__ uint64_t wsA[kWaves];
  __shared__ uint64_t wsB[kWaves];
  __shared__ uint64_t wsK[kWaves];
  __shared__ uint2 wsC[kWaves];
  __shared__ uint32_t bucket[256];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int t0 = tid * kPer;
  uint32_t c[kPer];
#pragma unroll
  for (int k = 0; k < kPer; k++) c[k] = t0 + k < numTiles ? tileCnt[t0 + k] : 0u;
  const uint32_t vis = tid < nb ? j.visPart[tid] : 0u;   // nb <= kSegBlocks
  // the count pass has read the chunk key sums: clear them for the next
  // projection to fill
  const int64_t nChunks = (j.n + kSegChunk - 1) / kSegChunk;
  for (int64_t k = tid; k < nChunks; k += kScanThreads) chunkKeys[k] = 0u;
  if (tid < 256) bucket[tid] = 0u;
  uint64_t pad = 0, raw = 0;
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    pad += c[k] ? seg_padded(c[k]) : 0u;
    raw += c[k];
  }
  // unbudgeted exclusive prefix (tile order), the chunk's start and end
  const uint64_t x = wave_incl_scan(pad);
  if (lane == 63) wsA[w] = x;
  __syncthreads();
  uint64_t acc0 = x - pad;                            // this thread's unbudgeted start
#pragma unroll
  for (int k = 0; k < kWaves; k++) {
    const uint64_t s = wsA[k];
    acc0 += k < w ? s : 0u;
  }
  const uint64_t q0 = __shfl(acc0, lane & ~(kShare - 1));           // the chunk's start
  const uint64_t qend = __shfl(acc0 + pad, lane | (kShare - 1));    // the chunk's unbudgeted end
  // an overflowing chunk: its first thread walks its 64 tiles in order and
  // leaves their kept counts (0 = dropped)
  const bool over = qend > cap;
  uint32_t dropped = 0;
  if (over && (tid & (kShare - 1)) == 0) {
    uint64_t acc = q0;
    for (int k = 0; k < kScanChunk; k++) {
      const int t = t0 + k;
      if (t >= numTiles) break;
      const uint32_t n = tileCnt[t];
      uint64_t p = n ? seg_padded(n) : 0u;
      if (acc + p > cap) { p = 0; dropped++; }
      acc += p;
      sc[t] = p ? n : 0u;
    }
  }
  __syncthreads();
  if (over) {
#pragma unroll
    for (int k = 0; k < kPer; k++) c[k] = t0 + k < numTiles ? sc[t0 + k] : 0u;
  }
  uint64_t kept = 0;
#pragma unroll
  for (int k = 0; k < kPer; k++) kept += c[k];
  // compact starts
  const uint64_t y = wave_incl_scan(kept);
  const uint64_t rsum = wave_incl_scan(raw);
  const uint32_t dsum = wave_incl_scan(dropped), vsum = wave_incl_scan(vis);
  if (lane == 63) {
    wsK[w] = y;
    wsB[w] = rsum;
    wsC[w] = make_uint2(dsum, vsum);
  }
  __syncthreads();
  uint64_t start = y - kept;
#pragma unroll
  for (int k = 0; k < kWaves; k++) {
    const uint64_t s = wsK[k];
    start += k < w ? s : 0u;
  }
  uint32_t place[kPer];   // tiles counted into the same bucket before this one
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const uint2 rg = make_uint2((uint32_t)start, (uint32_t)(start + c[k]));
    if (t0 + k < numTiles) {
      ranges[t0 + k] = rg;
      place[k] = atomicAdd(&bucket[tile_bucket(rg)], 1u);
    }
    start += c[k];
  }
  if (tid == kScanThreads - 1) *j.numKeys = (uint32_t)start;
  if (tid == 0) {
    uint64_t r = 0;
    uint32_t d = 0, v = 0;
#pragma unroll
    for (int k = 0; k < kWaves; k++) { r += wsB[k]; d += wsC[k].x; v += wsC[k].y; }
    *j.totalKeys = r;
    if (d) atomicAdd(&j.stats[kStatDropped], (double)d);   // the views' scans run together
    *j.numVisible = v;
  }
  __syncthreads();
  // exclusive bucket offsets, heaviest bucket first: the first wave scans
  // four buckets per lane
  if (w == 0) {
    uint32_t n[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      n[k] = bucket[255 - 4 * lane - k];
      sum += n[k];
    }
    uint32_t run = wave_incl_scan(sum) - sum;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      bucket[255 - 4 * lane - k] = run;
      run += n[k];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPer; k++)
    if (t0 + k < numTiles) order[bucket[tile_bucket(make_uint2(0u, c[k]))] + place[k]] = (uint32_t)(t0 + k);
}

// scatter pass: key (without mask) and cover-test constants of each Gaussian
// with keys. A conic that is not positive definite takes every block: its
// cover level is stored as infinity, which no exponent exceeds.
struct ScatterPrep {
  const uint32_t* __restrict__ depthKey;
  const float4* __restrict__ rec;
  int recFmt;
  uint64_t* sKey;
  float4* sG0;   // mx, my, A/2, B
  float4* sG1;   // C/2, L, -B/A, -B/C
  struct State {
    uint32_t dk;
    float4 g0, g1;
  };
  __device__ State load(int64_t i, uint32_t c) const {
    State s{0u, make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
    if (c != 0u) {
      const int64_t rs = rec_stride(recFmt);
      s.dk = depthKey[i];
      s.g0 = rec[rs * i + 0];
      s.g1 = rec[rs * i + 1];
    }
    return s;
  }
  __device__ void store(uint32_t k, int64_t i, uint32_t c, const State& s) const {
    if (c != 0u) {
      const float L = recFmt == 0 ? s.g1.z : gs_h2f(__float_as_uint(s.g1.w) >> 16);
      const gs_cover_splat g = gs_cover_prepare(s.g0.x, s.g0.y, s.g0.z, s.g0.w, s.g1.x, L);
      sKey[k] = seg_key(s.dk, (uint32_t)i, 0u);
      sG0[k] = make_float4(g.mx, g.my, g.hA, g.B);
      sG1[k] = make_float4(g.hC, g.pd ? g.L : __builtin_inff(), g.kA, g.kC);
    }
  }
};

// the scatter's bands of tile rows (gs_bands.h)
__device__ __forceinline__ SegBands seg_bands(const SegJob& j) {
  const int rows = gs_band_rows(*j.totalKeys, j.n, j.nb, j.tilesX, j.numTiles);
  return rows ? SegBands{j.numTiles / j.tilesX, rows} : SegBands{1, 1};
}

// Every (Gaussian, kept tile) key into its tile's segment: each tile's LDS
// counter starts at the tile's segment start plus this block's offset in
// the tile (the column scan), so a key's slot is one LDS atomic; the tile's
// block mask (gs_cover.h) rides in the low 4 bits.
template <bool kJobs>
__global__ __launch_bounds__(kSegThreads) void k_seg_scatter(SegJob arg, const SegJob* __restrict__ jobs) {
  const SegJob j = seg_job<kJobs>(arg, jobs, blockIdx.y);
  if (kJobs && j.skip) return;
  const uint32_t* __restrict__ blockStart = j.blockStart;
  const uint32_t* __restrict__ cnt = j.cnt;
  const uint2* __restrict__ rect = j.rect;
  const uint32_t* __restrict__ depthKey = j.depthKey;
  const float4* __restrict__ rec = j.rec;
  const int recFmt = j.recFmt, tilesX = j.tilesX, tileSize = j.tile, numTiles = j.numTiles;
  const uint32_t* __restrict__ table = j.table;
  const uint2* __restrict__ ranges = j.ranges;
  uint64_t* __restrict__ keys = j.keys;
  uint32_t* cur = seg_dyn;                            // numTiles: next slot of each tile
  uint8_t* dropped = (uint8_t*)(seg_dyn + numTiles);  // numTiles: tile dropped by the budget
  __shared__ uint4 sRc[kSegThreads];
  __shared__ uint64_t starts[kSegWords];
  __shared__ uint32_t owner[kSegWords];
  __shared__ uint2 wsum[kSegThreads / 64];
  __shared__ uint64_t sKey[kSegThreads];
  __shared__ float4 sG0[kSegThreads];
  __shared__ float4 sG1[kSegThreads];
  const int tid = threadIdx.x;
  const SegBands bands = seg_bands(j);
  const int lb = seg_logical_block(j.nb);
  const uint32_t* row = table + (int64_t)lb * numTiles;
  const int64_t lo = blockStart[lb], hi = blockStart[lb + 1];   // the count pass's blocks
  const SegRound sr{sRc, starts, owner, wsum};
  seg_rounds(lo, hi, cnt, rect, tilesX, bands, sr, ScatterPrep{depthKey, rec, recFmt, sKey, sG0, sG1},
             [&]() {
#pragma unroll 4
               for (int t = tid; t < numTiles; t += kSegThreads) {
                 const uint2 rg = ranges[t];
                 cur[t] = rg.x + row[t];
                 dropped[t] = rg.y == rg.x;
               }
             },
             [&](uint32_t g, uint32_t tile, uint32_t tx, uint32_t ty) {
               const uint32_t pos = atomicAdd(&cur[tile], 1u);
               if (dropped[tile]) return;   // tile dropped by the budget (shaders.js:406-407)
               const float4 a = sG0[g], b = sG1[g];
               const gs_cover_splat sg{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, 1};
               const uint32_t mask = gs_cover_tile_mask(&sg, (int)tx, (int)ty, tileSize);
               keys[pos] = sKey[g] | mask;
             });
}

// x from lane ^ m, for 64-bit x: m = 1, 2 as DPP quad permutes on the VALU; 4,
// 8 and 16 as LDS swizzles, which need no address; 32 as a ds_bpermute (flip:
// its byte address, 4 (lane ^ 32), computed once)
template <int kM>
__device__ __forceinline__ uint64_t lane_xor_u64(uint64_t x, int flip) {
  const int lo = (int)(uint32_t)x, hi = (int)(uint32_t)(x >> 32);
  int a, b;
  if constexpr (kM == 1) {
    a = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xf, 0xf, false);   // quad_perm [1,0,3,2]
    b = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xf, 0xf, false);
  } else if constexpr (kM == 2) {
    a = __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xf, 0xf, false);   // quad_perm [2,3,0,1]
    b = __builtin_amdgcn_mov_dpp(hi, 0x4E, 0xf, 0xf, false);
  } else if constexpr (kM == 32) {
    a = __builtin_amdgcn_ds_bpermute(flip, lo);
    b = __builtin_amdgcn_ds_bpermute(flip, hi);
  } else {
    a = __builtin_amdgcn_ds_swizzle(lo, (kM << 10) | 0x1f);   // bit mode: lane' = (lane & 0x1f) ^ kM
    b = __builtin_amdgcn_ds_swizzle(hi, (kM << 10) | 0x1f);
  }
  return ((uint64_t)(uint32_t)b << 32) | (uint32_t)a;
}

// One compare-exchange stage (k, j) of the bitonic network over 256 keys,
// element i = 4 lane + r in v[r]: partners at distance j < 4 are in the same
// lane (one compare orders both), others in lane ^ (j / 4).
template <uint32_t k, uint32_t j>
__device__ __forceinline__ void bitonic_stage(uint64_t (&v)[4], uint32_t lane, int flip) {
  if constexpr (j < 4) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      if (r & (int)j) continue;
      const bool ascending = ((4u * lane + (uint32_t)r) & k) == 0u;
      const uint64_t a = v[r], b = v[r | (int)j];
      const bool keep = (a < b) == ascending;
      v[r] = keep ? a : b;
      v[r | (int)j] = keep ? b : a;
    }
  } else {
    uint64_t o[4];
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = lane_xor_u64<(int)(j / 4)>(v[r], flip);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t i = 4u * lane + (uint32_t)r;
      const bool keepMin = ((i & j) == 0u) == ((i & k) == 0u);
      const bool lt = v[r] < o[r];
      v[r] = keepMin == lt ? v[r] : o[r];
    }
  }
}

template <uint32_t k, uint32_t j>
__device__ __forceinline__ void bitonic_merge_steps(uint64_t (&v)[4], uint32_t lane, int flip) {
  bitonic_stage<k, j>(v, lane, flip);
  if constexpr (j > 1) bitonic_merge_steps<k, j / 2>(v, lane, flip);
}

template <uint32_t k>
__device__ __forceinline__ void bitonic_blocks(uint64_t (&v)[4], uint32_t lane, int flip) {
  bitonic_merge_steps<k, k / 2>(v, lane, flip);
  if constexpr (k < 256) bitonic_blocks<k * 2>(v, lane, flip);
}

// Ascending bitonic sort of 256 keys within one wave, keys 4 lane .. 4 lane
// + 3 in v[0..3]: no LDS traffic except the exchanges at lane distances of
// 4 and more, no barriers. Bound by the compares and selects; the exchanges
// are written out because __shfl_xor computes its ds_bpermute address anew
// for each of them (1M Gaussians: sort 31.5 -> 28.1 us, 8 views 245 -> 214).
__device__ __forceinline__ void wave_sort256(uint64_t (&v)[4]) {
  bitonic_blocks<2>(v, __lane_id(), (int)((__lane_id() ^ 32u) << 2));
}

// Sorts m <= kChunk keys: R = ceil(m / 256) runs of 256 sorted by waves
// (the last padded with ~0), then merged pairwise in LDS (merge path, P
// outputs per thread per level; with three runs the last pair of the first
// level has no partner and is copied). Returns the LDS buffer holding the
// sorted keys (sorted[0, m)).
constexpr uint32_t kChunk = 4 * 256;

__device__ __forceinline__ uint64_t* seg_sort_chunk(const uint64_t* __restrict__ src, uint32_t m, uint64_t* sa, uint64_t* sb) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
  // runs of 256 keys: as many as m needs (a segment of 513-768 keys sorts
  // three runs, not four padded ones)
  const uint32_t R = (m + 255u) / 256u;
  // src is device memory: read through a global pointer
  const __attribute__((address_space(1))) uint64_t* gsrc = (const __attribute__((address_space(1))) uint64_t*)src;
  if (w < R) {
    uint64_t v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t i = 256u * w + 4u * lane + (uint32_t)r;
      v[r] = i < m ? gsrc[i] : ~0ull;
    }
    wave_sort256(v);
#pragma unroll
    for (int r = 0; r < 4; r++) sa[256u * w + 4u * lane + (uint32_t)r] = v[r];
  }
  __syncthreads();
  uint64_t* in = sa;
  uint64_t* out = sb;
  const uint32_t N = 256u * R;
  // outputs per thread: a power of two, so a thread's outputs never straddle
  // two merged pairs (2W >= 512); with three runs 192 threads write 4 each
  const uint32_t P = R == 3u ? 4u : R;
  for (uint32_t W = 256u; W < N; W <<= 1) {
    // thread tid writes outputs [tid P, tid P + P) of N; the pair at base
    // merges A = [base, base + na) and B = [base + na, base + na + nb), the
    // last pair possibly shorter (nb = 0: A is copied)
    const uint32_t o = tid * P;
    if (o < N) {
      const uint32_t base = o / (2u * W) * (2u * W);
      const uint32_t na = N - base < W ? N - base : W;
      const uint32_t nb = N - base - na < W ? N - base - na : W;
      const uint64_t* A = in + base;
      const uint64_t* B = A + na;
      const uint32_t d = o - base;
      uint32_t lo = d > nb ? d - nb : 0u, hi = d < na ? d : na;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (A[mid] < B[d - mid - 1u]) lo = mid + 1u;
        else hi = mid;
      }
      uint32_t ia = lo, ib = d - lo;
      for (uint32_t q = 0; q < P; q++) {
        const bool takeA = ib >= nb || (ia < na && A[ia] < B[ib]);
        out[o + q] = takeA ? A[ia++] : B[ib++];
      }
    }
    __syncthreads();
    uint64_t* t = in;
    in = out;
    out = t;
  }
  return in;
}

// out[0, na + nb) = merge of the sorted runs A and B (keys are distinct):
// each thread finds where its 8 outputs start by a merge-path search.
__device__ void seg_merge(const uint64_t* A, uint32_t na, const uint64_t* B, uint32_t nb, uint64_t* out) {
  const uint32_t N = na + nb;
  for (uint32_t o = threadIdx.x * 8u; o < N; o += kBlock * 8u) {
    uint32_t lo = o > nb ? o - nb : 0u, hi = o < na ? o : na;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (A[mid] < B[o - mid - 1u]) lo = mid + 1u;
      else hi = mid;
    }
    uint32_t ia = lo, ib = o - lo;
    const uint32_t e = o + 8u < N ? o + 8u : N;
    for (uint32_t q = o; q < e; q++) {
      const bool takeA = ib >= nb || (ia < na && A[ia] < B[ib]);
      out[q] = takeA ? A[ia++] : B[ib++];
    }
  }
}

// Sorts src[0, len) of more than kChunk keys by kChunk-key runs merged
// pairwise in global memory (src <-> other, both overwritten) and writes the
// raster values to vals.
__device__ __forceinline__ void seg_sort_merge(uint64_t* src, uint64_t* other, uint32_t len,
                                               uint32_t* __restrict__ vals, uint64_t* sa, uint64_t* sb) {
  const uint32_t tid = threadIdx.x;
  for (uint32_t c0 = 0; c0 < len; c0 += kChunk) {
    const uint32_t m = len - c0 < kChunk ? len - c0 : kChunk;
    const uint64_t* sorted = seg_sort_chunk(src + c0, m, sa, sb);
    for (uint32_t i = tid; i < m; i += kBlock) src[c0 + i] = sorted[i];
    __syncthreads();
  }
  uint64_t* dst = other;
  for (uint32_t wdt = kChunk; wdt < len; wdt <<= 1) {
    for (uint32_t a = 0; a < len; a += 2u * wdt) {
      const uint32_t na = len - a < wdt ? len - a : wdt;
      const uint32_t nb = len - a - na < wdt ? len - a - na : wdt;
      seg_merge(src + a, na, src + a + na, nb, dst + a);
    }
    __syncthreads();
    uint64_t* t = src;
    src = dst;
    dst = t;
  }
  for (uint32_t i = tid; i < len; i += kBlock) vals[i] = seg_val(src[i]);
  __syncthreads();
}

// Sorts a segment of more than kChunk keys (a tile under large splats holds
// thousands): a sample of the keys gives splitters, one pass counts the keys
// of each bucket between them, a second one moves the keys into their buckets
// (keys -> tmp), and each bucket, kBucketKeys on average, is sorted in LDS.
// Every key is read three times and written once however long the segment
// is, where pairwise merging of 1024-key runs reads and writes all of them
// once more per doubling, with a dependent search in global memory per eight
// keys. A bucket that came out larger than kChunk is merged that way.
// The splitters are whole keys (depth, id), so equal depths split too.
// A 1920x1080 view of 1M Gaussians with most keys in such tiles: 7596 us with
// the merges alone, 1261 with the buckets; already at 1025 keys (three
// buckets) two scans and three short sorts cost less than one global merge.
constexpr uint32_t kBucketKeys = 512;
constexpr uint32_t kMaxBuckets = 128;
constexpr uint32_t kSamplesPerBucket = 8;   // kMaxBuckets * 8 = kChunk samples at most

struct SegBuckets {
  uint64_t split[kMaxBuckets];   // bucket b: split[b - 1] <= key < split[b]
  uint32_t at[kMaxBuckets + 1];  // counts, then the buckets' next slots
};

// buckets' index of a key: the number of splitters at or below it (kMaxBuckets
// a power of two; unused splitters are ~0, above every key)
__device__ __forceinline__ uint32_t seg_bucket(const SegBuckets& sk, uint32_t top, uint64_t key) {
  uint32_t b = 0;
  for (uint32_t step = top; step > 0u; step >>= 1)
    if (sk.split[b + step - 1u] <= key) b += step;
  return b;
}

__device__ __forceinline__ void seg_sort_buckets(uint64_t* keys, uint64_t* tmp, uint32_t len,
                                                 uint32_t* __restrict__ vals, uint64_t* sa, uint64_t* sb,
                                                 SegBuckets& sk) {
  const uint32_t tid = threadIdx.x;
  uint32_t nb = (len + kBucketKeys - 1u) / kBucketKeys;
  nb = nb < kMaxBuckets ? nb : kMaxBuckets;
  // sorted samples in LDS (staged through tmp, which is free until the buckets move there)
  const uint32_t S = kSamplesPerBucket * nb;
  for (uint32_t i = tid; i < S; i += kBlock) tmp[i] = keys[(uint32_t)((uint64_t)i * len / S)];
  __syncthreads();
  const uint64_t* sorted = seg_sort_chunk(tmp, S, sa, sb);
  for (uint32_t i = tid; i < kMaxBuckets; i += kBlock) {
    sk.split[i] = i + 1u < nb ? sorted[(i + 1u) * kSamplesPerBucket] : ~0ull;
    sk.at[i] = 0u;
  }
  __syncthreads();
  uint32_t top = 1;   // largest power of two of the search: buckets 0 .. 2 top - 1
  while (2u * top < nb) top <<= 1;
  for (uint32_t i = tid; i < len; i += kBlock) atomicAdd(&sk.at[seg_bucket(sk, top, keys[i])], 1u);
  __syncthreads();
  // exclusive scan of the counts: each bucket's first slot
  if (tid < 64u) {
    uint32_t run = 0;
    for (uint32_t b0 = 0; b0 < kMaxBuckets; b0 += 64u) {
      const uint32_t c = sk.at[b0 + tid];
      const uint32_t x = wave_incl_scan(c);
      sk.at[b0 + tid] = run + x - c;
      run += __shfl(x, 63);
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < len; i += kBlock) {
    const uint64_t k = keys[i];
    tmp[atomicAdd(&sk.at[seg_bucket(sk, top, k)], 1u)] = k;
  }
  __syncthreads();   // at[b] is now the bucket's end
  for (uint32_t b = 0; b < nb; b++) {
    const uint32_t o = b ? sk.at[b - 1u] : 0u, m = sk.at[b] - o;
    if (m == 0u) continue;
    if (m > kChunk) {
      seg_sort_merge(tmp + o, keys + o, m, vals + o, sa, sb);
      continue;
    }
    const uint64_t* r = seg_sort_chunk(tmp + o, m, sa, sb);
    for (uint32_t i = tid; i < m; i += kBlock) vals[o + i] = seg_val(r[i]);
    __syncthreads();   // the next bucket's runs overwrite the LDS
  }
}

// One block per tile: sorts the tile's segment and writes the raster values
// (id | mask << 28) in order: in LDS up to kChunk keys, by buckets above.
// Blocks take the tiles in the raster launch order (most keys first), so the
// long segments start early instead of trailing the launch.
// Batched: view blockIdx.x, tile rank blockIdx.y, so the launch starts every
// view's heaviest tiles first.
// Everything is inlined and held to the registers of 8 waves per SIMD (56,
// nothing spilled; LDS allows 9 blocks per CU): called out of line, the LDS
// pointers became generic ones and the accesses flat (1M Gaussians: 36.1 ->
// 31.5 us).
template <bool kJobs>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_seg_sort(SegJob arg, const SegJob* __restrict__ jobs) {
  const SegJob j = seg_job<kJobs>(arg, jobs, kJobs ? blockIdx.x : 0);
  if (kJobs && j.skip) return;
  const uint32_t rank = kJobs ? blockIdx.y : blockIdx.x;
  if (kJobs && rank >= (uint32_t)j.numTiles) return;
  uint64_t* __restrict__ keys = j.keys;
  uint32_t* __restrict__ vals = j.ids;
  __shared__ uint64_t sa[kChunk];
  __shared__ uint64_t sb[kChunk];
  __shared__ SegBuckets sk;
  const uint2 r = j.ranges[j.tileOrder[rank]];
  const uint32_t s = r.x, len = r.y - r.x;
  const uint32_t tid = threadIdx.x;
  if (len == 0u) return;
  if (len == 1u) {
    if (tid == 0) vals[s] = seg_val(keys[s]);
    return;
  }
  if (len > kChunk) {
    seg_sort_buckets(keys + s, j.tmp + s, len, vals + s, sa, sb, sk);
    return;
  }
  const uint64_t* sorted = seg_sort_chunk(keys + s, len, sa, sb);
  for (uint32_t i = tid; i < len; i += kBlock) vals[s + i] = seg_val(sorted[i]);
}

// one pass: histogram, per-digit scan (with digit totals), stable scatter
// nOut != nullptr: drop keys equal to ~0 and store the count kept there
template <typename KeyT>
static void radix_pass(hipStream_t st, const SortScratch& s, const KeyT* kin, const uint32_t* vin,
                       KeyT* kout, uint32_t* vout, const uint32_t* dN, int shift, uint32_t* nOut) {
  if (nOut) k_radix_hist<KeyT, true><<<s.G, kBlock, 0, st>>>(kin, dN, shift, s.G, s.hist);
  else k_radix_hist<KeyT, false><<<s.G, kBlock, 0, st>>>(kin, dN, shift, s.G, s.hist);
  k_radix_scan<<<256, kBlock, 0, st>>>(s.hist, s.G, s.totals);
  if (nOut)
    k_radix_scatter<KeyT, true, true><<<s.G, kBlock, 0, st>>>(kin, vin, dN, shift, s.G, s.hist, kout, vout, s.totals,
                                                             nOut);
  else
    k_radix_scatter<KeyT, true, false><<<s.G, kBlock, 0, st>>>(kin, vin, dN, shift, s.G, s.hist, kout, vout,
                                                              s.totals, nullptr);
}

// Stable LSD sort of (key, val) pairs by key bits [bit0, bit1), 8 per pass.
// Pass p reads the previous pass's output (the input for p = 0; vals = iota
// when vin is null) and writes (k1, v1) for even p, (k2, v2) for odd p. The
// input may alias (k2, v2): it is consumed by the first pass. nKept !=
// nullptr: the first pass drops keys equal to ~0, stores the number kept in
// *nKept, and the later passes sort that many.
template <typename KeyT>
static void radix_sort(hipStream_t st, const SortScratch& s, const KeyT* kin, const uint32_t* vin,
                       KeyT* k1, uint32_t* v1, KeyT* k2, uint32_t* v2, const uint32_t* dN,
                       int bit0, int bit1, const KeyT** kres, const uint32_t** vres, uint32_t* nKept = nullptr) {
  const KeyT* ki = kin;
  const uint32_t* vi = vin;
  bool odd = false;
  for (int b = bit0; b < bit1; b += 8) {
    KeyT* ko = odd ? k2 : k1;
    uint32_t* vo = odd ? v2 : v1;
    const bool first = b == bit0;
    radix_pass<KeyT>(st, s, ki, vi, ko, vo, first || !nKept ? dN : nKept, b, first ? nKept : nullptr);
    ki = ko;
    vi = vo;
    odd = !odd;
  }
  *kres = ki;
  *vres = vi;
}

int64_t seg_group(int64_t n) {
  // the blocks take whole chunks by cost, so the group only sets their number
  static_assert(kSegBlocks <= kScanThreads, "one scan thread per block");
  const int64_t g = (n + kSegBlocks - 1) / kSegBlocks;
  return g > kSegMinGroup ? g : kSegMinGroup;
}

int tile_bits(int numTiles) {
  int b = 0;
  while ((1 << b) < numTiles) b++;
  return b < 1 ? 1 : b;
}

int seg_blocks(int64_t n) {
  const int64_t G = seg_group(n);
  return (int)((n + G - 1) / G);
}

// The five tile-segment stages for V jobs (kJobs: from the device array
// jobs, view from the block index; else the one job j by value); maxTiles:
// the most tiles of any job. Every job has the same Gaussian count (nb).
template <bool kJobs>
static void seg_launches(hipStream_t st, const SegJob& j, const SegJob* jobs, int V, int maxTiles) {
  static const bool ldsRaised = [] {
    // the per-tile LDS arrays at kMaxSegTiles: 5 B per tile in the scatter, 4 in the others
    const int dyn = kMaxSegTiles * 5;
    (void)hipFuncSetAttribute((const void*)k_seg_count<kJobs>, hipFuncAttributeMaxDynamicSharedMemorySize, dyn);
    (void)hipFuncSetAttribute((const void*)k_seg_scan<kJobs, 16>, hipFuncAttributeMaxDynamicSharedMemorySize, dyn);
    (void)hipFuncSetAttribute((const void*)k_seg_scatter<kJobs>, hipFuncAttributeMaxDynamicSharedMemorySize, dyn);
    return true;
  }();
  (void)ldsRaised;
  const unsigned v = (unsigned)V;
  k_seg_count<kJobs><<<dim3((unsigned)j.nb, v), kSegThreads, (size_t)maxTiles * 4, st>>>(j, jobs);
  k_seg_colscan<kJobs><<<dim3((unsigned)((maxTiles + 15) / 16), v), kBlock, 0, st>>>(j, jobs);
  const dim3 sg(1u, v);
  const size_t sl = (size_t)maxTiles * 4;
  if (maxTiles <= kScanThreads) k_seg_scan<kJobs, 1><<<sg, kScanThreads, sl, st>>>(j, jobs);
  else if (maxTiles <= 2 * kScanThreads) k_seg_scan<kJobs, 2><<<sg, kScanThreads, sl, st>>>(j, jobs);
  else if (maxTiles <= 4 * kScanThreads) k_seg_scan<kJobs, 4><<<sg, kScanThreads, sl, st>>>(j, jobs);
  else if (maxTiles <= 8 * kScanThreads) k_seg_scan<kJobs, 8><<<sg, kScanThreads, sl, st>>>(j, jobs);
  else k_seg_scan<kJobs, 16><<<sg, kScanThreads, sl, st>>>(j, jobs);
  k_seg_scatter<kJobs><<<dim3((unsigned)j.nb, v), kSegThreads, (size_t)maxTiles * 5, st>>>(j, jobs);
  if (kJobs) k_seg_sort<kJobs><<<dim3(v, (unsigned)maxTiles), kBlock, 0, st>>>(j, jobs);
  else k_seg_sort<kJobs><<<dim3((unsigned)maxTiles), kBlock, 0, st>>>(j, jobs);
}

void launch_bin_sort_views(hipStream_t st, const SegJob* dJobs, const SegJob* hJobs, int V) {
  int maxTiles = 0;
  for (int k = 0; k < V; k++)
    if (!hJobs[k].skip) maxTiles = maxTiles > hJobs[k].numTiles ? maxTiles : hJobs[k].numTiles;
  if (maxTiles > 0) seg_launches<true>(st, hJobs[0], dJobs, V, maxTiles);
}

void launch_bin_sort(hipStream_t st, const BinArgs& a, BinOut& out) {
  const SortScratch& s = a.scratch;
  const int tb = tile_bits(a.numTiles);
  const int tpasses = (tb + 7) / 8;
  const int Gc = (int)((a.n + kBlock - 1) / kBlock);
  if (a.mode == 2 && a.numTiles <= kMaxSegTiles) {
    // tile segments: count table, column scan, budgeted scan, scatter, per-tile sort
    SegJob j{};
    j.n = a.n;
    j.cap = a.cap;
    j.nb = seg_blocks(a.n);
    j.tilesX = a.tilesX;
    j.tile = a.tile;
    j.numTiles = a.numTiles;
    j.recFmt = a.recFmt;
    j.rec = const_cast<float4*>(a.rec);
    j.depthKey = const_cast<uint32_t*>(a.depthKey);
    j.rect = const_cast<uint2*>(a.rect);
    j.cnt = const_cast<uint32_t*>(a.cnt);
    j.chunkKeys = s.chunkKeys;
    j.blockStart = s.blockStart;
    j.table = s.segTable;
    j.visPart = s.visPart;
    j.tileCnt = s.tileCnt;
    j.ranges = a.ranges;
    j.tileOrder = a.tileOrder;
    j.numKeys = a.numKeys;
    j.numVisible = a.numVisible;
    j.totalKeys = a.totalKeys;
    j.stats = a.stats;
    j.keys = (uint64_t*)a.tkA;
    j.tmp = (uint64_t*)a.tkB;
    j.ids = a.tvA;
    seg_launches<false>(st, j, nullptr, 1, j.numTiles);
    out.keys = nullptr;
    out.ids = a.tvA;
    out.keyBytes = 0;
    out.tileOrder = a.tileOrder;
    return;
  }
  if (a.mode == 0 || a.mode == 2) {   // mode 2 lands here above kMaxSegTiles tiles
    // 1) stable sort of the Gaussians by depth bits, values = ids
    const uint32_t* dk;
    const uint32_t* order;
    radix_sort<uint32_t>(st, s, a.depthKey, nullptr, a.dkA, a.dvA, a.dkB, a.dvB, a.dN, 0, 32, &dk, &order,
                         s.nDepth);
    // 2) per-Gaussian key counts in depth order -> offsets -> one key per tile
    k_count_partials<<<Gc, kBlock, 0, st>>>(order, a.cnt, a.rect, a.depthKey, s.nDepth, s.cntS, s.rectS, nullptr,
                                            s.partials, s.vpartials);
    k_count_top<<<1, 1024, 0, st>>>(s.partials, s.vpartials, Gc, a.cap, a.numKeys, a.totalKeys, a.numVisible, a.stats);
    k_emit<false><<<Gc, kBlock, 0, st>>>(order, s.cntS, s.rectS, nullptr, s.nDepth, s.partials, a.tilesX, a.tile, a.cap,
                                         a.rec, a.recFmt, a.tkA, a.tvA);
    // 3) stable sort by tile id
    const uint32_t* tk;
    const uint32_t* tv;
    radix_sort<uint32_t>(st, s, (const uint32_t*)a.tkA, a.tvA, (uint32_t*)a.tkB, a.tvB,
                         (uint32_t*)a.tkA, a.tvA, a.numKeys, 0, 8 * tpasses, &tk, &tv);
    out.keys = tk;
    out.ids = tv;
    out.keyBytes = 4;
    launch_fill_u32(st, (uint32_t*)a.ranges, 2 * (int64_t)a.numTiles, 0u);
    k_tile_ranges<uint32_t><<<1024, 256, 0, st>>>(tk, a.numKeys, 0, a.numTiles, a.ranges);
    k_tile_order<<<1, 1024, 0, st>>>(a.ranges, a.numTiles, a.tileOrder);
  } else {
    k_count_partials<<<Gc, kBlock, 0, st>>>(nullptr, a.cnt, a.rect, a.depthKey, a.dN, s.cntS, s.rectS, s.dkS,
                                            s.partials, s.vpartials);
    k_count_top<<<1, 1024, 0, st>>>(s.partials, s.vpartials, Gc, a.cap, a.numKeys, a.totalKeys, a.numVisible, a.stats);
    k_emit<true><<<Gc, kBlock, 0, st>>>(nullptr, s.cntS, s.rectS, s.dkS, a.dN, s.partials, a.tilesX, a.tile, a.cap,
                                        a.rec, a.recFmt, a.tkA, a.tvA);
    const uint64_t* tk;
    const uint32_t* tv;
    radix_sort<uint64_t>(st, s, (const uint64_t*)a.tkA, a.tvA, (uint64_t*)a.tkB, a.tvB,
                         (uint64_t*)a.tkA, a.tvA, a.numKeys, 0, 32 + 8 * tpasses, &tk, &tv);
    out.keys = tk;
    out.ids = tv;
    out.keyBytes = 8;
    launch_fill_u32(st, (uint32_t*)a.ranges, 2 * (int64_t)a.numTiles, 0u);
    k_tile_ranges<uint64_t><<<1024, 256, 0, st>>>(tk, a.numKeys, 32, a.numTiles, a.ranges);
    k_tile_order<<<1, 1024, 0, st>>>(a.ranges, a.numTiles, a.tileOrder);
  }
  out.tileOrder = a.tileOrder;
}

}  // namespace gs
