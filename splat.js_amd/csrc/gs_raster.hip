// gs_raster.hip — per-tile alpha compositing, forward and backward
// (the reference's `render` pass, shaders.js:511-702).
//
// One workgroup per tile, one thread per pixel, each wave an 8x8 block: by
// default 16x16 tiles (256 threads, 4 waves) and batches of 256 keys; tiles
// of 8 or 32 pixels and batches of 64 or 128 are the other shapes (Shape
// below). The tile's sorted keys are consumed in batches: the waves load
// the batch's raster records into LDS (lane l of a wave one record of each
// 64-key chunk it stages), then every pixel walks the batch from LDS
// (broadcast reads). Each key carries the mask of the tile's quadrants whose
// pixels may take the splat (gs_cover.h, set by the binning pass): a wave
// visits only the splats of its quadrant's bit, a splat with an empty mask
// is not even loaded, and a wave leaves a splat early once no lane is inside
// the cutoff or takes it. The batch size changes no result (each pixel still
// walks its keys in order); the tile size changes which keys exist (the
// tile rectangles and the entry budget are per tile), as in the restatement
// run at the same tile size. The forward stops the whole tile once
// every pixel has reached T < 1e-4. Both passes evaluate alpha with
// gs_expf_raster (gs_math.h), as the restatement's raster passes do.
//
// Forward (shaders.js:556-585) writes the image, the final transmittance T
// and `end` (one past the last key the pixel processed); in training it also
// evaluates the Charbonnier loss per pixel (shaders.js:589-618) and stores
// dL/dC, so the backward pass needs no second loss read.
//
// Backward (shaders.js:620-700) walks each tile from the largest `end` of
// its pixels down to the first key (each wave from the largest `end` of its
// own pixels), recomputing each pixel's transmittance
// in front of a splat from the stored final T (Tb = Ta/(1-a), through one
// reciprocal that also scales the colour-behind sum S). It visits the keys
// that some lane took in the forward, which leaves words of 64 keys for this
// (RasterBufs::took). Per visit, the 10 screen-space gradient terms are summed
// over lanes (one DPP step, then the wave's own LDS scratch; WaveRed below).
//   GS_ACCUM_FIXED: the 16-lane groups of a wave (4x4 pixels each) walk lists
//                   of their own, from a word per group. A wave is done with a
//                   batch of 128 keys when its longest list is: a splat that
//                   misses a group costs it nothing, where a walk of the whole
//                   wave's keys left half of the lanes idle. The groups' sums
//                   are added to the batch's sums in LDS; these go to the
//                   Gaussians' accumulators with one atomic per key, term and
//                   tile once the batch is done.
//                   Each pixel's term is converted to i32 first,
//                   i32(clamp(v * 16384, -1e9, 1e9)), exactly as the
//                   reference's atomicAdd on atomic<i32> (shaders.js:529-541);
//                   integer sums commute, so the result is deterministic and
//                   bit-identical to any other summation order. (Under the
//                   Charbonnier loss the three colour terms cannot reach the
//                   clamp and convert without it.)
//   GS_ACCUM_F32:   plain f32 sums (atomic add order is not deterministic). A
//                   wave walks its keys as one, and adds its 64 pixels' sums
//                   to the Gaussian's accumulator with one atomic per term: a
//                   float added in LDS costs several times an integer one, so
//                   the groups' lists took 1160 us where this takes 666 (1M
//                   Gaussians at 1600x900, forward and backward).
//
// Training under the Charbonnier loss runs both passes in one launch: the
// loss gradient of a pixel needs only that pixel, so a block runs its tile's
// backward right after the forward (k_raster_fwd_bwd, and the persistent
// k_raster_fwd_bwd_views over a batched step's views). The two passes share
// one LDS array, and the backward stages the tile's records again while
// they are still in L2 from the forward. Renders, and the L1 + D-SSIM loss
// (whose gradient needs neighbouring pixels), run the passes apart.
//
// What bounds both visit loops is instruction issue: vector instructions
// where the chip is full, and on small images, with about one wave per SIMD,
// every instruction, scalar ones included (~4 cycles each there). So the
// masks of a forward visit live in scalar registers, with one instruction to
// clear a bit. Backward with lists per group (fixed-point sums) against a walk
// of the wave's keys with an atomic per wave: 20k Gaussians at 320x240 87 -> 64 us, 600k at
// 1237x933 389 -> 315; forward and backward in one launch, 160 Gaussians at
// 64x64 28 -> 24, 123k at 737x411 93 -> 79, 1M at 1600x900 566 -> 543, 8 views
// of 1M 3865 -> 3745. Where splats cover whole tiles the lists of a wave are
// all alike and their making is extra work: 1M large Gaussians, two views
// at 1920x1080, 883 -> 985. Added to the Gaussians directly, the groups'
// sums were bound by the rate of atomics (389 -> 787 at 1237x933).
#include <type_traits>

#include "gs_kernels.h"

namespace gs {

__device__ __forceinline__ int tile_of_block(const RasterBufs& b) { return (int)b.tileOrder[blockIdx.x]; }

// Shape of a raster launch: kT x kT pixel tiles, one thread per pixel, in
// waves of 8x8 pixel blocks (wave w: block column w % (kT/8), block row
// w / (kT/8); each 16 lanes a 4x4 block of it, row by row), and kB keys
// staged in LDS per round, in chunks of 64 keys (one ballot word each).
// Each key carries 4 cover bits, one per quadrant of the tile (kT/2 x kT/2
// pixels, bit 2 row + column): a wave tests its quadrant's bit (at kT = 16
// the quadrant is the wave's own block; at kT = 32 four waves share one; at
// kT = 8 the one wave spans all four and tests whether any bit is set).
template <int kT, int kB>
struct Shape {
  static constexpr int T = kT, B = kB;
  static constexpr int kThreads = kT * kT;
  static constexpr int kWaves = kThreads / 64;
  static constexpr int kChunks = kB / 64;
  static constexpr int kBW = kT / 8;            // 8x8 blocks per tile row
  static constexpr int kMasks = kT == 8 ? 1 : 4;
  // occupancy the launches with a backward are compiled for: 8 waves per SIMD
  // (at most 64 VGPRs; left free, the compiler takes 72, and the persistent
  // grid, sized by occupancy, shrinks); 8-pixel tiles are held below that by
  // their LDS anyway
  static constexpr int kBwdWavesPerEU = kT == 8 ? 1 : 8;
  static_assert((kT == 8 || kT == 16 || kT == 32) && (kB == 64 || kB == 128 || kB == 256), "raster shape");
  __device__ static int mask_slot(int w) {
    if constexpr (kT == 8) {
      return 0;
    } else {
      constexpr int h = kBW / 2;   // blocks per quadrant row
      return 2 * ((w / kBW) / h) + (w % kBW) / h;
    }
  }
};

// LDS of the raster passes, carved from one array that the kernel declares,
// so a launch that runs both passes holds the larger layout, not both.
// Forward: records sA, sB, sC (16 B each per key), the chunk masks per
// quadrant, the loss partials; backward: the records of a batch of kKeys keys
// and one that no lane takes, the waves' reduction scratch, the groups'
// lists, the batch's gradient sums, the block's largest end. Sizes in float4.
// 128 keys keep a block of 16-pixel tiles at 18.8 KB, eight to a CU.
constexpr int kRedStride = 68;   // words between a wave's 64-word rows (see WaveRed)
constexpr int kGroups = 4;       // 16-lane groups of a wave, each a 4x4 pixel block
template <class S>
struct RasterLds {
  // Keys per batch of the backward: 128, and 64 where the block is one wave
  // (8-pixel tiles) and its forward stages no more than 128, since the CU then
  // runs as many waves as its LDS holds blocks: 7.4 KB instead of 13.2. 1M
  // Gaussians at 1920x1080, batches of 128: 1559 -> 1164 us (1505 when the
  // backward held no lists and sums). With 256 the forward alone holds 12 KB.
  static constexpr int kKeys = S::B < 128 || (S::T == 8 && S::B == 128) ? 64 : 128;
  static constexpr int kFwd = 3 * S::B + (S::kChunks * S::kMasks * 8 + 3 * S::kWaves * 8 + 15) / 16;
  static constexpr int kRed = S::kWaves * 5 * kRedStride / 4;   // the waves' reduction scratch
  static constexpr int kLists = S::kWaves * kGroups * kKeys / 16;   // a byte per key and group
  static constexpr int kSums = (kKeys + 1) * 10 / 4 + 1;            // the batch's gradient sums
  static constexpr int kBwd = 3 * (kKeys + 1) + kRed + kLists + kSums + 1;   // one record more: nobody's
  static constexpr int kBoth = kFwd > kBwd ? kFwd : kBwd;
};

struct PixelMap {
  int x, y;        // pixel
};

// What the forward with the loss leaves for the backward at a thread's
// pixel: dL/dC (w = 1 for a valid target pixel, 0 otherwise, and 0 outside
// the image), the final T and `end`. Handed over in registers when both
// passes run in one launch.
struct PixelState {
  float4 g;
  float T;
  uint32_t end;
};
template <class S>
__device__ __forceinline__ PixelMap pixel_of_thread(const Cam& cam, int tile, int tid) {
  const int tx = tile % cam.tilesX, ty = tile / cam.tilesX;
  const int w = tid >> 6, l = tid & 63;
  PixelMap m;
  m.x = tx * S::T + (w % S::kBW) * 8 + (l & 3) + 4 * ((l >> 4) & 1);
  m.y = ty * S::T + (w / S::kBW) * 8 + ((l >> 2) & 3) + 4 * (l >> 5);
  return m;
}

// Stores the staged chunk's ballots of the cover bits the waves test (lane
// l of the calling wave holds key 64 c + l of the batch; keys past the
// segment end have cover 0 and contribute no bits).
template <class S>
__device__ __forceinline__ void store_masks(uint32_t cover, uint64_t* m) {
  const bool lead = (threadIdx.x & 63) == 0;
  if constexpr (S::kMasks == 1) {
    const uint64_t bal = wave_ballot(cover != 0u);
    if (lead) m[0] = bal;
  } else {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const uint64_t bal = wave_ballot(((cover >> q) & 1u) != 0u);
      if (lead) m[q] = bal;
    }
  }
}

// m without bit `bit`, in one scalar instruction (the compiler takes two or three)
__device__ __forceinline__ void clear_bit(uint64_t& m, int bit) {
  asm("s_bitset0_b64 %0, %1" : "+s"(m) : "s"(bit));
}

// the same when `mask` is empty (left to the compiler: five instructions)
__device__ __forceinline__ void clear_bit_if_none(uint64_t& m, int bit, uint64_t mask) {
  asm("s_cmp_lg_u64 %1, 0\n\ts_cbranch_scc1 .Lgs_some%=\n\ts_bitset0_b64 %0, %2\n.Lgs_some%=:"
      : "+s"(m) : "s"(mask), "s"(bit) : "scc");
}

// the OR over the first n lanes (the others hold 0), in a scalar register
template <int n>
__device__ __forceinline__ uint32_t or_lanes(uint32_t v) {
  v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, false);   // row_ror 8, 4, 2, 1
  v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x124, 0xf, 0xf, false);
  v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x122, 0xf, 0xf, false);
  v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x121, 0xf, 0xf, false);
  uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
#pragma unroll
  for (int l = 16; l < n; l += 16) r |= (uint32_t)__builtin_amdgcn_readlane((int)v, l);
  return r;
}

// `old` with lane `lane` set to v (both uniform)
__device__ int write_lane(int v, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

// Byte offset j * size of a staged record as a VGPR value the compiler
// cannot recompute: every LDS read of record j then shares this one address
// register (the compiler otherwise moves the uniform offset into a fresh
// VGPR before each group of reads).
__device__ __forceinline__ uint32_t lds_offset(uint32_t bytes) {
  uint32_t v;
  asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "s"(bytes));
  return v;
}

template <typename T>
__device__ __forceinline__ const T& lds_at(const void* base, uint32_t off) {
  return *(const T*)((const char*)base + off);
}

// The exponent clamped to [0, 87] in one v_med3_f32 (fminf(fmaxf()) takes
// two): max(e, 0) is the reference's (shaders.js:565); the upper clamp only
// keeps the exp's argument in range, since e > eCut (<= 80) is never taken.
// e is finite (bounded conic and offsets), where med3 equals the pair.
__device__ __forceinline__ float clamp_e(float e) { return __builtin_amdgcn_fmed3f(e, 0.0f, 87.0f); }

__device__ __forceinline__ float max3abs(float a, float b, float c) {
  return fmaxf(fmaxf(fabsf(a), fabsf(b)), fabsf(c));
}

// 1/x for x in [2^-9, 1]: hardware reciprocal estimate plus one Newton step
// with fused residual. Equal to IEEE 1.0f/x for all 75,497,473 floats of that
// range (exhaustive check on gfx950); callers guarantee the range.
__device__ __forceinline__ float rcp_exact_unit(float x) {
  float r = __builtin_amdgcn_rcpf(x);
  const float e = fmaf(-x, r, 1.0f);
  return fmaf(r, e, r);
}

// The record's colours as f32: stored as f32 (recFmt 0: (r, g, b, opa) is
// the third float4) or as bf16 / fp16 pairs in the second float4's z, w
// (recFmt 1, 2), which decode exactly.
__device__ __forceinline__ float4 record_colour(int recFmt, const float4& r1, float w) {
  const uint32_t rg = __float_as_uint(r1.z), bl = __float_as_uint(r1.w);
  if (recFmt == 2)
    return make_float4(dec16<2>(rg), dec16<2>(rg >> 16), dec16<2>(bl), w);
  return make_float4(dec16<1>(rg), dec16<1>(rg >> 16), dec16<1>(bl), w);
}

// First word (of one per 4x4 block, a wave's four next to each other) of RasterBufs::took for 64-key chunk `c`
// (below the tile's keys / 64, rounded up) of the tile whose keys start at s.
// Tiles lie in key order, so the rows of two
// tiles never overlap: s / 64 grows by at least the earlier tile's chunks
// less one, and the tile index by one.
template <class S>
__device__ __forceinline__ size_t took_word(uint32_t s, int tile, uint32_t c) {
  return ((size_t)(s >> 6) + (uint32_t)tile + c) * (S::kWaves * kGroups);
}

// One tile of the forward pass, by the whole 256-thread block. The block's
// threads must all call it (it synchronises), and nothing else may use the
// block's LDS until every thread has returned. What the backward needs of the
// keys that are taken: kTookGroups, each 16-lane group's; kTookWaves, each
// wave's, as the word of its first group (a scalar word: no lane writes).
constexpr int kTookNone = 0, kTookGroups = 1, kTookWaves = 2;
template <class S, int kLoss, int kTook>
__device__ __forceinline__ void raster_fwd_tile(const Cam& cam, const Cut& cut, const RasterBufs& b, int tile,
                                                float4* lds, PixelState* out = nullptr) {
  float4* const sA = lds;              // mx, my, A, B
  float4* const sB = lds + S::B;       // C, opa*comp, L, 0
  float4* const sC = lds + 2 * S::B;   // r, g, b, opa
  uint64_t (*const sMask)[S::kMasks] = reinterpret_cast<uint64_t (*)[S::kMasks]>(lds + 3 * S::B);
  double (*const sStat)[S::kWaves] = reinterpret_cast<double (*)[S::kWaves]>(&sMask[S::kChunks][0]);
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const int mslot = S::mask_slot(wv);
  const PixelMap pm = pixel_of_thread<S>(cam, tile, tid);
  const int x = pm.x, y = pm.y;
  const bool inside = x < cam.W && y < cam.H;
  const float px = (float)x + 0.5f, py = (float)y + 0.5f;
  const uint2 rg = b.ranges[tile];
  const uint32_t s = __builtin_amdgcn_readfirstlane(rg.x), e = __builtin_amdgcn_readfirstlane(rg.y);
  if (out) *out = PixelState{make_float4(0.0f, 0.0f, 0.0f, 0.0f), 0.0f, s};
  float T = 1.0f, C0 = 0.0f, C1 = 0.0f, C2 = 0.0f;
  uint32_t end = s;
  // lanes still compositing, in scalar registers: a lane is done once outside
  // the image or once T < 1e-4
  uint64_t run = wave_ballot(inside);
  for (uint32_t base = s; base < e; base += S::B) {
    if (__syncthreads_or(run != 0ull) == 0) break;
    // wave w stages chunks w, w + kWaves, ... (lane l: key 64 c + l)
    for (int c = wv; c < S::kChunks; c += S::kWaves) {
      const int j = 64 * c + lane;
      const uint32_t k = base + (uint32_t)j;
      uint32_t cover = 0;
      if (k < e) {
        const uint32_t v = b.ids[k];
        cover = v >> kMaskShift;
        if (cover != 0u) {           // splats no block of the tile can take stay unloaded
          const uint32_t id = v & kIdMask;
          if (b.recFmt == 0) {
            sA[j] = b.rec[4 * id + 0];
            sB[j] = b.rec[4 * id + 1];
            sC[j] = b.rec[4 * id + 2];
          } else {
            const float4 r1 = b.rec[3 * id + 1];
            sA[j] = b.rec[3 * id + 0];
            sB[j] = r1;
            sC[j] = record_colour(b.recFmt, r1, 0.0f);
          }
        }
      }
      store_masks<S>(cover, sMask[c]);
    }
    __syncthreads();
    const uint32_t cnt = min((uint32_t)S::B, e - base);
    if (run != 0ull) {
      for (int c = 0; c < S::kChunks; c++) {
        uint64_t m = uniform64(sMask[c][mslot]);
        int tkLo = 0, tkHi = 0;   // kTookGroups: lane k holds the lanes that take key k of the chunk
        uint64_t took = m;        // kTookWaves: the keys that some lane takes
        while (m) {
          const int bit = (int)__builtin_ctzll(m);
          clear_bit(m, bit);
          // Only lanes that take the splat (still running, inside the cutoff,
          // alpha >= A_MIN) update their state; the wave leaves as soon as
          // there is none. The masks are combined in scalar registers.
          const uint32_t jo = lds_offset((uint32_t)bit * 16u);
          const float4 a = lds_at<float4>(sA + 64 * c, jo);
          const float2 bb = lds_at<float2>(sB + 64 * c, jo);   // C, opa*comp
          asm volatile("" ::"v"(bb.y));                         // one 8-byte read
          const float dx = px - a.x, dy = py - a.y;
          const float t2 = fmaf(bb.x * dy, dy, (a.z * dx) * dx);
          // clamped to [0, 87]: an exponent above 87 > eCut is never taken,
          // and the exp below needs its argument in [-87, 0]
          const float ee = clamp_e(fmaf(0.5f, t2, (a.w * dx) * dy));
          const uint64_t live = run & wave_ballot(ee <= cut.eCut);
          uint64_t take = 0ull;
          if (live != 0ull) {
            const float araw = bb.y * gs_expf_raster(-ee);
            const float alpha = fminf(0.99f, araw);
            take = live & wave_ballot(alpha >= cut.aMin);
            if (__builtin_amdgcn_inverse_ballot_w64(take)) {
              const float4 c4 = lds_at<float4>(sC + 64 * c, jo);
              const float w = T * alpha;
              C0 = fmaf(w, c4.x, C0);
              C1 = fmaf(w, c4.y, C1);
              C2 = fmaf(w, c4.z, C2);
              T = T * (1.0f - alpha);
            }
            // T only falls here, so a lane reaches T < 1e-4 on this splat
            // exactly when it is still running and now below; that happens
            // once per pixel, so its bookkeeping sits behind a scalar branch
            if (kTook == kTookGroups) {
              tkLo = write_lane((int)(uint32_t)take, bit, tkLo);
              tkHi = write_lane((int)(uint32_t)(take >> 32), bit, tkHi);
            }
            const uint64_t fin = run & wave_ballot(T < 1e-4f);
            if (fin != 0ull) {
              if (__builtin_amdgcn_inverse_ballot_w64(fin)) end = base + (uint32_t)(64 * c + bit) + 1u;
              run &= ~fin;
              if (run == 0ull) m = 0ull;
            }
          }
          if (kTook == kTookWaves) clear_bit_if_none(took, bit, take);
        }
        if (kTook == kTookWaves && 64u * (uint32_t)c < cnt && lane == 0) {
          ulonglong2* tw = (ulonglong2*)(b.took + took_word<S>(s, tile, ((base - s) >> 6) + (uint32_t)c) + wv * kGroups);
          tw[0] = make_ulonglong2(took, 0ull);
          tw[1] = make_ulonglong2(0ull, 0ull);
        }
        if (kTook == kTookGroups && 64u * (uint32_t)c < cnt) {
          const uint64_t w0 = wave_ballot(((uint32_t)tkLo & 0xffffu) != 0u), w1 = wave_ballot(((uint32_t)tkLo >> 16) != 0u);
          const uint64_t w2 = wave_ballot(((uint32_t)tkHi & 0xffffu) != 0u), w3 = wave_ballot(((uint32_t)tkHi >> 16) != 0u);
          if (lane == 0) {
            ulonglong2* tw = (ulonglong2*)(b.took + took_word<S>(s, tile, ((base - s) >> 6) + (uint32_t)c) + wv * kGroups);
            tw[0] = make_ulonglong2(w0, w1);
            tw[1] = make_ulonglong2(w2, w3);
          }
        }
        if (run == 0ull) break;
      }
      if (__builtin_amdgcn_inverse_ballot_w64(run)) end = base + cnt;
    }
  }
  double st0 = 0.0, st1 = 0.0, st2 = 0.0;
  if (inside) {
    const int64_t pi = (int64_t)y * cam.W + x;
    const float o0 = C0 + T * cam.bg[0], o1 = C1 + T * cam.bg[1], o2 = C2 + T * cam.bg[2];
    b.img[pi] = make_float4(o0, o1, o2, 1.0f - T);
    if (kLoss) {
      b.T[pi] = T;
      b.end[pi] = end;
      if (out) {
        out->T = T;
        out->end = end;
      }
    }
    if (kLoss == 1) {
      const uint32_t pk = b.tgt[cam.tgtOffset + pi];
      float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if ((pk >> 24) != 0u) {
        const float o[3] = {o0, o1, o2};
        float err[3], root[3], gg[3];
        for (int c = 0; c < 3; c++) {
          const float tc = (float)((pk >> (8 * c)) & 0xffu) / 255.0f;
          err[c] = (cam.gain * o[c] + cam.bias) - tc;
          root[c] = sqrtf(err[c] * err[c] + 0.0009f);
          gg[c] = cam.gain * (err[c] / root[c]);
        }
        g = make_float4(gg[0], gg[1], gg[2], 1.0f);
        st0 = (double)dot3(err, err);
        st1 = (double)(((root[0] + root[1]) + root[2]) - 0.09f);
        st2 = 1.0;
      }
      b.gC[pi] = g;
      if (out) out->g = g;
    }
  }
  if (kLoss == 1) {
    for (int o = 32; o > 0; o >>= 1) {
      st0 += __shfl_xor(st0, o);
      st1 += __shfl_xor(st1, o);
      st2 += __shfl_xor(st2, o);
    }
    if ((tid & 63) == 0) { sStat[0][wv] = st0; sStat[1][wv] = st1; sStat[2][wv] = st2; }
    __syncthreads();
    if (tid < 3) {
      double v = sStat[tid][0];
      for (int w = 1; w < S::kWaves; w++) v += sStat[tid][w];
      if (v != 0.0) atomicAdd(&stat_line(b.stats, (uint32_t)tile)[tid], v);
    }
  }
}

// ---- reduction of a visit's 10 values over each 16-lane group ----
// A visit's terms are summed over a group (a DPP row) in two steps:
//  1. l ^ 15 (row_mirror, across bit 3 of the lane index) as two DPP adds per
//     output, each writing one half of the row through the DPP bank mask (no
//     selects): lanes 0-7 of each 16-lane row keep values 0-4, lanes 8-15
//     values 5-9, so 10 values become 5 per lane;
//  2. through the wave's own LDS scratch: register i goes to word 68 i +
//     lane, so the 8 words of one value and row lie next to each other
//     (68, not 64: 16 lanes' 16-byte reads then meet distinct banks). Lane
//     4 q + p (q < 10) reads value q's 8 words of row p and adds them: value
//     q's total of group p, which it adds to the sums of the key that the
//     group visited.
// Why LDS: on gfx950 a DPP add, a select or a compare issues in ~4.2 cycles
// per wave and SIMD, a plain add, multiply or FMA in ~2.4, a permlane swap in
// ~8.1 (measured, independent chains, 8 waves per SIMD). Lane exchanges for
// all steps cost about 110 issue cycles per visit, this about 60.
// Leaving step 1 to LDS as well would take half as many cycles again, but
// would fill the LDS pipe. The matrix cores don't help: an MFMA holds the
// SIMD's vector issue for its whole time (16-32 cycles) here.
// The reads of a visit's words are issued one visit later, before that
// visit's arithmetic, which hides their latency; LDS serves a wave's
// operations in order, so they precede the later visit's writes.
// The asm block starts with two wait states for the DPP read of a value that
// the previous VALU instruction wrote. Every step runs with all 64 lanes
// active (every branch of the visit loop is wave-uniform, and every wave of a
// block is full): a DPP add whose source lane were inactive would leave its
// output unwritten.
template <typename T>
__device__ __forceinline__ uint32_t as_u(T v) { return __builtin_bit_cast(uint32_t, v); }
template <typename T>
__device__ __forceinline__ T from_u(uint32_t v) { return __builtin_bit_cast(T, v); }

#define GS_DPP_M(OP, O, LO, HI) \
  OP " " O ", " LO ", " LO " row_mirror row_mask:0xf bank_mask:0x3\n\t" \
  OP " " O ", " HI ", " HI " row_mirror row_mask:0xf bank_mask:0xc\n\t"
#define GS_ROW_STEP(OP)                \
  "s_nop 1\n\t"                       \
  GS_DPP_M(OP, "%0", "%5", "%10")      \
  GS_DPP_M(OP, "%1", "%6", "%11")      \
  GS_DPP_M(OP, "%2", "%7", "%12")      \
  GS_DPP_M(OP, "%3", "%8", "%13")      \
  GS_DPP_M(OP, "%4", "%9", "%14")

// step 1
template <typename T>
__device__ __forceinline__ void row_halve(const T* v, T* h5) {
  static_assert(sizeof(T) == 4, "32-bit terms");
  if constexpr (std::is_same<T, float>::value) {
    asm volatile(GS_ROW_STEP("v_add_f32_dpp")
                 : "=&v"(h5[0]), "=&v"(h5[1]), "=&v"(h5[2]), "=&v"(h5[3]), "=&v"(h5[4])
                 : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]),
                   "v"(v[5]), "v"(v[6]), "v"(v[7]), "v"(v[8]), "v"(v[9]));
  } else {
    asm volatile(GS_ROW_STEP("v_add_u32_dpp")
                 : "=&v"(h5[0]), "=&v"(h5[1]), "=&v"(h5[2]), "=&v"(h5[3]), "=&v"(h5[4])
                 : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]),
                   "v"(v[5]), "v"(v[6]), "v"(v[7]), "v"(v[8]), "v"(v[9]));
  }
}
#undef GS_ROW_STEP
#undef GS_DPP_M

// x of the lane that a DPP quad permutation selects
template <int kCtrl, typename T>
__device__ __forceinline__ T quad(T x) {
  return from_u<T>((uint32_t)__builtin_amdgcn_mov_dpp((int)as_u(x), kCtrl, 0xf, 0xf, false));
}

// A wave's reduction scratch (5 rows of 64 words at red): where lane l writes
// and reads, and the slot of the sums it adds to (lane 4 q + p: q).
template <typename T>
struct WaveRed {
  T* wr;
  const T* rd;
  int slot;        // the value this lane sums and adds, clamped to 9
  bool flusher;    // lane 4 q + p, q < 10
  __device__ __forceinline__ WaveRed(float4* red, int lane) {
    const int q = lane >> 2, qc = q < 10 ? q : 9;
    wr = reinterpret_cast<T*>(red) + lane;
    rd = reinterpret_cast<const T*>(red) + kRedStride * (qc % 5) + 16 * (lane & 3) + 8 * (qc / 5);
    slot = qc;
    flusher = q < 10;
  }
  __device__ __forceinline__ void write(const T* h5) const {
#pragma unroll
    for (int i = 0; i < 5; i++) wr[kRedStride * i] = h5[i];
  }
  __device__ __forceinline__ void read(T* w8) const {
    const uint4 a = reinterpret_cast<const uint4*>(rd)[0], b = reinterpret_cast<const uint4*>(rd)[1];
    w8[0] = from_u<T>(a.x); w8[1] = from_u<T>(a.y); w8[2] = from_u<T>(a.z); w8[3] = from_u<T>(a.w);
    w8[4] = from_u<T>(b.x); w8[5] = from_u<T>(b.y); w8[6] = from_u<T>(b.z); w8[7] = from_u<T>(b.w);
  }
  // the 16-lane total of this lane's slot in group lane & 3
  __device__ __forceinline__ T total(const T* w8) const {
    return ((w8[0] + w8[1]) + (w8[2] + w8[3])) + ((w8[4] + w8[5]) + (w8[6] + w8[7]));
  }
  // the wave's total of this lane's slot, in the quad's four lanes
  __device__ __forceinline__ T wave_total(const T* w8) const {
    T s = total(w8);
    s = s + quad<0xB1>(s);   // quad_perm [1,0,3,2]
    return s + quad<0x4E>(s);   // quad_perm [2,3,0,1]
  }
};

// GS_ACCUM_FIXED: adds a visit's group totals to the batch's sums in LDS (the
// flushing lanes). The asm keeps the reads of the words ahead of the branch,
// where nothing waits for them yet.
__device__ __forceinline__ void add_group_sums(uint32_t* sum, int key, int slot, uint32_t r, bool flusher) {
  asm volatile("" : "+v"(r));
  if (!flusher) return;
  atomicAdd(reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(sum) + (__umul24((uint32_t)key, 40u) + 4u * (uint32_t)slot)), r);
}

// GS_ACCUM_F32: adds a visit's wave totals to Gaussian g's accumulator row (a
// lane per slot; zeros skipped). The asm keeps the total's last add ahead of
// the branch.
__device__ __forceinline__ void add_wave_sums(float* accum, uint32_t g, int slot, float r, bool flusher) {
  asm volatile("" : "+v"(r));
  if (flusher && r != 0.0f) unsafeAtomicAdd(accum + (uint64_t)g * 12 + (uint32_t)slot, r);
}

// kClampColour false: dL/dC is bounded (the Charbonnier loss: |dL/dC| <=
// gain * |err| / sqrt(err^2 + d^2) <= gain), so the colour terms
// 16384 dL/dC * alpha * T (alpha * T <= 1) stay far inside the +-1e9 clamp
// and convert without it.
// One tile of the backward pass, by the whole block (as raster_fwd_tile).
template <class S, int kAccum, bool kClampColour>
__device__ __forceinline__ void raster_bwd_tile(const Cam& cam, const Cut& cut, const RasterBufs& b, void* accum,
                                                int tile, float4* lds, const PixelState* in = nullptr) {
  // three 16-byte records per staged splat, all at one index: one LDS address
  constexpr int kKeys = RasterLds<S>::kKeys, kWords = S::kWaves * kGroups;
  constexpr int kPart = kKeys / S::kWaves;   // keys that a wave stages and flushes
  static_assert(kKeys / 64 * kGroups <= 64 && kWords <= 64, "one lane per chunk and group, and per block");
  static_assert(kKeys <= 256 && (kPart % 64 == 0 || 64 % kPart == 0), "list entries are bytes; a part lies in a chunk");
  float4* const sA = lds;              // mx, my, A, B
  float4* const sB = lds + (kKeys + 1);       // C, opa*comp, -0.5 cnorm, id (bits)
  float4* const sC = lds + 2 * (kKeys + 1);   // r, g, b, opa
  float4* const sRed = lds + 3 * (kKeys + 1);
  uint8_t* const sList = reinterpret_cast<uint8_t*>(sRed + RasterLds<S>::kRed);
  using AccT = typename std::conditional<kAccum == 0, uint32_t, float>::type;
  AccT* const sSum = reinterpret_cast<AccT*>(sRed + RasterLds<S>::kRed + RasterLds<S>::kLists);   // 10 per key
  uint32_t& sEnd = *reinterpret_cast<uint32_t*>(sSum + 10 * (kKeys + 1));
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const PixelMap pm = pixel_of_thread<S>(cam, tile, tid);
  const int x = pm.x, y = pm.y;
  const bool inside = x < cam.W && y < cam.H;
  const float px = (float)x + 0.5f, py = (float)y + 0.5f;
  // the tile's range and the block's largest end are the same in every
  // lane; read through readfirstlane so the compiler keeps the key indices
  // and the visit masks derived from them in scalar registers (as LDS and
  // global loads they would count as per-lane values, and every mask
  // operation of the visit loop would run on the VALU)
  const uint2 rg = b.ranges[tile];
  const uint32_t s = __builtin_amdgcn_readfirstlane(rg.x);
  const int64_t pi = (int64_t)y * cam.W + x;
  // The words of the last visit wait in the wave's scratch until the next
  // visit (or the end of the tile); before the first visit they are zeros,
  // which add nothing.
  const WaveRed<AccT> red(sRed + wv * (5 * kRedStride / 4), lane);
  {
    const AccT z[5] = {};
    red.write(z);
  }
  if constexpr (kAccum == 0)
    for (int k = wv * 10 * kPart + lane; k < (wv + 1) * 10 * kPart; k += 64) sSum[k] = 0u;
  int lastKey = 0;                           // fixed: of the group this lane adds for
  const int keyFrom = 4 * 16 * (lane & 3);   // a lane of it, as ds_bpermute counts
  uint32_t lastId = 0;                       // f32: the Gaussian of the last visit
  uint8_t* const lists = sList + wv * kGroups * kKeys;        // the wave's
  const uint8_t* const list = lists + (lane >> 4) * kKeys;    // this lane's group's
  float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float Ta = 0.0f;
  uint32_t myEnd = s;
  if (in) {   // the forward of this launch left them in registers
    g = in->g;
    if (g.w != 0.0f) {
      Ta = in->T;
      myEnd = in->end;
    }
  } else if (inside) {
    g = b.gC[pi];
    if (g.w != 0.0f) {
      Ta = b.T[pi];
      myEnd = b.end[pi];
    }
  }
  if (tid == 0) {
    sEnd = s;
    sA[kKeys] = sB[kKeys] = sC[kKeys] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);   // alpha 0: no lane takes it
  }
  __syncthreads();
  if (myEnd > s) atomicMax(&sEnd, myEnd);
  __syncthreads();
  const uint32_t endMax = __builtin_amdgcn_readfirstlane(sEnd);
  // this wave's largest end: keys at or past it are past every lane's end,
  // so the wave leaves them out of its visit set (they would add nothing)
  uint32_t we = myEnd;
  for (int o = 32; o > 0; o >>= 1) we = max(we, (uint32_t)__shfl_xor((int)we, o));
  const uint32_t waveEnd = __builtin_amdgcn_readfirstlane(we);
  const float gC[3] = {g.x, g.y, g.z};
  // GS_ACCUM_FIXED: the x16384 fixed-point scale rides on dL/dC from the
  // start, so on every product with it (dot(gC, c), dot(gC, S), galpha) and
  // on every term, which carries galpha or gC. Scaling by a power of two is
  // exact, so each scaled value equals the value times 16384 bit for bit;
  // the only exceptions are values whose unscaled form is subnormal, and
  // terms that small truncate to zero either way.
  constexpr float kS = kAccum == 0 ? kFixed : 1.0f;
  const float gCs[3] = {gC[0] * kS, gC[1] * kS, gC[2] * kS};
  // 16384 dot(gC, S) of the colour-behind sum S, which enters only through it
  float GS = fmaf(gCs[2], cam.bg[2], fmaf(gCs[1], cam.bg[1], gCs[0] * cam.bg[0])) * Ta;
  // fixed: this wave's part of the last batch's sums to the Gaussians' accumulators
  const auto flush = [&]() {
    if constexpr (kAccum == 0) {
#pragma unroll 1
      for (int k = 10 * kPart * wv + lane; k < 10 * kPart * (wv + 1); k += 64) {
        const uint32_t v = sSum[k];
        if (v != 0u) {
          sSum[k] = 0u;
          const uint32_t key = __umul24((uint32_t)k, 6554u) >> 16;   // k / 10 for k < 16384
          const uint32_t id = __float_as_uint(sB[key].w);
          atomicAdd((uint32_t*)accum + (uint64_t)id * 12 + ((uint32_t)k - __umul24(key, 10u)), v);
        }
      }
    }
  };
  // One visit, straight-line for all 64 lanes: the record at LDS offset
  // offset() from the three arrays' starts a0, b0 and c0 (behind the reads of
  // the previous visit's words); before(): the key lies before this lane's end. Lanes that do not take the splat (outside the
  // image, past their `end`, outside the cutoff, alpha below A_MIN, their
  // group past its list) keep their state and contribute zero terms. Some
  // lane took the splat in the forward, so there is nothing to vote on.
  // add(w8): the previous visit's words to its sums; ready(): ahead of this
  // visit's reduction. Returns the record's id.
  const auto visit = [&](const float4* a0, const float4* b0, const float4* c0, auto&& offset, auto&& before,
                         auto&& add, auto&& ready) __attribute__((always_inline)) {
    AccT w8[8];
    red.read(w8);   // the previous visit's words
    const uint32_t jo = offset();
    const float4 a = lds_at<float4>(a0, jo);
    const float4 bb = lds_at<float4>(b0, jo);   // C, opa*comp, -0.5 cnorm, id
    const float dx = px - a.x, dy = py - a.y;
    const float cA = a.z, cB = a.w, cC = bb.x;
    const float t2 = fmaf(cC * dy, dy, (cA * dx) * dx);
    // clamped to [0, 87] as in the forward pass
    const float e = clamp_e(fmaf(0.5f, t2, (cB * dx) * dy));
    const float G = gs_expf_raster(-e);
    const float araw = bb.y * G;
    const float alpha = fminf(0.99f, araw);
    const bool contrib = before() && e <= cut.eCut && alpha >= cut.aMin;
    const float4 c4 = lds_at<float4>(c0, jo);
    // Tb = Ta / (1 - alpha), S / (1 - alpha) through one reciprocal.
    // 1 - alpha lies in [0.0099, 1] (alpha in [0, 0.99]); on [2^-9, 1]
    // v_rcp_f32 refined by one FMA Newton step equals the correctly
    // rounded 1/x for every float (checked exhaustively on gfx950). A
    // lane that does not take the splat has alpha 0 here: its reciprocal
    // is exactly 1, so Tb = Ta and aT = 0 without a select each.
    const float alphaE = contrib ? alpha : 0.0f;
    const float rom = rcp_exact_unit(1.0f - alphaE);
    const float Tb = Ta * rom;
    add(w8);
    const float gcol = fmaf(gCs[2], c4.z, fmaf(gCs[1], c4.y, gCs[0] * c4.x));   // scaled
    // Every term is a product with galpha or aT, which are zero for the
    // lanes that do not take the splat (all other factors are finite).
    const float galphaS = (contrib && !(araw > 0.99f)) ? fmaf(gcol, Tb, -(GS * rom)) : 0.0f;
    const float aT = alphaE * Tb;
    const float ga = galphaS * araw;
    const float gq = ga * bb.z;
    const float gqdx = gq * dx;
    float v[10];
    v[0] = ga * (cA * dx + cB * dy);
    v[1] = ga * (cB * dx + cC * dy);
    v[2] = gqdx * dx;
    v[3] = 2.0f * (gqdx * dy);        // the middle conic term is 2 gq dx dy
    v[4] = (gq * dy) * dy;
    v[5] = galphaS * c4.w * G;
    v[6] = ga * (1.0f - c4.w);
    v[7] = gCs[0] * aT;
    v[8] = gCs[1] * aT;
    v[9] = gCs[2] * aT;
    GS = fmaf(gcol, aT, GS);
    Ta = Tb;
    AccT cur[10];
    if constexpr (kAccum == 0) {
      // i32(clamp(v * 16384, -1e9, 1e9)) per pixel; v already carries the
      // scale. Terms beyond the clamp are rare, so one test of the largest
      // magnitude stands for the clamps of the seven terms that carry
      // galpha (they are NaN together, and then so is the maximum; a NaN
      // converts to the lower clamp).
      const float m = max3abs(max3abs(max3abs(v[0], v[1], v[2]), v[3], v[4]), v[5], v[6]);
      if (wave_ballot(!(m <= 1.0e9f)) != 0ull) {
#pragma unroll
        for (int q = 0; q < 7; q++) v[q] = fminf(fmaxf(v[q], -1.0e9f), 1.0e9f);
      }
#pragma unroll
      for (int q = 0; q < 10; q++)
        cur[q] = (q >= 7 && kClampColour) ? (uint32_t)(int32_t)fminf(fmaxf(v[q], -1.0e9f), 1.0e9f)
                                           : (uint32_t)(int32_t)v[q];
    } else {
#pragma unroll
      for (int q = 0; q < 10; q++) cur[q] = v[q];
    }
    ready();
    AccT h[5];
    row_halve<AccT>(cur, h);
    red.write(h);
    return __float_as_uint(bb.w);
  };
  // batches start at multiples of 64 keys from s, so that their chunks are
  // the forward's chunks
  for (uint32_t hi = endMax; hi > s; ) {
    const uint32_t lo = s + (hi - s - 1u) / kKeys * kKeys;
    const int n = (int)(hi - lo);
    // lane 4 c + q: this wave's word of chunk c and group q (those of chunks
    // that the wave did not reach may be stale)
    const uint32_t first = lo + 64u * (uint32_t)(lane / kGroups);   // the chunk's first key
    uint64_t words = 0ull;
    if (lane < kKeys / 64 * kGroups && first < waveEnd) {
      words = b.took[took_word<S>(s, tile, ((lo - s) >> 6) + (uint32_t)(lane / kGroups)) + wv * kGroups + lane % kGroups];
      if (waveEnd - first < 64u) words &= (1ull << (waveEnd - first)) - 1ull;
    }
    __syncthreads();   // the last batch's visits are done
    if (hi != endMax) flush();
#pragma unroll 1
    for (int p0 = wv * kPart; p0 < (wv + 1) * kPart && p0 < n; p0 += 64) {
      const int j = p0 + lane;
      const uint64_t* tw = b.took + took_word<S>(s, tile, ((lo - s) >> 6) + (uint32_t)(p0 >> 6));
      const uint64_t word = lane < kWords ? tw[lane] : 0ull;
      // keys that some block of the tile took: only these are loaded
      const uint64_t any = ((uint64_t)or_lanes<kWords>((uint32_t)(word >> 32)) << 32) | or_lanes<kWords>((uint32_t)word);
      if (lane < kPart && j < n && ((any >> (j & 63)) & 1ull) != 0ull) {
        const uint32_t id = b.ids[lo + (uint32_t)j] & kIdMask;
        if (b.recFmt == 0) {
          const float4 r1 = b.rec[4 * id + 1];
          sA[j] = b.rec[4 * id + 0];
          sC[j] = b.rec[4 * id + 2];
          sB[j] = make_float4(r1.x, r1.y, b.rec[4 * id + 3].y, __uint_as_float(id));
        } else {
          const float4 r1 = b.rec[3 * id + 1];
          const float4 d = b.rec[3 * id + 2];   // comp, -0.5 cnorm, 1 - opa, opa
          sA[j] = b.rec[3 * id + 0];
          sC[j] = record_colour(b.recFmt, r1, d.w);
          sB[j] = make_float4(r1.x, r1.y, d.y, __uint_as_float(id));
        }
      }
    }
    __syncthreads();
    const int pastEnd = (int)(myEnd - lo);   // this lane's end as an index of the batch
    if constexpr (kAccum == 0) {
      // each group's keys, last one first, then the record that nobody takes
      constexpr uint32_t kNone = 0x01010101u * (uint32_t)kKeys;
      int have[kGroups] = {};
      for (int k = lane; k < kGroups * kKeys / 8; k += 64)
        reinterpret_cast<uint2*>(lists)[k] = make_uint2(kNone, kNone);
#pragma unroll
      for (int c = kKeys / 64 - 1; c >= 0; c--) {
#pragma unroll
        for (int q = 0; q < kGroups; q++) {
          const uint32_t mLo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)words, kGroups * c + q);
          const uint32_t mHi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(words >> 32), kGroups * c + q);
          const uint64_t m = ((uint64_t)mHi << 32) | mLo;
          const int cnt = __builtin_popcountll(m);
          const uint32_t below = __builtin_amdgcn_mbcnt_hi(mHi, __builtin_amdgcn_mbcnt_lo(mLo, 0u));
          if (__builtin_amdgcn_inverse_ballot_w64(m))
            lists[kKeys * q + have[q] + cnt - 1 - (int)below] = (uint8_t)(64 * c + lane);
          have[q] += cnt;
        }
      }
      const int steps = max(max(have[0], have[1]), max(have[2], have[3]));
      if (steps != 0) {
        int nextKey = (int)list[0];
        for (int step = 0; step < steps; step++) {
          int key = 0;
          visit(sA, sB, sC,
                [&]() {
                  key = nextKey;
                  nextKey = (int)list[step + 1 < kKeys ? step + 1 : 0];
                  return (uint32_t)key * 16u;
                },
                [&]() { return key < pastEnd; },
                [&](const AccT* w8) { add_group_sums(sSum, lastKey, red.slot, red.total(w8), red.flusher); },
                // the next key has arrived by now: waited for here, not behind the writes
                [&]() { asm volatile("" : "+v"(nextKey)); });
          lastKey = __builtin_amdgcn_ds_bpermute(keyFrom, key);
        }
      }
      // the last visit's words, while its batch is staged
      AccT w8[8];
      red.read(w8);
      add_group_sums(sSum, lastKey, red.slot, red.total(w8), red.flusher);
      const AccT z[5] = {};
      red.write(z);
    } else {
      // the keys that some group of the wave took, last one first
#pragma unroll 1
      for (int c = kKeys / 64 - 1; c >= 0; c--) {
        uint32_t mLo = 0u, mHi = 0u;
#pragma unroll
        for (int q = 0; q < kGroups; q++) {
          mLo |= (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)words, kGroups * c + q);
          mHi |= (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(words >> 32), kGroups * c + q);
        }
        uint64_t m = ((uint64_t)mHi << 32) | mLo;
        const int past = pastEnd - 64 * c;
        while (m) {
          const int bit = 63 - __builtin_clzll(m);
          clear_bit(m, bit);
          const uint32_t id =
              visit(sA + 64 * c, sB + 64 * c, sC + 64 * c, [&]() { return lds_offset((uint32_t)bit * 16u); },
                    [&]() { return bit < past; },
                    [&](const AccT* w8) {
                      add_wave_sums((float*)accum, lastId, red.slot, red.wave_total(w8), red.flusher && (lane & 3) == 0);
                    },
                    [] {});
          lastId = id;
        }
      }
    }
    hi = lo;
  }
  if constexpr (kAccum == 0) {
    __syncthreads();
    if (endMax > s) flush();
  } else {
    AccT w8[8];
    red.read(w8);
    add_wave_sums((float*)accum, lastId, red.slot, red.wave_total(w8), red.flusher && (lane & 3) == 0);
  }
}

template <class S, int kLoss>
__global__ __launch_bounds__(S::kThreads) void k_raster_fwd(Cam cam, Cut cut, RasterBufs b) {
  __shared__ float4 lds[RasterLds<S>::kFwd];
  raster_fwd_tile<S, kLoss, kLoss == 2 ? kTookGroups : kTookNone>(cam, cut, b, tile_of_block(b), lds);
}

template <class S, int kAccum, bool kClampColour>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu(S::kBwdWavesPerEU))) void k_raster_bwd(Cam cam, Cut cut, RasterBufs b, void* accum) {
  __shared__ float4 lds[RasterLds<S>::kBwd];
  raster_bwd_tile<S, kAccum, kClampColour>(cam, cut, b, accum, tile_of_block(b), lds);
}

// A training step's forward with the Charbonnier loss and its backward in
// one launch: the loss gradient of a pixel needs only that pixel, so each
// block runs the backward of its tile right after the forward (each thread
// keeps its pixel's T, end and dL/dC in registers; they are stored too,
// for the debug readbacks).
template <class S, int kAccum, bool kClampColour>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu(S::kBwdWavesPerEU))) void k_raster_fwd_bwd(Cam cam, Cut cut, RasterBufs b, void* accum) {
  __shared__ float4 lds[RasterLds<S>::kBoth];   // the two passes' layouts share it
  const int tile = tile_of_block(b);
  PixelState ps;
  raster_fwd_tile<S, 1, kAccum == 0 ? kTookGroups : kTookWaves>(cam, cut, b, tile, lds, &ps);
  __syncthreads();   // the forward's last LDS reads are done
  raster_bwd_tile<S, kAccum, kClampColour>(cam, cut, b, accum, tile, lds, &ps);
}

// ---- several views in one persistent launch ----
// Work item w in [0, off[V]) is tile tileOrder_v[w - off[v]] of the view v
// with off[v] <= w < off[v + 1]: each view's tiles in its own heaviest-first
// order, the views one after another. Each block takes the next item from
// the queue counter (zeroed before the launch) until the items run out, so
// every block leaves once the counter passes off[V].
struct ViewItem {
  int v;
  int tile;
};

__device__ __forceinline__ bool next_item(const ViewBlock* __restrict__ vb, uint32_t* queue, ViewItem& it) {
  __shared__ uint32_t sWork;
  __syncthreads();   // the previous item's LDS reads are done
  if (threadIdx.x == 0) sWork = atomicAdd(queue, 1u);
  __syncthreads();
  const uint32_t w = __builtin_amdgcn_readfirstlane(sWork);
  const int V = vb->count;
  if (w >= vb->off[V]) return false;
  int v = 0;
  while (w >= vb->off[v + 1]) v++;
  it.v = v;
  it.tile = (int)gs_global(vb->bufs[v].tileOrder)[w - vb->off[v]];
  return true;
}

// Forward with the Charbonnier loss and backward of every view's tiles in
// one persistent launch: each work item's tile runs both passes back to
// back, as k_raster_fwd_bwd does for one view.
template <class S, int kAccum, bool kClampColour>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu(S::kBwdWavesPerEU))) void
k_raster_fwd_bwd_views(const ViewBlock* __restrict__ vb, Cut cut, uint32_t* queue) {
  __shared__ float4 lds[RasterLds<S>::kBoth];
  ViewItem it;
  while (next_item(vb, queue, it)) {
    // read in place (the block is read-only here): copies held every camera
    // and buffer field in scalar registers across the whole tile and spilled
    // some of them. The buffers' pointers stay generic (flat accesses): a
    // copy with each loaded as a global pointer (global_bufs) took 0.2-0.4%
    // longer.
    const Cam& cam = vb->cams[it.v];
    const RasterBufs& b = vb->bufs[it.v];
    PixelState ps;
    raster_fwd_tile<S, 1, kAccum == 0 ? kTookGroups : kTookWaves>(cam, cut, b, it.tile, lds, &ps);
    __syncthreads();   // the forward's last LDS reads are done
    raster_bwd_tile<S, kAccum, kClampColour>(cam, cut, b, gs_global(vb->accum[it.v]), it.tile, lds, &ps);
  }
}

// one view of a batched step, one block per tile (camera and buffers from
// device memory), forward with the loss and backward in one launch
template <class S, int kAccum, bool kClampColour>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu(S::kBwdWavesPerEU))) void k_raster_fwd_bwd_view(const ViewBlock* __restrict__ vb, int v,
                                                                     Cut cut) {
  const Cam cam = vb->cams[v];
  const RasterBufs b = global_bufs(vb->bufs[v]);
  __shared__ float4 lds[RasterLds<S>::kBoth];
  const int tile = tile_of_block(b);
  PixelState ps;
  raster_fwd_tile<S, 1, kAccum == 0 ? kTookGroups : kTookWaves>(cam, cut, b, tile, lds, &ps);
  __syncthreads();
  raster_bwd_tile<S, kAccum, kClampColour>(cam, cut, b, gs_global(vb->accum[v]), tile, lds, &ps);
}

// f(Shape<tile, batch>{}) for a supported shape (checked by the callers)
template <int kT, typename F>
static void with_batch(int batch, F&& f) {
  if (batch == 64) f(Shape<kT, 64>{});
  else if (batch == 128) f(Shape<kT, 128>{});
  else f(Shape<kT, 256>{});
}

template <typename F>
static void with_shape(const RasterShape& sh, F&& f) {
  if (sh.tile == 8) with_batch<8>(sh.batch, f);
  else if (sh.tile == 32) with_batch<32>(sh.batch, f);
  else with_batch<16>(sh.batch, f);
}

size_t raster_took_bytes(int tile, int w, int h, int64_t keys) {
  // rows of one word per 4x4 pixels, up to took_word's last
  const size_t tiles = (size_t)((w + tile - 1) / tile) * (size_t)((h + tile - 1) / tile);
  return ((size_t)keys / 64 + tiles + 1) * (size_t)(tile * tile / 16) * 8;
}

bool raster_shape_ok(int tile, int batch) {
  return (tile == 8 || tile == 16 || tile == 32) && (batch == 64 || batch == 128 || batch == 256);
}

void launch_raster_fwd_bwd_view(hipStream_t st, const RasterShape& sh, const ViewBlock* vb, int v, int numTiles,
                                const Cut& cut, int accumMode, bool boundedColourGrad) {
  with_shape(sh, [&](auto shape) {
    using S = decltype(shape);
    if (accumMode != 0) k_raster_fwd_bwd_view<S, 1, true><<<numTiles, S::kThreads, 0, st>>>(vb, v, cut);
    else if (boundedColourGrad) k_raster_fwd_bwd_view<S, 0, false><<<numTiles, S::kThreads, 0, st>>>(vb, v, cut);
    else k_raster_fwd_bwd_view<S, 0, true><<<numTiles, S::kThreads, 0, st>>>(vb, v, cut);
  });
}

void launch_raster_fwd(hipStream_t st, const RasterShape& sh, const Cam& cam, const Cut& cut, const RasterBufs& b,
                       int loss) {
  const dim3 grid((unsigned)cam.numTiles);
  with_shape(sh, [&](auto shape) {
    using S = decltype(shape);
    if (loss == 1) k_raster_fwd<S, 1><<<grid, S::kThreads, 0, st>>>(cam, cut, b);
    else if (loss == 2) k_raster_fwd<S, 2><<<grid, S::kThreads, 0, st>>>(cam, cut, b);
    else k_raster_fwd<S, 0><<<grid, S::kThreads, 0, st>>>(cam, cut, b);
  });
}

void launch_raster_bwd(hipStream_t st, const RasterShape& sh, const Cam& cam, const Cut& cut, const RasterBufs& b,
                       int accumMode, void* accum, bool boundedColourGrad) {
  const dim3 grid((unsigned)cam.numTiles);
  with_shape(sh, [&](auto shape) {
    using S = decltype(shape);
    if (accumMode != 0) k_raster_bwd<S, 1, true><<<grid, S::kThreads, 0, st>>>(cam, cut, b, accum);
    else if (boundedColourGrad) k_raster_bwd<S, 0, false><<<grid, S::kThreads, 0, st>>>(cam, cut, b, accum);
    else k_raster_bwd<S, 0, true><<<grid, S::kThreads, 0, st>>>(cam, cut, b, accum);
  });
}

void launch_raster_fwd_bwd(hipStream_t st, const RasterShape& sh, const Cam& cam, const Cut& cut, const RasterBufs& b,
                           int accumMode, void* accum, bool boundedColourGrad) {
  const dim3 grid((unsigned)cam.numTiles);
  with_shape(sh, [&](auto shape) {
    using S = decltype(shape);
    if (accumMode != 0) k_raster_fwd_bwd<S, 1, true><<<grid, S::kThreads, 0, st>>>(cam, cut, b, accum);
    else if (boundedColourGrad) k_raster_fwd_bwd<S, 0, false><<<grid, S::kThreads, 0, st>>>(cam, cut, b, accum);
    else k_raster_fwd_bwd<S, 0, true><<<grid, S::kThreads, 0, st>>>(cam, cut, b, accum);
  });
}

void launch_raster_fwd_bwd_views(hipStream_t st, const RasterShape& sh, const ViewBlock* vb, const Cut& cut,
                                 int accumMode, bool boundedColourGrad, uint32_t* queue, int blocks) {
  with_shape(sh, [&](auto shape) {
    using S = decltype(shape);
    if (accumMode != 0) k_raster_fwd_bwd_views<S, 1, true><<<blocks, S::kThreads, 0, st>>>(vb, cut, queue);
    else if (boundedColourGrad) k_raster_fwd_bwd_views<S, 0, false><<<blocks, S::kThreads, 0, st>>>(vb, cut, queue);
    else k_raster_fwd_bwd_views<S, 0, true><<<blocks, S::kThreads, 0, st>>>(vb, cut, queue);
  });
}

// blocks of the persistent launches of one shape: as many as fit on the
// device at once
int raster_views_blocks(int device, const RasterShape& sh) {
  int cus = 0, per = 1;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) cus = 256;
  with_shape(sh, [&](auto shape) {
    using S = decltype(shape);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_raster_fwd_bwd_views<S, 0, false>, S::kThreads, 0) !=
        hipSuccess)
      per = 1;
  });
  if (per < 1) per = 1;
  return cus * per;
}

}  // namespace gs
