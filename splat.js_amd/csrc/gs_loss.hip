// gs_loss.hip — L1 + lambda * D-SSIM loss (textbook; the reference trains
// with Charbonnier only, shaders.js:11-12).
//
//   L = sum over valid pixels p and channels c of
//       (1 - lambda) |x - y| + lambda (1 - ssim_c(p))
//   x = gain * C + bias (rendered, exposure-adjusted), y = target
//   ssim (Wang et al. 2004): 11x11 Gaussian window, sigma 1.5, C1 = 0.01^2,
//   C2 = 0.03^2, zero padding outside the image. An invalid target pixel
//   (undistortion border, alpha byte 0) enters every window as zero in both
//   images, like the padding, so the loss does not depend on what is
//   rendered there and its dL/dC is zero, as its valid flag (gC.w = 0) tells
//   the backward pass.
//
// Two LDS-tiled passes over 32x16 pixel tiles with a 5-pixel halo:
//   k_ssim_fwd  blurs x, y, x^2, y^2, xy (separable: 26 rows x 32 columns
//               horizontally, then 32 x 16 vertically), forms ssim and its
//               partials A = dS/dmu_x - 2 mu_x dS/dvar_x - mu_y dS/dcov,
//               B = dS/dvar_x, Cm = dS/dcov (zero at invalid pixels), and
//               accumulates the loss.
//   k_ssim_bwd  blurs A, B, Cm back (the window is symmetric) and forms
//               dL/dx = (1 - lambda) sign(x - y) - lambda (A~ + 2 x B~ + y Cm~),
//               dL/dC = gain * dL/dx.
// A block gives two waves to each colour channel. A thread blurs eight
// columns of a row from 18 inputs it holds, then four rows of a column from
// 14, and asks for all its global inputs before it uses the first. A thread
// per output over 16x16 tiles read 11 inputs for each, through the LDS, and a
// halo of 1.6 pixels per pixel instead of 1.1: at 1237x933 the passes took 75
// and 58 us, now 58 and 43; at 320x240 13.3 and 10.8, now 10.8 and 7.1. Half
// of that is issued instructions (1470 per thread, forward), half the latency
// of five stages that wait for each other at 18 waves per CU.
// Every sum adds its taps in ascending order, as a thread per output would.
#include <cmath>

#include "gs_kernels.h"

namespace gs {

// The loss kernels' own image tiling (independent of the raster's tiles):
// 32 x 16 pixels per block, with a 5-pixel halo for the 11-tap windows.
constexpr int kTileX = 32, kTileY = 16;
constexpr int kTaps = 11, kHalo = kTaps / 2;
constexpr int kRegX = kTileX + 2 * kHalo, kRegY = kTileY + 2 * kHalo;   // 42 x 26 with the halo
constexpr int kInW = 44;                        // words per input row in LDS (16-byte aligned)
constexpr int kOutX = 8, kOutY = 4;             // outputs per thread of the horizontal, vertical blur
constexpr int kChThreads = 128;                 // threads per channel
constexpr int kLossThreads = 3 * kChThreads;
constexpr int kLoads = (kRegX * kRegY + kLossThreads - 1) / kLossThreads;   // input pixels per thread
static_assert(kRegY * (kTileX / kOutX) <= kChThreads, "a row's column group per thread");
static_assert(kTileX * (kTileY / kOutY) == kChThreads, "a column's row group per thread");

__host__ __device__ __forceinline__ int ssim_tiles_x(const Cam& cam) { return (cam.W + kTileX - 1) / kTileX; }

struct SsimWin {
  float g[kHalo + 1];   // tap q and tap 10 - q: g[min(q, 10 - q)]
};

// the taps as vector registers: an instruction with a scalar operand issues
// at half the rate
__device__ __forceinline__ void load_taps(const SsimWin& win, float (&w)[kHalo + 1]) {
#pragma unroll
  for (int q = 0; q <= kHalo; q++) {
    w[q] = win.g[q];
    asm("" : "+v"(w[q]));
  }
}
__device__ __forceinline__ float tap(const float (&w)[kHalo + 1], int q) { return w[q <= kHalo ? q : kTaps - 1 - q]; }

// v / 255 for v = 0..255, rounded as the division is (every value checked)
__device__ __forceinline__ float unorm8(uint32_t v) {
  const float f = (float)v, q = f * (1.0f / 255.0f);
  return fmaf(fmaf(-q, 255.0f, f), 1.0f / 255.0f, q);
}

__device__ __forceinline__ void load_xy(const Cam& cam, const RasterBufs& b, int gx, int gy, float* x,
                                        float* y, bool& valid) {
  valid = false;
  for (int c = 0; c < 3; c++) { x[c] = 0.0f; y[c] = 0.0f; }
  if (gx < 0 || gy < 0 || gx >= cam.W || gy >= cam.H) return;
  const int64_t pi = (int64_t)gy * cam.W + gx;
  const uint32_t pk = b.tgt[cam.tgtOffset + pi];
  const float4 o = b.img[pi];
  valid = (pk >> 24) != 0u;
  if (!valid) return;
  const float oc[3] = {o.x, o.y, o.z};
  for (int c = 0; c < 3; c++) {
    x[c] = cam.gain * oc[c] + cam.bias;
    y[c] = unorm8((pk >> (8 * c)) & 0xffu);
  }
}

// 18 consecutive LDS words (16-byte aligned)
__device__ __forceinline__ void load_row(const float* p, float (&v)[kOutX + kTaps - 1]) {
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const float4 q = *(const float4*)(p + 4 * k);
    v[4 * k] = q.x; v[4 * k + 1] = q.y; v[4 * k + 2] = q.z; v[4 * k + 3] = q.w;
  }
  const float2 q = *(const float2*)(p + 16);
  v[16] = q.x; v[17] = q.y;
}

__device__ __forceinline__ void store_row(float* p, const float (&v)[kOutX]) {
  *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
  *(float4*)(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}

// Word of row r in a blurred plane of kRegY x kTileX words. The two row
// groups of a wave read rows four apart, 128 words: swapping every second
// group's even and odd rows puts them in different halves of the banks.
__device__ __forceinline__ int blurred_row(int r) { return (r ^ ((r >> 2) & 1)) * kTileX; }

// Vertical blur of S planes: out[s][o] for the kOutY rows from row r0 (a
// multiple of kOutY) of column c.
template <int S>
__device__ __forceinline__ void blur_down(const float* planes, const float (&w)[kHalo + 1], int r0, int c,
                                          float (&out)[S][kOutY]) {
#pragma unroll
  for (int s = 0; s < S; s++)
#pragma unroll
    for (int o = 0; o < kOutY; o++) out[s][o] = 0.0f;
#pragma unroll
  for (int i = 0; i < kOutY + kTaps - 1; i++) {
    const float* p = planes + blurred_row(r0 + i) + c;
#pragma unroll
    for (int s = 0; s < S; s++) {
      const float v = p[s * kRegY * kTileX];
#pragma unroll
      for (int o = 0; o < kOutY; o++)
        if (i >= o && i - o < kTaps) out[s][o] = fmaf(tap(w, i - o), v, out[s][o]);
    }
  }
}

__global__ __launch_bounds__(kLossThreads) void k_ssim_fwd(Cam cam, SsimWin win, float lambda, RasterBufs b,
                                                           float* __restrict__ part) {
  // the inputs (x and y planes per channel), then, in their place, the
  // horizontal blurs of x, y, xx, yy, xy per channel
  constexpr int kIn = kRegY * kInW, kBl = kRegY * kTileX;
  __shared__ __align__(16) float lds[15 * kBl > 6 * kIn ? 15 * kBl : 6 * kIn];
  __shared__ double sStat[3][kLossThreads / 64];
  const int tid = threadIdx.x, ch = tid / kChThreads, ct = tid % kChThreads;
  const int tile = blockIdx.x;
  const int tx = tile % ssim_tiles_x(cam), ty = tile / ssim_tiles_x(cam);
  const int ox = tx * kTileX - kHalo, oy = ty * kTileY - kHalo;
  float w[kHalo + 1];
  load_taps(win, w);
  // every load of the block's inputs in flight before the first is used
  uint32_t pk[kLoads];
  float4 im[kLoads];
#pragma unroll
  for (int l = 0; l < kLoads; l++) {
    const int k = tid + l * kLossThreads, gx = ox + k % kRegX, gy = oy + k / kRegX;
    pk[l] = 0u;
    im[l] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (gx >= 0 && gy >= 0 && gx < cam.W && gy < cam.H && k < kRegX * kRegY) {
      const int64_t pi = (int64_t)gy * cam.W + gx;
      pk[l] = b.tgt[cam.tgtOffset + pi];
      im[l] = b.img[pi];
    }
  }
#pragma unroll
  for (int l = 0; l < kLoads; l++) {
    const int k = tid + l * kLossThreads, at = k / kRegX * kInW + k % kRegX;
    if (k >= kRegX * kRegY) break;
    const float oc[3] = {im[l].x, im[l].y, im[l].z};
    const bool v = (pk[l] >> 24) != 0u;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      lds[2 * q * kIn + at] = v ? cam.gain * oc[q] + cam.bias : 0.0f;
      lds[(2 * q + 1) * kIn + at] = v ? unorm8((pk[l] >> (8 * q)) & 0xffu) : 0.0f;
    }
  }
  // this thread's pixels: column lx, rows ly .. ly + 3 of the tile
  const int lx = ct % kTileX, ly = ct / kTileX * kOutY;
  const int px = tx * kTileX + lx, py = ty * kTileY + ly;
  bool valid[kOutY];
#pragma unroll
  for (int o = 0; o < kOutY; o++)
    valid[o] = px < cam.W && py + o < cam.H && (b.tgt[cam.tgtOffset + (int64_t)(py + o) * cam.W + px] >> 24) != 0u;
  __syncthreads();
  float xv[kOutY], yv[kOutY], h[5][kOutX];
  const int hr = ct / (kTileX / kOutX), hc = ct % (kTileX / kOutX) * kOutX;
  {
    const float* sx = lds + 2 * ch * kIn;
#pragma unroll
    for (int o = 0; o < kOutY; o++) {
      const int at = (ly + o + kHalo) * kInW + lx + kHalo;
      xv[o] = sx[at];
      yv[o] = sx[kIn + at];
    }
    if (hr < kRegY) {
      float vx[kOutX + kTaps - 1], vy[kOutX + kTaps - 1];
      load_row(sx + hr * kInW + hc, vx);
      load_row(sx + kIn + hr * kInW + hc, vy);
#pragma unroll
      for (int s = 0; s < 5; s++)
#pragma unroll
        for (int o = 0; o < kOutX; o++) h[s][o] = 0.0f;
#pragma unroll
      for (int i = 0; i < kOutX + kTaps - 1; i++) {
        const float v[5] = {vx[i], vy[i], vx[i] * vx[i], vy[i] * vy[i], vx[i] * vy[i]};
#pragma unroll
        for (int o = 0; o < kOutX; o++)
          if (i >= o && i - o < kTaps)
#pragma unroll
            for (int s = 0; s < 5; s++) h[s][o] = fmaf(tap(w, i - o), v[s], h[s][o]);
      }
    }
  }
  __syncthreads();
  float* bl = lds + 5 * ch * kBl;
  if (hr < kRegY)
#pragma unroll
    for (int s = 0; s < 5; s++) store_row(bl + s * kBl + blurred_row(hr) + hc, h[s]);
  __syncthreads();
  double st0 = 0.0, st1 = 0.0, st2 = 0.0;
  if (px < cam.W && py < cam.H) {
    const int64_t npx = (int64_t)cam.W * cam.H;
    const float C1 = 0.0001f, C2 = 0.0009f;
    float m[5][kOutY];
    blur_down<5>(bl, w, ly, lx, m);
#pragma unroll
    for (int o = 0; o < kOutY; o++) {
      if (py + o >= cam.H) break;
      const int64_t pi = (int64_t)(py + o) * cam.W + px;
      const float ux = m[0][o], uy = m[1][o];
      const float vx = m[2][o] - ux * ux, vy = m[3][o] - uy * uy, cxy = m[4][o] - ux * uy;
      const float N1 = 2.f * ux * uy + C1, N2 = 2.f * cxy + C2;
      const float D1 = ux * ux + uy * uy + C1, D2 = vx + vy + C2;
      const float S = (N1 * N2) / (D1 * D2);
      float A = 0.f, Bv = 0.f, Cv = 0.f;
      if (valid[o]) {
        const float err = xv[o] - yv[o];
        st0 += (double)(err * err);
        st1 += (double)((1.f - lambda) * fabsf(err) + lambda * (1.f - S));
        st2 += ch == 0 ? 1.0 : 0.0;
        const float dmx = (2.f * uy * N2) / (D1 * D2) - S * (2.f * ux) / D1;
        const float dvx = -S / D2;
        const float dcxy = 2.f * N1 / (D1 * D2);
        A = dmx - 2.f * ux * dvx - uy * dcxy;
        Bv = dvx;
        Cv = dcxy;
      }
      part[(int64_t)(3 * ch + 0) * npx + pi] = A;
      part[(int64_t)(3 * ch + 1) * npx + pi] = Bv;
      part[(int64_t)(3 * ch + 2) * npx + pi] = Cv;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    st0 += __shfl_xor(st0, o);
    st1 += __shfl_xor(st1, o);
    st2 += __shfl_xor(st2, o);
  }
  const int wv = tid >> 6;
  if ((tid & 63) == 0) { sStat[0][wv] = st0; sStat[1][wv] = st1; sStat[2][wv] = st2; }
  __syncthreads();
  if (tid < 3) {
    double v = 0.0;
    for (int k = 0; k < kLossThreads / 64; k++) v += sStat[tid][k];
    if (v != 0.0) atomicAdd(&stat_line(b.stats, blockIdx.x)[tid], v);
  }
}

__global__ __launch_bounds__(kLossThreads) void k_ssim_bwd(Cam cam, SsimWin win, float lambda, RasterBufs b,
                                                           const float* __restrict__ part) {
  // A, B and Cm per channel, then, in their place, their horizontal blurs,
  // then the gradients
  constexpr int kIn = kRegY * kInW, kBl = kRegY * kTileX;
  __shared__ __align__(16) float lds[9 * kIn];
  static_assert(9 * kBl <= 9 * kIn && 3 * kTileX * kTileY <= 9 * kIn, "the later stages fit");
  const int tid = threadIdx.x, ch = tid / kChThreads, ct = tid % kChThreads;
  const int tile = blockIdx.x;
  const int tx = tile % ssim_tiles_x(cam), ty = tile / ssim_tiles_x(cam);
  const int ox = tx * kTileX - kHalo, oy = ty * kTileY - kHalo;
  const int64_t npx = (int64_t)cam.W * cam.H;
  float w[kHalo + 1];
  load_taps(win, w);
  float v9[kLoads][9];
#pragma unroll
  for (int l = 0; l < kLoads; l++) {
    const int k = tid + l * kLossThreads, gx = ox + k % kRegX, gy = oy + k / kRegX;
    const bool in = gx >= 0 && gy >= 0 && gx < cam.W && gy < cam.H && k < kRegX * kRegY;
    const float* p = part + ((int64_t)gy * cam.W + gx);
#pragma unroll
    for (int s = 0; s < 9; s++) v9[l][s] = in ? p[(int64_t)s * npx] : 0.0f;
  }
  // this thread's pixels: column lx, rows ly .. ly + 3 of the tile
  const int lx = ct % kTileX, ly = ct / kTileX * kOutY;
  const int px = tx * kTileX + lx, py = ty * kTileY + ly;
  float xs[kOutY], ys[kOutY];
  bool valid[kOutY];
#pragma unroll
  for (int o = 0; o < kOutY; o++) {
    float x[3], y[3];
    load_xy(cam, b, px, py + o, x, y, valid[o]);
    xs[o] = ch == 0 ? x[0] : ch == 1 ? x[1] : x[2];
    ys[o] = ch == 0 ? y[0] : ch == 1 ? y[1] : y[2];
  }
#pragma unroll
  for (int l = 0; l < kLoads; l++) {
    const int k = tid + l * kLossThreads, at = k / kRegX * kInW + k % kRegX;
    if (k >= kRegX * kRegY) break;
#pragma unroll
    for (int s = 0; s < 9; s++) lds[s * kIn + at] = v9[l][s];
  }
  __syncthreads();
  float h[3][kOutX];
  const int hr = ct / (kTileX / kOutX), hc = ct % (kTileX / kOutX) * kOutX;
  if (hr < kRegY) {
#pragma unroll
    for (int s = 0; s < 3; s++) {
      float v[kOutX + kTaps - 1];
      load_row(lds + (3 * ch + s) * kIn + hr * kInW + hc, v);
#pragma unroll
      for (int o = 0; o < kOutX; o++) {
        h[s][o] = 0.0f;
#pragma unroll
        for (int q = 0; q < kTaps; q++) h[s][o] = fmaf(tap(w, q), v[o + q], h[s][o]);
      }
    }
  }
  __syncthreads();
  float* bl = lds + 3 * ch * kBl;
  if (hr < kRegY)
#pragma unroll
    for (int s = 0; s < 3; s++) store_row(bl + s * kBl + blurred_row(hr) + hc, h[s]);
  __syncthreads();
  float m[3][kOutY];
  blur_down<3>(bl, w, ly, lx, m);
  __syncthreads();
#pragma unroll
  for (int o = 0; o < kOutY; o++) {
    const float dssim = m[0][o] + 2.f * xs[o] * m[1][o] + ys[o] * m[2][o];
    const float err = xs[o] - ys[o];
    const float d = -lambda * dssim + (1.f - lambda) * (err > 0.f ? 1.f : (err < 0.f ? -1.f : 0.f));
    lds[(ch * kTileY + ly + o) * kTileX + lx] = valid[o] ? cam.gain * d : 0.0f;
  }
  __syncthreads();
  for (int k = tid; k < kTileX * kTileY; k += kLossThreads) {
    const int x = tx * kTileX + k % kTileX, y = ty * kTileY + k / kTileX;
    if (x >= cam.W || y >= cam.H) continue;
    const int64_t pi = (int64_t)y * cam.W + x;
    const bool v = (b.tgt[cam.tgtOffset + pi] >> 24) != 0u;
    b.gC[pi] = make_float4(lds[k], lds[kTileX * kTileY + k], lds[2 * kTileX * kTileY + k], v ? 1.0f : 0.0f);
  }
}

void launch_loss_l1ssim(hipStream_t st, const Cam& cam, float lambda, const RasterBufs& b, float* scratch) {
  SsimWin w;
  double g[kTaps], s = 0.0;
  for (int i = 0; i < kTaps; i++) {
    g[i] = std::exp(-((i - kHalo) * (i - kHalo)) / (2.0 * 1.5 * 1.5));
    s += g[i];
  }
  for (int i = 0; i <= kHalo; i++) w.g[i] = (float)(g[i] / s);
  const dim3 grid((unsigned)(ssim_tiles_x(cam) * ((cam.H + kTileY - 1) / kTileY)));
  k_ssim_fwd<<<grid, kLossThreads, 0, st>>>(cam, w, lambda, b, scratch);
  k_ssim_bwd<<<grid, kLossThreads, 0, st>>>(cam, w, lambda, b, scratch);
}

}  // namespace gs
