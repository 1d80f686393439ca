// gs_readback.hip — what the host reads: a rendered view, the statistics of a
// loss or PSNR read, and the Gaussians in the caller's layout (readGaussians,
// trainer.js:797-817): 16 floats and 3K coefficients per row, from the 16-byte
// planes. All are written over PCIe straight into pinned host memory.
//
// The device lays the rows out and decodes 16-bit coefficients, so that the
// host only has to copy whole blocks: its loop over the planes took 7 of the
// 17 ms of a 73 MB read. The writes are what bounds it (PCIe); the reads come
// from HBM at a fraction of its rate.
#include "gs_kernels.h"

namespace gs {

// rows [first, first + count): 4 threads per row, one 16-byte piece each
__global__ __launch_bounds__(kBlock) void k_param_rows(int64_t cap, int64_t first, int64_t count,
                                                      const float4* __restrict__ P, float4* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k < 4 * count) out[k] = P[(k & 3) * cap + first + (k >> 2)];
}

// one thread per coefficient: C = 3K of a row, from planes of 4 floats
// (kFmt 0) or of 8 bf16 or fp16 (1, 2)
template <int kFmt>
__global__ __launch_bounds__(kBlock) void k_sh_rows(int64_t cap, int64_t first, int64_t count, int C,
                                                   const void* __restrict__ SH, float* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k >= count * C) return;
  const uint32_t r = (uint32_t)k / (uint32_t)C, j = (uint32_t)k - r * (uint32_t)C;
  if constexpr (kFmt == 0) {
    out[k] = ((const float*)SH)[((j >> 2) * cap + first + r) * 4 + (j & 3u)];
  } else {
    const uint32_t b = ((const uint16_t*)SH)[((j >> 3) * cap + first + r) * 8 + (j & 7u)];
    out[k] = kFmt == 2 ? gs_h2f(b) : gs_bf2f(b);
  }
}

// One block: the statistics src into pinned memory, the loss window cleared
// (all but its dropped keys), and with a PSNR read also src and the camera
// gradient rows. What a copy and up to three memsets did in launches of their
// own, some 3 us each: four evaluated 979x546 views 469 -> 439 us.
__global__ __launch_bounds__(1024) void k_stats_read(double* src, double* window, double* __restrict__ out, bool clearSrc,
                                                     uint32_t* __restrict__ camGrad, int64_t camWords) {
  for (int i = threadIdx.x; i < kStatDoubles; i += 1024) {
    out[i] = src[i];
    if (clearSrc) src[i] = 0.0;
    if (i < kStatDropped) window[i] = 0.0;   // the same thread read it above where it is src
  }
  for (int64_t i = threadIdx.x; i < camWords; i += 1024) camGrad[i] = 0u;
}

void launch_stats_read(hipStream_t st, double* src, double* window, double* out, bool clearSrc, uint32_t* camGrad,
                       int64_t camWords) {
  k_stats_read<<<1, 1024, 0, st>>>(src, window, out, clearSrc, camGrad, camWords);
}

// pixels of a view as they are; PCIe bounds it
__global__ __launch_bounds__(kBlock) void k_pixels(int64_t count, const float4* __restrict__ img, float4* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k < count) out[k] = img[k];
}

void launch_pixels(hipStream_t st, int64_t count, const float4* img, float* out) {
  if (count <= 0) return;
  k_pixels<<<(unsigned)((count + kBlock - 1) / kBlock), kBlock, 0, st>>>(count, img, (float4*)out);
}

void launch_param_rows(hipStream_t st, int64_t cap, int64_t first, int64_t count, const float4* P, float* out) {
  if (count <= 0) return;
  k_param_rows<<<(unsigned)((4 * count + kBlock - 1) / kBlock), kBlock, 0, st>>>(cap, first, count, P, (float4*)out);
}

void launch_sh_rows(hipStream_t st, int fmt, int64_t cap, int64_t first, int64_t count, int C, const void* SH,
                    float* out) {
  const int64_t m = count * C;   // at most a pinned block's floats
  if (m <= 0) return;
  const unsigned g = (unsigned)((m + kBlock - 1) / kBlock);
  if (fmt == 0) k_sh_rows<0><<<g, kBlock, 0, st>>>(cap, first, count, C, SH, out);
  else if (fmt == 1) k_sh_rows<1><<<g, kBlock, 0, st>>>(cap, first, count, C, SH, out);
  else k_sh_rows<2><<<g, kBlock, 0, st>>>(cap, first, count, C, SH, out);
}

}  // namespace gs
