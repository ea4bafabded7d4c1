// image.hip — the output stage on the device, where the image already is:
// the 8-bit conversion the PNG writer applies (main.cpp:25-31) and the
// reference-free noise estimate NoiseStats (math/image.h:35-182).
//
// Every per-pixel value is the reference's float expression in its order
// (built with -ffp-contract=off, so nothing is fused): luminance, the 1-2-1
// blur of interior pixels (which never reach the clamped border), the
// gradient edge test and the two normalised residuals are bit-identical.
// The reference sums luminance and residuals in double in row order; here
// the sums are double too, in a tree order, so the float results can differ
// only where a double sum lands within its own rounding error of a float
// rounding boundary. The median and 95th percentile are selected exactly:
// the residuals are non-negative floats, whose bit patterns order like the
// values, and a three-pass radix select (11, 11 and 10 bits, both ranks at
// once) finds the k-th smallest pattern with k computed as the reference
// computes it. Nothing leaves the device until the result.
//
// NoiseStats is five launches. Bound at 1920x1080 by launches and their
// latency rather than by the 33 MB it moves: every work-group adds the few
// hundred partial results of the launch before itself instead of leaving
// that to a launch of one work-group, the first digit is counted where the
// keys are made, and a pass has at most 1024 work-groups, because each adds
// its counts to the same words and one address takes about 85 M atomics a
// second. 73 us of the device's time; 2048 work-groups, four 8-bit passes and a
// one-thread scan of each took 12 launches and 205 us.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <mutex>

#include "launch.h"

namespace xnh {
namespace {

constexpr int kImgThreads = 256;
constexpr uint32_t kNoKey = 0xFFFFFFFFu;   // above every non-negative float's bit pattern
constexpr int kImgHistWords = 2048 + 2 * 2048 + 2 * 1024;
static_assert(sizeof(ImgState::hist0) + sizeof(ImgState::hist1) + sizeof(ImgState::hist2) == 4 * kImgHistWords,
              "digit counts follow each other");

__device__ __forceinline__ double wave_sumd(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

__device__ __forceinline__ uint32_t wave_sumu(uint32_t v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// image.h:94-95: the running maximum starts at 0 and takes a value only if
// it compares greater (a NaN never does); combining partial maxima by the
// same rule gives the same result
__device__ __forceinline__ float gt_max(float m, float v) { return v > m ? v : m; }

__device__ __forceinline__ float wave_gt_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = gt_max(v, __shfl_xor(v, o));
  return v;
}

// std::max(a, b) returns b only when a < b
__device__ __forceinline__ float std_max(float a, float b) { return a < b ? b : a; }

// Block sums (kImgThreads threads); red holds one slot per wave.
__device__ double block_sumd(double v, double* red) {
  v = wave_sumd(v);
  const int w = static_cast<int>(threadIdx.x >> 6), nw = static_cast<int>(blockDim.x >> 6);
  if ((threadIdx.x & 63u) == 0u) red[w] = v;
  __syncthreads();
  double t = 0.0;
  for (int k = 0; k < nw; ++k) t += red[k];
  __syncthreads();
  return t;
}

__global__ void __launch_bounds__(kImgThreads) k_img_from_accum(const float4* accum, float inv_spp, int w, int h,
                                                                float* img) {
  // the swapchain layout (cpu_tiled.cpp:224-234): pixel row y goes to row h-1-y
  const int p = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (p >= w * h) return;
  const int y = p / w, x = p - y * w;
  const float4 a = accum[p];
  float* o = img + 3 * (static_cast<size_t>(h - 1 - y) * w + x);
  o[0] = a.x * inv_spp;
  o[1] = a.y * inv_spp;
  o[2] = a.z * inv_spp;
}

// image.h:127-135 and 137-146: luminance, and per-block double sums of it.
// Clears the digit counts of the passes that follow.
__global__ void __launch_bounds__(kImgThreads) k_img_lum(const float* img, int n, float* lum, double* part,
                                                         ImgState* st) {
  __shared__ double red[kImgThreads / 64];
  const int tid = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  const int stride = static_cast<int>(gridDim.x * blockDim.x);
  for (int k = tid; k < kImgHistWords; k += stride) st->hist0[k] = 0u;   // hist0, hist1 and hist2 follow each other
  double acc = 0.0;
  for (int i = tid; i < n; i += stride) {
    const float r = img[3 * static_cast<size_t>(i)], g = img[3 * static_cast<size_t>(i) + 1],
                b = img[3 * static_cast<size_t>(i) + 2];
    const float l = 0.2126f * r + 0.7152f * g + 0.0722f * b;
    lum[i] = l;
    acc += static_cast<double>(l);
  }
  const double t = block_sumd(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// image.h:51-57 (average luminance, edge threshold and epsilon, by every
// work-group in the same order) and image.h:63-98 for every interior pixel:
// the edge test, the residual
// against the blur and its two normalised forms. key[i] is the absolute
// form's bit pattern for a counted pixel, kNoKey otherwise; per block the
// double sums of both forms, the maximum and the count. The keys' first
// digits are counted on the way.
__global__ void __launch_bounds__(kImgThreads) k_img_resid(const float* lum, int w, int h, const double* part,
                                                           ImgState* st, uint32_t* key, double* part2, float* pmax,
                                                           uint32_t* pcnt) {
  __shared__ double red[kImgThreads / 64];
  __shared__ float redm[kImgThreads / 64];
  __shared__ uint32_t redc[kImgThreads / 64];
  __shared__ uint32_t lh[2048];
  const int n = w * h;
  double sum = 0.0;
  for (int k = static_cast<int>(threadIdx.x); k < static_cast<int>(gridDim.x); k += kImgThreads) sum += part[k];
  for (int k = static_cast<int>(threadIdx.x); k < 2048; k += kImgThreads) lh[k] = 0u;
  const float avg = static_cast<float>(block_sumd(sum, red) / static_cast<double>(n));
  const float edge = std_max(1e-6f, avg * 0.1f), eps = std_max(1e-8f, avg * avg * 1e-4f);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->avg = avg;
    st->edge = edge;
    st->eps = eps;
  }
  double s2 = 0.0, s1 = 0.0;
  float mx = 0.f;
  uint32_t cnt = 0u;
  for (int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); i < n;
       i += static_cast<int>(gridDim.x * blockDim.x)) {
    const int y = i / w, x = i - y * w;
    uint32_t k = kNoKey;
    if (x >= 1 && x < w - 1 && y >= 1 && y < h - 1) {
      const float gx = 0.5f * (lum[i + 1] - lum[i - 1]);
      const float gy = 0.5f * (lum[i + w] - lum[i - w]);
      const float grad = sqrtf(gx * gx + gy * gy);
      if (!(grad >= edge)) {
        // image.h:152-174 at an interior pixel: weights 1 2 1 / 2 4 2 / 1 2 1
        // summed row by row, left to right, then divided by 16
        float s = 0.f;
        s += 1.f * lum[i - w - 1];
        s += 2.f * lum[i - w];
        s += 1.f * lum[i - w + 1];
        s += 2.f * lum[i - 1];
        s += 4.f * lum[i];
        s += 2.f * lum[i + 1];
        s += 1.f * lum[i + w - 1];
        s += 2.f * lum[i + w];
        s += 1.f * lum[i + w + 1];
        const float bl = s / 16.f;
        const float r = lum[i] - bl;
        const float den = bl * bl + eps;
        const float q2 = (r * r) / den;
        const float q1 = fabsf(r) / sqrtf(den);
        s2 += static_cast<double>(q2);
        s1 += static_cast<double>(q1);
        mx = gt_max(mx, q1);
        ++cnt;
        k = __float_as_uint(q1);
        if (k != kNoKey) atomicAdd(&lh[k >> 21], 1u);
      }
    }
    key[i] = k;
  }
  const double t2 = block_sumd(s2, red);
  const double t1 = block_sumd(s1, red);
  const float wm = wave_gt_max(mx);
  const uint32_t wc = wave_sumu(cnt);
  const int wv = static_cast<int>(threadIdx.x >> 6), nw = static_cast<int>(blockDim.x >> 6);
  if ((threadIdx.x & 63u) == 0u) {
    redm[wv] = wm;
    redc[wv] = wc;
  }
  __syncthreads();
  for (int k = static_cast<int>(threadIdx.x); k < 2048; k += kImgThreads)
    if (lh[k]) atomicAdd(&st->hist0[k], lh[k]);
  if (threadIdx.x == 0) {
    float m = 0.f;
    uint32_t c = 0u;
    for (int k = 0; k < nw; ++k) {
      m = gt_max(m, redm[k]);
      c += redc[k];
    }
    part2[2 * blockIdx.x] = t2;
    part2[2 * blockIdx.x + 1] = t1;
    pmax[blockIdx.x] = m;
    pcnt[blockIdx.x] = c;
  }
}

// The digit whose count holds the given rank, and the rank within it (block
// of kImgThreads threads, kBins a multiple of that; every thread gets both).
struct Pick {
  uint32_t digit, rank;
};
template <int kBins>
__device__ Pick block_pick(const uint32_t* hist, uint32_t rank) {
  __shared__ uint32_t wsum[kImgThreads / 64];
  __shared__ Pick found;
  constexpr int per = kBins / kImgThreads;
  const int lane = static_cast<int>(threadIdx.x & 63u), wv = static_cast<int>(threadIdx.x >> 6);
  const int b0 = static_cast<int>(threadIdx.x) * per;
  uint32_t c[per], sum = 0u;
  for (int k = 0; k < per; ++k) {
    c[k] = hist[b0 + k];
    sum += c[k];
  }
  uint32_t inc = sum;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o);
    if (lane >= o) inc += t;
  }
  if (threadIdx.x == 0) found = Pick{0u, rank};
  if (lane == 63) wsum[wv] = inc;
  __syncthreads();
  uint32_t cum = inc - sum;
  for (int k = 0; k < wv; ++k) cum += wsum[k];
  for (int k = 0; k < per; ++k) {
    if (rank >= cum && rank < cum + c[k]) found = Pick{static_cast<uint32_t>(b0 + k), rank - cum};
    cum += c[k];
  }
  __syncthreads();
  const Pick r = found;
  __syncthreads();
  return r;
}

// image.h:100-118: totals, the three means, and the two ranks
// k = (size_t)(p * (float)(n - 1)) of image.h:176-186, their first digits, and
// the counts of the second digits of the keys that carry them.
__global__ void __launch_bounds__(kImgThreads) k_img_second(const uint32_t* key, int n, const double* part2,
                                                            const float* pmax, const uint32_t* pcnt, ImgState* st) {
  __shared__ double red[kImgThreads / 64];
  __shared__ float redm[kImgThreads / 64];
  __shared__ uint32_t redc[kImgThreads / 64];
  __shared__ uint32_t lh[2][2048];
  double s2 = 0.0, s1 = 0.0;
  float mx = 0.f;
  uint32_t cnt = 0u;
  for (int k = static_cast<int>(threadIdx.x); k < static_cast<int>(gridDim.x); k += kImgThreads) {
    s2 += part2[2 * k];
    s1 += part2[2 * k + 1];
    mx = gt_max(mx, pmax[k]);
    cnt += pcnt[k];
  }
  for (int k = static_cast<int>(threadIdx.x); k < 4096; k += kImgThreads) lh[k >> 11][k & 2047] = 0u;
  const double t2 = block_sumd(s2, red);
  const double t1 = block_sumd(s1, red);
  const float wm = wave_gt_max(mx);
  const uint32_t wc = wave_sumu(cnt);
  const int wv = static_cast<int>(threadIdx.x >> 6), nw = static_cast<int>(blockDim.x >> 6);
  if ((threadIdx.x & 63u) == 0u) {
    redm[wv] = wm;
    redc[wv] = wc;
  }
  __syncthreads();
  float m = 0.f;
  uint32_t c = 0u;
  for (int k = 0; k < nw; ++k) {
    m = gt_max(m, redm[k]);
    c += redc[k];
  }
  Pick p[2] = {{0u, 0u}, {0u, 0u}};
  if (c > 0u) {
    p[0] = block_pick<2048>(st->hist0, static_cast<uint32_t>(0.50f * static_cast<float>(c - 1u)));
    p[1] = block_pick<2048>(st->hist0, static_cast<uint32_t>(0.95f * static_cast<float>(c - 1u)));
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->count = c;
    st->max_abs = m;
    st->mean_sq = c > 0u ? static_cast<float>(t2 / static_cast<double>(c)) : 0.f;
    st->mean_abs = c > 0u ? static_cast<float>(t1 / static_cast<double>(c)) : 0.f;
    for (int t = 0; t < 2; ++t) {
      st->prefix[t] = p[t].digit;
      st->rank[t] = p[t].rank;
    }
  }
  for (int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); i < n;
       i += static_cast<int>(gridDim.x * blockDim.x)) {
    const uint32_t k = key[i];
    if (k == kNoKey) continue;
    for (int t = 0; t < 2; ++t)
      if ((k >> 21) == p[t].digit) atomicAdd(&lh[t][(k >> 10) & 2047u], 1u);
  }
  __syncthreads();
  for (int k = static_cast<int>(threadIdx.x); k < 4096; k += kImgThreads)
    if (lh[k >> 11][k & 2047]) atomicAdd(&st->hist1[k >> 11][k & 2047], lh[k >> 11][k & 2047]);
}

// The second digits, and the counts of the last ten bits of the keys that
// carry both. prefix and rank of st are the first digit's (written by the
// launch before).
__global__ void __launch_bounds__(kImgThreads) k_img_third(const uint32_t* key, int n, ImgState* st) {
  __shared__ uint32_t lh[2][1024];
  for (int k = static_cast<int>(threadIdx.x); k < 2048; k += kImgThreads) lh[k >> 10][k & 1023] = 0u;
  uint32_t pre[2] = {0u, 0u};
  if (st->count > 0u)
    for (int t = 0; t < 2; ++t) pre[t] = (st->prefix[t] << 11) | block_pick<2048>(st->hist1[t], st->rank[t]).digit;
  __syncthreads();
  for (int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); i < n;
       i += static_cast<int>(gridDim.x * blockDim.x)) {
    const uint32_t k = key[i];
    if (k == kNoKey) continue;
    for (int t = 0; t < 2; ++t)
      if ((k >> 10) == pre[t]) atomicAdd(&lh[t][k & 1023u], 1u);
  }
  __syncthreads();
  for (int k = static_cast<int>(threadIdx.x); k < 2048; k += kImgThreads)
    if (lh[k >> 10][k & 1023]) atomicAdd(&st->hist2[k >> 10][k & 1023], lh[k >> 10][k & 1023]);
}

// The selected keys (one work-group).
__global__ void __launch_bounds__(kImgThreads) k_img_select(ImgState* st) {
  if (st->count == 0u) return;
  uint32_t keys[2];
  for (int t = 0; t < 2; ++t) {
    const Pick b = block_pick<2048>(st->hist1[t], st->rank[t]);
    const Pick c = block_pick<1024>(st->hist2[t], b.rank);
    keys[t] = (((st->prefix[t] << 11) | b.digit) << 10) | c.digit;
  }
  __syncthreads();   // every thread has read prefix and rank
  if (threadIdx.x < 2) st->prefix[threadIdx.x] = threadIdx.x == 0 ? keys[0] : keys[1];
}

// main.cpp:28-30 with the writer's vertical flip: file row r is framebuffer
// row h-1-r. powf is taken as the double power rounded to float, which is
// the correctly rounded powf; glibc's powf differs from it on 671,164 of the
// 1,065,353,217 floats in [0, 1] and none of them changes the byte.
__global__ void __launch_bounds__(kImgThreads) k_img_rgb8(const float* img, int w, int h, uint8_t* out) {
  const int q = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (q >= 3 * w * h) return;
  const int r = q / (3 * w), k = q - r * 3 * w;
  float v = img[3 * static_cast<size_t>(h - 1 - r) * w + k];
  v = v < 0.f ? 0.f : (1.f < v ? 1.f : v);   // std::clamp
  const float c = static_cast<float>(pow(static_cast<double>(v), static_cast<double>(1.f / 2.2f)));
  out[q] = static_cast<uint8_t>(static_cast<uint32_t>(255.99f * c));
}

int img_blocks(int n) {
  const int b = (n + kImgThreads - 1) / kImgThreads;
  return b < 1 ? 1 : (b > kImgMaxBlocks ? kImgMaxBlocks : b);
}

}  // namespace

hipError_t launch_img_from_accum(hipStream_t s, const float4* accum, float inv_spp, int w, int h, float* img) {
  const int n = w * h;
  hipLaunchKernelGGL(k_img_from_accum, dim3((n + kImgThreads - 1) / kImgThreads), dim3(kImgThreads), 0, s, accum,
                     inv_spp, w, h, img);
  return hipGetLastError();
}

hipError_t launch_noise_stats(hipStream_t s, const float* img, int w, int h, ImgScratch sc) {
  const int n = w * h, nb = img_blocks(n);
  hipLaunchKernelGGL(k_img_lum, dim3(nb), dim3(kImgThreads), 0, s, img, n, sc.lum, sc.part, sc.st);
  hipLaunchKernelGGL(k_img_resid, dim3(nb), dim3(kImgThreads), 0, s, sc.lum, w, h, sc.part, sc.st, sc.key, sc.part2,
                     sc.pmax, sc.pcnt);
  hipLaunchKernelGGL(k_img_second, dim3(nb), dim3(kImgThreads), 0, s, sc.key, n, sc.part2, sc.pmax, sc.pcnt, sc.st);
  hipLaunchKernelGGL(k_img_third, dim3(nb), dim3(kImgThreads), 0, s, sc.key, n, sc.st);
  hipLaunchKernelGGL(k_img_select, dim3(1), dim3(kImgThreads), 0, s, sc.st);
  return hipGetLastError();
}

// ---- scratch of the allocation-free NoiseStats entry point ----------------
// One static device array per GPU, carved into the ImgScratch fields for
// images of at most kImgStaticMaxPixels. The launch sequence above writes
// every scratch word it later reads within the same call (the partial sums
// per block, the keys per pixel; k_img_lum clears the digit counts), so nothing needs clearing between calls. Calls that
// overlap on one GPU share the array and race.
namespace {
constexpr size_t align256(size_t x) { return (x + 255u) & ~static_cast<size_t>(255u); }
constexpr size_t kStOffLum = 0;
constexpr size_t kStOffKey = align256(kStOffLum + sizeof(float) * kImgStaticMaxPixels);
constexpr size_t kStOffPart = align256(kStOffKey + sizeof(uint32_t) * kImgStaticMaxPixels);
constexpr size_t kStOffPart2 = align256(kStOffPart + sizeof(double) * kImgMaxBlocks);
constexpr size_t kStOffPmax = align256(kStOffPart2 + sizeof(double) * 2 * kImgMaxBlocks);
constexpr size_t kStOffPcnt = align256(kStOffPmax + sizeof(float) * kImgMaxBlocks);
constexpr size_t kStOffState = align256(kStOffPcnt + sizeof(uint32_t) * kImgMaxBlocks);
constexpr size_t kStBytes = align256(kStOffState + sizeof(ImgState));
static_assert(kStBytes == kImgStaticScratchBytes, "static scratch size");

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch[kMaxDevices] = {};   // the array's device address, per device
}  // namespace

static __device__ __align__(256) unsigned char scratch[kStBytes];

hipError_t img_static_scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[device]) return hipSuccess;
  int cur = -1;
  hipError_t e = hipGetDevice(&cur);
  if (e != hipSuccess) return e;
  if (cur != device) return hipErrorInvalidDevice;   // the address is the current device's
  void* p = nullptr;
  e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  if (!p) return hipErrorInvalidSymbol;
  g_scratch[device] = static_cast<unsigned char*>(p);
  return hipSuccess;
}

hipError_t img_static_scratch(int device, ImgScratch* sc) {
  if (device < 0 || device >= kMaxDevices || !sc) return hipErrorInvalidDevice;
  unsigned char* base = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    base = g_scratch[device];
  }
  if (!base) return hipErrorNotInitialized;
  sc->lum = reinterpret_cast<float*>(base + kStOffLum);
  sc->key = reinterpret_cast<uint32_t*>(base + kStOffKey);
  sc->part = reinterpret_cast<double*>(base + kStOffPart);
  sc->part2 = reinterpret_cast<double*>(base + kStOffPart2);
  sc->pmax = reinterpret_cast<float*>(base + kStOffPmax);
  sc->pcnt = reinterpret_cast<uint32_t*>(base + kStOffPcnt);
  sc->st = reinterpret_cast<ImgState*>(base + kStOffState);
  return hipSuccess;
}

hipError_t launch_img_rgb8(hipStream_t s, const float* img, int w, int h, uint8_t* out) {
  const int q = 3 * w * h;
  hipLaunchKernelGGL(k_img_rgb8, dim3((q + kImgThreads - 1) / kImgThreads), dim3(kImgThreads), 0, s, img, w, h, out);
  return hipGetLastError();
}

}  // namespace xnh
