// textons.hip -- texton filter bank and k-means (reference: textons/texton.cu,
// textons/kmeans.cu).
//
// Filter bank: exact FP32 correlation in the reference order (x offset
// outer, y offset inner, fused multiply-add), clamp-to-edge borders.  Each
// block stages a clamped image tile with halo in LDS; each thread computes 8
// vertically adjacent outputs so one column of tile values feeds 8
// independent accumulation chains.  Coefficients are wave-uniform (scalar
// loads).
//
// k-means: one kernel per iteration.  Every block forms the centroids from
// the int32 sums in LDS while its pixels' responses load, takes the 32 or 64
// distances per pixel on the matrix cores in the reference order, labels its
// pixels (argmin with strict '<') and adds them to the next iteration's sums
// (wrap-around, exact and order independent).  A device-side done flag lets
// all iterations be enqueued without host round trips.
#include <algorithm>
#include <cstddef>

#include "dmsc_device.hpp"
#include "dmsc_internal.hpp"
#include "kernels.hpp"

namespace dmsc {
namespace {

constexpr int TX = 64, TY = 32, RPT = 8;  // tile 64 x 32, 8 rows per thread

template <int R>
__global__ __launch_bounds__(256) void k_texton_conv(int w, int h, const float* __restrict__ grey,
                                                     const float* __restrict__ coeffs,
                                                     int first_filter, float* __restrict__ out) {
  constexpr int LW = TX + 2 * R, LH = TY + 2 * R, D = 2 * R + 1;
  __shared__ float tile[LH][LW + 1];
  const int f = first_filter + blockIdx.z;
  const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY;
  for (int i = threadIdx.x; i < LW * LH; i += 256) {
    const int ly = i / LW, lx = i - ly * LW;
    const int gx = dev::clampi(x0 + lx - R, 0, w - 1), gy = dev::clampi(y0 + ly - R, 0, h - 1);
    tile[ly][lx] = grey[(size_t)gy * w + gx];
  }
  __syncthreads();
  const int tx = threadIdx.x & 63, ty = (threadIdx.x >> 6) * RPT;
  const float* c = coeffs + (size_t)(f < 17 ? f * 169 : 17 * 169 + (f - 17) * 361);
  float acc[RPT];
#pragma unroll
  for (int k = 0; k < RPT; k++) acc[k] = 0.0f;
#pragma unroll 1
  for (int dx = 0; dx < D; dx++) {
    float col[RPT + 2 * R];
#pragma unroll
    for (int j = 0; j < RPT + 2 * R; j++) col[j] = tile[ty + j][tx + dx];
#pragma unroll
    for (int dy = 0; dy < D; dy++) {
      const float cf = c[dx * D + dy];
#pragma unroll
      for (int k = 0; k < RPT; k++) acc[k] = fmaf(col[k + dy], cf, acc[k]);
    }
  }
  const int gx = x0 + tx;
  if (gx < w) {
    const size_t n = (size_t)w * h;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int gy = y0 + ty + k;
      if (gy < h) out[(size_t)f * n + (size_t)gy * w + gx] = acc[k];
    }
  }
}

__global__ void k_zero(float* p, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0f;
}

// ------------------------------------------------------------------ k-means
// Cluster count K is 32 (texton_choice 1) or 64 (texton_choice 2); the
// state is sized for 64 and indexed with stride K.
constexpr int kMaxK = 64;
// Copies of the global sums.  Block b adds its own to copy b % 4, so an
// address meets a quarter of the blocks' atomic adds; the next iteration adds
// the copies up (8 copies measured the same).
constexpr int kCopies = 4;
// Blocks of an iteration: at least three chunks of 256 pixels each once every
// CU has a block, up to the 768 that are resident at once.  Forming the
// centroids costs a block as much as labelling several chunks: at 481x321
// with 32 clusters 256 / 512 / 603 blocks take 13.9 / 15.6 / 16.6 us, at
// 1024x768 with 64 clusters 256 / 512 / 768 / 1024 / 3072 blocks 60 / 54 /
// 53 / 59 / 73 us.
inline int km_blocks(int n) {
  const int chunks = div_up(n, 256);
  return std::min(chunks, std::min(768, std::max(256, chunks / 3)));
}

struct KmSums {
  uint32_t mass[kNFilters * kMaxK];  // [filter][cluster], int32 wrap-around sums
  uint32_t count[kMaxK];
};

struct KmState {
  int changes[3];           // label changes, by iteration modulo 3
  unsigned int done;        // set when an iteration changed no label
  unsigned int iterations;  // iterations executed
  unsigned int pad[11];
  // iteration it forms its centroids from sums[it % 3], adds to sums[(it + 1)
  // % 3] and clears sums[(it + 2) % 3] (and the change counts likewise)
  KmSums sums[3][kCopies];
};

__global__ __launch_bounds__(256) void k_km_clear(uint32_t* st) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i < sizeof(KmState) / 4) st[i] = 0;
}

// kmeans.cu:14-35 assignInitialClusters (6x6 grid capped at 31) for K = 32,
// kmeans.cu:37-55 assignInitialClusters_64 (8x8 grid) for K = 64.
template <int K>
__device__ __forceinline__ int km_initial_label(int p, int w, int h) {
  const int y = p / w, x = p - y * w;
  constexpr int G = K == 64 ? 8 : 6;
  const int c = (y / ((h - 1) / G + 1)) * G + x / ((w - 1) / G + 1);
  return (K == 32 && c >= 32) ? 31 : c;
}

// The block's int32 sums, in NC copies taken by lane so that a wave whose
// pixels share a label does not queue on one address; the copies lie 8
// banks apart.
template <int K>
struct KmBlockSums {
  static constexpr int NC = K == 32 ? 8 : 4;
  static constexpr int kStride = (kNFilters + 1) * K + 8;  // the row after the filters holds the counts
  uint32_t v[NC * kStride];

  __device__ __forceinline__ void clear() {
    for (int i = threadIdx.x; i < NC * kStride; i += 256) v[i] = 0;
  }
  // kmeans.cu:57-103 findCentroids / 106-153 findCentroids_64: (int)(1e5 *
  // response) (INTCONFACTOR, kmeans.h:16) of one pixel to cluster c
  __device__ __forceinline__ void add(const float (&x)[kNFilters], int c) {
    uint32_t* s = v + (threadIdx.x % NC) * kStride + c;
#pragma unroll
    for (int f = 0; f < kNFilters; f++) atomicAdd(s + f * K, (uint32_t)(int)(100000.0f * x[f]));
    atomicAdd(s + kNFilters * K, 1u);
  }
  __device__ __forceinline__ void flush(KmSums* out) const {
    for (int i = threadIdx.x; i < (kNFilters + 1) * K; i += 256) {
      uint32_t t = 0;
#pragma unroll
      for (int k = 0; k < NC; k++) t += v[k * kStride + i];
      if (t) atomicAdd(i < kNFilters * K ? out->mass + i : out->count + (i - kNFilters * K), t);
    }
  }
};

// Initial labels and their sums.
template <int K>
__global__ __launch_bounds__(256) void k_km_init(int w, int h, const float* __restrict__ resp, int* __restrict__ labels,
                                                 KmState* st) {
  __shared__ KmBlockSums<K> bs;
  const int n = w * h, p = blockIdx.x * 256 + threadIdx.x;
  float x[kNFilters];
#pragma unroll
  for (int f = 0; f < kNFilters; f++) x[f] = resp[(size_t)f * n + min(p, n - 1)];
  bs.clear();
  __syncthreads();
  if (p < n) {
    const int c = km_initial_label<K>(p, w, h);
    labels[p] = c;
    bs.add(x, c);
  }
  __syncthreads();
  bs.flush(&st->sums[0][blockIdx.x % kCopies]);
}

// One iteration.  The stop test (kmeans.cu:712: no label changed) is taken
// from the change count the previous iteration left; every block reads the
// same count, so all agree.
//
// Distances (kmeans.cu:296-338 makeDots + SGEMM(alpha -2, beta 1), 447-472
// findDiffLabels): dist_c = fma(-2, x.c, |x|^2 + |c|^2), x.c a chain of
// fused multiply-adds over the filters in order, strict '<' from 1e7.  One
// v_mfma_f32_32x32x1_2b_f32 per filter takes a wave's 64 pixels (two blocks
// of 32 columns, the B operand: each lane its own pixel's response) against
// 32 centroids (the rows: lane l holds centroid l % 32, the same in both
// blocks); with one step of k per instruction every result is exactly that
// chain.  A lane ends with 16 clusters (8 (r / 4) + 4 (l / 32) + r % 4) of
// two pixels, and its partner 32 lanes away with the other 16.
//
// Earlier forms of an iteration at 481x321 with 32 clusters: sums by a
// kernel of their own (17 us, 603 blocks adding 1,088 words each to one set
// of sums) and FP32 distances on the vector units (21 us); or BF16 MFMA
// distances with an exact re-check of near ties and the sums fused (40 us;
// 196 us with 64 clusters at 1024x768).  This takes 13.9 us (53 us).
typedef float f32x32 __attribute__((ext_vector_type(32)));
template <int K>
__global__ __launch_bounds__(256, 3) void k_km_pass(int n, const float* __restrict__ resp, int* __restrict__ labels,
                                                    KmState* st, int it) {
  static_assert(256 % K == 0, "a thread's centroid entries belong to one cluster");
  __shared__ KmBlockSums<K> bs;
  __shared__ float cent[kNFilters][K];
  __shared__ float cdot[K];
  __shared__ int schanges;
  const int lane = threadIdx.x & 63;
  // everything the block needs is loaded before any of it is waited for: the
  // stop test, the sums and the first pixels' responses
  const bool stop = st->done || (it > 0 && st->changes[(it - 1) % 3] <= 0);
  const KmSums* in = st->sums[it % 3];
  constexpr int NE = (kNFilters * K + 255) / 256;
  uint32_t count = 0, mass[NE];
#pragma unroll
  for (int k = 0; k < kCopies; k++) count += in[k].count[threadIdx.x % K];
#pragma unroll
  for (int e = 0; e < NE; e++) {
    mass[e] = 0;
    const int i = min((int)threadIdx.x + 256 * e, kNFilters * K - 1);
#pragma unroll
    for (int k = 0; k < kCopies; k++) mass[e] += in[k].mass[i];
  }
  int p = blockIdx.x * 256 + threadIdx.x;
  float x[kNFilters];
#pragma unroll
  for (int f = 0; f < kNFilters; f++) x[f] = resp[(size_t)f * n + min(p, n - 1)];
  int old = labels[min(p, n - 1)];
  if (stop) {
    if (blockIdx.x == 0 && threadIdx.x == 0) st->done = 1;
    return;
  }
  if (threadIdx.x == 0) schanges = 0;
  bs.clear();
  // kmeans.cu:268-286 finishCentroids(_64): an empty cluster gives NaN, which
  // never wins a comparison
#pragma unroll
  for (int e = 0; e < NE; e++) {
    const int i = threadIdx.x + 256 * e;
    if (i < kNFilters * K) (&cent[0][0])[i] = (float)(int)mass[e] / (100000.0f * (float)count);
  }
  if (blockIdx.x == 0) {
    uint32_t* z = reinterpret_cast<uint32_t*>(st->sums[(it + 2) % 3]);
    for (int i = threadIdx.x; i < (int)(sizeof(KmSums) * kCopies / 4); i += 256) z[i] = 0;
    if (threadIdx.x == 0) st->changes[(it + 1) % 3] = 0;
  }
  __syncthreads();
  if (threadIdx.x < K) {  // makeSelfDots of the centroids
    float d = 0.0f;
#pragma unroll
    for (int f = 0; f < kNFilters; f++) d = fmaf(cent[f][threadIdx.x], cent[f][threadIdx.x], d);
    cdot[threadIdx.x] = d;
  }
  __syncthreads();
  for (;;) {
    float pd = 0.0f;  // makeSelfDots of the pixel
#pragma unroll
    for (int f = 0; f < kNFilters; f++) pd = fmaf(x[f], x[f], pd);
    const float pdo = __shfl_xor(pd, 32, 64);
    const bool hi = lane >= 32;
    const float pd0 = hi ? pdo : pd, pd1 = hi ? pd : pdo;  // pixels lane % 32 and 32 + lane % 32 of the wave
    float best0 = 10000000.0f, best1 = 10000000.0f;
    int c0 = -1, c1 = -1;
#pragma unroll 1
    for (int t = 0; t < K; t += 32) {
      f32x32 d;
#pragma unroll
      for (int r = 0; r < 32; r++) d[r] = 0.0f;
#pragma unroll
      for (int f = 0; f < kNFilters; f++)
        d = __builtin_amdgcn_mfma_f32_32x32x1f32(cent[f][t + (lane & 31)], x[f], d, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int c = t + 8 * (r / 4) + 4 * (lane >> 5) + r % 4;
        const float cd = cdot[c];
        const float d0 = fmaf(-2.0f, d[r], pd0 + cd), d1 = fmaf(-2.0f, d[16 + r], pd1 + cd);
        if (d0 < best0) { best0 = d0; c0 = c; }
        if (d1 < best1) { best1 = d1; c1 = c; }
      }
    }
    // each lane keeps its own pixel and hands its partner the other one
    const float ob = __shfl_xor(hi ? best0 : best1, 32, 64);
    const int oc = __shfl_xor(hi ? c0 : c1, 32, 64);
    const float mb = hi ? best1 : best0;
    const int mc = hi ? c1 : c0;
    // the smaller distance, then the lower index; -1 (no distance below 1e7) only if both are
    const int bl = oc < 0 ? mc : mc < 0 ? oc : (ob < mb || (ob == mb && oc < mc)) ? oc : mc;
    bool changed = false;
    if (p < n) {
      changed = bl != old;
      labels[p] = bl;
      if (bl >= 0) bs.add(x, bl);  // -1: in no cluster
    }
    const unsigned long long m = __ballot(changed);
    if (lane == 0 && m) atomicAdd(&schanges, __popcll(m));
    p += gridDim.x * 256;
    if (p - (int)threadIdx.x >= n) break;
#pragma unroll
    for (int f = 0; f < kNFilters; f++) x[f] = resp[(size_t)f * n + min(p, n - 1)];
    old = labels[min(p, n - 1)];
  }
  __syncthreads();
  bs.flush(&st->sums[(it + 1) % 3][blockIdx.x % kCopies]);
  if (threadIdx.x == 0) {
    if (schanges) atomicAdd(&st->changes[it % 3], schanges);
    if (blockIdx.x == 0) st->iterations = it + 1;
  }
}

}  // namespace

int launch_texton_conv(hipStream_t s, int w, int h, const float* grey, const float* d_coeffs, float* resp) {
  dim3 grid(div_up(w, TX), div_up(h, TY), 17);
  hipLaunchKernelGGL(k_texton_conv<6>, grid, dim3(256), 0, s, w, h, grey, d_coeffs, 0, resp);
  grid.z = 16;
  hipLaunchKernelGGL(k_texton_conv<9>, grid, dim3(256), 0, s, w, h, grey, d_coeffs, 17, resp);
  const size_t n = (size_t)w * h;
  hipLaunchKernelGGL(k_zero, dim3(div_up(n, 256)), dim3(256), 0, s, resp + 33 * n, n);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}

size_t kmeans_state_bytes() { return sizeof(KmState); }

namespace {
template <int K>
int run_kmeans(hipStream_t s, int w, int h, const float* resp, int* labels, KmState* st, int max_iter) {
  const int n = w * h;
  hipLaunchKernelGGL(k_km_clear, dim3(div_up(sizeof(KmState) / 4, 256)), dim3(256), 0, s, (uint32_t*)st);
  hipLaunchKernelGGL(k_km_init<K>, dim3(div_up(n, 256)), dim3(256), 0, s, w, h, resp, labels, st);
  for (int it = 0; it < max_iter; it++)
    hipLaunchKernelGGL(k_km_pass<K>, dim3(km_blocks(n)), dim3(256), 0, s, n, resp, labels, st, it);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}
}  // namespace

int launch_kmeans(hipStream_t s, int w, int h, int k, const float* resp, int* labels, void* state, int max_iter) {
  KmState* st = (KmState*)state;
  if ((uintptr_t)state % 16) return fail(DMSC_ERR_INTERNAL, "k-means state misaligned");
  if (k == 64) return run_kmeans<64>(s, w, h, resp, labels, st, max_iter);
  if (k == 32) return run_kmeans<32>(s, w, h, resp, labels, st, max_iter);
  return fail(DMSC_ERR_ARG, "k-means supports 32 or 64 clusters");
}

const int* kmeans_iterations_ptr(const void* state) {
  return reinterpret_cast<const int*>(&static_cast<const KmState*>(state)->iterations);
}

int kmeans_read_state(hipStream_t s, const void* state, int* changes, int* iterations) {
  struct Head {
    int changes[3];
    unsigned int done, iterations;
  } h;
  static_assert(offsetof(Head, iterations) == offsetof(KmState, iterations), "the state's head");
  DMSC_HIP(hipMemcpyAsync(&h, state, sizeof(h), hipMemcpyDeviceToHost, s));
  DMSC_HIP(hipStreamSynchronize(s));
  const int last = (int)h.iterations - 1;
  if (iterations) *iterations = (int)h.iterations;
  if (changes) *changes = last >= 0 ? h.changes[last % 3] : 0;
  return DMSC_OK;
}

}  // namespace dmsc
