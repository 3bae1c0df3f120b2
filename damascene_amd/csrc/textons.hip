// textons.hip -- texton filter bank and k-means (reference: textons/texton.cu,
// textons/kmeans.cu).
//
// Filter bank: exact FP32 correlation in the reference order (x offset
// outer, y offset inner, fused multiply-add), clamp-to-edge borders, on the
// matrix cores.
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

// The bank's filters 0..16 have radius 6 and 17..32 radius 9 (filter 33 is
// zero).  v_mfma_f32_16x16x1_4b_f32 adds four blocks of a 16 x 16 outer product
// with one step of k: row i is filter i of a scale, a column one of the wave's
// 64 pixels (block l / 16, lane l its own pixel's value), so 16 filters of 64
// pixels advance by one tap and every sum is the reference's fmaf chain.  A
// block takes 64 x 4 RW pixels, RW rows per wave; its grey tile and the 16
// filters' taps lie in LDS.  The 17th filter of radius 6 runs on the vector
// units beside them.  One filter per block and 8 pixels per thread took 28 +
// 45 us at 481x321 (88 + 155 us at 1024x768); one launch of both scales takes
// 38 us (136 us), of which the MFMAs are 18 (85) and the responses' stores,
// 21 MB (107 MB), most of the rest.
constexpr int TX = 64;
constexpr int kRows16 = 16;  // filters on the matrix cores
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTaps9 = 19 * 19 * kRows16, kTaps6 = 13 * 13 * kRows16;
template <int R, int RW>
constexpr int bank_lds() {  // floats: the tile and the taps
  return (TX + 2 * R) * (4 * RW + 2 * R) + (2 * R + 1) * (2 * R + 1) * kRows16;
}

template <int R, int RW, bool ODD>
__device__ __forceinline__ void texton_bank(float* lds, int w, int h, const float* __restrict__ grey,
                                            const float* __restrict__ bank, const float* __restrict__ odd,
                                            float* __restrict__ out) {
  constexpr int LW = TX + 2 * R, TY = 4 * RW, LH = TY + 2 * R, D = 2 * R + 1;
  float* taps = lds;  // [dx][dy][filter]
  float* tile = lds + D * D * kRows16;
  const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY;
  for (int i = threadIdx.x; i < LW * LH; i += 256) {
    const int ly = i / LW, lx = i - ly * LW;
    const int gx = dev::clampi(x0 + lx - R, 0, w - 1), gy = dev::clampi(y0 + ly - R, 0, h - 1);
    tile[i] = grey[(size_t)gy * w + gx];
  }
  for (int i = threadIdx.x; i < D * D * kRows16 / 4; i += 256)
    reinterpret_cast<float4*>(taps)[i] = reinterpret_cast<const float4*>(bank)[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, ty = (threadIdx.x >> 6) * RW;
  const float* col = tile + ty * LW + lane;
  const float* tap = taps + (lane & 15);
  f32x16 acc[RW];
  float acc_odd[RW];
#pragma unroll
  for (int k = 0; k < RW; k++) {
#pragma unroll
    for (int r = 0; r < 16; r++) acc[k][r] = 0.0f;
    acc_odd[k] = 0.0f;
  }
#pragma unroll 1
  for (int dx = 0; dx < D; dx++) {
    float v[D + RW - 1], a[D];
#pragma unroll
    for (int dy = 0; dy < D; dy++) a[dy] = tap[(dx * D + dy) * kRows16];
#pragma unroll
    for (int j = 0; j < D + RW - 1; j++) v[j] = col[j * LW + dx];
#pragma unroll
    for (int dy = 0; dy < D; dy++)
#pragma unroll
      for (int k = 0; k < RW; k++) {
        acc[k] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[dy], v[dy + k], acc[k], 0, 0, 0);
        if (ODD) acc_odd[k] = fmaf(v[dy + k], odd[dx * D + dy], acc_odd[k]);
      }
  }
  const size_t n = (size_t)w * h;
#pragma unroll
  for (int k = 0; k < RW; k++) {
    const int y = y0 + ty + k;
    if (y >= h) continue;
    const size_t row = (size_t)y * w;
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const int x = x0 + 16 * b + (lane & 15);
      if (x < w)
#pragma unroll
        for (int r = 0; r < 4; r++) out[(size_t)(4 * (lane >> 4) + r) * n + row + x] = acc[k][4 * b + r];
    }
    // the odd filter of this scale; the last plane of the bank is zero
    if (x0 + lane < w) out[(size_t)kRows16 * n + row + x0 + lane] = ODD ? acc_odd[k] : 0.0f;
  }
}

template <int RW>
__global__ __launch_bounds__(256) void k_texton_bank(int w, int h, const float* __restrict__ grey,
                                                     const float* __restrict__ taps, float* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) float lds[bank_lds<9, RW>()];
  if (blockIdx.z == 0)  // the longer blocks first
    texton_bank<9, RW, false>(lds, w, h, grey, taps, nullptr, out + (size_t)17 * w * h);
  else
    texton_bank<6, RW, true>(lds, w, h, grey, taps + kTaps9, taps + kTaps9 + kTaps6, out);
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

// Taps of radius 9's 16 filters, radius 6's first 16 ([tap][filter] each,
// tap = dx (2 R + 1) + dy) and radius 6's last one.
std::vector<float> texton_taps() {
  const TextonBank& b = texton_bank();
  std::vector<float> t;
  t.reserve(kTaps9 + kTaps6 + 169);
  for (int i = 0; i < 361; i++)
    for (int f = 0; f < kRows16; f++) t.push_back(b.coeffs[17 * 169 + (size_t)f * 361 + i]);
  for (int i = 0; i < 169; i++)
    for (int f = 0; f < kRows16; f++) t.push_back(b.coeffs[(size_t)f * 169 + i]);
  for (int i = 0; i < 169; i++) t.push_back(b.coeffs[(size_t)kRows16 * 169 + i]);
  return t;
}

int launch_texton_conv(hipStream_t s, int w, int h, const float* grey, const float* d_taps, float* resp) {
  // two rows per wave halve the reads of the taps and the tile's frame, and
  // pay once the grid is several rounds deep (1024x768, 3,072 blocks: 136
  // against 147 us); at 481x321 (656 blocks, fewer than the chip holds) one
  // row per wave balances better (38 against 42 us)
  const int blocks2 = div_up(w, TX) * div_up(h, 8) * 2;
  if (blocks2 >= 2048)
    hipLaunchKernelGGL(k_texton_bank<2>, dim3(div_up(w, TX), div_up(h, 8), 2), dim3(256), 0, s, w, h, grey, d_taps,
                       resp);
  else
    hipLaunchKernelGGL(k_texton_bank<1>, dim3(div_up(w, TX), div_up(h, 4), 2), dim3(256), 0, s, w, h, grey, d_taps,
                       resp);
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
