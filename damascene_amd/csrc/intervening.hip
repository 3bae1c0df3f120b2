// intervening.hip -- intervening-contour affinities on the radius-5 disc
// (reference: intervening/intervening.cu).
//
// The affinity of a pixel and a disc point is exp(-(1 - C(ic)) / sigma), ic
// the strongest boundary crossed on the walk to the point (walks.hpp) and C a
// falling logistic; the matrix is then symmetrised, M(p, q) = (walk from p +
// walk from q) / 2.  Two exponentials per entry and the walks' integer tests
// took 272 us at 640x480, and clearing and symmetrising the matrix 66 us more.
// Here:
//  * The affinity is a falling function g of ic (each of its steps is
//    monotone in floating point too), so g of the largest crossed value is
//    the smallest g of the crossed pixels: g is evaluated once per staged
//    pixel, as unsigned bits (g >= 0), and an entry is a minimum over LDS
//    values.
//  * The pixels crossed are the same for every pixel whose window is not
//    clipped: their offsets are compiled into the kernel (418 reads for the 80
//    points).  Near the image's edges 36 points have a second set: a constant
//    per point, with a bit for each pair of the window's reaches, tells when.
//    The launch needs no table in memory, so nothing is allocated or copied
//    for it and a caller may capture it.
//  * A thread takes both walks of each of its entries and writes the
//    symmetrised value once: no clearing, no second kernel.
// It takes 27 us at 640x480 (100 MB written) and 15 us at 160x120 (140 us
// before), where most waves touch an edge; with a table in memory of the set
// each clipped window takes, waves waited on it: 30 and 18 us.
#include <utility>

#include "dmsc_device.hpp"
#include "dmsc_internal.hpp"
#include "kernels.hpp"
#include "walks.hpp"

namespace dmsc {
namespace {

__device__ inline float c_ic_ss(float ic) {  // intervening.cu:32-42 (project exp, as above)
  float val = 1.8682f;
  val += (ic / 0.3130f) * -1.3113f;
  const float post = 1.0f / (1.0f + dev::exp_exact(-val));
  if (!isfinite(post)) return 0;
  if (post < 0) return 0;
  if (post > 1) return 1;
  return post;
}

// intervening.cu:28-30, with the project exp in place of the device expf
__device__ inline float affinity(float c, float rs) { return dev::exp_exact(-(1 - c) * rs); }

constexpr int ITX = 64, ITY = 4, HALO = 6;            // a walk reaches 5 pixels, its crossings one more
constexpr int LW = ITX + 2 * HALO, LH = ITY + 2 * HALO;
// Columns past the image that one block clears.  With a pitch for larger images
// than this one there is more to clear than the image's blocks should: at 32x32
// with the pitch of 640x480 they took 355 us where k_clear_pad takes 14 (and 14
// at 640x480 with as many columns again, where one block took 11.5 ms).
constexpr int kPadPiece = 4096;

// Smallest g on a walk of W from the pixel at `b` (its tile position less
// the halo) to point D.
template <bool SECOND, int D, int... K>
__device__ __forceinline__ uint32_t walk_min(const uint32_t* b, uint32_t g, std::integer_sequence<int, K...>) {
  constexpr const Walks& W = SECOND ? kSecondWalks : kFullWalks;
  ((g = min(g, b[(HALO + W.ey[D][K]) * LW + HALO + W.ex[D][K]])), ...);
  return g;
}
template <bool SECOND, int D>
__device__ __forceinline__ uint32_t walk_min(const uint32_t* b, uint32_t g0) {
  return walk_min<SECOND, D>(b, g0, std::make_integer_sequence<int, (SECOND ? kSecondWalks : kFullWalks).n[D]>());
}

struct Pixel {
  const uint32_t* b;  // tile position less the halo
  int x, y, w, h;
  uint32_t g0;  // g(0): nothing crossed
};

// Affinity (its bits) of the walk from the pixel (x, y), at b, to point D
// inside its window, which may be clipped.
template <int D>
__device__ __forceinline__ uint32_t any_walk(const uint32_t* b, int x, int y, const Pixel& P) {
  uint32_t g = walk_min<false, D>(b, P.g0);
  if constexpr (constexpr uint32_t kSecond = kWalkRules.second[D]; kSecond != 0) {
    const int at = walk_bit(D, walk_reach(walk_dy(D), y, P.h), walk_reach(walk_dx(D), x, P.w));
    if (__builtin_amdgcn_ubfe(kSecond, at, 1)) g = walk_min<true, D>(b, P.g0);
  }
  return g;
}

// M(p, p + D): the mean of the two walks, 0 past the image.
template <int D, bool FULL>
__device__ __forceinline__ float entry(const Pixel& P) {
  constexpr int dy = walk_dy(D), dx = walk_dx(D), R = kWalkArea - 1 - D;  // R: the way back
  if constexpr (dy == 0 && dx == 0) {
    return 1.0f;
  } else {
    const uint32_t* q = P.b + dy * LW + dx;
    if constexpr (FULL) {
      return 0.5f * (__uint_as_float(walk_min<false, D>(P.b, P.g0)) +
                     __uint_as_float(walk_min<false, R>(q, P.g0)));
    } else {
      const int x = P.x + dx, y = P.y + dy;
      const bool in = x >= 0 && y >= 0 && x < P.w && y < P.h;
      const float there = __uint_as_float(any_walk<D>(P.b, P.x, P.y, P));
      const float back = __uint_as_float(any_walk<R>(q, x, y, P));
      return in ? 0.5f * (there + back) : 0.0f;
    }
  }
}

template <bool FULL, int... D>
__device__ __forceinline__ void entries(const Pixel& P, float* __restrict__ M, size_t pitch, bool live,
                                        std::integer_sequence<int, D...>) {
  if constexpr (FULL) {
    ((M[(size_t)D * pitch] = entry<D, true>(P)), ...);
  } else {
    auto put = [&](int d, float v) {
      if (live) M[(size_t)d * pitch] = v;
    };
    (put(D, entry<D, false>(P)), ...);
  }
}

__global__ __launch_bounds__(256) void k_affinities(int w, int h, float rs, const float* __restrict__ mpb,
                                                    float* __restrict__ M, size_t pitch) {
  // the way back from a point past the tile's frame is formed and dropped:
  // five rows and columns of slack on each side
  __shared__ uint32_t tile[(LH + 10) * LW + 10];
  uint32_t* t0 = tile + 5 * LW + 5;
  const int bx = blockIdx.x * ITX, by = blockIdx.y * ITY;
  const uint32_t g0 = __float_as_uint(affinity(c_ic_ss(0.0f), rs));
  for (int i = threadIdx.x; i < (LH + 10) * LW + 10; i += 256) tile[i] = g0;
  __syncthreads();
  for (int i = threadIdx.x; i < LW * LH; i += 256) {
    const int ly = i / LW, lx = i - ly * LW;
    const int gx = dev::clampi(bx + lx - HALO, 0, w - 1), gy = dev::clampi(by + ly - HALO, 0, h - 1);
    const float v = mpb[(size_t)gy * w + gx];
    // the walks take the maximum with 0 first
    if (v > 0.0f) t0[i] = __float_as_uint(affinity(c_ic_ss(v), rs));
  }
  __syncthreads();
  const int tx = threadIdx.x % ITX, ty = threadIdx.x / ITX;
  const int x = bx + tx, y = by + ty;
  const bool live = x < w && y < h;
  const Pixel P{t0 + ty * LW + tx, min(x, w - 1), min(y, h - 1), w, h, g0};
  float* row = M + (live ? (size_t)y * w + x : 0);
  // no window of the pixel's or its disc points' is clipped
  const bool full = x >= 10 && y >= 10 && x < w - 10 && y < h - 10;
  constexpr std::make_integer_sequence<int, kWalkArea> all;
  if (__all(full)) entries<true>(P, row, pitch, live, all);
  else entries<false>(P, row, pitch, live, all);
  // a few columns past the image, a row per block; more: k_clear_pad
  const int n = w * h, pad = (int)pitch - n, blocks = gridDim.x * gridDim.y;
  if (pad > kPadPiece) return;
  for (int d = blockIdx.y * gridDim.x + blockIdx.x; d < kWalkArea; d += blocks)
    for (int i = threadIdx.x; i < pad; i += 256) M[(size_t)d * pitch + n + i] = 0.0f;
}

__global__ __launch_bounds__(256) void k_clear_pad(int n, float* __restrict__ M, size_t pitch) {
  const size_t at = (size_t)n + (size_t)blockIdx.x * kPadPiece;
  for (size_t i = at + threadIdx.x; i < min(at + kPadPiece, pitch); i += 256) M[blockIdx.y * pitch + i] = 0.0f;
}

}  // namespace

int launch_intervene(hipStream_t s, int w, int h, const float* mpb, float* M, int pitch, float sigma) {
  hipLaunchKernelGGL(k_affinities, dim3(div_up(w, ITX), div_up(h, ITY)), dim3(256), 0, s, w, h, 1.0f / sigma, mpb, M,
                     (size_t)pitch);
  if (const int pad = pitch - w * h; pad > kPadPiece)
    hipLaunchKernelGGL(k_clear_pad, dim3(div_up(pad, kPadPiece), kWalkArea), dim3(256), 0, s, w * h, M, (size_t)pitch);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}

}  // namespace dmsc
