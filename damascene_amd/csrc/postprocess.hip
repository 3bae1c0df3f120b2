// postprocess.hip -- thinned gPb and sigmoid normalisation (reference:
// postprocess/skeleton.cu).
//
// PostProcess: the thin mask starts as nonmax-mPb > 0.05 (normalizewrtmpb),
// is thinned to a fixed point by eight 3x3 look-up-table passes per
// iteration (applyLut: each pass reads the image the previous pass left and
// clears the pixels whose neighbourhood code the table marks), masks gPb
// (mask), and both gPb and the thin map go through the sigmoid
// normalisation (normalizeSigmoid).  NormalizeGpbAll applies the same
// sigmoid to the eight oriented gPb planes.
//
// The mask lives in u8 ping-pong buffers between launches and as bits within
// one: a launch runs two whole iterations and reports for each whether it
// removed a pixel; the host stops after the first iteration that removed
// none, as the reference does.
#include <vector>

#include "dmsc_device.hpp"
#include "dmsc_internal.hpp"
#include "kernels.hpp"

namespace dmsc {
namespace {

// skeleton.cu:104-129: the neighbourhood codes each of the eight tables
// marks.  The code of a pixel sums 2^(r + 3c) over its non-zero neighbours
// at (row - 1 + r, col - 1 + c), r, c in 0..2 (weights 1 8 64 / 2 16 128 /
// 4 32 256), neighbours outside the image contributing nothing.
constexpr int kLutCodes[8][8] = {
    {89, 91, 217, 219, -1, -1, -1, -1},          {152, 153, 216, 217, 408, 409, 472, 473},
    {23, 31, 55, 63, -1, -1, -1, -1},            {26, 27, 30, 31, 90, 91, 94, 95},
    {464, 472, 496, 504, -1, -1, -1, -1},        {50, 51, 54, 55, 306, 307, 310, 311},
    {308, 310, 436, 438, -1, -1, -1, -1},        {176, 180, 240, 244, 432, 436, 496, 500}};

// Two iterations of the eight passes.  A pass reaches one pixel, so a wave
// with a 64 x 64 pixel window gets the 32 x 32 pixels at its middle right:
// lane r holds row r as 64 bits, a pass takes the rows above and below from
// the neighbour lanes and evaluates its codes for the whole row at once.
// Bound by launch latency: combine to postprocess at 160x120 takes 148 us with
// one launch here, 235 with a seed, two counter clears and sixteen passes of
// 3.5 us each and a look by the host after each iteration.
// seed: the mask is nmax > 0.05 instead of `in`.
constexpr int kPpHalo = 16, kPpOwn = 32;

template <int L>
__device__ __forceinline__ void pp_pass(unsigned long long& v, unsigned long long& gone) {
  const int lane = threadIdx.x & 63;
  unsigned long long up = __shfl_up(v, 1, 64), dn = __shfl_down(v, 1, 64);
  if (lane == 0) up = 0;
  if (lane == 63) dn = 0;
  const unsigned long long n[9] = {up << 1, v << 1, dn << 1, up, v, dn, up >> 1, v >> 1, dn >> 1};
  unsigned long long clear = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    if (kLutCodes[L][k] < 0) continue;
    unsigned long long hit = ~0ull;
#pragma unroll
    for (int i = 0; i < 9; i++) hit &= (kLutCodes[L][k] >> i & 1) ? n[i] : ~n[i];
    clear |= hit;
  }
  gone |= clear & v;
  v &= ~clear;
}

__device__ __forceinline__ bool pp_iteration(unsigned long long& v, unsigned long long own) {
  unsigned long long gone = 0;
  pp_pass<0>(v, gone);
  pp_pass<1>(v, gone);
  pp_pass<2>(v, gone);
  pp_pass<3>(v, gone);
  pp_pass<4>(v, gone);
  pp_pass<5>(v, gone);
  pp_pass<6>(v, gone);
  pp_pass<7>(v, gone);
  return __ballot((gone & own) != 0) != 0;
}

__global__ __launch_bounds__(256) void k_pp_thin(int w, int h, int ntx, int ntiles, const float* __restrict__ seed,
                                                 const uint8_t* __restrict__ in, uint8_t* __restrict__ out,
                                                 uint8_t* __restrict__ removed) {
  const int lane = threadIdx.x & 63, tile = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile >= ntiles) return;
  const int x0 = tile % ntx * kPpOwn - kPpHalo, y0 = tile / ntx * kPpOwn - kPpHalo;
  const int x = x0 + lane;
  unsigned long long v = 0;
#pragma unroll 16
  for (int r = 0; r < 64; r++) {
    const int y = y0 + r;
    const bool inside = x >= 0 && x < w && y >= 0 && y < h;
    const size_t p = inside ? (size_t)y * w + x : 0;
    const bool on = seed ? seed[p] > 0.05f : in[p] != 0;
    const unsigned long long m = __ballot(inside && on);
    if (lane == r) v = m;
  }
  const bool mid = lane >= kPpHalo && lane < kPpHalo + kPpOwn;
  const unsigned long long own = mid ? ((1ull << kPpOwn) - 1) << kPpHalo : 0;
  const int first = pp_iteration(v, own), second = pp_iteration(v, own);
  if (lane == 0) removed[tile] = (uint8_t)(first + 2 * second);
  // two rows of the middle per store
#pragma unroll 4
  for (int r = 0; r < kPpOwn; r += 2) {
    const int row = kPpHalo + r + (lane >> 5), bit = kPpHalo + (lane & 31);
    const unsigned long long m = __shfl(v, row, 64);
    const int yy = y0 + row, xx = x0 + bit;
    if (xx < w && yy < h) out[(size_t)yy * w + xx] = (m >> bit) & 1;
  }
}

// skeleton.cu:84-99 normalizeSigmoid (FP32 arithmetic; the source's double
// literals are single precision on the reference's target).
__device__ __forceinline__ float pp_sigmoid(float val) {
  val = (val <= 0.0f) ? 0.0f : ((val * 1.2f > 1.0f) ? 1.0f : 1.2f * val);
  val = 1.0f / (1.0f + expf(2.6433f - 10.7998f * val));
  return (val - 0.0667f) / 0.9333f;
}

// skeleton.cu:69-82 mask, then normalizeSigmoid on gPb and on the thin map.
__global__ void k_pp_finish(int n, float* __restrict__ gpb, const uint8_t* __restrict__ thin,
                            float* __restrict__ gpb_thin) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const float g = gpb[p];
  const float t = thin[p] ? g : 0.0f;
  gpb[p] = pp_sigmoid(g);
  gpb_thin[p] = pp_sigmoid(t);
}

// skeleton.cu:227-245 SigmoidGpbAll.
__global__ void k_pp_sigmoid_all(int npix, int norient, int pitch, float* __restrict__ all) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npix) return;
  for (int o = 0; o < norient; o++) {
    float v = all[(size_t)o * pitch + p];
    v = (v * 1.2f > 1.0f) ? 1.0f : v * 1.2f;
    if (v < 0.0f) v = 0.0f;
    v = 1.0f / (1.0f + expf(2.6433f - 10.7998f * v));
    all[(size_t)o * pitch + p] = (v - 0.0667f) / 0.9333f;
  }
}

}  // namespace

int run_postprocess(Ctx* ctx, int w, int h, float* gpb, const float* nmax, float* gpb_thin, int* iterations) {
  hipStream_t s = ctx->stream;
  const int n = w * h;
  void* base;
  const size_t nb = ((size_t)n + 255) & ~(size_t)255;
  const int ntx = div_up(w, kPpOwn), ntiles = ntx * div_up(h, kPpOwn);
  DMSC_TRY(ctx->scratch(5, 2 * nb + (size_t)ntiles, &base));
  uint8_t* a = (uint8_t*)base;
  uint8_t* b = a + nb;
  uint8_t* removed = b + nb;
  std::vector<uint8_t> flags(ntiles);
  const dim3 g1(div_up(n, 256));
  int it = 0;
  bool more = true;
  // skeleton.cu:143-167: repeat the eight passes until one iteration removes
  // nothing; a pixel can only be removed once, so at most n + 1 iterations
  // (a second iteration behind one that removed nothing changes nothing)
  while (more && it <= n) {
    hipLaunchKernelGGL(k_pp_thin, dim3(div_up(ntiles, 4)), dim3(256), 0, s, w, h, ntx, ntiles, it ? nullptr : nmax, b,
                       a, removed);
    DMSC_HIP(hipGetLastError());
    DMSC_HIP(hipMemcpyAsync(flags.data(), removed, (size_t)ntiles, hipMemcpyDeviceToHost, s));
    DMSC_HIP(hipStreamSynchronize(s));
    int any = 0;
    for (uint8_t f : flags) any |= f;
    it += any & 1 ? 2 : 1;
    more = any == 3;
    if (more) std::swap(a, b);
  }
  hipLaunchKernelGGL(k_pp_finish, g1, dim3(256), 0, s, n, gpb, a, gpb_thin);
  DMSC_HIP(hipGetLastError());
  if (iterations) *iterations = it;
  return DMSC_OK;
}

int launch_normalize_gpb_all(hipStream_t s, int npix, int norient, int pitch, float* all) {
  hipLaunchKernelGGL(k_pp_sigmoid_all, dim3(div_up(npix, 256)), dim3(256), 0, s, npix, norient, pitch, all);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}

}  // namespace dmsc
