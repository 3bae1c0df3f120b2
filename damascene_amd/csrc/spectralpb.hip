// spectralpb.hip -- oriented spectral Pb (reference: sPb/spectralPb.cu).
//
// For eigenvectors 1..nvec-1: mirror with border 3, correlate with the 8
// first-derivative-of-Gaussian 7x7 filters (u outer, v inner, fused
// multiply-add) and accumulate |response| / sqrt(lambda_i).  One lane per
// pixel keeps the 8 oriented sums for all eigenvectors in registers; the
// filters run on the matrix cores (edgefilter.hpp) over tiles staged in LDS
// eight vectors at a time.
#include "dmsc_device.hpp"
#include "dmsc_internal.hpp"
#include "edgefilter.hpp"
#include "kernels.hpp"

namespace dmsc {
namespace {

struct SpbScale {
  float s[32];  // 1/sqrt(lambda_i)
};

__global__ __launch_bounds__(edge::NT, 3) void k_spectral_pb(int w, int h, int nvec, const float* __restrict__ V,
                                                          edge::Filters F, SpbScale S, float* __restrict__ spb,
                                                          size_t pitch) {
  using namespace edge;
  __shared__ float tile[kChunk * kTile];
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const int x = blockIdx.x * TX + tx, y = blockIdx.y * TY + ty;
  const size_t n = (size_t)w * h;
  float a[2][kTaps];
  taps(F.K, a);
  float res[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int i0 = 1; i0 < nvec; i0 += kChunk) {
    if (i0 > 1) __syncthreads();
    stage(tile, V, n, i0, nvec, w, h);
    __syncthreads();
    const float* t = tile + ty * LW + tx;
#pragma unroll 1
    for (int c = 0; c < kChunk && i0 + c < nvec; c += 2) {
      f32x4 s0[2], s1[2];
      respond2(t + c * kTile, t + (c + 1) * kTile, a, s0, s1);
      const float e0 = S.s[i0 + c], e1 = i0 + c + 1 < nvec ? S.s[i0 + c + 1] : 0.f;
#pragma unroll
      for (int o = 0; o < 8; o++) res[o] = fmaf(fabsf(s0[o >> 2][o & 3]), e0, res[o]);
      if (i0 + c + 1 < nvec)
#pragma unroll
        for (int o = 0; o < 8; o++) res[o] = fmaf(fabsf(s1[o >> 2][o & 3]), e1, res[o]);
    }
  }
  if (x < w && y < h)
#pragma unroll
    for (int o = 0; o < 8; o++) spb[(size_t)o * pitch + (size_t)y * w + x] = res[o];
}

}  // namespace

// spectralPb.cu:673-795
int launch_spectral_pb(hipStream_t s, const float* h_eigvals, const float* d_eigvecs, int w, int h, int nvec,
                       float* spb, int pitch) {
  if (nvec > 32) return fail(DMSC_ERR_ARG, "spectral_pb: at most 32 vectors");
  SpbScale S;
  for (int i = 0; i < 32; i++) S.s[i] = 0.f;
  for (int i = 1; i < nvec; i++) S.s[i] = 1.0f / sqrtf(h_eigvals[i]);
  hipLaunchKernelGGL(k_spectral_pb, dim3(div_up(w, edge::TX), div_up(h, edge::TY)), dim3(edge::NT), 0, s, w, h, nvec,
                     d_eigvecs, edge::filters(), S, spb, (size_t)pitch);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}

}  // namespace dmsc
