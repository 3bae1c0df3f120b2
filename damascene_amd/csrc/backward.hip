// backward.hip -- differentiable spectral Pb + combine.
//
// The reference has no backward pass; its forward is combine.cu:24-70
// (combinedG_o = sum_k w_k C_{k,o} over the 12 cue x scale planes),
// spectralPb.cu:651-659 (sPb_o = sum_i |K_o * mirror3(v_i)| / sqrt(lambda_i))
// and globalPb.cu:5-49 (gPbAll_o = combinedG_o + 0.0139 sPb_o, gPb = max_o).
// Here the weights are free parameters,
//   params = [w_0 .. w_11, gamma, eta_0 .. eta_{nvec-1}]   (eta_0 unused),
//   gPbAll_o = sum_k w_k C_{k,o} + gamma * sum_{i>=1} eta_i |R_{i,o}|,
//   R_{i,o}  = K_o correlated with v_i mirrored by 3 pixels,
//   gPbPre   = max_o gPbAll_o (strict '>', the lowest orientation wins ties),
// and the backward pass gives, from g = dL/dgPbPre and o* = argmax:
//   dL/dw_k    = sum_p g C_{k,o*}
//   dL/dgamma  = sum_p g sPb_{o*}
//   dL/deta_i  = gamma sum_p g |R_{i,o*}|
//   dL/dv_i    = mirror^T K^T (g gamma eta_i sign(R_{i,o*}) at orientation o*)
// The forward forms every value in the pipeline's operation order, so with
// params = (combine weights, 0.0139, 1/sqrt(lambda_i)) its gPbAll is
// bit-identical to the pipeline's.  Parameter gradients are block partial
// sums in FP64 reduced in a fixed order (deterministic).
#include "dmsc_device.hpp"
#include "dmsc_internal.hpp"
#include "edgefilter.hpp"
#include "kernels.hpp"

namespace dmsc {
namespace {

using edge::f32x4;
constexpr int kTaps = edge::kTaps;

struct Cues {
  const float* c[4];  // Bg, Cga, Cgb, Tg: [24][cue_pitch], scale-major then orientation
};

__global__ __launch_bounds__(edge::NT, 3) void k_dspb_forward(int w, int h, int nvec, const float* __restrict__ V,
                                                              edge::Filters F, const float* __restrict__ prm, Cues C,
                                                              size_t cue_pitch, float* __restrict__ all, size_t pitch,
                                                              float* __restrict__ gpb_pre, int* __restrict__ amax) {
  using namespace edge;
  __shared__ float tile[kChunk * kTile];
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const int x = blockIdx.x * TX + tx, y = blockIdx.y * TY + ty;
  const size_t n = (size_t)w * h;
  float res[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  {
    float a[2][kTaps];
    taps(F.K, a);
    for (int i0 = 1; i0 < nvec; i0 += kChunk) {
      if (i0 > 1) __syncthreads();
      stage(tile, V, n, i0, nvec, w, h);
      __syncthreads();
      const float* t = tile + ty * LW + tx;
#pragma unroll 1
      for (int c = 0; c < kChunk && i0 + c < nvec; c += 2) {
        f32x4 s0[2], s1[2];
        respond2(t + c * kTile, t + (c + 1) * kTile, a, s0, s1);
        const bool two = i0 + c + 1 < nvec;
        const float e0 = prm[13 + i0 + c], e1 = two ? prm[13 + i0 + c + 1] : 0.f;
#pragma unroll
        for (int o = 0; o < 8; o++) res[o] = fmaf(fabsf(s0[o >> 2][o & 3]), e0, res[o]);
        if (two)
#pragma unroll
          for (int o = 0; o < 8; o++) res[o] = fmaf(fabsf(s1[o >> 2][o & 3]), e1, res[o]);
      }
    }
  }
  if (x >= w || y >= h) return;
  const size_t p = (size_t)y * w + x;
  const float gamma = prm[12];
  float m = -200.0f;
  int mo = 0;
#pragma unroll
  for (int o = 0; o < 8; o++) {
    float a2 = 0.f;
#pragma unroll
    for (int k = 0; k < 12; k++) a2 = fmaf(C.c[k / 3][(size_t)((k % 3) * 8 + o) * cue_pitch + p], prm[k], a2);
    const float v = fmaf(gamma, res[o], a2);
    if (all) all[(size_t)o * pitch + p] = v;
    if (v > m) {
      m = v;
      mo = o;
    }
  }
  gpb_pre[p] = m;
  amax[p] = mo;
}

// Sum over the block in a fixed order (waves' butterfly sums, then the
// waves in order); thread 0 of each wave leaves its part in red[slot].
__device__ __forceinline__ void wave_part(double v, double (*red)[edge::NT / 64], int slot) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[slot][threadIdx.x >> 6] = v;
}

// Per pixel: R_{i,o*} for every vector (same order as the forward, so the
// signs are the forward's), the scattered values s_i = g gamma eta_i
// sign(R_{i,o*}) for the second kernel, and block partial sums of the
// parameter gradients (np = 13 + nvec values per block).  The responses of
// all eight orientations come from the matrix cores and o*'s is selected:
// the wave's chain for one orientation alone (an LDS read of the tap per
// lane) is slower.
__global__ __launch_bounds__(edge::NT, 3) void k_dspb_backward1(int w, int h, int nvec, const float* __restrict__ V,
                                                                edge::Filters F, const float* __restrict__ prm, Cues C,
                                                                size_t cue_pitch, const float* __restrict__ grad,
                                                                const int* __restrict__ amax, float* __restrict__ S,
                                                                double* __restrict__ part) {
  using namespace edge;
  __shared__ float tile[kChunk * kTile];
  __shared__ double red[13 + kMaxDiffVec][NT / 64];
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const int x = blockIdx.x * TX + tx, y = blockIdx.y * TY + ty;
  const bool in = x < w && y < h;
  const size_t n = (size_t)w * h, p = in ? (size_t)y * w + x : 0;
  const float g = in ? grad[p] : 0.f;
  const int o = in ? amax[p] : 0;
  const float gamma = prm[12];
  const int np = 13 + nvec;
  const int blk = blockIdx.y * gridDim.x + blockIdx.x;
  float spb = 0.f;
  {
    float a[2][kTaps];
    taps(F.K, a);
    for (int i0 = 1; i0 < nvec; i0 += kChunk) {
      if (i0 > 1) __syncthreads();
      stage(tile, V, n, i0, nvec, w, h);
      __syncthreads();
      const float* t = tile + ty * LW + tx;
#pragma unroll 1
      for (int c = 0; c < kChunk && i0 + c < nvec; c += 2) {
        f32x4 s0[2], s1[2];
        respond2(t + c * kTile, t + (c + 1) * kTile, a, s0, s1);
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const int i = i0 + c + e;
          if (i >= nvec) break;
          float r = 0.f;
#pragma unroll
          for (int k = 0; k < 8; k++) r = o == k ? (e ? s1[k >> 2][k & 3] : s0[k >> 2][k & 3]) : r;
          const float eta = prm[13 + i];
          spb = fmaf(fabsf(r), eta, spb);
          const float sg = r > 0.f ? 1.f : (r < 0.f ? -1.f : 0.f);
          if (in) S[(size_t)i * n + p] = g * gamma * eta * sg;
          wave_part((double)g * (double)gamma * (double)fabsf(r), red, 13 + i);
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 12; k++) {
    const float c = in ? C.c[k / 3][(size_t)((k % 3) * 8 + o) * cue_pitch + p] : 0.f;
    wave_part((double)g * (double)c, red, k);
  }
  wave_part((double)g * (double)spb, red, 12);
  wave_part(0.0, red, 13);  // eta_0 (vector 0 is not used)
  __syncthreads();
  if ((int)threadIdx.x < np) {
    double t = red[threadIdx.x][0];
#pragma unroll
    for (int k = 1; k < NT / 64; k++) t += red[threadIdx.x][k];
    part[(size_t)blk * np + threadIdx.x] = t;
  }
}

// dL/dv_i at pixel (a, b): every mirrored position (X, Y) that reflects to
// (a, b) -- X = a + 3, and 2 - a near the left edge or 2w + 2 - a near the
// right (dev::mirror with border 3) -- collects K_{o*}(u, v) s_i from the
// pixels (X - 3 - u, Y - 3 - v) whose 7 x 7 window read it.
//
// A block owns 32 x 8 pixels and stages the argmax and the scattered values
// of its pixels and a 3-pixel frame in LDS (every position above lies within
// 3 pixels of (a, b)), eight vectors at a time as two float4 per pixel: one
// tap is two 16-byte LDS reads, the tap's filter value and eight
// multiply-adds.  Read straight from memory, the 49 x 9 gathers per pixel
// took 144 us at 481x321 with 8 vectors; this takes 15.6 us.
constexpr int GX = 32, GY = 8, GW = GX + 6, GH = GY + 6;

__global__ __launch_bounds__(256) void k_dspb_backward2(int w, int h, int nvec, edge::Filters F,
                                                        const int* __restrict__ amax, const float* __restrict__ S,
                                                        float* __restrict__ dV) {
  __shared__ float sk[8 * kTaps];
  __shared__ float4 ss[2][GH * GW];
  __shared__ int so[GH * GW];  // first tap of the pixel's filter
  const size_t n = (size_t)w * h;
  const int bx = blockIdx.x * GX, by = blockIdx.y * GY;
  for (int k = threadIdx.x; k < 8 * kTaps; k += 256) sk[k] = F.K[k];
  const int a = bx + (int)(threadIdx.x % GX), b = by + (int)(threadIdx.x / GX);
  const bool in = a < w && b < h;
  const size_t p = in ? (size_t)b * w + a : 0;
  int px[2], py[2], nx = 0, ny = 0;
  px[nx++] = a + 3;
  if (a <= 2) px[nx++] = 2 - a;
  else if (a >= w - 3) px[nx++] = 2 * w + 2 - a;
  py[ny++] = b + 3;
  if (b <= 2) py[ny++] = 2 - b;
  else if (b >= h - 3) py[ny++] = 2 * h + 2 - b;
  if (in) dV[p] = 0.f;  // vector 0 does not enter the forward
  for (int i0 = 1; i0 < nvec; i0 += 8) {
    __syncthreads();
    for (int k = threadIdx.x; k < GH * GW; k += 256) {
      const int y = by - 3 + k / GW, x = bx - 3 + k % GW;
      const bool ok = x >= 0 && y >= 0 && x < w && y < h;
      const size_t q = ok ? (size_t)y * w + x : 0;
      float v[8];
#pragma unroll
      for (int c = 0; c < 8; c++) v[c] = ok && i0 + c < nvec ? S[(size_t)(i0 + c) * n + q] : 0.f;
      ss[0][k] = make_float4(v[0], v[1], v[2], v[3]);
      ss[1][k] = make_float4(v[4], v[5], v[6], v[7]);
      so[k] = ok ? amax[q] * kTaps : 0;
    }
    __syncthreads();
    if (!in) continue;
    float acc[8];
#pragma unroll
    for (int c = 0; c < 8; c++) acc[c] = 0.f;
    for (int jy = 0; jy < ny; jy++)
      for (int jx = 0; jx < nx; jx++)
        for (int u = -3; u <= 3; u++) {
          const int xs = px[jx] - 3 - u;
          if (xs < 0 || xs >= w) continue;
#pragma unroll
          for (int vv = -3; vv <= 3; vv++) {
            const int ys = py[jy] - 3 - vv;
            if (ys < 0 || ys >= h) continue;
            const int k = (ys - by + 3) * GW + xs - bx + 3;
            const float kv = sk[so[k] + (3 + u) + (3 + vv) * 7];
            const float4 lo = ss[0][k], hi = ss[1][k];
            acc[0] = fmaf(kv, lo.x, acc[0]);
            acc[1] = fmaf(kv, lo.y, acc[1]);
            acc[2] = fmaf(kv, lo.z, acc[2]);
            acc[3] = fmaf(kv, lo.w, acc[3]);
            acc[4] = fmaf(kv, hi.x, acc[4]);
            acc[5] = fmaf(kv, hi.y, acc[5]);
            acc[6] = fmaf(kv, hi.z, acc[6]);
            acc[7] = fmaf(kv, hi.w, acc[7]);
          }
        }
#pragma unroll
    for (int c = 0; c < 8; c++)
      if (i0 + c < nvec) dV[(size_t)(i0 + c) * n + p] = acc[c];
  }
}

// Parameter gradients: block j sums parameter j's partials, each thread a
// strided subset, then the threads' sums in a fixed order.
__global__ __launch_bounds__(256) void k_dspb_reduce(int nblk, int np, const double* __restrict__ part,
                                                     float* __restrict__ gp) {
  __shared__ double red[4];
  const int j = blockIdx.x;
  double v = 0;
  for (int b = threadIdx.x; b < nblk; b += 256) v += part[(size_t)b * np + j];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) gp[j] = (float)(((red[0] + red[1]) + red[2]) + red[3]);
}

}  // namespace

int spb_combine_forward(Ctx* ctx, int w, int h, int cue_pitch, const float* bg, const float* cga, const float* cgb,
                        const float* tg, int nvec, const float* V, const float* prm, float* all, int pitch,
                        float* gpb_pre, int* amax) {
  if (nvec < 2 || nvec > kMaxDiffVec) return fail(DMSC_ERR_ARG, "nvec must be in [2, %d]", kMaxDiffVec);
  hipLaunchKernelGGL(k_dspb_forward, dim3(div_up(w, edge::TX), div_up(h, edge::TY)), dim3(edge::NT), 0, ctx->stream, w,
                     h, nvec, V, edge::filters(), prm, Cues{{bg, cga, cgb, tg}}, (size_t)cue_pitch, all, (size_t)pitch, gpb_pre, amax);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}

int spb_combine_backward(Ctx* ctx, int w, int h, int cue_pitch, const float* bg, const float* cga, const float* cgb,
                         const float* tg, int nvec, const float* V, const float* prm, const int* amax,
                         const float* grad, float* grad_prm, float* dV) {
  if (nvec < 2 || nvec > kMaxDiffVec) return fail(DMSC_ERR_ARG, "nvec must be in [2, %d]", kMaxDiffVec);
  const size_t n = (size_t)w * h;
  const dim3 g1(div_up(w, edge::TX), div_up(h, edge::TY)), g2(div_up(w, GX), div_up(h, GY));
  const int nblk = (int)(g1.x * g1.y), np = 13 + nvec;
  const size_t s_bytes = (sizeof(float) * nvec * n + 255) & ~(size_t)255;
  void* scr;
  DMSC_TRY(ctx->scratch(4, s_bytes + sizeof(double) * (size_t)nblk * np, &scr));
  float* S = (float*)scr;
  double* part = (double*)((char*)scr + s_bytes);
  hipLaunchKernelGGL(k_dspb_backward1, g1, dim3(edge::NT), 0, ctx->stream, w, h, nvec, V, edge::filters(), prm,
                     Cues{{bg, cga, cgb, tg}}, (size_t)cue_pitch, grad, amax, S, part);
  hipLaunchKernelGGL(k_dspb_backward2, g2, dim3(256), 0, ctx->stream, w, h, nvec, edge::filters(), amax, S, dV);
  hipLaunchKernelGGL(k_dspb_reduce, dim3(np), dim3(256), 0, ctx->stream, nblk, np, part, grad_prm);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}

}  // namespace dmsc
