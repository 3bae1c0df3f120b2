// edgefilter.hpp -- the eight 7x7 oriented derivative filters of spectral Pb
// (spectralPb.cu:651-659) on the matrix cores, shared by the pipeline's
// spectral Pb and the differentiable forward and backward.
//
// v_mfma_f32_4x4x1_16b_f32 adds 16 independent 4 x 4 outer products of FP32
// values, every element one fused multiply-add: its A operand (lane 4b + i)
// holds one tap of filter i (the same for all 16 blocks b), its B operand
// (lane l) one input value of pixel l, and lane l's four result registers
// are pixel l's sums for the four filters.  Two accumulators hold the eight
// orientations, and the sums run tap by tap in the reference's order (u
// outer, v inner), bit-identical to a chain of fmaf.
//
// A wave's 98 tap operands stay in registers for all its vectors.  With one
// thread per pixel and the 392 taps as scalar operands, the taps (four times
// the scalar registers) were reloaded for every vector and the waves waited
// on those loads: k_spectral_pb took 82 us at 160x120 and 188 us at 481x321
// (8 vectors; 2 x 8 x 49 flop per pixel and vector), and takes 10 and 20
// us here; the differentiable forward at 481x321 went from 205 to 27 us.
#pragma once
#include "dmsc_device.hpp"
#include "tables.hpp"

namespace dmsc {
namespace edge {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTaps = 49;
constexpr int TX = 64, TY = 4, NT = TX * TY;         // block: 64 x 4 pixels, one row per wave
constexpr int LW = TX + 6, LH = TY + 6;              // tile with its mirrored 3-pixel frame
constexpr int kChunk = 8;                            // vectors staged at a time
constexpr int kTile = LW * LH;

struct Filters {
  float K[8 * kTaps];  // slot o: filter index (3+u) + (3+v)*7 (spectralPb.cu:100)
};

inline const Filters& filters() {  // constants, built once
  static const Filters f = [] {
    Filters t;
    spb_filters(t.K);
    return t;
  }();
  return f;
}

// Vectors i0 .. i0 + kChunk - 1 (those below nvec) of the block's tile, the
// mirrored frame included.
__device__ __forceinline__ void stage(float* tile, const float* __restrict__ V, size_t n, int i0, int nvec, int w,
                                      int h) {
  for (int k = threadIdx.x; k < kTile; k += NT) {
    const int ly = k / LW, lx = k - ly * LW;
    // mirrored coordinates (border 3), clamped to [0, w + 6) before reflecting
    const int gx = dev::mirror(dev::clampi(blockIdx.x * TX + lx, 0, w + 5), 3, w);
    const int gy = dev::mirror(dev::clampi(blockIdx.y * TY + ly, 0, h + 5), 3, h);
    const float* v = V + (size_t)i0 * n + (size_t)gy * w + gx;
    float t[kChunk];
#pragma unroll
    for (int c = 0; c < kChunk; c++) t[c] = i0 + c < nvec ? v[(size_t)c * n] : 0.f;
#pragma unroll
    for (int c = 0; c < kChunk; c++) tile[c * kTile + k] = t[c];
  }
}

// The lane's A operands: tap t of filters lane % 4 and 4 + lane % 4.
__device__ __forceinline__ void taps(const float* K, float (&a)[2][kTaps]) {
  const int i = threadIdx.x & 3;
#pragma unroll
  for (int t = 0; t < kTaps; t++) {
    a[0][t] = K[i * kTaps + t];
    a[1][t] = K[(4 + i) * kTaps + t];
  }
}

// Responses of the lane's pixel to two vectors: t0 and t1 point at their
// tile values at (row - 3, column - 3).
__device__ __forceinline__ void respond2(const float* t0, const float* t1, const float (&a)[2][kTaps],
                                         f32x4 (&s0)[2], f32x4 (&s1)[2]) {
  s0[0] = s0[1] = s1[0] = s1[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < 7; u++)
#pragma unroll
    for (int v = 0; v < 7; v++) {
      const float x0 = t0[v * LW + u], x1 = t1[v * LW + u];
      s0[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[0][u + 7 * v], x0, s0[0], 0, 0, 0);
      s1[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[0][u + 7 * v], x1, s1[0], 0, 0, 0);
      s0[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[1][u + 7 * v], x0, s0[1], 0, 0, 0);
      s1[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[1][u + 7 * v], x1, s1[1], 0, 0, 0);
    }
}

}  // namespace edge
}  // namespace dmsc
