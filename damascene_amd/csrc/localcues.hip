// localcues.hip -- brightness / colour / texture gradients (reference:
// localcues/localcues.cu, gradient.cu, rotate.cu, parabola.cu).
//
// All 4 channels x 4 rotations (16 frames) are processed together so every
// launch has enough waves to fill 256 CUs:
//   1. labels:    quantised L/a/b (25 bins) or textons (32/64), mirrored (border
//                 30) and scattered through the Bresenham rotation tables into
//                 uint8 rotated frames (255 = outside the rotated image);
//   2. integrals: per-bin 2-D inclusive counts, stored as uint16 modulo
//                 2^16: every half-disc count is a signed sum of four corners
//                 whose true value lies in [0, 2r^2], so modular arithmetic
//                 recovers it exactly at half the bytes of int32.  A frame's
//                 integral is BP/8 planes of 8 bins (16 bytes) per rotated
//                 pixel: a wave's 16-byte gathers of one plane at consecutive
//                 pixels read one contiguous run;
//   3. gradients: per pixel, scale and split: 4+4 corner gathers per bin,
//                 optional bin blur, normalisation to sum 8 and chi-squared
//                 with the reference's 32-slot tree sums (64 textons: two
//                 lanes per pixel, one 32-bin half each);
//   4. parabola:  Savitzky-Golay smoothing of each mirrored gradient plane
//                 over the filter's non-zero taps (v outer, u inner, fma).
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>

#include "dmsc_device.hpp"
#include "dmsc_internal.hpp"
#include "kernels.hpp"

namespace dmsc {

namespace {

constexpr int kFrames = 16;
constexpr int kRadii[4] = {3, 5, 10, 20};

struct FrameGeom {
  int w, h, bw, bh;
  int nw[4], nh[4];
  long long lab_off[kFrames];  // byte offset of frame f = ch*4 + o (label buffer)
  long long int_off[kFrames];  // uint16 element offset of frame f (integral buffer)
  long long band_off[kFrames];  // uint16 element offset of frame f's band sums (k_integral_strip)
  long long row_off[kFrames];   // uint32 word offset of frame f's row carries (k_integral_strip)
  int tab_off[4];              // offset of orientation o's tables: bX[bw] bY[bw] gX[bh] gY[bh]
  int rect[4][4][8];           // [orientation][radius index][corner A..H]
  int tbp;                     // bins per integral pixel of the texture frames (32 or 64)
};

// Bins stored per integral-image pixel of frame f: 32 for the L/a/b frames
// (25 used), 32 or 64 for the texton frames 12..15.
__device__ __forceinline__ int bin_pitch(const FrameGeom& g, int f) { return f >= 12 ? g.tbp : 32; }

// Element index (uint16) of bin `bin` at rotated pixel `pix` of frame f:
// plane bin / 8 holds 8 bins per pixel.
__device__ __forceinline__ size_t int_index(const FrameGeom& g, int f, long long pix, int bin) {
  const int o = f & 3;
  const size_t npx = (size_t)g.nw[o] * g.nh[o];
  return (size_t)g.int_off[f] + (size_t)(bin >> 3) * npx * 8 + (size_t)pix * 8 + (bin & 7);
}

struct CueOut {
  float* p[4];  // Bg, Cga, Cgb, Tg; each [24][pitch]
};

__global__ void k_fill_u8(uint8_t* p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0xff;
}

// gradient.cu:210-223 (quantizeImage, mirrorImage) + rotate.cu:247-259
// (bresenhamRotate): one mirrored pixel per thread, frames f0, f0 + 1, ...
__global__ void k_cue_labels(FrameGeom g, int f0, const float* __restrict__ L, const float* __restrict__ A,
                             const float* __restrict__ B, const int* __restrict__ tex,
                             const int* __restrict__ tabs, uint8_t* __restrict__ frames) {
  const int X = blockIdx.x * blockDim.x + threadIdx.x, Y = blockIdx.y;
  const int f = f0 + blockIdx.z, ch = f >> 2, o = f & 3;
  if (X >= g.bw) return;
  const size_t si = (size_t)dev::mirror(Y, kBorder, g.h) * g.w + dev::mirror(X, kBorder, g.w);
  int lab;
  if (ch == 3) {
    lab = tex[si];
  } else {
    const float v = (ch == 0 ? L : ch == 1 ? A : B)[si];
    lab = (int)floorf(v * 25.0f);
    if (lab == 25) lab = 24;
  }
  const int* t = tabs + g.tab_off[o];
  const int rx = t[2 * g.bw + Y] + t[X];
  const int ry = t[2 * g.bw + g.bh + Y] + t[g.bw + X];
  frames[g.lab_off[f] + (size_t)ry * g.nw[o] + rx] = (uint8_t)lab;
}

// gradient.cu:66-87: per-bin inclusive prefix counts along each row of a
// rotated frame with BP bins per pixel.  Block = one row; thread = (bin,
// one of 256/BP row segments).  Frames f0 + blockIdx.y.
template <int BP>
__global__ __launch_bounds__(256) void k_integral_rows(FrameGeom g, int f0, const uint8_t* __restrict__ frames,
                                                       uint16_t* __restrict__ I) {
  constexpr int NSEG = 256 / BP;
  extern __shared__ uint8_t row[];
  __shared__ uint32_t segtot[NSEG][BP];
  const int f = f0 + blockIdx.y, o = f & 3, y = blockIdx.x;
  const int nw = g.nw[o];
  if (y >= g.nh[o]) return;
  const uint8_t* src = frames + g.lab_off[f] + (size_t)y * nw;
  for (int i = threadIdx.x; i < nw; i += 256) row[i] = src[i];
  __syncthreads();
  const int bin = threadIdx.x % BP, seg = threadIdx.x / BP;
  const int len = (nw + NSEG - 1) / NSEG, x0 = seg * len, x1 = min(nw, x0 + len);
  uint32_t c = 0;
  for (int x = x0; x < x1; x++) c += (row[x] == bin);
  segtot[seg][bin] = c;
  __syncthreads();
  uint32_t run = 0;
  for (int s = 0; s < seg; s++) run += segtot[s][bin];
  uint16_t* dst = I + int_index(g, f, (long long)y * nw, bin);
  for (int x = x0; x < x1; x++) {
    run += (row[x] == bin);
    dst[(size_t)x * 8] = (uint16_t)run;
  }
}

// gradient.cu:89-103: column pass, two bins per thread, modulo 2^16.
__global__ __launch_bounds__(256) void k_integral_cols(FrameGeom g, int f0, uint16_t* __restrict__ I) {
  const int f = f0 + blockIdx.y, o = f & 3;
  const int nw = g.nw[o], nh = g.nh[o], pairs = bin_pitch(g, f) / 2;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;  // (x, bin pair)
  if (t >= nw * pairs) return;
  const int x = t / pairs, pr = t - x * pairs;
  uint32_t* col = reinterpret_cast<uint32_t*>(I + int_index(g, f, x, 2 * pr));
  const size_t stride = (size_t)nw * 4;  // u32 words per plane row
  uint32_t lo = 0, hi = 0;
  int y = 0;
  for (; y + 8 <= nh; y += 8) {
    uint32_t v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = col[(size_t)(y + k) * stride];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      lo += v[k] & 0xffffu;
      hi += v[k] >> 16;
      col[(size_t)(y + k) * stride] = (lo & 0xffffu) | (hi << 16);
    }
  }
  for (; y < nh; y++) {
    const uint32_t v = col[(size_t)y * stride];
    lo += v & 0xffffu;
    hi += v >> 16;
    col[(size_t)y * stride] = (lo & 0xffffu) | (hi << 16);
  }
}

// Single-write integral images.  A frame is cut into bands of kBand rows and
// strips of 64 columns; one wave owns a (strip, band) and lane x one column.
// Going down the band's rows it keeps, per bin, the running sum of the
// strip's row prefixes, L(x, y) = number of the bin's labels in the strip's
// columns <= x of the band's rows <= y: per row and bin a compare, the two
// mbcnt instructions that count the wave's matching lanes below (accumulating
// into L) and an add with carry for the lane's own match.  Then
//   I(x, y) = C_b(x) + R_s(y) + L(x, y)  (modulo 2^16 per bin)
// with R_s(y) the same sum over the band's strips left of s (the last lane's
// L of those strips, scanned over the strips by k_strip_carry) and C_b(x)
// that of the earlier bands' last rows (k_band_carry).  Pass 1 (FINAL =
// false) leaves each row's last-lane L and each band's last row; pass 2
// recomputes L and writes every integral value once: a wave's store to one
// plane is one contiguous kilobyte.  No barriers and no LDS: with one block
// per band whose 16 waves exchanged their row totals through LDS at a
// barrier per row the two passes took 143 + 126 us (L/a/b frames) and 55 +
// 51 us (texton frames) at 481x321, and take 64 + 30 and 30 + 17 us.  Pass 1
// is bound by its VALU instructions (about 8 per pixel and bin pair).
constexpr int kBand = 16;
constexpr int kStrip = 64;

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t add_u16x2(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) + __builtin_bit_cast(u16x2, b));
}

template <int BP, int NBU, bool FINAL>
__global__ __launch_bounds__(256) void k_integral_strip(FrameGeom g, int f0, int4 first,
                                                        const uint8_t* __restrict__ frames,
                                                        uint16_t* __restrict__ bands, uint32_t* __restrict__ rows,
                                                        const uint32_t* __restrict__ carry,
                                                        uint16_t* __restrict__ I) {
  constexpr int NQ = BP / 2;          // words per record (two bins each)
  constexpr int NQU = (NBU + 1) / 2;  // words holding used bins (labels are < NBU; higher bins stay 0)
  // blocks of a channel's four frames follow each other: first = the first
  // block of orientations 1, 2, 3 and of the next channel; numbered
  // XCD-aware, so neighbouring strips, whose stores share cache lines (a
  // frame's rows are not line-aligned), mostly meet in one L2
  const int lb = dev::xcd_block(blockIdx.x, gridDim.x);
  const int ch = lb / first.w, in_ch = lb - ch * first.w;
  const int o = in_ch < first.x ? 0 : in_ch < first.y ? 1 : in_ch < first.z ? 2 : 3, f = f0 + 4 * ch + o;
  const int blk = in_ch - (o == 0 ? 0 : o == 1 ? first.x : o == 2 ? first.y : first.z);
  const int nw = g.nw[o], nh = g.nh[o], ns = (nw + kStrip - 1) / kStrip;
  const int lane = threadIdx.x & 63;
  const int unit = blk * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int b = unit / ns, s = unit - b * ns;
  const int y0 = b * kBand;
  if (y0 >= nh) return;  // past this frame's last band
  const int y1 = min(nh, y0 + kBand), x = s * kStrip + lane;
  const bool in = x < nw;
  uint32_t L[2 * NQU];
#pragma unroll
  for (int k = 0; k < 2 * NQU; k++) L[k] = 0;
  uint16_t* rec = bands + g.band_off[f] + ((size_t)b * nw + (in ? x : 0)) * BP;
  uint32_t C[NQU];
#pragma unroll
  for (int q = 0; q < NQU; q++) C[q] = 0;
  if (FINAL) {
#pragma unroll
    for (int q = 0; q < NQ; q += 4)
      if (q < NQU) {
        const uint4 v = *reinterpret_cast<const uint4*>(rec + 2 * q);
        C[q] = v.x;
        if (q + 1 < NQU) C[q + 1] = v.y;
        if (q + 2 < NQU) C[q + 2] = v.z;
        if (q + 3 < NQU) C[q + 3] = v.w;
      }
  }
  const uint8_t* lab = frames + g.lab_off[f] + x;
  size_t row = (size_t)g.row_off[f] + ((size_t)y0 * ns + s) * NQ;  // this row's and strip's record
  const size_t npx = (size_t)nw * nh;
  uint4* dst = reinterpret_cast<uint4*>(I + g.int_off[f]) + (size_t)y0 * nw + x;
  constexpr int kAhead = 4;  // rows whose labels are loaded together, one group ahead
  uint32_t next[kAhead];
#pragma unroll
  for (int r = 0; r < kAhead; r++) next[r] = in && y0 + r < y1 ? (uint32_t)lab[(size_t)(y0 + r) * nw] : 255u;
#pragma unroll 1
  for (int yb = y0; yb < y1; yb += kAhead) {
    uint32_t cur[kAhead];
#pragma unroll
    for (int r = 0; r < kAhead; r++) {
      cur[r] = next[r];
      const int y = yb + kAhead + r;
      next[r] = in && y < y1 ? (uint32_t)lab[(size_t)y * nw] : 255u;
    }
#pragma unroll
    for (int r = 0; r < kAhead; r++) {
      if (yb + r >= y1) break;
      uint32_t R[NQU];
#pragma unroll
      for (int q = 0; q < NQU; q++) R[q] = FINAL ? carry[row + q] : 0u;  // wave-uniform: scalar loads
#pragma unroll
      for (int k0 = 0; k0 < NBU; k0 += 5) {  // five masks at a time: none is read right after its compare
        unsigned long long m[5];
#pragma unroll
        for (int k = k0; k < k0 + 5 && k < NBU; k++) m[k - k0] = __ballot(cur[r] == (uint32_t)k);
#pragma unroll
        for (int k = k0; k < k0 + 5 && k < NBU; k++)
          L[k] = __builtin_amdgcn_mbcnt_hi((uint32_t)(m[k - k0] >> 32),
                                           __builtin_amdgcn_mbcnt_lo((uint32_t)m[k - k0], L[k])) +
                 (cur[r] == (uint32_t)k);
      }
      uint32_t W[NQ];
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        W[q] = 0;
        if (q < NQU) {
          W[q] = __builtin_amdgcn_perm(L[2 * q + 1], L[2 * q], 0x05040100u);  // low halves
          if (FINAL) W[q] = add_u16x2(add_u16x2(W[q], C[q]), R[q]);
        }
      }
      if (FINAL) {
        if (in)
#pragma unroll
          for (int q = 0; q < NQ; q += 4) dst[(size_t)(q / 4) * npx] = make_uint4(W[q], W[q + 1], W[q + 2], W[q + 3]);
      } else {
        uint4* rd = reinterpret_cast<uint4*>(rows + row);
        if (lane == kStrip - 1)
#pragma unroll
          for (int q = 0; q < NQ; q += 4) rd[q / 4] = make_uint4(W[q], W[q + 1], W[q + 2], W[q + 3]);
        if (in && yb + r == y1 - 1) {
          uint4* bd = reinterpret_cast<uint4*>(rec);
#pragma unroll
          for (int q = 0; q < NQ; q += 4) bd[q / 4] = make_uint4(W[q], W[q + 1], W[q + 2], W[q + 3]);
        }
      }
      row += (size_t)ns * NQ;
      dst += nw;
    }
  }
}

// Rows of last-lane sums -> exclusive prefix over the row's strips (in
// place); one thread per (row, word).
__global__ __launch_bounds__(256) void k_strip_carry(FrameGeom g, int f0, uint32_t* __restrict__ rows) {
  const int f = f0 + blockIdx.y, o = f & 3;
  const int ns = (g.nw[o] + kStrip - 1) / kStrip, nq = bin_pitch(g, f) / 2;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= g.nh[o] * nq) return;
  const int y = e / nq, q = e - y * nq;
  uint32_t* p = rows + g.row_off[f] + (size_t)y * ns * nq + q;
  uint32_t acc = 0;
  for (int s0 = 0; s0 < ns; s0 += 8) {
    uint32_t t[8];
#pragma unroll
    for (int k = 0; k < 8; k++) t[k] = s0 + k < ns ? p[(size_t)(s0 + k) * nq] : 0u;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (s0 + k < ns) p[(size_t)(s0 + k) * nq] = acc;
      acc = add_u16x2(acc, t[k]);
    }
  }
}

// Each band's last row, completed by its strips' carries, -> exclusive
// prefix over the bands of each frame (in place).  A block owns 32 pieces of
// a row (one column's 16 bytes each) and 8 groups of threads that share the
// frame's bands: every group sums its bands, the groups' sums meet in LDS,
// and each writes its bands' prefixes (one chain over 58 bands per thread
// was 20 us at 481x321 for the L/a/b and for the texton frames; this is 11).
constexpr int kCarryCols = 32, kCarrySegs = 8;
__global__ __launch_bounds__(256) void k_band_carry(FrameGeom g, int f0, const uint32_t* __restrict__ rows,
                                                    uint16_t* __restrict__ bands) {
  __shared__ uint4 sums[kCarrySegs][kCarryCols];
  const int f = f0 + blockIdx.y, o = f & 3;
  const int nw = g.nw[o], nh = g.nh[o], nb = (nh + kBand - 1) / kBand, n4 = bin_pitch(g, f) / 8;
  const int ns = (nw + kStrip - 1) / kStrip;
  const int c = threadIdx.x % kCarryCols, seg = threadIdx.x / kCarryCols;
  const int e = blockIdx.x * kCarryCols + c;
  const bool in = e < nw * n4;
  const int s = in ? e / n4 / kStrip : 0, q = in ? e % n4 : 0;
  uint4* p = reinterpret_cast<uint4*>(bands + g.band_off[f]) + (in ? e : 0);
  const uint4* r = reinterpret_cast<const uint4*>(rows + g.row_off[f]) + (size_t)s * n4 + q;
  const size_t stride = (size_t)nw * n4;
  const int per = (nb + kCarrySegs - 1) / kCarrySegs, b0 = seg * per, b1 = min(nb, b0 + per);
  auto add = [](uint4& a, const uint4& v) {
    a.x = add_u16x2(a.x, v.x);
    a.y = add_u16x2(a.y, v.y);
    a.z = add_u16x2(a.z, v.z);
    a.w = add_u16x2(a.w, v.w);
  };
  auto band = [&](int b) {
    uint4 t = p[(size_t)b * stride];
    add(t, r[(size_t)(min(nh, (b + 1) * kBand) - 1) * ns * n4]);
    return t;
  };
  uint4 acc = make_uint4(0u, 0u, 0u, 0u);
  if (in)
#pragma unroll 8
    for (int b = b0; b < b1; b++) add(acc, band(b));
  sums[seg][c] = acc;
  __syncthreads();
  acc = make_uint4(0u, 0u, 0u, 0u);
  for (int k = 0; k < seg; k++) add(acc, sums[k][c]);
  if (!in) return;
  for (int b = b0; b < b1; b += 4) {
    uint4 t[4];
#pragma unroll
    for (int k = 0; k < 4; k++) t[k] = band(min(b + k, nb - 1));
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (b + k < b1) {
        p[(size_t)(b + k) * stride] = acc;
        add(acc, t[k]);
      }
  }
}

struct BlurK {
  float k[16];
};

// rotate.cu:352-370: zero-padded correlation over bins.  A padding term
// fma(0, k, s) leaves s unchanged (s >= +0, k finite), so it is not formed.
template <int NB, int KR>
__device__ __forceinline__ void blur_bins(float (&v)[32], const BlurK& bk) {
  float c[NB];
#pragma unroll
  for (int i = 0; i < NB; i++) {
    float s = 0.f;
#pragma unroll
    for (int nk = 0; nk < 2 * KR + 1; nk++) {
      const int j = i - KR + nk;
      if (j >= 0 && j < NB) s = fmaf(v[j], bk.k[nk], s);
    }
    c[i] = s;
  }
#pragma unroll
  for (int i = 0; i < NB; i++) v[i] = c[i];
}

// rotate.cu:263-475 computeGradient: one (pixel, scale, split) per thread.
// NB bins, KR blur radius (0 = no blur).  Output plane of channel ch:
// [scale][slot] with slot o+4 for the top/bottom split (sense A) and slot o
// for the left/right split (sense B) (gradient.cu:240-241).
// c[i0] - c[i1] + c[i2] - c[i3] of packed corner counts, two bins per word,
// each half modulo 2^16 on its own.
template <int NB>
__device__ __forceinline__ void corner_sum(const uint32_t (&pk)[8][16], int i0, int i1, int i2, int i3,
                                           uint32_t (&out)[16]) {
#pragma unroll
  for (int e = 0; e < 16; e++)
    out[e] = 2 * e < NB ? __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, pk[i0][e]) -
                                                           __builtin_bit_cast(u16x2, pk[i1][e]) +
                                                           __builtin_bit_cast(u16x2, pk[i2][e]) -
                                                           __builtin_bit_cast(u16x2, pk[i3][e]))
                        : 0u;
}

// n / s for the values that occur in chi^2 (0 or n in [2^-80, 2^7], s
// in [2^-17, 2^10]), where no scaling is needed: Newton steps with fused
// multiply-adds from the hardware reciprocal, whose last correction rounds
// correctly (Markstein, IBM J. Res. Dev. 34, 1990), so the quotient is the
// IEEE one.  It saves the scaling and fix-up instructions of the general
// sequence and leaves no branch per bin.
__device__ __forceinline__ float div_exact(float n, float s) {
  float r = __builtin_amdgcn_rcpf(s);
  r = fmaf(fmaf(-s, r, 1.0f), r, r);
  float q = n * r;
  q = fmaf(fmaf(-s, q, n), r, q);
  return fmaf(fmaf(-s, q, n), r, q);
}

// chi^2 of one split of the half-disc pair from the packed corner counts:
// a = c[i0] - c[i1] + c[i2] - c[i3], b = c[j0] - c[j1] + c[j2] - c[j3] per
// bin (uint16 modulo arithmetic recovers the exact counts), optional bin
// blur, normalisation to sum 8 and 0.5 * sum (a-b)^2/(a+b) with the
// reference's 32-slot tree sums (rotate.cu:352-472).
// PAIR: the pixel's 64 bins are split over this lane (32 bins in pk) and
// its neighbour lane (lane ^ 1); each 32-slot tree sum is completed with the
// partner's as lo + hi (rotate.cu:384-389 adds slot 32 to slot 0), and IEEE
// addition being commutative both lanes hold the same total.
template <int NB, int KR, bool PAIR = false>
__device__ __forceinline__ float chi2_split(const uint32_t (&pa)[16], const uint32_t (&pb)[16],
                                            const BlurK& bk) {
  static_assert(!PAIR || (NB == 32 && KR == 0), "paired halves hold 32 unblurred bins");
  float a[32], b[32];
#pragma unroll
  for (int e = 0; e < 32; e++) {
    a[e] = e < NB ? (float)((pa[e / 2] >> (16 * (e & 1))) & 0xffffu) : 0.f;
    b[e] = e < NB ? (float)((pb[e / 2] >> (16 * (e & 1))) & 0xffffu) : 0.f;
  }
  if constexpr (KR > 0) {
    blur_bins<NB, KR>(a, bk);
    blur_bins<NB, KR>(b, bk);
  }
  // slots NB..31 hold +0 and every other slot is >= +0, so the tree sums
  // skip the additions of those zeros (x + 0 = x exactly) and the chi terms
  // of the empty slots are not formed
  float t32[32];
#pragma unroll
  for (int i = 0; i < 32; i++) t32[i] = a[i];
  float sa = dev::tree32z<NB>(t32);
  if (PAIR) sa = sa + __shfl_xor(sa, 1, 64);
  const float na = (sa != 0.f) ? div_exact(8.0f, sa) : 0.f;
#pragma unroll
  for (int i = 0; i < 32; i++) t32[i] = b[i];
  float sb = dev::tree32z<NB>(t32);
  if (PAIR) sb = sb + __shfl_xor(sb, 1, 64);
  const float nb = (sb != 0.f) ? div_exact(8.0f, sb) : 0.f;
#pragma unroll
  for (int i = 0; i < 32; i++) {
    float chi = 0.f;
    if (i < NB) {
      const float ai = a[i] * na, bi = b[i] * nb;
      const float s = ai + bi, d = ai - bi;
      const float quot = div_exact(d * d, s);  // NaN for an empty bin
      chi = s != 0.f ? quot : 0.f;
    }
    t32[i] = chi;
  }
  float c = dev::tree32z<NB>(t32);
  if (PAIR) c = c + __shfl_xor(c, 1, 64);
  return 0.5f * c;
}

// The pixels of a block: a 16 x 16 patch, 16 x 4 per wave.  In a rotated
// frame a run of image pixels is a slanted line (orientation 2: a diagonal,
// 3: nearly a column), so 64 pixels of one image row touch up to 64 cache
// lines per corner load and use 16 bytes of each; a patch stays compact in
// every orientation.  With runs of 64 pixels the three launches took 352 /
// 181 / 178 us at 481x321, and take 249 / 147 / 114 us (8 x 8 per wave 251 /
// 152 / 123, 32 x 2 274 / 154 / 134), near four fifths of the VALU issue rate.
constexpr int GWX = 16, GPX = 16, GPY = 256 / GPX;

// Both splits of one (pixel, scale, orientation): the eight corners A..H
// are loaded once (uint16 counts, 8 bins per 16-byte load) and feed
//   sense A (top/bottom, slot o+4): a = A-C+E-D, b = H-F+D-E
//   sense B (left/right, slot o):   a = A-F+G-B, b = H-C+B-G
// (rotate.cu:400-445; gradient.cu:240-241).
// Blocks: blockIdx.x runs over (patch, scale) with the scale fastest,
// numbered XCD-aware, so each XCD handles a contiguous band of image rows at
// all three scales and its L2 keeps the band's rotated integral rows (plus
// the corner reach above and below) for every gather; blockIdx.y is the
// (channel, orientation).
template <int NB, int KR>
__global__ __launch_bounds__(256, 3) void k_gradients(FrameGeom g, int ch0, int rad0, const int* __restrict__ tabs,
                                                   const uint16_t* __restrict__ I, BlurK bk,
                                                   float* __restrict__ grads, size_t plane) {
  const int bl = dev::xcd_block(blockIdx.x, gridDim.x);
  const int scale = bl % 3, patch = bl / 3, ntx = (g.w + GPX - 1) / GPX;
  const int ch = ch0 + (blockIdx.y >> 2), o = blockIdx.y & 3, f = ch * 4 + o;
  const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
  const int x = (patch % ntx) * GPX + (wv % (GPX / GWX)) * GWX + ln % GWX;
  const int y = (patch / ntx) * GPY + (wv / (GPX / GWX)) * (64 / GWX) + ln / GWX;
  if (x >= g.w || y >= g.h) return;
  const int p = y * g.w + x;
  const int* t = tabs + g.tab_off[o];
  const int ix = x + kBorder, iy = y + kBorder;
  const int rx = t[2 * g.bw + iy] + t[ix];
  const int ry = t[2 * g.bw + g.bh + iy] + t[g.bw + ix];
  const long long pix = (long long)ry * g.nw[o] + rx;
  const int* rc = g.rect[o][rad0 + scale];
  const uint4* base = reinterpret_cast<const uint4*>(I + g.int_off[f]);
  const size_t npx = (size_t)g.nw[o] * g.nh[o];
  constexpr int NQ = (NB + 7) / 8;
  uint32_t pk[8][16];
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const uint4* src = base + (size_t)(rc[c] + pix);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (q < NQ) {
        const uint4 v = src[q * npx];
        pk[c][4 * q] = v.x;
        pk[c][4 * q + 1] = v.y;
        pk[c][4 * q + 2] = v.z;
        pk[c][4 * q + 3] = v.w;
      } else {
        pk[c][4 * q] = pk[c][4 * q + 1] = pk[c][4 * q + 2] = pk[c][4 * q + 3] = 0u;
      }
    }
  }
  // corner indices: A0 B1 C2 D3 E4 F5 G6 H7
  uint32_t ta[16], tb[16], la[16], lb[16];
  corner_sum<NB>(pk, 0, 2, 4, 3, ta);
  corner_sum<NB>(pk, 7, 5, 3, 4, tb);
  corner_sum<NB>(pk, 0, 5, 6, 1, la);
  corner_sum<NB>(pk, 7, 2, 1, 6, lb);
  const float top = chi2_split<NB, KR>(ta, tb, bk);
  const float left = chi2_split<NB, KR>(la, lb, bk);
  float* dst = grads + (size_t)((ch * 3 + scale) * 8) * plane + p;
  dst[(size_t)(o + 4) * plane] = top;
  dst[(size_t)o * plane] = left;
}

// The texture channel with 64 textons (rotate.cu:780-782,
// computeGradient<64, 64, false, *>): lanes 2p and 2p+1 share pixel p,
// holding bins 0..31 and 32..63 of every corner (integral planes 0..3 and
// 4..7).  Output as k_gradients.
constexpr int GHX = 16, GHY = 8;  // a block's patch: four waves of 8 x 4 pixels
__global__ __launch_bounds__(256, 3) void k_gradients64(FrameGeom g, int rad0, const int* __restrict__ tabs,
                                                     const uint16_t* __restrict__ I, float* __restrict__ grads,
                                                     size_t plane) {
  const int bl = dev::xcd_block(blockIdx.x, gridDim.x);  // (patch, scale), as k_gradients
  const int scale = bl % 3, patch = bl / 3, ntx = (g.w + GHX - 1) / GHX;
  const int ch = 3, o = blockIdx.y, f = ch * 4 + o;
  const int wv = threadIdx.x >> 6, ln = (threadIdx.x & 63) >> 1, half = threadIdx.x & 1;
  const int xx = (patch % ntx) * GHX + (wv & 1) * 8 + ln % 8, yy = (patch / ntx) * GHY + (wv >> 1) * 4 + ln / 8;
  const bool live = xx < g.w && yy < g.h;
  // both lanes of a pair agree; all lanes reach the shuffles
  const int x = live ? xx : g.w - 1, y = live ? yy : g.h - 1, p = y * g.w + x;
  const int* t = tabs + g.tab_off[o];
  const int ix = x + kBorder, iy = y + kBorder;
  const int rx = t[2 * g.bw + iy] + t[ix];
  const int ry = t[2 * g.bw + g.bh + iy] + t[g.bw + ix];
  const long long pix = (long long)ry * g.nw[o] + rx;
  const int* rc = g.rect[o][rad0 + scale];
  const size_t npx = (size_t)g.nw[o] * g.nh[o];
  const uint4* base = reinterpret_cast<const uint4*>(I + g.int_off[f]) + (size_t)(4 * half) * npx;  // planes 4h..4h+3
  uint32_t pk[8][16];
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const uint4* src = base + (size_t)(rc[c] + pix);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const uint4 v = src[q * npx];
      pk[c][4 * q] = v.x;
      pk[c][4 * q + 1] = v.y;
      pk[c][4 * q + 2] = v.z;
      pk[c][4 * q + 3] = v.w;
    }
  }
  BlurK none{};
  uint32_t ta[16], tb[16], la[16], lb[16];
  corner_sum<32>(pk, 0, 2, 4, 3, ta);
  corner_sum<32>(pk, 7, 5, 3, 4, tb);
  corner_sum<32>(pk, 0, 5, 6, 1, la);
  corner_sum<32>(pk, 7, 2, 1, 6, lb);
  const float top = chi2_split<32, 0, true>(ta, tb, none);
  const float left = chi2_split<32, 0, true>(la, lb, none);
  if (live && half == 0) {
    float* dst = grads + (size_t)((ch * 3 + scale) * 8) * plane + p;
    dst[(size_t)(o + 4) * plane] = top;
    dst[(size_t)o * plane] = left;
  }
}

// Parabola smoothing (parabola.cu:75-124 / parabola_kernel.cu:1-30) of all
// planes of a channel group in one launch.
// Each thread computes QX horizontally adjacent outputs from a tile staged
// in LDS.  The filter of a radius and orientation is a list of pieces of
// four horizontally adjacent taps, row by row (v ascending, the reference's
// outer loop) and u ascending within a row, that cover its non-zero taps:
// per piece a scalar load of the four coefficients and three 16-byte LDS
// reads feed 4 QX multiply-adds.  A covered tap outside the ellipse has
// coefficient 0 and fma(x, 0, acc) == acc for finite x (acc starts at +0 and
// can never become -0), so the sums equal the reference's zero-skipping loop
// bit for bit.  The ellipse (axes r and r/4) holds a fifth of its square:
// dense rows of 2 r + 1 taps took 120 us per channel at radius 20 (481x321),
// 330 us for all 96 planes in nine launches; the lists take 128 us in one (59 us
// of multiply-adds, 44 us of LDS reads; staging the tile row by row, with one
// row's loads in flight, cost another 50).
constexpr int QX = 8, QCOLS = 16, QTX = QX * QCOLS, QTY = 32, QNT = QCOLS * QTY;

__host__ __device__ constexpr int q_lw(int r) { return QTX - QX + 2 * r / 4 * 4 + 12; }  // tile row, floats
__host__ __device__ constexpr int q_lh(int r) { return QTY + 2 * r; }

struct ParabolaJobs {
  int n;                              // (channel, scale) pairs, largest radius first
  int ch[12], scale[12], radius[12];
  int first[12][8], count[12][8];     // pieces of the pair's orientations
};

__global__ __launch_bounds__(QNT) void k_parabola(int w, int h, ParabolaJobs J, const float* __restrict__ grads,
                                                  size_t gplane, const float4* __restrict__ coef,
                                                  const int* __restrict__ at, CueOut out, int pitch) {
  extern __shared__ float4 tile4[];
  float* tile = reinterpret_cast<float*>(tile4);
  const int job = blockIdx.z >> 3, o = blockIdx.z & 7;
  const int ch = J.ch[job], scale = J.scale[job], R = J.radius[job], LW = q_lw(R), LH = q_lh(R);
  const float* src = grads + (size_t)((ch * 3 + scale) * 8 + o) * gplane;
  const int x0 = blockIdx.x * QTX, y0 = blockIdx.y * QTY;
  const int lane = threadIdx.x & 63;
  // tile columns past the image only feed discarded outputs: clamp into the
  // mirrored range [0, w + 2*border) before reflecting
  int gx[3];
#pragma unroll
  for (int k = 0; k < 3; k++)
    gx[k] = dev::mirror(dev::clampi(x0 + lane + 64 * k - R + kBorder, 0, w + 2 * kBorder - 1), kBorder, w);
  constexpr int kRows = 3;  // tile rows per wave whose loads are in flight together
  for (int l0 = threadIdx.x >> 6; l0 < LH; l0 += kRows * (QNT / 64)) {
    float t[kRows][3];
#pragma unroll
    for (int r = 0; r < kRows; r++) {
      const int ly = l0 + r * (QNT / 64);
      const int gy = dev::mirror(dev::clampi(y0 + ly - R + kBorder, 0, h + 2 * kBorder - 1), kBorder, h);
      const float* row = src + (size_t)gy * w;
#pragma unroll
      for (int k = 0; k < 3; k++) t[r][k] = row[gx[k]];
    }
#pragma unroll
    for (int r = 0; r < kRows; r++) {
      const int ly = l0 + r * (QNT / 64);
#pragma unroll
      for (int k = 0; k < 3; k++)
        if (ly < LH && lane + 64 * k < LW) tile[ly * LW + lane + 64 * k] = t[r][k];
    }
  }
  __syncthreads();
  const int tx = (threadIdx.x % QCOLS) * QX, ty = threadIdx.x / QCOLS;
  const int first = J.first[job][o], last = first + J.count[job][o];
  const float4* base = tile4 + (ty * LW + tx) / 4;
  float acc[QX];
#pragma unroll
  for (int j = 0; j < QX; j++) acc[j] = 0.0f;
#pragma unroll 4
  for (int i = first; i < last; i++) {
    const float4 c = coef[i];
    const float4* p = base + at[i];
    const float4 a = p[0], b = p[1], d = p[2];
    const float seg[12] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, d.x, d.y, d.z, d.w};
    const float cf[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int j = 0; j < QX; j++) acc[j] = fmaf(seg[j + u], cf[u], acc[j]);
  }
  float* dst = out.p[ch] + (size_t)(scale * 8 + o) * pitch;
  const int gy = y0 + ty;
  if (gy < h)
#pragma unroll
    for (int j = 0; j < QX; j++)
      if (x0 + tx + j < w) dst[(size_t)gy * w + x0 + tx + j] = acc[j];
}

// ---------------------------------------------------------------- host plan

struct CuePlan {
  int w = -1, h = -1;
  FrameGeom g;
  size_t lab_bytes = 0, int_elems = 0, band_elems = 0, row_words = 0;
  int* d_tabs = nullptr;
  // smoothing filters as pieces of four taps: coefficients, float4 offset of
  // the piece in a tile of its radius, and [radius][orientation] ranges
  float4* d_piece_coef = nullptr;
  int* d_piece_at = nullptr;
  int piece_first[4][8], piece_count[4][8];
  BlurK blur_bg, blur_cg;
  int kr_bg = 0, kr_cg = 0;
  ~CuePlan() {
    if (d_tabs) (void)hipFree(d_tabs);
    if (d_piece_coef) (void)hipFree(d_piece_coef);
    if (d_piece_at) (void)hipFree(d_piece_at);
  }
};

int build_plan(hipStream_t s, int w, int h, int tbp, CuePlan& P) {
  FrameGeom& g = P.g;
  memset(&g, 0, sizeof(g));
  g.w = w; g.h = h; g.bw = w + 2 * kBorder; g.bh = h + 2 * kBorder;
  g.tbp = tbp;
  std::vector<int> tabs;
  std::vector<int> bX(g.bw), bY(g.bw), gX(g.bh), gY(g.bh);
  for (int o = 0; o < 4; o++) {
    const float thetaPi = -float(o) / float(8);
    if (rotation_tables(g.bw, g.bh, thetaPi, &g.nw[o], &g.nh[o], bX.data(), bY.data(), gX.data(), gY.data()))
      return fail(DMSC_ERR_INTERNAL, "rotation tables failed for %dx%d", w, h);
    g.tab_off[o] = (int)tabs.size();
    tabs.insert(tabs.end(), bX.begin(), bX.end());
    tabs.insert(tabs.end(), bY.begin(), bY.end());
    tabs.insert(tabs.end(), gX.begin(), gX.end());
    tabs.insert(tabs.end(), gY.begin(), gY.end());
    for (int ri = 0; ri < 4; ri++)
      halfdisc_offsets(w, h, thetaPi, kRadii[ri], bX.data(), bY.data(), gX.data(), gY.data(), g.nw[o],
                       g.rect[o][ri]);
  }
  // Every gather below must stay inside its rotated frame: verify on the host
  // (labels scatter over the whole mirrored image; corners around every
  // interior pixel for all radii).
  for (int o = 0; o < 4; o++) {
    const int* t = tabs.data() + g.tab_off[o];
    const int *tbX = t, *tbY = t + g.bw, *tgX = t + 2 * g.bw, *tgY = t + 2 * g.bw + g.bh;
    for (int Y = 0; Y < g.bh; Y++)
      for (int X = 0; X < g.bw; X++) {
        const int rx = tgX[Y] + tbX[X], ry = tgY[Y] + tbY[X];
        if (rx < 0 || ry < 0 || rx >= g.nw[o] || ry >= g.nh[o])
          return fail(DMSC_ERR_INTERNAL, "rotation maps outside the frame (o=%d)", o);
      }
    long long lo_off = 0, hi_off = 0;
    for (int ri = 0; ri < 4; ri++)
      for (int k = 0; k < 8; k++) {
        lo_off = std::min(lo_off, (long long)g.rect[o][ri][k]);
        hi_off = std::max(hi_off, (long long)g.rect[o][ri][k]);
      }
    const long long npx = (long long)g.nw[o] * g.nh[o];
    for (int y = 0; y < h; y++)
      for (int x = 0; x < w; x++) {
        const int X = x + kBorder, Y = y + kBorder;
        const long long pix = (long long)(tgY[Y] + tbY[X]) * g.nw[o] + (tgX[Y] + tbX[X]);
        if (pix + lo_off < 0 || pix + hi_off >= npx)
          return fail(DMSC_ERR_INTERNAL, "half-disc corners leave the frame (o=%d)", o);
      }
  }
  size_t lo = 0, io = 0, bo = 0, ro = 0;
  for (int f = 0; f < kFrames; f++) {
    const int o = f & 3;
    g.lab_off[f] = (long long)lo;
    g.int_off[f] = (long long)io;
    g.band_off[f] = (long long)bo;
    g.row_off[f] = (long long)ro;
    lo += ((size_t)g.nw[o] * g.nh[o] + 255) & ~(size_t)255;
    io += (size_t)g.nw[o] * g.nh[o] * (f >= 12 ? tbp : 32);
    bo += (size_t)div_up(g.nh[o], kBand) * g.nw[o] * (f >= 12 ? tbp : 32);
    ro += (size_t)g.nh[o] * div_up(g.nw[o], kStrip) * (f >= 12 ? tbp : 32) / 2;
  }
  P.lab_bytes = lo;
  P.int_elems = io;
  P.band_elems = bo;
  P.row_words = ro;
  DMSC_HIP(hipMalloc(&P.d_tabs, sizeof(int) * tabs.size()));
  DMSC_HIP(hipMemcpy(P.d_tabs, tabs.data(), sizeof(int) * tabs.size(), hipMemcpyHostToDevice));
  std::vector<float4> piece_coef;
  std::vector<int> piece_at;
  for (int ri = 0; ri < 4; ri++) {
    const int r = kRadii[ri], len = 2 * r + 1;
    std::vector<float> filt((size_t)8 * len * len);
    parabola_filters(r, filt.data());
    for (int o = 0; o < 8; o++) {
      P.piece_first[ri][o] = (int)piece_coef.size();
      for (int v = 0; v < len; v++) {
        const float* row = filt.data() + ((size_t)o * len + v) * len;
        int u0 = len, u1 = -1;  // columns holding the row's non-zero taps
        for (int u = 0; u < len; u++)
          if (row[u] != 0.0f) {
            u0 = std::min(u0, u);
            u1 = u;
          }
        for (int u = u0 & ~3; u <= u1; u += 4) {
          auto tap = [&](int k) { return k < len ? row[k] : 0.0f; };
          piece_coef.push_back(make_float4(tap(u), tap(u + 1), tap(u + 2), tap(u + 3)));
          piece_at.push_back((v * q_lw(r) + u) / 4);
        }
      }
      P.piece_count[ri][o] = (int)piece_coef.size() - P.piece_first[ri][o];
    }
  }
  DMSC_HIP(hipMalloc(&P.d_piece_coef, sizeof(float4) * piece_coef.size()));
  DMSC_HIP(hipMemcpy(P.d_piece_coef, piece_coef.data(), sizeof(float4) * piece_coef.size(), hipMemcpyHostToDevice));
  DMSC_HIP(hipMalloc(&P.d_piece_at, sizeof(int) * piece_at.size()));
  DMSC_HIP(hipMemcpy(P.d_piece_at, piece_at.data(), sizeof(int) * piece_at.size(), hipMemcpyHostToDevice));
  // gradient.cu:233: blur sigma = (int)(sigma * nbins) -> Bg 2, Cg 1
  memset(&P.blur_bg, 0, sizeof(BlurK));
  memset(&P.blur_cg, 0, sizeof(BlurK));
  blur_kernel((float)(int)(0.1f * 25.0f), P.blur_bg.k, &P.kr_bg);
  blur_kernel((float)(int)(0.05f * 25.0f), P.blur_cg.k, &P.kr_cg);
  if (P.kr_bg != 6 || P.kr_cg != 3) return fail(DMSC_ERR_INTERNAL, "unexpected blur radii");
  P.w = w;
  P.h = h;
  (void)s;
  return DMSC_OK;
}

// Integral images of frames f0 .. f0 + nf - 1: BP bins per record, NBU of
// them used (the L/a/b frames hold 25 quantised bins in 32-bin records; the
// unused bins stay 0).
template <int BP, int NBU>
int integral_strips(hipStream_t s, const FrameGeom& g, int f0, int nf, const uint8_t* frames, uint16_t* bands,
                    uint32_t* rows, uint16_t* I) {
  int first[5] = {0}, row_words = 0, col_quads = 0;
  for (int o = 0; o < 4; o++) {
    first[o + 1] = first[o] + div_up(div_up(g.nw[o], kStrip) * div_up(g.nh[o], kBand), 4);
    row_words = std::max(row_words, g.nh[o] * (BP / 2));
    col_quads = std::max(col_quads, g.nw[o] * (BP / 8));
  }
  const int4 at = make_int4(first[1], first[2], first[3], first[4]);
  const dim3 grid(first[4] * (nf / 4));
  hipLaunchKernelGGL((k_integral_strip<BP, NBU, false>), grid, dim3(256), 0, s, g, f0, at, frames, bands,
                     rows, nullptr, nullptr);
  hipLaunchKernelGGL(k_strip_carry, dim3(div_up(row_words, 256), nf), dim3(256), 0, s, g, f0, rows);
  hipLaunchKernelGGL(k_band_carry, dim3(div_up(col_quads, kCarryCols), nf), dim3(256), 0, s, g, f0, rows, bands);
  hipLaunchKernelGGL((k_integral_strip<BP, NBU, true>), grid, dim3(256), 0, s, g, f0, at, frames, bands,
                     nullptr, rows, I);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}

// Byte offsets in the scratch arena: label frames (at 0), integral images,
// raw gradient planes, band sums, row carries.
struct ScratchLayout {
  size_t ints, grads, bands, rows, total;
};
ScratchLayout scratch_layout(const CuePlan& P) {
  ScratchLayout a;
  a.ints = P.lab_bytes;
  a.grads = a.ints + P.int_elems * sizeof(uint16_t);
  a.bands = a.grads + (size_t)4 * 24 * P.w * P.h * sizeof(float);
  a.rows = a.bands + P.band_elems * sizeof(uint16_t);
  a.total = a.rows + P.row_words * sizeof(uint32_t) + 1024;
  return a;
}

struct PlanCache {
  std::map<std::tuple<int, int, int>, std::unique_ptr<CuePlan>> plans;
};

}  // namespace

// Plans are cached per (w, h, texture bin pitch) and context; the map is
// shared by all contexts (and host threads), so it is only touched under
// plan_lock(), and a context's plans are dropped when it is destroyed.
static std::map<const Ctx*, PlanCache>& plan_caches() {
  static std::map<const Ctx*, PlanCache> caches;
  return caches;
}
static std::mutex& plan_lock() {
  static std::mutex m;
  return m;
}

static int get_plan(Ctx* ctx, int w, int h, int tbp, CuePlan** out) {
  const auto key = std::make_tuple(w, h, tbp);
  {
    std::lock_guard<std::mutex> lk(plan_lock());
    PlanCache& pc = plan_caches()[ctx];
    auto it = pc.plans.find(key);
    if (it != pc.plans.end()) {
      *out = it->second.get();
      return DMSC_OK;
    }
  }
  // built outside the lock: only this context's thread builds its plans
  std::unique_ptr<CuePlan> p(new CuePlan());
  DMSC_TRY(build_plan(ctx->stream, w, h, tbp, *p));
  std::lock_guard<std::mutex> lk(plan_lock());
  auto it = plan_caches()[ctx].plans.emplace(key, std::move(p)).first;
  *out = it->second.get();
  return DMSC_OK;
}

void release_local_cues(const Ctx* ctx) {
  std::lock_guard<std::mutex> lk(plan_lock());
  plan_caches().erase(ctx);
}

// localcues.cu:257-300 localCues, in two parts that may run on two streams:
// part 1 the L, a and b channels (frames 0..11: labels, integral images,
// Bg and Cg gradients and their parabola fits), which do not need the
// textons; part 2 the texton channel (frames 12..15: Tg); part 3 both.
// local_cues_prepare builds the plan and sizes the scratch arena first, so
// the parts only launch kernels and never reallocate while the other part
// runs.
int local_cues_prepare(Ctx* ctx, int w, int h, int ntex) {
  if (ntex != 32 && ntex != 64) return fail(DMSC_ERR_ARG, "local cues support 32 or 64 textons");
  CuePlan* P;
  DMSC_TRY(get_plan(ctx, w, h, ntex, &P));
  void* scratch;
  return ctx->scratch(1, scratch_layout(*P).total, &scratch);
}

int launch_local_cues_part(Ctx* ctx, hipStream_t s, int part, int w, int h, const float* L, const float* A,
                           const float* B, const int* tex, int ntex, float* bg, float* cga, float* cgb, float* tg,
                           int pitch, float* grads_out, hipEvent_t hist_done) {
  if (ntex != 32 && ntex != 64) return fail(DMSC_ERR_ARG, "local cues support 32 or 64 textons");
  if (part < 1 || part > 3) return fail(DMSC_ERR_INTERNAL, "bad local-cue part %d", part);
  const int tbp = ntex;
  CuePlan* P;
  DMSC_TRY(get_plan(ctx, w, h, tbp, &P));
  const FrameGeom& g = P->g;
  const int n = w * h;
  void* scratch;
  const ScratchLayout at = scratch_layout(*P);
  DMSC_TRY(ctx->scratch(1, at.total, &scratch));
  uint8_t* frames = (uint8_t*)scratch;
  uint16_t* I = (uint16_t*)((char*)scratch + at.ints);
  float* grads = grads_out ? grads_out : (float*)((char*)scratch + at.grads);
  uint16_t* bands = (uint16_t*)((char*)scratch + at.bands);
  uint32_t* rows = (uint32_t*)((char*)scratch + at.rows);
  const bool colour = part & 1, texture = part & 2;
  // frames of channel ch are f = 4 ch + o; the texture frames 12..15 come last
  const size_t split = (size_t)g.lab_off[12];
  const int f0 = colour ? 0 : 12, nf = (colour ? 12 : 0) + (texture ? 4 : 0);
  const size_t fill0 = colour ? 0 : split, fill1 = texture ? P->lab_bytes : split;
  hipLaunchKernelGGL(k_fill_u8, dim3(div_up(fill1 - fill0, 256)), dim3(256), 0, s, frames + fill0, fill1 - fill0);
  hipLaunchKernelGGL(k_cue_labels, dim3(div_up(g.bw, 256), g.bh, nf), dim3(256), 0, s, g, f0, L, A, B, tex,
                     P->d_tabs, frames);
  int maxh = 0, maxw = 0;
  for (int o = 0; o < 4; o++) { maxh = std::max(maxh, g.nh[o]); maxw = std::max(maxw, g.nw[o]); }
  if (colour) {
    if (integral_pass == 1) {
      DMSC_TRY((integral_strips<32, 25>(s, g, 0, 12, frames, bands, rows, I)));
    } else {
      hipLaunchKernelGGL(k_integral_rows<32>, dim3(maxh, 12), dim3(256), (size_t)maxw, s, g, 0, frames, I);
      hipLaunchKernelGGL(k_integral_cols, dim3(div_up(maxw * 32 / 2, 256), 12), dim3(256), 0, s, g, 0, I);
    }
  }
  if (texture) {
    if (integral_pass == 1) {
      if (tbp == 32) DMSC_TRY((integral_strips<32, 32>(s, g, 12, 4, frames, bands, rows, I)));
      else DMSC_TRY((integral_strips<64, 64>(s, g, 12, 4, frames, bands, rows, I)));
    } else {
      if (tbp == 32)
        hipLaunchKernelGGL(k_integral_rows<32>, dim3(maxh, 4), dim3(256), (size_t)maxw, s, g, 12, frames, I);
      else
        hipLaunchKernelGGL(k_integral_rows<64>, dim3(maxh, 4), dim3(256), (size_t)maxw, s, g, 12, frames, I);
      hipLaunchKernelGGL(k_integral_cols, dim3(div_up(maxw * tbp / 2, 256), 4), dim3(256), 0, s, g, 12, I);
    }
  }
  const size_t plane = (size_t)n;
  const int patches = div_up(w, GPX) * div_up(h, GPY);
  BlurK none;
  memset(&none, 0, sizeof(none));
  // Bg: channel 0, radii {3,5,10}; Cga/Cgb: channels 1-2, radii {5,10,20};
  // Tg: channel 3, radii {5,10,20}.
  if (colour) {
    hipLaunchKernelGGL((k_gradients<25, 6>), dim3(patches * 3, 4), dim3(256), 0, s, g, 0, 0,
                       P->d_tabs, I, P->blur_bg, grads, plane);
    hipLaunchKernelGGL((k_gradients<25, 3>), dim3(patches * 3, 8), dim3(256), 0, s, g, 1, 1,
                       P->d_tabs, I, P->blur_cg, grads, plane);
  }
  if (texture) {
    if (ntex == 64)
      hipLaunchKernelGGL(k_gradients64, dim3(div_up(w, GHX) * div_up(h, GHY) * 3, 4), dim3(256), 0, s, g, 1, P->d_tabs, I,
                         grads, plane);
    else
      hipLaunchKernelGGL((k_gradients<32, 0>), dim3(patches * 3, 4), dim3(256), 0, s, g, 3, 1,
                         P->d_tabs, I, none, grads, plane);
  }
  if (hist_done) DMSC_HIP(hipEventRecord(hist_done, s));
  CueOut out{{bg, cga, cgb, tg}};
  ParabolaJobs J;
  J.n = 0;
  for (int ri = 3; ri >= 0; ri--)  // longest blocks first
    for (int ch = 0; ch < 4; ch++) {
      const int scale = ri - (ch == 0 ? 0 : 1);  // Bg: radii 3, 5, 10; the others 5, 10, 20
      if (scale < 0 || scale > 2 || (ch < 3 ? !colour : !texture)) continue;
      J.ch[J.n] = ch;
      J.scale[J.n] = scale;
      J.radius[J.n] = kRadii[ri];
      std::copy(P->piece_first[ri], P->piece_first[ri] + 8, J.first[J.n]);
      std::copy(P->piece_count[ri], P->piece_count[ri] + 8, J.count[J.n]);
      J.n++;
    }
  static_assert(q_lw(3) % 4 == 0 && q_lw(5) % 4 == 0 && q_lw(10) % 4 == 0 && q_lw(20) % 4 == 0 && q_lw(20) <= 192,
                "float4-aligned tile rows of at most three columns per lane");
  hipLaunchKernelGGL(k_parabola, dim3(div_up(w, QTX), div_up(h, QTY), J.n * 8), dim3(QNT),
                     sizeof(float) * q_lw(J.radius[0]) * q_lh(J.radius[0]), s, w, h, J, grads, plane, P->d_piece_coef,
                     P->d_piece_at, out, pitch);
  DMSC_HIP(hipGetLastError());
  return DMSC_OK;
}

int launch_local_cues(Ctx* ctx, int w, int h, const float* L, const float* A, const float* B,
                      const int* tex, int ntex, float* bg, float* cga, float* cgb, float* tg, int pitch,
                      float* grads_out) {
  DMSC_TRY(local_cues_prepare(ctx, w, h, ntex));
  return launch_local_cues_part(ctx, ctx->stream, 3, w, h, L, A, B, tex, ntex, bg, cga, cgb, tg, pitch, grads_out);
}

}  // namespace dmsc
