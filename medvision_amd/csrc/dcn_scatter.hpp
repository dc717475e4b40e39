// Which corners of a sample are summed in LDS, and at what scale: shared by the kernels of the deformable backward pass.
#pragma once
#include "dcn_mfma.hpp"

namespace mv {

constexpr unsigned kOob = 0x80000000u;  // byte offset beyond every buffer: loads give 0, atomics are dropped
constexpr int kRsrcFlags = 0x00020000;

// ---- bricks and tiles of the LDS scatter (dcn_backward_scatter.hip) ---------------------------------
// A brick is 2^bd x 2^bh x 2^bw output positions; its tile the td x th x tw input voxels centred on the
// reach of the brick's undeformed taps.  A corner is "local" when its voxel lies in
// the tile of its position's brick: local corners are summed in LDS by the scatter kernel, all
// others are added to the gradient buffer by the tap kernel, 128 bytes per request.
struct ScatterShape {
  int bd, bh, bw, td, th, tw;
  int nbd, nbh, nbw;   // bricks along the axes
  int terms;      // corners that a voxel of a tile can take: positions of the brick times taps
  int narrow;     // 32-bit sums instead of 64-bit ones (dcn_scatter_plan)
  int turns;      // blocks of sixteen channels of a workgroup (wide images)
};
struct TileOrigin { int d, h, w; };
__device__ __forceinline__ TileOrigin tile_origin(const DcnDims &s, const ScatterShape &t, int bz, int by, int bx) {
  TileOrigin o;
  o.d = (bz << t.bd) * s.sd - s.pd - (t.td - (((1 << t.bd) - 1) * s.sd + (s.kd - 1) * s.dd + 1)) / 2;
  o.h = (by << t.bh) * s.sh - s.ph - (t.th - (((1 << t.bh) - 1) * s.sh + (s.kh - 1) * s.dh + 1)) / 2;
  o.w = (bx << t.bw) * s.sw - s.pw - (t.tw - (((1 << t.bw) - 1) * s.sw + (s.kw - 1) * s.dw + 1)) / 2;
  return o;
}
// bit c: corner c (z-major) of the sample whose first corner is voxel (id, ih, iw) lies in the tile;
// `first` its cell index there
__device__ __forceinline__ unsigned tile_bits(const ScatterShape &t, const TileOrigin &o, int id, int ih, int iw, int &first) {
  const int zd = id - o.d, zh = ih - o.h, zw = iw - o.w;
  const bool fd[2] = {zd >= 0 && zd < t.td, zd >= -1 && zd < t.td - 1};
  const bool fh[2] = {zh >= 0 && zh < t.th, zh >= -1 && zh < t.th - 1};
  const bool fw[2] = {zw >= 0 && zw < t.tw, zw >= -1 && zw < t.tw - 1};
  unsigned bits = 0;
#pragma unroll
  for (int c = 0; c < 8; c++) bits |= (fd[c >> 2] && fh[(c >> 1) & 1] && fw[c & 1]) ? 1u << c : 0u;
  first = (zd * t.th + zh) * t.tw + zw;
  return bits;
}

// The LDS sums are fixed point (LDS float atomics retire one lane at a time: 0.33 lanes a clock, 64-bit integer ones 6.4, or 10.7 where
// sixteen lanes add to neighbouring words).  Every term is w * mask * gcol with 0 <= w <= 1, so
//   |term| <= max|mask| * max|grad_output| * max_{c,k} sum_o |Wt[o,c,k]|  =: bound < 2^ex,
// and a voxel takes at most one corner of each (position, tap) of the brick: positions * taps terms.
// Terms are scaled by 2^(shift - ex), shift = min(50, 62 - ceil(log2(terms))), and rounded to
// integers (adding 1.5 * 2^52 in fp64 leaves round(x) in the low mantissa bits for |x| < 2^51):
// a term loses less than 2^-shift of the bound (2^-49 for up to 4096 terms), and the sum of a
// voxel stays below 2^63.  words[0..2] hold the bit patterns of the three maxima (of |.|, so they
// order like unsigned integers; a NaN or infinity anywhere gives a non-finite bound, and then no
// corner is treated as local).
constexpr double kRoundMagic = 6755399441055744.0;  // 1.5 * 2^52
struct ScatterScale { bool valid; double up, down; };
__device__ __forceinline__ ScatterScale scatter_scale(const unsigned *__restrict__ words, int terms, bool has_mask) {
  const float bound = 1.001f * __uint_as_float(words[0]) * __uint_as_float(words[1]) *
                      (has_mask ? __uint_as_float(words[2]) : 1.f);
  ScatterScale r;
  r.valid = bound < __builtin_inff() && bound == bound;
  int ex = 0;
  frexpf(fmaxf(bound, 1e-30f), &ex);  // bound < 2^ex
  const int shift = min(50, 62 - (32 - __clz(terms - 1)));
  r.up = ldexp(1.0, shift - ex);
  r.down = ldexp(1.0, ex - shift);
  return r;
}
// round(w * scaled) as a 64-bit integer; the low word of the magic number's bit pattern is zero
__device__ __forceinline__ unsigned long long fixed_term(float w, double scaled) {
  const double x = fma(static_cast<double>(w), scaled, kRoundMagic);
  const unsigned lo = static_cast<unsigned>(__double2loint(x)), hi = static_cast<unsigned>(__double2hiint(x)) - 0x43380000u;
  return (static_cast<unsigned long long>(hi) << 32) | lo;
}

}  // namespace mv
