// Pieces shared by the matrix-core (MFMA) kernels of the 3-D deformable convolution.
#pragma once
#include "dcn_common.hpp"

namespace mv {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Element-type traits of the matrix-core kernels.  Every operand piece is 16 bytes per lane (`kPiece` elements): a product of
// 16 x 16 (`run16`; 16-bit types v_mfma_f32_16x16x32, fp32 four v_mfma_f32_16x16x4_f32, element t of the piece in instruction
// t) covers a "slice" of 4 * kPiece channels or rows: lane l holds row / column l % 16 and the slice's piece l / 16;
// accumulator register r of lane l is row 4 * (l / 16) + r, column l % 16.
template <typename T> struct Mfma;
template <> struct Mfma<__half> {
  static constexpr int kPiece = 8;
  static __device__ __forceinline__ float4_t run16(u32x4 a, u32x4 b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ float lo(unsigned w) {
    return __half2float(__ushort_as_half(static_cast<unsigned short>(w & 0xffffu)));
  }
  static __device__ __forceinline__ float hi(unsigned w) {
    return __half2float(__ushort_as_half(static_cast<unsigned short>(w >> 16)));
  }
  static __device__ __forceinline__ float element(const u32x4 &r, int i) { return i % 2 ? hi(r[i / 2]) : lo(r[i / 2]); }
  // two values rounded to nearest even and packed, in one instruction (v_cvt_pk_f16_f32; not as inline assembly, around which the
  // compiler leaves no wait for a matrix instruction that is still writing a or b)
  static __device__ __forceinline__ unsigned pack2(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((float2_t{a, b}), half2_t));
  }
  // v[0..7] += w * piece
  static __device__ __forceinline__ void fma_piece(float (&v)[8], float w, u32x4 r) {
    v[0] += w * lo(r.x); v[1] += w * hi(r.x); v[2] += w * lo(r.y); v[3] += w * hi(r.y);
    v[4] += w * lo(r.z); v[5] += w * hi(r.z); v[6] += w * lo(r.w); v[7] += w * hi(r.w);
  }
  static __device__ __forceinline__ u32x4 pack(const float (&v)[8]) {
    return u32x4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])};
  }
};
template <> struct Mfma<__hip_bfloat16> {
  static constexpr int kPiece = 8;
  static __device__ __forceinline__ float4_t run16(u32x4 a, u32x4 b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ float lo(unsigned w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float hi(unsigned w) { return __uint_as_float(w & 0xffff0000u); }
  static __device__ __forceinline__ float element(const u32x4 &r, int i) { return i % 2 ? hi(r[i / 2]) : lo(r[i / 2]); }
  // two values rounded to nearest even and packed, in one instruction (v_cvt_pk_bf16_f32; not as inline assembly, around which the
  // compiler leaves no wait for a matrix instruction that is still writing a or b)
  static __device__ __forceinline__ unsigned pack2(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((float2_t{a, b}), bf16x2_t));
  }
  static __device__ __forceinline__ void fma_piece(float (&v)[8], float w, u32x4 r) {
    v[0] += w * lo(r.x); v[1] += w * hi(r.x); v[2] += w * lo(r.y); v[3] += w * hi(r.y);
    v[4] += w * lo(r.z); v[5] += w * hi(r.z); v[6] += w * lo(r.w); v[7] += w * hi(r.w);
  }
  static __device__ __forceinline__ u32x4 pack(const float (&v)[8]) {
    return u32x4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])};
  }
};
template <> struct Mfma<float> {
  static constexpr int kPiece = 4;
  static __device__ __forceinline__ float4_t run16(u32x4 a, u32x4 b, float4_t c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
  }
  static __device__ __forceinline__ float element(const u32x4 &r, int i) { return __uint_as_float(r[i]); }
  static __device__ __forceinline__ void fma_piece(float (&v)[4], float w, u32x4 r) {
    v[0] += w * __uint_as_float(r.x); v[1] += w * __uint_as_float(r.y);
    v[2] += w * __uint_as_float(r.z); v[3] += w * __uint_as_float(r.w);
  }
  static __device__ __forceinline__ u32x4 pack(const float (&v)[4]) {
    return u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
  }
};

// x [B, C, P] -> xt [B, P, Cp], channel c at (c / unit) * unit_p + c % unit, zeros elsewhere (Cp = C / unit * unit_p, a multiple of
// 16 bytes; unit = unit_p: no padding).  64 positions x 128 bytes of channels per workgroup through LDS; rows of any
// alignment, 16 bytes at a time all the same.  (U: the element as an integer of its size.)
//   ([8, 256, 100 x 152] fp16: 29 us with 64 positions, 41 us with 128 positions x 256 bytes; [128, 7 x 45 x 18], whose
//   rows are not aligned: 4 us, 12 us element by element.)
constexpr int kMovePos = 64;
template <typename U>
__device__ __forceinline__ void dcn_move_block(const U *__restrict__ x, U *__restrict__ xt, const int C, const int Cp, const int unit,
                                               const int unit_p, const long P, const long bx, const int b, const int bz) {
  constexpr int V = 16 / sizeof(U), CH = 128 / sizeof(U), PITCH = kMovePos + V, PG = kMovePos / V;
  typedef unsigned int piece_t __attribute__((ext_vector_type(4), aligned(2)));   // (element alignment: the hardware takes it)
  __shared__ __attribute__((aligned(16))) U stage[CH * PITCH];
  const long p0 = bx * kMovePos;
  const int c0 = bz * CH, cn = min(CH, Cp - c0), np = static_cast<int>(min(static_cast<long>(kMovePos), P - p0));
#pragma unroll
  for (int u = 0; u < CH * PG / 256; u++) {
    const int i = threadIdx.x + u * 256, c = i / PG, at = i % PG * V;
    if (c >= cn) continue;
    int from_c = c0 + c;
    bool real = true;
    if (unit != unit_p) {
      const int r = from_c % unit_p;
      real = r < unit;
      from_c = from_c / unit_p * unit + r;
    }
    const U *from = x + (static_cast<long>(b) * C + from_c) * P + p0 + at;
    if (!real) {
      *reinterpret_cast<u32x4 *>(stage + c * PITCH + at) = u32x4{0u, 0u, 0u, 0u};
    } else if (at + V <= np) {
      *reinterpret_cast<u32x4 *>(stage + c * PITCH + at) = *reinterpret_cast<const piece_t *>(from);
    } else {
      for (int e = 0; at + e < np; e++) stage[c * PITCH + at + e] = from[e];
    }
  }
  __syncthreads();
  const int groups = cn / V;
  for (int i = threadIdx.x; i < np * groups; i += 256) {
    const int p = i / groups, cg = i - p * groups;
    U out[V];
#pragma unroll
    for (int e = 0; e < V; e++) out[e] = stage[(cg * V + e) * PITCH + p];
    u32x4 packed;
    __builtin_memcpy(&packed, out, 16);
    *reinterpret_cast<u32x4 *>(xt + (static_cast<long>(b) * P + p0 + p) * Cp + c0 + cg * V) = packed;
  }
}

// The 8 trilinear corners of one (tap, position), z-major order: `at[c]` = voxel index * scale + add
// for a corner inside the volume, `outside` otherwise (also when the sample itself is void, i.e.
// not -1 < p < size on every axis, or the lane is not live); w[c] the trilinear weight; ld/lh/lw
// the fractions.  Branch-free: a corner is inside iff its index is, which per axis reads
//   low  index valid  <=>  0 <= p < size        high index valid  <=>  -1 < p < size - 1.
// Positions are exact in fp32 for 16-bit offsets (integer grid position + offset); fp32 tensors
// pass them in fp64 (floor and fraction taken there, the fraction rounded once to fp32).
struct CornerTaps {
  unsigned at[8];
  float w[8];
  float ld, lh, lw;
};
template <typename P>
__device__ __forceinline__ void corner_taps(const DcnDims &s, P pd, P ph, P pw, bool live,
                                            unsigned scale, unsigned add, unsigned outside,
                                            CornerTaps &t) {
  const P fd = floor(pd), fh = floor(ph), fw = floor(pw);
  t.ld = static_cast<float>(pd - fd); t.lh = static_cast<float>(ph - fh); t.lw = static_cast<float>(pw - fw);
  const bool vd[2] = {pd >= P(0) && pd < static_cast<P>(s.D), pd > P(-1) && pd < static_cast<P>(s.D - 1)};
  const bool vh[2] = {ph >= P(0) && ph < static_cast<P>(s.H), ph > P(-1) && ph < static_cast<P>(s.H - 1)};
  const bool vw[2] = {live && pw >= P(0) && pw < static_cast<P>(s.W), live && pw > P(-1) && pw < static_cast<P>(s.W - 1)};
  const int base = (static_cast<int>(fd) * s.H + static_cast<int>(fh)) * s.W + static_cast<int>(fw);
  const unsigned first = static_cast<unsigned>(base) * scale + add;  // wraps harmlessly when base < 0
  const unsigned sw = scale, sh = static_cast<unsigned>(s.W) * scale, sd = static_cast<unsigned>(s.H * s.W) * scale;
  const float wd[2] = {1.f - t.ld, t.ld}, wh[2] = {1.f - t.lh, t.lh}, ww[2] = {1.f - t.lw, t.lw};
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const int a = c >> 2, bb = (c >> 1) & 1, e = c & 1;
    t.at[c] = (vd[a] && vh[bb] && vw[e]) ? first + a * sd + bb * sh + e * sw : outside;
    t.w[c] = wd[a] * wh[bb] * ww[e];
  }
}

}  // namespace mv
