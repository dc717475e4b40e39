// Gradient of the input of the deformable convolution, local corners: summed in LDS, then added to the buffer.
//
//   gx[corner_n(k, q), c] += w_n * mask * gcol[c, k, q],   gcol[c, k, q] = sum_o Wt[o, c, k] * gy[o, q]
//
// A workgroup owns a brick of positions and 16 (fp32: 8) channels; its sixteen wavefronts split the brick's groups of 32
// positions and, where there are fewer than sixteen, the taps.  Two taps at a time: the lower half-wavefront works out tap k of
// the group's positions, the upper half tap k + 1; gcol comes from the 16 x 16 MFMA with the channels as rows (fp32: the
// eight channels of both taps), so a lane holds position l % 16 of a block and four channels.  Corners in the brick's tile are
// integer additions to LDS; afterwards the tile's non-zero sums are added to the gradient buffer, one global atomic per
// (voxel, channel) of the tile instead of one per (position, tap, corner, channel).
//
// NARROW (dense layers of 16-bit tensors, see dcn_scatter_plan): 32-bit sums.  (Two of them per 64-bit addition: 11.3 terms a clock and compute unit
// against 10.3, and more vector instructions to make the words: 556 us against 504 us.)  They leave 30 - ceil(log2(positions * taps)) bits for a term (17 for 3 x 3 x 3 taps), so the scale comes from the data: a
// first sweep over the brick's taps forms gcol alone (matrix cores, no geometry) and takes max |gcol| of the workgroup;
// every term is then below max |gcol| * max |mask| < 2^ex and is rounded to a multiple of 2^(ex - shift) (adding
// 1.5 * 2^23 in fp32 leaves round(x) in the low mantissa bits for |x| < 2^22).  The error of a voxel's sum stays below
// terms * 2^(ex - shift - 1), about 2^-15 of the values it sums for the 3 x 3 x 3 layer — a sixteenth of the last bit of the
// 16-bit result.  Otherwise a 64-bit word per channel, scale from the global maxima.
//
// What bounds it: the LDS additions (six to seven 64-bit lanes a clock and compute unit) and the 64-byte atomics of the tiles
// (21 G a second on the whole chip).  Busy, bf16 [2, 32 -> 64, 48^3] (32-bit sums, 496 us): vector issue 61 %, LDS 54 % (61 % of
// that bank conflicts: cells at random places); fp16 [8, 256 -> 256, 100 x 152] (64-bit, 1185 us): 47 %, 37 %, texture addressers 39 %.
#include "dcn_scatter.hpp"

namespace mv {

// Tiles of input voxels: their pitches are constants, so that the corners of a sample are immediate offsets (with pitches at run
// time: 603 us against 504 us for bf16 [2, 32 -> 64, 48^3]).
template <int D, int H, int W> struct Tile { static constexpr int TD = D, TH = H, TW = W, VOX = D * H * W, NC = D > 1 ? 8 : 4; };
constexpr int kScatterMinShift = 14;  // fewer bits per term: 64-bit words
__host__ __device__ constexpr int scatter32_shift(int terms) {
  int bits = 0;
  while ((1L << bits) < terms) bits++;
  return bits < 8 ? 22 : 30 - bits;   // (a term stays below 2^22)
}
// sums between voxels: the channels of a workgroup, and one to spread the banks
template <bool NARROW> constexpr int kScatterStride = NARROW ? 17 : 9;

// KEEP: slices of grad_output (of 4 * kPiece output channels) that a wavefront keeps in registers over the taps: 4, or 8 with half
// the wavefronts for wide layers, whose further slices cost 64 cache look-ups each for every tap.
template <typename T, bool NARROW, typename S, int KEEP>
__global__ __launch_bounds__(KEEP == 4 ? 1024 : 512) void dcn_backward_scatter_kernel(
    const T *__restrict__ off, const T *__restrict__ mask, const T *__restrict__ gyt,
    const T *__restrict__ wa, float *__restrict__ gxt, const DcnDims s, const ScatterShape shape,
    const unsigned *__restrict__ bounds) {
  using M = Mfma<T>;
  using P = typename std::conditional<(sizeof(T) == 2), float, double>::type;
  constexpr int PC = M::kPiece, SL = 4 * PC, CH = NARROW ? 16 : 8, NC = S::NC, WAVES = KEEP == 4 ? 16 : 8;
  using Sum = typename std::conditional<NARROW, int, unsigned long long>::type;
  constexpr int STRIDE = kScatterStride<NARROW>;
  __shared__ Sum tile[S::VOX * STRIDE];
  __shared__ float recs[WAVES][5][64];   // cell and corner bits, mask (times the scale), ld, lh, lw
  __shared__ unsigned wgmax;
  const ScatterScale scale = scatter_scale(bounds, shape.terms, mask != nullptr);
  if (!scale.valid) return;  // (a NaN or infinity somewhere: every corner went through the tap kernel)
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int n = lane % 32, half = lane / 32, p16 = lane % 16, j = lane / 16;
  const unsigned brick = xcd_contiguous(blockIdx.x, gridDim.x);
  const int bx = brick % shape.nbw, by = (brick / shape.nbw) % shape.nbh, bz = brick / (shape.nbw * shape.nbh);
  const int c0 = blockIdx.y * CH, b = blockIdx.z;
  const int dgi = c0 / s.cpd, g = c0 / s.cpg;
  const long bg = static_cast<long>(b) * s.dg + dgi;
  const int steps = s.opg / SL, cblocks = s.cpg / 16;
  const int groups = (1 << (shape.bd + shape.bh + shape.bw)) / 32;   // of 32 positions
  const int pwaves = min(groups, 8);                                 // wavefronts over the groups; the others over the taps
  const int share = wave / pwaves, shares = WAVES / pwaves;
  const int per = (s.K + shares - 1) / shares, k0 = min(share * per, s.K), k1 = min(s.K, k0 + per);
  const TileOrigin origin = tile_origin(s, shape, bz, by, bx);

  for (int i = threadIdx.x; i < S::VOX * STRIDE; i += WAVES * 64) tile[i] = 0;
  if (threadIdx.x == 0) wgmax = 0u;
  __syncthreads();

  // position of brick index i, columns fastest
  auto position = [&](int i, bool &live) {
    const int od = (bz << shape.bd) + (i >> (shape.bh + shape.bw)), oh = (by << shape.bh) + ((i >> shape.bw) & ((1 << shape.bh) - 1)),
              ow = (bx << shape.bw) + (i & ((1 << shape.bw) - 1));
    live = od < s.Do && oh < s.Ho && ow < s.Wo;
    return (static_cast<long>(min(od, s.Do - 1)) * s.Ho + min(oh, s.Ho - 1)) * s.Wo + min(ow, s.Wo - 1);
  };
  // grad_output of the lane's column in the two 16-position blocks of a group (MFMA B operand)
  const T *grow[2];
  bool glive[2];
  u32x4 keep[2][KEEP];
  auto load_keep = [&](int pg) {
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      bool on;
      const long qb = position(pg * 32 + blk * 16 + p16, on);
      const T *from = gyt + (static_cast<long>(b) * s.Q + qb) * s.Cout + g * s.opg + j * PC;
#pragma unroll
      for (int st = 0; st < KEEP; st++)
        keep[blk][st] = on && st < steps ? *reinterpret_cast<const u32x4 *>(from + st * SL) : u32x4{0u, 0u, 0u, 0u};
      grow[blk] = from;
      glive[blk] = on;
    }
  };
  // Rows of the weight of tap k: NARROW its 16 channels; else the 8 channels of tap k in rows 0 - 7 and of tap k + 1 in rows 8 - 15
  // (zeros when that is not the wavefront's)
  const long tap_stride = static_cast<long>(cblocks) * steps * 64 * PC;
  const T *wrow = wa + (static_cast<long>(g) * s.K * cblocks + (c0 - g * s.cpg) / 16) * steps * (64 * PC) +
                  (NARROW ? lane : j * 16 + p16 % 8 + (c0 - g * s.cpg) % 16) * PC + (NARROW ? 0 : p16 / 8 * tap_stride);
  auto load_weight = [&](int k, int st) {
    const bool on = NARROW || k + p16 / 8 < k1;
    return on && st < steps ? *reinterpret_cast<const u32x4 *>(wrow + k * tap_stride + static_cast<long>(st) * (64 * PC)) : u32x4{0u, 0u, 0u, 0u};
  };
  // gcol of both blocks of the group (the further slices of wide layers are read again for every tap)
  auto product = [&](const u32x4 (&w)[KEEP], int k, float4_t (&acc)[2]) {
    acc[0] = acc[1] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < KEEP; st++)
      if (st < steps) {
        acc[0] = M::run16(w[st], keep[0][st], acc[0]);
        acc[1] = M::run16(w[st], keep[1][st], acc[1]);
      }
    for (int st = KEEP; KEEP > 4 && st < steps; st++) {
      const u32x4 wf = load_weight(k, st);
#pragma unroll
      for (int blk = 0; blk < 2; blk++) {
        const u32x4 bf = glive[blk] ? *reinterpret_cast<const u32x4 *>(grow[blk] + st * SL) : u32x4{0u, 0u, 0u, 0u};
        acc[blk] = M::run16(wf, bf, acc[blk]);
      }
    }
  };
  auto load_weights = [&](int k, u32x4 (&w)[KEEP]) {
#pragma unroll
    for (int st = 0; st < KEEP; st++) w[st] = load_weight(k, st);
  };

  float up = 1.f, down = 1.f;
  if constexpr (NARROW) {
    // ---- first sweep: max |gcol| over the brick's positions, the taps and the channels --------------------------
    float top = 0.f;
    for (int pg = wave % pwaves; pg < groups; pg += pwaves) {
      load_keep(pg);
      for (int k = k0; k < k1; k++) {
        u32x4 w[KEEP];
        load_weights(k, w);
        float4_t acc[2];
        product(w, k, acc);
#pragma unroll
        for (int i = 0; i < 4; i++) top = fmaxf(top, fmaxf(fabsf(acc[0][i]), fabsf(acc[1][i])));
      }
    }
    for (int sh = 32; sh > 0; sh >>= 1) top = fmaxf(top, __shfl_xor(top, sh));
    if (lane == 0 && top > 0.f) atomicMax(&wgmax, __float_as_uint(top));
    __syncthreads();
    const float bound = fmaxf(1.001f * __uint_as_float(wgmax), 1e-30f) * (mask ? __uint_as_float(bounds[2]) : 1.f);
    if (!(bound > 0.f)) return;  // nothing but zeros to add (the whole workgroup leaves together)
    const int shift = scatter32_shift(shape.terms);
    int ex = 0;
    frexpf(bound, &ex);  // bound < 2^ex
    up = ldexpf(1.f, shift - ex);
    down = ldexpf(1.f, ex - shift);
  }
  constexpr float kMagic = 12582912.f;  // 1.5 * 2^23
  float(*rec)[64] = recs[wave];

  for (int pg = wave % pwaves; pg < groups; pg += pwaves) {
    bool live;
    const long q = position(pg * 32 + n, live);
    const int ow = q % s.Wo, oh = (q / s.Wo) % s.Ho, od = q / (static_cast<long>(s.Wo) * s.Ho);
    const int bd = od * s.sd - s.pd, bh = oh * s.sh - s.ph, bw = ow * s.sw - s.pw;
    load_keep(pg);
    int kt = k0 + half;  // the lane's own tap
    const T *o = off + (bg * s.nd * s.K + static_cast<long>(s.nd) * kt) * s.Q + q;
    const T *mk = mask ? mask + (bg * s.K + kt) * s.Q + q : nullptr;
    int ki = kt / (s.kh * s.kw), kj = (kt / s.kw) % s.kh, kk = kt % s.kw;
    P fd = P(0), fh = P(0), fw = P(0);
    float fm = 1.f;
    if (kt < k1) {
      dcn_offsets(s, o, fd, fh, fw);
      if (mk) fm = load(mk);
    }
    for (int k = k0; k < k1; k += 2) {
      // weight pieces of the two taps (the taps' geometry below hides their latency)
      u32x4 wpair[NARROW ? 2 : 1][KEEP];
#pragma unroll
      for (int u = 0; u < (NARROW ? 2 : 1); u++) load_weights(min(k + u, s.K - 1), wpair[u]);
      {
        P pd = fd + static_cast<P>(bd + ki * s.dd);
        const P ph = fh + static_cast<P>(bh + kj * s.dh), pw = fw + static_cast<P>(bw + kk * s.dw);
        if (NC == 4) pd = P(0);   // images: the only slice
        const float m = fm;
        const bool tap_on = kt < k1;
        kt += 2;
        o += 2 * s.nd * s.Q;
        if (mk) mk += 2 * s.Q;
#pragma unroll
        for (int u = 0; u < 2; u++)
          if (++kk == s.kw) { kk = 0; if (++kj == s.kh) { kj = 0; ++ki; } }
        if (kt < k1) {  // the next pair's offsets are in flight during this pair's adds
          dcn_offsets(s, o, fd, fh, fw);
          if (mk) fm = load(mk);
        }
        CornerTaps t;
        corner_taps<P>(s, pd, ph, pw, live && tap_on, 1u, 0u, ~0u, t);
        int first;
        unsigned bits = tile_bits(shape, origin, static_cast<int>(floor(pd)), static_cast<int>(floor(ph)), static_cast<int>(floor(pw)), first);
        unsigned inside = 0;
#pragma unroll
        for (int c = 0; c < NC; c++) inside |= t.at[c] != ~0u ? 1u << c : 0u;
        bits &= inside;
        rec[0][lane] = __uint_as_float(static_cast<unsigned>(first) * 256u + bits);
        rec[1][lane] = NARROW ? m * up : m;
        rec[2][lane] = t.ld; rec[3][lane] = t.lh; rec[4][lane] = t.lw;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

#pragma unroll
      for (int u = 0; u < (NARROW ? 2 : 1); u++) {
        if (k + u >= k1) break;
        float4_t acc[2];
        product(wpair[u], k + u, acc);
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
          const int at = (NARROW ? u : j / 2) * 32 + blk * 16 + p16;
          const int word = __float_as_int(rec[0][at]);
          const float m = rec[1][at], ld = rec[2][at], lh = rec[3][at], lw = rec[4][at];
          const unsigned bits = static_cast<unsigned>(word) & 255u;
          const float wd[2] = {1.f - ld, ld}, wh[2] = {1.f - lh, lh}, ww[2] = {1.f - lw, lw};
          // (NARROW: channel 4 j + r of a voxel is its sum j + 4 r, so that the lanes of neighbouring voxels use all banks)
          // the lane's sums of the first corner (the record's cell may lie before the tile: its corners do not)
          char *const cell0 = reinterpret_cast<char *>(tile) + ((word >> 8) * STRIDE + (NARROW ? j : 4 * (j % 2))) * static_cast<int>(sizeof(Sum));
          float gv[4];
          double gd[4];
#pragma unroll
          for (int r = 0; r < 4; r++) {
            gv[r] = acc[blk][r] * m;
            if constexpr (!NARROW) gd[r] = static_cast<double>(gv[r]) * scale.up;
          }
#pragma unroll
          for (int c = 0; c < NC; c++) {
            const int ca = c >> 2, cb = (c >> 1) & 1, ce = c & 1;
            if ((bits >> c) & 1u) {
              const float wc = wd[ca] * wh[cb] * ww[ce];
              Sum *dst = reinterpret_cast<Sum *>(cell0 + (ca * (S::TH * S::TW) + cb * S::TW + ce) * (STRIDE * static_cast<int>(sizeof(Sum))));
#pragma unroll
              for (int r = 0; r < 4; r++) {
                if constexpr (NARROW)
                  __hip_atomic_fetch_add(dst + 4 * r, __float_as_int(fmaf(wc, gv[r], kMagic)) - 0x4B400000, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP);
                else
                  __hip_atomic_fetch_add(dst + r, fixed_term(wc, gd[r]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
              }
            }
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
  __syncthreads();
  // ---- the tile's voxels inside the volume go to the gradient buffer, all channels of a voxel at once -----------
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(
      gxt + static_cast<long>(b) * s.P * s.Cin, 0, static_cast<int>(s.P * s.Cin * 4), kRsrcFlags);
  const unsigned cin4 = static_cast<unsigned>(s.Cin) * 4u;
  const int slot = threadIdx.x % CH, ch = NARROW ? slot % 4 * 4 + slot / 4 : slot;
  for (int cell = threadIdx.x / CH; cell < S::VOX; cell += WAVES * 64 / CH) {
    const int zw = cell % S::TW + origin.w, zh = cell / S::TW % S::TH + origin.h, zd = cell / (S::TW * S::TH) + origin.d;
    const Sum sum = tile[cell * STRIDE + slot];
    const float v = NARROW ? static_cast<float>(sum) * down
                           : static_cast<float>(static_cast<double>(static_cast<long long>(sum)) * scale.down);
    if (zd >= 0 && zd < s.D && zh >= 0 && zh < s.H && zw >= 0 && zw < s.W && v != 0.f)
      __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(
          v, gr, static_cast<unsigned>((zd * s.H + zh) * s.W + zw) * cin4 + static_cast<unsigned>(c0 + ch) * 4u, 0, 0);
  }
}

using TileVolume = Tile<10, 14, 14>;    // 4 x 8 x 8 positions: two voxels to spare at stride 1
using TileStrided = Tile<12, 12, 13>;   // 4 x 4 x 4 positions: stride 2, dilation
using TileImage = Tile<1, 44, 44>;      // 32 x 32 positions (16 x 16 at stride 2)
using TileSmall = Tile<1, 28, 28>;      // 16 x 16 or 8 x 8 positions, two workgroups on a compute unit

// The brick and its tile: the first of the list whose tile holds the reach of the brick's undeformed taps with two voxels to spare
// on either side, or one, if none has two.  Images with fewer workgroups than compute units take a smaller brick (77 us ->
// 35 us for [1, 256 -> 128, 27 x 58]); volumes do not (the halo of 4 x 4 x 4 positions is most of their tile: 117 us
// against 78 us for [2, 16 -> 128, 7 x 19 x 32]).  False: no brick fits.
//
// Width of the sums: 32 bits round every term to 14 - 22 bits of the workgroup's largest, which is worth their speed in dense
// layers alone (16-bit tensors, the first brick fits: unit strides, taps close together; up to 128 output channels).  bf16 training
// step of [2, 32 -> 64, 48^3]: 1178 us, 1393 us with 64-bit sums.  Strided and wide layers have 64-bit sums, as good as fp32 ones:
// where the output's gradient is 2^-14 of what it is elsewhere in the brick, 32 bits left them 2 - 20 % off.  Training steps, 32
// against 64 bits: [8, 256 -> 256, 100 x 152] fp16 2315 / 2337 us; stride 2, [8, 128 -> 128, 100 x 152] 332 / 370 us and
// [2, 32 -> 64, 48^3] 297 / 345 us.
bool dcn_scatter_plan(const DcnDims &s, int dtype, ScatterShape &shape) {
  static const int volumes[2][6] = {{2, 3, 3, 10, 14, 14}, {2, 2, 2, 12, 12, 13}};
  static const int images[4][6] = {{0, 5, 5, 1, 44, 44}, {0, 4, 4, 1, 28, 28}, {0, 4, 4, 1, 44, 44}, {0, 3, 3, 1, 28, 28}};
  const bool image = s.nd == 2;
  const int st[3] = {s.sd, s.sh, s.sw}, kn[3] = {s.kd, s.kh, s.kw}, dl[3] = {s.dd, s.dh, s.dw}, on[3] = {s.Do, s.Ho, s.Wo};
  int best = -1;
  bool dense = false;
  for (int i = 0; i < (image ? 4 : 2); i++) {
    const int *e = image ? images[i] : volumes[i];
    long spare = 1 << 20, bricks = s.B;
    for (int a = 0; a < 3; a++) {
      const long extent = static_cast<long>((1 << e[a]) - 1) * st[a] + static_cast<long>(kn[a] - 1) * dl[a] + 1;
      if (!image || a > 0) spare = std::min(spare, e[3 + a] - extent);
      bricks *= (on[a] + (1 << e[a]) - 1) >> e[a];
    }
    if (spare < 2 || (1L << (e[0] + e[1] + e[2])) * s.K >= (1L << 20)) continue;
    dense = dense || i == 0;
    const int rank = (spare >= 4 ? 2 : 0) + (image && bricks * (s.Cin / (dtype == MV_F32 ? 8 : 16)) >= 256 ? 1 : 0);
    if (rank <= best) continue;
    best = rank;
    shape = ScatterShape{e[0], e[1], e[2], e[3], e[4], e[5], 0, 0, (1 << (e[0] + e[1] + e[2])) * s.K, 0};
  }
  if (best < 0 || s.Cin / 8 > 65535) return false;
  shape.narrow = dense && dtype != MV_F32 && s.opg <= 128 && scatter32_shift(shape.terms) >= kScatterMinShift;
  shape.nbh = (s.Ho + (1 << shape.bh) - 1) >> shape.bh;
  shape.nbw = (s.Wo + (1 << shape.bw) - 1) >> shape.bw;
  return static_cast<long>(shape.nbh) * shape.nbw * ((s.Do + (1 << shape.bd) - 1) >> shape.bd) < (1L << 31);
}

template <typename T, typename S>
static int scatter_launch(const void *off, const void *mask, const void *gyt, const void *wf, float *gxt, const DcnDims &s,
                          const ScatterShape &shape, const unsigned *bounds, hipStream_t stream) {
  const int nbd = (s.Do + (1 << shape.bd) - 1) >> shape.bd;
  const bool wide = s.opg > 4 * 64 / static_cast<int>(sizeof(T));
  const dim3 grid(static_cast<unsigned>(nbd) * shape.nbh * shape.nbw, s.Cin / (shape.narrow ? 16 : 8), s.B);
#define MV_SCATTER(NARROWV, KEEPV)                                                                                    \
  hipLaunchKernelGGL((dcn_backward_scatter_kernel<T, NARROWV, S, KEEPV>), grid, dim3(KEEPV == 4 ? 1024 : 512), 0, stream,     \
                     static_cast<const T *>(off), static_cast<const T *>(mask), static_cast<const T *>(gyt),          \
                     static_cast<const T *>(wf), gxt, s, shape, bounds)
  if (shape.narrow) {
    if constexpr (sizeof(T) == 2) MV_SCATTER(true, 4);   // (never wide)
  } else {
    if (wide) MV_SCATTER(false, 8); else MV_SCATTER(false, 4);
  }
#undef MV_SCATTER
  return check_launch("dcn_backward_scatter_kernel");
}

int dcn_scatter(const void *off, const void *mask, const void *gyt, const void *wf, float *gxt, const DcnDims &s,
                const ScatterShape &shape, const unsigned *bounds, int dtype, hipStream_t stream) {
#define MV_SCATTER_TILE(T, S) scatter_launch<T, S>(off, mask, gyt, wf, gxt, s, shape, bounds, stream)
#define MV_SCATTER_AS(T)                                                                                              \
  (shape.th == TileVolume::TH ? MV_SCATTER_TILE(T, TileVolume)                                                          \
   : shape.th == TileStrided::TH ? MV_SCATTER_TILE(T, TileStrided)                                                      \
   : shape.th == TileImage::TH ? MV_SCATTER_TILE(T, TileImage) : MV_SCATTER_TILE(T, TileSmall))
  if (dtype == MV_F16) return MV_SCATTER_AS(__half);
  if (dtype == MV_F32) return MV_SCATTER_AS(float);
  return MV_SCATTER_AS(__hip_bfloat16);
#undef MV_SCATTER_AS
#undef MV_SCATTER_TILE
}

}  // namespace mv
