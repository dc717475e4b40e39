// Gradient of the input of the deformable convolution, local corners: summed in LDS, then added to the buffer.
//
//   gx[corner_n(k, q), c] += w_n * mask * gcol[c, k, q],   gcol[c, k, q] = sum_o Wt[o, c, k] * gy[o, q]
//
// A workgroup owns a brick of positions and 16 channels (8 where 64-bit sums of 16 are beyond the LDS); its wavefronts split the
// brick's groups of 32 positions and, where there are fewer groups than wavefronts, the taps.  Two taps at a time: every lane works
// out one sample, a cell of the tile and the weights of its corners.  gcol comes from the 16 x 16 MFMA with the positions as rows, so
// that a row of sixteen lanes holds sixteen channels of one position (eight of two taps): the sample's words reach them as DPP row
// broadcasts, which the multiplications take as an operand, and an LDS addition meets four (eight) cells of 64 contiguous bytes.
// Per term: multiply, convert, add.  Corners outside the tile or the volume have weight 0 in a cell that exists: no branches.
//   (Channels as rows, a lane holding one position and four channels, needed the samples' words from LDS, a branch per corner
//   and additions to 16 places: bf16 [2, 32 -> 64, 48^3] 496 us, then 338 us (348 us with today's larger tile); fp16 [8, 256 -> 256, 100 x 152] 1185 us, now 510 us.)
// Afterwards the tile's non-zero sums are added to the gradient buffer, one global atomic per (voxel, channel) of the tile
// instead of one per (position, tap, corner, channel).
//
// NARROW (dense layers of 16-bit tensors, see dcn_scatter_plan): 32-bit sums.  They leave 31 - log2(positions * taps) bits for
// a term (18 for 3 x 3 x 3 taps), so the scale comes from the data: a first sweep over the brick's taps forms gcol alone (matrix
// cores, no geometry; 17 us) and takes max |gcol| of the workgroup; every term is then below max |gcol| * max |mask| <
// 2^ex and is rounded to a multiple of 2^(ex - shift).  The error of a voxel's sum stays below terms * 2^(ex - shift - 1), whatever its own
// size: 1.3 % of the workgroup's largest term for 3 x 3 x 3 taps if all roundings agreed.  With gradients of even size it is far less
// (fp16 [2, 32 -> 64, 48^3], sigma = 2: 2.18e-4 rms of the gradient, of which rounding the result is 2.07e-4).  Otherwise a 64-bit word
// per channel, scale from the global maxima.
//
// What bounds it: the LDS additions (64 lanes of 32 bits in 4 clocks, of 64 bits in 6, whatever the cells) behind phases that leave
// the LDS idle, since a tile fills the compute unit: the first group's inputs, the sweep, the tile's atomics (40 us).  Busy: bf16
// [2, 32 -> 64, 48^3] vector issue 51 %, LDS 40 %; fp16 [8, 256 -> 256, 100 x 152] 46 %, 28 %, texture addressers 37 %.
#include "dcn_scatter.hpp"

namespace mv {

// Tiles of input voxels: their pitches are constants, so that the corners of a sample are immediate offsets (with pitches at run
// time: 603 us against 504 us for bf16 [2, 32 -> 64, 48^3]).
// Channels of a workgroup: 16, and 8 where 64-bit sums of 16 are beyond the LDS.
template <int D, int H, int W> struct Tile {
  static constexpr int TD = D, TH = H, TW = W, VOX = D * H * W, NC = D > 1 ? 8 : 4;
  static constexpr bool WIDE = D == 1 && W > H;
  template <bool NARROW> static constexpr int channels = VOX * 16 * (NARROW ? 4 : 8) <= 160 * 1024 ? 16 : 8;
};
constexpr int kScatter32Terms = 1 << 16;  // more (fewer than 14 bits each): 64-bit words
// the largest shift <= 22 with terms * 2^shift < 2^31
__host__ __device__ constexpr int scatter32_shift(int terms) {
  int shift = 22;
  while (shift > 0 && (static_cast<long>(terms) << shift) > 0x7fffffffL) shift--;
  return shift;
}

template <int... I, typename F> __device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}
// The value that lane FROM of the lane's row of sixteen holds.  CH == 8: lane FROM for the row's lower half, FROM + 8 for the upper.
template <int CH, int FROM> __device__ __forceinline__ int row_word(int v) {
  constexpr int kRowBroadcast = 0x150;
  if constexpr (CH == 16) return __builtin_amdgcn_mov_dpp(v, kRowBroadcast + FROM, 0xf, 0xf, true);
  const int low = __builtin_amdgcn_mov_dpp(v, kRowBroadcast + FROM, 0xf, 0xf, true);
  return __builtin_amdgcn_update_dpp(low, v, kRowBroadcast + (FROM + 8) % 16, 0xf, 0xc, false);
}
template <int CH, int FROM> __device__ __forceinline__ float row_value(float v) {
  return __int_as_float(row_word<CH, FROM>(__float_as_int(v)));
}
// round(x) for |x| < 2^31 in one instruction (in the register of x: around inline assembly the compiler leaves no wait for a matrix instruction
// that still reads a register which the result would get)
__device__ __forceinline__ int round_word(float x) {
  int r = __float_as_int(x);
  asm("v_cvt_rpi_i32_f32 %0, %0" : "+v"(r));
  return r;
}

// A value that is the same in all lanes, in a scalar register
__device__ __forceinline__ float uniform(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }

// One axis of a tile that starts at voxel `origin` and whose cells low .. high - 1 lie in the volume.
struct TileAxis {
  float origin, low, high, low1, high1;
  __device__ __forceinline__ TileAxis(int first, int cells, int voxels)
      : origin(uniform(static_cast<float>(first))), low(uniform(static_cast<float>(max(0, -first)))),
        high(uniform(static_cast<float>(min(cells, voxels - first)))), low1(uniform(low - 1.f)), high1(uniform(high - 1.f)) {}
  // The weights of two neighbouring cells of the tile, of which it returns the first.  A corner outside has weight 0: a sample on the
  // tile's edge has its cells moved by one, any other one outside both weights 0 (NaN positions too), so that every cell exists.
  template <int CELLS, typename P> __device__ __forceinline__ float sample(P p, float &w0, float &w1) const {
    const P f = floor(p);
    const float frac = static_cast<float>(p - f), z = static_cast<float>(f - static_cast<P>(origin));
    const float u0 = z >= low && z < high ? 1.f - frac : 0.f, u1 = z >= low1 && z < high1 ? frac : 0.f;
    const float first = fminf(fmaxf(z, 0.f), static_cast<float>(CELLS - 2));
    const bool moved = z != first;
    w0 = moved ? u1 : u0;
    w1 = moved ? u0 : u1;
    return first;
  }
};

// KEEP: slices of grad_output (of 4 * kPiece output channels) that a wavefront keeps in registers over the taps: 2 or 4, or 8 with
// half the wavefronts for wide layers, whose further slices cost 64 cache look-ups each for every tap.
template <typename T, bool NARROW, typename S, int KEEP>
__global__ __launch_bounds__(KEEP <= 4 ? 1024 : 512) void dcn_backward_scatter_kernel(
    const T *__restrict__ off, const T *__restrict__ mask, const T *__restrict__ gyt,
    const T *__restrict__ wa, float *__restrict__ gxt, const DcnDims s, const ScatterShape shape,
    const unsigned *__restrict__ bounds) {
  using M = Mfma<T>;
  using P = typename std::conditional<(sizeof(T) == 2), float, double>::type;
  constexpr int PC = M::kPiece, SL = 4 * PC, ES = sizeof(T), CH = S::template channels<NARROW>, NC = S::NC, ND = NC == 8 ? 3 : 2;
  constexpr int WAVES = KEEP <= 4 ? 16 : 8;
  constexpr int TAPS = CH == 16 ? 2 : 1;   // products per pair of taps
  // positions of a group: 64 where eight slices of the weight come from the caches for every tap (with sixteen wavefronts of 32
  // positions 620 us instead of 500 for fp16 [8, 256 -> 256, 100 x 152])
  constexpr int SETS = KEEP == 8 && S::WIDE ? 2 : 1, BLOCKS = 2 * SETS, GROUP = 16 * BLOCKS;
  using Sum = typename std::conditional<NARROW, int, unsigned long long>::type;
  constexpr int CELL = CH * static_cast<int>(sizeof(Sum));
  __shared__ __attribute__((aligned(16))) Sum tile[S::VOX * CH];
  __shared__ unsigned wgmax;
  const ScatterScale scale = scatter_scale(bounds, shape.terms, mask != nullptr);
  if (!scale.valid) return;  // (a NaN or infinity somewhere: every corner went through the tap kernel)
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int p16 = lane % 16, j = lane / 16;
  // the lane's own sample: position n of a group, the first or second tap of a pair
  const int n = p16 / 4 % 2 * 16 + 4 * j + p16 % 4, half = p16 / 8;
  // (the channel blocks of a brick next to each other on one XCD: they read the same grad_output and offsets)
  const int turns = CH == 16 && KEEP == 8 ? shape.turns : 1;   // blocks of CH channels, one after the other
  const unsigned shares_of_brick = s.Cin / (CH * turns), workgroups = shape.nbd * shape.nbh * shape.nbw * s.B * shares_of_brick;
  if (linear_block() >= workgroups) return;
  const unsigned id = xcd_contiguous(linear_block(), workgroups), brick = id / shares_of_brick;
  int c0 = static_cast<int>(id % shares_of_brick) * (CH * turns);
  const int bx = brick % shape.nbw, by = brick / shape.nbw % shape.nbh, bz = brick / (shape.nbw * shape.nbh) % shape.nbd,
            b = brick / (shape.nbw * shape.nbh * shape.nbd);
  const int dgi = c0 / s.cpd, g = c0 / s.cpg;
  const long bg = static_cast<long>(b) * s.dg + dgi;
  const int steps = s.opg / SL, cblocks = s.cpg / 16;
  const int groups = (1 << (shape.bd + shape.bh + shape.bw)) / GROUP;
  const int pwaves = min(groups, WAVES);   // wavefronts over the groups; the others over the taps
  const int share = wave / pwaves, shares = WAVES / pwaves;
  const int per = (s.K + shares - 1) / shares, k0 = min(share * per, s.K), k1 = min(s.K, k0 + per);
  const TileOrigin origin = tile_origin(s, shape, bz, by, bx);

  // position of brick index i, columns fastest
  struct Position { int d, h, w, q; bool live; };
  auto position = [&](int i) {
    Position p;
    const int od = (bz << shape.bd) + (i >> (shape.bh + shape.bw)), oh = (by << shape.bh) + ((i >> shape.bw) & ((1 << shape.bh) - 1)),
              ow = (bx << shape.bw) + (i & ((1 << shape.bw) - 1));
    p.live = od < s.Do && oh < s.Ho && ow < s.Wo;
    p.d = min(od, s.Do - 1); p.h = min(oh, s.Ho - 1); p.w = min(ow, s.Wo - 1);
    p.q = (p.d * s.Ho + p.h) * s.Wo + p.w;
    return p;
  };
  // grad_output of the lane's row in the blocks of 16 positions of group `loaded` (MFMA A operand)
  u32x4 keep[BLOCKS][KEEP];
  auto gradient = [&](const Position &p, int st) {
    return p.live && st < steps ? *reinterpret_cast<const u32x4 *>(gyt + (static_cast<long>(b) * s.Q + p.q) * s.Cout + g * s.opg + j * PC + st * SL)
                                : u32x4{0u, 0u, 0u, 0u};
  };
  int loaded = -1;
  bool some = false;   // (any position of the group exists)
  auto load_keep = [&](int pg) {
    if (pg == loaded) return;
    loaded = pg;
    bool mine = false;
#pragma unroll
    for (int blk = 0; blk < BLOCKS; blk++) {
      const Position p = position(pg * GROUP + blk * 16 + p16);
#pragma unroll
      for (int st = 0; st < KEEP; st++) keep[blk][st] = gradient(p, st);
      mine = mine || p.live;
    }
    some = __any(mine) != 0;
  };
  // Columns of the weight of tap k: the 16 channels; of eight channels tap k in columns 0 - 7 and tap k + 1 in columns 8 - 15.  No
  // branches: slices that do not exist meet zeros of grad_output, the tap behind the wavefront's last one samples of weight 0 (and the
  // buffer ends behind the last of all).
  const int tap_bytes = s.cpg * s.opg * ES;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(wa + static_cast<long>(g) * s.K * s.cpg * s.opg), 0, s.K * tap_bytes, kRsrcFlags);
  int cl = c0 - g * s.cpg;
  const unsigned wlane = static_cast<unsigned>((CH == 16 ? lane : j * 16 + p16 % 8 + cl % 16) * 16 + (CH == 16 ? 0 : half * tap_bytes));
  auto load_weight = [&](int k, int st) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, wlane, k * tap_bytes + (cl / 16 * steps + min(st, steps - 1)) * 1024, 0));
  };
  constexpr int AHEAD = SETS == 2 ? 4 : KEEP;   // slices requested behind the product before (the registers hold no more)
  auto load_weights = [&](int k, u32x4 (&w)[AHEAD]) {
#pragma unroll
    for (int st = 0; st < AHEAD; st++) w[st] = load_weight(k, st);
  };
  // gcol of the blocks of the group (the further slices of wide layers are read again for every tap)
  auto product = [&](const u32x4 (&w)[AHEAD], int k, int pg, float4_t (&acc)[BLOCKS]) {
#pragma unroll
    for (int blk = 0; blk < BLOCKS; blk++) acc[blk] = float4_t{0.f, 0.f, 0.f, 0.f};
    u32x4 now[AHEAD], then[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) now[i] = w[i];
#pragma unroll
    for (int from = 0; from < KEEP; from += AHEAD) {
#pragma unroll
      for (int i = 0; i < AHEAD; i++)
        if (from + AHEAD + i < KEEP) then[i] = load_weight(k, from + AHEAD + i);
      if (AHEAD < KEEP) __builtin_amdgcn_sched_barrier(0);   // (the registers hold no more of the weight)
#pragma unroll
      for (int i = 0; i < AHEAD; i++)
#pragma unroll
        for (int blk = 0; blk < BLOCKS; blk++) acc[blk] = M::run16(keep[blk][from + i], now[i], acc[blk]);
      if (AHEAD < KEEP) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < AHEAD; i++) now[i] = then[i];
    }
    for (int st = KEEP; KEEP > 4 && st < steps; st++) {
      const u32x4 wf = load_weight(k, st);
#pragma unroll
      for (int blk = 0; blk < BLOCKS; blk++)
        acc[blk] = M::run16(gradient(position(pg * GROUP + blk * 16 + p16), st), wf, acc[blk]);
    }
  };
  // ---- a group's samples -----------------------------------------------------------------------------------------
  int bd[SETS], bh[SETS], bw[SETS];
  unsigned at0[SETS];
  bool live[SETS];
  // offsets and mask as they are stored: requested a pair ahead, converted where they are used
  T rd[SETS], rh[SETS], rw[SETS], rm[SETS];
  const unsigned step = static_cast<unsigned>(s.Q) * ES;
  auto request = [&](int k) {
    const bool second = half && k + 1 < s.K;   // (beyond the last tap: the first of the pair)
    const char *o = reinterpret_cast<const char *>(off + (bg * s.K + k) * ND * s.Q), *m = reinterpret_cast<const char *>(mask + (bg * s.K + k) * s.Q);
#pragma unroll
    for (int e = 0; e < SETS; e++) {
      const unsigned at = at0[e] + (second ? ND * step : 0u);
      if (ND == 3) rd[e] = *reinterpret_cast<const T *>(o + at);
      rh[e] = *reinterpret_cast<const T *>(o + (ND - 2) * static_cast<long>(step) + at);
      rw[e] = *reinterpret_cast<const T *>(o + (ND - 1) * static_cast<long>(step) + at);
      if (mask) rm[e] = *reinterpret_cast<const T *>(m + (at0[e] + (second ? step : 0u)));
    }
  };
  const int kfirst = min(k0, s.K - 1);   // (k0 == K: a share without taps)
  auto open = [&](int pg) {
#pragma unroll
    for (int e = 0; e < SETS; e++) {
      const Position own = position(pg * GROUP + e * 32 + n);
      bd[e] = own.d * s.sd - s.pd; bh[e] = own.h * s.sh - s.ph; bw[e] = own.w * s.sw - s.pw;
      at0[e] = static_cast<unsigned>(own.q) * ES;
      live[e] = own.live;
    }
    request(kfirst);
  };
  u32x4 weights[AHEAD];   // of the next product, requested behind the one before

  // The first group's inputs are on their way while the tile is cleared.
  open(wave % pwaves);
  load_keep(wave % pwaves);
  load_weights(kfirst, weights);
  for (int i = threadIdx.x; i < S::VOX * CELL / 16; i += WAVES * 64) reinterpret_cast<u32x4 *>(tile)[i] = u32x4{0u, 0u, 0u, 0u};
  if (threadIdx.x == 0) wgmax = 0u;
  __syncthreads();

  float up = 1.f, down = 1.f;
  if constexpr (NARROW) {
    // ---- first sweep: max |gcol| over the brick's positions, the taps and the channels --------------------------
    float top = 0.f;
    for (int pg = wave % pwaves; pg < groups; pg += pwaves) {
      load_keep(pg);
      if (!some) continue;
      for (int k = k0; k < k1; k++) {
        float4_t acc[BLOCKS];
        product(weights, k, pg, acc);
        load_weights(k + 1 < k1 ? k + 1 : k0, weights);
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
  const TileAxis ad(origin.d, S::TD, s.D), ah(origin.h, S::TH, s.H), aw(origin.w, S::TW, s.W);
  char *const sums = reinterpret_cast<char *>(tile) + p16 % CH * sizeof(Sum);

  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(
      gxt + static_cast<long>(b) * s.P * s.Cin, 0, static_cast<int>(s.P * s.Cin * 4), kRsrcFlags);
  constexpr int CELLS = 64 / CH, TURNS = (S::TW + CELLS - 1) / CELLS;   // cells of a turn
  const int first = lane / CH;
  const unsigned turn_bytes = static_cast<unsigned>(CELLS * s.Cin) * 4u, place = static_cast<unsigned>(first * s.Cin + lane % CH) * 4u;
  for (int turn = 0; turn < turns; turn++) {
    for (int pg = wave % pwaves; pg < groups; pg += pwaves) {
      if (groups > pwaves) {
        load_keep(pg);
        if (pg != wave % pwaves || turn > 0) open(pg);
      }
      if (!some) continue;   // (positions beyond the output)
      int kt = k0 + half;  // the lane's own tap
      int ki = kt / (s.kh * s.kw), kj = (kt / s.kw) % s.kh, kk = kt % s.kw;
      for (int k = k0; k < k1; k += 2) {
        // the lane's samples: byte offset of the first cell, the corners' weights times the mask (and the scale)
        int cell[SETS];
        float w[SETS][NC];
#pragma unroll
        for (int e = 0; e < SETS; e++) {
          float m = mask ? static_cast<float>(load(&rm[e])) : 1.f;
          m = live[e] && kt < k1 ? (NARROW ? m * up : m) : 0.f;
          float wd[2] = {1.f, 0.f}, wh[2], ww[2], at = 0.f;
          if constexpr (ND == 3) at = ad.sample<S::TD>(static_cast<P>(load(&rd[e])) + static_cast<P>(bd[e] + ki * s.dd), wd[0], wd[1]);
          const float ath = ah.sample<S::TH>(static_cast<P>(load(&rh[e])) + static_cast<P>(bh[e] + kj * s.dh), wh[0], wh[1]);
          const float atw = aw.sample<S::TW>(static_cast<P>(load(&rw[e])) + static_cast<P>(bw[e] + kk * s.dw), ww[0], ww[1]);
          at = fmaf(at, static_cast<float>(S::TH), ath);
          cell[e] = static_cast<int>(fmaf(at, static_cast<float>(S::TW), atw)) * CELL;
#pragma unroll
          for (int c = 0; c < NC; c++) w[e][c] = m * wd[c >> 2] * wh[(c >> 1) & 1] * ww[c & 1];
        }
        request(k + 2 < k1 ? k + 2 : kfirst);
        kt += 2;
#pragma unroll
        for (int u = 0; u < 2; u++)
          if (++kk == s.kw) { kk = 0; if (++kj == s.kh) { kj = 0; ++ki; } }
        unrolled(std::make_integer_sequence<int, TAPS>{}, [&](auto uc) {
          constexpr int u = decltype(uc)::value;
          if (k + u >= k1) return;
          float4_t acc[BLOCKS];
          product(weights, k + u, pg, acc);
          const int next = k + (CH == 16 ? u + 1 : 2);
          load_weights(next < k1 ? next : kfirst, weights);
          unrolled(std::make_integer_sequence<int, 8 * SETS>{}, [&](auto ic) {
            constexpr int i = decltype(ic)::value, e = i / 8, FROM = u * 8 + i % 8;   // position 4 j + i % 4 of block i / 4
            const float gv = acc[i / 4][i % 4];
            char *const dst = sums + row_word<CH, FROM>(cell[e]);
            const double gd = static_cast<double>(gv) * scale.up;
#pragma unroll
            for (int c = 0; c < NC; c++) {
              Sum *const to = reinterpret_cast<Sum *>(dst + ((c >> 2) * (S::TH * S::TW) + ((c >> 1) & 1) * S::TW + (c & 1)) * CELL);
              const float wc = row_value<CH, FROM>(w[e][c]);
              if constexpr (NARROW) __hip_atomic_fetch_add(to, round_word(wc * gv), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
              else __hip_atomic_fetch_add(to, fixed_term(wc, gd), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
          });
        });
      }
    }
    if (turn + 1 < turns) {   // the next turn's first weights
      cl += CH;
      load_weights(kfirst, weights);
    }
    __syncthreads();
    // ---- the tile's voxels inside the volume go to the gradient buffer, all channels of a voxel at once: a row of the tile per
    // wavefront, whose place is then scalar arithmetic ------------------------------------------------------------
    for (int row = wave; row < S::TD * S::TH; row += WAVES) {
      const int zd = row / S::TH + origin.d, zh = row % S::TH + origin.h;
      if (zd < 0 || zd >= s.D || zh < 0 || zh >= s.H) continue;
      const unsigned at = static_cast<unsigned>(((zd * s.H + zh) * s.W + origin.w) * s.Cin + c0) * 4u + place;   // (may lie before the row)
      Sum *const from = tile + row * S::TW * CH + lane;
#pragma unroll
      for (int u = 0; u < TURNS; u++) {
        const int cell = u * CELLS + first, zw = cell + origin.w;
        if (S::TW % CELLS && u == TURNS - 1 && cell >= S::TW) continue;
        const Sum sum = from[u * 64];
        if (turn + 1 < turns) from[u * 64] = 0;
        const float v = NARROW ? static_cast<float>(sum) * down
                               : static_cast<float>(static_cast<double>(static_cast<long long>(sum)) * scale.down);
        if (zw >= 0 && zw < s.W && v != 0.f)
          __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(v, gr, at + u * turn_bytes, 0, 0);
      }
    }
    c0 += CH;
    if (turn + 1 < turns) __syncthreads();
  }
}

// 4 x 8 x 8 positions at stride 1: six voxels to spare along d, four along h and w.  A voxel more on either side along d costs 20 % more of
// the tile's atomics (10 us for bf16 [2, 32 -> 64, 48^3]) and leaves two thirds of the corners that the tap kernel adds one by
// one (offsets of sigma = 2: 8.4 -> 5.7 %; that kernel 504 -> 462 us); 12 x 14 x 15 and 11 x 15 x 15 were no faster, layers of small offsets
// do not change.
using TileVolume = Tile<12, 14, 14>;
using TileStrided = Tile<12, 12, 13>;   // 4 x 4 x 4 positions: dilation, 64-bit sums
using TileDeep = Tile<9, 10, 14>;       // 4 x 4 x 8 positions, 64-bit sums of 16-bit tensors
using TileDeepStrided = Tile<8, 12, 13>;   // 2 x 4 x 4 positions, the same at stride 2
template <typename S> constexpr bool kDeep = std::is_same<S, TileDeep>::value || std::is_same<S, TileDeepStrided>::value;
using TileImage = Tile<1, 44, 44>;      // 32 x 32 positions, 32-bit sums; 16 x 16 positions whose taps are further apart
using TileWide = Tile<1, 28, 44>;       // 16 x 32 positions (8 x 16 at stride 2), 64-bit sums of 16-bit tensors
using TileSmall = Tile<1, 28, 28>;      // 16 x 16 or 8 x 8 positions
// The same for fp32, 8 channels: twice the workgroups for the few large bricks that fp32 has (backward pass of [1, 256 -> 128, 27 x 58] 155 us,
// 165 us with 16; with twice as many bricks 16 would be 3 - 5 % faster).
struct TileSmallF32 : TileSmall {
  template <bool NARROW> static constexpr int channels = 8;
};

// Voxels along one axis that the undeformed taps of neighbouring positions reach
static long dcn_reach(int positions, int stride, int taps, int dilation) {
  return (positions - 1L) * stride + (taps - 1L) * dilation + 1;
}
// Dense layers: positions and taps close together along every axis, a rule of the layer whatever the tiles hold (tiles that grew by two voxels
// took layers of stride (2, 1, 1), dilation (3, 1, 1) and 7 x 3 x 3 taps with them, whose 32-bit sums were 14 - 18 % off there).
static bool dcn_dense(const DcnDims &s) {
  if (s.nd == 2) return dcn_reach(32, s.sh, s.kh, s.dh) <= 42 && dcn_reach(32, s.sw, s.kw, s.dw) <= 42;
  return dcn_reach(4, s.sd, s.kd, s.dd) <= 8 && dcn_reach(8, s.sh, s.kh, s.dh) <= 12 && dcn_reach(8, s.sw, s.kw, s.dw) <= 12;
}
// Among them, volumes that take bricks of 4 x 8 x 8 positions.  Those whose taps reach further have bricks of 4 x 4 x 4 (also where the
// larger tile would hold them): two bits more for a term, and one maximum for a quarter of the positions.
static bool dcn_dense_large(const DcnDims &s) {
  return dcn_reach(4, s.sd, s.kd, s.dd) <= 6 && dcn_reach(8, s.sh, s.kh, s.dh) <= 10 && dcn_reach(8, s.sw, s.kw, s.dw) <= 10;
}

// The brick and its tile: the first of the list whose tile holds the reach of the brick's undeformed taps with two voxels to spare
// on either side, or one, if none has two.  Images with fewer workgroups than compute units take a smaller brick (77 us ->
// 35 us for [1, 256 -> 128, 27 x 58]); volumes do not (the halo of 4 x 4 x 4 positions is most of their tile: 117 us
// against 78 us for [2, 16 -> 128, 7 x 19 x 32]).  False: no brick fits.
//
// 16-bit images with 64-bit sums have smaller tiles of 16 channels instead of 44 x 44 of 8: half the samples to work out, and
// 5.5 million requests of 64 bytes instead of 9.9 of 32 for [8, 256 -> 256, 100 x 152].  Where no brick of 16-bit images gives a
// workgroup to every compute unit, the one of most workgroups (backward passes of fp16 [2, 128 -> 256, 36 x 18] 150 -> 112 us,
// [1, 64 -> 64, 24 x 24] 109 -> 72 us, [1, 256 -> 128, 27 x 58] 124 -> 109 us).  Taps too far apart for those tiles (3 x 3 taps from dilation 9 on)
// have 16 x 16 positions in 44 x 44 of 8 channels, up to dilation 13 (backward pass at dilation 12, every corner left to the tap kernel
// and with this tile: fp16 [2, 64 -> 64, 64 x 64] 142 and 121 us, [2, 256 -> 256, 64 x 64] 305 and 264 us); so have dense images,
// with 16 channels, where 32 x 32 positions leave fewer than four voxels to spare (fp16 [2, 128 -> 128, 112 x 120] at dilation 5: 302 us
// with 8 x 8 positions in 28 x 28, 233 us).
//
// Tensors of fp32 keep the largest bricks: every addition of a tile's sums to memory rounds.  Images, with the lists of 16-bit ones
// ([1, 64 -> 64, 24 x 24] in 8 x 8 positions, not 32 x 32): gradient 1.56e-7 (rms) off instead of 1.52e-7, backward pass 100 instead
// of 125 us, [2, 128 -> 128, 112 x 208] 658 instead of 730 us.  Volumes ([4, 16 -> 16, 17 x 43 x 30] with 9 x 10 x 14 of 16 channels): 1.5e-7
// instead of 1.3e-7, 244 instead of 343 us.
//
// Volumes of 16-bit tensors with 64-bit sums have smaller tiles of 16 channels too, where they leave three voxels to spare:
// bf16 [4, 32 -> 128, 57 x 51 x 27] at stride 2 472 us with 12 x 12 x 13 of 8, 407 us with 8 x 12 x 13 of 16 (the tap kernel, which
// adds the corners beyond the smaller bricks' tiles, 236 -> 275 us).  With 32-bit sums, where 16 channels fit the larger tile, smaller ones
// only cost more halo (30 layers of fewer than 256 workgroups: 2 % slower).
//
// Width of the sums: 32 bits round every term to 14 - 22 bits of the workgroup's largest, which is worth their speed in dense
// layers alone (dcn_dense; 16-bit tensors, up to 128 output channels).  Backward passes with 32 and with 64 bits: bf16 volumes
// [2, 32 -> 64, 48^3] 838 and 1140 us, [2, 64 -> 64, 24 x 32 x 32] 436 and 553 us; fp16 images [2, 64 -> 128, 100 x 152] 173 - 189 and
// 183 - 187 us, [2, 128 -> 128, 112 x 208] 283 - 304 and 290 - 297 us: no gain any more.  Strided and wide layers have 64-bit sums, as good as
// fp32 ones: where the output's gradient is 2^-14 of what it is elsewhere in the brick, 32 bits left them 2 - 20 % off.
bool dcn_scatter_plan(const DcnDims &s, int dtype, ScatterShape &shape) {
  static const int volumes[2][6] = {{2, 3, 3, 12, 14, 14}, {2, 2, 2, 12, 12, 13}};
  static const int deep[2][6] = {{2, 2, 3, 9, 10, 14}, {1, 2, 2, 8, 12, 13}};
  static const int large_images[4][6] = {{0, 5, 5, 1, 44, 44}, {0, 4, 4, 1, 28, 28}, {0, 4, 4, 1, 44, 44}, {0, 3, 3, 1, 28, 28}};
  static const int images[4][6] = {{0, 4, 5, 1, 28, 44}, {0, 4, 4, 1, 28, 28}, {0, 3, 4, 1, 28, 44}, {0, 3, 3, 1, 28, 28}};
  static const int far_images[1][6] = {{0, 4, 4, 1, 44, 44}};
  const bool image = s.nd == 2;
  const int st[3] = {s.sd, s.sh, s.sw}, kn[3] = {s.kd, s.kh, s.kw}, dl[3] = {s.dd, s.dh, s.dw}, on[3] = {s.Do, s.Ho, s.Wo};
  // voxels to spare in a tile; workgroups
  const auto spare_of = [&](const int *e) {
    long spare = 1 << 20;
    for (int a = image ? 1 : 0; a < 3; a++)
      spare = std::min(spare, e[3 + a] - (static_cast<long>((1 << e[a]) - 1) * st[a] + static_cast<long>(kn[a] - 1) * dl[a] + 1));
    return (1L << (e[0] + e[1] + e[2])) * s.K >= (1L << 20) ? -1 : spare;
  };
  const auto workgroups = [&](const int *e, int channels) {
    long bricks = s.B;
    for (int a = 0; a < 3; a++) bricks *= (on[a] + (1 << e[a]) - 1) >> e[a];
    return bricks * (s.Cin / channels);
  };
  const auto choose = [&](const int (*list)[6], int count, int channels) {
    int best = -1;
    const int *taken = nullptr;
    for (int i = 0; i < count; i++) {
      const int *e = list[i];
      const long spare = spare_of(e);
      if (spare < 2) continue;
      const int rank = (spare >= 4 ? 2 : 0) + (image && workgroups(e, channels) >= 256 ? 1 : 0);
      if (rank < best || (rank == best && !(image && dtype != MV_F32 && workgroups(taken, channels) < 256))) continue;
      best = rank;
      taken = e;
      shape = ScatterShape{e[0], e[1], e[2], e[3], e[4], e[5], 0, 0, 0, (1 << (e[0] + e[1] + e[2])) * s.K, 0, 1};
    }
    return best >= 0;
  };
  // (offsets and weights at 32-bit byte offsets from scalar bases)
  if (s.Cin / 8 > 65535 || s.Q >= (1L << 28) || static_cast<long>(s.K) * s.cpg * s.opg * (dtype == MV_F32 ? 4 : 2) >= (1L << 31)) return false;
  bool fits = false;
  if (dtype != MV_F32 && s.opg <= 128 && dcn_dense(s)) {
    fits = image ? choose(large_images, 4, 16) : choose(dcn_dense_large(s) ? volumes : volumes + 1, 1, 16);
    shape.narrow = fits && shape.terms <= kScatter32Terms;
  }
  if (!shape.narrow) {
    const int (*const small)[6] = image || dtype == MV_F32 ? nullptr : spare_of(deep[0]) >= 3 ? deep : spare_of(deep[1]) >= 3 ? deep + 1 : nullptr;
    fits = image ? (dtype == MV_F32 ? choose(large_images, 4, 8) : choose(images, 4, 16)) : small ? choose(small, 1, 16) : choose(volumes, 2, 8);
    const int taken[6] = {shape.bd, shape.bh, shape.bw, shape.td, shape.th, shape.tw};
    if (image && (!fits || spare_of(taken) < 4) && spare_of(far_images[0]) >= (fits ? 4 : 2)) fits = choose(far_images, 1, 8);
  }
  if (!fits) return false;
  shape.nbd = (s.Do + (1 << shape.bd) - 1) >> shape.bd;
  shape.nbh = (s.Ho + (1 << shape.bh) - 1) >> shape.bh;
  shape.nbw = (s.Wo + (1 << shape.bw) - 1) >> shape.bw;
  // wide images: 32 channels in two turns, which share grad_output, while that leaves four workgroups per compute unit
  // (fp16 [8, 256 -> 256, 100 x 152]: 500 us, 575 us in one turn, four turns the same)
  shape.turns = image && static_cast<double>(shape.nbd) * shape.nbh * shape.nbw * s.B * (s.Cin / 16) >= 2048 ? 2 : 1;
  return static_cast<double>(shape.nbd) * shape.nbh * shape.nbw * s.B * (s.Cin / 8) < static_cast<double>(1L << 31);
}

template <typename T, typename S>
static int scatter_launch(const void *off, const void *mask, const void *gyt, const void *wf, float *gxt, const DcnDims &s,
                          const ScatterShape &shape, const unsigned *bounds, hipStream_t stream) {
  const int slices = s.opg / (64 / static_cast<int>(sizeof(T)));
#define MV_SCATTER(NARROWV, KEEPV)                                                                                    \
  hipLaunchKernelGGL((dcn_backward_scatter_kernel<T, NARROWV, S, KEEPV>),                                              \
                     linear_grid(static_cast<long>(shape.nbd) * shape.nbh * shape.nbw * s.B *                           \
                                     (s.Cin / (S::template channels<NARROWV> * (KEEPV == 8 && S::template channels<NARROWV> == 16 ? shape.turns : 1))), \
                                 KEEPV <= 4 ? 1024 : 512),                                                              \
                     dim3(KEEPV <= 4 ? 1024 : 512), 0, stream,                                                         \
                     static_cast<const T *>(off), static_cast<const T *>(mask), static_cast<const T *>(gyt),          \
                     static_cast<const T *>(wf), gxt, s, shape, bounds)
  if (shape.narrow) {
    if constexpr (sizeof(T) == 2 && !kDeep<S> && !S::WIDE) {   // (those have 64-bit sums)
      if (slices <= 2) MV_SCATTER(true, 2); else MV_SCATTER(true, 4);
    }
  } else if constexpr (!((kDeep<S> || S::WIDE) && sizeof(T) == 4)) {   // (never of those)
    if (slices <= 2) MV_SCATTER(false, 2);
    else if (slices <= 4) MV_SCATTER(false, 4);
    else MV_SCATTER(false, 8);
  }
#undef MV_SCATTER
  return check_launch("dcn_backward_scatter_kernel");
}

int dcn_scatter(const void *off, const void *mask, const void *gyt, const void *wf, float *gxt, const DcnDims &s,
                const ScatterShape &shape, const unsigned *bounds, int dtype, hipStream_t stream) {
#define MV_SCATTER_TILE(T, S) scatter_launch<T, S>(off, mask, gyt, wf, gxt, s, shape, bounds, stream)
#define MV_SCATTER_AS(T)                                                                                              \
  (shape.td == TileDeep::TD ? MV_SCATTER_TILE(T, TileDeep)                                                             \
   : shape.td == TileDeepStrided::TD ? MV_SCATTER_TILE(T, TileDeepStrided)                                              \
   : shape.th == TileVolume::TH ? MV_SCATTER_TILE(T, TileVolume)                                                          \
   : shape.th == TileStrided::TH ? MV_SCATTER_TILE(T, TileStrided)                                                      \
   : shape.th == TileImage::TH ? MV_SCATTER_TILE(T, TileImage)                                                        \
   : shape.tw == TileWide::TW ? MV_SCATTER_TILE(T, TileWide)                                                            \
                              : scatter_launch<T, std::conditional<sizeof(T) == 4, TileSmallF32, TileSmall>::type>(off, mask, gyt, wf, gxt, s, shape, bounds, stream))
  if (dtype == MV_F16) return MV_SCATTER_AS(__half);
  if (dtype == MV_F32) return MV_SCATTER_AS(float);
  return MV_SCATTER_AS(__hip_bfloat16);
#undef MV_SCATTER_AS
#undef MV_SCATTER_TILE
}

}  // namespace mv
