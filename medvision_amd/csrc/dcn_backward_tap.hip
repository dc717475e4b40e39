// Backward of the deformable convolution on the matrix cores: gradients of the offsets, the mask and the weight, and the
// far corners of the gradient of the input (dcn3d_mfma_backward.hip has the equations and the kernels around this one).
//
// One workgroup = one TAP, a range of positions and a chunk of input channels.  With the tap fixed,
//   * its weight block Wt_k [channels x output channels] sits in registers for the whole range,
//   * the gradient of that block, gw_k = gy col_k^T, stays in accumulators over the range (added to memory once),
//   * the column values mask * Z(x) go from the lanes that blend them through LDS into that product,
// so that there is no column buffer and no second gather of x, and a layer of a few thousand positions has taps x ranges
// workgroups instead of one wavefront per 32 positions.  64 positions at a time, grad_output of them in LDS:
//   1  gcol = Wt_k^T gy (16 x 16 MFMA, rows = channels), through LDS to the load layout (position l / 4, 16-byte piece
//      l % 4: a voxel's pieces are one cache look-up);
//   2  every wavefront samples 16 positions: the corners' pieces are loaded once and used twice, blended into the column
//      value and differenced against gcol.  The trilinear form is blended axis by axis, which passes the differences that
//      its derivatives are made of: along w four per channel (images: two), along h two (one), along d one.  Sums over the channels
//      are taken of these differences, and the blends over the axes that are left are done once per position.  (One sum per
//      corner, differenced at the end, is 16 instead of 23 vector instructions per channel, images 8 instead of 11, and loses the
//      digits that nearly equal corners share: 4e-5 of sum |gcol * step| on an input of 64 and 64 + one step of fp16.  That
//      form took 496 us against 493 us for bf16 [2, 32 -> 64, 48^3], 728 us against 762 us for fp16 images
//      [8, 256 -> 256, 100 x 152].);
//   3  gw_k += gy col_k^T, a quarter of the output channels per wavefront, both operands by transposing LDS reads.
// Corners that the LDS scatter does not take are listed when the records are made, and their 32 channels are added as
// 128 contiguous bytes.
// What bounds it: narrow layers the vector instructions of the samples (184 per 16 positions and 32 channels, and as many more
// for everything else; vector issue 68 %) and the latency of the gathers (48 % of the wavefronts' time in waits), wide ones LDS
// (35 %; vector issue 31 %, matrix cores 21 %) and the same waits (49 %), and everywhere the atomics of the far corners (64 bytes per corner
// and 16 channels, 21 G of them a second at best).
//   (bf16 [2, 32 -> 64, 48^3]: 390 us; the data and weight kernels before it took 670 us.  fp16 images
//   [8, 256 -> 256, 100 x 152]: 538 us, 587 with
//   grad_output of a tile loaded when it begins, 4380 before.  [1, 128 -> 128, 7 x 45 x 18]: 60 us, 790 us before.)
#include "dcn_scatter.hpp"

#include <algorithm>

namespace mv {

// One 16-byte piece (kPiece neighbouring channels of a position) of an LDS block [piece][position]: rows of 69 pieces, so that
// eight pieces of a position, the four pieces of neighbouring positions and one piece of sixteen positions fall on different banks
// (rows of 68: eight pieces of a position on four sets of banks; fp16 [8, 256 -> 256, 100 x 152] 616 us, 582 us with 69).
constexpr int kTapTile = 64, kTapPitch = kTapTile + 5;   // positions per turn
__device__ __forceinline__ int tap_slot(int piece, int position) { return piece * kTapPitch + position; }

// Operand of a product over positions from such a block: row `block * 16 + lane % 16` (a channel), the kPiece positions
// 4 * kPiece * ks + ... that belong to lane group lane / 16.  16-bit: two transposing reads (lane 4 e + t of a group of sixteen
// addresses channels 4 t .. 4 t + 3 of position e, lane i gets channel i of the four positions).
template <typename T> __device__ __forceinline__ u32x4 tap_transposed(const u32x4 *base, int block, int ks, int lane) {
  const int kc = lane / 16, i = lane % 16;
  if constexpr (sizeof(T) == 2) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 *lds_ptr;
    const int piece = block * 2 + (i % 4) / 2, half = i % 2, position = ks * 32 + kc * 8 + i / 4;
    const auto at = [&](int add) {
      return (lds_ptr)(reinterpret_cast<s16x4 *>(const_cast<u32x4 *>(base + tap_slot(piece, position + add))) + half);
    };
    union { s16x4 h[2]; u32x4 u; } r;
    r.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(at(0));
    r.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(at(4));
    return r.u;
  } else {
    const int piece = block * 4 + i / 4;
    union { unsigned e[4]; u32x4 u; } r;
#pragma unroll
    for (int t = 0; t < 4; t++) r.e[t] = reinterpret_cast<const unsigned *>(base + tap_slot(piece, ks * 16 + kc * 4 + t))[i % 4];
    return r.u;
  }
}

// A launch's part of the layer: all of it, unless the shares of the offset and mask gradients (`partial`) are limited
// to fewer taps or positions at a time.
struct TapPiece { int k_first, taps, q_first, positions; };

// workgroups per compute unit that the registers should leave room for
template <typename T, int NC, int OBW, int CBW>
constexpr int TAP_WAVES = OBW * CBW >= 8 || (NC == 8 && (sizeof(T) == 4 || OBW >= 2)) ? 2 : OBW == 1 && CBW == 2 && sizeof(T) == 2 ? 4 : 3;

// blocks of 16 channels of gcol per wavefront: two where that halves the reads of grad_output from LDS (a block of four positions each
// would do too, but the registers leave room for two: fp16 [8, 256 -> 256, 100 x 152] 638 -> 616 us, four 740 us;
// bf16 [2, 128 -> 128, 112 x 208] training step 312 -> 295 us)
template <typename T, int NC, int OBW, int CBW> constexpr int TAP_BLOCKS = CBW == 4 ? 2 : 1;

// OBW: blocks of 16 output channels per wavefront (every fourth block of the 64 * OBW rows from row0; layers with more rows
// take several passes, gcol and all that follows from it being sums over them).  CBW: blocks of 16 input channels of a
// chunk.  NC: corners, 8 for volumes, 4 for images.
template <typename T, int NC, int OBW, int CBW>
__global__ __launch_bounds__(256, (TAP_WAVES<T, NC, OBW, CBW>)) void dcn_backward_tap_kernel(
    const T *__restrict__ xt, const T *__restrict__ off, const T *__restrict__ mask, const T *__restrict__ gyt,
    const T *__restrict__ wf, float *__restrict__ gxt, T *__restrict__ goff, T *__restrict__ gmask,
    float *__restrict__ partial, float *__restrict__ gw, const DcnDims s, const unsigned *__restrict__ bounds,
    const ScatterShape shape, const int chunks, const int shares, const int range, const unsigned ranges, const int row0, const TapPiece piece) {
  using M = Mfma<T>;
  using P = typename std::conditional<(sizeof(T) == 2), float, double>::type;  // position type
  constexpr int PC = M::kPiece, SL = 4 * PC, ES = sizeof(T), CW = 16 * CBW, ROWS = 64 * OBW;
  constexpr int BPI = SL / 16, ITEMS = CBW / BPI, KS = kTapTile / SL;   // 16-channel blocks per item; items; K steps of a tile
  constexpr int STEPS = ROWS / SL, STAGED = ROWS * kTapTile / PC / 256;
  constexpr int RW = 12, kRecs = 2 * kTapTile, GP = CW + 4;
  __shared__ __attribute__((aligned(16))) unsigned rec[kRecs][RW];          // at[NC], ld, lh, lw, mask (12 words: sixteen rows on different banks)
  __shared__ u32x4 gyl[ROWS / PC * kTapPitch];                               // grad_output, pieces of output channels
  __shared__ u32x4 col[CW / PC * kTapPitch];                                 // column values, pieces of input channels
  __shared__ __attribute__((aligned(16))) float gcol[kTapTile][GP];
  __shared__ uint2 far_list[2][kTapTile * NC];   // {offset in the gradient buffer | position, mask * weight}
  __shared__ int far_count[2];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int j = lane % 16, kc = lane / 16;   // matrix layout
  const int lj = lane / 4, lk = lane % 4;    // load layout
  // (taps and chunks of one range next to each other, on one XCD: they gather the same part of x and read the same gy)
  const unsigned inner = piece.taps * s.dg * chunks, workgroups = ranges * inner * s.B;
  if (linear_block() >= workgroups) return;
  const unsigned wg = xcd_contiguous(linear_block(), workgroups);
  const int k = piece.k_first + static_cast<int>(wg % piece.taps), slice = static_cast<int>(wg / piece.taps % (s.dg * chunks));
  const int dgi = slice / chunks, part = slice % chunks, b = static_cast<int>(wg / inner / ranges);
  const int c0 = dgi * s.cpd + part * CW, g = c0 / s.cpg;
  const int within = static_cast<int>(wg / inner % ranges) * range;   // < 2^31: within.. is a range of the piece
  const long q0 = piece.q_first + static_cast<long>(within);
  const int count = min(range, piece.positions - within);   // positions of the range
  const long bg = static_cast<long>(b) * s.dg + dgi;
  const int rows = min(ROWS, s.opg - row0), steps = rows / SL;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(xt + static_cast<long>(b) * s.P * s.Cin), 0, static_cast<int>(s.P * s.Cin * ES), kRsrcFlags);
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(
      gxt + static_cast<long>(b) * s.P * s.Cin, 0, static_cast<int>(s.P * s.Cin * 4), kRsrcFlags);
  const bool split = bounds && scatter_scale(bounds, shape.terms, mask != nullptr).valid;

  // gcol: a wavefront forms WB blocks of sixteen channels for CBW / WB blocks of sixteen positions; its rows of the weight stay
  // in registers for the whole range
  constexpr int WB = TAP_BLOCKS<T, NC, OBW, CBW>, WP = CBW / WB;
  const int wblock = wave % (CBW / WB) * WB, wfirst = wave / (CBW / WB) * WP;
  u32x4 wreg[WB][STEPS];
#pragma unroll
  for (int w = 0; w < WB; w++) {
    const T *src = wf + (((static_cast<long>(g) * s.K + k) * (s.cpg / 16) + (c0 - g * s.cpg) / 16 + wblock + w) * (s.opg / SL) + row0 / SL) * (64 * PC) + lane * PC;
#pragma unroll
    for (int st = 0; st < STEPS; st++)
      wreg[w][st] = st < steps ? *reinterpret_cast<const u32x4 *>(src + st * (64 * PC)) : u32x4{0u, 0u, 0u, 0u};
  }
  // grad_output of a tile, loaded a tile ahead where the registers allow it, elsewhere during the tile's last product, when those of the
  // corners are free (loads at the start of the tile had nothing to hide behind: the step above 1456 -> 1407 us): thread t has piece t % NP of positions t / NP +
  // u * 256 / NP (positions and rows that do not exist: zeros)
  constexpr bool AHEAD = STAGED <= 4;
  constexpr int NP = ROWS / PC;
  const int cout_bytes = s.Cout * ES, tpiece = tid % NP, tposition = tid / NP;
  const __amdgpu_buffer_rsrc_t gyr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(gyt + (static_cast<long>(b) * s.Q + q0) * s.Cout), 0, count * cout_bytes, kRsrcFlags);
  const unsigned stage_at = tpiece * PC < rows ? static_cast<unsigned>(tposition * cout_bytes + tpiece * 16) : kOob;
  u32x4 *const keep_at = gyl + tap_slot(tpiece, tposition);
  u32x4 staged[STAGED];
  auto stage = [&](int tile) {
#pragma unroll
    for (int u = 0; u < STAGED; u++)
      staged[u] = __builtin_amdgcn_raw_buffer_load_b128(gyr, stage_at, (tile * kTapTile + u * (256 / NP)) * cout_bytes + (g * s.opg + row0) * ES, 0);
  };
  auto keep = [&] {
#pragma unroll
    for (int u = 0; u < STAGED; u++) keep_at[u * (256 / NP)] = staged[u];
  };

  // ---- records: thread t < 128 works out position t of the next two tiles; its offsets are requested a block ahead -----
  const int ti = k / (s.kh * s.kw), tj = (k / s.kw) % s.kh, tk = k % s.kw;
  const T *const ob = off + (bg * s.nd * s.K + s.nd * k) * s.Q, *const mb = mask ? mask + (bg * s.K + k) * s.Q : nullptr;
  P fd = P(0), fh = P(0), fw = P(0);
  float fm = 1.f;
  auto request = [&](int first) {
    const long q = q0 + min(first + tid, count - 1);
    dcn_offsets(s, ob + q, fd, fh, fw);
    if (mb) fm = load(mb + q);
  };
  auto publish = [&](int first) {
    const bool live = first + tid < count;
    const int qc = static_cast<int>(q0) + min(first + tid, count - 1);
    const int ow = qc % s.Wo, t = qc / s.Wo, oh = t % s.Ho, od = t / s.Ho;
    P pd = fd + static_cast<P>(od * s.sd - s.pd + ti * s.dd);
    const P ph = fh + static_cast<P>(oh * s.sh - s.ph + tj * s.dh), pw = fw + static_cast<P>(ow * s.sw - s.pw + tk * s.dw);
    if (NC == 4) pd = P(0);   // images: the only slice
    CornerTaps ct;
    corner_taps<P>(s, pd, ph, pw, live, static_cast<unsigned>(s.Cin) * ES, 0u, kOob, ct);
    unsigned *r = rec[tid];
#pragma unroll
    for (int c = 0; c < NC; c += 4) *reinterpret_cast<u32x4 *>(r + c) = u32x4{ct.at[c], ct.at[c + 1], ct.at[c + 2], ct.at[c + 3]};
    *reinterpret_cast<float4 *>(r + NC) = make_float4(ct.ld, ct.lh, ct.lw, fm);
    int first_cell;
    const unsigned local = split ? tile_bits(shape, tile_origin(s, shape, od >> shape.bd, oh >> shape.bh, ow >> shape.bw),
                                             static_cast<int>(floor(pd)), static_cast<int>(floor(ph)), static_cast<int>(floor(pw)), first_cell) : 0u;
    int listed = 0;   // (the wavefront is one tile)
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const bool is_far = ct.at[c] != kOob && !((local >> c) & 1u);
      const unsigned long long owners = __ballot(is_far);
      // (a voxel's channels start at a multiple of 128 bytes: the position fits below)
      if (is_far)
        far_list[wave][listed + __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(owners >> 32),
                                                         __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(owners), 0u))] =
            make_uint2(ct.at[c] * (4u / ES) | static_cast<unsigned>(lane), __float_as_uint(fm * ct.w[c]));
      listed += __popcll(owners);
    }
    if (lane == 0) far_count[wave] = listed;
  };

  float4_t acc[OBW][CBW];
#pragma unroll
  for (int o = 0; o < OBW; o++)
#pragma unroll
    for (int c = 0; c < CBW; c++) acc[o][c] = float4_t{0.f, 0.f, 0.f, 0.f};

  // lane l % 4 stores component l % 4 of its position (d, h, w, mask)
  float *pout = nullptr;
  T *tout = nullptr;
  {
    const int p = wave * 16 + lj;
    if (partial)
      pout = partial + (((bg * piece.taps + k - piece.k_first) * shares + row0 / ROWS * chunks + part) * piece.positions + within + p) * 4 + lk;
    else if (lk == 3) tout = gmask ? gmask + (bg * s.K + k) * s.Q + q0 + p : nullptr;
    else if (lk + s.nd >= 3) tout = goff + (bg * s.nd * s.K + s.nd * k + lk + s.nd - 3) * s.Q + q0 + p;
  }
  if (tid < kRecs) request(0);
  stage(0);
  const int tiles = (count + kTapTile - 1) / kTapTile;
  for (int tile = 0; tile < tiles; tile++) {
    const int half = tile & 1;
    __syncthreads();   // the tile before has been read
    keep();
    if (half == 0 && tid < kRecs) {
      publish(tile * kTapTile);
      if (tile + 2 < tiles) request(tile * kTapTile + kRecs);
    }
    __syncthreads();
    // ---- the sampling pieces of this wavefront's sixteen positions are on their way during the product ---------------
    const int p = wave * 16 + lj;
    const unsigned *r = rec[half * kTapTile + p];
    unsigned at[NC];
#pragma unroll
    for (int c = 0; c < NC; c += 4) {
      const u32x4 a = *reinterpret_cast<const u32x4 *>(r + c);
      at[c] = a.x + lk * 16u; at[c + 1] = a.y + lk * 16u; at[c + 2] = a.z + lk * 16u; at[c + 3] = a.w + lk * 16u;
    }
    const float4 e = *reinterpret_cast<const float4 *>(r + NC);   // ld, lh, lw, mask
    constexpr int SETS = NC == 4 && ITEMS > 1 ? 2 : 1;   // items whose corners are in registers (volumes: one, for occupancy)
    u32x4 raw[SETS][NC];
    auto gather = [&](u32x4 (&to)[NC], int item) {
#pragma unroll
      for (int c = 0; c < NC; c++) to[c] = __builtin_amdgcn_raw_buffer_load_b128(xr, at[c], (c0 + item * SL) * ES, 0);
    };
    gather(raw[0], 0);
    if (AHEAD) stage(tile + 1);   // (beyond the last one: zeros)
    {
      float4_t gc[WB][WP];
#pragma unroll
      for (int w = 0; w < WB; w++)
#pragma unroll
        for (int n = 0; n < WP; n++) gc[w][n] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < STEPS; st++)
#pragma unroll
        for (int n = 0; n < WP; n++) {
          const u32x4 gy = gyl[tap_slot(st * 4 + kc, (wfirst + n) * 16 + j)];
#pragma unroll
          for (int w = 0; w < WB; w++) gc[w][n] = M::run16(wreg[w][st], gy, gc[w][n]);
        }
#pragma unroll
      for (int w = 0; w < WB; w++)
#pragma unroll
        for (int n = 0; n < WP; n++)
          *reinterpret_cast<float4 *>(&gcol[(wfirst + n) * 16 + j][(wblock + w) * 16 + 4 * kc]) = make_float4(gc[w][n][0], gc[w][n][1], gc[w][n][2], gc[w][n][3]);
    }
    __syncthreads();   // gcol is complete
    // sums over the lane's channels: differences along w (along h, d), value
    float sw[NC / 2], sh[NC / 4], sd = 0.f, sv = 0.f;
#pragma unroll
    for (int c = 0; c < NC / 2; c++) sw[c] = 0.f;
#pragma unroll
    for (int c = 0; c < NC / 4; c++) sh[c] = 0.f;
#pragma unroll
    for (int item = 0; item < ITEMS; item++) {
      if (SETS == 2 && item + 1 < ITEMS) gather(raw[(item + 1) % SETS], item + 1);
      const u32x4(&x)[NC] = raw[item % SETS];
      float gv[PC], v[PC];
#pragma unroll
      for (int i = 0; i < PC; i += 4) {
        const float4 t = *reinterpret_cast<const float4 *>(&gcol[p][item * SL + lk * PC + i]);
        gv[i] = t.x; gv[i + 1] = t.y; gv[i + 2] = t.z; gv[i + 3] = t.w;
      }
#pragma unroll
      for (int i = 0; i < PC; i++) {
        float row[NC / 2], plane[NC / 4];   // blended along w; along w and h
#pragma unroll
        for (int c = 0; c < NC / 2; c++) {
          const float first = M::element(x[2 * c], i), step = M::element(x[2 * c + 1], i) - first;
          sw[c] = fmaf(step, gv[i], sw[c]);
          row[c] = fmaf(e.z, step, first);
        }
#pragma unroll
        for (int c = 0; c < NC / 4; c++) {
          const float step = row[2 * c + 1] - row[2 * c];
          sh[c] = fmaf(step, gv[i], sh[c]);
          plane[c] = fmaf(e.y, step, row[2 * c]);
        }
        float value = plane[0];
        if constexpr (NC == 8) {
          const float step = plane[1] - plane[0];
          sd = fmaf(step, gv[i], sd);
          value = fmaf(e.x, step, plane[0]);
        }
        sv = fmaf(value, gv[i], sv);
        v[i] = e.w * value;
      }
      col[tap_slot(item * 4 + lk, p)] = M::pack(v);
      if (SETS == 1 && item + 1 < ITEMS) gather(raw[0], item + 1);
    }
    const auto mix = [](float f, float a, float b) { return fmaf(f, b - a, a); };
    float t0 = sd, t1 = sh[0], t2 = mix(e.y, sw[0], sw[1]), t3 = sv;
    if constexpr (NC == 8) {
      t1 = mix(e.x, sh[0], sh[1]);
      t2 = mix(e.x, t2, mix(e.y, sw[2], sw[3]));
    }
    // the four pieces of a position: lane l % 4 ends with the sum of component l % 4
#define MV_QUAD(v, ctrl) __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), ctrl, 0xf, 0xf, true))
    {
      const bool odd = lk & 1, upper = lk & 2;
      const float u0 = (odd ? t1 : t0) + MV_QUAD(odd ? t0 : t1, 0xB1);   // xor 1: components 0 | 1
      const float u1 = (odd ? t3 : t2) + MV_QUAD(odd ? t2 : t3, 0xB1);   // components 2 | 3
      const float sum = (upper ? u1 : u0) + MV_QUAD(upper ? u0 : u1, 0x4E);
      const float out = lk < 3 ? e.w * sum : sum;
      if (tile * kTapTile + p < count) {
        if (partial) pout[tile * (kTapTile * 4)] = out;
        else if (tout) tout[tile * kTapTile] = store_cast<T>(out);
      }
    }
#undef MV_QUAD
    __syncthreads();   // the tile's column values are complete
    // ---- far corners: 32 lanes add an entry's channels, 32 at a time -------------------------------------------------
    const int far = __builtin_amdgcn_readfirstlane(far_count[half]), n = tid % 32;
    for (int i = tid / 32; i < far; i += 8) {
      const uint2 entry = far_list[half][i];
      const float w = __uint_as_float(entry.y);
      const float *src = gcol[entry.x & 63u];
      const unsigned base = (entry.x & ~127u) + static_cast<unsigned>(c0 + n) * 4u;
#pragma unroll
      for (int c = 0; c < CW; c += 32)
        __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(w * src[c + n], gr, base + c * 4u, 0, 0);
    }
    if (!AHEAD) stage(tile + 1);   // (beyond the last one: zeros)
    // ---- gw += gy col^T, a quarter of the rows per wavefront -------------------------------------------------------
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      u32x4 a[OBW];
#pragma unroll
      for (int o = 0; o < OBW; o++) a[o] = tap_transposed<T>(gyl, o * 4 + wave, ks, lane);
#pragma unroll
      for (int c = 0; c < CBW; c++) {
        const u32x4 bf = tap_transposed<T>(col, c, ks, lane);
#pragma unroll
        for (int o = 0; o < OBW; o++) acc[o][c] = M::run16(a[o], bf, acc[o][c]);
      }
    }
  }
  // accumulator register r of lane l: output channel 4 * (l / 16) + r of its block, input channel l % 16
#pragma unroll
  for (int o = 0; o < OBW; o++) {
    const int row = (o * 4 + wave) * 16;
    if (row >= rows) continue;
#pragma unroll
    for (int c = 0; c < CBW; c++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        atomicAdd(gw + (static_cast<long>(k) * s.Cout + g * s.opg + row0 + row + 4 * kc + i) * s.cpg + c0 - g * s.cpg + c * 16 + j,
                  acc[o][c][i]);
  }
}

// The chunks' shares of the offset and mask gradients, summed.
template <typename T>
__global__ __launch_bounds__(256) void dcn_backward_partial_kernel(const float4 *__restrict__ partial, T *__restrict__ goff,
                                                                   T *__restrict__ gmask, const DcnDims s, const int chunks,
                                                                   const TapPiece piece) {
  const long q = blockIdx.x * 256L + threadIdx.x, row = blockIdx.y + static_cast<long>(blockIdx.z) * s.dg * piece.taps;
  if (q >= piece.positions) return;
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int c = 0; c < chunks; c++) {
    const float4 v = partial[(row * chunks + c) * piece.positions + q];
    sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
  }
  const long bgk = row / piece.taps * s.K + piece.k_first + row % piece.taps;
  T *go = goff + bgk * s.nd * s.Q + piece.q_first + q;
  if (s.nd == 3) *go = store_cast<T>(sum.x);
  go[(s.nd - 2) * s.Q] = store_cast<T>(sum.y);
  go[(s.nd - 1) * s.Q] = store_cast<T>(sum.z);
  if (gmask) gmask[bgk * s.Q + piece.q_first + q] = store_cast<T>(sum.w);
}

// Chunks of 64 input channels for 16-bit images (four corners; grad_output of a tile then serves twice the channels), 32
// for volumes and fp32, whose eight corners or wider pieces would leave too few registers for two workgroups on a SIMD,
// and where a group is no multiple of 64.
static int tap_chunk(const DcnDims &s, int dtype) {
  return dtype != MV_F32 && s.nd == 2 && s.cpd % 64 == 0 && s.cpg % 64 == 0 ? 64 : 32;
}
static int tap_chunks(const DcnDims &s, int dtype) { return s.cpd / tap_chunk(s, dtype); }
// rows of a pass: 256 (fp32: 128) output channels keep grad_output of 64 positions within 32 KB of LDS
static int tap_rows(int dtype) { return dtype == MV_F32 ? 128 : 256; }
static int tap_shares(const DcnDims &s, int dtype) { return tap_chunks(s, dtype) * ((s.opg + tap_rows(dtype) - 1) / tap_rows(dtype)); }

constexpr long kTapRange = 64 * kTapTile;   // positions of a workgroup at most

// Taps and positions of a launch (TapPiece): as many as keep the shares of several chunks within `budget` bytes, fewer positions
// only where a single tap is beyond it, one range of them at least.
static long tap_share_bytes(const DcnDims &s, int dtype) { return static_cast<long>(s.B) * s.dg * tap_shares(s, dtype) * 16; }
static void tap_pieces(const DcnDims &s, int dtype, size_t budget, long &taps, long &positions) {
  taps = s.K;
  positions = s.Q;
  if (tap_shares(s, dtype) == 1) return;
  const long fits = static_cast<long>(std::min(budget, static_cast<size_t>(1) << 62)) / tap_share_bytes(s, dtype);   // taps x positions
  taps = std::min(std::max(fits / s.Q, 1L), static_cast<long>(s.K));
  if (fits < s.Q) positions = std::min(std::max(fits / kTapRange, 1L) * kTapRange, s.Q);
}
size_t dcn_tap_partial_bytes(const DcnDims &s, int dtype, size_t budget) {
  if (tap_shares(s, dtype) == 1) return 0;
  long taps, positions;
  tap_pieces(s, dtype, budget, taps, positions);
  return static_cast<size_t>(tap_share_bytes(s, dtype)) * taps * positions;
}
bool dcn_tap_supported(const DcnDims &s, int dtype) {
  // (a range of 4096 positions of grad_output within 32-bit byte offsets)
  return s.Q < (1L << 31) && s.Cout <= 65536 && static_cast<long>(s.dg) * tap_chunks(s, dtype) <= 65535 && static_cast<long>(s.dg) * s.K <= 65535;
}

// Ranges of positions.  The workgroups of a launch do the same work, so that they should fill the places on the chip (`slots`) a whole
// number of times: with about four workgroups per compute unit bf16 [2, 32 -> 64, 48^3] had 1458 workgroups on 1024 places (446 us,
// now 1998: 411 us), fp16 [8, 256 -> 256, 100 x 152] 1152 on 512 (745 us, now 1440: 653 us).  Every workgroup costs a few tiles of
// its own: the weight and the first offsets (as long as 1.5 tiles), and a block of the weight gradient, `block` fp32 atomics
// at 64 bytes per request, 21 G a second, a tile taking 3.7 us (of those two layers; the ranges hardly depend on it: with 1 to 16 us the
// backward passes of twelve layers of all instances differ by at most 4 %, most by 1).  fp32 layers keep four workgroups per compute unit: each addition
// rounds their weight gradient (2.2e-7 rms of it with the ranges of 16-bit layers, 1.9e-7 with these, [2, 64 -> 128, 36 x 40]), at
// 3 to 5 % of a training step.
static long tap_ranges(long tiles, long others, long slots, long block) {
  const double own = 1.5 + static_cast<double>(slots) * block / 16 / (21e9 * 3.7e-6);
  long best = 0;
  double least = 0.0;
  const long first = (tiles + kTapRange / kTapTile - 1) / (kTapRange / kTapTile);
  for (long per = std::min(tiles, kTapRange / kTapTile); per >= 1; per--) {
    const long ranges = (tiles + per - 1) / per, rounds = (ranges * others + slots - 1) / slots;
    const double cost = rounds * (per + own);
    if (best == 0 || cost < least) { best = ranges; least = cost; }
  }
  return std::max(best, first);
}

// workgroups of an instance that the chip holds at a time (256 compute units; a property of the compiled kernel)
template <typename T, int NC, int OBW, int CBW> static long tap_places() {
  static const long places = [] {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(&dcn_backward_tap_kernel<T, NC, OBW, CBW>), 256, 0) != hipSuccess)
      (void)hipGetLastError();
    return 256L * std::max(n, 1);
  }();
  return places;
}

template <typename T, int NC, int CBW>
static int tap_launch(const T *xt, const T *off, const T *mask, const T *gyt, const T *wf, float *gxt, T *goff,
                      T *gmask, float *partial, float *gw, const DcnDims &s, const unsigned *bounds, const ScatterShape &shape, int dtype,
                      const TapPiece &piece, hipStream_t stream) {
  const int chunks = tap_chunks(s, dtype), shares = tap_shares(s, dtype);
  const int rows = std::min(static_cast<int>(s.opg), s.opg <= 64 ? 64 : s.opg <= 128 || sizeof(T) == 4 ? 128 : 256);
  const long others = static_cast<long>(piece.taps) * s.dg * chunks * s.B, tiles = (piece.positions + static_cast<long>(kTapTile) - 1) / kTapTile;
  const long slots = s.opg <= 64 ? tap_places<T, NC, 1, CBW>() : s.opg <= 128 || sizeof(T) == 4 ? tap_places<T, NC, 2, CBW>()
                                                                                                     : tap_places<T, NC, sizeof(T) == 2 ? 4 : 2, CBW>();
  const long four = std::max(1L, 1024 / others), few = std::min(std::max(1L, (tiles + four - 1) / four), kTapRange / kTapTile);
  const long ranges = sizeof(T) == 4 ? (tiles + few - 1) / few : tap_ranges(tiles, others, slots, static_cast<long>(rows) * (16 * CBW));
  const long per = (tiles + ranges - 1) / ranges;
  MV_REQUIRE(static_cast<double>(ranges) * others < static_cast<double>(1L << 31), "grid too large");
  const dim3 grid = linear_grid(ranges * others, 256);
  const int range = static_cast<int>(per * kTapTile);
#define MV_TAP(OBWV, ROW)                                                                                               \
  hipLaunchKernelGGL((dcn_backward_tap_kernel<T, NC, OBWV, CBW>), grid, dim3(256), 0, stream, xt, off, mask, gyt, wf, gxt,     \
                     goff, gmask, partial, gw, s, bounds, shape, chunks, shares, range, static_cast<unsigned>(ranges), ROW, piece)
  if (s.opg <= 64) {
    MV_TAP(1, 0);
  } else if (s.opg <= 128 || sizeof(T) == 4) {
    for (int row = 0; row < s.opg; row += 128) MV_TAP(2, row);
  } else if constexpr (sizeof(T) == 2) {
    for (int row = 0; row < s.opg; row += 256) MV_TAP(4, row);
  }
#undef MV_TAP
  int st = check_launch("dcn_backward_tap_kernel");
  if (st || !partial) return st;
  hipLaunchKernelGGL((dcn_backward_partial_kernel<T>), dim3(static_cast<unsigned>((piece.positions + 255L) / 256), s.dg * piece.taps, s.B),
                     dim3(256), 0, stream, reinterpret_cast<const float4 *>(partial), goff, gmask, s, shares, piece);
  return check_launch("dcn_backward_partial_kernel");
}

// `bounds` null: no scatter kernel runs, every corner of the gradient of the input is added here.  `partial`: memory of
// dcn_tap_partial_bytes(s, dtype, budget).
int dcn_tap_backward(const void *xt, const void *off, const void *mask, const void *gyt, const void *wf,
                     float *gxt, void *goff, void *gmask, float *partial, size_t budget, float *gw, const DcnDims &s,
                     const unsigned *bounds, const ScatterShape &shape, int dtype, hipStream_t stream) {
  if (tap_shares(s, dtype) == 1) partial = nullptr;
  long taps, positions;
  tap_pieces(s, dtype, budget, taps, positions);
#define MV_TAP_AS(T, NC, CBW)                                                                                          \
  tap_launch<T, NC, CBW>(static_cast<const T *>(xt), static_cast<const T *>(off), static_cast<const T *>(mask),           \
                         static_cast<const T *>(gyt), static_cast<const T *>(wf), gxt, static_cast<T *>(goff),            \
                         static_cast<T *>(gmask), partial, gw, s, bounds, shape, dtype, piece, stream)
  const bool wide = tap_chunk(s, dtype) == 64, image = s.nd == 2;
  for (long k = 0; k < s.K; k += taps)
    for (long q = 0; q < s.Q; q += positions) {
      const TapPiece piece{static_cast<int>(k), static_cast<int>(std::min(taps, s.K - k)), static_cast<int>(q),
                           static_cast<int>(std::min(positions, s.Q - q))};
      const int st = dtype == MV_F32 ? (image ? MV_TAP_AS(float, 4, 2) : MV_TAP_AS(float, 8, 2))
                     : dtype == MV_F16 ? (wide ? MV_TAP_AS(__half, 4, 4) : image ? MV_TAP_AS(__half, 4, 2) : MV_TAP_AS(__half, 8, 2))
                     : wide ? MV_TAP_AS(__hip_bfloat16, 4, 4) : image ? MV_TAP_AS(__hip_bfloat16, 4, 2) : MV_TAP_AS(__hip_bfloat16, 8, 2);
      if (st) return st;
    }
#undef MV_TAP_AS
  return MV_OK;
}

}  // namespace mv
