// Matrix-core forward of the deformable convolution for fp16 / bf16 / fp32 tensors, images and volumes.
//
//   y[b, o, q] = sum_{k, c} Wt[o, c, k] * col[c, k, q] + bias[o],
//   col[c, k, q] = mask[k, q] * Z(x[b, c], p(k, q))           (zero-padded trilinear / bilinear sample)
//
// is a GEMM whose right operand, the column matrix, exists 16 pieces (of 16 bytes: 8 or 4 channels of a position) at a
// time in LDS.  The contraction runs over the flat sequence of pieces (tap, deformable group, channels), so that any
// channel count that is a multiple of a piece fills the K steps of the matrix instruction.
//
// Layout: x channels-last [B, P, C] (workspace): ONE 16-byte load per corner brings the channels of a piece, and the four
// lanes of a position fetch four neighbouring pieces, usually one cache line, together.  Weights in fragment order
// (workspace): a wavefront's operand is one coalesced 16-byte load per lane.
//
// Workgroup = PT positions x up to 16 * W * OBW output channels, W wavefronts:
//   records   a thread works out one (unit, position): the corners' byte offsets and weights (times the mask) go
//             to LDS, 64 * W of them at a time; a unit is a tap of one deformable group.  Their offsets are requested a window ahead.
//   samples   an item = 64 / LP positions x LP pieces: load, blend, write the piece to LDS.  The corners of the next item are on
//             their way while one is blended, also across the product in between.
//   product   16 pieces of K against the wavefront's rows of the weight, v_mfma_f32_16x16x32 (fp32: 16x16x4).
// LP: the cache takes a load by the 128-byte lines that it touches (4.6 clocks each when they come from the L2, whatever is read of them), so
// eight neighbouring lanes read a whole line of a corner where its channels are that many (fp16 [8, 256 -> 256, 100 x 152] 274 -> 249 us
// with 64 positions, fp16 [2, 128 -> 64, 24^3] 98 -> 90, fp32 243 -> 217); four, half a line, elsewhere.
// PT, W: 32 positions use a weight fragment twice; 16 give a layer of a few thousand positions twice the workgroups, whose
// wavefronts then share the positions and split the pieces.  Wide images take 64 positions and eight wavefronts, which halves the reads of the
// weights, two thirds of the cache's work ([8, 256 -> 256, 100 x 152] fp16 298 -> 274 us, with LP = 8 299 -> 245; fp32, batch 4,
// 715 -> 648); the rule is at the launch.  (128 positions of sixteen wavefronts: 292 us, one workgroup per compute unit waits at
// its barriers; volumes, whose eight corners leave too few registers, fp16 [128 -> 256, 16 x 16 x 90] 127 us with 32 positions and 139 with 64.)
// What bounds it: the look-ups of the corners and weights in the vector caches, narrow layers the blend too (a multiply-add per channel and
// corner); small layers the latency of the chain load - blend - product.
//   (Images fp16 [8, 256 -> 256, 100 x 152]: 566 us with 16 positions per wavefront and the weights through LDS;
//   bf16 [4, 256 -> 64, 121 x 21] stride 2: 83 us, 21 us now; bf16 [1, 128 -> 32, 6 x 22 x 34]: 100 us, 30 us now.)
#include "dcn_mfma.hpp"
#include <algorithm>

namespace mv {

// ---- layouts: x [B, C, P] -> xt [B, P, C] and the weight fragments, one launch --------------------------------------
// weight [Cout, cpg, K] -> [group][16-row block][K step][lane][piece]: lane l holds row l % 16 and flat piece 4 * step + l / 16
// (tap piece / (cpg / PC), channels piece % (cpg / PC)); pieces beyond the last one are zeros
template <typename U>
__device__ __forceinline__ void dcn_flat_fragments_block(const U *__restrict__ wt, U *__restrict__ wf, const DcnDims &s, const long id) {
  constexpr int PC = 16 / sizeof(U);
  const int per_tap = s.cpg / PC, steps = (s.K * per_tap + 3) / 4, blocks = s.opg / 16;
  if (id >= static_cast<long>(s.groups) * blocks * steps * 64) return;
  const int lane = id % 64;
  long r = id / 64;
  const int st = r % steps; r /= steps;
  const int mb = r % blocks, g = static_cast<int>(r / blocks);
  const int piece = st * 4 + lane / 16, k = piece / per_tap, c = piece % per_tap * PC;
  const U *src = wt + (static_cast<long>(g * s.opg + mb * 16 + lane % 16) * s.cpg + c) * s.K + k;
  U out[PC];
#pragma unroll
  for (int i = 0; i < PC; i++) out[i] = k < s.K ? src[static_cast<long>(i) * s.K] : U(0);
  u32x4 packed;
  __builtin_memcpy(&packed, out, 16);
  *reinterpret_cast<u32x4 *>(wf + id * PC) = packed;
}

// the first of the two alone, for callers outside this file: elements of 2 or 4 bytes, channels in whole 16 bytes
template <typename U>
__global__ __launch_bounds__(256) void channels_last_kernel(const U *__restrict__ x, U *__restrict__ xt, const int C, const long P) {
  dcn_move_block<U>(x, xt, C, C, C, C, P, blockIdx.x, blockIdx.y, blockIdx.z);
}
int channels_last(const void *x, void *xt, int B, int C, long P, int elem_bytes, hipStream_t stream) {
  const long blocks = (P + kMovePos - 1) / kMovePos;
  const int ch = 128 / elem_bytes;
  MV_REQUIRE(blocks < (1L << 31) && B <= 65535 && (C + ch - 1) / ch <= 65535, "volume too large");
  const dim3 grid(static_cast<unsigned>(blocks), B, (C + ch - 1) / ch);
  if (elem_bytes == 2)
    hipLaunchKernelGGL((channels_last_kernel<unsigned short>), grid, dim3(256), 0, stream, static_cast<const unsigned short *>(x), static_cast<unsigned short *>(xt), C, P);
  else
    hipLaunchKernelGGL((channels_last_kernel<unsigned int>), grid, dim3(256), 0, stream, static_cast<const unsigned int *>(x), static_cast<unsigned int *>(xt), C, P);
  return check_launch("channels_last_kernel");
}

template <typename U>
__global__ __launch_bounds__(256) void dcn_columns_layout_kernel(const U *__restrict__ x, U *__restrict__ xt,
                                                                 const U *__restrict__ wt, U *__restrict__ wf, const DcnDims s,
                                                                 const unsigned pblocks, const unsigned moves) {
  if (blockIdx.x < moves) {
    const unsigned bx = blockIdx.x % pblocks, r = blockIdx.x / pblocks;
    dcn_move_block<U>(x, xt, s.Cin, s.Cin, s.Cin, s.Cin, s.P, bx, static_cast<int>(r % s.B), static_cast<int>(r / s.B));
  } else {
    dcn_flat_fragments_block<U>(wt, wf, s, (blockIdx.x - moves) * 256L + threadIdx.x);
  }
}

// ---- the layer ---------------------------------------------------------------------------------------------------------
constexpr int kColPieces = 16;   // pieces of a product: four K steps

template <typename T, int NC, int PT, int OBW, int W, int LP>
__global__ __launch_bounds__(kWave * W, W == 8 ? 4 : OBW == 4 && (PT == 32 || NC == 8) ? 2 : (OBW == 1 ? 4 : 3)) void dcn_forward_columns_kernel(
    const T *__restrict__ xt, const T *__restrict__ off, const T *__restrict__ mask, const T *__restrict__ wf,
    const T *__restrict__ bias, T *__restrict__ y, const DcnDims s) {
  using M = Mfma<T>;
  using P = typename std::conditional<(sizeof(T) == 2), float, double>::type;  // position type
  constexpr int PC = M::kPiece, ES = sizeof(T), PG = PT / 16, TG = kWave * W / PT;   // position groups; units of a window
  constexpr int PIECES = kColPieces, KS = PIECES / 4;
  constexpr int ITEMS = KS * PG / W;                                           // items of a wavefront per product
  constexpr unsigned kOutside = 0x80000000u;                                   // beyond the buffer: such loads return zeros
  constexpr int RW = 2 * NC + 4, PITCH = PT + (LP == 8 ? 1 : 4);   // (records 4 dwords further apart than they are long, a position's pieces: banks)
  constexpr int LG = PT * LP / kWave, LS = W / LG;   // items side by side on the positions; groups of LP pieces a wavefront is on at a time
  static_assert(LG * LS == W && ITEMS * W * kWave == PT * kColPieces && kColPieces % (LS * LP) == 0, "items of a product are shared out evenly");
  __shared__ __attribute__((aligned(16))) unsigned rec[TG * PT][RW];           // [unit][position]: at[NC], mask * w[NC]
  __shared__ u32x4 col[2][PIECES * PITCH];                                 // [piece][position]
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int j = lane % 16, kc = lane / 16;   // matrix layout
  const int lj = lane / LP, lk = lane % LP;  // load layout
  const int row_chunks = (s.opg + 16 * W * OBW - 1) / (16 * W * OBW);
  const int g = blockIdx.y / row_chunks, row0 = blockIdx.y % row_chunks * (16 * W * OBW), b = blockIdx.z;
  // (an XCD takes a contiguous eighth of the positions: its L2 then holds an eighth of the input and the offsets' reach)
  const long q0 = static_cast<long>(xcd_contiguous(blockIdx.x, gridDim.x)) * PT;
  const int dgn = s.cpd < s.cpg ? s.cpg / s.cpd : 1, dg0 = g * s.cpg / s.cpd;
  const int units = s.K * dgn, up = (dgn == 1 ? s.cpg : s.cpd) / PC;   // pieces per unit
  const int total = units * up, steps_all = (total + 3) / 4;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(xt + static_cast<long>(b) * s.P * s.Cin), 0, static_cast<int>(s.P * s.Cin * ES), 0x00020000);

  // ---- records ------------------------------------------------------------------------------------------------------
  const int ru = tid / PT, rp = tid % PT;   // this thread's unit of a window and position
  const long rq = min(q0 + rp, s.Q - 1);
  const bool rlive = q0 + rp < s.Q;
  int base_d, base_h, base_w;
  {
    const int qi = static_cast<int>(rq), ow = qi % s.Wo, t = qi / s.Wo, oh = t % s.Ho, od = t / s.Ho;
    base_d = od * s.sd - s.pd; base_h = oh * s.sh - s.ph; base_w = ow * s.sw - s.pw;
  }
  P fd = P(0), fh = P(0), fw = P(0);
  float fm = 1.f;
  auto request = [&](int first) {
    const int u = min(first + ru, units - 1), k = u / dgn;
    const long bg = static_cast<long>(b) * s.dg + dg0 + u - k * dgn;
    dcn_offsets(s, off + (bg * s.K + k) * s.nd * s.Q + rq, fd, fh, fw);
    if (mask) fm = load(mask + (bg * s.K + k) * s.Q + rq);
  };
  auto publish = [&](int first) {
    const int u = first + ru, k = u / dgn;
    const int ti = k / (s.kh * s.kw), tj = (k / s.kw) % s.kh, tk = k % s.kw;
    P pd = fd + static_cast<P>(base_d + ti * s.dd);
    const P ph = fh + static_cast<P>(base_h + tj * s.dh), pw = fw + static_cast<P>(base_w + tk * s.dw);
    if (NC == 4) pd = P(0);   // images: the only slice
    CornerTaps t;
    corner_taps<P>(s, pd, ph, pw, rlive && u < units, static_cast<unsigned>(s.Cin) * ES, 0u, kOutside, t);
    unsigned *r = rec[tid];
#pragma unroll
    for (int c = 0; c < NC; c += 4) {
      *reinterpret_cast<u32x4 *>(r + c) = u32x4{t.at[c], t.at[c + 1], t.at[c + 2], t.at[c + 3]};
      *reinterpret_cast<float4 *>(r + NC + c) = make_float4(fm * t.w[c], fm * t.w[c + 1], fm * t.w[c + 2], fm * t.w[c + 3]);
    }
  };

  // ---- samples: item i of a product: slot = wave + W i, positions 64 / LP * (slot % LG), group slot / LG of LP pieces of the
  // product; a wavefront's items form one sequence over the window, LS groups apart -----------------------------------
  const int p = wave % LG * (kWave / LP) + lj;   // (slot % LG is the same for all of them)
  const bool whole = LP == 8 || up % 4 == 0;     // a group of pieces belongs to one unit
  const int per_unit = up / LP;              // (`whole`)
  // (division by the pieces of a unit: the high half of a product, exact while piece * up < 2^32)
  const unsigned magic = up == 1 ? 0u : 0xffffffffu / static_cast<unsigned>(up) + 1u;
  u32x4 raw[NC];
  const unsigned *rnow = nullptr;            // the record of the item on its way
  int nu = 0, nr = 0;                        // the next item: unit of the window and group of it (`whole`), or group of the window
  auto gather = [&](int window, int limit) {
    unsigned add;
    int scalar_add = g * s.cpg * ES;
    if (whole) {
      const int u = min(nu, min(TG, units - window) - 1);   // (past the last one: loaded for nothing)
      rnow = rec[u * PT + p];
      add = static_cast<unsigned>(lk) * 16u;
      scalar_add += nr * (16 * LP);
      if (dgn > 1) scalar_add += (window + u) % dgn * (s.cpd * ES);
      nr += LS;
      while (nr >= per_unit) { nr -= per_unit; nu++; }
    } else {
      const int piece = min(nr * 4 + lk, limit - 1);
      const int u = up == 1 ? piece : static_cast<int>(__umulhi(static_cast<unsigned>(piece), magic)), r = piece - u * up;
      rnow = rec[u * PT + p];
      add = static_cast<unsigned>((dgn == 1 ? r * PC : (window + u) % dgn * s.cpd + r * PC) * ES);
      nr += LS;
    }
#pragma unroll
    for (int c = 0; c < NC; c += 4) {
      const u32x4 a = *reinterpret_cast<const u32x4 *>(rnow + c);
#pragma unroll
      for (int t = 0; t < 4; t++) raw[c + t] = __builtin_amdgcn_raw_buffer_load_b128(xr, a[t] + add, scalar_add, 0);
    }
  };
  // `left`: pieces of the window from this product's first one on
  auto blend = [&](int left, int i, u32x4 *to) {
    const int piece = (wave / LG + i * LS) * LP + lk;
    float v[PC];
#pragma unroll
    for (int e = 0; e < PC; e++) v[e] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; c += 4) {
      const float4 w = *reinterpret_cast<const float4 *>(rnow + NC + c);
      M::fma_piece(v, w.x, raw[c]); M::fma_piece(v, w.y, raw[c + 1]);
      M::fma_piece(v, w.z, raw[c + 2]); M::fma_piece(v, w.w, raw[c + 3]);
    }
    // (pieces beyond the last one meet weights that are zero, or the next window's: they must be zero themselves)
    to[piece * PITCH + p] = piece < left ? M::pack(v) : u32x4{0u, 0u, 0u, 0u};
  };

  float4_t acc[OBW][PG];
#pragma unroll
  for (int o = 0; o < OBW; o++)
#pragma unroll
    for (int n = 0; n < PG; n++) acc[o][n] = float4_t{0.f, 0.f, 0.f, 0.f};
  const int blocks = s.opg / 16;
  const T *wsrc[OBW];
#pragma unroll
  for (int o = 0; o < OBW; o++)   // (blocks beyond the last one repeat it; their products are not used)
    wsrc[o] = wf + (static_cast<long>(g) * blocks + min(row0 / 16 + o * W + wave, blocks - 1)) * steps_all * (64 * PC) + lane * PC;

  request(0);
  int buf = 0;
  for (int window = 0; window < units; window += TG) {
    __syncthreads();   // the records have been read
    publish(window);
    if (window + TG < units) request(window + TG);
    __syncthreads();
    const int limit = min(TG, units - window) * up, step0 = window * up / 4;   // (TG is a multiple of four)
    nu = 0;
    nr = wave / LG;
    if (whole) while (nr >= per_unit) { nr -= per_unit; nu++; }
    gather(window, limit);
    for (int first = 0; first < limit; first += PIECES) {
      u32x4 a[OBW][KS];
#pragma unroll
      for (int st = 0; st < KS; st++) {
        const int step = min(step0 + first / 4 + st, steps_all - 1);
#pragma unroll
        for (int o = 0; o < OBW; o++) a[o][st] = *reinterpret_cast<const u32x4 *>(wsrc[o] + static_cast<long>(step) * (64 * PC));
      }
#pragma unroll
      for (int i = 0; i < ITEMS; i++) {
        blend(limit - first, i, col[buf]);
        if (i + 1 < ITEMS || first + PIECES < limit) gather(window, limit);
      }
      __syncthreads();   // the pieces are complete (and the other buffer has been read)
#pragma unroll
      for (int st = 0; st < KS; st++)
#pragma unroll
        for (int n = 0; n < PG; n++) {
          const u32x4 bf = col[buf][(st * 4 + kc) * PITCH + n * 16 + j];
#pragma unroll
          for (int o = 0; o < OBW; o++) acc[o][n] = M::run16(a[o][st], bf, acc[o][n]);
        }
      buf ^= 1;
    }
  }
  // accumulator register r of lane l: output channel 4 * (l / 16) + r of its block, position l % 16 of its group
#pragma unroll
  for (int o = 0; o < OBW; o++) {
    const int row = row0 + (o * W + wave) * 16 + 4 * kc;
    if (row >= s.opg) continue;
    float bv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) bv[r] = bias ? load(bias + g * s.opg + row + r) : 0.f;
#pragma unroll
    for (int n = 0; n < PG; n++) {
      const long q = q0 + n * 16 + j;
      if (q < s.Q) {
#pragma unroll
        for (int r = 0; r < 4; r++)
          y[(static_cast<long>(b) * s.Cout + g * s.opg + row + r) * s.Q + q] = store_cast<T>(acc[o][n][r] + bv[r]);
      }
    }
  }
}

// dcn3d_mfma.hip: large volumes with few channels; -1: not for this layer
int dcn_shared_taps_forward(const void *xt, const void *off, const void *mask, const void *wf, const void *bias, void *y,
                            const DcnDims &s, int dtype, hipStream_t stream);

static size_t columns_align(size_t v) { return (v + 255) / 256 * 256; }
static long columns_steps(const DcnDims &s, int pc) { return (static_cast<long>(s.K) * (s.cpg / pc) + 3) / 4; }

bool dcn_columns_supported(const DcnDims &s, int dtype) {
  if (dtype != MV_F16 && dtype != MV_BF16 && dtype != MV_F32) return false;
  const int es = dtype == MV_F32 ? 4 : 2, pc = 16 / es;
  if (s.cpg % pc || s.cpd % pc || s.opg % 16 || (s.cpd < s.cpg && s.cpg % s.cpd) || (s.cpd > s.cpg && s.cpd % s.cpg)) return false;
  if (s.B > 65535 || s.Q >= (1L << 31) || s.K > 65536) return false;
  // 32-bit byte offsets into a sample; pieces of a window below 2^16
  return static_cast<long>(s.P) * s.Cin * es < (1L << 31) && 16L * (s.cpg / pc) < 65536 && static_cast<long>(s.K) * s.cpg < (1L << 30);
}

size_t dcn_columns_workspace_bytes(const DcnDims &s, int dtype) {
  const size_t es = dtype == MV_F32 ? 4 : 2;
  return columns_align(static_cast<size_t>(s.B) * s.P * s.Cin * es) +
         columns_align(static_cast<size_t>(s.Cout / 16) * columns_steps(s, static_cast<int>(16 / es)) * 1024);
}

// images (the kernels with four corners)
static bool columns_image(const DcnDims &s) { return s.nd == 2 && s.D == 1 && s.kd == 1 && s.pd == 0; }

// What a workgroup takes: `positions` of an image or volume, `waves` wavefronts of `blocks` blocks of 16 output channels each; the grid is
// tiles x chunks x samples.
struct ColumnsPlan {
  int positions, waves, blocks;
  long tiles, chunks;
};

void dcn_columns_plan(const DcnDims &s, int dtype, ColumnsPlan &plan) {
  // Positions per workgroup: 32 as long as that gives every compute unit two workgroups, otherwise 16; then fewer output
  // channels per workgroup (each share repeats the samples) until there is one for every compute unit.
  int pt = 32, obw = s.opg <= 64 ? 1 : (s.opg <= 128 ? 2 : 4);
  auto groups_of = [&](int p, int o) { return (s.Q + p - 1) / p * s.B * s.groups * ((s.opg + 64 * o - 1) / (64 * o)); };
  if (groups_of(pt, obw) < 512) pt = 16;
  while (obw > 1 && groups_of(pt, obw) < 256) obw /= 2;
  // Wide images: 64 positions and eight wavefronts per workgroup, as long as enough of them remain.  Their time goes in steps of 256
  // workgroups: fp16 [256 -> 256, 64 x n] 44 against 40 us with n = 128, 46 and 51 with 160, 49 and 65 with 224, 66 and 64 with 300, 68 and 88 with 450,
  // 100 and 119 with 700; fp32, bound by its products too, 326 and 277 us with 350, 330 and 367 with 450, 489 and 452 with 520, 494 and 537 with 700.
  // Not where their last tile holds much that does not exist (small images in large batches: fp16 [200, 256 -> 256] of 7 x 7 43 us and 65 with 32,
  // 10 x 10 64 and 87; of 5 x 5, as long as 7 x 7 there, 36 with 32, 4 x 4 24).
  const long positions64 = (s.Q + 63) / 64 * 64, positions32 = (s.Q + 31) / 32 * 32;
  const bool wide = columns_image(s) && s.opg > 128 && groups_of(64, 4) >= (dtype == MV_F32 ? 640 : 160) && positions64 * 8 <= positions32 * 9;
  plan.positions = wide ? 64 : pt;
  plan.waves = wide ? 8 : 4;
  plan.blocks = wide ? 2 : obw;
  const int rows = 16 * plan.waves * plan.blocks;   // (as the kernel has it: its groups and chunks are numbered by them)
  plan.tiles = (s.Q + plan.positions - 1) / plan.positions;
  plan.chunks = s.groups * static_cast<long>((s.opg + rows - 1) / rows);
}

template <typename T, int NC>
static int columns_run(const void *x, const void *off, const void *mask, const void *wt, const void *bias, void *y,
                       const DcnDims &s, void *workspace, hipStream_t stream) {
  using U = typename std::conditional<(sizeof(T) == 2), unsigned short, unsigned int>::type;
  T *xt = static_cast<T *>(workspace);
  T *wf = reinterpret_cast<T *>(static_cast<char *>(workspace) + columns_align(static_cast<size_t>(s.B) * s.P * s.Cin * sizeof(T)));
  const int ch = 128 / static_cast<int>(sizeof(T));
  const long pblocks = (s.P + kMovePos - 1) / kMovePos, moves = pblocks * s.B * ((s.Cin + ch - 1) / ch);
  const long frags = (static_cast<long>(s.Cout / 16) * columns_steps(s, 16 / static_cast<int>(sizeof(T))) * 64 + 255) / 256;
  MV_REQUIRE(moves + frags < (1L << 31), "volume too large");
  hipLaunchKernelGGL((dcn_columns_layout_kernel<U>), dim3(static_cast<unsigned>(moves + frags)), dim3(256), 0, stream,
                     static_cast<const U *>(x), reinterpret_cast<U *>(xt), static_cast<const U *>(wt), reinterpret_cast<U *>(wf), s,
                     static_cast<unsigned>(pblocks), static_cast<unsigned>(moves));
  int st = check_launch("dcn_columns_layout_kernel");
  if (st) return st;
  if constexpr (sizeof(T) == 2 && NC == 8) {
    st = dcn_shared_taps_forward(xt, off, mask, wf, bias, y, s, sizeof(T) == 2 && std::is_same<T, __half>::value ? MV_F16 : MV_BF16, stream);
    if (st >= 0) return st;
  }
  ColumnsPlan plan;
  dcn_columns_plan(s, sizeof(T) == 2 ? MV_F16 : MV_F32, plan);
  MV_REQUIRE(plan.tiles < (1L << 31) && plan.chunks <= 65535, "grid too large");
  const dim3 grid(static_cast<unsigned>(plan.tiles), static_cast<unsigned>(plan.chunks), s.B);
  // 16-byte pieces of a corner that a load takes from each position: eight, whole 128-byte lines, where a unit's channels allow it.
  const bool eights = std::min(s.cpd, s.cpg) % (8 * Mfma<T>::kPiece) == 0;
#define MV_COLUMNS_LP(PTV, OBWV, WV, LPV)                                                                              \
  hipLaunchKernelGGL((dcn_forward_columns_kernel<T, NC, PTV, OBWV, WV, LPV>), grid, dim3(kWave * WV), 0, stream, xt,     \
                     static_cast<const T *>(off), static_cast<const T *>(mask), wf, static_cast<const T *>(bias), static_cast<T *>(y), s)
#define MV_COLUMNS(PTV, OBWV, WV)                                                                                      \
  if (plan.positions == PTV && plan.blocks == OBWV && plan.waves == WV) {                                              \
    if (eights) MV_COLUMNS_LP(PTV, OBWV, WV, 8);                                                                       \
    else MV_COLUMNS_LP(PTV, OBWV, WV, 4);                                                                              \
    return check_launch("dcn_forward_columns_kernel");                                                                 \
  }
  if constexpr (NC == 4) { MV_COLUMNS(64, 2, 8) }
  MV_COLUMNS(32, 1, 4)
  MV_COLUMNS(32, 2, 4)
  MV_COLUMNS(32, 4, 4)
  MV_COLUMNS(16, 1, 4)
  MV_COLUMNS(16, 2, 4)
  MV_COLUMNS(16, 4, 4)
#undef MV_COLUMNS
#undef MV_COLUMNS_LP
  return fail(MV_INVALID_ARGUMENT, "no kernel for this plan");
}

int dcn_columns_forward(const void *x, const void *off, const void *mask, const void *wt, const void *bias, void *y,
                        const DcnDims &s, int dtype, void *workspace, hipStream_t stream) {
  const bool image = columns_image(s);
#define MV_COLUMNS_AS(T) \
  (image ? columns_run<T, 4>(x, off, mask, wt, bias, y, s, workspace, stream) : columns_run<T, 8>(x, off, mask, wt, bias, y, s, workspace, stream))
  if (dtype == MV_F16) return MV_COLUMNS_AS(__half);
  if (dtype == MV_F32) return MV_COLUMNS_AS(float);
  return MV_COLUMNS_AS(__hip_bfloat16);
#undef MV_COLUMNS_AS
}

}  // namespace mv
