// RoIAlign BACKWARD of plain boxes with few cells per axis (fp16 detection heads on volumes) by the voxels' owners: no global
// atomics, no fp32 copy of the gradient to clear and to fold.  Same results as the reference's one-thread-per-output kernel
// with eight atomicAdd per sample (csrc/cuda/roi_align_3d_cuda_kernel.cuh:90-202).
//
// A box's samples are separable, so a roi's share of the gradient is
//     grad[z, y, x][c] += sum_pd Wz[z][pd] P[c, pd][y, x],   P[c, pd][y, x] = sum_(ph, pw) gout[c][pd][ph][pw] Wy[y][ph] Wx[x][pw]
// with a short matrix per axis (up to 8 cells).  A wavefront owns a brick of 8 x 8 x 8 voxels and 16 channels: their sums are
// accumulators.  It takes the rois that touch the brick one after the other.  Both sums are products on the matrix cores, for two
// channels and 16 voxels (two rows of the brick) at a time:
//   * P: rows (channel, pd), K = (ph, pw) with cells padded to rows of eight, so that a lane's 16-byte piece of the left operand is
//     one row of cells as it lies in grad_output, and its piece of the right one a row of Wx times one number of Wy, formed in
//     registers from the roi's tables, which a small launch before has left in memory.
//   * over pd: rows (channel', z), K = (channel, pd), block-diagonal in the channel with Wz in the blocks: the accumulator of the
//     first product is the right operand of the second as it stands.
// The gradient of a roi's 16 channels is one run of memory of 10 KB or so.  It comes to LDS as it lies there (loads of its rows of
// cells straight into registers, 16 bytes of 64 different cache lines each, kept the texture addressers 85 % busy: 800 us for
// 4000 rois x 256 channels x 7^3), the next roi's while the present one's products run.  The order of the sums is the order of the rois.
//
// Two small launches before: the rois' tables, and the bricks' lists of rois.  The two wavefronts of a workgroup have neighbouring
// bricks along x: rows of the gradient are written 32 bytes at a time (16 bytes of a single brick are 547 MB for a gradient of 226;
// four bricks, 64 bytes, wait for the longest of four lists).
#include "common.hpp"
#include "roi_geometry.hpp"
#include "sampling.hpp"
#include "dcn_mfma.hpp"

#include <algorithm>

namespace mv {

bool roi_pool_applies(int dtype, const RoiProblem &p);   // roi_pool.hip

constexpr int kBrickThreads = 256, kBrickWaves = kBrickThreads / kWave;
constexpr int kBrickCells = 8, kBrickChannels = 16;
constexpr int kBrickTried = 4;                 // records that a thread fetches together
constexpr int kBrickEdge = 8;                  // voxels of a brick along each axis
constexpr int kBrickPad = 128;                 // bytes behind the copy of the last roi's gradient

// What the tables kernel leaves about a roi: first and last voxel of its box per axis (low and high half; first > last: the roi
// touches nothing; bit 15: more samples than a wavefront has lanes) and the image.  Its tables are rows of eight fp32 weights, one per voxel along x, then y, then z, the axes
// padded to whole bricks; only the rows of the bricks that the box touches are written.  A row of y holds cell c at
// c % 4 * 2 + c / 4, the two cells of a lane side by side; where there is no cell c + 4, cell c stands there too.
struct BrickRoi { unsigned span[3]; int image; };
constexpr unsigned kBrickMany = 0x8000u;

__host__ __device__ inline int brick_up(int n) { return (n + kBrickEdge - 1) / kBrickEdge * kBrickEdge; }
__host__ __device__ inline int brick_rows(const RoiProblem &p) { return brick_up(p.W) + brick_up(p.H) + brick_up(p.D); }
// where the rows of y and z start
__device__ __forceinline__ int brick_row_y(const RoiProblem &p) { return brick_up(p.W); }
__device__ __forceinline__ int brick_row_z(const RoiProblem &p) { return brick_up(p.W) + brick_up(p.H); }

// One workgroup per roi, a wavefront per axis; further ones copy the last roi's gradient to a place with room behind it (a row of
// cells is read as 16 bytes, more than it may have behind it at the end of a tensor).
__global__ __launch_bounds__(3 * kWave) void roi_brick_tables_kernel(const float *__restrict__ rois, BrickRoi *__restrict__ recs,
                                                                     float *__restrict__ tables, const RoiProblem p,
                                                                     const __half *__restrict__ last, __half *__restrict__ copy, const int slab) {
  if (blockIdx.x >= static_cast<unsigned>(p.R)) {
    const int at = ((blockIdx.x - p.R) * 3 * kWave + threadIdx.x) * 8, end = slab + kBrickPad / 2;
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (at + i < end) copy[at + i] = at + i < slab ? last[at + i] : store_cast<__half>(0.f);
    return;
  }
  const int n = blockIdx.x, a = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const float *roi = rois + static_cast<long>(n) * roi_columns(3, 0);
  const int image = static_cast<int>(roi[0]), nc = a == 0 ? p.ow : a == 1 ? p.oh : p.od, sz = a == 0 ? p.W : a == 1 ? p.H : p.D;
  const bool empty = image < 0 || image >= p.N;
  // (the expressions of build_geom; an extent of at least 1 has a grid of at least 1)
  const double start = static_cast<double>(roi[1 + a]) * p.scale, ext = fmax(static_cast<double>(roi[4 + a]) * p.scale - start, 1.0);
  const int grid = p.sampling_ratio > 0 ? p.sampling_ratio : static_cast<int>(ceil(ext / static_cast<double>(nc)));
  const double bin = ext / static_cast<double>(nc), step = bin / static_cast<double>(grid), per = 1.0 / step;
  auto tap = [&](int cell, int sub, int &lo, int &hi, float &frac) {   // (local_coord's expression)
    const double v = start + cell * bin + static_cast<double>(static_cast<float>(sub) + .5f) * step;
    return clamped_tap<float>(v, sz, lo, hi, frac, p.order);
  };
  // Positions grow with the sample, so the box runs from the first valid sample to the last: both are among the 64 from, and up to,
  // the ones that this estimate gives (fmin and fmax make 0 and the last of a position that is not a number).
  int first = 0x7fff, last_voxel = -1;
  if (!empty) {
    const long entries = static_cast<long>(nc) * grid;
    const double top = static_cast<double>(entries - 1);
    const long e0 = static_cast<long>(fmin(fmax(floor((-1.0 - start) * per - 0.5) - 2.0, 0.0), top));
    const long e1 = static_cast<long>(fmax(fmin(ceil((sz - start) * per - 0.5) + 2.0, top), 0.0));
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const long e = i == 0 ? min(e0 + lane, entries - 1) : max(e1 - lane, 0L);
      int lo, hi;
      float frac;
      int cell = 0;
      long sub = e;
      while (sub >= grid && cell + 1 < nc) { sub -= grid; cell++; }
      if (tap(cell, static_cast<int>(sub), lo, hi, frac)) {
        first = min(first, lo);
        last_voxel = max(last_voxel, hi);
      }
    }
  }
#pragma unroll
  for (int m = 1; m < kWave; m *= 2) {
    first = min(first, __shfl_xor(first, m));
    last_voxel = max(last_voxel, __shfl_xor(last_voxel, m));
  }
  if (lane == 0) {
    const bool many = static_cast<long>(nc) * grid > kWave;
    recs[n].span[a] = static_cast<unsigned>(first) | (many ? kBrickMany : 0u) | static_cast<unsigned>(max(last_voxel, 0)) << 16;
    if (a == 0) recs[n].image = image;
  }
  const int cell = a == 1 && lane % kBrickCells >= max(nc, 4) ? lane % kBrickCells - 4 : lane % kBrickCells;
  const float inv = 1.f / static_cast<float>(grid);
  float *rows = tables + (static_cast<long>(n) * brick_rows(p) + (a == 0 ? 0 : a == 1 ? brick_row_y(p) : brick_row_z(p))) * kBrickCells;
  for (int r0 = first / kBrickEdge * kBrickEdge; r0 <= last_voxel; r0 += kWave / kBrickCells) {
    const int row = r0 + lane / kBrickCells;
    float w = 0.f;
    if (cell < nc && row >= first && row <= last_voxel) {
      // the cell's samples that can reach the row, a few more on either side
      const double from = start + cell * bin, below = row == 0 ? -1.0 : row - 1.0, above = row >= sz - 2 ? sz : row + 1.0;
      const int s0 = static_cast<int>(fmin(fmax(floor((below - from) * per - 0.5) - 2.0, 0.0), static_cast<double>(grid - 1)));
      const int s1 = static_cast<int>(fmax(fmin(ceil((above - from) * per - 0.5) + 2.0, static_cast<double>(grid - 1)), 0.0));
      for (int s = s0; s <= s1; s++) {
        int lo, hi;
        float frac;
        if (!tap(cell, s, lo, hi, frac)) continue;
        if (lo == row) w += (1.f - frac) * inv;
        if (hi == row) w += frac * inv;
      }
    }
    rows[row * kBrickCells + (a == 1 ? lane % 4 * 2 + lane / 4 % 2 : cell)] = w;
  }
}

// The rois that touch a brick, in their order: a workgroup per brick.  An entry is the roi's number, with a bit for the upper
// four rows of the brick, one for the lower four, and one for the form with all bits (see brick_exact).
constexpr unsigned kBrickUpper = 1u << 30, kBrickLower = 1u << 31, kBrickExact = 1u << 29, kBrickNumber = kBrickExact - 1;

// Whether a roi's gradient has all bits of its weights: those that the kernel which adds box by box works out in fp32, not as products of 16-bit
// numbers (a slice that does not fit its operand, boxes or samples beyond its tables, and what its loads would reach past the tensor's end).
__device__ __forceinline__ bool brick_exact(const unsigned (&span)[3]) {
  int extent[3];
  bool many = false;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    extent[a] = static_cast<int>(span[a] >> 16) - static_cast<int>(span[a] & 0x7fffu) + 1;
    many = many || (span[a] & kBrickMany) || extent[a] > 32;
  }
  return many || extent[1] * ((extent[0] + 3) & ~3) > 224;
}

__global__ __launch_bounds__(kBrickThreads) void roi_brick_lists_kernel(const uint4 *__restrict__ recs, unsigned *__restrict__ lists,
                                                                        unsigned *__restrict__ lengths, const int R, const int nx,
                                                                        const int ny, const int nz) {
  __shared__ unsigned counts[2][kBrickTried * kBrickWaves];
  unsigned id = blockIdx.x;
  unsigned *const list = lists + static_cast<long>(id) * R;
  const int first[3] = {static_cast<int>(id % nx) * kBrickEdge, static_cast<int>(id / nx % ny) * kBrickEdge,
                        static_cast<int>(id / nx / ny % nz) * kBrickEdge};
  const int image = id / nx / ny / nz;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  unsigned have = 0;
  int turn = 0;
  for (int base = 0; base < R; base += kBrickTried * kBrickThreads, turn ^= 1) {
    uint4 rec[kBrickTried];
    unsigned long hits[kBrickTried];
#pragma unroll
    for (int i = 0; i < kBrickTried; i++) rec[i] = recs[min(base + i * kBrickThreads + static_cast<int>(threadIdx.x), R - 1)];
#pragma unroll
    for (int i = 0; i < kBrickTried; i++) {
      const int k = base + i * kBrickThreads + static_cast<int>(threadIdx.x);
      const unsigned span[3] = {rec[i].x, rec[i].y, rec[i].z};
      bool hit = k < R && static_cast<int>(rec[i].w) == image;
#pragma unroll
      for (int a = 0; a < 3; a++) {
        const int lo = static_cast<int>(span[a] & 0x7fffu) - first[a], hi = static_cast<int>(span[a] >> 16) - first[a];
        hit = hit && lo <= hi && lo < kBrickEdge && hi >= 0;
        if (a == 1) rec[i].x = static_cast<unsigned>(k) | (lo < kBrickEdge / 2 ? kBrickUpper : 0) | (hi >= kBrickEdge / 2 ? kBrickLower : 0);
      }
      if (brick_exact(span)) rec[i].x |= kBrickExact;
      hits[i] = __ballot(hit);
      if (lane == 0) counts[turn][i * kBrickWaves + wave] = __popcll(hits[i]);
    }
    __syncthreads();   // (the counts of a turn are read before this barrier of the next one, and written again behind it)
#pragma unroll
    for (int i = 0; i < kBrickTried; i++)
#pragma unroll
      for (int w = 0; w < kBrickWaves; w++) {
        if (w == wave && (hits[i] >> lane & 1)) list[have + __popcll(hits[i] & ((1UL << lane) - 1))] = rec[i].x;
        have += counts[turn][i * kBrickWaves + w];
      }
  }
  if (threadIdx.x == 0) lengths[id] = have;
}

// The operands of the products are fp16 numbers.  In the ordinary form the weights Wy Wx and the sums P are rounded to them once (11 bits) and Wz is
// two numbers side by side in K.  Where the first product's K has room, below eight rows of cells, rows stand in it twice, the second time with
// what the rounding left of their weights.  Wy Wx is scaled by kBrickWeight, so that P of small gradients is not a subnormal number of a few bits.
// In the form with all bits (22 of them) Wy Wx, P and Wz are all two numbers, what is left of a weight in products of its own.  It is for rois whose
// gradients the kernel that adds box by box works out in fp32 (brick_exact): P is kept four times as large and its rest 256 times, so that gradients
// of 1e-5 lose nothing.  Bricks whose sums overflow with that or in the ordinary form (|P| > 16376) have the form too: the first number of P is scaled
// down to 1 / 128 (64 cells of the type's largest fit), its rest up to 16.  Wz is scaled by what makes the products' sum the result.
// Error against 64 bits (2.07e-4 of it the result's own rounding) here and box by box, 200 rois of up to 12 voxels: four rows 2.93e-4 and 3.61e-4,
// seven 3.53e-4 and 3.62e-4, eight 3.59e-4 and 3.60e-4; 100 rois of 16 - 24 voxels: 2.07e-4 with all bits (3.5e-4 without) and 2.07e-4; gradients of
// 1e-5 2.24e-3 (own 2.15e-3) and 3.02e-3, on 100 rois of 16 - 24 voxels 8.27e-3 both, all of it the result's own (8.32e-3 with the scales for large sums).
// Backward pass of 4000 rois x 256 channels x 7^3: 500 us (box by box 795); with P as two numbers for all rois, so that no values need a second time,
// 555, and 1000 rois of 4^3 x 128 98 and 115 (box by box 151).  Gradients of 4000 throughout, where all bricks do: 1.6 ms.  100 rois of 16 - 24 voxels
// x 128 x 7^3: 220 us with all bits, 125 without, 403 box by box.
constexpr float kBrickWeight = 4.f;
// The form with all bits: factors of Wy Wx, of the first number of P from what these give, back to that, and of Wz for the two numbers
struct BrickScales {
  float weight, down, up, value, rest;
  __device__ __forceinline__ explicit BrickScales(const bool large)
      : weight(large ? 16.f : 256.f), down(large ? 1.f / 2048 : 1.f / 64), up(large ? 2048.f : 64.f), value(large ? 128.f : 1.f / 4),
        rest(large ? 1.f / 16 : 1.f / 256) {}
};
typedef _Float16 brick_half4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ brick_half4 brick_pack(const float (&w)[4]) {
  return __builtin_bit_cast(brick_half4, uint2{Mfma<__half>::pack2(w[0], w[1]), Mfma<__half>::pack2(w[2], w[3])});
}
__device__ __forceinline__ u32x4 brick_pair(const brick_half4 a, const brick_half4 b) {
  const uint2 x = __builtin_bit_cast(uint2, a), y = __builtin_bit_cast(uint2, b);
  return u32x4{x.x, x.y, y.x, y.y};
}
struct BrickLeft { brick_half4 value, rest; };
__device__ __forceinline__ BrickLeft brick_left(const float (&w)[4], const float scale) {
  const float v[4] = {w[0] * scale, w[1] * scale, w[2] * scale, w[3] * scale};
  BrickLeft l;
  l.value = brick_pack(v);
  float rest[4];
#pragma unroll
  for (int r = 0; r < 4; r++) rest[r] = v[r] - static_cast<float>(l.value[r]);
  l.rest = brick_pack(rest);
  return l;
}
__device__ __forceinline__ u32x4 brick_sums(const float4_t &part) {
  const float v[4] = {part[0], part[1], part[2], part[3]};
  const brick_half4 sums = brick_pack(v);
  return brick_pair(sums, sums);
}
__device__ __forceinline__ u32x4 brick_sums_exact(const float4_t &part, const BrickScales &scales) {
  const float v[4] = {part[0] * scales.down, part[1] * scales.down, part[2] * scales.down, part[3] * scales.down};
  brick_half4 high = brick_pack(v), rest;
  asm("" : "+v"(high));   // (or the compiler forms it a second time, element by element, for the rest)
#pragma unroll
  for (int r = 0; r < 4; r++) rest[r] = static_cast<_Float16>(__builtin_fmaf(static_cast<float>(high[r]), -scales.up, part[r]));
  return brick_pair(high, rest);
}

// Sums that do not come out finite are formed again, with all bits and in turns.  (A weight of zero times a gradient that is not finite is not a
// number, and it would reach every voxel of the brick.)  First the sums without such gradients, then what the positive infinities reach (1 stands
// for them), then what the negative ones do; a gradient that is not a number counts as both.  The turns' results add up, inf - inf = NaN.  (4000 rois
// x 256 channels x 7^3 with one infinity 500 us, all NaN 2.2 ms, infinities of both signs alone 3.4; term by term in fp32, without a product, one
// infinity took 17.7 ms.)
enum BrickTurn { kBrickAll, kBrickFinite, kBrickPlus, kBrickMinus };
constexpr unsigned kBrickHasPlus = 2, kBrickHasMinus = 4, kBrickHasNan = 8;   // what a brick's gradients have
struct BrickKinds { unsigned plus = 0, minus = 0, nan = 0, now = 0; };        // not 0: there are some (`now`: for the present turn)
// A word of two gradients in a turn
__device__ __forceinline__ unsigned brick_screen(const unsigned v, const int turn, BrickKinds &has) {
  const unsigned special = ((v & 0x7c007c00u) + 0x04000400u) & 0x80008000u;   // (a sign bit each, as all of these)
  const unsigned nan = special & ((v & 0x03ff03ffu) + 0x7fff7fffu), inf = special ^ nan;
  has.plus |= inf & ~v; has.minus |= inf & v; has.nan |= nan;
  const unsigned on = nan | (inf & (turn == kBrickPlus ? ~v : v));
  const unsigned now = turn == kBrickFinite ? v & ~(special | (special - (special >> 15))) : (on >> 1) - (on >> 5);   // (0x4000 - 0x0400: 1)
  has.now |= now & 0x7fff7fffu;
  return now;
}

// What a workgroup works on: 1 << LOG_WX bricks side by side, 16 channels of an image; `part` of `parts` workgroups that share them.
template <int LOG_WX>
struct BrickPlace {
  int X0, Y0, Z0, c_base, image, part;
  long brick;      // the first one's number, among those of all images
  int bricks;      // of them that there are
  bool none;
  __device__ __forceinline__ BrickPlace(const RoiProblem &p, const int nx, const int ny, const int nz, const int cblocks, const int parts,
                                        const unsigned total) {
    // eight runs of regions, one per die, neighbours one after the other: they read the same rois' gradients
    const unsigned run = (total + 7) / 8;
    unsigned id = (blockIdx.x % 8) * run + blockIdx.x / 8;
    none = blockIdx.x / 8 >= run || id >= total;
    part = id % parts; id /= parts;
    const int rx = id % nx; id /= nx;
    const int ry = id % ny; id /= ny;
    const int rz = id % nz; id /= nz;
    c_base = static_cast<int>(id % cblocks) * kBrickChannels;
    image = id / cblocks;
    X0 = rx * kBrickEdge << LOG_WX; Y0 = ry * kBrickEdge; Z0 = rz * kBrickEdge;
    const int along = (p.W + kBrickEdge - 1) / kBrickEdge;
    brick = ((static_cast<long>(image) * nz + rz) * ny + ry) * along + (rx << LOG_WX);
    bricks = min(1 << LOG_WX, along - (rx << LOG_WX));
  }
};

// whether all of a wavefront's sums are
__device__ __forceinline__ bool brick_finite(const float4_t (&acc)[kBrickChannels / 2][4]) {
  float check = 0.f;
#pragma unroll
  for (int i = 0; i < kBrickChannels / 2; i++)
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int r = 0; r < 4; r++) check = fmaf(acc[i][k][r], 0.f, check);
  return __ballot(!(check == 0.f)) == 0;
}

// The wavefronts' sums to the gradient.  acc[i][k], register r: channel 2 i + quad / 2, voxel z = quad % 2 * 4 + r, y = 2 k + col / 8,
// x = col % 8 of the brick.  Not `first`: `mark` where a sum is positive is added to what is there.
template <int LOG_WX>
__device__ __forceinline__ void brick_finish(const float4_t (&acc)[kBrickChannels / 2][4], const BrickPlace<LOG_WX> &at, __half *__restrict__ grad,
                                             const RoiProblem &p, unsigned char *const lds, const bool first, const float mark) {
  constexpr int wxn = 1 << LOG_WX, RX = kBrickEdge << LOG_WX, TZ = kBrickEdge;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));   // (nothing of this is formed before a brick's turns and kept)
  const int lane = tid % kWave, bx = tid / kWave * kBrickEdge, col = lane % 16, quad = lane / 16;
  // through LDS, so that rows of the region go out whole: [channel][z][y][x], a little room between channels against bank conflicts
  __half *const stage = reinterpret_cast<__half *>(lds);
  constexpr int channel = (TZ * 64 << LOG_WX) + 8;
#pragma unroll
  for (int i = 0; i < kBrickChannels / 2; i++)
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        stage[(2 * i + quad / 2) * channel + ((quad % 2 * 4 + r) * 8 + 2 * k + col / 8) * RX + bx + col % 8] =
            store_cast<__half>(first ? acc[i][k][r] : acc[i][k][r] > 0.f ? mark : 0.f);
  __syncthreads();
  constexpr int kPieces = kBrickChannels * wxn * TZ * 8;
#pragma unroll 4
  for (int i = tid; i < kPieces; i += kWave * wxn) {
    const int px = i & (wxn - 1), row = (i >> LOG_WX) & (TZ * 8 - 1), cl = (i >> LOG_WX) / (TZ * 8);
    const int y = at.Y0 + row % 8, z = at.Z0 + row / 8, x = at.X0 + px * 8;
    if (at.c_base + cl >= p.C || y >= p.H || z >= p.D || x >= p.W) continue;
    const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + cl * channel + row * RX + px * 8);
    __half *dst = grad + (((static_cast<long>(at.image) * p.C + at.c_base + cl) * p.D + z) * p.H + y) * p.W + x;
    if (first && x + 8 <= p.W) {   // one store: global memory takes any alignment
      typedef unsigned int V __attribute__((ext_vector_type(4), aligned(2)));
      *reinterpret_cast<V *>(dst) = v;
    } else {
      __half e[8];
      __builtin_memcpy(e, &v, sizeof(v));
#pragma unroll
      for (int k = 0; k < 8; k++)
        if (x + k < p.W) dst[k] = first ? e[k] : store_cast<__half>(load(dst + k) + load(&e[k]));
    }
  }
}

// the lane's number, worked out where it is used: kept, it would be one register too many.  (The instructions are the compiler's own: around
// inline assembly it leaves no wait for a matrix instruction that still reads or writes the register that the result gets.)
__device__ __forceinline__ int brick_lane() {
  unsigned none = 0;
  asm volatile("" : "+s"(none));
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, none));
}

// where part `k` of `parts` of a list begins
__device__ __forceinline__ int brick_share(const int length, const int k, const int parts) {
  return static_cast<int>(static_cast<long>(length) * k / parts);
}

template <int LOG_WX, bool SHARED>
__global__ __launch_bounds__(kWave << LOG_WX, 2) void roi_brick_backward_kernel(
    const __half *__restrict__ gout, const __half *__restrict__ last, const float *__restrict__ tables, const unsigned *__restrict__ lists,
    const unsigned *__restrict__ lengths, __half *__restrict__ grad, const RoiProblem p, const int nx, const int ny, const int nz,
    const int cblocks, const unsigned total, const int pieces, const int ring, const int parts, float4_t *__restrict__ partial) {
  using M = Mfma<__half>;
  // A ring of `ring` kilobytes and one more for each wavefront, for the rois' gradients, `pieces` of them each; at the end the sums.
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  __shared__ unsigned special;
  const BrickPlace<LOG_WX> place(p, nx, ny, nz, cblocks, SHARED ? parts : 1, total);
  if (place.none) return;
  const int X0 = place.X0, Y0 = place.Y0, Z0 = place.Z0, c_base = place.c_base;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int bx = wave * kBrickEdge;
  const int col = lane % 16, quad = lane / 16;
  const int cells = p.od * p.oh * p.ow, ohw = p.oh * p.ow;
  const long slab = static_cast<long>(p.C) * cells;
  const int rows = brick_rows(p);
  unsigned char *const ring_lds = lds + wave * (ring + 1) * 1024;
  // the lane's first row of cells (ph = quad) there, of channel col / 8 and plane col % 8 (beyond the last: any, its weights are 0),
  // in elements; the second is four rows on, or the same
  const int piece = col / 8 * cells + min(col % 8, p.od - 1) * ohw + quad * p.ow;

  const bool own_block = col / 8 == quad / 2;
  const bool twice = quad + 4 >= p.oh;   // the lane's second row is its first again
  const unsigned to_second = twice ? 0 : 8 * p.ow;

  if (threadIdx.x == 0) special = 0;
  __syncthreads();
  // the brick's list, or this part of it; a wavefront beyond the last column of bricks has none
  const long brick = place.brick + wave;
  int have = wave < place.bricks ? static_cast<int>(lengths[brick]) : 0, begin = 0;
  if (SHARED) {
    begin = brick_share(have, place.part, parts);
    have = brick_share(have, place.part + 1, parts) - begin;
  }
  const unsigned *const list = lists + brick * p.R + begin;
  // [two channels][two rows of voxels]: z = quad % 2 * 4 + r of channel quad / 2 at voxel (y = col / 8, x = col % 8)
  float4_t acc[kBrickChannels / 2][4];
  unsigned bits = 0;   // 1: the sums are not all finite; then what the gradients have
#pragma unroll 1
  for (int turn = kBrickAll;;) {
#pragma unroll
    for (int i = 0; i < kBrickChannels / 2; i++)
#pragma unroll
      for (int k = 0; k < 4; k++) acc[i][k] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (have > 0) {
      unsigned entries = list[min(brick_lane(), have - 1)];   // 64 at a time, one per lane
      auto entry = [&](const int i) {
        if (i % kWave == 0 && i > 0) {
          entries = list[min(i + brick_lane(), have - 1)];
          asm volatile("" : "+v"(entries));   // (a wait here and not where it is used, which would be one for all that is on its way)
        }
        return static_cast<unsigned>(__builtin_amdgcn_readlane(entries, i % kWave));
      };
      // what a lane needs of a roi's tables: its voxel's row of x, its rows' pairs of y, and four weights of z
      struct Weights { float4 x0, x1; float2 y[4]; float4 z; };
      auto fetch = [&](unsigned n, Weights &w) {
        // (its places there, in bytes)
        const unsigned at = brick_lane(), c = at % 16, q = at / 16;
        const unsigned at_x = (X0 + bx + c % 8) * (kBrickCells * 4), at_y = (brick_row_y(p) + Y0 + c / 8) * (kBrickCells * 4) + q * 8,
                       at_z = (brick_row_z(p) + Z0 + c % 8) * (kBrickCells * 4) + q % 2 * 16;
        const char *tab = reinterpret_cast<const char *>(tables + static_cast<long>(n) * rows * kBrickCells);
        const float4 *x = reinterpret_cast<const float4 *>(tab + at_x);
        w.x0 = x[0];
        w.x1 = x[1];
#pragma unroll
        for (int k = 0; k < 4; k++) w.y[k] = *reinterpret_cast<const float2 *>(tab + (at_y + 2 * k * kBrickCells * 4));
        w.z = *reinterpret_cast<const float4 *>(tab + at_z);
      };
      // A roi's gradient of the 16 channels is one run of memory.  It comes to LDS as it is, 1024 bytes a load, from the 4-byte
      // boundary before it; returns the elements between that and its start.
      // Pieces `from` to `to` of it go to the ring's places from `at` on; the piece that comes to the first place when others are
      // before it goes behind the last place too, so that what lies across the ring's end can be read in one.
      struct Run { u32x4 src; int odd; };
      auto run_of = [&](const unsigned of) {
        const bool end = of == static_cast<unsigned>(p.R) - 1u;
        const long from = (end ? 0L : of * slab) + static_cast<long>(c_base) * cells;   // in elements
        const unsigned char *const start = reinterpret_cast<const unsigned char *>((end ? last : gout) + from);
        const int odd = static_cast<int>(reinterpret_cast<unsigned long long>(start) & 2);
        const long behind = (end ? slab * 2 + kBrickPad : p.R * slab * 2) - from * 2 + odd;
        const unsigned long long base = reinterpret_cast<unsigned long long>(start - odd);
        return Run{u32x4{static_cast<unsigned>(base), static_cast<unsigned>(base >> 32) & 0xffffu,
                         static_cast<unsigned>(min(behind, 0x7ffffff0L)), 0x00020000u}, odd};
      };
      // (Written out: behind the compiler's own form every read of LDS waits for all the loads that are on their way to it.  The waits
      // that it places for other loads count these among them, so that they are longer than they need be, never shorter.)
      const unsigned ring_at = __builtin_amdgcn_readfirstlane(
          static_cast<unsigned>(reinterpret_cast<unsigned long long>((__attribute__((address_space(3))) unsigned char *)ring_lds)));
      auto to_lds = [&](const Run &run, const int at, const int place) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     : : "s"(__builtin_amdgcn_readfirstlane(ring_at + place * 1024)), "v"(at), "s"(run.src) : "memory");
      };
      auto bring = [&](const Run &run, int place, const int from, const int to) {
        int at = brick_lane() * 16 + from * 1024;
        // (m0 is the compiler's own: it cannot be named as changed, so it gets back what it had; and five waits before the loads, what they need
        // where the compiler has just fetched their scalars from vector registers)
        unsigned kept;
        asm volatile("s_mov_b32 %0, m0\n\ts_nop 4" : "=s"(kept) : "s"(run.src));
#pragma unroll 1
        for (int i = from; i < to; i++, at += 1024) {
          to_lds(run, at, place);
          if (place == 0 && i > 0) to_lds(run, at, ring);
          place = place + 1 == ring ? 0 : place + 1;
        }
        asm volatile("s_mov_b32 m0, %0" : : "s"(kept));
        return place;
      };
      const int early = min(ring - pieces, pieces);   // pieces that come in before the present roi has been read
      // Pairs of channels are read four ahead; behind the fourth of the last sweep the next roi's gradient may come in.
      u32x4 slot[4][2];
      auto read = [&](unsigned at, const unsigned end, u32x4 (&s)[2]) {   // (a roi begins before the end and is no longer than the ring)
        typedef unsigned int V __attribute__((ext_vector_type(4), aligned(4)));
        const unsigned char *const from = ring_lds + min(at, at - end);
        s[0] = *reinterpret_cast<const V *>(from);
        s[1] = *reinterpret_cast<const V *>(from + to_second);
      };
      // the present roi's gradient as a turn has it, in LDS; whether there is anything
      auto screen = [&](int place, const int turn) {
        BrickKinds has;
        unsigned char *const mine = ring_lds + brick_lane() * 16;
#pragma unroll 2
        for (int i = 0; i < pieces; i++) {
          u32x4 *const at = reinterpret_cast<u32x4 *>(mine + place * 1024);
          u32x4 v = *at;
#pragma unroll
          for (int j = 0; j < 4; j++) v[j] = brick_screen(v[j], turn, has);
          *at = v;
          if (place == 0 && i > 0) at[ring * 64] = v;
          place = place + 1 == ring ? 0 : place + 1;
        }
        const auto any = [](const unsigned word, const unsigned bit) { return __ballot(word != 0) != 0 ? bit : 0u; };
        bits |= any(has.plus, kBrickHasPlus) | any(has.minus, kBrickHasMinus) | any(has.nan, kBrickHasNan);
        return any(has.now, 1u) != 0;
      };
      Weights w;
      unsigned e = entry(0);
      fetch(e & kBrickNumber, w);
      Run here = run_of(e & kBrickNumber);
      int first = 0, next_place = bring(here, 0, 0, pieces);   // in the ring: of the present roi, of the next
      for (int done = 0; done < have; done++) {
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");   // the gradient is here, and the tables
        asm volatile("" : "+v"(w.x0.x), "+v"(w.x0.y), "+v"(w.x0.z), "+v"(w.x0.w), "+v"(w.x1.x), "+v"(w.x1.y), "+v"(w.x1.z), "+v"(w.x1.w));
        asm volatile("" : "+v"(w.y[0].x), "+v"(w.y[0].y), "+v"(w.y[1].x), "+v"(w.y[1].y), "+v"(w.y[2].x), "+v"(w.y[2].y), "+v"(w.y[3].x),
                          "+v"(w.y[3].y), "+v"(w.z.x), "+v"(w.z.y), "+v"(w.z.z), "+v"(w.z.w));
        const bool idle = turn != kBrickAll && !screen(first, turn);
        const bool more = done + 1 < have;
        const unsigned e2 = more ? entry(done + 1) : e, n2 = e2 & kBrickNumber;
        const Run run2 = run_of(n2);
        int first2 = next_place;
        Weights w2;
        fetch(n2, w2);
        if (more) next_place = bring(run2, first2, 0, early);
        const float ws[4] = {own_block ? w.z.x : 0.f, own_block ? w.z.y : 0.f, own_block ? w.z.z : 0.f, own_block ? w.z.w : 0.f};
        const float xs[8] = {w.x0.x, w.x0.y, w.x0.z, w.x0.w, w.x1.x, w.x1.y, w.x1.z, w.x1.w};
        // (from the 4-byte boundary, and shifted after: 16 bytes at a 2-byte boundary take LDS 60 clocks, 660 instead of 380 us of all)
        const unsigned at = (piece + here.odd / 2) / 2 * 4 + first * 1024, end = ring * 1024;
        const unsigned shift = (piece + here.odd / 2) % 2 * 16;
        const int pair = 4 * cells;   // bytes from two channels to the next
        const BrickLeft left = brick_left(ws, 1.f / kBrickWeight);
        const u32x4 left_both = brick_pair(left.value, left.rest);
        const bool upper = !idle && (e & kBrickUpper) != 0, lower = !idle && (e & kBrickLower) != 0;
        const BrickScales scales(turn != kBrickAll);
        // Two pairs of rows of voxels, or with all bits (EXACT) one, whose operands take as many registers.  `over`: the roi's last sweep.
        auto sweep = [&](auto k0_, auto exact_, const bool over) {
          constexpr bool EXACT = decltype(exact_)::value;
          constexpr int K0 = decltype(k0_)::value, KN = EXACT ? 1 : 2, FORMS = EXACT ? 2 : 1;
          unsigned from = at, second = to_second;
          asm volatile("" : "+v"(second));
          const float taken = second == 0 ? -1.f : 0.f;   // the second row is the first again
          float weight = EXACT ? scales.weight : kBrickWeight;
          u32x4 right[FORMS][KN][2], left_value{}, left_rest{};   // the second form: what the rounding left of the first
          if constexpr (EXACT) {
            asm volatile("" : "+v"(from), "+v"(weight));   // (nothing below is formed for several sweeps and kept: that takes more registers than there are)
            const BrickLeft l = brick_left(ws, scales.value), small = brick_left(ws, scales.rest);
            left_value = brick_pair(l.value, small.value);
            left_rest = brick_pair(l.rest, small.rest);
          }
#pragma unroll
          for (int k = 0; k < KN; k++)
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
              const float y = (ks == 0 ? w.y[K0 + k].x : w.y[K0 + k].y) * weight;
              float f[8];
#pragma unroll
              for (int j = 0; j < 8; j++) f[j] = y * xs[j];
              right[0][k][ks] = M::pack(f);
              if (ks == 1) {
#pragma unroll
                for (int j = 0; j < 8; j++) f[j] = fmaf(M::element(right[0][k][1], j), taken, f[j]);
                right[0][k][1] = M::pack(f);
              }
              if constexpr (EXACT) {   // (the first row's stand in the second one's place already where that is free)
#pragma unroll
                for (int j = 0; j < 8; j++) f[j] = (f[j] - M::element(right[0][k][ks], j)) * (ks == 0 ? 1.f + taken : 1.f);
                right[FORMS - 1][k][ks] = M::pack(f);
              }
            }
#pragma unroll
          for (int i = 0; i < 4; i++) read(from + i * pair, end, slot[i]);
#pragma unroll
          for (int i = 0; i < kBrickChannels / 2; i++) {
            u32x4 g[2];
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
              const u32x4 v = slot[i % 4][ks];
              g[ks] = u32x4{__builtin_amdgcn_alignbit(v.y, v.x, shift), __builtin_amdgcn_alignbit(v.z, v.y, shift),
                            __builtin_amdgcn_alignbit(v.w, v.z, shift), v.w >> shift};
            }
            float4_t part[KN];
#pragma unroll
            for (int k = 0; k < KN; k++) part[k] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int form = FORMS - 1; form >= 0; form--)
#pragma unroll
              for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int k = 0; k < KN; k++) part[k] = M::run16(g[ks], right[form][k][ks], part[k]);
            if (i < 4) read(from + (i + 4) * pair, end, slot[i]);
            if (i == 3 && over) {
#pragma unroll
              for (int j = 0; j < 4; j++) asm volatile("" : "+v"(slot[j][0]), "+v"(slot[j][1]) : : "memory");   // they have been read
              if (more) next_place = bring(run2, next_place, early, pieces);
            }
#pragma unroll
            for (int k = 0; k < KN; k++) {
              if constexpr (EXACT) {
                const u32x4 sums = brick_sums_exact(part[k], scales);
                acc[i][K0 + k] = M::run16(left_value, sums, M::run16(left_rest, sums, acc[i][K0 + k]));
              } else {
                acc[i][K0 + k] = M::run16(left_both, brick_sums(part[k]), acc[i][K0 + k]);
              }
            }
          }
        };
        // (one condition after the other, not two branches of one: where those meet, all sums are copied)
        using std::integral_constant;
        const bool exact = turn == kBrickFinite || (e & kBrickExact) != 0 || ((e & kBrickNumber) == static_cast<unsigned>(p.R) - 1u && c_base + kBrickChannels >= p.C);
        if (!exact && upper) sweep(integral_constant<int, 0>(), std::false_type(), !lower);
        if (!exact && lower) sweep(integral_constant<int, 2>(), std::false_type(), true);
        unsigned all_bits = __builtin_amdgcn_readfirstlane(exact ? 1 : 0);
        asm volatile("" : "+s"(all_bits));
        if (all_bits != 0 && upper) {
          sweep(integral_constant<int, 0>(), std::true_type(), false);
          sweep(integral_constant<int, 1>(), std::true_type(), !lower);
        }
        if (all_bits != 0 && lower) {
          sweep(integral_constant<int, 2>(), std::true_type(), false);
          sweep(integral_constant<int, 3>(), std::true_type(), true);
        }
        if (idle && more) {
          asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");   // the screened gradient has been written: its places may be taken
          next_place = bring(run2, next_place, early, pieces);
        }
        e = e2; w = w2; here = run2; first = first2;
      }
    }
    if (turn == kBrickAll && !brick_finite(acc)) bits = 1;
    if constexpr (SHARED) {
      if (have == 0) return;
    } else {   // (both wavefronts take the same turns: they leave their sums together)
      if (bits != 0 && brick_lane() == 0) atomicOr(&special, bits);
      __syncthreads();
      bits = __builtin_amdgcn_readfirstlane(special);
    }
    if (turn == kBrickAll && bits != 0) {
      turn = kBrickFinite;
      continue;
    }
    const bool infinite = (bits & (kBrickHasPlus | kBrickHasMinus)) != 0, first = turn <= kBrickFinite;
    const float mark = turn == kBrickMinus ? -INFINITY : infinite ? INFINITY : NAN;   // for what the later turns' gradients reach
    if constexpr (SHARED) {
      float4_t *to =
          partial + ((brick * cblocks + c_base / kBrickChannels) * parts + place.part) * (kBrickChannels / 2 * 4 * kWave) + brick_lane();
      asm volatile("" : "+v"(to));   // (the addresses are not formed before the turns and kept)
      if (turn == kBrickAll) {
#pragma unroll
        for (int i = 0; i < kBrickChannels / 2; i++)
#pragma unroll
          for (int k = 0; k < 4; k++) to[(i * 4 + k) * kWave] = acc[i][k];
      } else {
#pragma unroll
        for (int i = 0; i < kBrickChannels / 2; i++)
#pragma unroll
          for (int k = 0; k < 4; k++) {
            float4_t sum = acc[i][k];
#pragma unroll
            for (int r = 0; r < 4; r++) sum[r] = first ? sum[r] : sum[r] > 0.f ? mark : 0.f;
            if (!first) sum += to[0];
            to[0] = sum;
            to += kWave;
            asm volatile("" : "+v"(to) : : "memory");   // (one after the other: together they take more registers than there are)
          }
      }
    } else {
      brick_finish<LOG_WX>(acc, place, grad, p, lds, first, mark);
    }
    if (turn == kBrickFinite && (bits & (kBrickHasPlus | kBrickHasNan))) turn = kBrickPlus;
    else if ((turn == kBrickFinite || (turn == kBrickPlus && infinite)) && (bits & (kBrickHasMinus | kBrickHasNan))) turn = kBrickMinus;
    else return;
    if constexpr (!SHARED) __syncthreads();   // the sums have been read and are in memory
  }
}

// The sums of the parts.
template <int LOG_WX>
__global__ __launch_bounds__(kWave << LOG_WX) void roi_brick_fold_kernel(
    const unsigned *__restrict__ lengths, __half *__restrict__ grad, const RoiProblem p, const int nx, const int ny, const int nz,
    const int cblocks, const unsigned total, const int parts, const float4_t *__restrict__ partial) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const BrickPlace<LOG_WX> place(p, nx, ny, nz, cblocks, 1, total);
  if (place.none) return;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int have = wave < place.bricks ? static_cast<int>(lengths[place.brick + wave]) : 0;
  float4_t acc[kBrickChannels / 2][4];
#pragma unroll
  for (int i = 0; i < kBrickChannels / 2; i++)
#pragma unroll
    for (int k = 0; k < 4; k++) acc[i][k] = float4_t{0.f, 0.f, 0.f, 0.f};
  const float4_t *from = partial + ((place.brick + wave) * cblocks + place.c_base / kBrickChannels) * parts * (kBrickChannels / 2 * 4 * kWave) + lane;
  for (int part = 0; part < parts; part++, from += kBrickChannels / 2 * 4 * kWave) {
    if (brick_share(have, part, parts) == brick_share(have, part + 1, parts)) continue;   // (left nothing)
#pragma unroll
    for (int i = 0; i < kBrickChannels / 2; i++)
#pragma unroll
      for (int k = 0; k < 4; k++) acc[i][k] += from[(i * 4 + k) * kWave];
  }
  brick_finish<LOG_WX>(acc, place, grad, p, lds, true, 0.f);
}

static size_t brick_tables_bytes(const RoiProblem &p) {
  return (static_cast<size_t>(p.R) * brick_rows(p) * kBrickCells * sizeof(float) + 255) / 256 * 256;
}

static long brick_count(const RoiProblem &p) {
  return static_cast<long>(p.N) * (brick_up(p.D) / kBrickEdge) * (brick_up(p.H) / kBrickEdge) * (brick_up(p.W) / kBrickEdge);
}
static long brick_waves(const RoiProblem &p) { return brick_count(p) * ((p.C + kBrickChannels - 1) / kBrickChannels); }

// Workgroups that share a brick and 16 channels, for maps of few such pairs whose bricks have many rois each (a roi is one serial chain for a
// wavefront); their sums go through memory (32 KB for a wavefront) and another launch.  2048 wavefronts run at a time.  Forward and backward
// pass, one workgroup and as many as make 2048 wavefronts: [4,64,11,27,28] with 3510 rois of 7^3 cells 873 and 435 us, [2,83,24,29,25] with 484
// of 4^3 271 and 190; [2,24,35,93,28] with 369 of 2^3, four rois per five bricks, 59 and 66.
// Lists differ in length, and the longest is the end of the launch: 4096 wavefronts, half as long, even that out where lists are long.  2048 and
// 4096: [1,128,36,27,46] with 2424 rois of 4^3, 20 per brick, 530 and 403 us, [1,128,9,76,38] with 2543 of 7^3, 25 per brick, 575 and 453,
// [1,128,12,48,65] with 932 of 5^3, 9 per brick, 331 and 315; [1,64,22,57,38] with 243 of 7^3, 2 per brick, 80 and 89, [2,32,19,95,25] with 568, 2
// per brick, 70 and 78.
static int brick_parts(const RoiProblem &p) {
  if (4L * p.R < 5 * brick_count(p)) return 1;
  const long wavefronts = p.R >= 8 * brick_count(p) ? 4096 : 2048;
  return static_cast<int>(std::max(wavefronts / brick_waves(p), 1L));   // (at most eight: roi_brick_applies asks for 480 pairs)
}

// Kilobytes of a roi's 16 channels (and behind them: a row of cells may be read as 16 bytes, and rows up to the eighth), and of a wavefront's
// ring: as much as lets eight wavefronts share a compute unit's LDS, or one roi's
static int brick_pieces(const RoiProblem &p) { return (kBrickChannels * p.od * p.oh * p.ow * 2 + 2 + kBrickPad + 1023) / 1024; }
static int brick_ring(const RoiProblem &p) { return std::max(std::min(2 * brick_pieces(p), 18), brick_pieces(p)); }

bool roi_brick_applies(int dtype, const RoiProblem &p) {
  if (dtype != MV_F16 || p.ndim != 3 || p.od > kBrickCells || p.oh > kBrickCells || p.ow > kBrickCells || !roi_pool_applies(dtype, p)) return false;
  if (p.D > 0x7fff || p.H > 0x7fff || p.W > 0x7fff) return false;
  const long slab = static_cast<long>(p.C) * p.od * p.oh * p.ow * 2;   // bytes of a roi's gradient
  if (slab < kBrickPad || slab + kBrickPad >= (1L << 31)) return false;
  if (static_cast<long>(p.R) * brick_rows(p) * kBrickCells * 4 >= (1L << 31) || p.R >= (1 << 29)) return false;
  // Small maps have too few bricks to fill the chip, and few channels leave most of a product idle; there the kernel that adds box by box is
  // the faster one.  Forward and backward pass there -> here: [1,16,14,40,66] with 163 rois of 7^3 cells (90 bricks) 37 -> 54 us,
  // [4,36,10,20,26] with 112 (96 bricks) 59 -> 72, [2,19,6,125,50] with 89 of 8^3 (224 bricks) 38 -> 42; [2,16,12,94,77] with 987 (480 bricks) 84 -> 77,
  // [1,32,18,57,123] with 463 91 -> 83, [2,256,10,64,67] with 363 of 5^3 173 -> 130.  Over 2500 heads of 16 - 4000 rois, 2^3 - 8^3 cells, 16 - 256 channels
  // and up to 64 x 128 x 128 voxels 1.20 times as fast in geometric mean (1.05 below 800 pairs of a brick and 16 channels, 1.42 from 4096 on), one in
  // twenty-five slower by more than a tenth.  (The small ones stay for their values too: box by box, zero times an infinity reaches the whole box.)
  // Gradients that fill a wavefront's ring: hardly any of the next roi's comes in beside the present one's products, so that long lists take twice
  // as long as others.  500 such heads (8^3 cells), box by box / here: below two rois for five bricks 1.30 (from 4096 wavefronts on) to 0.90 (below
  // 800), up to five for four 1.05 from 2048 wavefronts on and 0.76 - 0.95 below, beyond 0.80 - 0.87 ([4,128,48,60,21] with 3808 rois 1215 and 1946 us).
  if (brick_ring(p) < std::min(2 * brick_pieces(p), brick_pieces(p) + 4) &&
      (brick_waves(p) >= 2048 ? 4L * p.R >= 5 * brick_count(p) : 5L * p.R >= 2 * brick_count(p)))
    return false;
  return brick_count(p) * p.C >= 7680 && brick_waves(p) * 16 < (1L << 31) - 8;
}

static size_t brick_lists_bytes(const RoiProblem &p) { return (static_cast<size_t>(brick_count(p)) * (p.R + 1) * 4 + 255) / 256 * 256; }
static size_t brick_partial_bytes(const RoiProblem &p) {
  const int parts = brick_parts(p);
  return parts > 1 ? static_cast<size_t>(brick_waves(p)) * parts * kBrickChannels * 512 * sizeof(float) : 0;
}

// Lists grow with rois times bricks: where they would take more than 256 MB and more than the fp32 copy of the gradient of the kernel
// with atomics (more than 512 rois per channel on large maps), that kernel stays.
size_t roi_brick_workspace(int dtype, const RoiProblem &p) {
  if (!roi_brick_applies(dtype, p)) return 0;
  const size_t bytes = brick_tables_bytes(p) + brick_lists_bytes(p) + brick_partial_bytes(p) + static_cast<size_t>(p.R) * sizeof(BrickRoi) +
                       static_cast<size_t>(p.C) * p.od * p.oh * p.ow * 2 + kBrickPad;
  const size_t copy = static_cast<size_t>(p.N) * p.C * p.D * p.H * p.W * sizeof(float);
  return bytes <= std::max(copy, static_cast<size_t>(256) << 20) ? bytes : 0;
}

// Writes all of grad_input.  -1: not for these kernels, or a workspace that is too small for them.
int roi_brick_backward(const void *grad_output, const void *rois, void *grad_input, int dtype, const RoiProblem &p, void *workspace,
                       size_t capacity, hipStream_t s) {
  const size_t wanted = roi_brick_workspace(dtype, p);
  if (wanted == 0 || capacity < wanted || reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return -1;
  float *const tables = static_cast<float *>(workspace);
  unsigned *const lists = reinterpret_cast<unsigned *>(static_cast<char *>(workspace) + brick_tables_bytes(p));
  unsigned *const lengths = lists + brick_count(p) * p.R;
  float4_t *const partial = reinterpret_cast<float4_t *>(reinterpret_cast<char *>(lists) + brick_lists_bytes(p));
  BrickRoi *const recs = reinterpret_cast<BrickRoi *>(reinterpret_cast<char *>(partial) + brick_partial_bytes(p));
  __half *const copy = reinterpret_cast<__half *>(recs + p.R);
  const int slab = p.C * p.od * p.oh * p.ow;
  const int copies = (slab + kBrickPad / 2 + 3 * kWave * 8 - 1) / (3 * kWave * 8);
  // (rows of eight cells have to lie at 4-byte boundaries: what a shift brings in is one cell short of that)
  if (p.ow == kBrickCells && reinterpret_cast<uintptr_t>(grad_output) % 4 != 0) return -1;
  const int pieces = brick_pieces(p), ring = brick_ring(p);
  const int log_wx = p.W > kBrickEdge ? 1 : 0;
  const int nx = (p.W + (8 << log_wx) - 1) >> (3 + log_wx), ny = brick_up(p.H) / kBrickEdge, cblocks = (p.C + kBrickChannels - 1) / kBrickChannels;
  const int nz = brick_up(p.D) / kBrickEdge;
  const int parts = brick_parts(p);
  const long regions = static_cast<long>(p.N) * cblocks * nz * ny * nx, total = regions * parts;
  const float *const r = static_cast<const float *>(rois);
  const __half *const g = static_cast<const __half *>(grad_output);
  __half *const grad = static_cast<__half *>(grad_input);
  const size_t sums = static_cast<size_t>(kBrickChannels) * ((512 << log_wx) + 8) * 2, rings = static_cast<size_t>(ring + 1) * 1024 << log_wx;
  hipLaunchKernelGGL(roi_brick_tables_kernel, dim3(p.R + copies), dim3(3 * kWave), 0, s, r, recs, tables, p, g + static_cast<long>(p.R - 1) * slab,
                     copy, slab);
  hipLaunchKernelGGL(roi_brick_lists_kernel, dim3(static_cast<unsigned>(brick_count(p))), dim3(kBrickThreads), 0, s,
                     reinterpret_cast<const uint4 *>(recs), lists, lengths, p.R, brick_up(p.W) / kBrickEdge, ny, nz);
  auto grid = [](long n) { return dim3(static_cast<unsigned>((n + 7) / 8 * 8)); };
#define MV_BRICK(LOG_WX, SHARED)                                                                                               \
  hipLaunchKernelGGL((roi_brick_backward_kernel<LOG_WX, SHARED>), grid(total), dim3(kWave << LOG_WX), std::max(sums, rings), s, g, copy, tables, \
                     lists, lengths, grad, p, nx, ny, nz, cblocks, static_cast<unsigned>(total), pieces, ring, parts, partial)
#define MV_BRICK_FOLD(LOG_WX)                                                                                                  \
  hipLaunchKernelGGL((roi_brick_fold_kernel<LOG_WX>), grid(regions), dim3(kWave << LOG_WX), sums, s, lengths, grad, p, nx, ny, nz, \
                     cblocks, static_cast<unsigned>(regions), parts, partial)
  if (parts == 1) {
    if (log_wx) MV_BRICK(1, false); else MV_BRICK(0, false);
  } else if (log_wx) {
    MV_BRICK(1, true);
    MV_BRICK_FOLD(1);
  } else {
    MV_BRICK(0, true);
    MV_BRICK_FOLD(0);
  }
#undef MV_BRICK
#undef MV_BRICK_FOLD
  return check_launch("roi_brick_backward_kernel");
}

}  // namespace mv
