// RoIAlign / RoIAlignRotated BACKWARD of heads that the separable kernels do not take (rotated boxes, sampling grids above
// four), by the voxels' owners: no global atomics, no fp32 copy of the gradient to clear and to fold.  Same results as the
// reference's one-thread-per-output kernel with one atomicAdd per sample corner
// (csrc/cuda/roi_align_rotated_3d_cuda_kernel.cuh:124-265 and the 2-D twin).
//
// A workgroup owns a tile of 64 voxels (8 x 4 x 2, images 8 x 8) and 64 channels and writes their gradient once.  It lists
// the rois whose samples' bounding box meets the tile; each of its two wavefronts takes rois from the list.  A roi's
// contribution is a matrix product, gradient[voxel][channel] = sum over cells of weight[voxel][cell] *
// grad_output[cell][channel], where weight[voxel][cell] is the mean over the cell's samples of the corner weights that
// fall on the voxel.  The wavefront picks the cells that reach the tile (32 columns at a time, of several rois where one
// has fewer), works their samples out once -- for all the channels -- and adds the corner weights to a table of 32-bit
// fixed-point numbers in LDS (quanta of 2^-30 of a cell's whole weight -- of the part of it that one voxel can get where a
// cell has many samples -- so finer than the fp32 product of the three fractions that they are made of); the table then is the left operand of matrix-core products with the
// gradient's rows, which a transposing copy has laid out channels-last.  Products keep the table's precision: 16-bit
// gradients are exact operands and the weights are split into two fp16 or three bf16 numbers, fp32 ones use the fp32
// matrix instructions; sums are fp32.
//
// Why owners: the samples' 8 corners times channels are 1.4 G additions for 1000 rois of 7^3 cells, 2^3 samples and 64
// channels; summed in LDS boxes per roi and added to memory, the boxes' scan and 64-byte global atomics (21 G a second)
// took the time.  Here the additions are products (70 GFLOP with what the tiles' padding wastes), the corner weights are
// added once per sample instead of once per channel, and what bounds the kernel is the samples' arithmetic (every
// cell is worked out by each of the ~10 tiles it reaches) and the conversion of the tables: vector issue 70 %, waits 40 % of the
// wavefronts' time, LDS 14 %.  A sample's eight corners are added without branches, those outside the tile as zeros, and in tiles off the image's border
// its voxels are its position's floor: 358 us, 440 with a branch per corner and the clamped taps everywhere.
// Small tiles: a tile's products are dense, and cells that reach it fill a larger one less.
// Training step of 1000 rois with 7^3 cells on [2,64,48,96,96] fp16: 2080 -> 550 us, of which this kernel takes 358 us (26 us for
// the layout; the box kernel, its fp32 sums and their fold took 1.8 ms).
#include "common.hpp"
#include "roi_geometry.hpp"
#include "sampling.hpp"
#include "roi_taps.hpp"
#include "dcn_mfma.hpp"

namespace mv {

constexpr int kOwnThreads = 128, kOwnWaves = kOwnThreads / kWave;
constexpr int kOwnChannels = 64, kOwnVoxels = 64;
constexpr int kOwnColumns = 32;    // cells of one table
constexpr int kOwnPitch = 36;      // words between a table's voxels: rows stay 16-byte aligned and spread over the banks
constexpr int kOwnRois = 512;      // rois listed at a time
constexpr int kOwnTried = 2;       // rois that a thread tries at a time: their bounds are fetched together

// What the layout kernel leaves about the rois: their geometry, the bounds of the voxels that their samples reach, and the
// map from a tile's middle to the middle of the cells that can reach it, in cells, with half their extent.
struct OwnBox { float map[3][3], offset[3], reach[3], unused; };
static_assert(sizeof(OwnBox) == 64 && sizeof(RoiGeom) == 192, "a box record is one cache line, a geometry record 24 doubles");
constexpr int kOwnPart = 47;   // word of a geometry record, behind its last member: the part of a cell's whole weight that one voxel can get
struct OwnRois {
  RoiGeom *geom;    // [R]
  OwnBox *box;      // [R]
  float4 *first;    // [R]: first voxel along x, y, z, and the image's number
  float4 *last;     // [R]: last voxel along x, y, z
};
constexpr size_t kOwnRoiBytes = sizeof(RoiGeom) + sizeof(OwnBox) + 2 * sizeof(float4);

__device__ inline void own_geometry(const float *roi, const unsigned n, const OwnRois &out, const RoiProblem &p) {
  double sn[3], cs[3];
#pragma unroll
  for (int a = 0; a < 3; a++) roi_trig(roi, p, a, sn[a], cs[a]);
  RoiGeom g;
  build_geom(g, roi, p, sn, cs);
  const int cells[3] = {p.ow, p.oh, p.od};
  bool empty = g.batch < 0 || g.grid[0] <= 0 || g.grid[1] <= 0 || (p.ndim == 3 && g.grid[2] <= 0);
  float lo[3] = {-1.f, -1.f, -1.f}, hi[3] = {1.f, 1.f, 1.f};
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (a >= p.ndim) continue;
    double c = g.centre[a], reach = 1.001;
#pragma unroll
    for (int j = 0; j < 3; j++) {
      if (j >= p.ndim) continue;
      const double first = local_coord(g, j, 0, 0), last = local_coord(g, j, cells[j] - 1, g.grid[j] - 1);
      c += g.rot[3 * a + j] * 0.5 * (first + last);
      reach += fabs(g.rot[3 * a + j] * 0.5 * (last - first));
    }
    reach += 1e-6 * fabs(c);   // (the bounds are rounded to fp32)
    lo[a] = static_cast<float>(c - reach);
    hi[a] = static_cast<float>(c + reach);
    if (!(c - reach <= c + reach)) empty = true;   // NaN
  }
  out.geom[n] = g;
  // The part of a cell's whole weight that one voxel can get, as a power of two.  A sample's weight is at most the integral, over
  // its cell of the sample lattice, of the voxel's weight function widened by half that cell: (b + e) / spacing per axis, e the
  // lattice cell's extent along the voxel axis, b the function's own integral (1; 1.5 at a border, whose voxel also takes the
  // samples beyond it; 2 on an axis of one voxel).  (1 down to an eighth: three bits of 30 do not matter, and rois of one part
  // share tables.)
  double most = 1.0;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (a >= p.ndim) continue;
    double e = 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++)
      if (j < p.ndim) e += fabs(g.rot[3 * a + j] * g.sub[j]);
    most *= (((a == 0 ? p.W : a == 1 ? p.H : p.D) == 1 ? 2.0 : 1.5) + e) / fabs(g.sub[a]);
  }
  float part = 1.f;
  if (most * 1.0001 < g.count)   // (not for NaN)
    while (part > 1e-9f && 0.5 * part * g.count >= fmax(most * 1.0001, 1.0)) part *= 0.5f;
  reinterpret_cast<float *>(out.geom + n)[kOwnPart] = part < 0.125f ? part : 1.f;
  out.first[n] = make_float4(empty ? 3e38f : lo[0], lo[1], lo[2], __int_as_float(g.batch));
  out.last[n] = make_float4(hi[0], hi[1], hi[2], 0.f);
  OwnBox box;
  const double ext[3] = {3.5, p.ndim == 3 ? 1.5 : 3.5, p.ndim == 3 ? 0.5 : 0.0};   // half a tile
  const int size[3] = {p.W, p.H, p.D};
#pragma unroll
  for (int j = 0; j < 3; j++) {
    // (a cell's samples start and end half their spacing inside it)
    double offset = -g.start[j], reach = 1e-6 - 0.5 * g.sub[j], slack = fabs(g.start[j]);
#pragma unroll
    for (int a = 0; a < 3; a++) {
      if (a >= p.ndim) continue;
      offset -= g.rot[3 * a + j] * g.centre[a];
      reach += fabs(g.rot[3 * a + j]) * (ext[a] + 1.0);
      slack += fabs(g.rot[3 * a + j]) * (fabs(g.centre[a]) + size[a] + 8.0);
    }
    slack = 1e-6 * slack / g.bin[j] + 1e-4;   // (the map is evaluated in fp32)
    const bool small = j < p.ndim && g.bin[j] > 1e-9 && slack < 1e6;
#pragma unroll
    for (int a = 0; a < 3; a++) box.map[j][a] = small && a < p.ndim ? static_cast<float>(g.rot[3 * a + j] / g.bin[j]) : 0.f;
    box.offset[j] = small ? static_cast<float>(offset / g.bin[j]) : 0.f;
    box.reach[j] = small ? static_cast<float>(reach / g.bin[j] + slack) : 1e9f;   // otherwise: every cell
  }
  box.unused = 0.f;
  out.box[n] = box;
}

// grad_output [roi][channel][cell] -> [roi][cell][channel], then the rois' records, and by the workgroups that are left the
// clearing of the gradient's `cleared` elements
constexpr int kOwnClearPieces = 16;   // 16-byte pieces that a thread clears
template <typename U>
__global__ __launch_bounds__(256) void roi_own_layout_kernel(const U *__restrict__ x, U *__restrict__ xt,
                                                             const float *__restrict__ rois, const OwnRois recs,
                                                             const RoiProblem p, const unsigned pblocks, const unsigned moves,
                                                             U *__restrict__ grad, const long cleared) {
  if (blockIdx.x < moves) {
    const unsigned bx = blockIdx.x % pblocks, r = blockIdx.x / pblocks;
    dcn_move_block<U>(x, xt, p.C, p.C, p.C, p.C, static_cast<long>(p.od) * p.oh * p.ow, bx, static_cast<int>(r % p.R),
                      static_cast<int>(r / p.R));
    return;
  }
  const unsigned n = (blockIdx.x - moves) * 256 + threadIdx.x;
  if (blockIdx.x - moves >= (p.R + 255u) / 256u) {
    constexpr int per = 16 / static_cast<int>(sizeof(U));
    const U zeros[per] = {};
    long at = (blockIdx.x - moves - (p.R + 255u) / 256u) * (256L * kOwnClearPieces * per) + static_cast<long>(threadIdx.x) * per;
#pragma unroll
    for (int i = 0; i < kOwnClearPieces; i++, at += 256 * per) {
      if (at + per <= cleared) {
        __builtin_memcpy(grad + at, zeros, sizeof(zeros));   // one store: global memory takes any alignment
      } else {
        for (long k = at; k < cleared; k++) grad[k] = 0;
      }
    }
    return;
  }
  if (n < static_cast<unsigned>(p.R)) own_geometry(rois + static_cast<long>(n) * roi_columns(p.ndim, p.rotated), n, recs, p);
}

__device__ __forceinline__ void own_wave_sync() {   // LDS of one wavefront is in order: only the compiler has to keep it
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// round(x) for 0 <= x < 2^31 in one instruction (in the register of x: around inline assembly the compiler leaves no wait for a matrix instruction
// that still reads a register which the result would get)
__device__ __forceinline__ unsigned own_round(float x) {
  unsigned r = __float_as_uint(x);
  asm("v_cvt_rpi_i32_f32 %0, %0" : "+v"(r));
  return r;
}

typedef float own_acc __attribute__((ext_vector_type(16)));
typedef unsigned own_u32x4 __attribute__((ext_vector_type(4)));

// The table's rows of one lane as operands: how many the weights are split into, their scale, and the split.
template <typename T> struct OwnSplit;
template <> struct OwnSplit<__half> {
  static constexpr int parts = 2;
  static constexpr float scale = 1.f / 32768.f, back = 1.f / 32768.f;   // weights up to 2^15: the second part stays a normal number
  typedef _Float16 V __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ void split(const float (&w)[8], V (&v)[parts]) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
      v[0][e] = static_cast<_Float16>(w[e]);
      v[1][e] = static_cast<_Float16>(w[e] - static_cast<float>(v[0][e]));
    }
  }
  static __device__ __forceinline__ own_acc mfma(V a, own_u32x4 b, own_acc c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, __builtin_bit_cast(V, b), c, 0, 0, 0);
  }
};
template <> struct OwnSplit<__hip_bfloat16> {
  static constexpr int parts = 3;
  static constexpr float scale = 1.f / 1073741824.f, back = 1.f;
  typedef __bf16 V __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ void split(const float (&w)[8], V (&v)[parts]) {
    // (truncated: the parts hold eight bits each of the fp32 number's 24)
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      float a = w[e], b = w[e + 1];
#pragma unroll
      for (int i = 0; i < parts; i++) {
        const unsigned ua = __float_as_uint(a), ub = __float_as_uint(b);
        reinterpret_cast<unsigned *>(&v[i])[e / 2] = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
        a -= __uint_as_float(ua & 0xffff0000u);
        b -= __uint_as_float(ub & 0xffff0000u);
      }
    }
  }
  static __device__ __forceinline__ own_acc mfma(V a, own_u32x4 b, own_acc c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(V, b), c, 0, 0, 0);
  }
};
template <> struct OwnSplit<float> {
  static constexpr int parts = 1;
  static constexpr float scale = 1.f / 1073741824.f, back = 1.f;
};

struct OwnTile {
  int x, y, z, image, group;
  __device__ __forceinline__ OwnTile(unsigned id, int nx, int ny, int nz, int groups) {
    x = id % nx; id /= nx;
    group = id % groups; id /= groups;
    y = id % ny; id /= ny;
    z = id % nz;
    image = id / nz;
  }
};

// The lane's column of product n: 16-bit channels come in pairs, one load for both products; fp32 ones a product apart, so
// that the second product is left out where a group has at most 32 channels.
template <typename T>
__device__ __forceinline__ int own_channel(int l32, int n) { return sizeof(T) == 2 ? 2 * l32 + n : 32 * n + l32; }

// Writes half of a tile's gradient from the lanes that hold the sums: v[n][i] is voxel 32 half_tile + 8 (i / 4) +
// 4 (lane / 32) + i % 4 of channel own_channel(lane % 32, n), so a lane has four voxels along x of eight rows.
template <typename T, int TX, int TY, int TZ>
__device__ __forceinline__ void own_write(T *__restrict__ grad, const RoiProblem &p, const OwnTile &tile, const int half_tile,
                                          const own_acc (&v)[2]) {
  const int lane = threadIdx.x % kWave, x0 = tile.x * TX + 4 * (lane / 32);
#pragma unroll
  for (int n = 0; n < 2; n++) {
    const int channel = tile.group * kOwnChannels + own_channel<T>(lane % 32, n);
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int row = half_tile * 4 + g, y = tile.y * TY + row % TY, z = tile.z * TZ + row / TY;
      if (channel >= p.C || y >= p.H || z >= p.D) continue;
      T out[4];
#pragma unroll
      for (int x = 0; x < 4; x++) out[x] = store_cast<T>(v[n][4 * g + x] * OwnSplit<T>::back);
      T *dst = grad + ((((static_cast<long>(tile.image) * p.C + channel) * p.D + z) * p.H + y) * p.W + x0);
      if (x0 + 4 <= p.W) {   // one store: global memory takes any alignment
        typedef unsigned V __attribute__((ext_vector_type(sizeof(T)), aligned(sizeof(T))));
        V o;
        __builtin_memcpy(&o, out, sizeof(o));
        *reinterpret_cast<V *>(dst) = o;
      } else {
#pragma unroll
        for (int x = 0; x < 4; x++)
          if (x0 + x < p.W) dst[x] = out[x];
      }
    }
  }
}

// The parts of tiles that several workgroups have shared, [tile][part][half][n, i][lane].
template <typename T, int TX, int TY, int TZ>
__global__ __launch_bounds__(kOwnThreads) void roi_own_fold_kernel(const float *__restrict__ partial, T *__restrict__ grad,
                                                                   const RoiProblem p, const int nx, const int ny, const int nz,
                                                                   const int groups, const int parts) {
  own_acc v[2];
#pragma unroll
  for (int n = 0; n < 2; n++)
#pragma unroll
    for (int i = 0; i < 16; i++) v[n][i] = 0.f;
  const float *src = partial + static_cast<long>(blockIdx.x) * parts * kOwnChannels * kOwnVoxels + threadIdx.x / kWave * 2048 + threadIdx.x % kWave;
  for (int k = 0; k < parts; k++, src += kOwnChannels * kOwnVoxels)
#pragma unroll
    for (int n = 0; n < 2; n++)
#pragma unroll
      for (int i = 0; i < 16; i++) v[n][i] += src[(n * 16 + i) * kWave];
  own_write<T, TX, TY, TZ>(grad, p, OwnTile(blockIdx.x, nx, ny, nz, groups), threadIdx.x / kWave, v);
}

// gt: grad_output channels-last, [roi][cell][channel].
// `parts` workgroups share a tile, every parts-th roi each, and leave their sums in `partial` where that is more than one.
// `cleared`: the gradient holds zeros, tiles without rois are left alone.
template <typename T, bool ROT, int TX, int TY, int TZ>
__global__ __launch_bounds__(kOwnThreads, 3) void roi_own_backward_kernel(const T *__restrict__ gt,
                                                                          const OwnRois recs,
                                                                          T *__restrict__ grad, const RoiProblem p,
                                                                          const int nx, const int ny, const int nz,
                                                                          const int groups, const unsigned total, const int parts,
                                                                          const int cleared, float *__restrict__ partial) {
  static_assert(TX * TY * TZ == kOwnVoxels && TX == 8, "tile of 64 voxels");
  typedef OwnSplit<T> S;
  __shared__ __attribute__((aligned(16))) unsigned tables[kOwnWaves * kOwnVoxels * kOwnPitch];   // at the end: the wavefronts' sums
  // the rois whose bounds meet the tile; those with cells that reach it, their first cell and the further ones per axis
  __shared__ unsigned short listed[kOwnRois], reaching[kOwnRois];
  __shared__ unsigned corners[kOwnRois], beyonds[kOwnRois];
  __shared__ unsigned picked[kOwnWaves][kOwnColumns + kWave];
  __shared__ __attribute__((aligned(16))) unsigned rows_of[kOwnWaves][kOwnColumns];
  __shared__ unsigned n_listed, n_reaching, next, special;
  static_assert(sizeof(tables) >= kOwnChannels * kOwnVoxels * sizeof(float), "room for the sums");
  // eight runs of tiles, one per die: neighbouring tiles write parts of the same cache lines
  const unsigned run = (total + 7) / 8, id = (blockIdx.x % 8) * run + blockIdx.x / 8;
  if (blockIdx.x / 8 >= run || id >= total) return;
  const int part = id % parts;
  const OwnTile tile(id / parts, nx, ny, nz, groups);
  const int image = tile.image, c_base = tile.group * kOwnChannels;
  const int t0[3] = {tile.x * TX, tile.y * TY, tile.z * TZ};
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int half = lane / 32, l32 = lane % 32;
  unsigned *const table = tables + wave * kOwnVoxels * kOwnPitch;
  unsigned *const mine = picked[wave];
  unsigned *const rows = rows_of[wave];
  const unsigned cells = static_cast<unsigned>(p.od) * p.oh * p.ow;
  // the lane's columns of the two products (16-bit: C is even)
  const int channel0 = min(c_base + own_channel<T>(l32, 0), p.C - (sizeof(T) == 2 ? 2 : 1));
  const T *const gcol = gt + channel0;
  const int to_second = sizeof(T) == 2 ? 1 : min(c_base + own_channel<T>(l32, 1), p.C - 1) - channel0;
  const bool wide = sizeof(T) == 2 || p.C - c_base > 32;
  const double mid[3] = {t0[0] + 0.5 * (TX - 1), t0[1] + 0.5 * (TY - 1), t0[2] + 0.5 * (TZ - 1)};
  constexpr double ext[3] = {0.5 * (TX - 1), 0.5 * (TY - 1), 0.5 * (TZ - 1)};

  // No sample that reaches the tile is moved onto the image's border (order 1).
  const bool interior = p.order == 1 && t0[0] > 0 && t0[0] + TX < p.W && t0[1] > 0 && t0[1] + TY < p.H && (TZ == 1 || (t0[2] > 0 && t0[2] + TZ < p.D));
  if (threadIdx.x == 0) special = 0;
  bool any = false;   // the tile has a roi (the same for all threads)

  own_acc acc[2][2];
  // Products give NaN for weight 0 times an infinite gradient.  A tile whose sums come out not finite is done again with
  // `careful` set, term by term and without the terms of weight 0.
  for (int careful = 0; careful < 2; careful++) {
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
      for (int n = 0; n < 2; n++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[m][n][i] = 0.f;
    int columns = 0;   // of the table in use
    unsigned part_bits = __float_as_uint(1.f);   // kOwnPart of the rois in the table

    auto multiply = [&] {
      const float unit = S::scale * __uint_as_float(part_bits);
      own_wave_sync();
      if (careful) {
        for (int k = 0; k < columns; k++) {
          const T *src = gcol + static_cast<long>(rows[k]) * p.C;
          const float g0 = static_cast<float>(load(src)), g1 = static_cast<float>(load(src + to_second));
#pragma unroll
          for (int m = 0; m < 2; m++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
              const unsigned q = table[(m * 32 + 8 * (i / 4) + 4 * half + i % 4) * kOwnPitch + k];
              if (q != 0) {
                const float w = static_cast<float>(q) * unit;
                acc[m][0][i] += w * g0;
                acc[m][1][i] += w * g1;
              }
            }
        }
        own_wave_sync();
      }
      for (int k0 = 0; k0 < columns; k0 += 16) {
        const own_u32x4 ra = *reinterpret_cast<const own_u32x4 *>(rows + k0 + half * 8);
        const own_u32x4 rb = *reinterpret_cast<const own_u32x4 *>(rows + k0 + half * 8 + 4);
        const unsigned row[8] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y, rb.z, rb.w};
        unsigned x0[8], x1[8];   // the lane's two channels of eight cells, as they lie in memory (16-bit: both in x0)
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const unsigned *src = reinterpret_cast<const unsigned *>(gcol + static_cast<long>(row[e]) * p.C);
          x0[e] = src[0];
          if constexpr (sizeof(T) == 4) x1[e] = src[to_second];
        }
        float w[2][8];
#pragma unroll
        for (int m = 0; m < 2; m++) {
          own_u32x4 *cell = reinterpret_cast<own_u32x4 *>(table + (m * 32 + l32) * kOwnPitch + k0 + half * 8);
          const own_u32x4 qa = cell[0], qb = cell[1];
          cell[0] = own_u32x4{0, 0, 0, 0};
          cell[1] = own_u32x4{0, 0, 0, 0};
          const unsigned q[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
          for (int e = 0; e < 8; e++) w[m][e] = static_cast<float>(q[e]) * unit;
        }
        if (careful) continue;
        if constexpr (sizeof(T) == 2) {
          own_u32x4 b[2];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            b[0][e] = __builtin_amdgcn_perm(x0[2 * e + 1], x0[2 * e], 0x05040100u);
            b[1][e] = __builtin_amdgcn_perm(x0[2 * e + 1], x0[2 * e], 0x07060302u);
          }
#pragma unroll
          for (int m = 0; m < 2; m++) {
            typename S::V v[S::parts];
            S::split(w[m], v);
#pragma unroll
            for (int n = 0; n < 2; n++)
#pragma unroll
              for (int i = 0; i < S::parts; i++) acc[m][n] = S::mfma(v[i], b[n], acc[m][n]);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; e++)
#pragma unroll
            for (int m = 0; m < 2; m++)
              acc[m][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[m][e], __uint_as_float(x0[e]), acc[m][0], 0, 0, 0);
          if (wide) {
#pragma unroll
            for (int e = 0; e < 8; e++)
#pragma unroll
              for (int m = 0; m < 2; m++)
                acc[m][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[m][e], __uint_as_float(x1[e]), acc[m][1], 0, 0, 0);
          }
        }
      }
      columns = 0;
      own_wave_sync();
    };

    auto one_roi = [&](const RoiGeom &g, const unsigned bits, const unsigned n, const unsigned corner, const unsigned beyond) {
      const int first[3] = {static_cast<int>(corner & 1023u), static_cast<int>((corner >> 10) & 1023u), static_cast<int>(corner >> 20)};
      const int num[3] = {static_cast<int>(beyond & 1023u) + 1, static_cast<int>((beyond >> 10) & 1023u) + 1, static_cast<int>(beyond >> 20) + 1};
      double reach[3];   // of a cell's samples along the voxel axes
#pragma unroll
      for (int a = 0; a < 3; a++) {
        reach[a] = 1.000001 + ext[a];
#pragma unroll
        for (int j = 0; j < 3; j++)
          if (j < p.ndim) reach[a] += fabs(g.rot[3 * a + j]) * (0.5 * (g.grid[j] - 1) * g.sub[j]);
      }
      const int count = g.count, boxed = num[0] * num[1] * num[2];
      const float inv_x = 1.f / static_cast<float>(num[0]), inv_y = 1.f / static_cast<float>(num[1]);
      const float quanta = 1073741824.f / (__uint_as_float(bits) * static_cast<float>(count));
      const float inv_gx = 1.f / static_cast<float>(g.grid[0]), inv_gy = 1.f / static_cast<float>(g.grid[1]);
      for (int i0 = 0; i0 < boxed; i0 += kWave) {
        // each cell of the box is tried on its own
        const int i = i0 + lane;
        const int q1 = static_cast<int>((static_cast<float>(i) + 0.5f) * inv_x);
        const int q2 = static_cast<int>((static_cast<float>(q1) + 0.5f) * inv_y);
        const int at[3] = {first[0] + i - q1 * num[0], first[1] + q1 - q2 * num[1], first[2] + q2};
        bool hit = i < boxed;
        double local[3];
#pragma unroll
        for (int j = 0; j < 3; j++) local[j] = j < p.ndim ? g.start[j] + (at[j] + 0.5) * g.bin[j] : 0.0;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          if (a >= p.ndim) continue;
          double c = local[a];
          if (ROT) c = g.rot[3 * a] * local[0] + g.rot[3 * a + 1] * local[1] + g.rot[3 * a + 2] * local[2] + g.centre[a];
          hit = hit && fabs(c - mid[a]) <= reach[a];
        }
        const unsigned long hits = __ballot(hit);
        int left = __popcll(hits);
        if (left == 0) continue;
        own_wave_sync();
        if (hit) mine[__popcll(hits & ((1UL << lane) - 1))] = static_cast<unsigned>(at[0]) | at[1] << 10 | at[2] << 20;
        own_wave_sync();
        for (int done = 0; left > 0;) {
          if (columns == kOwnColumns || bits != part_bits) {
            multiply();
            part_bits = bits;
          }
          const int m = min(left, kOwnColumns - columns);
          // lanes: m cells (rounded up to a power of two) times parts of their samples
          const int log_m = m > 1 ? 32 - __clz(m - 1) : 0, parts = kWave >> log_m;
          const int k = lane & ((1 << log_m) - 1), part = lane >> log_m;
          if (k < m) {
            const unsigned packed = mine[done + k];
            const unsigned cx = packed & 1023u, cy = (packed >> 10) & 1023u, cz = packed >> 20;
            if (part == 0) rows[columns + k] = n * cells + (cz * p.oh + cy) * p.ow + cx;
            unsigned *const column = table + columns + k;
            unsigned *const aside = column + (part & 15) * kOwnPitch;   // (lanes of one cell apart; 15 voxels and the farthest corner are in the table)
            static_assert(15 + ((TZ > 1 ? TY : 0) + 1) * TX + 1 < kOwnVoxels, "room for every corner");
            const double bx = g.start[0] + cx * g.bin[0], by = g.start[1] + cy * g.bin[1], bz = g.start[2] + cz * g.bin[2];
            for (int s = part; s < count; s += parts) {
              int s1, s2;
              if (count < (1 << 21)) {   // (exact in fp32)
                s1 = static_cast<int>((static_cast<float>(s) + 0.5f) * inv_gx);
                s2 = static_cast<int>((static_cast<float>(s1) + 0.5f) * inv_gy);
              } else {
                s1 = s / g.grid[0];
                s2 = s1 / g.grid[1];
              }
              const double x = bx + static_cast<double>(static_cast<float>(s - s1 * g.grid[0]) + .5f) * g.sub[0];
              const double y = by + static_cast<double>(static_cast<float>(s1 - s2 * g.grid[1]) + .5f) * g.sub[1];
              const double z = p.ndim == 3 ? bz + static_cast<double>(static_cast<float>(s2) + .5f) * g.sub[2] : 0.0;
              double rx = x, ry = y, rz = z;
              if (ROT) {
                rx = g.rot[0] * x + g.rot[1] * y + g.rot[2] * z + g.centre[0];
                ry = g.rot[3] * x + g.rot[4] * y + g.rot[5] * z + g.centre[1];
                rz = p.ndim == 3 ? g.rot[6] * x + g.rot[7] * y + g.rot[8] * z + g.centre[2] : 0.0;
              }
              // the first of the sample's two voxels along each axis, in the tile, and the fraction to the second one
              int ix = 0, iy = 0, iz = 0;
              float fx = 0.f, fy = 0.f, fz = 0.f;
              bool inside = true;
              if (interior) {
                const double gx = floor(rx), gy = floor(ry), gz = floor(rz);
                fx = static_cast<float>(rx - gx); fy = static_cast<float>(ry - gy);
                ix = static_cast<int>(gx) - t0[0]; iy = static_cast<int>(gy) - t0[1];
                if (TZ > 1) {
                  fz = static_cast<float>(rz - gz);
                  iz = static_cast<int>(gz) - t0[2];
                }
              } else {
                int hi;   // (the next voxel, or the same with a fraction of 0)
                inside = clamped_tap<float>(rz, p.D, iz, hi, fz, p.order) && clamped_tap<float>(ry, p.H, iy, hi, fy, p.order) &&
                         clamped_tap<float>(rx, p.W, ix, hi, fx, p.order);
                ix -= t0[0]; iy -= t0[1]; iz -= t0[2];
              }
              const auto in = [&](int i, int n, float w) { return inside && static_cast<unsigned>(i) < static_cast<unsigned>(n) && w != 0.f; };
              const float wx[2] = {1.f - fx, fx}, wy[2] = {1.f - fy, fy}, wz[2] = {1.f - fz, fz};
              const bool ox[2] = {in(ix, TX, wx[0]), in(ix + 1, TX, wx[1])}, oy[2] = {in(iy, TY, wy[0]), in(iy + 1, TY, wy[1])},
                         oz[2] = {in(iz, TZ, wz[0]), in(iz + 1, TZ, wz[1])};
              unsigned *const first_corner = column + ((iz * TY + iy) * TX + ix) * kOwnPitch;
              // (corners outside the tile, or of weight 0, add nothing to a place that exists: no branches)
#pragma unroll
              for (int c = 0; c < (TZ > 1 ? 8 : 4); c++) {
                const int bx_ = c & 1, by_ = (c >> 1) & 1, bz_ = c >> 2;
                const bool on = ox[bx_] && oy[by_] && oz[bz_];
                unsigned *const to = (on ? first_corner : aside) + ((bz_ * TY + by_) * TX + bx_) * kOwnPitch;
                const unsigned term = max(own_round(wz[bz_] * wy[by_] * wx[bx_] * quanta), 1u);
                __hip_atomic_fetch_add(to, on ? term : 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
              }
            }
          }
          columns += m; done += m; left -= m;
        }
      }
    };

    // the rois that reach the tile, a list at a time
    const int rois = part < p.R ? (p.R - part + parts - 1) / parts : 0;
    for (int base = 0; base < rois;) {
      __syncthreads();
      if (threadIdx.x == 0) { n_listed = 0; n_reaching = 0; next = 0; }
      __syncthreads();
      int have = 0;
      while (base < rois && have + kOwnTried * kOwnThreads <= kOwnRois) {
        float4 lo[kOwnTried], hi[kOwnTried];
#pragma unroll
        for (int i = 0; i < kOwnTried; i++) {
          const int r = part + parts * min(base + i * kOwnThreads + static_cast<int>(threadIdx.x), rois - 1);
          lo[i] = recs.first[r];
          hi[i] = recs.last[r];
        }
#pragma unroll
        for (int i = 0; i < kOwnTried; i++) {
          const int k = base + i * kOwnThreads + static_cast<int>(threadIdx.x);
          const bool hit = k < rois && __float_as_int(lo[i].w) == image && lo[i].x <= static_cast<float>(t0[0] + TX - 1) &&
                           lo[i].y <= static_cast<float>(t0[1] + TY - 1) && lo[i].z <= static_cast<float>(t0[2] + TZ - 1) &&
                           hi[i].x >= static_cast<float>(t0[0]) && hi[i].y >= static_cast<float>(t0[1]) && hi[i].z >= static_cast<float>(t0[2]);
          const unsigned long hits = __ballot(hit);
          unsigned at = 0;
          if (lane == 0 && hits) at = atomicAdd(&n_listed, static_cast<unsigned>(__popcll(hits)));
          at = __builtin_amdgcn_readfirstlane(at);
          if (hit) listed[at + __popcll(hits & ((1UL << lane) - 1))] = part + parts * k;
        }
        base += kOwnTried * kOwnThreads;
        __syncthreads();
        have = n_listed;
        __syncthreads();
      }
      have = __builtin_amdgcn_readfirstlane(have);
      if (have == 0) continue;
      if (!any) {
        any = true;
        for (unsigned i = 4 * threadIdx.x; i < kOwnWaves * kOwnVoxels * kOwnPitch; i += 4 * kOwnThreads)
          *reinterpret_cast<own_u32x4 *>(tables + i) = own_u32x4{0, 0, 0, 0};
        if (lane < kOwnColumns) rows[lane] = 0;
      }
      // the cells of a listed roi whose samples can reach the tile: a box of cells in the roi's own frame
      for (int i0 = wave * kWave; i0 < have; i0 += kOwnThreads) {
        bool hit = i0 + lane < have;
        unsigned r = 0, corner = 0, beyond = 0;
        if (hit) {
          r = listed[i0 + lane];
          const OwnBox b = recs.box[r];
#pragma unroll
          for (int j = 0; j < 3; j++) {
            if (j >= p.ndim) continue;
            const float last = static_cast<float>((j == 0 ? p.ow : j == 1 ? p.oh : p.od) - 1);
            float c = b.offset[j];
#pragma unroll
            for (int a = 0; a < 3; a++) c = fmaf(b.map[j][a], static_cast<float>(mid[a]), c);
            const float lo = fmaxf(ceilf(c - b.reach[j] - 1.f), 0.f), hi = fminf(floorf(c + b.reach[j]), last);
            if (lo <= hi) {
              corner |= static_cast<unsigned>(lo) << (10 * j);
              beyond |= static_cast<unsigned>(hi - lo) << (10 * j);
            } else {
              hit = false;
            }
          }
        }
        const unsigned long hits = __ballot(hit);
        unsigned at = 0;
        if (lane == 0 && hits) at = atomicAdd(&n_reaching, static_cast<unsigned>(__popcll(hits)));
        at = __builtin_amdgcn_readfirstlane(at);
        if (hit) {
          at += __popcll(hits & ((1UL << lane) - 1));
          reaching[at] = r; corners[at] = corner; beyonds[at] = beyond;
        }
      }
      __syncthreads();
      have = __builtin_amdgcn_readfirstlane(n_reaching);
      // A wavefront takes the next roi, and fetches its geometry, before it works on the one at hand; a record is loaded with
      // a double per lane and read from there (held by the scalar loads that the compiler makes of it otherwise, the sample
      // loop loads it again every time).
      auto take = [&](unsigned &n, unsigned &corner, unsigned &beyond, uint2 &rec) {
        unsigned at = 0;
        if (lane == 0) at = atomicAdd(&next, 1u);
        at = __builtin_amdgcn_readfirstlane(at);
        if (at >= static_cast<unsigned>(have)) return false;
        n = __builtin_amdgcn_readfirstlane(reaching[at]);
        corner = __builtin_amdgcn_readfirstlane(corners[at]);
        beyond = __builtin_amdgcn_readfirstlane(beyonds[at]);
        rec = reinterpret_cast<const uint2 *>(recs.geom + n)[min(lane, 23)];
        return true;
      };
      unsigned n, corner, beyond;
      uint2 rec;
      bool more = take(n, corner, beyond, rec);
      while (more) {
        RoiGeom g;
        auto from = [&](int i) {
          return __hiloint2double(__builtin_amdgcn_readlane(rec.y, i), __builtin_amdgcn_readlane(rec.x, i));
        };
#pragma unroll
        for (int i = 0; i < 9; i++) g.rot[i] = from(i);
#pragma unroll
        for (int a = 0; a < 3; a++) { g.centre[a] = from(9 + a); g.start[a] = from(12 + a); g.bin[a] = from(15 + a); g.sub[a] = from(18 + a); }
        g.grid[0] = __builtin_amdgcn_readlane(rec.x, 21); g.grid[1] = __builtin_amdgcn_readlane(rec.y, 21);
        g.grid[2] = __builtin_amdgcn_readlane(rec.x, 22); g.count = __builtin_amdgcn_readlane(rec.x, 23);
        const unsigned bits = __builtin_amdgcn_readlane(rec.y, kOwnPart / 2);
        const unsigned n0 = n, corner0 = corner, beyond0 = beyond;
        more = take(n, corner, beyond, rec);
        one_roi(g, bits, n0, corner0, beyond0);
      }
    }
    if (!any) break;
    if (columns > 0) multiply();
    float check = 0.f;
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
      for (int n = 0; n < 2; n++)
#pragma unroll
        for (int i = 0; i < 16; i++) check = fmaf(acc[m][n][i], 0.f, check);
    if (!careful && __ballot(!(check == 0.f)) != 0 && lane == 0) special = 1;
    __syncthreads();
    if (careful || special == 0) break;
  }

  if (!any && cleared) return;
  // each wavefront hands half of the tile's sums to the other and writes the other half
  static_assert(kOwnWaves == 2, "a half of the tile for each wavefront");
  float *const sums = reinterpret_cast<float *>(tables);
#pragma unroll
  for (int m = 0; m < 2; m++)
    if (any && wave != m) {
#pragma unroll
      for (int n = 0; n < 2; n++)
#pragma unroll
        for (int i = 0; i < 16; i++) sums[(m * 32 + n * 16 + i) * kWave + lane] = acc[m][n][i];
    }
  if (any) __syncthreads();
#pragma unroll
  for (int m = 0; m < 2; m++)
    if (wave == m) {
      if (any) {
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
          for (int i = 0; i < 16; i++) acc[m][n][i] += sums[(m * 32 + n * 16 + i) * kWave + lane];
      }
      if (parts == 1) {
        own_write<T, TX, TY, TZ>(grad, p, tile, m, acc[m]);
      } else {
        float *dst = partial + (static_cast<long>(id) * kOwnVoxels + m * 32) * kWave + lane;
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
          for (int i = 0; i < 16; i++) dst[(n * 16 + i) * kWave] = acc[m][n][i];
      }
    }
}

static unsigned own_groups(const RoiProblem &p) { return (p.C + kOwnChannels - 1) / kOwnChannels; }
static long own_tiles(const RoiProblem &p) {
  const int ty = p.ndim == 3 ? 4 : 8, tz = p.ndim == 3 ? 2 : 1;
  return static_cast<long>(p.N) * ((p.W + 7) / 8) * ((p.H + ty - 1) / ty) * ((p.D + tz - 1) / tz);
}
static size_t own_copy_bytes(int dtype, const RoiProblem &p) {
  return (static_cast<size_t>(p.R) * p.od * p.oh * p.ow * p.C * dtype_size(dtype) + 255) / 256 * 256;
}

// Workgroups that share a tile: small maps with many rois have too few tiles to fill the compute units (six workgroups each,
// and several rounds of them, since tiles differ in their rois), and every tile then has many rois; sixteen parts at
// most, of 16 rois at least.
static int own_parts(const RoiProblem &p) {
  const long wanted = 4096 / std::max(own_tiles(p) * static_cast<long>(own_groups(p)), 1L);
  return static_cast<int>(std::max(std::min({wanted, 16L, static_cast<long>(p.R / 16)}), 1L));
}
static size_t own_partial_bytes(const RoiProblem &p) {
  const int parts = own_parts(p);
  return parts > 1 ? static_cast<size_t>(own_tiles(p)) * own_groups(p) * parts * kOwnChannels * kOwnVoxels * sizeof(float) : 0;
}

// 16- and 32-bit tensors, orders 0 / 1, channels in whole 16-byte pieces (the copy's rows).
bool roi_own_applies(int dtype, const RoiProblem &p) {
  if (dtype != MV_F16 && dtype != MV_BF16 && dtype != MV_F32) return false;
  if ((p.order != 0 && p.order != 1) || p.C % (16 / static_cast<int>(dtype_size(dtype))) != 0) return false;
  const long cells = static_cast<long>(p.od) * p.oh * p.ow;
  if (cells > 1024 || p.R > 65535 || cells * p.R >= (1L << 31)) return false;
  // A table costs the same for one channel as for 64 of a group, and fp32 products are eight times as long as fp16 ones: where
  // cells are smaller than voxels (one sample each, dozens of them in a tile) and channels few, the kernel that sums roi by
  // roi is the faster one.  [1,C,17,28,45], training steps of n rois of 7^3 cells, that kernel -> this one: fp16, C = 16, 300
  // rois (5 cells per voxel) 147 -> 112 us, 700 163 -> 177; C = 32, 1490 410 -> 318; fp32, C = 32, 60 140 -> 110, 1490 415 ->
  // 453; C = 64, 1490 789 -> 712.
  const double per_voxel = static_cast<double>(cells) * p.R / (static_cast<double>(p.N) * p.D * p.H * p.W);
  if (p.ndim == 3 && (dtype == MV_F32 ? p.C < 64 && per_voxel > 2.0 : p.C < 32 && per_voxel > 8.0)) return false;
  // Rois far apart on a large fp32 map with one sample a cell (or an adaptive grid, which often is one): most of the time is the
  // writing of zeros, and the fill before the atomics does that faster.  What the atomics cost is the voxels of the boxes, whatever their
  // cells, so the line is in rois per voxel: of 46 drawn training steps with boxes of 1 - 24 voxels all 28 from 1 / 1600 on are faster here, 1.05 -
  // 2.6 times ([2,256,17,72,115], 760 rois of 4^3 cells, 750 -> 481 us; [4,128,36,120,39], 347 of 7^3, 867 -> 739; [4,32,31,61,109], 1012 of
  // 5^3, 459 -> 323), those below 1 / 2000 mostly not ([4,128,28,55,117], 231 of 7^3, 467 -> 520; [4,256,37,107,87], 266 of 5^3, 1276 -> 1484).
  // The error against 64 bits is a third (1.0e-7 and 3.2e-7, six of them).
  const double voxels = static_cast<double>(p.N) * p.D * p.H * p.W;
  if (p.ndim == 3 && dtype == MV_F32 && p.sampling_ratio < 2 && per_voxel < 0.25 && p.R * 1600.0 < voxels && own_tiles(p) * own_groups(p) > 4096)
    return false;
  return own_tiles(p) * own_groups(p) < (1L << 31) - 8 && cells * p.R / 32 * own_groups(p) < (1L << 30);
}

size_t roi_own_workspace(int dtype, const RoiProblem &p) {
  return roi_own_applies(dtype, p) ? own_copy_bytes(dtype, p) + own_partial_bytes(p) + static_cast<size_t>(p.R) * kOwnRoiBytes : 0;
}

// Writes all of grad_input.  -1: not for these kernels, or a workspace that is too small for them.
int roi_own_backward(const void *grad_output, const void *rois, void *grad_input, int dtype, const RoiProblem &p, void *workspace,
                     size_t capacity, hipStream_t s) {
  if (!roi_own_applies(dtype, p) || capacity < roi_own_workspace(dtype, p)) return -1;
  const int es = static_cast<int>(dtype_size(dtype));
  char *const after = static_cast<char *>(workspace) + own_copy_bytes(dtype, p);
  float *const partial = reinterpret_cast<float *>(after);
  OwnRois recs;
  recs.geom = reinterpret_cast<RoiGeom *>(after + own_partial_bytes(p));
  recs.box = reinterpret_cast<OwnBox *>(recs.geom + p.R);
  recs.first = reinterpret_cast<float4 *>(recs.box + p.R);
  recs.last = recs.first + p.R;
  const unsigned pblocks = (p.od * p.oh * p.ow + kMovePos - 1) / kMovePos;
  const int parts = own_parts(p);
  // A tile's rows are 16 or 32 bytes and reach 2 TB/s at best.  Where nearly all tiles have no roi (one meets some 20 of them) a
  // streaming fill, in the launch of the layouts, is the faster way to their zeros: 16 rois on [4,128,36,101,44] fp32 170 -> 151
  // us, fp16 104 -> 81; 120 rois (47 tiles a roi) fp32 256 -> 275.
  const bool clear = parts == 1 && 64L * p.R <= own_tiles(p);
  const long elements = clear ? static_cast<long>(p.N) * p.C * p.D * p.H * p.W : 0, block_elements = 256L * kOwnClearPieces * (16 / es);
  const unsigned moves = pblocks * p.R * ((p.C * es + 127) / 128);
  const unsigned blocks = moves + (p.R + 255) / 256 + static_cast<unsigned>((elements + block_elements - 1) / block_elements);
  const float *const r = static_cast<const float *>(rois);
  if (es == 2)
    hipLaunchKernelGGL((roi_own_layout_kernel<unsigned short>), dim3(blocks), dim3(256), 0, s, static_cast<const unsigned short *>(grad_output),
                       static_cast<unsigned short *>(workspace), r, recs, p, pblocks, moves,
                       static_cast<unsigned short *>(grad_input), elements);
  else
    hipLaunchKernelGGL((roi_own_layout_kernel<unsigned int>), dim3(blocks), dim3(256), 0, s, static_cast<const unsigned int *>(grad_output),
                       static_cast<unsigned int *>(workspace), r, recs, p, pblocks, moves,
                       static_cast<unsigned int *>(grad_input), elements);
  int st = check_launch("roi_own_layout_kernel");
  if (st) return st;
  const int groups = static_cast<int>(own_groups(p));
  const unsigned tiles = static_cast<unsigned>(own_tiles(p) * groups), total = tiles * parts;
  const dim3 grid((total + 7) / 8 * 8), block(kOwnThreads);
#define MV_OWN_AS(TYPE, ROTV, TY, TZ)                                                                                   \
  do {                                                                                                                 \
    const int nx = (p.W + 7) / 8, ny = (p.H + TY - 1) / TY, nz = (p.D + TZ - 1) / TZ;                                    \
    hipLaunchKernelGGL((roi_own_backward_kernel<TYPE, ROTV, 8, TY, TZ>), grid, block, 0, s, static_cast<const TYPE *>(workspace), recs, \
                       static_cast<TYPE *>(grad_input), p, nx, ny, nz, groups, total, parts, clear, partial);           \
    if (parts > 1)                                                                                                     \
      hipLaunchKernelGGL((roi_own_fold_kernel<TYPE, 8, TY, TZ>), dim3(tiles), block, 0, s, partial, static_cast<TYPE *>(grad_input), p, \
                         nx, ny, nz, groups, parts);                                                                   \
  } while (0)
#define MV_OWN(TYPE)                                                                                                    \
  do {                                                                                                                 \
    if (p.ndim == 3) { if (p.rotated) MV_OWN_AS(TYPE, true, 4, 2); else MV_OWN_AS(TYPE, false, 4, 2); }                  \
    else { if (p.rotated) MV_OWN_AS(TYPE, true, 8, 1); else MV_OWN_AS(TYPE, false, 8, 1); }                              \
  } while (0)
  switch (dtype) {
    case MV_F32: MV_OWN(float); break;
    case MV_F16: MV_OWN(__half); break;
    default: MV_OWN(__hip_bfloat16);
  }
#undef MV_OWN
#undef MV_OWN_AS
  return check_launch("roi_own_backward_kernel");
}

}  // namespace mv
