// RoIAlign heads on IMAGES with plain boxes and small outputs (up to 16 x 16 cells per roi): forward and backward.
// Results as the reference's csrc/cuda/roi_align_2d_cuda_kernel.cuh:11-180; fp32 arithmetic for every type.
//
// Both passes use that the samples of a plain box are separable: a pixel's weight in a cell is wy[cell row] *
// wx[cell column], each the sum over the cell's samples on that axis, so that with G = the 7 x 7 cells of a channel
//     forward  G = Wy box Wx^T,        backward  box += Wy^T G Wx
// are two small matrix products per channel each.  They run on the fp32 matrix cores (16 x 16 x 4, exact fp32
// products and sums), the first one on the 16-bit ones where the pixels or gradients are 16-bit (PlaneHalf).  A dense product gives 0 x infinity for a pixel or gradient that no sample's weight reaches, so
// sums that come out not finite are formed again without the terms of weight 0 (one test per finished sum; the second
// pass runs for such channels and tiles alone).  The accumulator of the first product is the right-hand operand of the second as it stands:
// lane l holds column l % 16 and the four rows 4 (l / 16) + r, and a product's step r takes K = one row per lane
// group, so a suitable order of the rows (that is: of the lanes' loads) is all the second product needs - no
// LDS, no exchange between lanes.
//
// Forward, one workgroup = (roi, some channels): the pixels that some sample touches are listed per axis (rows one by
// one, columns in groups of four), so that large rois with a small sampling grid read only what they use.  A lane's
// piece of a 16 x 16 piece of the box is one 16-byte load (16-bit tensors: 8 bytes), straight from the feature map.
//   (1000 rois of 4 - 64 pixels, adaptive grid, 256 channels, 7 x 7 cells, fp32, [2, 256, 200, 304]: 480 us when the
//   boxes went through LDS and three barriers per chunk of channels; 157 us now, matrix cores 42 % and texture addressers 58 % busy (168 us
//   with a channel per product).  fp16, 1613 rois of 3 - 25 pixels x 256 channels: 147 us with a channel per fp32 product, 122 us with
//   two, 108 us with the first product on the 16-bit cores.)
//
// Backward, one workgroup = (16 x 16 pixels, some channels): it looks up the rois that touch its pixels, works out
// its pixels' weights for eight rois at a time and adds roi after roi into accumulators that stay in registers.  No
// atomics, no fp32 copy of the gradient, every pixel written once, sums in the order of the rois.
//   (The same head: 1030 us with one atomic per touched pixel, roi and channel; 147 us now: matrix cores 51 %, vector issue 32 %.  16-bit
//   gradients, 14 x 14 cells: fp16 1499 rois x 256 channels 304 us with fp32 products, 207 us; bf16 1689 x 128 207 us, 143 us.)
// What bounds them: the matrix cores (three 32-clock instructions per roi, tile and channel backward, eight with 16 cells; 4 x pieces + 2
// per row piece and channel forward, + 4 with 16 cells; a first product of 16-bit values takes a quarter, forward, or less) and the latency of the loads.
#include <algorithm>

#include "common.hpp"
#include "roi_geometry.hpp"
#include "sampling.hpp"

namespace mv {

constexpr int kPlaneThreads = 256, kPlaneWaves = kPlaneThreads / kWave;
constexpr int kPlaneTile = 16;       // pixels per side of a matrix piece
constexpr unsigned kPlaneNowhere = 0x80000000u;   // beyond every buffer: the load returns zeros
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned plane_u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t plane_product(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Values of a 16-bit tensor, as they are stored, times fp32 weights, on the 16-bit matrix cores: a weight is the sum of
// three 16-bit parts, which stand next to each other in K against the same values.  Every product is exact in fp32, and
// the parts hold the weight's 24 bits (bf16) or leave less than 2^-28 (fp16, whose weights, at most 1, are kept times 2^14).
// All products of a sum are 16 x 16 x 32 ones: where a 16 x 16 x 16 one took the result of a 16 x 16 x 32 one as its third
// operand, the compiler left no wait between them, and it read the old registers.
template <typename T> struct PlaneHalf;
template <> struct PlaneHalf<__half> {
  using E = _Float16;
  static constexpr float kScale = 16384.f;
  typedef _Float16 v4 __attribute__((ext_vector_type(4)));
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4_t product(v8 a, v8 b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <> struct PlaneHalf<__hip_bfloat16> {
  using E = __bf16;
  static constexpr float kScale = 1.f;
  typedef __bf16 v4 __attribute__((ext_vector_type(4)));
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4_t product(v8 a, v8 b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
template <> struct PlaneHalf<float> { static constexpr float kScale = 1.f; };

// One axis of a plain roi: v(cell, sub) = start + cell * bin + (sub + .5) * step (local_coord's expression)
struct PlaneAxis {
  double start, bin, step, inv_step, inv_grid;
  int cells, grid, size;
  __device__ __forceinline__ void set(float lo_, float hi_, double scale, int cells_, int ratio, int size_) {
    const double lo = static_cast<double>(lo_) * scale, hi = static_cast<double>(hi_) * scale;
    const double ext = fmax(hi - lo, 1.0);
    start = lo;
    cells = cells_;
    size = size_;
    grid = ratio > 0 ? ratio : static_cast<int>(ceil(ext / static_cast<double>(cells_)));
    bin = ext / static_cast<double>(cells_);
    step = bin / static_cast<double>(grid > 0 ? grid : 1);
    inv_step = 1.0 / step;
    inv_grid = 1.0 / static_cast<double>(grid > 0 ? grid : 1);
  }
  __device__ __forceinline__ double at(int cell, int sub) const {
    return start + cell * bin + static_cast<double>(static_cast<float>(sub) + .5f) * step;
  }
  // w[cell] = sum of the weights that the cell's samples give to pixel x (1 / grid included); true when there is one
  template <int CELLS>
  __device__ __forceinline__ bool pixel_weights(int x, int order, float *w) const {
#pragma unroll
    for (int k = 0; k < CELLS; k++) w[k] = 0.f;
    // samples within one pixel of x (towards a border: up to the end of the closed interval), one more on either side
    const double entries = static_cast<double>(cells) * grid;
    const double from = x == 0 ? -1.0 : x - 1.0, to = x == size - 1 ? static_cast<double>(size) : x + 1.0;
    const double e0 = fmax(floor((from - start) * inv_step - 0.5) - 1.0, 0.0);
    const double e1 = fmin(ceil((to - start) * inv_step - 0.5) + 1.0, entries - 1.0);
    if (!(e0 <= e1)) return false;   // (also when the roi holds NaN)
    const float inv = static_cast<float>(inv_grid);
    int cell = static_cast<int>((e0 + 0.5) * inv_grid), sub = static_cast<int>(e0 - static_cast<double>(cell) * grid);
    float sum = 0.f;   // of the current cell
    bool any = false;
    for (int left = static_cast<int>(e1 - e0); left >= 0; left--) {
      int lo, hi;
      float f;
      if (clamped_tap<float>(at(cell, sub), size, lo, hi, f, order))
        sum += (lo == x ? (1.f - f) * inv : 0.f) + (hi == x ? f * inv : 0.f);
      if (++sub == grid || left == 0) {
        if (sum != 0.f) {
          w[cell] = sum;
          any = true;
        }
        sum = 0.f;
        sub = 0;
        cell++;
      }
    }
    return any;
  }
};

// N neighbouring elements, 2 or 4
template <typename T, int N> struct PlaneCells { T v[N]; };
template <typename T, int N> __device__ __forceinline__ PlaneCells<T, N> plane_load_cells(__amdgpu_buffer_rsrc_t rsrc, unsigned off, int soff) {
  PlaneCells<T, N> r;
  if constexpr (sizeof(T) * N == 4) {
    const auto w = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, soff, 0);
    __builtin_memcpy(&r, &w, 4);
  } else if constexpr (sizeof(T) * N == 8) {
    const auto w = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, soff, 0);
    __builtin_memcpy(&r, &w, 8);
  } else {
    const auto w = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, soff, 0);
    __builtin_memcpy(&r, &w, 16);
  }
  return r;
}

template <typename T> __device__ __forceinline__ void plane_store(__amdgpu_buffer_rsrc_t rsrc, unsigned off, int soff, float v) {
  const T t = store_cast<T>(v);
  if constexpr (sizeof(T) == 2) {
    unsigned short w;
    __builtin_memcpy(&w, &t, 2);
    __builtin_amdgcn_raw_buffer_store_b16(w, rsrc, off, soff, 0);
  } else {
    unsigned w;
    __builtin_memcpy(&w, &t, 4);
    __builtin_amdgcn_raw_buffer_store_b32(w, rsrc, off, soff, 0);
  }
}

// Launch order of the forward pass: rois by image and place, so that the workgroups of an XCD (a contiguous eighth of the
// order) read overlapping boxes at about the same time from one L2.  In the order of the rois every box came from
// beyond the L2s (960 MB for the head above, at the 5 TB/s of a copy).  One workgroup, a counting sort; the order inside
// a bucket is whatever the atomics give (it changes the schedule, not the results).
constexpr int kPlaneBuckets = 1024, kPlaneSizes = 16, kPlaneOrderMax = 16384;
__global__ __launch_bounds__(1024) void roi_plane_order_kernel(const float *__restrict__ rois, unsigned *__restrict__ order,
                                                               const RoiProblem p, const int side) {
  __shared__ unsigned count[kPlaneBuckets], start[kPlaneBuckets];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  auto bucket = [&](int i) {
    const float *r = rois + static_cast<long>(i) * 5;
    const float scale = 0.5f * static_cast<float>(p.scale) * side;
    const int bx = static_cast<int>(fminf(fmaxf((r[1] + r[3]) * scale / p.W, 0.f), side - 1.f));
    const int by = static_cast<int>(fminf(fmaxf((r[2] + r[4]) * scale / p.H, 0.f), side - 1.f));
    const int b = static_cast<int>(fminf(fmaxf(r[0], 0.f), p.N - 1.f));
    // largest boxes first: steps of a factor of two
    const float area = fmaxf((r[3] - r[1]) * static_cast<float>(p.scale) + 2.f, 3.f) * fmaxf((r[4] - r[2]) * static_cast<float>(p.scale) + 2.f, 3.f);
    const int size = static_cast<int>(fminf(fmaxf(16.f - log2f(area), 0.f), kPlaneSizes - 1.f));
    return size * (kPlaneBuckets / kPlaneSizes) + (b * side + by) * side + bx;
  };
  count[tid] = 0;
  __syncthreads();
  for (int i = tid; i < p.R; i += 1024) atomicAdd(&count[bucket(i)], 1u);
  __syncthreads();
  {   // exclusive sums: within the wavefront, then over the wavefronts
    __shared__ unsigned total[16];
    const unsigned mine = count[tid];
    unsigned sum = mine;
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) {
      const unsigned up = __shfl_up(sum, d);
      if (lane >= d) sum += up;
    }
    if (lane == kWave - 1) total[wave] = sum;
    __syncthreads();
    unsigned before = 0;
    for (int w = 0; w < wave; w++) before += total[w];
    start[tid] = before + sum - mine;
  }
  __syncthreads();
  for (int i = tid; i < p.R; i += 1024) order[atomicAdd(&start[bucket(i)], 1u)] = static_cast<unsigned>(i);
}

// ---- forward ---------------------------------------------------------------------------------------
constexpr int kPlaneRows = 128, kPlaneGroups = 32;   // listed rows, groups of four columns
constexpr int kPlaneAtOnce = 4, kPlaneSteps = 4;     // channels of a step, steps loaded or in flight
constexpr int kPlaneChannels = 256;                  // of a workgroup at most

template <typename T, int CELLS>
__global__ __launch_bounds__(kPlaneThreads, 4) void roi_plane_forward_kernel(const T *__restrict__ feat,
                                                                             const float *__restrict__ rois, T *__restrict__ out,
                                                                             const RoiProblem p, const int channels_per_block,
                                                                             const unsigned *__restrict__ order) {
  constexpr int PITCH = CELLS + 1, ES = sizeof(T);
  __shared__ float wy[kPlaneRows][PITCH];            // listed row, cell row
  __shared__ float wx[4 * kPlaneGroups][PITCH];      // column of a listed group, cell column
  __shared__ int row_of[kPlaneRows], column_of[kPlaneGroups];
  __shared__ float pixel[2][kWave][PITCH];           // weights of the pixels being listed
  __shared__ int count[2];
  const unsigned cblocks = (p.C + channels_per_block - 1) / channels_per_block;
  const unsigned id = blockIdx.x, n = order ? order[id / cblocks] : id / cblocks;
  const int c_begin = (id % cblocks) * channels_per_block, c_count = min(channels_per_block, p.C - c_begin);
  const float *roi = rois + static_cast<long>(n) * 5;
  const int tid = threadIdx.x, lane = tid % kWave, cells = p.oh * p.ow;
  T *dst = out + (static_cast<long>(n) * p.C + c_begin) * cells;
  const int b = __builtin_amdgcn_readfirstlane(static_cast<int>(roi[0]));
  const bool image = b >= 0 && b < p.N;
  const long plane = static_cast<long>(p.H) * p.W;
  const T *src = feat + (static_cast<long>(image ? b : 0) * p.C + c_begin) * plane;
  if (tid < 2) count[tid] = image ? 0 : -1;
  for (int i = tid; i < kPlaneRows * PITCH; i += kPlaneThreads) (&wy[0][0])[i] = 0.f;
  for (int i = tid; i < 4 * kPlaneGroups * PITCH; i += kPlaneThreads) (&wx[0][0])[i] = 0.f;
  __syncthreads();
  if (image && tid < 2 * kWave) {
    // wavefront 0 lists the columns, wavefront 1 the rows: 64 pixels of the box at a time
    const int axis = tid / kWave;
    PlaneAxis A;
    A.set(roi[1 + axis], roi[3 + axis], p.scale, axis == 0 ? p.ow : p.oh, p.sampling_ratio, axis == 0 ? p.W : p.H);
    int listed = 0;
    if (A.grid > 0) {
      const double first = A.at(0, 0), last = A.at(A.cells - 1, A.grid - 1);
      if (last >= -1.0 && first <= A.size) {
        const int lo = static_cast<int>(fmin(fmax(floor(first), 0.0), A.size - 1.0));
        const int hi = static_cast<int>(fmin(fmax(floor(last) + 1.0, 0.0), A.size - 1.0));
        const int room = axis == 0 ? kPlaneGroups : kPlaneRows;
        for (int x0 = lo; x0 <= hi && listed <= room; x0 += kWave) {
          const int x = x0 + lane;
          float *w = pixel[axis][lane];
          const bool any = x <= hi && A.template pixel_weights<CELLS>(x, p.order, w);
          const unsigned long long touched = __ballot(any);
          if (axis == 0) {
            // a group starts at every fourth column of the box; the image's last one is moved back into the row
            unsigned long long groups = touched | (touched >> 1);
            groups = (groups | (groups >> 2)) & 0x1111111111111111ull;
            const int mine = lane & ~3, k = listed + __popcll(groups & ((1ull << mine) - 1));
            if (((groups >> mine) & 1) && k < room) {
              const int start = min(x0 + mine, p.W - 4);
              if (lane == mine) column_of[k] = start;
              if (any)
                for (int c = 0; c < CELLS; c++) wx[4 * k + x - start][c] = w[c];
            }
            listed += __popcll(groups);
          } else {
            const int k = listed + __popcll(touched & ((1ull << lane) - 1));
            if (any && k < room) {
              row_of[k] = x;
              for (int c = 0; c < CELLS; c++) wy[k][c] = w[c];
            }
            listed += __popcll(touched);
          }
        }
      }
    }
    if (lane == 0) count[axis] = listed;
  }
  __syncthreads();
  const int groups = __builtin_amdgcn_readfirstlane(count[0]), rows = __builtin_amdgcn_readfirstlane(count[1]);
  if (groups <= 0 || rows <= 0) {   // no sample touches the image
    for (int i = tid; i < c_count * cells; i += kPlaneThreads) dst[i] = store_cast<T>(0.f);
    return;
  }
  if (groups > kPlaneGroups || rows > kPlaneRows || p.W < 4) {
    // more pixels than the lists hold: every output walks its samples
    PlaneAxis X, Y;
    X.set(roi[1], roi[3], p.scale, p.ow, p.sampling_ratio, p.W);
    Y.set(roi[2], roi[4], p.scale, p.oh, p.sampling_ratio, p.H);
    const float samples = static_cast<float>(X.grid) * static_cast<float>(Y.grid);
    for (int i = tid; i < c_count * cells; i += kPlaneThreads) {
      const int c = i / cells, r = i - c * cells, ph = r / p.ow, pw = r - ph * p.ow;
      float acc = 0.f;
      for (int iy = 0; iy < Y.grid; iy++)
        for (int ix = 0; ix < X.grid; ix++)
          acc += sample_clamped<T>(src + c * plane, 1, p.H, p.W, 0.0, Y.at(ph, iy), X.at(pw, ix), p.order);
      dst[i] = store_cast<T>(acc / samples);
    }
    return;
  }
  constexpr int PAIR = 16 / CELLS, SUMS = kPlaneAtOnce / PAIR;   // channels side by side in the columns of the products
  const int m = lane % 16, q = lane / 16, mc = m % CELLS, mine = m / CELLS;   // the lane's cell and its channel of the pair
  const bool cell_lane = m < CELLS;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int y_pieces = (rows + 15) / 16, x_pieces = (groups + 3) / 4;
  const int plane_bytes = static_cast<int>(plane) * ES;   // < 2^27, checked by the host
  // The steps (channels, row piece, column piece) of the wavefront form one sequence; a step's loads are issued a few
  // steps ahead.  (Every step issues the same number of loads, beyond the last one to nowhere, so that the wait
  // for a step's loads leaves the later ones' in flight.)
  struct Step { int c0, yp, xp; };
  auto next_of = [&](Step st) {
    if (++st.xp == x_pieces) {
      st.xp = 0;
      if (++st.yp == y_pieces) { st.yp = 0; st.c0 += kPlaneWaves * kPlaneAtOnce; }
    }
    return st;
  };
  auto issue = [&](PlaneCells<T, 4> (&v)[kPlaneAtOnce], const Step &st) {
    // (channels beyond the last one: zeros; the clamp is a vector instruction, so its result goes back to a scalar)
    const int cs = min(kPlaneAtOnce, c_count - st.c0);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T *>(src + static_cast<long>(cs > 0 ? st.c0 : 0) * plane), 0,
        __builtin_amdgcn_readfirstlane(max(cs, 0) * plane_bytes), 0x00020000);
    const int row = st.yp * 16 + m, g = st.xp * 4 + q;
    const unsigned off = row < rows && g < groups ? static_cast<unsigned>((row_of[row] * p.W + column_of[g]) * ES) : kPlaneNowhere;
#pragma unroll
    for (int c = 0; c < kPlaneAtOnce; c++) v[c] = plane_load_cells<T, 4>(rsrc, off, c * plane_bytes);
  };
  f32x4_t sum[SUMS], t[SUMS];
  static_assert(kPlaneChannels <= 32 * kPlaneWaves * kPlaneAtOnce, "a bit for each of the wavefront's groups of channels");
  unsigned special = 0;   // the groups whose sums are not finite
  unsigned out_off[4];   // the lane's four outputs of a channel
#pragma unroll
  for (int r = 0; r < 4; r++)
    out_off[r] = mc < p.ow && 4 * q + r < p.oh ? static_cast<unsigned>((mine * cells + (4 * q + r) * p.ow + mc) * ES) : kPlaneNowhere;
  auto columns = [&](const PlaneCells<T, 4> (&v)[kPlaneAtOnce], const Step &st, auto first) {
    const int g = st.xp * 4 + q;
    // (of two channels, the weights meet the first one in columns 0 - 7 and the second one in columns 8 - 15)
    if constexpr (ES == 2) {
      using H = PlaneHalf<T>;
      typename H::v8 part[2][PAIR];   // first and second parts; third parts
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float w = g < groups ? wx[4 * g + u][mc] * H::kScale : 0.f;
        const typename H::E first_part = static_cast<typename H::E>(w);
        const float left = w - static_cast<float>(first_part);
        const typename H::E second_part = static_cast<typename H::E>(left);
        const typename H::E third_part = static_cast<typename H::E>(left - static_cast<float>(second_part));
#pragma unroll
        for (int i = 0; i < PAIR; i++) {
          const typename H::E none = static_cast<typename H::E>(0.f);
          part[0][i][u] = mine == i ? first_part : none;
          part[0][i][4 + u] = mine == i ? second_part : none;
          part[1][i][u] = mine == i ? third_part : none;
          part[1][i][4 + u] = none;
        }
      }
#pragma unroll
      for (int k = 0; k < 2; k++)
#pragma unroll
        for (int i = 0; i < PAIR; i++)
#pragma unroll
          for (int c = 0; c < SUMS; c++) {
            const typename H::v4 a = __builtin_bit_cast(typename H::v4, v[c * PAIR + i]);
            t[c] = H::product(__builtin_shufflevector(a, a, 0, 1, 2, 3, 0, 1, 2, 3), part[k][i],
                              decltype(first)::value && k == 0 && i == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : t[c]);
          }
    } else {
      float bx[PAIR][4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float w = g < groups ? wx[4 * g + u][mc] : 0.f;
#pragma unroll
        for (int i = 0; i < PAIR; i++) bx[i][u] = mine == i ? w : 0.f;
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int i = 0; i < PAIR; i++)
#pragma unroll
          for (int c = 0; c < SUMS; c++)
            t[c] = plane_product(load(&v[c * PAIR + i].v[u]), bx[i][u],
                                 decltype(first)::value && u == 0 && i == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : t[c]);
    }
  };
  auto row_sums = [&](const Step &st, auto first) {
    // register r of lane group q: listed row 16 yp + 4 q + r
    float ay[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int k = st.yp * 16 + 4 * q + r;
      ay[r] = cell_lane && k < rows ? wy[k][mc] * (1.f / PlaneHalf<T>::kScale) : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int c = 0; c < SUMS; c++)
        sum[c] = plane_product(ay[r], t[c][r], decltype(first)::value && r == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : sum[c]);
  };
  auto products = [&](const PlaneCells<T, 4> (&v)[kPlaneAtOnce], const Step &st) {
    if (st.xp == 0) columns(v, st, std::true_type{});
    else columns(v, st, std::false_type{});
    if (st.xp + 1 < x_pieces) return;
    if (st.yp == 0) row_sums(st, std::true_type{});
    else row_sums(st, std::false_type{});
    if (st.yp + 1 < y_pieces) return;
    float check = 0.f;   // stays zero unless a sum is infinite or NaN
#pragma unroll
    for (int c = 0; c < SUMS; c++)
#pragma unroll
      for (int r = 0; r < 4; r++) check = fmaf(sum[c][r], 0.f, check);
    if (__ballot(!(check == 0.f)) != 0) {
      special |= 1u << (st.c0 / (kPlaneWaves * kPlaneAtOnce));
      return;
    }
    const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(
        dst + static_cast<long>(st.c0) * cells, 0,
        __builtin_amdgcn_readfirstlane(min(kPlaneAtOnce, c_count - st.c0) * cells * ES), 0x00020000);
#pragma unroll
    for (int c = 0; c < SUMS; c++)   // (channels beyond the last one are beyond the buffer)
#pragma unroll
      for (int r = 0; r < 4; r++) plane_store<T>(to, out_off[r], c * PAIR * cells * ES, sum[c][r]);
  };
  // kPlaneSteps sets of load registers used in turn: the loads of the next kPlaneSteps - 1 steps are in flight
  Step step[kPlaneSteps];
  PlaneCells<T, 4> v[kPlaneSteps][kPlaneAtOnce];
  step[0] = Step{wave * kPlaneAtOnce, 0, 0};
#pragma unroll
  for (int u = 0; u + 1 < kPlaneSteps; u++) {
    issue(v[u], step[u]);
    step[u + 1] = next_of(step[u]);
  }
  while (step[0].c0 < c_count) {
#pragma unroll
    for (int u = 0; u < kPlaneSteps; u++) {
      issue(v[(u + kPlaneSteps - 1) % kPlaneSteps], step[(u + kPlaneSteps - 1) % kPlaneSteps]);
      if (step[u].c0 < c_count) products(v[u], step[u]);
      step[u] = next_of(step[(u + kPlaneSteps - 1) % kPlaneSteps]);
    }
  }
  for (; special != 0; special &= special - 1) {   // again, output by output, without the pixels of weight 0
    const int c0 = (__builtin_ctz(special) * kPlaneWaves + wave) * kPlaneAtOnce, outputs = min(kPlaneAtOnce, c_count - c0) * cells;
    for (int i = lane; i < outputs; i += kWave) {
      const int c = i / cells, r = i - c * cells, ph = r / p.ow, pw = r - ph * p.ow;
      const T *from = src + (c0 + c) * plane;
      float acc = 0.f;
      for (int k = 0; k < rows; k++) {
        if (wy[k][ph] == 0.f) continue;
        const T *row = from + static_cast<long>(row_of[k]) * p.W;
        float along = 0.f;
        for (int x = 0; x < 4 * groups; x++)
          if (wx[x][pw] != 0.f) along = fmaf(wx[x][pw], load(row + column_of[x / 4] + x % 4), along);
        acc = fmaf(wy[k][ph], along, acc);
      }
      dst[c0 * cells + i] = store_cast<T>(acc);
    }
  }
}

// ---- backward ----------------------------------------------------------------------------------------
constexpr int kPlaneAhead = 2;      // rois whose gradients are loaded or in flight
constexpr int kPlaneBatch = 8;      // rois whose pixel weights are worked out together
constexpr int kPlaneQueue = 1024;   // rois looked through at a time
constexpr int kPlaneBackwardChannels = 8;   // of a wavefront

// A wavefront has CH channels of the tile.  SPLIT: several workgroups share a tile's rois (few tiles, many rois) and
// add to the fp32 buffer `acc`; otherwise a pixel is written once, to `grad` (added to what is there when
// `accumulate`).
template <typename T, int CELLS, int CH, bool SPLIT>
__global__ __launch_bounds__(kPlaneThreads, CELLS == 8 ? 4 : 2) void roi_plane_backward_kernel(
    const T *__restrict__ gout, const float *__restrict__ rois, T *__restrict__ grad, float *__restrict__ acc_buffer,
    const RoiProblem p, const int tiles_x, const int tiles_y, const int accumulate) {
  constexpr int PITCH = CELLS + 1, ES = sizeof(T);
  constexpr int STEPS = CELLS / 4;                  // K steps of four cells
  constexpr int PER = 16 / CELLS;                   // channels per first product: rows (channel, cell row)
  constexpr int PIECES = CH / PER;                  // first products (and loads) per roi
  __shared__ float weights[kPlaneBatch][2][kPlaneTile][PITCH];   // roi, axis, pixel, cell
  __shared__ unsigned queue[kPlaneQueue];
  __shared__ int wave_count[kPlaneQueue / kWave];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  // (neighbouring tiles, which share rois, on one XCD: its L2 then holds their gradients)
  const int id = static_cast<int>(xcd_contiguous(blockIdx.x, gridDim.x)), tile = id % (tiles_x * tiles_y), image = id / (tiles_x * tiles_y);
  const int x0 = (tile % tiles_x) * kPlaneTile, y0 = (tile / tiles_x) * kPlaneTile;
  const int c0 = (blockIdx.y * kPlaneWaves + wave) * CH, c_count = min(CH, p.C - c0);   // (may be <= 0: nothing to load or store)
  const int cells = p.oh * p.ow;
  const int m = lane % 16, q = lane / 16;
  const int parts = gridDim.z, part = blockIdx.z;
  f32x4_t acc[CH];
#pragma unroll
  for (int c = 0; c < CH; c++) acc[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // The row of the first product's left operand that this lane loads, row 4 a + r: the accumulator leaves it in lane
  // group a, register r, where the second product wants cell row a + 4 s of a channel in step s.  Its STEPS cells, one
  // per K step, are neighbours: one load.
  const int a = m / 4, r_of = m % 4, ph = CELLS == 8 ? a + 4 * (r_of % 2) : a + 4 * r_of, c_of = CELLS == 8 ? r_of / 2 : 0;
  const int pw = q * STEPS;
  const int have = p.ow - pw;   // cells of the load that belong to the row
  // (16-bit tensors: a word that begins within the gradients and ends beyond them reads as zero, so the last row's last
  // load is moved back to end with the row, and its cells down by as many places)
  const int back = ES == 2 && ph == p.oh - 1 && have > 0 && have < STEPS ? STEPS - have : 0;
  const unsigned off = ph < p.oh && pw < p.ow ? static_cast<unsigned>((c_of * cells + ph * p.ow + pw - back) * ES) : kPlaneNowhere;
  const int pair_bytes = PER * cells * ES;
  // (the minimum and maximum become one vector instruction, after which the compiler takes the descriptor for divergent
  // and wraps every load in a loop over the lanes: back to a scalar)
  const int roi_bytes = __builtin_amdgcn_readfirstlane(max(c_count, 0) * cells * ES);
  auto fetch = [&](PlaneCells<T, STEPS> (&v)[PIECES], unsigned roi) {
    const T *g = gout + (static_cast<long>(roi) * p.C + c0) * cells;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(g), 0, roi_bytes, 0x00020000);
#pragma unroll
    for (int i = 0; i < PIECES; i++) v[i] = plane_load_cells<T, STEPS>(rsrc, off, i * pair_bytes);
  };
  // (a load that reaches past its row of cells brings the next row's, channel's or roi's: cleared, 0 x inf is not 0)
  using Bits = typename std::conditional<ES * STEPS == 4, unsigned, unsigned long long>::type;   // of a 16-bit load
  const Bits keep = have >= STEPS ? static_cast<Bits>(~0ull) : have <= 0 ? 0 : (static_cast<Bits>(1) << (16 * have)) - 1;
  auto add = [&](PlaneCells<T, STEPS> (&v)[PIECES], int bi) {
    using H = PlaneHalf<T>;
    float wx[STEPS], wy[STEPS];
#pragma unroll
    for (int t = 0; t < STEPS; t++) {
      wx[t] = weights[bi][0][m][pw + t] * H::kScale;
      wy[t] = weights[bi][1][m][q + 4 * t] * (1.f / H::kScale);
    }
    // (products of different channels next to each other: each waits for the one before it of its own channel)
    f32x4_t t[PIECES];
    constexpr f32x4_t zero = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if constexpr (ES == 2) {
      // the gradients stand twice (four times) in K, against the weights' parts
      constexpr int PRODUCTS = STEPS / 2;
      typename H::v8 parts[PRODUCTS];
#pragma unroll
      for (int k = 0; k < STEPS; k++) {
        const typename H::E first = static_cast<typename H::E>(wx[k]);
        const float left = wx[k] - static_cast<float>(first);
        const typename H::E second = static_cast<typename H::E>(left);
        parts[0][k] = first;
        parts[0][STEPS + k] = second;
        if constexpr (STEPS == 2) parts[0][2 * STEPS + k] = static_cast<typename H::E>(left - static_cast<float>(second));
        else parts[PRODUCTS - 1][k] = static_cast<typename H::E>(left - static_cast<float>(second));
        parts[PRODUCTS - 1][8 - STEPS + k] = static_cast<typename H::E>(0.f);
      }
#pragma unroll
      for (int k = 0; k < PRODUCTS; k++)
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
          Bits bits;
          __builtin_memcpy(&bits, &v[i], sizeof(bits));
          bits = (bits >> (16 * back)) & keep;
          typename H::v8 g;
          if constexpr (STEPS == 2) g = __builtin_bit_cast(typename H::v8, plane_u32x4{bits, bits, bits, bits});
          else g = __builtin_bit_cast(typename H::v8, plane_u32x4{static_cast<unsigned>(bits), static_cast<unsigned>(bits >> 32), static_cast<unsigned>(bits), static_cast<unsigned>(bits >> 32)});
          t[i] = H::product(g, parts[k], k == 0 ? zero : t[i]);
        }
    } else {
#pragma unroll
      for (int k = 0; k < STEPS; k++)
#pragma unroll
        for (int i = 0; i < PIECES; i++)
          t[i] = plane_product(k < have ? load(&v[i].v[k]) : 0.f, wx[k], k == 0 ? zero : t[i]);
    }
#pragma unroll
    for (int s = 0; s < STEPS; s++)
#pragma unroll
      for (int c = 0; c < CH; c++) acc[c] = plane_product(wy[s], t[c / PER][c % PER * STEPS + s], acc[c]);
  };

  auto touches = [&](int i) {
    if (i >= p.R || (SPLIT && i % parts != part)) return false;
    const float *r = rois + static_cast<long>(i) * 5;
    const float scale = static_cast<float>(p.scale);
    const float xl = r[1] * scale, yl = r[2] * scale;
    const float xh = fmaxf(r[3] * scale, xl + 1.f), yh = fmaxf(r[4] * scale, yl + 1.f);
    // (a sample touches the pixels within one of it; one more for rounding.  Written so that NaN misses.)
    return static_cast<int>(r[0]) == image && r[0] > -1.f && xh >= x0 - 2.f && xl <= x0 + kPlaneTile + 1.f && yh >= y0 - 2.f &&
           yl <= y0 + kPlaneTile + 1.f;
  };
  // weights of column (axis 0) or row (axis 1) k of the tile in the cells of roi i
  auto weigh = [&](int i, int axis, int k, float *w) {
    const float *r = rois + static_cast<long>(i) * 5;
    PlaneAxis A;
    A.set(r[1 + axis], r[3 + axis], p.scale, axis == 0 ? p.ow : p.oh, p.sampling_ratio, axis == 0 ? p.W : p.H);
    const int x = (axis == 0 ? x0 : y0) + k;
    if (x < A.size && A.grid > 0) {
      A.template pixel_weights<CELLS>(x, p.order, w);
    } else {
#pragma unroll
      for (int c = 0; c < CELLS; c++) w[c] = 0.f;
    }
  };

  for (int base = 0; base < p.R; base += kPlaneQueue) {
    // ---- rois that touch the tile, in order, of the next kPlaneQueue ---------------------------------
    constexpr int kTests = kPlaneQueue / kPlaneThreads;
    __syncthreads();
    unsigned long long hits[kTests];
#pragma unroll
    for (int u = 0; u < kTests; u++) {
      hits[u] = __ballot(touches(base + u * kPlaneThreads + tid));
      if (lane == 0) wave_count[u * kPlaneWaves + wave] = __popcll(hits[u]);
    }
    __syncthreads();
    int listed = 0;
#pragma unroll
    for (int u = 0; u < kTests; u++) {
      int at = listed;
      for (int w = 0; w < kPlaneWaves; w++) {
        if (w == wave) at = listed;
        listed += wave_count[u * kPlaneWaves + w];
      }
      if ((hits[u] >> lane) & 1)
        queue[at + __popcll(hits[u] & ((1ull << lane) - 1))] = static_cast<unsigned>(base + u * kPlaneThreads + tid);
    }
    __syncthreads();
    if (listed == 0) continue;
    PlaneCells<T, STEPS> v[kPlaneAhead][PIECES];
#pragma unroll
    for (int u = 0; u + 1 < kPlaneAhead; u++) fetch(v[u], __builtin_amdgcn_readfirstlane(queue[min(u, listed - 1)]));
    for (int q0 = 0; q0 < listed; q0 += kPlaneBatch) {
      const int batch = min(kPlaneBatch, listed - q0);
      __syncthreads();   // the weights before have been used
      {
        // weights: thread = (roi of the batch, one of the tile's 16 columns or 16 rows)
        const int bi = tid / (2 * kPlaneTile), k = tid % (2 * kPlaneTile), axis = k / kPlaneTile;
        if (bi < batch) weigh(queue[q0 + bi], axis, k % kPlaneTile, weights[bi][axis][k % kPlaneTile]);
      }
      __syncthreads();
      // The loads of the next kPlaneAhead - 1 rois are in flight while one is added.  (Loads under a condition would make
      // the compiler wait for all of them: past the last roi it is loaded again.)
      for (int b0 = 0; b0 < batch; b0 += kPlaneAhead) {
#pragma unroll
        for (int u = 0; u < kPlaneAhead; u++) {
          fetch(v[(u + kPlaneAhead - 1) % kPlaneAhead],
                __builtin_amdgcn_readfirstlane(queue[min(q0 + b0 + u + kPlaneAhead - 1, listed - 1)]));
          if (b0 + u < batch) add(v[u], b0 + u);
        }
      }
    }
  }
  __syncthreads();   // the weights are free
  float check = 0.f;   // stays zero unless a sum is infinite or NaN
#pragma unroll
  for (int c = 0; c < CH; c++)
#pragma unroll
    for (int r = 0; r < 4; r++) check = fmaf(acc[c][r], 0.f, check);
  if (__ballot(!(check == 0.f)) != 0) {
    // this wavefront's channels again, roi by roi, without the terms of weight 0
    static_assert(kPlaneBatch >= kPlaneWaves, "a slot of weights for each wavefront");
    float(*mine)[kPlaneTile][PITCH] = weights[wave];
#pragma unroll
    for (int c = 0; c < CH; c++) acc[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto wave_sync = [] {   // LDS of one wavefront is in order: only the compiler has to keep it
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    };
    for (int i0 = 0; i0 < p.R; i0 += kWave)
      for (unsigned long long hits = __ballot(touches(i0 + lane)); hits != 0; hits &= hits - 1) {
        const int i = i0 + __builtin_ctzll(hits);
        wave_sync();
        if (lane < 2 * kPlaneTile) weigh(i, lane / kPlaneTile, lane % kPlaneTile, mine[lane / kPlaneTile][lane % kPlaneTile]);
        wave_sync();
        const T *g = gout + (static_cast<long>(i) * p.C + c0) * cells;
        for (int k = 0; k < cells; k++) {
          const int gy = k / p.ow, gx = k - gy * p.ow;
          const float wx = mine[0][m][gx];
#pragma unroll
          for (int c = 0; c < CH; c++) {
            if (c >= c_count) continue;
            const float v = load(g + static_cast<long>(c) * cells + k);
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const float wy = mine[1][4 * q + r][gy];
              if (wx != 0.f && wy != 0.f) acc[c][r] = fmaf(wy, wx * v, acc[c][r]);
            }
          }
        }
      }
  }
  const int x = x0 + m;
  if (x >= p.W) return;
  const long plane = static_cast<long>(p.H) * p.W;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int y = y0 + 4 * q + r;
    if (y >= p.H) continue;
    const long at = (static_cast<long>(image) * p.C + c0) * plane + static_cast<long>(y) * p.W + x;
    if constexpr (SPLIT) {
#pragma unroll
      for (int c = 0; c < CH; c++)
        if (c < c_count && acc[c][r] != 0.f) atomic_add(acc_buffer + at + c * plane, acc[c][r]);
    } else {
      T *d = grad + at;
      if (accumulate) {   // (all reads ahead of the first write: one round trip)
        T old[CH];
#pragma unroll
        for (int c = 0; c < CH; c++)
          if (c < c_count) old[c] = d[c * plane];
#pragma unroll
        for (int c = 0; c < CH; c++)
          if (c < c_count) acc[c][r] += load(&old[c]);
      }
#pragma unroll
      for (int c = 0; c < CH; c++)
        if (c < c_count) d[c * plane] = store_cast<T>(acc[c][r]);
    }
  }
}

bool roi_plane_applies(int dtype, const RoiProblem &p) {
  return p.ndim == 2 && !p.rotated && p.oh * p.ow >= 4 && (p.order == 0 || p.order == 1) && p.oh <= 16 && p.ow <= 16 && p.R > 0 &&
         (dtype == MV_F32 || dtype == MV_F16 || dtype == MV_BF16) && static_cast<long>(p.H) * p.W < (1L << 25);
}
static bool plane_small(const RoiProblem &p) { return p.oh <= 8 && p.ow <= 8; }

// Bytes of workspace that the forward pass can make use of: four per roi where ordering them pays for the ~7 us it takes
// (features well beyond an L2, enough rois).
size_t roi_plane_forward_workspace(int dtype, const RoiProblem &p) {
  if (!roi_plane_applies(dtype, p) || p.R < 256 || p.R > kPlaneOrderMax || p.N > kPlaneBuckets / kPlaneSizes) return 0;
  const long bytes = static_cast<long>(p.N) * p.C * p.H * p.W * static_cast<long>(dtype_size(dtype));
  return bytes >= (16L << 20) ? static_cast<size_t>(p.R) * 4 : 0;
}

// -1: not for this problem
int roi_plane_forward(const void *input, const void *rois, void *output, int dtype, const RoiProblem &p, void *workspace,
                      size_t capacity, hipStream_t s) {
  if (!roi_plane_applies(dtype, p)) return -1;
  unsigned *order = nullptr;
  const size_t need = roi_plane_forward_workspace(dtype, p);
  if (need > 0 && workspace != nullptr && capacity >= need && reinterpret_cast<uintptr_t>(workspace) % 4 == 0) {
    order = static_cast<unsigned *>(workspace);
    int side = 1;
    while ((side + 1) * (side + 1) * p.N <= kPlaneBuckets / kPlaneSizes) side++;
    hipLaunchKernelGGL(roi_plane_order_kernel, dim3(1), dim3(1024), 0, s, static_cast<const float *>(rois), order, p, side);
  }
  // Channels per workgroup: the lists cost ~3 us, so as many channels as leave eight workgroups per compute unit.
  int cpb = kPlaneChannels;
  while (cpb > 16 && static_cast<long>(p.R) * ((p.C + cpb - 1) / cpb) < 4096) cpb /= 2;
  const long cblocks = (p.C + cpb - 1) / cpb;
  if (cblocks * p.R >= (1L << 31)) return -1;
  const dim3 grid(static_cast<unsigned>(p.R * cblocks)), block(kPlaneThreads);
  const float *r = static_cast<const float *>(rois);
#define MV_PLANE_FORWARD(TYPE)                                                                                       \
  do {                                                                                                               \
    if (plane_small(p))                                                                                              \
      hipLaunchKernelGGL((roi_plane_forward_kernel<TYPE, 8>), grid, block, 0, s, static_cast<const TYPE *>(input), r, \
                         static_cast<TYPE *>(output), p, cpb, order);                                                        \
    else                                                                                                             \
      hipLaunchKernelGGL((roi_plane_forward_kernel<TYPE, 16>), grid, block, 0, s, static_cast<const TYPE *>(input),   \
                         r, static_cast<TYPE *>(output), p, cpb, order);                                                     \
  } while (0)
  switch (dtype) {
    case MV_F32: MV_PLANE_FORWARD(float); break;
    case MV_F16: MV_PLANE_FORWARD(__half); break;
    default: MV_PLANE_FORWARD(__hip_bfloat16);
  }
#undef MV_PLANE_FORWARD
  return check_launch("roi_plane_forward_kernel");
}

// Workgroups that share a tile's rois: 1 while the tiles and channels alone fill the chip (0: not for this problem).
int roi_plane_backward_parts(int dtype, const RoiProblem &p) {
  if (!roi_plane_applies(dtype, p)) return 0;
  const int ch = kPlaneBackwardChannels * kPlaneWaves;
  const long groups = static_cast<long>(p.N) * ((p.W + kPlaneTile - 1) / kPlaneTile) * ((p.H + kPlaneTile - 1) / kPlaneTile) *
                      ((p.C + ch - 1) / ch);
  // (a part should have a few dozen rois to look through)
  return static_cast<int>(std::max(1L, std::min({768L / groups, static_cast<long>(p.R) / 32, 64L})));
}

// parts == 1: `grad` is written (added to when `accumulate`); else the sums are added to the fp32 buffer `acc` (zeros).
int roi_plane_backward(const void *grad_output, const void *rois, void *grad, float *acc, int dtype, const RoiProblem &p,
                       int parts, bool accumulate, hipStream_t s) {
  const int ch = kPlaneBackwardChannels * kPlaneWaves;
  const int tx = (p.W + kPlaneTile - 1) / kPlaneTile, ty = (p.H + kPlaneTile - 1) / kPlaneTile;
  const long tiles = static_cast<long>(p.N) * tx * ty, cblocks = (p.C + ch - 1) / ch;
  if (tiles >= (1L << 31) || cblocks > 65535) return -1;
  const dim3 grid(static_cast<unsigned>(tiles), static_cast<unsigned>(cblocks), parts), block(kPlaneThreads);
  const float *r = static_cast<const float *>(rois);
#define MV_PLANE_BACKWARD(TYPE, CELLSV, SPLITV)                                                                      \
  hipLaunchKernelGGL((roi_plane_backward_kernel<TYPE, CELLSV, kPlaneBackwardChannels, SPLITV>), grid, block, 0, s,                       \
                     static_cast<const TYPE *>(grad_output), r, static_cast<TYPE *>(grad), acc, p, tx, ty, accumulate ? 1 : 0)
#define MV_PLANE_BACKWARD_OF(TYPE)                                                                                    \
  do {                                                                                                               \
    if (plane_small(p)) { if (parts > 1) MV_PLANE_BACKWARD(TYPE, 8, true); else MV_PLANE_BACKWARD(TYPE, 8, false); } \
    else { if (parts > 1) MV_PLANE_BACKWARD(TYPE, 16, true); else MV_PLANE_BACKWARD(TYPE, 16, false); }         \
  } while (0)
  switch (dtype) {
    case MV_F32: MV_PLANE_BACKWARD_OF(float); break;
    case MV_F16: MV_PLANE_BACKWARD_OF(__half); break;
    default: MV_PLANE_BACKWARD_OF(__hip_bfloat16);
  }
#undef MV_PLANE_BACKWARD_OF
#undef MV_PLANE_BACKWARD
  return check_launch("roi_plane_backward_kernel");
}

}  // namespace mv
