// Elastic deformation of volumes: the warp of warp.hip by a displacement field that is never written.  The field is the order-3
// upsampling of a small control grid over the window [border, n - border] of each axis, as the order-3 affine engine gives it for an
// unrotated roi (reference: aug_cuda/aug_spatial.py:560-600 upsamples, :655-668 warps).
//
// A workgroup owns 32 x 8 columns of eight voxels.  The upsampling is separable: the control points that its rows need are contracted along x
// for its 32 columns (to LDS), each thread contracts them along y where the four slices change, and a voxel's displacement is four products
// per component.  Same taps, weights and order of the sums as the separable form of roi_resample_cubic_kernel; the displacement is rounded to the
// image's type, as a field of that type holds it.
//
// Why: on fp16 [96 x 192 x 192] with 8^3 control points the field cost 32 us to write, 10 us to convert, and 12 (6) of the 20 (10) bytes that
// the two warps after it, 28 us (image) and 21 us (labels), move per voxel.  Now 27 and 18 us, bound by vector issue (positions in 32 bits: with
// those of warp.hip in 64 bits 31 and 23.5 us).  Augmentation of fp16 [128 x 256 x 256] in four stages: 205 -> 175 us, where the host's work
// begins to show (140 us).
#include "common.hpp"
#include "sampling.hpp"

#include <algorithm>

namespace mv {

constexpr int kElX = 32, kElY = 8, kElZ = 8;      // voxels of a workgroup; a thread has a column along z
constexpr int kElThreads = kElX * kElY;
constexpr int kElRows = 100;                      // rows of control points (y, z) that a workgroup's voxels may need
constexpr int kElGrid = 16;                       // control points per axis

struct ElasticShape {
  int C, D, H, W, gd, gh, gw;
  double border;
};
struct ElasticTaps {
  int idx[4];
  float w[4];
};

// The taps of output index `i` of `n` on an axis of `points` control points
__device__ __forceinline__ ElasticTaps elastic_taps(int i, int n, int points, double border) {
  const double ext = static_cast<double>(points) - 2.0 * border, bin = ext / n;
  const double v = (0.5 * points - 0.5) + (-0.5 * ext + i * bin + 0.5 * bin);
  ElasticTaps t;
  if (!cubic_tap<float>(v, points, t.idx, t.w)) {
#pragma unroll
    for (int k = 0; k < 4; k++) { t.idx[k] = 0; t.w[k] = 0.f; }
  }
  return t;
}

// The taps of position i + off on an axis of `size` voxels, those of clamped_tap on the open interval (-1, size), without 64-bit
// arithmetic: i + floor(off) is the position's floor, and off - floor(off) its fraction, rounded once.  `nearest`: the voxel at order 0, by the
// fraction as it is before that rounding (floor(off) + 0.5 is a number of 32 bits, so the comparison is exact).
__device__ __forceinline__ bool elastic_tap(int i, float off, int size, int &lo, int &hi, float &frac, int &nearest) {
  const float f = floorf(off);
  const bool near = fabsf(off) < 1e6f;   // (farther is outside, and not a number too)
  const int base = i + static_cast<int>(near ? f : 0.f);
  frac = off - f;
  const bool inside = near && base < size && (base >= 0 || (base == -1 && frac > 0.f));
  const bool border = base < 0 || base >= size - 1;
  if (border) frac = 0.f;
  lo = min(max(base, 0), size - 1);
  hi = min(lo + 1, size - 1);
  nearest = !border && off > f + 0.5f ? hi : lo;
  return inside;
}

// T: the image's type; int: label maps at order 0
template <typename T>
__global__ __launch_bounds__(kElThreads, 6) void elastic_warp_kernel(const T *__restrict__ img, const float *__restrict__ grid,
                                                                  T *__restrict__ out, const ElasticShape s, const int tiles_z) {
  __shared__ ElasticTaps taps_x[kElX], taps_y[kElY], taps_z[kElZ];
  extern __shared__ float lines[];   // [slice][row][component][x]
  const int tid = threadIdx.x, lx = tid % kElX, ly = tid / kElX;
  const int x0 = blockIdx.x * kElX, y0 = blockIdx.y * kElY, z0 = blockIdx.z % tiles_z * kElZ, b = blockIdx.z / tiles_z;
  if (tid < kElX) taps_x[tid] = elastic_taps(min(x0 + tid, s.W - 1), s.W, s.gw, s.border);
  else if (tid < kElX + kElY) taps_y[tid - kElX] = elastic_taps(min(y0 + tid - kElX, s.H - 1), s.H, s.gh, s.border);
  else if (tid < kElX + kElY + kElZ) taps_z[tid - kElX - kElY] = elastic_taps(min(z0 + tid - kElX - kElY, s.D - 1), s.D, s.gd, s.border);
  __syncthreads();
  const auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int first_y = uniform(taps_y[0].idx[0]), ny = uniform(taps_y[kElY - 1].idx[3]) - first_y + 1;
  const int first_z = uniform(taps_z[0].idx[0]), nz = uniform(taps_z[kElZ - 1].idx[3]) - first_z + 1;
  {
    const ElasticTaps e = taps_x[lx];   // (kElThreads is a multiple of kElX)
    const float *const g = grid + static_cast<long>(b) * 3 * s.gd * s.gh * s.gw;
    for (int r = ly; r < nz * ny * 3; r += kElY) {
      const int component = r % 3, zy = r / 3, y = zy % ny, z = zy / ny;
      const float *row = g + ((component * s.gd + first_z + z) * s.gh + first_y + y) * s.gw;
      lines[r * kElX + lx] = e.w[0] * row[e.idx[0]] + e.w[1] * row[e.idx[1]] + e.w[2] * row[e.idx[2]] + e.w[3] * row[e.idx[3]];
    }
  }
  __syncthreads();
  const int x = x0 + lx, y = y0 + ly;
  if (x >= s.W || y >= s.H) return;
  const ElasticTaps ey = taps_y[ly];
  const long P = static_cast<long>(s.D) * s.H * s.W;
  const int count = min(kElZ, s.D - z0);
  float c[4][3];
  int at[4] = {-1, -1, -1, -1};   // the slices that c holds
  for (int k = 0; k < count; k++) {
    const ElasticTaps ez = taps_z[k];
    int want[4];
#pragma unroll
    for (int j = 0; j < 4; j++) want[j] = uniform(ez.idx[j]) - first_z;
    if (want[0] != at[0] || want[1] != at[1] || want[2] != at[2] || want[3] != at[3]) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        at[j] = want[j];
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const float *col = lines + ((want[j] * ny - first_y) * 3 + a) * kElX + lx;
          c[j][a] = ey.w[0] * col[ey.idx[0] * 3 * kElX] + ey.w[1] * col[ey.idx[1] * 3 * kElX] + ey.w[2] * col[ey.idx[2] * 3 * kElX] +
                    ey.w[3] * col[ey.idx[3] * 3 * kElX];
        }
      }
    }
    float off[3];   // z, y, x
#pragma unroll
    for (int a = 0; a < 3; a++) {
      off[a] = ez.w[0] * c[0][a] + ez.w[1] * c[1][a] + ez.w[2] * c[2][a] + ez.w[3] * c[3][a];
      if constexpr (sizeof(T) == 2) {
        const T rounded = store_cast<T>(off[a]);
        off[a] = load(&rounded);
      }
    }
    const int z = z0 + k;
    int zi[2], yi[2], xi[2], zn, yn, xn;
    float lz, lh, lw;
    const bool live_z = elastic_tap(z, off[0], s.D, zi[0], zi[1], lz, zn), live_y = elastic_tap(y, off[1], s.H, yi[0], yi[1], lh, yn),
               live = elastic_tap(x, off[2], s.W, xi[0], xi[1], lw, xn) && live_z && live_y;
    const unsigned q = static_cast<unsigned>((z * s.H + y) * s.W + x);
    if constexpr (std::is_same<T, int>::value) {
      const unsigned from = static_cast<unsigned>((zn * s.H + yn) * s.W + xn);
      for (int ch = 0; ch < s.C; ch++) {
        const long plane = (static_cast<long>(b) * s.C + ch) * P;
        (out + plane)[q] = live ? (img + plane)[from] : 0;
      }
    } else {
      const float hz = 1.f - lz, hy = 1.f - lh, hx = 1.f - lw;
      unsigned at_row[4];
#pragma unroll
      for (int n = 0; n < 4; n++) at_row[n] = static_cast<unsigned>((zi[n / 2] * s.H + yi[n % 2]) * s.W);
      const float w_row[4] = {hz * hy, hz * lh, lz * hy, lz * lh};
      for (int ch = 0; ch < s.C; ch++) {
        const long plane = (static_cast<long>(b) * s.C + ch) * P;
        const T *const from = img + plane;
        float v = 0.f;
        if (live) {
#pragma unroll
          for (int n = 0; n < 4; n++) {
            v += w_row[n] * hx * load(from + (at_row[n] + static_cast<unsigned>(xi[0])));
            v += w_row[n] * lw * load(from + (at_row[n] + static_cast<unsigned>(xi[1])));
          }
        }
        (out + plane)[q] = store_cast<T>(v);
      }
    }
  }
}

// rows of control points that `voxels` neighbouring voxels need at most
static long elastic_rows(int voxels, int n, int points, double border) {
  return std::min(static_cast<long>(points), static_cast<long>(voxels * (points - 2.0 * border) / n) + 5);
}

}  // namespace mv

extern "C" {

int mv_elastic_warp_3d_applies(int dtype, int batch, int depth, int height, int width, int grid_d, int grid_h, int grid_w, float border) {
  using namespace mv;
  if (dtype != MV_F32 && dtype != MV_F16 && dtype != MV_BF16 && dtype != MV_I32) return 0;
  if (batch <= 0 || depth <= 0 || height <= 0 || width <= 0 || !(border >= 0.f)) return 0;
  for (int points : {grid_d, grid_h, grid_w})
    if (points < 2 || points > kElGrid || !(points > 2.f * border)) return 0;
  if (static_cast<long>(depth) * height * width >= (1L << 31) || (height + kElY - 1) / kElY > 65535 ||
      (depth + kElZ - 1L) / kElZ * batch > 65535)
    return 0;
  return elastic_rows(kElY, height, grid_h, border) * elastic_rows(kElZ, depth, grid_d, border) <= kElRows;
}

int mv_elastic_warp_3d(const void *img, const void *grid, void *output, int dtype, int batch, int channels, int depth, int height,
                       int width, int grid_d, int grid_h, int grid_w, float border, void *stream) {
  using namespace mv;
  MV_REQUIRE(mv_elastic_warp_3d_applies(dtype, batch, depth, height, width, grid_d, grid_h, grid_w, border) && channels > 0,
             "volume or control grid out of range (mv_elastic_warp_3d_applies)");
  MV_REQUIRE(img && grid && output, "null pointer argument");
  const ElasticShape s{channels, depth, height, width, grid_d, grid_h, grid_w, static_cast<double>(border)};
  const int tiles_z = (depth + kElZ - 1) / kElZ;
  const dim3 blocks((width + kElX - 1) / kElX, (height + kElY - 1) / kElY, tiles_z * batch);
  const size_t lds = elastic_rows(kElY, height, grid_h, border) * elastic_rows(kElZ, depth, grid_d, border) * (3 * kElX * sizeof(float));
  hipStream_t st = static_cast<hipStream_t>(stream);
#define MV_ELASTIC(T)                                                                                                  \
  hipLaunchKernelGGL((elastic_warp_kernel<T>), blocks, dim3(kElThreads), lds, st, static_cast<const T *>(img),              \
                     static_cast<const float *>(grid), static_cast<T *>(output), s, tiles_z)
  if (dtype == MV_I32) MV_ELASTIC(int);
  else if (dtype == MV_F16) MV_ELASTIC(__half);
  else if (dtype == MV_BF16) MV_ELASTIC(__hip_bfloat16);
  else MV_ELASTIC(float);
#undef MV_ELASTIC
  return check_launch("elastic_warp_kernel");
}

}  // extern "C"
