// Backward of the 3-D deformable convolution for fp16 / bf16 / fp32 tensors, built around the
// matrix cores and channels-last buffers.
//
//   gcol[c, k, q] = sum_o Wt[o, c, k] * gy[o, q]                    (GEMM, MFMA)
//   gx[corner_n(k, q), c] += w_n * mask * gcol                       (scatter: LDS tiles + fp32 atomics)
//   goff_a[k, q] = mask * sum_c gcol * dZ/dp_a ,  gmask[k, q] = sum_c gcol * Z
//   gw[o, c, k]  = sum_{b, q} gy[o, q] * col[c, k, q]                (GEMM over positions, MFMA)
//
// Tap kernel (dcn_backward_tap.hip): everything but the gradient of the input, and of that the corners that
// the scatter kernel leaves.
// Scatter kernels (unit-stride layers whose taps fit their tile): the corners that land near their
// position are summed per brick of positions in a fixed-point LDS tile and reach the gradient buffer as one
// atomic per (voxel, channel) of the tile.
#include "dcn_pad.hpp"
#include "dcn_scatter.hpp"

#include <atomic>
#include <cstdlib>

namespace mv {

// max |p[i]| as a bit pattern, folded into *out (which starts at 0) with one atomic per workgroup
__device__ __forceinline__ void fold_max(unsigned bits, unsigned *out) {
  __shared__ unsigned part[4];
  for (int sh = 32; sh > 0; sh >>= 1) bits = max(bits, static_cast<unsigned>(__shfl_xor(static_cast<int>(bits), sh)));
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = bits;
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned m = max(max(part[0], part[1]), max(part[2], part[3]));
    // (atomics on one address retire one after the other: a workgroup that cannot raise the value it
    // reads — possibly an older one, which is never above the current one — leaves it alone)
    if (m > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, m);
  }
}
// (block `bid` of `nblocks`: the kernels below call these bodies with their own block index or with a
// share of a launch that does several small jobs at once)
template <typename T>
__device__ __forceinline__ void dcn_absmax_block(const T *__restrict__ p, long n, unsigned *out, const unsigned bid,
                                                 const unsigned nblocks) {
  constexpr int V = 16 / sizeof(T);  // elements per 16-byte load
  float m = 0.f;
  bool bad = false;
  auto take = [&](T e) {
    const float v = fabsf(static_cast<float>(load(&e)));
    bad = bad || !(v == v);
    m = fmaxf(m, v);
  };
  const long head = min(n, static_cast<long>((16 - reinterpret_cast<size_t>(p) % 16) % 16 / sizeof(T)));
  const long groups = (n - head) / V, tid = bid * 256L + threadIdx.x;
  // four independent loads per lane and step
  for (long i = bid * 1024L + threadIdx.x; i < groups; i += nblocks * 1024L) {
    union { u32x4 u; T e[V]; } piece[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
      piece[u].u = i + u * 256 < groups ? *reinterpret_cast<const u32x4 *>(p + head + (i + u * 256) * V) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int j = 0; j < V; j++) take(piece[u].e[j]);
  }
  if (tid < head) take(p[tid]);
  const long tail = head + groups * V;
  if (tid < n - tail) take(p[tail + tid]);
  fold_max(bad ? 0x7fc00000u : __float_as_uint(m), out);
}
// max over (group, c, k) of sum_o |Wt[o, c, k]|: a workgroup takes 64 columns, its four wavefronts
// a quarter of the rows each
template <typename T>
__device__ __forceinline__ void dcn_weight_colsum_block(const T *__restrict__ wt, const DcnDims s, unsigned *out, const unsigned bid) {
  __shared__ float part[4][64];
  const long cols = static_cast<long>(s.cpg) * s.K, id = bid * 64L + threadIdx.x % 64;
  const int wave = threadIdx.x / 64;
  float sum = 0.f;
  if (id < cols * s.groups) {
    const long g = id / cols, ck = id - g * cols;
    for (int o = wave; o < s.opg; o += 4) sum += fabsf(static_cast<float>(load(wt + (g * s.opg + o) * cols + ck)));
  }
  part[wave][threadIdx.x % 64] = sum;
  __syncthreads();
  if (wave == 0) sum = part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x];
  fold_max(wave == 0 ? (sum == sum ? __float_as_uint(sum) : 0x7fc00000u) : 0u, out);
}

// dcn_backward_tap.hip
size_t dcn_tap_partial_bytes(const DcnDims &s, int dtype);
bool dcn_tap_supported(const DcnDims &s, int dtype);
int dcn_tap_backward(const void *xt, const void *off, const void *mask, const void *gyt, const void *wf,
                     float *gxt, void *goff, void *gmask, float *partial, float *gw, const DcnDims &s, const unsigned *bounds,
                     int dtype, hipStream_t stream);

// ---- gradient of the input, local corners: summed in LDS, then added to the buffer ----------------
// A workgroup owns a brick of positions and eight channels; its sixteen wavefronts are kScatterSplit
// groups of eight, every group covers the positions of the brick (32 per wavefront at a time) and
// takes a contiguous share of the taps.  gcol comes from the 16 x 16 MFMA with the channels as
// rows: lane l holds position l % 16 of a 16-position block and the channels l / 16 and l / 16 + 4,
// so one LDS add instruction covers 16 positions x 4 adjacent channels; a voxel's 8 sums are 9
// qwords apart from the next voxel's to spread the banks.  After the taps the tile's non-zero sums are converted and added
// to the gradient buffer: one global atomic per (voxel, channel) of the tile instead of one per
// (position, tap, corner, channel).
constexpr int kScatterSplit = 2, kScatterWaves = 8 * kScatterSplit, kScatterStride = 9;
constexpr int kScatterKeep = 4;  // slices of grad_output a wavefront keeps in registers over the taps (all of them)

// Element (output channel o of the padded layer p, channel cl of its group, tap k) of the real layer's weight
template <typename T>
__device__ __forceinline__ T padded_weight(const T *__restrict__ wt, const DcnDims &s, const DcnPad &pad, int o, int cl, int k) {
  const int g = o / pad.p.opg, ol = o - g * pad.p.opg, u = cl / pad.unit_p, r = cl - u * pad.unit_p;
  return ol < s.opg && r < pad.unit ? wt[(static_cast<long>(g * s.opg + ol) * s.cpg + u * pad.unit + r) * s.K + k] : store_cast<T>(0.f);
}

// weight [Cout, cpg, K] -> A pieces [group][tap][8-channel block][row step][lane][kPiece]: lane l
// is MFMA row l % 16 = channel (row / 4) + 4 * (row % 2) of the block (rows 4j + 2, 4j + 3 repeat
// rows 4j, 4j + 1 and are not used), element i the output channel g*opg + step*4*kPiece +
// (l/16)*kPiece + i
template <typename T>
__device__ __forceinline__ void dcn_weight_afragments8_block(const T *__restrict__ wt, T *__restrict__ wa, const DcnDims &real, const DcnPad &pad, const unsigned bid) {
  const DcnDims &s = pad.p;
  constexpr int PC = Mfma<T>::kPiece;
  const int cblocks = s.cpg / 8, steps = s.opg / (4 * PC);
  const long total = static_cast<long>(s.groups) * s.K * cblocks * steps * 64;
  const long id = bid * 256L + threadIdx.x;
  if (id >= total) return;
  const int lane = id % 64;
  long r = id / 64;
  const int st = r % steps; r /= steps;
  const int cb = r % cblocks; r /= cblocks;
  const int k = r % s.K;
  const int g = static_cast<int>(r / s.K);
  const int row = lane % 16, cl = cb * 8 + row / 4 + 4 * (row % 2);
  const int o = g * s.opg + st * 4 * PC + (lane / 16) * PC;
  for (int i = 0; i < PC; i++) wa[id * PC + i] = padded_weight(wt, real, pad, o + i, cl, k);
}

template <typename T, typename S>
__global__ __launch_bounds__(kScatterWaves * 64) void dcn_backward_scatter_kernel(
    const T *__restrict__ off, const T *__restrict__ mask, const T *__restrict__ gyt,
    const T *__restrict__ wa, float *__restrict__ gxt, const DcnDims s, const int nbh, const int nbw,
    const unsigned *__restrict__ bounds) {
  using M = Mfma<T>;
  using P = typename std::conditional<(sizeof(T) == 2), float, double>::type;
  constexpr int PC = M::kPiece, SL = 4 * PC;
  constexpr int VOX = S::TD * S::TH * S::TW;
  constexpr int GROUPS = S::BD * S::BH * S::BW / 32;  // 32-position groups of the brick
  static_assert(VOX <= kTileVoxMax && GROUPS % 8 == 0, "brick and tile sizes");
  __shared__ unsigned long long tile[VOX * kScatterStride];
  __shared__ __attribute__((aligned(16))) float recs[kScatterWaves][32][8];
  const ScatterScale scale = scatter_scale(bounds, S::BD * S::BH * S::BW * s.K, mask != nullptr);
  if (!scale.valid) return;  // every corner went through the data kernel
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int n = lane % 32, p16 = lane % 16, j = lane / 16;
  const int tg = wave / 8;
  const unsigned brick = xcd_contiguous(blockIdx.x, gridDim.x);
  const int bx = brick % nbw, by = (brick / nbw) % nbh, bz = brick / (nbw * nbh);
  const int c0 = blockIdx.y * 8, b = blockIdx.z;
  const int dgi = c0 / s.cpd, g = c0 / s.cpg, cb = (c0 - g * s.cpg) / 8;
  const long bg = static_cast<long>(b) * s.dg + dgi;
  const int cblocks = s.cpg / 8, steps = s.opg / SL;
  const TileOrigin origin = tile_origin<S>(s, bz, by, bx);

  for (int i = threadIdx.x; i < VOX * kScatterStride; i += kScatterWaves * 64) tile[i] = 0ull;
  __syncthreads();

  // position of brick index i, columns fastest
  auto position = [&](int i, bool &live) {
    const int od = bz * S::BD + i / (S::BH * S::BW), oh = by * S::BH + (i / S::BW) % S::BH, ow = bx * S::BW + i % S::BW;
    live = od < s.Do && oh < s.Ho && ow < s.Wo;
    return (static_cast<long>(min(od, s.Do - 1)) * s.Ho + min(oh, s.Ho - 1)) * s.Wo + min(ow, s.Wo - 1);
  };
  for (int pg = wave % 8; pg < GROUPS; pg += 8) {
  // the lane's own position for the taps (both halves of the wavefront compute them)
  bool live;
  const long q = position(pg * 32 + n, live);
  const int ow = q % s.Wo, oh = (q / s.Wo) % s.Ho, od = q / (static_cast<long>(s.Wo) * s.Ho);
  const int bd = od * s.sd - s.pd, bh = oh * s.sh - s.ph, bw = ow * s.sw - s.pw;
  // grad_output of the lane's column in the two 16-position blocks (MFMA B operand)
  bool blive[2];
  const T *grow[2];
  u32x4 keep[2][kScatterKeep];
#pragma unroll
  for (int blk = 0; blk < 2; blk++) {
    const long qb = position(pg * 32 + blk * 16 + p16, blive[blk]);
    grow[blk] = gyt + (static_cast<long>(b) * s.Q + qb) * s.Cout + g * s.opg + j * PC;
#pragma unroll
    for (int st = 0; st < kScatterKeep; st++)
      keep[blk][st] = (blive[blk] && st < steps) ? *reinterpret_cast<const u32x4 *>(grow[blk] + st * SL)
                                                : u32x4{0u, 0u, 0u, 0u};
  }
  const int per = (s.K + kScatterSplit - 1) / kScatterSplit, k0 = min(tg * per, s.K), k1 = min(s.K, k0 + per);
  const T *o = off + (bg * s.nd * s.K + static_cast<long>(s.nd) * k0) * s.Q + q;
  const T *mk = mask ? mask + (bg * s.K + k0) * s.Q + q : nullptr;
  float(*rec)[8] = recs[wave];

  int ki = k0 / (s.kh * s.kw), kj = (k0 / s.kw) % s.kh, kk = k0 % s.kw;
  P fd = P(0), fh = P(0), fw = P(0);
  float fm = 1.f;
  if (k0 < k1) {
    dcn_offsets(s, o, fd, fh, fw);
    if (mk) fm = load(mk);
  }
  // weight pieces of the current tap, loaded one tap ahead
  const long tap_stride = static_cast<long>(cblocks) * steps * 64 * PC;
  const T *afrag = wa + (((static_cast<long>(g) * s.K + k0) * cblocks + cb) * steps * 64 + lane) * PC;
  u32x4 wcur[kScatterKeep];
#pragma unroll
  for (int st = 0; st < kScatterKeep; st++)
    wcur[st] = (k0 < k1 && st < steps) ? *reinterpret_cast<const u32x4 *>(afrag + static_cast<long>(st) * (64 * PC))
                                       : u32x4{0u, 0u, 0u, 0u};
  for (int k = k0; k < k1; k++) {
    u32x4 wnext[kScatterKeep];
#pragma unroll
    for (int st = 0; st < kScatterKeep; st++)
      wnext[st] = (k + 1 < k1 && st < steps)
                      ? *reinterpret_cast<const u32x4 *>(afrag + tap_stride + static_cast<long>(st) * (64 * PC))
                      : u32x4{0u, 0u, 0u, 0u};
    {
      const P pd = fd + static_cast<P>(bd + ki * s.dd), ph = fh + static_cast<P>(bh + kj * s.dh),
              pw = fw + static_cast<P>(bw + kk * s.dw);
      const float m = fm;
      o += s.nd * s.Q;
      if (mk) mk += s.Q;
      if (++kk == s.kw) { kk = 0; if (++kj == s.kh) { kj = 0; ++ki; } }
      if (k + 1 < k1) {  // the next tap's offsets are in flight during this tap's adds
        dcn_offsets(s, o, fd, fh, fw);
        if (mk) fm = load(mk);
      }
      CornerTaps t;
      corner_taps<P>(s, pd, ph, pw, live, 1u, 0u, ~0u, t);
      int first;
      unsigned bits = tile_bits<S>(origin, static_cast<int>(floor(pd)), static_cast<int>(floor(ph)),
                                static_cast<int>(floor(pw)), first);
      unsigned inside = 0;
#pragma unroll
      for (int c = 0; c < 8; c++) inside |= t.at[c] != ~0u ? 1u << c : 0u;
      bits &= inside;
      if (lane < 32) {
        float4 *dst = reinterpret_cast<float4 *>(rec[n]);
        dst[0] = make_float4(__int_as_float(first), __uint_as_float(bits), m, t.ld);
        dst[1] = make_float4(t.lh, t.lw, 0.f, 0.f);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int st = 0; st < kScatterKeep; st++)
      if (st < steps) {
        acc[0] = M::run16(wcur[st], keep[0][st], acc[0]);
        acc[1] = M::run16(wcur[st], keep[1][st], acc[1]);
      }
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      const float4 *src = reinterpret_cast<const float4 *>(rec[blk * 16 + p16]);
      const float4 ra = src[0], rb = src[1];
      const int first = __float_as_int(ra.x);
      const unsigned bits = __float_as_uint(ra.y);
      // the lane's two channels, times the mask and the fixed-point scale
      const double gv[2] = {static_cast<double>(acc[blk][0] * ra.z) * scale.up,
                            static_cast<double>(acc[blk][1] * ra.z) * scale.up};
      const float wd[2] = {1.f - ra.w, ra.w}, wh[2] = {1.f - rb.x, rb.x}, ww[2] = {1.f - rb.y, rb.y};
      // the lane's qword of the first corner, as a 32-bit byte offset worked out once: the corners
      // differ by constants that go into the instructions' offset fields
      char *const cell0 = reinterpret_cast<char *>(tile) + (static_cast<unsigned>(first) * kScatterStride + j) * 8u;
#pragma unroll
      for (int c = 0; c < 8; c++) {
        const int ca = c >> 2, cb2 = (c >> 1) & 1, ce = c & 1;
        if ((S::TD > 1 || ca == 0) && ((bits >> c) & 1u)) {  // images have no second slice
          const float wc = wd[ca] * wh[cb2] * ww[ce];
          unsigned long long *dst = reinterpret_cast<unsigned long long *>(
              cell0 + (ca * (S::TH * S::TW) + cb2 * S::TW + ce) * (kScatterStride * 8));
#pragma unroll
          for (int r = 0; r < 2; r++)
            __hip_atomic_fetch_add(dst + 4 * r, fixed_term(wc, gv[r]), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    afrag += tap_stride;
#pragma unroll
    for (int st = 0; st < kScatterKeep; st++) wcur[st] = wnext[st];
  }
  }
  __syncthreads();
  // ---- the tile's voxels inside the volume go to the gradient buffer, 8 channels per voxel --------
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(
      gxt + static_cast<long>(b) * s.P * s.Cin, 0, static_cast<int>(s.P * s.Cin * 4), kRsrcFlags);
  const unsigned cin4 = static_cast<unsigned>(s.Cin) * 4u;
  const int ch = threadIdx.x % 8;
  for (int cell = threadIdx.x / 8; cell < VOX; cell += kScatterWaves * 8) {
    const int zw = cell % S::TW + origin.w, zh = (cell / S::TW) % S::TH + origin.h, zd = cell / (S::TW * S::TH) + origin.d;
    const unsigned long long sum = tile[cell * kScatterStride + ch];
    if (zd >= 0 && zd < s.D && zh >= 0 && zh < s.H && zw >= 0 && zw < s.W && sum != 0ull) {
      const double v = static_cast<double>(static_cast<long long>(sum)) * scale.down;
      __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(
          static_cast<float>(v), gr,
          static_cast<unsigned>((zd * s.H + zh) * s.W + zw) * cin4 + static_cast<unsigned>(c0 + ch) * 4u, 0, 0);
    }
  }
}

// ---- the same sums in 32-bit cells, for 16-bit tensors ---------------------------------------------
// A workgroup owns a brick and SIXTEEN channels (all 16 rows of the 16 x 16 MFMA): the taps, the
// records and grad_output serve twice the channels, an LDS add moves 4 bytes instead of 8 and a term
// costs one fma and one subtraction.  32 bits leave 30 - ceil(log2(positions * taps)) bits for a
// term (17 for 3 x 3 x 3 taps), so the scale comes from the data: a first sweep over the brick's
// taps forms gcol alone (matrix cores, no geometry) and takes max |gcol| of the workgroup; every
// term is then below max |gcol| * max |mask| < 2^ex and is rounded to a multiple of 2^(ex - shift)
// (adding 1.5 * 2^23 in fp32 leaves round(x) in the low mantissa bits for |x| < 2^22).  The error of
// a voxel's sum stays below terms * 2^(ex - shift - 1), about 2^-15 of the values it sums for the
// 3 x 3 x 3 layer — a sixteenth of the last bit of the 16-bit result.
constexpr int kScatter32Stride = 17;    // dwords between voxels: 16 channels and one to spread the banks
constexpr int kScatter32MinShift = 14;  // fewer bits per term: the 64-bit kernel takes the layer
__host__ __device__ constexpr int scatter32_shift(int terms) {
  int bits = 0;
  while ((1L << bits) < terms) bits++;
  return 30 - bits;
}

// weight [Cout, cpg, K] -> A pieces [group][tap][16-channel block][row step][lane][kPiece]: lane l is
// MFMA row l % 16 = channel l % 16 of the block, element i the output channel
// g*opg + step*4*kPiece + (l/16)*kPiece + i
template <typename T>
__device__ __forceinline__ void dcn_weight_afragments16_block(const T *__restrict__ wt, T *__restrict__ wa, const DcnDims &real, const DcnPad &pad, const unsigned bid) {
  const DcnDims &s = pad.p;
  constexpr int PC = Mfma<T>::kPiece;
  const int cblocks = s.cpg / 16, steps = s.opg / (4 * PC);
  const long total = static_cast<long>(s.groups) * s.K * cblocks * steps * 64;
  const long id = bid * 256L + threadIdx.x;
  if (id >= total) return;
  const int lane = id % 64;
  long r = id / 64;
  const int st = r % steps; r /= steps;
  const int cb = r % cblocks; r /= cblocks;
  const int k = r % s.K;
  const int g = static_cast<int>(r / s.K);
  const int cl = cb * 16 + lane % 16;
  const int o = g * s.opg + st * 4 * PC + (lane / 16) * PC;
  for (int i = 0; i < PC; i++) wa[id * PC + i] = padded_weight(wt, real, pad, o + i, cl, k);
}

template <typename T, typename S>
__global__ __launch_bounds__(kScatterWaves * 64) void dcn_backward_scatter32_kernel(
    const T *__restrict__ off, const T *__restrict__ mask, const T *__restrict__ gyt,
    const T *__restrict__ wa, float *__restrict__ gxt, const DcnDims s, const int nbh, const int nbw,
    const unsigned *__restrict__ bounds) {
  using M = Mfma<T>;
  using P = typename std::conditional<(sizeof(T) == 2), float, double>::type;
  constexpr int PC = M::kPiece, SL = 4 * PC;
  constexpr int VOX = S::TD * S::TH * S::TW;
  constexpr int GROUPS = S::BD * S::BH * S::BW / 32;  // 32-position groups of the brick
  static_assert(VOX <= kTileVoxMax && GROUPS % 8 == 0, "brick and tile sizes");
  __shared__ int tile[VOX * kScatter32Stride];
  __shared__ __attribute__((aligned(8))) float recs[kScatterWaves][64][6];
  __shared__ unsigned wgmax;
  // (the validity of the data kernel's split: no NaN or infinity anywhere, products finite)
  if (!scatter_scale(bounds, S::BD * S::BH * S::BW * s.K, mask != nullptr).valid) return;
  const float mask_max = mask ? __uint_as_float(bounds[2]) : 1.f;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int n = lane % 32, p16 = lane % 16, j = lane / 16;
  const int tg = wave / 8;
  const unsigned brick = xcd_contiguous(blockIdx.x, gridDim.x);
  const int bx = brick % nbw, by = (brick / nbw) % nbh, bz = brick / (nbw * nbh);
  const int c0 = blockIdx.y * 16, b = blockIdx.z;
  const int dgi = c0 / s.cpd, g = c0 / s.cpg, cb = (c0 - g * s.cpg) / 16;
  const long bg = static_cast<long>(b) * s.dg + dgi;
  const int cblocks = s.cpg / 16, steps = s.opg / SL;
  const TileOrigin origin = tile_origin<S>(s, bz, by, bx);
  const int per = (s.K + kScatterSplit - 1) / kScatterSplit, k0 = min(tg * per, s.K), k1 = min(s.K, k0 + per);
  const long tap_stride = static_cast<long>(cblocks) * steps * 64 * PC;
  const T *afrag0 = wa + (((static_cast<long>(g) * s.K + k0) * cblocks + cb) * steps * 64 + lane) * PC;

  for (int i = threadIdx.x; i < VOX * kScatter32Stride; i += kScatterWaves * 64) tile[i] = 0;
  if (threadIdx.x == 0) wgmax = 0u;
  __syncthreads();

  // position of brick index i, columns fastest
  auto position = [&](int i, bool &live) {
    const int od = bz * S::BD + i / (S::BH * S::BW), oh = by * S::BH + (i / S::BW) % S::BH, ow = bx * S::BW + i % S::BW;
    live = od < s.Do && oh < s.Ho && ow < s.Wo;
    return (static_cast<long>(min(od, s.Do - 1)) * s.Ho + min(oh, s.Ho - 1)) * s.Wo + min(ow, s.Wo - 1);
  };
  // grad_output of the lane's column in the two 16-position blocks of a group (MFMA B operand)
  auto load_keep = [&](int pg, u32x4 (&keep)[2][kScatterKeep]) {
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      bool blive;
      const long qb = position(pg * 32 + blk * 16 + p16, blive);
      const T *grow = gyt + (static_cast<long>(b) * s.Q + qb) * s.Cout + g * s.opg + j * PC;
#pragma unroll
      for (int st = 0; st < kScatterKeep; st++)
        keep[blk][st] = (blive && st < steps) ? *reinterpret_cast<const u32x4 *>(grow + st * SL) : u32x4{0u, 0u, 0u, 0u};
    }
  };
  auto load_weights = [&](const T *afrag, bool on, u32x4 (&w)[kScatterKeep]) {
#pragma unroll
    for (int st = 0; st < kScatterKeep; st++)
      w[st] = (on && st < steps) ? *reinterpret_cast<const u32x4 *>(afrag + static_cast<long>(st) * (64 * PC))
                                 : u32x4{0u, 0u, 0u, 0u};
  };

  // ---- first sweep: max |gcol| over the brick's positions, the taps and the 16 channels -----------
  {
    float top = 0.f;
    for (int pg = wave % 8; pg < GROUPS; pg += 8) {
      u32x4 keep[2][kScatterKeep];
      load_keep(pg, keep);
      const T *afrag = afrag0;
      for (int k = k0; k < k1; k++) {
        u32x4 w[kScatterKeep];
        load_weights(afrag, true, w);
        afrag += tap_stride;
        float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int st = 0; st < kScatterKeep; st++)
          if (st < steps) {
            acc[0] = M::run16(w[st], keep[0][st], acc[0]);
            acc[1] = M::run16(w[st], keep[1][st], acc[1]);
          }
#pragma unroll
        for (int i = 0; i < 4; i++) top = fmaxf(top, fmaxf(fabsf(acc[0][i]), fabsf(acc[1][i])));
      }
    }
    for (int sh = 32; sh > 0; sh >>= 1) top = fmaxf(top, __shfl_xor(top, sh));
    if (lane == 0 && top > 0.f) atomicMax(&wgmax, __float_as_uint(top));
  }
  __syncthreads();
  const float bound = fmaxf(1.001f * __uint_as_float(wgmax), 1e-30f) * mask_max;
  if (!(bound > 0.f)) return;  // nothing but zeros to add (the whole workgroup leaves together)
  const int shift = scatter32_shift(S::BD * S::BH * S::BW * s.K);
  int ex = 0;
  frexpf(bound, &ex);  // bound < 2^ex
  const float up = ldexpf(1.f, shift - ex), down = ldexpf(1.f, ex - shift);
  constexpr float kMagic = 12582912.f;  // 1.5 * 2^23

  for (int pg = wave % 8; pg < GROUPS; pg += 8) {
  // the taps are worked out two at a time: the lower half-wavefront takes tap k of the group's 32
  // positions, the upper half tap k + 1
  const int hh = lane / 32;
  bool live;
  const long q = position(pg * 32 + n, live);
  const int ow = q % s.Wo, oh = (q / s.Wo) % s.Ho, od = q / (static_cast<long>(s.Wo) * s.Ho);
  const int bd = od * s.sd - s.pd, bh = oh * s.sh - s.ph, bw = ow * s.sw - s.pw;
  u32x4 keep[2][kScatterKeep];
  load_keep(pg, keep);
  int kt = k0 + hh;  // the lane's own tap
  const T *o = off + (bg * s.nd * s.K + static_cast<long>(s.nd) * kt) * s.Q + q;
  const T *mk = mask ? mask + (bg * s.K + kt) * s.Q + q : nullptr;
  float(*rec)[6] = recs[wave];

  int ki = kt / (s.kh * s.kw), kj = (kt / s.kw) % s.kh, kk = kt % s.kw;
  P fd = P(0), fh = P(0), fw = P(0);
  float fm = 1.f;
  if (kt < k1) {
    dcn_offsets(s, o, fd, fh, fw);
    if (mk) fm = load(mk);
  }
  const T *afrag = afrag0;
  for (int k = k0; k < k1; k += 2) {
    // weight pieces of the two taps (the taps' geometry below hides their latency)
    u32x4 wpair[2][kScatterKeep];
    load_weights(afrag, true, wpair[0]);
    load_weights(afrag + tap_stride, k + 1 < k1, wpair[1]);
    {
      const P pd = fd + static_cast<P>(bd + ki * s.dd), ph = fh + static_cast<P>(bh + kj * s.dh),
              pw = fw + static_cast<P>(bw + kk * s.dw);
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
      unsigned bits = tile_bits<S>(origin, static_cast<int>(floor(pd)), static_cast<int>(floor(ph)),
                                static_cast<int>(floor(pw)), first);
      unsigned inside = 0;
#pragma unroll
      for (int c = 0; c < 8; c++) inside |= t.at[c] != ~0u ? 1u << c : 0u;
      bits &= inside;
      float2 *dst = reinterpret_cast<float2 *>(rec[lane]);
      dst[0] = make_float2(__int_as_float(first), __uint_as_float(bits));
      dst[1] = make_float2(m * up, t.ld);
      dst[2] = make_float2(t.lh, t.lw);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

#pragma unroll
    for (int u = 0; u < 2; u++) {
      if (k + u >= k1) break;
      float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int st = 0; st < kScatterKeep; st++)
        if (st < steps) {
          acc[0] = M::run16(wpair[u][st], keep[0][st], acc[0]);
          acc[1] = M::run16(wpair[u][st], keep[1][st], acc[1]);
        }
#pragma unroll
      for (int blk = 0; blk < 2; blk++) {
        const float2 *src = reinterpret_cast<const float2 *>(rec[u * 32 + blk * 16 + p16]);
        const float2 ra = src[0], rb = src[1], rc = src[2];
        const int first = __float_as_int(ra.x);
        const unsigned bits = __float_as_uint(ra.y);
        // the lane's four channels 4j .. 4j + 3, times the mask and the fixed-point scale
        const float gv[4] = {acc[blk][0] * rb.x, acc[blk][1] * rb.x, acc[blk][2] * rb.x, acc[blk][3] * rb.x};
        const float wd[2] = {1.f - rb.y, rb.y}, wh[2] = {1.f - rc.x, rc.x}, ww[2] = {1.f - rc.y, rc.y};
        // the lane's first dword of the first corner, as a 32-bit byte offset worked out once: the
        // corners and channels differ by constants that go into the instructions' offset fields
        char *const cell0 = reinterpret_cast<char *>(tile) + (static_cast<unsigned>(first) * kScatter32Stride + 4 * j) * 4u;
#pragma unroll
        for (int c = 0; c < 8; c++) {
          const int ca = c >> 2, cb2 = (c >> 1) & 1, ce = c & 1;
          if ((S::TD > 1 || ca == 0) && ((bits >> c) & 1u)) {  // images have no second slice
            const float wc = wd[ca] * wh[cb2] * ww[ce];
            int *dst = reinterpret_cast<int *>(cell0 + (ca * (S::TH * S::TW) + cb2 * S::TW + ce) * (kScatter32Stride * 4));
#pragma unroll
            for (int r = 0; r < 4; r++)
              __hip_atomic_fetch_add(dst + r, __float_as_int(fmaf(wc, gv[r], kMagic)) - 0x4B400000, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    afrag += 2 * tap_stride;
  }
  }
  __syncthreads();
  // ---- the tile's voxels inside the volume go to the gradient buffer, 16 channels per voxel -------
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(
      gxt + static_cast<long>(b) * s.P * s.Cin, 0, static_cast<int>(s.P * s.Cin * 4), kRsrcFlags);
  const unsigned cin4 = static_cast<unsigned>(s.Cin) * 4u;
  const int ch = threadIdx.x % 16;
  for (int cell = threadIdx.x / 16; cell < VOX; cell += kScatterWaves * 4) {
    const int zw = cell % S::TW + origin.w, zh = (cell / S::TW) % S::TH + origin.h, zd = cell / (S::TW * S::TH) + origin.d;
    const int sum = tile[cell * kScatter32Stride + ch];
    if (zd >= 0 && zd < s.D && zh >= 0 && zh < s.H && zw >= 0 && zw < s.W && sum != 0)
      __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(
          static_cast<float>(sum) * down, gr,
          static_cast<unsigned>((zd * s.H + zh) * s.W + zw) * cin4 + static_cast<unsigned>(c0 + ch) * 4u, 0, 0);
  }
}

// gxt [B, P, Cs] fp32 -> gx [B, C, P] T, added to what gx holds (`accumulate`) or in its place; 64 positions x up to
// kAddChunk channels per workgroup.  The source may hold padded channels: channel c at (c / unit) * unit_p + c % unit.
constexpr int kAddChunk = 64;
struct AddShared { __attribute__((aligned(16))) float f[64][kAddChunk + 4]; };   // (16-byte writes; reads along the positions)
template <typename T>
__device__ __forceinline__ void dcn_planar_add_block(AddShared &stage, const float *__restrict__ gxt, T *__restrict__ gx, int C, long P,
                                                     const unsigned bx, const int b, const int bz, const int accumulate,
                                                     const int Cs, const int unit, const int unit_p) {
  const long p0 = static_cast<long>(bx) * 64;
  const int c0 = bz * kAddChunk, cn = min(kAddChunk, C - c0);
  const int count = static_cast<int>(min(static_cast<long>(64), P - p0)) * cn;
  const float *src = gxt + (static_cast<long>(b) * P + p0) * Cs;
  for (int i = threadIdx.x; i < count; i += 256) {
    const int pp = i / cn, c = c0 + i % cn;
    stage.f[pp][c - c0] = src[static_cast<long>(pp) * Cs + c / unit * unit_p + c % unit];
  }
  __syncthreads();
  const int lp = threadIdx.x % 64;
  if (p0 + lp < P)
    for (int c = threadIdx.x / 64; c < cn; c += 4) {
      T *d = gx + (static_cast<long>(b) * C + c0 + c) * P + p0 + lp;
      *d = store_cast<T>(accumulate ? load(d) + stage.f[lp][c] : stage.f[lp][c]);
    }
}

// The same move with 16-byte reads (units and channels in fours, an aligned buffer).  EVEN: P a multiple of 64 and the gradient
// aligned, so that a lane takes V = 16 / sizeof(T) neighbouring positions of one channel in one write; otherwise a
// wavefront writes 64 neighbouring elements.  ([4, 256, 38 * 30 * 125] fp16: 431 us through the kernel above.)
template <typename T, bool EVEN>
__device__ __forceinline__ void dcn_planar_add_wide_block(AddShared &stage, const float *__restrict__ gxt, T *__restrict__ gx, int C, long P,
                                                          const unsigned bx, const int b, const int bz, const int accumulate,
                                                          const int Cs, const int unit, const int unit_p) {
  constexpr int V = 16 / static_cast<int>(sizeof(T));
  const long p0 = static_cast<long>(bx) * 64;
  const int c0 = bz * kAddChunk, cn = min(kAddChunk, C - c0);   // cn: a multiple of 4
  const int pn = EVEN ? 64 : static_cast<int>(min(64L, P - p0));
  const float *src = gxt + (static_cast<long>(b) * P + p0) * Cs;
  float4 in[4];
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int i = threadIdx.x + u * 256, pp = i / 16, cq = i % 16;
    in[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (cq * 4 < cn && (EVEN || pp < pn)) {   // (the accumulation buffer is read once and the result not read here again: nontemporal)
      typedef float f32x4 __attribute__((ext_vector_type(4)));
      const int c = c0 + cq * 4, at = unit == unit_p ? c : c / unit * unit_p + c % unit;
      const f32x4 t = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(src + static_cast<long>(pp) * Cs + at));
      in[u] = make_float4(t.x, t.y, t.z, t.w);
    }
  }
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int i = threadIdx.x + u * 256, pp = i / 16, cq = i % 16;
    *reinterpret_cast<float4 *>(&stage.f[pp][cq * 4]) = in[u];
  }
  __syncthreads();
  if constexpr (EVEN) {
    constexpr int PG = 64 / V;   // position groups per channel
    for (int i = threadIdx.x; i < cn * PG; i += 256) {
      const int c = i / PG, pg = i % PG;
      T *d = gx + (static_cast<long>(b) * C + c0 + c) * P + p0 + pg * V;
      union { u32x4 u; T e[V]; } piece;
      if (accumulate) {
        piece.u = *reinterpret_cast<const u32x4 *>(d);
#pragma unroll
        for (int e = 0; e < V; e++) piece.e[e] = store_cast<T>(load(&piece.e[e]) + stage.f[pg * V + e][c]);
      } else {
#pragma unroll
        for (int e = 0; e < V; e++) piece.e[e] = store_cast<T>(stage.f[pg * V + e][c]);
      }
      __builtin_nontemporal_store(piece.u, reinterpret_cast<u32x4 *>(d));
    }
  } else {
    const int lp = threadIdx.x % 64;
    if (lp < pn) {
      T *d = gx + (static_cast<long>(b) * C + c0) * P + p0 + lp;
      for (int c = threadIdx.x / 64; c < cn; c += 16) {   // (cn is a multiple of four: four channels per turn, reads first)
        T old[4];
        if (accumulate)
#pragma unroll
          for (int u = 0; u < 4; u++)
            if (c + 4 * u < cn) old[u] = d[(c + 4 * u) * P];
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (c + 4 * u < cn)
            d[(c + 4 * u) * P] = store_cast<T>(accumulate ? load(&old[u]) + stage.f[lp][c + 4 * u] : stage.f[lp][c + 4 * u]);
      }
    }
  }
}
// MODE 0: the plain move, 1: 16-byte reads, 2: 16-byte writes as well
template <typename T, int MODE>
__device__ __forceinline__ void dcn_planar_add_mode(AddShared &stage, const float *__restrict__ gxt, T *__restrict__ gx, int C, long P, const unsigned bx,
                                                    const int b, const int bz, const int accumulate, const int Cs, const int unit,
                                                    const int unit_p) {
  if constexpr (MODE == 0) dcn_planar_add_block<T>(stage, gxt, gx, C, P, bx, b, bz, accumulate, Cs, unit, unit_p);
  else dcn_planar_add_wide_block<T, MODE == 2>(stage, gxt, gx, C, P, bx, b, bz, accumulate, Cs, unit, unit_p);
}
static int planar_add_mode(const void *src, const void *dst, int unit, long P) {
  auto aligned16 = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  return unit % 4 || !aligned16(src) ? 0 : (P % 64 == 0 && aligned16(dst) ? 2 : 1);
}
template <typename T, int MODE>
__global__ __launch_bounds__(256) void dcn_planar_add_kernel(const float *__restrict__ gxt, T *__restrict__ gx, int C, long P,
                                                             int accumulate) {
  __shared__ AddShared stage;
  dcn_planar_add_mode<T, MODE>(stage, gxt, gx, C, P, blockIdx.x, blockIdx.y, blockIdx.z, accumulate, C, C, C);
}

__device__ __forceinline__ void dcn_zero_f32_block(float *p, long n, const unsigned bid, const unsigned nblocks) {
  for (long i = bid * 256L + threadIdx.x; i < n; i += nblocks * 256L) p[i] = 0.f;
}

// One pass over a slab of grad_output[b, o, .]: its sum into the fp32 bias accumulator and (`out`
// given) its largest magnitude as a bit pattern into *out.  Workgroup = (o, b, slab of `slab_len`
// positions); about 512 workgroups in all — enough loads in flight for the memory system, and few enough
// for the atomics on the one word of the maximum, which retire one after the other (~10 ns each).
static long gy_slab_len(const DcnDims &s) {
  const long rows = static_cast<long>(s.Cout) * s.B;
  const long slabs = std::max(1L, std::min((s.Q + 2047) / 2048, (512 + rows - 1) / rows));
  return ((s.Q + slabs - 1) / slabs + 1023) / 1024 * 1024;
}
template <typename T>
__device__ __forceinline__ void dcn_gy_sum_max_block(const T *__restrict__ gy, float *__restrict__ gb32, unsigned *out,
                                                     const DcnDims s, const long slab_len, const unsigned bid) {
  constexpr int V = 16 / static_cast<int>(sizeof(T));
  __shared__ float sums[4];
  const unsigned slabs = static_cast<unsigned>((s.Q + slab_len - 1) / slab_len);
  const unsigned slab = bid % slabs, r = bid / slabs;
  const int b = static_cast<int>(r % s.B), o = static_cast<int>(r / s.B);
  const T *src = gy + (static_cast<long>(b) * s.Cout + o) * s.Q;
  long q0 = static_cast<long>(slab) * slab_len;
  const long q_end = min(q0 + slab_len, s.Q);
  float v = 0.f, m = 0.f;
  bool bad = false;
  auto take = [&](T e) {
    const float x = static_cast<float>(load(&e));
    v += x;
    bad = bad || !(x == x);
    m = fmaxf(m, fabsf(x));
  };
  if (reinterpret_cast<uintptr_t>(src + q0) % 16 == 0) {
    // 16-byte pieces, four independent loads per lane and step
    const long groups = (q_end - q0) / V;
    const u32x4 *pieces = reinterpret_cast<const u32x4 *>(src + q0);
    for (long i = threadIdx.x; i < groups; i += 1024) {
      union { u32x4 u; T e[V]; } raw[4];
#pragma unroll
      for (int u = 0; u < 4; u++) raw[u].u = i + u * 256 < groups ? pieces[i + u * 256] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int e = 0; e < V; e++) take(raw[u].e[e]);
    }
    q0 += groups * V;
  }
  for (long q = q0 + threadIdx.x; q < q_end; q += 256) take(src[q]);
  for (int sh = 32; sh > 0; sh >>= 1) v += __shfl_xor(v, sh);
  if (threadIdx.x % kWave == 0) sums[threadIdx.x / kWave] = v;
  if (out) fold_max(bad ? 0x7fc00000u : __float_as_uint(m), out);   // (contains the barrier)
  else __syncthreads();
  if (threadIdx.x == 0) atomicAdd(gb32 + o, (sums[0] + sums[1]) + (sums[2] + sums[3]));
}

// The small jobs in front of the tap kernel in two launches (a dependent launch costs ~2.7 us before its first
// instruction, and kernels of a few microseconds do not fill the machine): first the two layout passes, the weight
// fragments and the zero fill of the accumulators and of the maxima's words; then the maxima and the bias sums, which need those
// words at zero.
struct PrepareJobs {
  unsigned x_end, gy_end, f16_end, fsc_end, zero_end;   // block ranges of the first launch
  unsigned px, pq;                                      // blocks of positions of the input / the output
};
template <typename T>
__global__ __launch_bounds__(256) void dcn_backward_prepare_kernel(const T *__restrict__ x, T *__restrict__ xt,
                                                                   const T *__restrict__ gy, T *__restrict__ gyt,
                                                                   const T *__restrict__ wt, T *__restrict__ wb,
                                                                   T *__restrict__ wa, float *__restrict__ zero,
                                                                   const long nz, const DcnDims s, const DcnPad pad, const PrepareJobs j) {
  using U = typename std::conditional<(sizeof(T) == 2), unsigned short, unsigned int>::type;
  const unsigned id = blockIdx.x;
  if (id < j.gy_end) {   // (one body, and one LDS block, for both)
    const bool first = id < j.x_end;
    const unsigned r = first ? id : id - j.x_end, pb = first ? j.px : j.pq;
    dcn_move_block<U>(reinterpret_cast<const U *>(first ? x : gy), reinterpret_cast<U *>(first ? xt : gyt), first ? s.Cin : s.Cout,
                      first ? pad.p.Cin : pad.p.Cout, first ? pad.unit : s.opg, first ? pad.unit_p : pad.p.opg, first ? s.P : s.Q,
                      r % pb, static_cast<int>((r / pb) % s.B), static_cast<int>(r / pb / s.B));
  } else if (id < j.f16_end) {
    dcn_weight_afragments16_block<T>(wt, wb, s, pad, id - j.gy_end);
  } else if (id < j.fsc_end) {
    dcn_weight_afragments8_block<T>(wt, wa, s, pad, id - j.f16_end);
  } else {
    dcn_zero_f32_block(zero, nz, id - j.fsc_end, j.zero_end - j.fsc_end);
  }
}
template <typename T>
__global__ __launch_bounds__(256) void dcn_backward_maxima_kernel(const T *__restrict__ gy, const long ngy,
                                                                  const T *__restrict__ mask, const long nmask,
                                                                  const T *__restrict__ wt, const DcnDims s,
                                                                  unsigned *__restrict__ bounds, float *__restrict__ gb32,
                                                                  const long slab_len, const unsigned gy_blocks,
                                                                  const unsigned mask_blocks) {
  const unsigned id = blockIdx.x;
  if (id < gy_blocks) {
    // with a bias gradient to form the pass over grad_output also sums it, a workgroup per (o, b, slab)
    if (gb32) dcn_gy_sum_max_block<T>(gy, gb32, bounds, s, slab_len, id);
    else dcn_absmax_block<T>(gy, ngy, bounds, id, gy_blocks);
  } else if (id < gy_blocks + mask_blocks) dcn_absmax_block<T>(mask, nmask, bounds + 2, id - gy_blocks, mask_blocks);
  else dcn_weight_colsum_block<T>(wt, s, bounds + 1, id - gy_blocks - mask_blocks);
}

// The LDS scatter pays when its tile holds the reach of a brick's undeformed taps with a voxel to
// spare on either side (offsets beyond the tile still work, through the data kernel's atomics).
template <typename S>
static bool scatter_tile_applies(const DcnDims &s, int dtype) {
  // the scatter kernel keeps grad_output of its positions in registers: up to kScatterKeep slices
  // of 4 * kPiece output channels per group (128 for 16-bit tensors, 64 for fp32); wider layers
  // would repeat too much per 8-channel workgroup and keep the atomics
  if (s.opg > kScatterKeep * (dtype == MV_F32 ? 16 : 32)) return false;
  const int ed = (S::BD - 1) * s.sd + (s.kd - 1) * s.dd + 1, eh = (S::BH - 1) * s.sh + (s.kh - 1) * s.dh + 1,
            ew = (S::BW - 1) * s.sw + (s.kw - 1) * s.dw + 1;
  return (S::TD == 1 || ed + 2 <= S::TD) && eh + 2 <= S::TH && ew + 2 <= S::TW &&
         static_cast<long>(S::BD * S::BH * S::BW) * s.K < (1L << 20);
}

static size_t align256b(size_t v) { return (v + 255) / 256 * 256; }

bool dcn_mfma_backward_supported(const DcnDims &s, int dtype) {
  if (dtype != MV_F16 && dtype != MV_BF16 && dtype != MV_F32) return false;
  if (s.cpg % 32 || s.opg % 32 || s.cpd % 32) return false;
  if (s.B > 65535 || s.dg > 65535) return false;
  if (static_cast<long>(s.P) * s.Cin * 4 >= (1L << 31)) return false;  // 32-bit byte offsets
  return dcn_tap_supported(s, dtype);
}

// workspace: xt | gyt | weight fragments (16- and 8-channel blocks) | gxt (fp32) | gw (fp32) | gb (fp32) |
// the three maxima of the scatter scale (gxt .. maxima start at zero) | partial sums of the tap kernel
struct BackwardLayout {
  size_t xt, gyt, wb, wa, gxt, gw, gb, bounds, part, total;
};
// (the budget of an earlier design's column buffer, still stored and returned for callers that set it)
static std::atomic<size_t> &column_budget_cell() {
  static std::atomic<size_t> cell{[] {
    const char *e = getenv("MV_DCN_COLUMN_BYTES");
    return e ? static_cast<size_t>(strtoull(e, nullptr, 10)) : (static_cast<size_t>(1) << 30);
  }()};
  return cell;
}
void dcn_set_column_budget(size_t bytes) { column_budget_cell().store(bytes, std::memory_order_relaxed); }
size_t dcn_column_budget() { return column_budget_cell().load(std::memory_order_relaxed); }
static BackwardLayout backward_layout(const DcnDims &s, int dtype) {
  BackwardLayout l;
  const size_t es = dtype == MV_F32 ? 4 : 2;
  size_t at = 0;
  l.xt = at; at += align256b(static_cast<size_t>(s.B) * s.P * s.Cin * es);
  l.gyt = at; at += align256b(static_cast<size_t>(s.B) * s.Q * s.Cout * es);
  l.wb = at; at += align256b(static_cast<size_t>(s.Cout) * s.cpg * s.K * es);
  l.wa = at; at += align256b(2 * static_cast<size_t>(s.Cout) * s.cpg * s.K * es);  // 16 MFMA rows per 8 channels
  l.gxt = at; at += align256b(static_cast<size_t>(s.B) * s.P * s.Cin * 4);
  l.gw = at; at += align256b(static_cast<size_t>(s.Cout) * s.cpg * s.K * 4);
  l.gb = at; at += align256b(static_cast<size_t>(s.Cout) * 4);
  l.bounds = at; at += 256;
  l.part = at; at += align256b(dcn_tap_partial_bytes(s, dtype));
  l.total = at;
  return l;
}

size_t dcn_mfma_backward_workspace_bytes(const DcnDims &s, int dtype) { return backward_layout(s, dtype).total; }

template <typename T>
static int backward_run(const void *x, const void *off, const void *mask, const void *wt,
                        const void *gy, void *goff, void *gmask, const DcnDims &real, const DcnPad &pad, void *workspace,
                        float **gx32, float **gw32, float **gb32, int dtype, bool want_bias, hipStream_t stream) {
  const DcnDims &s = pad.p;
  const BackwardLayout l = backward_layout(s, dtype);
  char *ws = static_cast<char *>(workspace);
  T *xt = reinterpret_cast<T *>(ws + l.xt), *gyt = reinterpret_cast<T *>(ws + l.gyt), *wb = reinterpret_cast<T *>(ws + l.wb);
  float *gxt = reinterpret_cast<float *>(ws + l.gxt);
  *gx32 = gxt; *gw32 = reinterpret_cast<float *>(ws + l.gw); *gb32 = reinterpret_cast<float *>(ws + l.gb);
  const bool image = s.nd == 2;
  const bool tiles = image ? scatter_tile_applies<ImageBricks>(s, dtype) : scatter_tile_applies<VolumeBricks>(s, dtype);
  // 16-bit tensors: 32-bit cells and 16 channels per workgroup, while a term keeps enough bits
  const int terms = (image ? ImageBricks::BD * ImageBricks::BH * ImageBricks::BW
                           : VolumeBricks::BD * VolumeBricks::BH * VolumeBricks::BW) * s.K;
  const bool narrow = sizeof(T) == 2 && scatter32_shift(terms) >= kScatter32MinShift;
  T *wa = narrow ? wb : reinterpret_cast<T *>(ws + l.wa);   // (16-channel blocks: those of the tap kernel)
  unsigned *bounds = reinterpret_cast<unsigned *>(ws + l.bounds);
  const long frag_lanes = static_cast<long>(s.groups) * s.K * (s.cpg / 16) * (s.opg / (4 * Mfma<T>::kPiece)) * 64;
  const long scatter_lanes = tiles && !narrow ? static_cast<long>(s.groups) * s.K * (s.cpg / 8) * (s.opg / (4 * Mfma<T>::kPiece)) * 64 : 0;
  const long nz = static_cast<long>((l.part - l.gxt) / 4);
  const long ngy = static_cast<long>(s.B) * real.Cout * s.Q, nmask = static_cast<long>(s.B) * s.dg * s.K * s.Q;
  const long ncols = static_cast<long>(s.groups) * real.cpg * s.K;
  constexpr int CH = 128 / static_cast<int>(sizeof(T));   // channels of a move
  const long px = (s.P + kMovePos - 1) / kMovePos, pq = (s.Q + kMovePos - 1) / kMovePos;
  const long nx = px * s.B * ((s.Cin + CH - 1) / CH), ngyb = pq * s.B * ((s.Cout + CH - 1) / CH);
  const long nf16 = (frag_lanes + 255) / 256, nfsc = (scatter_lanes + 255) / 256, nzb = min((nz + 1023) / 1024, 4096L);
  MV_REQUIRE(nx + ngyb + nf16 + nfsc + nzb < (1L << 31), "volume too large");
  PrepareJobs j;
  j.x_end = static_cast<unsigned>(nx); j.gy_end = j.x_end + static_cast<unsigned>(ngyb);
  j.f16_end = j.gy_end + static_cast<unsigned>(nf16); j.fsc_end = j.f16_end + static_cast<unsigned>(nfsc);
  j.zero_end = j.fsc_end + static_cast<unsigned>(nzb);
  j.px = static_cast<unsigned>(px); j.pq = static_cast<unsigned>(pq);
  hipLaunchKernelGGL((dcn_backward_prepare_kernel<T>), dim3(j.zero_end), dim3(256), 0, stream, static_cast<const T *>(x), xt,
                     static_cast<const T *>(gy), gyt, static_cast<const T *>(wt), wb, wa, gxt, nz, real, pad, j);
  if (tiles || want_bias) {
    const long slab_len = gy_slab_len(real);
    const long sum_blocks = static_cast<long>(real.Cout) * s.B * ((s.Q + slab_len - 1) / slab_len);
    const unsigned gy_blocks = static_cast<unsigned>(want_bias ? sum_blocks : min((ngy + 8191) / 8192, 256L));
    const unsigned mask_blocks = mask && tiles ? static_cast<unsigned>(min((nmask + 8191) / 8192, 256L)) : 0u;
    const unsigned col_blocks = tiles ? static_cast<unsigned>((ncols + 63) / 64) : 0u;
    MV_REQUIRE(sum_blocks < (1L << 30), "grid too large");
    hipLaunchKernelGGL((dcn_backward_maxima_kernel<T>), dim3(gy_blocks + mask_blocks + col_blocks), dim3(256), 0, stream,
                       static_cast<const T *>(gy), ngy, static_cast<const T *>(mask), nmask, static_cast<const T *>(wt), real,
                       tiles ? bounds : nullptr, want_bias ? *gb32 : nullptr, slab_len, gy_blocks, mask_blocks);
  }
  int st = check_launch("dcn_backward_prepare_kernel");
  if (st) return st;
  st = dcn_tap_backward(xt, off, mask, gyt, wb, gxt, goff, gmask, reinterpret_cast<float *>(ws + l.part), *gw32, s,
                        tiles ? bounds : nullptr, dtype, stream);
  if (st || !tiles) return st;
  MV_REQUIRE(s.Cin / 8 <= 65535, "grid too large");
#define MV_LAUNCH_SCATTER(S)                                                                                      \
  {                                                                                                               \
    const long nbd = (s.Do + S::BD - 1) / S::BD, nbh = (s.Ho + S::BH - 1) / S::BH, nbw = (s.Wo + S::BW - 1) / S::BW; \
    MV_REQUIRE(nbd * nbh * nbw < (1L << 31), "grid too large");                                                   \
    if (narrow)                                                                                                   \
      hipLaunchKernelGGL((dcn_backward_scatter32_kernel<T, S>),                                                   \
                         dim3(static_cast<unsigned>(nbd * nbh * nbw), s.Cin / 16, s.B), dim3(kScatterWaves * 64), 0, \
                         stream, static_cast<const T *>(off), static_cast<const T *>(mask), gyt, wa, gxt, s,      \
                         static_cast<int>(nbh), static_cast<int>(nbw), bounds);                                   \
    else                                                                                                          \
      hipLaunchKernelGGL((dcn_backward_scatter_kernel<T, S>),                                                     \
                         dim3(static_cast<unsigned>(nbd * nbh * nbw), s.Cin / 8, s.B), dim3(kScatterWaves * 64), 0, \
                         stream, static_cast<const T *>(off), static_cast<const T *>(mask), gyt, wa, gxt, s,      \
                         static_cast<int>(nbh), static_cast<int>(nbw), bounds);                                   \
  }
  if (image) MV_LAUNCH_SCATTER(ImageBricks) else MV_LAUNCH_SCATTER(VolumeBricks)
#undef MV_LAUNCH_SCATTER
  return check_launch("dcn_backward_scatter_kernel");
}

// Runs the kernels of the layer, padded to channel counts that they take (`pad.p`; the layer itself when it has such):
// grad_offset / grad_mask are written, the fp32 gradients of input (channels-last) and weight (tap-major) of the padded
// layer and the bias accumulator (with `want_bias` the sums of grad_output over samples and positions) are
// returned for the caller to fold in.
int dcn_mfma_backward(const void *x, const void *off, const void *mask, const void *wt,
                      const void *gy, void *goff, void *gmask, const DcnDims &s, const DcnPad &pad, int dtype,
                      void *workspace, bool want_bias, float **gx32, float **gw32, float **gb32,
                      hipStream_t stream) {
  if (dtype == MV_F16)
    return backward_run<__half>(x, off, mask, wt, gy, goff, gmask, s, pad, workspace, gx32, gw32, gb32, dtype, want_bias, stream);
  if (dtype == MV_F32)
    return backward_run<float>(x, off, mask, wt, gy, goff, gmask, s, pad, workspace, gx32, gw32, gb32, dtype, want_bias, stream);
  return backward_run<__hip_bfloat16>(x, off, mask, wt, gy, goff, gmask, s, pad, workspace, gx32, gw32, gb32, dtype, want_bias, stream);
}

// dst [B, C, P] (element type of `dtype`) += src [B, P, C] fp32 (= src when not `accumulate`)
int planar_add_f32(const float *src, void *dst, int B, int C, long P, int dtype, bool accumulate, hipStream_t stream) {
  const long pblocks = (P + 63) / 64;
  MV_REQUIRE(pblocks < (1L << 31) && B <= 65535 && (C + kAddChunk - 1) / kAddChunk <= 65535, "volume too large");
  const dim3 grid(static_cast<unsigned>(pblocks), B, (C + kAddChunk - 1) / kAddChunk);
  const int mode = planar_add_mode(src, dst, C, P);
#define MV_PLANAR_ADD_AS(TYPE, MODE)                                                                                  \
  hipLaunchKernelGGL((dcn_planar_add_kernel<TYPE, MODE>), grid, dim3(256), 0, stream, src, static_cast<TYPE *>(dst), C, P, \
                     accumulate ? 1 : 0)
#define MV_PLANAR_ADD(TYPE)                                                                                           \
  do {                                                                                                               \
    if (mode == 2) MV_PLANAR_ADD_AS(TYPE, 2);                                                                         \
    else if (mode == 1) MV_PLANAR_ADD_AS(TYPE, 1);                                                                    \
    else MV_PLANAR_ADD_AS(TYPE, 0);                                                                                   \
  } while (0)
  if (dtype == MV_F16) MV_PLANAR_ADD(__half);
  else if (dtype == MV_F32) MV_PLANAR_ADD(float);
  else MV_PLANAR_ADD(__hip_bfloat16);
#undef MV_PLANAR_ADD
#undef MV_PLANAR_ADD_AS
  return check_launch("dcn_planar_add_kernel");
}

// grad_weight [Cout][cpg][K] += the tap-major fp32 accumulator [K][Cout][cpg] of the weight kernel
template <typename T>
__device__ __forceinline__ void dcn_weight_add_block(const float *__restrict__ acc, T *__restrict__ gw, const DcnDims &s, const DcnPad &pad,
                                                     const unsigned bid, const unsigned nblocks, const int accumulate) {
  const DcnDims &p = pad.p;
  const long n = static_cast<long>(s.Cout) * s.cpg * s.K;
  for (long i = bid * 256L + threadIdx.x; i < n; i += nblocks * 256L) {
    const int k = static_cast<int>(i % s.K), c = static_cast<int>(i / s.K % s.cpg), o = static_cast<int>(i / s.K / s.cpg);
    const int g = o / s.opg, u = c / pad.unit;
    const float v = acc[(static_cast<long>(k) * p.Cout + g * p.opg + o - g * s.opg) * p.cpg + u * pad.unit_p + c - u * pad.unit];
    gw[i] = store_cast<T>(accumulate ? load(gw + i) + v : v);
  }
}

// The folds behind the backward kernels in one launch: channels-last fp32 grad input -> grad_input,
// tap-major fp32 grad weight -> grad_weight, the fp32 bias sums -> grad_bias.
template <typename T, int MODE>
__global__ __launch_bounds__(256) void dcn_backward_fold_kernel(const float *__restrict__ gxt, T *__restrict__ gx,
                                                                const float *__restrict__ gw32, T *__restrict__ gw,
                                                                const float *__restrict__ gb32, T *__restrict__ gb,
                                                                const DcnDims s, const DcnPad pad, const unsigned pblocks,
                                                                const unsigned add_end, const unsigned weight_end,
                                                                const int accumulate) {
  __shared__ AddShared stage;
  const unsigned id = blockIdx.x;
  if (id < add_end)
    dcn_planar_add_mode<T, MODE>(stage, gxt, gx, s.Cin, s.P, id % pblocks, static_cast<int>((id / pblocks) % s.B),
                                       static_cast<int>(id / (pblocks * s.B)), accumulate, pad.p.Cin, pad.unit, pad.unit_p);
  else if (id < weight_end)
    dcn_weight_add_block<T>(gw32, gw, s, pad, id - add_end, weight_end - add_end, accumulate);
  else
    for (int o = threadIdx.x; o < s.Cout; o += 256) gb[o] = store_cast<T>((accumulate ? static_cast<float>(load(gb + o)) : 0.f) + gb32[o]);
}

// All three folds of a layer on the matrix-core path.
int dcn_backward_fold(const float *gxt, const float *gw32, const float *gb32, void *grad_input, void *grad_weight,
                      void *grad_bias, const DcnDims &s, const DcnPad &pad, int dtype, bool accumulate, hipStream_t stream) {
  const int mode = planar_add_mode(gxt, grad_input, pad.unit, s.P);
  const long pblocks = (s.P + 63) / 64, add_blocks = pblocks * s.B * ((s.Cin + kAddChunk - 1) / kAddChunk);
  const long n = static_cast<long>(s.Cout) * s.cpg * s.K, weight_blocks = min((n + 255) / 256, 1024L);
  const long bias_blocks = grad_bias ? 1 : 0;
  MV_REQUIRE(add_blocks + weight_blocks + bias_blocks < (1L << 31), "volume too large");
  const unsigned add_end = static_cast<unsigned>(add_blocks), weight_end = add_end + static_cast<unsigned>(weight_blocks);
#define MV_FOLD_AS(T, MODE)                                                                                          \
  hipLaunchKernelGGL((dcn_backward_fold_kernel<T, MODE>), dim3(weight_end + static_cast<unsigned>(bias_blocks)), dim3(256), 0, \
                     stream, gxt, static_cast<T *>(grad_input), gw32, static_cast<T *>(grad_weight),               \
                     gb32, static_cast<T *>(grad_bias), s, pad,                                                    \
                     static_cast<unsigned>(pblocks), add_end, weight_end, accumulate ? 1 : 0)
#define MV_FOLD(T)                                                                                                    \
  do {                                                                                                               \
    if (mode == 2) MV_FOLD_AS(T, 2);                                                                                  \
    else if (mode == 1) MV_FOLD_AS(T, 1);                                                                             \
    else MV_FOLD_AS(T, 0);                                                                                            \
  } while (0)
  if (dtype == MV_F16) MV_FOLD(__half);
  else if (dtype == MV_BF16) MV_FOLD(__hip_bfloat16);
  else MV_FOLD(float);
#undef MV_FOLD
#undef MV_FOLD_AS
  return check_launch("dcn_backward_fold_kernel");
}

}  // namespace mv
