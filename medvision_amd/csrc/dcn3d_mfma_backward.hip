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
// Scatter kernel (dcn_backward_scatter.hip; layers whose taps fit its tile): the corners that land near their
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
size_t dcn_tap_partial_bytes(const DcnDims &s, int dtype, size_t budget);
bool dcn_tap_supported(const DcnDims &s, int dtype);
int dcn_tap_backward(const void *xt, const void *off, const void *mask, const void *gyt, const void *wf,
                     float *gxt, void *goff, void *gmask, float *partial, size_t budget, float *gw, const DcnDims &s,
                     const unsigned *bounds, const ScatterShape &shape, int dtype, hipStream_t stream);
// dcn_backward_scatter.hip
bool dcn_scatter_plan(const DcnDims &s, int dtype, ScatterShape &shape);
int dcn_scatter(const void *off, const void *mask, const void *gyt, const void *wf, float *gxt, const DcnDims &s,
                const ScatterShape &shape, const unsigned *bounds, int dtype, hipStream_t stream);

// ---- layouts and folds -----------------------------------------------------------------------------
// Element (output channel o of the padded layer p, channel cl of its group, tap k) of the real layer's weight
template <typename T>
__device__ __forceinline__ T padded_weight(const T *__restrict__ wt, const DcnDims &s, const DcnPad &pad, int o, int cl, int k) {
  const int g = o / pad.p.opg, ol = o - g * pad.p.opg, u = cl / pad.unit_p, r = cl - u * pad.unit_p;
  return ol < s.opg && r < pad.unit ? wt[(static_cast<long>(g * s.opg + ol) * s.cpg + u * pad.unit + r) * s.K + k] : store_cast<T>(0.f);
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

// One pass over grad_output[b, o, .]: the sums of its rows into the fp32 bias accumulator and (`out` given) its largest magnitude as a
// bit pattern into *out.  About 512 workgroups in all — enough loads in flight for the memory system, and few enough for the
// atomics on the one word of the maximum, which retire one after the other (~10 ns each): a workgroup takes a slab of
// `slab_len` positions of a row, or (`rows` > 0: many rows) each of its wavefronts `rows` whole rows.
//   (2048 rows of 15 200 positions, fp16, a workgroup per row: 51 us; 26 us with a row per wavefront.  Rows that start at any element, in
//   the same 16-byte pieces: 15 251 positions 26 us, element by element 78 us.)
static long gy_rows(const DcnDims &s) { return static_cast<long>(s.Cout) * s.B; }
static long gy_slab_len(const DcnDims &s) {
  const long rows = gy_rows(s), slabs = std::max(1L, std::min((s.Q + 2047) / 2048, (512 + rows - 1) / rows));
  return ((s.Q + slabs - 1) / slabs + 1023) / 1024 * 1024;
}
static int gy_rows_per_wave(const DcnDims &s) {   // 0: slabs
  const long rows = gy_rows(s);
  return rows < 1024 ? 0 : static_cast<int>((rows + 2047) / 2048);
}
// sum and largest magnitude of src[q0 .. q_end), `threads` threads, PIECES independent 16-byte loads each, which have a sum each: an
// addition of a chain rounds by as much as the chain has grown (fp32, 8 rows of 15 200 positions and 64 threads: the bias gradient is
// off by 3.1e-7 (rms) with one sum per thread, 1.3e-7 with eight)
template <typename T, int PIECES>
__device__ __forceinline__ float gy_sum_max(const T *__restrict__ src, const long q0, const long q_end, const int thread, const int threads,
                                            float &m, bool &bad) {
  constexpr int V = 16 / static_cast<int>(sizeof(T));
  float sum[PIECES] = {};
  auto take = [&](T e, float &v) {
    const float x = static_cast<float>(load(&e));
    v += x;
    bad = bad || !(x == x);
    m = fmaxf(m, fabsf(x));
  };
  typedef unsigned int piece_t __attribute__((ext_vector_type(4), aligned(2)));   // (element alignment: the hardware takes it)
  const long groups = (q_end - q0) / V, rest = q0 + groups * V;
  const piece_t *pieces = reinterpret_cast<const piece_t *>(src + q0);
  for (long i = thread; i < groups; i += PIECES * threads) {
    union { u32x4 u; T e[V]; } raw[PIECES];
#pragma unroll
    for (int u = 0; u < PIECES; u++) raw[u].u = i + u * threads < groups ? static_cast<u32x4>(pieces[i + u * threads]) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int u = 0; u < PIECES; u++)
#pragma unroll
      for (int e = 0; e < V; e++) take(raw[u].e[e], sum[u]);
  }
  if (rest + thread < q_end) take(src[rest + thread], sum[0]);   // (fewer than V elements)
#pragma unroll
  for (int half = PIECES / 2; half > 0; half /= 2)
#pragma unroll
    for (int u = 0; u < half; u++) sum[u] += sum[u + half];
  return sum[0];
}
template <typename T>
__device__ __forceinline__ void dcn_gy_sum_max_block(const T *__restrict__ gy, float *__restrict__ gb32, unsigned *out,
                                                     const DcnDims s, const long slab_len, const int rows, const unsigned bid) {
  __shared__ float sums[4];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  float m = 0.f;
  bool bad = false;
  const long total = static_cast<long>(s.Cout) * s.B;
  if (rows > 0) {
    for (long r = (bid * 4L + wave) * rows, last = min(r + rows, total); r < last; r++) {   // (rows are [b][o])
      float v = gy_sum_max<T, 8>(gy + r * s.Q, 0, s.Q, lane, kWave, m, bad);
      for (int sh = 32; sh > 0; sh >>= 1) v += __shfl_xor(v, sh);
      if (lane == 0) atomicAdd(gb32 + r % s.Cout, v);
    }
    if (out) fold_max(bad ? 0x7fc00000u : __float_as_uint(m), out);
    return;
  }
  const unsigned slabs = static_cast<unsigned>((s.Q + slab_len - 1) / slab_len);
  const unsigned slab = bid % slabs, r = bid / slabs;
  const int b = static_cast<int>(r % s.B), o = static_cast<int>(r / s.B);
  const long q0 = static_cast<long>(slab) * slab_len;
  float v = gy_sum_max<T, 4>(gy + (static_cast<long>(b) * s.Cout + o) * s.Q, q0, min(q0 + slab_len, s.Q), threadIdx.x, 256, m, bad);
  for (int sh = 32; sh > 0; sh >>= 1) v += __shfl_xor(v, sh);
  if (lane == 0) sums[wave] = v;
  if (out) fold_max(bad ? 0x7fc00000u : __float_as_uint(m), out);   // (contains the barrier)
  else __syncthreads();
  if (threadIdx.x == 0) atomicAdd(gb32 + o, (sums[0] + sums[1]) + (sums[2] + sums[3]));
}

// The small jobs in front of the tap kernel in two launches (a dependent launch costs ~2.7 us before its first
// instruction, and kernels of a few microseconds do not fill the machine): first the two layout passes, the weight
// fragments and the zero fill of the accumulators and of the maxima's words; then the maxima and the bias sums, which need those
// words at zero.
struct PrepareJobs {
  unsigned x_end, gy_end, f16_end, zero_end;   // block ranges of the first launch
  unsigned px, pq;                                      // blocks of positions of the input / the output
};
template <typename T>
__global__ __launch_bounds__(256) void dcn_backward_prepare_kernel(const T *__restrict__ x, T *__restrict__ xt,
                                                                   const T *__restrict__ gy, T *__restrict__ gyt,
                                                                   const T *__restrict__ wt, T *__restrict__ wb,
                                                                   float *__restrict__ zero,
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
  } else {
    dcn_zero_f32_block(zero, nz, id - j.f16_end, j.zero_end - j.f16_end);
  }
}
template <typename T>
__global__ __launch_bounds__(256) void dcn_backward_maxima_kernel(const T *__restrict__ gy, const long ngy,
                                                                  const T *__restrict__ mask, const long nmask,
                                                                  const T *__restrict__ wt, const DcnDims s,
                                                                  unsigned *__restrict__ bounds, float *__restrict__ gb32,
                                                                  const long slab_len, const int rows, const unsigned gy_blocks,
                                                                  const unsigned mask_blocks) {
  const unsigned id = blockIdx.x;
  if (id < gy_blocks) {
    // with a bias gradient to form the pass over grad_output also sums it
    if (gb32) dcn_gy_sum_max_block<T>(gy, gb32, bounds, s, slab_len, rows, id);
    else dcn_absmax_block<T>(gy, ngy, bounds, id, gy_blocks);
  } else if (id < gy_blocks + mask_blocks) dcn_absmax_block<T>(mask, nmask, bounds + 2, id - gy_blocks, mask_blocks);
  else dcn_weight_colsum_block<T>(wt, s, bounds + 1, id - gy_blocks - mask_blocks);
}

static size_t align256b(size_t v) { return (v + 255) / 256 * 256; }

bool dcn_mfma_backward_supported(const DcnDims &s, int dtype) {
  if (dtype != MV_F16 && dtype != MV_BF16 && dtype != MV_F32) return false;
  if (s.cpg % 32 || s.opg % 32 || s.cpd % 32) return false;
  if (s.B > 65535 || s.dg > 65535) return false;
  if (static_cast<long>(s.P) * s.Cin * 4 >= (1L << 31)) return false;  // 32-bit byte offsets
  return dcn_tap_supported(s, dtype);
}

// workspace: xt | gyt | weight fragments | gxt (fp32) | gw (fp32) | gb (fp32) |
// the three maxima of the scatter scale (gxt .. maxima start at zero) | partial sums of the tap kernel
struct BackwardLayout {
  size_t xt, gyt, wb, gxt, gw, gb, bounds, part, total;
};
// Bytes that the partial sums may take: layers with more run in pieces (fewer taps or positions per launch).
static std::atomic<size_t> &column_budget_cell() {
  static std::atomic<size_t> cell{[] {
    const char *e = getenv("MV_DCN_COLUMN_BYTES");
    return e ? static_cast<size_t>(strtoull(e, nullptr, 10)) : (static_cast<size_t>(1) << 30);
  }()};
  return cell;
}
void dcn_set_column_budget(size_t bytes) { column_budget_cell().store(bytes, std::memory_order_relaxed); }
size_t dcn_column_budget() { return column_budget_cell().load(std::memory_order_relaxed); }
static BackwardLayout backward_layout(const DcnDims &s, int dtype, size_t budget) {
  BackwardLayout l;
  const size_t es = dtype == MV_F32 ? 4 : 2;
  size_t at = 0;
  l.xt = at; at += align256b(static_cast<size_t>(s.B) * s.P * s.Cin * es);
  l.gyt = at; at += align256b(static_cast<size_t>(s.B) * s.Q * s.Cout * es);
  l.wb = at; at += align256b(static_cast<size_t>(s.Cout) * s.cpg * s.K * es);
  l.gxt = at; at += align256b(static_cast<size_t>(s.B) * s.P * s.Cin * 4);
  l.gw = at; at += align256b(static_cast<size_t>(s.Cout) * s.cpg * s.K * 4);
  l.gb = at; at += align256b(static_cast<size_t>(s.Cout) * 4);
  l.bounds = at; at += 256;
  l.part = at; at += align256b(dcn_tap_partial_bytes(s, dtype, budget));
  l.total = at;
  return l;
}

size_t dcn_mfma_backward_workspace_bytes(const DcnDims &s, int dtype) { return backward_layout(s, dtype, dcn_column_budget()).total; }

template <typename T>
static int backward_run(const void *x, const void *off, const void *mask, const void *wt,
                        const void *gy, void *goff, void *gmask, const DcnDims &real, const DcnPad &pad, void *workspace,
                        float **gx32, float **gw32, float **gb32, int dtype, bool want_bias, hipStream_t stream) {
  const DcnDims &s = pad.p;
  const size_t budget = dcn_column_budget();
  const BackwardLayout l = backward_layout(s, dtype, budget);
  char *ws = static_cast<char *>(workspace);
  T *xt = reinterpret_cast<T *>(ws + l.xt), *gyt = reinterpret_cast<T *>(ws + l.gyt), *wb = reinterpret_cast<T *>(ws + l.wb);
  float *gxt = reinterpret_cast<float *>(ws + l.gxt);
  *gx32 = gxt; *gw32 = reinterpret_cast<float *>(ws + l.gw); *gb32 = reinterpret_cast<float *>(ws + l.gb);
  ScatterShape shape{};
  const bool tiles = dcn_scatter_plan(s, dtype, shape);
  unsigned *bounds = reinterpret_cast<unsigned *>(ws + l.bounds);
  const long frag_lanes = static_cast<long>(s.groups) * s.K * (s.cpg / 16) * (s.opg / (4 * Mfma<T>::kPiece)) * 64;
  const long nz = static_cast<long>((l.part - l.gxt) / 4);
  const long ngy = static_cast<long>(s.B) * real.Cout * s.Q, nmask = static_cast<long>(s.B) * s.dg * s.K * s.Q;
  const long ncols = static_cast<long>(s.groups) * real.cpg * s.K;
  constexpr int CH = 128 / static_cast<int>(sizeof(T));   // channels of a move
  const long px = (s.P + kMovePos - 1) / kMovePos, pq = (s.Q + kMovePos - 1) / kMovePos;
  const long nx = px * s.B * ((s.Cin + CH - 1) / CH), ngyb = pq * s.B * ((s.Cout + CH - 1) / CH);
  const long nf16 = (frag_lanes + 255) / 256, nzb = min((nz + 1023) / 1024, 4096L);
  MV_REQUIRE(nx + ngyb + nf16 + nzb < (1L << 31), "volume too large");
  PrepareJobs j;
  j.x_end = static_cast<unsigned>(nx); j.gy_end = j.x_end + static_cast<unsigned>(ngyb);
  j.f16_end = j.gy_end + static_cast<unsigned>(nf16); 
  j.zero_end = j.f16_end + static_cast<unsigned>(nzb);
  j.px = static_cast<unsigned>(px); j.pq = static_cast<unsigned>(pq);
  hipLaunchKernelGGL((dcn_backward_prepare_kernel<T>), dim3(j.zero_end), dim3(256), 0, stream, static_cast<const T *>(x), xt,
                     static_cast<const T *>(gy), gyt, static_cast<const T *>(wt), wb, gxt, nz, real, pad, j);
  if (tiles || want_bias) {
    const long slab_len = gy_slab_len(real);
    const int rows = gy_rows_per_wave(real);
    const long sum_blocks = rows > 0 ? (gy_rows(real) + 4L * rows - 1) / (4L * rows) : gy_rows(real) * ((s.Q + slab_len - 1) / slab_len);
    const unsigned gy_blocks = static_cast<unsigned>(want_bias ? sum_blocks : min((ngy + 8191) / 8192, 256L));
    const unsigned mask_blocks = mask && tiles ? static_cast<unsigned>(min((nmask + 8191) / 8192, 256L)) : 0u;
    const unsigned col_blocks = tiles ? static_cast<unsigned>((ncols + 63) / 64) : 0u;
    MV_REQUIRE(sum_blocks < (1L << 30), "grid too large");
    hipLaunchKernelGGL((dcn_backward_maxima_kernel<T>), dim3(gy_blocks + mask_blocks + col_blocks), dim3(256), 0, stream,
                       static_cast<const T *>(gy), ngy, static_cast<const T *>(mask), nmask, static_cast<const T *>(wt), real,
                       tiles ? bounds : nullptr, want_bias ? *gb32 : nullptr, slab_len, rows, gy_blocks, mask_blocks);
  }
  int st = check_launch("dcn_backward_prepare_kernel");
  if (st) return st;
  st = dcn_tap_backward(xt, off, mask, gyt, wb, gxt, goff, gmask, reinterpret_cast<float *>(ws + l.part), budget, *gw32, s,
                        tiles ? bounds : nullptr, shape, dtype, stream);
  return st || !tiles ? st : dcn_scatter(off, mask, gyt, wb, gxt, s, shape, bounds, dtype, stream);
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
