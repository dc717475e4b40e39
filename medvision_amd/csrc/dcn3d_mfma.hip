// Matrix-core forward of deformable layers on large volumes with 32 (fp16: or 64) channels and 64 output channels per group (16-bit
// tensors): the taps are worked out once per position and shared through LDS.  (dcn_forward_columns.hip: every other layer, the layouts of x and the
// weights, and the plan that both share.)
#include <cstdint>

#include "dcn_mfma.hpp"

namespace mv {

// A workgroup of four wavefronts owns 64 positions and alternates two phases
// per group of TG = 4 taps:
//   G  wavefront w takes tap w of the group with ONE position per lane (the offset planes are read
//      as 128 contiguous bytes), and leaves the 8 corner offsets and 8 mask-scaled weights as a
//      64-byte record in LDS; all lanes also bring the group's weight pieces into LDS;
//   B  wavefront w takes positions 16 w .. 16 w + 15 in the load layout (position l / 4, piece
//      l % 4), reads each tap's record as four broadcast 16-byte LDS reads, gathers, blends and
//      moves the piece to the matrix layout (position l % 16, piece l / 16) and multiplies.
// The offsets of the next group are requested a whole B phase ahead; no barrier separates the samples of a group from
// its products, and the registers leave room for five wavefronts per SIMD.  One convolution group must lie inside one
// deformable group, and a tap's weight pieces (SLICES x MB x 1 KB) are kept to 8 KB.
template <typename T, int SLICES>
__global__ __launch_bounds__(256, 5) void dcn_forward_shared_taps_kernel(
    const T *__restrict__ xt, const T *__restrict__ off, const T *__restrict__ mask,
    const T *__restrict__ wf, const T *__restrict__ bias, T *__restrict__ y, const DcnDims s) {
  using M = Mfma<T>;
  constexpr int PC = M::kPiece, SL = 4 * PC, ES = sizeof(T), TG = 4;
  constexpr int NC = 8, MB = 4;                   // corners; blocks of 16 output channels
  static_assert(sizeof(T) == 2, "16-bit tensors");
  constexpr int REC = 2 * NC;                     // dwords per record: NC corner offsets, NC weights
  constexpr int WT = SLICES * MB * 64;            // 16-byte weight pieces per tap
  constexpr int WREG = (TG * WT + 255) / 256;     // pieces a thread moves per group
  constexpr unsigned kOutside = 0x80000000u;      // beyond the buffer: such loads return zeros
  __shared__ __attribute__((aligned(16))) unsigned rec[TG][64][REC];
  __shared__ __attribute__((aligned(16))) u32x4 wl[TG * WT];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int j = lane % 16, kc = lane / 16;   // matrix layout: position (column) and piece of this lane
  const int lj = lane / 4, lk = lane % 4;    // load layout
  const int from = (4 * j + kc) * 4;         // ds_bpermute byte address of the lane holding this lane's piece
  // The workgroup's 64 positions are a brick of 8 x 4 x 2 output voxels (8 x 8 of a single slice):
  // their corners overlap far more than those of 64 positions along a row, which is what the vector
  // L1 sees.  Local index l of the brick is voxel (l / 32, (l / 8) % 4, l % 8); positions of a
  // brick that reach past the volume are dead.
  const int bdz = s.Do > 1 ? 2 : 1, bhy = 8 / bdz;
  const int nbw = (s.Wo + 7) / 8, nbh = (s.Ho + bhy - 1) / bhy;
  const int wg = xcd_contiguous(blockIdx.x, gridDim.x);
  const int w0 = (wg % nbw) * 8, h0 = ((wg / nbw) % nbh) * bhy, d0 = (wg / (nbw * nbh)) * bdz;
  auto position = [&](int l) -> long {   // linear output position of local index l, -1 when dead
    const int ow = w0 + l % 8, oh = h0 + (l / 8) % bhy, od = d0 + l / (8 * bhy);
    return (ow < s.Wo && oh < s.Ho && od < s.Do) ? (static_cast<long>(od) * s.Ho + oh) * s.Wo + ow : -1;
  };
  const int g = blockIdx.y, b = blockIdx.z;
  const int dgi = g * s.cpg / s.cpd;
  const long bg = static_cast<long>(b) * s.dg + dgi;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(xt + static_cast<long>(b) * s.P * s.Cin), 0, static_cast<int>(s.P * s.Cin * ES), 0x00020000);

  // phase G: this lane's position, its grid origin, and the planes it reads (scalar offsets per
  // tap and component; sizes below 2^31 bytes are checked by the host)
  const long qg = position(lane);
  const bool live = qg >= 0;
  const long qgc = live ? qg : s.Q - 1;
  float base_d, base_h, base_w;
  {
    const int ow = qgc % s.Wo, oh = (qgc / s.Wo) % s.Ho, od = qgc / (static_cast<long>(s.Wo) * s.Ho);
    base_d = static_cast<float>(od * s.sd - s.pd); base_h = static_cast<float>(oh * s.sh - s.ph);
    base_w = live ? static_cast<float>(ow * s.sw - s.pw) : -1e30f;   // a dead lane's samples are void
  }
  const int plane_bytes = static_cast<int>(s.Q) * ES;
  const __amdgpu_buffer_rsrc_t offr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(off + bg * 3 * s.K * s.Q), 0, 3 * s.K * plane_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t maskr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(mask ? mask + bg * s.K * s.Q : off), 0, mask ? s.K * plane_bytes : 0, 0x00020000);
  const unsigned q_bytes = static_cast<unsigned>(qgc) * ES;
  auto as_float = [](unsigned short bits) { T t; __builtin_memcpy(&t, &bits, 2); return load(&t); };
  // d, h, w offsets and the mask value of tap k, requested one group ahead (a tap beyond the
  // last one reads zeros: scalar offsets take part in the range check)
  unsigned short rd = 0, rh = 0, rw = 0, rm = 0;
  auto request = [&](int k) {
    const int first = 3 * k * plane_bytes;
    rd = __builtin_amdgcn_raw_buffer_load_b16(offr, q_bytes, first, 0);
    rh = __builtin_amdgcn_raw_buffer_load_b16(offr, q_bytes, first + plane_bytes, 0);
    rw = __builtin_amdgcn_raw_buffer_load_b16(offr, q_bytes, first + 2 * plane_bytes, 0);
    rm = __builtin_amdgcn_raw_buffer_load_b16(maskr, q_bytes, k * plane_bytes, 0);
  };
  // element strides of the channels-last input in bytes, and the corner offsets relative to the first
  const unsigned cb = s.Cin * ES, wb = static_cast<unsigned>(s.W) * cb, hwb = static_cast<unsigned>(s.H) * wb;
  // the group's weight pieces: piece `id` of the group = (tap id / WT, slice, block, lane)
  // (in wf [block][tap][slice][lane]; taps beyond the last one are loaded and not used)
  constexpr int tap_bytes = SLICES * 64 * 16;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(wf + static_cast<long>(g) * MB * s.K * SLICES * (64 * PC)), 0, MB * s.K * tap_bytes, 0x00020000);
  unsigned wsrc[WREG];
#pragma unroll
  for (int i = 0; i < WREG; i++) {
    const int id = i * 256 + tid, t = id / WT, rem = id % WT;
    const int ln = rem % 64, m = (rem / 64) % MB, cc = rem / (64 * MB);
    wsrc[i] = id < TG * WT ? static_cast<unsigned>(((m * s.K + t) * SLICES + cc) * 1024 + ln * 16) : kOutside;
  }

  float4_t acc[MB];
#pragma unroll
  for (int m = 0; m < MB; m++) acc[m] = float4_t{0.f, 0.f, 0.f, 0.f};

  // tap of this wavefront in the current group as (i, j, k) kernel indices: advanced by TG per group
  const int khw = s.kh * s.kw;
  int ki = wave / khw, kj = (wave % khw) / s.kw, kk = wave % s.kw;
  request(wave);
  for (int k0 = 0; k0 < s.K; k0 += TG) {
    const int taps = min(TG, s.K - k0);
    // ---- G: the group's weight pieces (requested first, stored last) and this wavefront's tap ----
    u32x4 wreg[WREG];
#pragma unroll
    for (int i = 0; i < WREG; i++) wreg[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, wsrc[i], k0 * tap_bytes, 0);
    const int k = k0 + wave;
    if (k < s.K) {
      const float m = mask ? as_float(rm) : 1.f;
      const float pd = base_d + static_cast<float>(ki * s.dd) + as_float(rd);
      const float ph = base_h + static_cast<float>(kj * s.dh) + as_float(rh);
      const float pw = base_w + static_cast<float>(kk * s.dw) + as_float(rw);
      // A corner is inside iff its index is: with f = floor(p) the low one iff 0 <= f < size, the
      // high one iff 0 <= f + 1 < size (a sample at -1 exactly keeps a high corner of weight 0).
      const float fd = floorf(pd), fh = floorf(ph), fw = floorf(pw);
      const float ld = pd - fd, lh = ph - fh, lw = pw - fw;
      // (huge positions saturate in the conversion and fail the unsigned comparisons)
      const int id = static_cast<int>(fd), ih = static_cast<int>(fh), iw = static_cast<int>(fw);
      const bool vd0 = static_cast<unsigned>(id) < static_cast<unsigned>(s.D), vd1 = static_cast<unsigned>(id + 1) < static_cast<unsigned>(s.D);
      const bool vh0 = static_cast<unsigned>(ih) < static_cast<unsigned>(s.H), vh1 = static_cast<unsigned>(ih + 1) < static_cast<unsigned>(s.H);
      const bool vw0 = static_cast<unsigned>(iw) < static_cast<unsigned>(s.W), vw1 = static_cast<unsigned>(iw + 1) < static_cast<unsigned>(s.W);
      const unsigned first = static_cast<unsigned>(id) * hwb + static_cast<unsigned>(ih) * wb + static_cast<unsigned>(iw) * cb;
      const float md1 = m * ld, md0 = m - md1;   // mask times the depth weights
      const float wh1 = lh, wh0 = 1.f - lh, ww1 = lw, ww0 = 1.f - lw;
      const float hw00 = wh0 * ww0, hw01 = wh0 * ww1, hw10 = wh1 * ww0, hw11 = wh1 * ww1;
      unsigned at[8];
      float w[8];
      at[0] = (vd0 && vh0 && vw0) ? first : kOutside;                 w[0] = md0 * hw00;
      at[1] = (vd0 && vh0 && vw1) ? first + cb : kOutside;            w[1] = md0 * hw01;
      at[2] = (vd0 && vh1 && vw0) ? first + wb : kOutside;            w[2] = md0 * hw10;
      at[3] = (vd0 && vh1 && vw1) ? first + wb + cb : kOutside;       w[3] = md0 * hw11;
      at[4] = (vd1 && vh0 && vw0) ? first + hwb : kOutside;           w[4] = md1 * hw00;
      at[5] = (vd1 && vh0 && vw1) ? first + hwb + cb : kOutside;      w[5] = md1 * hw01;
      at[6] = (vd1 && vh1 && vw0) ? first + hwb + wb : kOutside;      w[6] = md1 * hw10;
      at[7] = (vd1 && vh1 && vw1) ? first + hwb + wb + cb : kOutside; w[7] = md1 * hw11;
      unsigned *r = rec[wave][lane];
#pragma unroll
      for (int c = 0; c < NC; c += 4) {
        *reinterpret_cast<u32x4 *>(r + c) = u32x4{at[c], at[c + 1], at[c + 2], at[c + 3]};
        *reinterpret_cast<u32x4 *>(r + NC + c) = u32x4{__float_as_uint(w[c]), __float_as_uint(w[c + 1]),
                                                      __float_as_uint(w[c + 2]), __float_as_uint(w[c + 3])};
      }
    }
    request(k + TG);
    kk += TG;
    while (kk >= s.kw) { kk -= s.kw; kj++; }
    while (kj >= s.kh) { kj -= s.kh; ki++; }
#pragma unroll
    for (int i = 0; i < WREG; i++)
      if (i * 256 + tid < TG * WT) wl[i * 256 + tid] = wreg[i];
    __syncthreads();
    // ---- B: positions 16 * wave .. + 15, every tap of the group -----------------------------------
    for (int t = 0; t < taps; t++) {
      const unsigned *r = rec[t][16 * wave + lj];
      unsigned at[NC];
      float cw[NC];
#pragma unroll
      for (int c = 0; c < NC; c += 4) {
        const u32x4 a = *reinterpret_cast<const u32x4 *>(r + c), w4 = *reinterpret_cast<const u32x4 *>(r + NC + c);
        at[c] = a.x + lk * 16u; at[c + 1] = a.y + lk * 16u; at[c + 2] = a.z + lk * 16u; at[c + 3] = a.w + lk * 16u;
        cw[c] = __uint_as_float(w4.x); cw[c + 1] = __uint_as_float(w4.y);
        cw[c + 2] = __uint_as_float(w4.z); cw[c + 3] = __uint_as_float(w4.w);
      }
#pragma unroll
      for (int cc = 0; cc < SLICES; cc++) {
        const unsigned c0 = g * s.cpg + cc * SL;
        u32x4 raw[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) raw[c] = __builtin_amdgcn_raw_buffer_load_b128(xr, at[c], c0 * ES, 0);
        float v[PC];
#pragma unroll
        for (int i = 0; i < PC; i++) v[i] = 0.f;
#pragma unroll
        for (int c = 0; c < NC; c++) M::fma_piece(v, cw[c], raw[c]);
        const u32x4 mine = M::pack(v);   // piece lk of position lj; wanted: piece kc of position j
        const u32x4 bpiece = u32x4{
            static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(from, static_cast<int>(mine.x))),
            static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(from, static_cast<int>(mine.y))),
            static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(from, static_cast<int>(mine.z))),
            static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(from, static_cast<int>(mine.w)))};
#pragma unroll
        for (int mm = 0; mm < MB; mm++) acc[mm] = M::run16(wl[t * WT + (cc * MB + mm) * 64 + lane], bpiece, acc[mm]);
      }
    }
    __syncthreads();   // records and weight pieces may be overwritten
  }
  const long qo = position(16 * wave + j);
  if (qo < 0) return;
  // 16x16 accumulator layout: register r of lane l holds row 4 * (l / 16) + r, column l % 16.
  // All bias values first (the lane's four channels of a block are 8 contiguous bytes; no bias: an
  // empty range), then the stores: a load between two stores would wait for the first.
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T *>(bias), 0, bias ? s.Cout * ES : 0, 0x00020000);
  u32x2 braw[MB];
#pragma unroll
  for (int m = 0; m < MB; m++)
    braw[m] = __builtin_amdgcn_raw_buffer_load_b64(br, (g * s.opg + m * 16 + kc * 4) * ES, 0, 0);
#pragma unroll
  for (int m = 0; m < MB; m++) {
    const float bv[4] = {M::lo(braw[m].x), M::hi(braw[m].x), M::lo(braw[m].y), M::hi(braw[m].y)};
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int o = g * s.opg + m * 16 + kc * 4 + r;
      y[(static_cast<long>(b) * s.Cout + o) * s.Q + qo] = store_cast<T>(acc[m][r] + bv[r]);
    }
  }
}

// The layers that this kernel serves: volumes of many bricks (below four workgroups per compute unit the columns
// kernel's smaller ones win: 44 us against 30 us for fp16 [4, 64 -> 64, 16 x 38 x 26], stride 2), all of a group's channels in one
// slice (fp16: or two) of one deformable group, and 64 output channels.  There it is the faster one: fp16 [2, 32 -> 64, 32^3] 57 us
// against 64 us, bf16 55 and 63, fp16 [64 -> 64, 48^3] 152 and 159.  It repeats the samples for every 64 output channels, which the columns
// kernel shares among 256 (bf16 [2, 32 -> 128, 32^3] 95 against 78 us, fp16 [2, 64 -> 256, 32^3] 279 and 162); bf16 with 64 channels leaves
// it three wavefronts per SIMD (64 -> 64 48^3 192 against 167 us); and its bricks have to be full (fp16 [2, 32 -> 64, 37 x 29 x 33],
// 73 % of the positions alive: 73 against 69 us; 64 -> 64 120 and 107; [4, 64 -> 64, 9 x 45 x 51], 77 %: 136 and 124).
int dcn_shared_taps_forward(const void *xt, const void *off, const void *mask, const void *wf, const void *bias, void *y,
                            const DcnDims &s, int dtype, hipStream_t stream) {
  const int slices = s.cpg / 32;
  // bricks of 8 x 4 x 2 output voxels (8 x 8 of a single slice), one per workgroup
  const int bdz = s.Do > 1 ? 2 : 1, bhy = 8 / bdz;
  const long bricks = static_cast<long>((s.Wo + 7) / 8) * ((s.Ho + bhy - 1) / bhy) * ((s.Do + bdz - 1) / bdz);
  if (s.nd != 3 || s.cpg % 32 || slices < 1 || slices > (dtype == MV_F16 ? 2 : 1) || s.cpd % s.cpg || s.opg != 64 || bricks * s.B < 1024 ||
      s.Q * 20 < bricks * (64 * 17) || bricks >= (1L << 31) || s.groups > 65535 || 3L * s.K * s.Q * 2 >= (1L << 31) ||
      static_cast<long>(s.K) * slices * 4 * 1024 >= (1L << 31))
    return -1;
  const dim3 grid(static_cast<unsigned>(bricks), s.groups, s.B), block(256);
#define MV_SHARED_TAPS(T, SLICES)                                                                                     \
  hipLaunchKernelGGL((dcn_forward_shared_taps_kernel<T, SLICES>), grid, block, 0, stream, static_cast<const T *>(xt), \
                     static_cast<const T *>(off), static_cast<const T *>(mask), static_cast<const T *>(wf),           \
                     static_cast<const T *>(bias), static_cast<T *>(y), s)
  if (dtype == MV_F16) { if (slices == 1) MV_SHARED_TAPS(__half, 1); else MV_SHARED_TAPS(__half, 2); }
  else MV_SHARED_TAPS(__hip_bfloat16, 1);
#undef MV_SHARED_TAPS
  return check_launch("dcn_forward_shared_taps_kernel");
}

}  // namespace mv
