// gemm.hip — prefill-regime (m > 16) block-quantized GEMMs whose block sums are
// scaled in f32, on CDNA4 MFMA: f32 activations, and int8 activations
// (rq_quantize_act_i8).
//
// y[m, o] = sum_b scale[o, b] * P_b[m, o],  P_b = sum_{k in block b} x[m, k] * code[o, k]
//
// Raster's staged contraction (raster/compiler/ir/contract_stages.clj:25-31):
// the codes enter v_mfma_f32_32x32x16_bf16 as bf16 integers, which is exact
// (|code| <= 128 needs 8 significand bits), so every product is exact in f32;
// the f32 block scale then multiplies the f32 partial of the block (one FMA per
// output per block). x is carried as bf16 hi + lo (x = hi + lo + O(2^-17 |x|)),
// two MFMAs per product.
//
// int8 activations (qmatmul-i8-gemm!, raster/quant/kernels_k.clj:357-370, and the
// Q4_0 form of qmatmul-q4-composable, raster/quant/kernels.clj:140-184):
//   y[t, o] = sum_b ws[o, b] * xs[t, b] * dot_b(code[o] [- 8], xq[t])
// The codes of both sides enter the bf16 MFMA as exact integers (the Q4_0 zero
// point subtracted from the code, which is the -8 xsum fold) and a block's sum,
// below 2^19, is exact in f32: no int32 result to convert, and no sums to fold.
//
// Bound, f32 activations: the MFMAs (twice the bf16 GEMM's) and, at the operand rates of a CU,
// the activations: 4 bytes per element, so a fragment is loaded once per wave
// and used for 96 or 192 columns. Measured (128 x 96 tile, per MFMA and wave):
// 24 ns, of it 16.5 the MFMA itself, about 4 the activation loads and the
// producers, 2 the LDS reads, 2 the block scaling.
#include <algorithm>

#include "rq_internal.h"

namespace rq {

namespace {

typedef float f32x32 __attribute__((ext_vector_type(32)));

constexpr int kGbBlocks = 4;  // 32-blocks per step

// x = hi + lo, both RNE bf16, eight elements
__device__ __forceinline__ void split8(const f32x4& v0, const f32x4& v1, u32x4& hi, u32x4& lo) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float a = i < 2 ? v0[2 * i] : v1[2 * i - 4], b = i < 2 ? v0[2 * i + 1] : v1[2 * i - 3];
    hi[i] = pack2_bf16(a, b);
    lo[i] = pack2_bf16(a - __uint_as_float(hi[i] << 16), b - __uint_as_float(hi[i] & 0xFFFF0000u));
  }
}

// Reads from one array, at a lane's offset plus a uniform one: 32-bit offsets into a
// buffer resource, or (WIDE) 64-bit addresses.
template <bool WIDE>
struct Src {
  using Off = uint32_t;
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Src(const void* p, int64_t bytes) : r(buffer_rsrc(p, (uint32_t)bytes)) {}
  __device__ __forceinline__ u32x4 b128(Off v, Off s) const {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)v, (int)s, 0));
  }
  __device__ __forceinline__ u32x2 b64(Off v, Off s) const {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)s, 0));
  }
  __device__ __forceinline__ uint32_t b32(Off v, Off s) const {
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0);
  }
  __device__ __forceinline__ uint32_t b16(Off v, Off s) const {
    return __builtin_amdgcn_raw_buffer_load_b16(r, (int)v, (int)s, 0);
  }
};
template <>
struct Src<true> {
  using Off = uint64_t;
  const uint8_t* p;
  bool any;
  __device__ __forceinline__ Src(const void* q, int64_t bytes) : p(static_cast<const uint8_t*>(q)), any(bytes != 0) {}
  template <typename T>
  __device__ __forceinline__ T at(Off v, Off s) const {
    return any ? *reinterpret_cast<const T*>(p + v + s) : T{};
  }
  __device__ __forceinline__ u32x4 b128(Off v, Off s) const { return at<u32x4>(v, s); }
  __device__ __forceinline__ u32x2 b64(Off v, Off s) const { return at<u32x2>(v, s); }
  __device__ __forceinline__ uint32_t b32(Off v, Off s) const { return at<uint32_t>(v, s); }
  __device__ __forceinline__ uint32_t b16(Off v, Off s) const { return at<uint16_t>(v, s); }
};

// Blocks past the last one, which fill up a step, add zeros: rereading the last
// block and scaling its sum by 0 would make NaN where y is infinite. f32
// activations, whose sums can overflow, read as zero there, out of a resource of
// no bytes; the int8 sums cannot, so the codes there are the next tile's (zeros
// after the last), with scales from the zeros that each tile's scales end with.
template <bool WIDE>
struct ActBlock {
  using Off = typename Src<WIDE>::Off;
  Src<WIDE> x;
  Off off;  // of the block
  __device__ __forceinline__ ActBlock(const void* p, uint32_t x_bytes, int kb, int nkb, uint32_t block_bytes)
      : x(p, kb < nkb ? x_bytes : 0u), off(kb < nkb ? (Off)kb * block_bytes : 0u) {}
};

// bytes of the packed activations: bf16 hi + lo, or (int8) f32 block scales, of one
// block more per tile, and bf16 codes, of one block more
int64_t packed_bytes(int x_dtype, int64_t m, int64_t k) {
  const int64_t m32 = (m + 31) / 32 * 32;
  return x_dtype == kXtI8 ? m32 * (k / 32 + 1) * 4 + m32 * k * 2 + 2048 : m32 * k * 4;
}

}  // namespace

// x[M][K] (f32) -> xf[M/32][K/32][hi, lo][2][64][8] bf16: fragment (tile, kb,
// hl, j), lane l = row l % 32 of the tile, k = 32 kb + 16 (l / 32) + 8 j + 0..7.
// Rows up to the next multiple of 32 are zero. A workgroup copies 32 rows x 64 k.
__global__ __launch_bounds__(256) void pack_x32_split_kernel(const float* __restrict__ x, uint16_t* __restrict__ xf,
                                                             int M, int K) {
  const int nkb = K / 32, nq = (nkb + 1) / 2;
  const int tile = blockIdx.x / nq, kb = (blockIdx.x % nq) * 2 + ((threadIdx.x & 7) >> 2);
  if (kb >= nkb) return;
  const int row = threadIdx.x >> 3, cc = threadIdx.x & 3;  // 8-k chunk cc of the k-step
  const int m = tile * 32 + row;
  f32x4 v0 = {0.0f, 0.0f, 0.0f, 0.0f}, v1 = v0;
  if (m < M) {
    const f32x4* p = reinterpret_cast<const f32x4*>(x + (int64_t)m * K + 32 * kb + 8 * cc);
    v0 = p[0];
    v1 = p[1];
  }
  u32x4 hi, lo;
  split8(v0, v1, hi, lo);
  const int j = cc & 1, lane = row + 32 * (cc >> 1);
  u32x4* dst = reinterpret_cast<u32x4*>(xf) + (((int64_t)tile * nkb + kb) * 4 + j) * 64 + lane;
  dst[0] = hi;
  dst[128] = lo;
}

// int8 codes xq[M][K] and their block scales xs[M][K/32] -> the scales as
// [M/32][K/32 + 1][32], a tile's last block zero, and after them the same fragments
// (codes as bf16, exact) and a block of zeros.
__global__ __launch_bounds__(256) void pack_x32_i8_kernel(const int8_t* __restrict__ xq, const float* __restrict__ xs,
                                                          uint16_t* __restrict__ xf, int M, int K) {
  const int nkb = K / 32, nq = (nkb + 1) / 2;
  const int tile = blockIdx.x / nq, kb = (blockIdx.x % nq) * 2 + ((threadIdx.x & 7) >> 2);
  if (kb >= nkb) return;
  const int row = threadIdx.x >> 3, cc = threadIdx.x & 3;  // 8-k chunk cc of the k-step
  const int m = tile * 32 + row;
  u32x2 v = {0u, 0u};
  if (m < M) v = *reinterpret_cast<const u32x2*>(xq + (int64_t)m * K + 32 * kb + 8 * cc);
  const u32x2 p = q8_dword_bf16(v[0], 1.0f), q = q8_dword_bf16(v[1], 1.0f);
  const int64_t at = (int64_t)tile * nkb + kb;
  const int tiles = (M + 31) / 32;
  float* sf = reinterpret_cast<float*>(xf) + (at + tile) * 32 + row;
  u32x4* cf = reinterpret_cast<u32x4*>(reinterpret_cast<float*>(xf) + (int64_t)tiles * (nkb + 1) * 32) +
              (at * 2 + (cc & 1)) * 64 + row + 32 * (cc >> 1);
  cf[0] = u32x4{p[0], p[1], q[0], q[1]};
  if (cc == 0) sf[0] = m < M ? xs[(int64_t)m * nkb + kb] : 0.0f;
  if (kb == nkb - 1) {
    if (cc == 1) sf[32] = 0.0f;
    if (tile == tiles - 1) cf[128] = u32x4{0u, 0u, 0u, 0u};
  }
}

// Workgroup: WM x KG waves; tile 32 MF WM rows x 32 NF columns, a wave 32 MF x
// 32 NF of it over the steps s (of four 32-blocks) with s % KG = its kg (their
// sums are added in kg order at the end). All waves convert the next KG steps'
// codes to bf16 (16 codes per thread and task) into the other half of a
// double-buffered LDS ring while the current ones compute; one barrier per KG
// steps. Activation fragments go straight into registers, a block ahead: from
// the packed copy, or (PK false: calls that have no scratch) from x itself,
// split in registers, with the same result. WIDE: rows so long that a tile's
// weights or activations pass 4 GiB.
template <int FMT, typename ST, int XT, bool PK, bool WIDE, int MF, int NF, int WM, int KG>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WM * KG, 64 * WM * KG), amdgpu_waves_per_eu(1))) void
gemm_blk_kernel(const uint8_t* __restrict__ q, const ST* __restrict__ sc, const void* __restrict__ x,
                void* __restrict__ y, int M, int K, int N, int npad, int y_dtype, int tiles_m, uint32_t x_bytes) {
  constexpr int T = 64 * WM * KG, NB = kGbBlocks;
  constexpr int BM = 32 * MF * WM, BN = 32 * NF;
  constexpr int G = BN / 16;                 // 16-row weight groups of the tile
  constexpr int NT = G * KG * NB * 32 / T;   // conversion tasks per thread and step
  constexpr int NS = (BN * KG * NB + T - 1) / T;  // scales per thread and step
  constexpr bool I8 = XT == kXtI8;
  constexpr int AF = I8 ? 2 : 4;             // 16-byte pieces of an activation fragment
  static_assert(NT * T == G * KG * NB * 32, "whole tasks");
  struct Lds {
    u32x4 w[2][KG][NB][2][NF][64];  // code fragments [buffer][kg][block][half j][32-column fragment][lane]
    float s[2][KG][NB][BN];
  };
  constexpr int kRed = KG > 1 ? (KG - 1) * BM * BN * 4 : 16;
  __shared__ __attribute__((aligned(16))) uint8_t smem[sizeof(Lds) > kRed ? sizeof(Lds) : kRed];
  Lds& L = *reinterpret_cast<Lds*>(smem);

  const int nblk = (int)gridDim.x, bid = (int)blockIdx.x;
  // the row tiles of a column tile adjacent, each XCD a contiguous run
  const int xcd = bid & 7, per = nblk >> 3, rem = nblk & 7;
  const int tord = xcd * per + (xcd < rem ? xcd : rem) + (bid >> 3);
  const int tm = tord % tiles_m, tn = tord / tiles_m;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, kg = wave / WM;
  const int l32 = lane & 31, g = lane >> 5;
  const int nkb = K / 32, steps = (nkb + NB - 1) / NB, turns = (steps + KG - 1) / KG;
  const int n0 = tn * BN, m0 = tm * BM + wm * 32 * MF;

  // ---- conversion tasks: task t = tid + T i is row t % 16, half t / 16 % 2 of
  // block t / 32 % NB of kg t / 32 / NB % KG of the tile's 16-row group
  // t / 32 / NB / KG (clamped to the padded rows; blocks past the last one
  // reread it and get zero scales)
  constexpr uint32_t CB = FMT == RQ_Q8_0 ? 512u : 256u, RB = FMT == RQ_Q8_0 ? 32u : 16u;
  constexpr uint32_t HB = RB / 2;
  // the tile's own groups: offsets that do not grow with the weight's rows
  using Off = typename Src<WIDE>::Off;
  const int g0 = n0 / 16, g_last = min(G, npad / 16 - g0) - 1;
  const Src<WIDE> qs(q + (int64_t)g0 * nkb * CB, (int64_t)(g_last + 1) * nkb * CB);
  const Src<WIDE> ss(sc + (int64_t)g0 * nkb * 16, (int64_t)(g_last + 1) * nkb * 16 * (int)sizeof(ST));
  const int tr = tid & 15, th = (tid >> 4) & 1;
  u32x4 raw[NT];
  uint32_t rs[NS];
  auto wload = [&](int turn) {
#pragma unroll
    for (int i = 0; i < NT; i++) {
      const int u = (tid + T * i) >> 5, b = u % NB, k = u / NB % KG;
      const Off grp = (Off)min(u / NB / KG, g_last);
      const Off kb = (Off)min((turn * KG + k) * NB + b, nkb - 1);
      const Off off = (grp * (Off)nkb + kb) * CB + (Off)tr * RB + (Off)th * HB;
      if (FMT == RQ_Q8_0) {
        raw[i] = qs.b128(off, 0);
      } else {
        const u32x2 v = qs.b64(off, 0);
        raw[i] = u32x4{v[0], v[1], 0u, 0u};
      }
    }
#pragma unroll
    for (int i = 0; i < NS; i++) {
      // scale t = tid + T i: row t % 16 of block t / 16 % NB, kg, group as above
      const int t = tid + T * i, b = (t >> 4) % NB, k = (t >> 4) / NB % KG;
      const Off grp = (Off)min((t >> 4) / NB / KG, g_last);
      const int kb = (turn * KG + k) * NB + b;
      const Off off = ((grp * (Off)nkb + (Off)min(kb, nkb - 1)) * 16 + (Off)(t & 15)) * sizeof(ST);
      rs[i] = sizeof(ST) == 4 ? ss.b32(off, 0) : ss.b16(off, 0);
      if (kb >= nkb) rs[i] = 0u;
    }
  };
  auto wstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NT; i++) {
      const int u = (tid + T * i) >> 5, b = u % NB, k = u / NB % KG, grp = u / NB / KG;
      const int n = 16 * (grp & 1) + tr;
      if (FMT == RQ_Q8_0) {
        // 16 codes k = 16 th + 0..15: half j = 0 the first eight, j = 1 the rest
        u32x2 p[4];
#pragma unroll
        for (int d = 0; d < 4; d++) p[d] = q8_dword_bf16(raw[i][d], 1.0f);
        L.w[buf][k][b][0][grp >> 1][n + 32 * th] = u32x4{p[0][0], p[0][1], p[1][0], p[1][1]};
        L.w[buf][k][b][1][grp >> 1][n + 32 * th] = u32x4{p[2][0], p[2][1], p[3][0], p[3][1]};
      } else {
        // bytes 8 th + 0..7: low nibbles k = 8 th + 0..7 (lanes of half 0),
        // high nibbles 16 + 8 th + 0..7 (half 1), both j = th
#pragma unroll
        for (int h = 0; h < 2; h++) {
          uint32_t d[2] = {(raw[i][0] >> (4 * h)) & 0x0F0F0F0Fu, (raw[i][1] >> (4 * h)) & 0x0F0F0F0Fu};
          asm("" : "+v"(d[0]), "+v"(d[1]));  // byte-select conversions instead of a bit-field extract per nibble
          uint32_t o[4];
#pragma unroll
          for (int e = 0; e < 2; e++) {
            o[2 * e] = pack2_bf16((float)(d[e] & 0xFFu) - 8.0f, (float)((d[e] >> 8) & 0xFFu) - 8.0f);
            o[2 * e + 1] = pack2_bf16((float)((d[e] >> 16) & 0xFFu) - 8.0f, (float)(d[e] >> 24) - 8.0f);
          }
          L.w[buf][k][b][th][grp >> 1][n + 32 * h] = u32x4{o[0], o[1], o[2], o[3]};
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NS; i++) {
      const int t = tid + T * i, b = (t >> 4) % NB, k = (t >> 4) / NB % KG, grp = (t >> 4) / NB / KG;
      if (NS * T == BN * KG * NB || grp < G) L.s[buf][k][b][16 * grp + (t & 15)] = scale_from_bits<ST>(rs[i]);
    }
  };

  // ---- this wave's activation fragments: rows m0 + 32 f + lane % 32
  const int r32_last = (M + 31) / 32 - 1;
  const Off xc = I8 ? (Off)(r32_last + 1) * (Off)(nkb + 1) * 128u : 0u;  // I8: the codes, after the scales
  Off xo[MF], so[MF];
#pragma unroll
  for (int f = 0; f < MF; f++) {
    const Off t32 = (Off)min(m0 / 32 + f, r32_last);
    xo[f] = PK ? xc + t32 * (Off)nkb * (1024u * AF) + 16u * (Off)lane
               : (Off)min(m0 + 32 * f + l32, M - 1) * (Off)nkb * 128u + 64u * (Off)g;
    so[f] = t32 * (Off)(nkb + 1) * 128u + 16u * (Off)g;
  }
  u32x4 a[2][MF][AF];     // PK: hi j 0, 1, f32: lo j 0, 1; else the 16 f32
  f32x4 xs[2][I8 ? MF : 1][4];  // I8: the scales of rows 8 q + 4 g + 0..3
  auto aload = [&](int slot, int kb) {
    if constexpr (I8) {
      const Src<WIDE> src(x, x_bytes);
      const Off k = (Off)min(kb, nkb);
#pragma unroll
      for (int f = 0; f < MF; f++) {
#pragma unroll
        for (int i = 0; i < AF; i++) a[slot][f][i] = src.b128(xo[f] + 1024u * i, k * 2048u);
#pragma unroll
        for (int i = 0; i < 4; i++)
          xs[slot][f][i] = __builtin_bit_cast(f32x4, src.b128(so[f] + 32u * i, k * 128u));
      }
    } else {
      const ActBlock<WIDE> b(x, x_bytes, kb, nkb, PK ? 4096u : 128u);
#pragma unroll
      for (int f = 0; f < MF; f++)
#pragma unroll
        for (int i = 0; i < AF; i++) a[slot][f][i] = b.x.b128(xo[f] + (PK ? 1024u : 16u) * i, b.off);
    }
  };

  f32x16 acc[MF][NF];
#pragma unroll
  for (int f = 0; f < MF; f++)
#pragma unroll
    for (int c = 0; c < NF; c++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[f][c][e] = 0.0f;
  f32x16 zero;
#pragma unroll
  for (int e = 0; e < 16; e++) zero[e] = 0.0f;

  wload(0);
  aload(0, kg * NB);
  wstore(0);
  wload(1);
  __syncthreads();
  for (int t = 0; t < turns; t++) {
    const int buf = t & 1, kb0 = (t * KG + kg) * NB;
    wstore(buf ^ 1);
    wload(t + 2);
#pragma unroll
    for (int b = 0; b < NB; b++) {
      aload((b + 1) & 1, b + 1 < NB ? kb0 + b + 1 : kb0 + KG * NB);
      bf16x8 h[MF][2], l[MF][2];
#pragma unroll
      for (int f = 0; f < MF; f++) {
        const u32x4* r = a[b & 1][f];
#pragma unroll
        for (int j = 0; j < 2; j++) {
          u32x4 hv = r[j], lv = r[j];
          if (PK) {
            if (!I8) lv = r[AF - 2 + j];
          } else {
            split8(__builtin_bit_cast(f32x4, r[2 * j % AF]), __builtin_bit_cast(f32x4, r[(2 * j + 1) % AF]), hv, lv);
          }
          h[f][j] = __builtin_bit_cast(bf16x8, hv);
          l[f][j] = __builtin_bit_cast(bf16x8, lv);
        }
      }
#pragma unroll
      for (int c = 0; c < NF; c++) {
        const bf16x8 w0 = __builtin_bit_cast(bf16x8, L.w[buf][kg][b][0][c][lane]);
        const bf16x8 w1 = __builtin_bit_cast(bf16x8, L.w[buf][kg][b][1][c][lane]);
        const float s = L.s[buf][kg][b][32 * c + l32];
#pragma unroll
        for (int f = 0; f < MF; f++) {
          f32x16 p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h[f][0], w0, zero, 0, 0, 0);
          p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h[f][1], w1, p, 0, 0, 0);
          if (!I8) {
            p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l[f][0], w0, p, 0, 0, 0);
            p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l[f][1], w1, p, 0, 0, 0);
          }
#pragma unroll
          for (int e = 0; e < 16; e++)
            acc[f][c][e] = fmaf(I8 ? s * xs[b & 1][I8 ? f : 0][e / 4][e % 4] : s, p[e], acc[f][c][e]);
        }
      }
    }
    __syncthreads();
  }

  if (KG > 1) {
    // the kg waves' sums through LDS, added in kg order
    f32x16* red = reinterpret_cast<f32x16*>(smem);
    constexpr int W = WM * MF * NF * 64;
    const int at = wm * MF * NF * 64 + lane;
    if (kg > 0) {
#pragma unroll
      for (int f = 0; f < MF; f++)
#pragma unroll
        for (int c = 0; c < NF; c++) red[(kg - 1) * W + at + (f * NF + c) * 64] = acc[f][c];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int k = 0; k < KG - 1; k++)
#pragma unroll
      for (int f = 0; f < MF; f++)
#pragma unroll
        for (int c = 0; c < NF; c++) acc[f][c] += red[k * W + at + (f * NF + c) * 64];
  }

  // acc[f][c] register e: m = m0 + 32 f + 8 (e / 4) + 4 g + e % 4, n = n0 + 32 c + lane % 32
#pragma unroll
  for (int f = 0; f < MF; f++)
#pragma unroll
    for (int c = 0; c < NF; c++) {
      const int n = n0 + 32 * c + l32;
      if (n >= N) continue;
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int m = m0 + 32 * f + 8 * (e >> 2) + 4 * g + (e & 3);
        if (m >= M) continue;
        if (y_dtype == RQ_F32)
          static_cast<float*>(y)[(int64_t)m * N + n] = acc[f][c][e];
        else
          static_cast<uint16_t*>(y)[(int64_t)m * N + n] = (uint16_t)f32_to_bf16_bits(acc[f][c][e]);
      }
    }
}

// Role-split form for the larger tiles: eight waves, waves 0..3 (consumers) 32
// rows x 32 NF columns each, waves 4..7 (producers) load the codes RW - 1 steps
// ahead and convert step s + 2 into LDS buffer (s + 2) % 3 while the consumers
// run step s. A wave's loads complete in issue order, so a wave that loads both
// would wait for its codes (HBM) whenever it waits for activations (L2).
template <int FMT, typename ST, int XT, bool PK, int NF, int RA>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void gemm_blk_rs_kernel(
    const uint8_t* __restrict__ q, const ST* __restrict__ sc, const void* __restrict__ x, void* __restrict__ y, int M,
    int K, int N, int npad, int y_dtype, int tiles_m, uint32_t x_bytes) {
  constexpr int NB = kGbBlocks, RW = 3;
  constexpr int BM = 128, BN = 32 * NF, G = BN / 16;
  constexpr int NT = G * NB * 32 / 256;
  constexpr int NS = (BN * NB + 255) / 256;
  constexpr int TPS = NB * NF;  // tiles per step
  static_assert(NB % RA == 0 && (XT == kXtI8 ? NF % 2 == 0 : TPS % 3 == 0 && TPS % 4 == 0), "rings turn whole in a step");
  struct Lds {
    u32x4 w[3][NB][2][NF][64];
    float s[3][NB][BN];
  };
  __shared__ __attribute__((aligned(16))) Lds L;
  const int nblk = (int)gridDim.x, bid = (int)blockIdx.x;
  const int xcd = bid & 7, per = nblk >> 3, rem = nblk & 7;
  const int tord = xcd * per + (xcd < rem ? xcd : rem) + (bid >> 3);
  const int tm = tord % tiles_m, tn = tord / tiles_m;
  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nkb = K / 32, steps = (nkb + NB - 1) / NB;
  const int n0 = tn * BN;

  if (wave >= 4) {
    // ---- producer
    constexpr uint32_t CB = FMT == RQ_Q8_0 ? 512u : 256u, RB = FMT == RQ_Q8_0 ? 32u : 16u;
    constexpr uint32_t HB = RB / 2;
    const int g0 = n0 / 16, g_last = min(G, npad / 16 - g0) - 1;
    const __amdgpu_buffer_rsrc_t qr =
        buffer_rsrc(q + (int64_t)g0 * nkb * CB, (uint32_t)(g_last + 1) * (uint32_t)nkb * CB);
    const __amdgpu_buffer_rsrc_t sr =
        buffer_rsrc(sc + (int64_t)g0 * nkb * 16, (uint32_t)(g_last + 1) * (uint32_t)nkb * 16 * (uint32_t)sizeof(ST));
    const int tr = tid & 15, th = (tid >> 4) & 1;
    u32x4 raw[RW][NT];
    uint32_t rs[RW][NS];
    auto wload = [&](int slot, int step) {
#pragma unroll
      for (int i = 0; i < NT; i++) {
        const int u = (tid + 256 * i) >> 5, b = u % NB;
        const uint32_t grp = (uint32_t)min(u / NB, g_last);
        const uint32_t kb = (uint32_t)min(step * NB + b, nkb - 1);
        const uint32_t off = (grp * (uint32_t)nkb + kb) * CB + (uint32_t)tr * RB + (uint32_t)th * HB;
        if (FMT == RQ_Q8_0) {
          raw[slot][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(qr, (int)off, 0, 0));
        } else {
          const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(qr, (int)off, 0, 0));
          raw[slot][i] = u32x4{v[0], v[1], 0u, 0u};
        }
      }
#pragma unroll
      for (int i = 0; i < NS; i++) {
        const int t = tid + 256 * i, b = (t >> 4) % NB;
        const uint32_t grp = (uint32_t)min((t >> 4) / NB, g_last);
        const uint32_t kb = (uint32_t)min(step * NB + b, nkb - 1);
        const uint32_t off = ((grp * (uint32_t)nkb + kb) * 16 + (uint32_t)(t & 15)) * sizeof(ST);
        if (sizeof(ST) == 4)
          rs[slot][i] = __builtin_amdgcn_raw_buffer_load_b32(sr, (int)off, 0, 0);
        else
          rs[slot][i] = __builtin_amdgcn_raw_buffer_load_b16(sr, (int)off, 0, 0);
      }
    };
    auto wstore = [&](int slot, int buf, int step) {
#pragma unroll
      for (int i = 0; i < NT; i++) {
        const int u = (tid + 256 * i) >> 5, b = u % NB, grp = u / NB;
        const int n = 16 * (grp & 1) + tr;
        if (FMT == RQ_Q8_0) {
          u32x2 p[4];
#pragma unroll
          for (int d = 0; d < 4; d++) p[d] = q8_dword_bf16(raw[slot][i][d], 1.0f);
          L.w[buf][b][0][grp >> 1][n + 32 * th] = u32x4{p[0][0], p[0][1], p[1][0], p[1][1]};
          L.w[buf][b][1][grp >> 1][n + 32 * th] = u32x4{p[2][0], p[2][1], p[3][0], p[3][1]};
        } else {
#pragma unroll
          for (int h = 0; h < 2; h++) {
            uint32_t d[2] = {(raw[slot][i][0] >> (4 * h)) & 0x0F0F0F0Fu, (raw[slot][i][1] >> (4 * h)) & 0x0F0F0F0Fu};
            asm("" : "+v"(d[0]), "+v"(d[1]));
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 2; e++) {
              o[2 * e] = pack2_bf16((float)(d[e] & 0xFFu) - 8.0f, (float)((d[e] >> 8) & 0xFFu) - 8.0f);
              o[2 * e + 1] = pack2_bf16((float)((d[e] >> 16) & 0xFFu) - 8.0f, (float)(d[e] >> 24) - 8.0f);
            }
            L.w[buf][b][th][grp >> 1][n + 32 * h] = u32x4{o[0], o[1], o[2], o[3]};
          }
        }
      }
#pragma unroll
      for (int i = 0; i < NS; i++) {
        const int t = tid + 256 * i, b = (t >> 4) % NB, grp = (t >> 4) / NB;
        if (grp < G) L.s[buf][b][16 * grp + (t & 15)] = step * NB + b < nkb ? scale_from_bits<ST>(rs[slot][i]) : 0.0f;
      }
    };
#pragma unroll
    for (int s = 0; s < RW; s++) wload(s, s);
    wstore(0, 0, 0);
    wload(0, 3);
    wstore(1, 1, 1);
    wload(1, 4);
    __syncthreads();
    for (int s0 = 0; s0 < steps; s0 += 3) {
#pragma unroll
      for (int u = 0; u < 3; u++) {
        if (s0 + u < steps) {
          wstore((u + 2) % 3, (u + 2) % 3, s0 + u + 2);
          wload((u + 2) % 3, s0 + u + 5);
          __syncthreads();
        }
      }
    }
    return;
  }

  // ---- consumer
  const int l32 = lane & 31, g = lane >> 5;
  const int m0 = tm * BM + wave * 32;
  const int r32_last = (M + 31) / 32 - 1;
  f32x16 zero, acc[NF];
#pragma unroll
  for (int e = 0; e < 16; e++) zero[e] = 0.0f;
#pragma unroll
  for (int c = 0; c < NF; c++) acc[c] = zero;
  if constexpr (XT == kXtI8) {
    f32x32 zero2;
#pragma unroll
    for (int e = 0; e < 32; e++) zero2[e] = 0.0f;
    // int8 activations. Tiles in pairs of column fragments; the scales of a pair's
    // outputs, xs[row] ws[column], come from one 32x32x1 two-block f32 MFMA (one
    // rounding, as a multiply; 32 cycles a tile where 16 multiplies on the VALU
    // cost about 70 beside the FMAs that wait for them), issued ahead of the next
    // pair's MFMAs, beside which the pair before is scaled
    const uint32_t t32 = (uint32_t)min(m0 / 32, r32_last);
    const uint32_t so = t32 * (uint32_t)(nkb + 1) * 128u + 4u * (uint32_t)l32;
    const uint32_t xo = (uint32_t)(r32_last + 1) * (uint32_t)(nkb + 1) * 128u + t32 * (uint32_t)nkb * 2048u +
                        16u * (uint32_t)lane;
    constexpr int NP = NF / 2, TP = NB * NP;  // pairs per block and step
    const Src<false> xr(x, x_bytes);
    u32x4 a[RA][2];
    float xs[RA];
    auto aload = [&](int slot, int kb) {
      const uint32_t k = (uint32_t)min(kb, nkb);
#pragma unroll
      for (int i = 0; i < 2; i++) a[slot][i] = xr.b128(xo + 1024u * i, k * 2048u);
      xs[slot] = __uint_as_float(xr.b32(so, k * 128u));
    };
    f32x16 p[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++) p[1][i] = zero;
    bf16x8 w[2][2][2];  // [slot][tile of the pair][half]
    float ws[2];        // lanes 0..31 the pair's first column fragment, 32..63 its second
    f32x32 sc2[2];      // scales of the pair's outputs
    sc2[1] = zero2;
    auto wread = [&](int slot, int buf, int b, int q) {
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) w[slot][i][j] = __builtin_bit_cast(bf16x8, L.w[buf][b][j][2 * q + i][lane]);
      ws[slot] = L.s[buf][b][64 * q + lane];
    };
#pragma unroll
    for (int i = 0; i < RA - 1; i++) aload(i, i);
    __syncthreads();
    wread(0, 0, 0, 0);
    int buf = 0;
    for (int s = 0; s < steps; s++) {
      const int nbuf = buf == 2 ? 0 : buf + 1;
#pragma unroll
      for (int i = 0; i < TP; i++) {
        const int b = i / NP, q = i % NP, cur = i & 1, q1 = (i + TP - 1) % TP % NP;
        if (q == 0) aload((b + RA - 1) % RA, s * NB + b + RA - 1);
        wread(cur ^ 1, i + 1 < TP ? buf : nbuf, (i + 1) / NP % NB, (i + 1) % NP);
        sc2[cur] = __builtin_amdgcn_mfma_f32_32x32x1f32(xs[b % RA], ws[cur], zero2, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int t = 0; t < 2; t++)
            p[cur][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[b % RA][j]), w[cur][t][j],
                                                                j > 0 ? p[cur][t] : zero, 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
          for (int e = 0; e < 16; e++)
            acc[2 * q1 + t][e] = fmaf(sc2[cur ^ 1][16 * t + e], p[cur ^ 1][t][e], acc[2 * q1 + t][e]);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 12, 0);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      buf = nbuf;
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int e = 0; e < 16; e++)
        acc[NF - 2 + t][e] = fmaf(sc2[1][16 * t + e], p[1][t][e], acc[NF - 2 + t][e]);
  } else {
    const uint32_t xo = PK ? (uint32_t)min(m0 / 32, r32_last) * (uint32_t)nkb * 4096u + 16u * (uint32_t)lane
                           : (uint32_t)min(m0 + l32, M - 1) * (uint32_t)nkb * 128u + 64u * (uint32_t)g;
    u32x4 a[RA][4];
    auto aload = [&](int slot, int kb) {
      const ActBlock<false> b(x, x_bytes, kb, nkb, PK ? 4096u : 128u);
#pragma unroll
      for (int i = 0; i < 4; i++) a[slot][i] = b.x.b128(xo + (PK ? 1024u : 16u) * i, b.off);
    };
    f32x16 p[3];  // the block sums in flight
#pragma unroll
    for (int i = 0; i < 3; i++) p[i] = zero;
    bf16x8 w[3][2];
    float ws[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // scales of the column fragments j - 2 .. j + 1
    bf16x8 h[2], l[2], lp[2];  // the block's hi and lo fragments; the last tile's lo of the block before
    const bf16x8 none = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
    w[2][0] = w[2][1] = lp[0] = lp[1] = none;
    auto wread = [&](int j, int buf, int b, int c) {
      w[j % 3][0] = __builtin_bit_cast(bf16x8, L.w[buf][b][0][c][lane]);
      w[j % 3][1] = __builtin_bit_cast(bf16x8, L.w[buf][b][1][c][lane]);
      ws[j % 4] = L.s[buf][b][32 * c + l32];
    };
#pragma unroll
    for (int i = 0; i < RA - 1; i++) aload(i, i);
    __syncthreads();
    wread(0, 0, 0, 0);
    int buf = 0;
    for (int s = 0; s < steps; s++) {
      const int nbuf = buf == 2 ? 0 : buf + 1;
      // tile j of the step: a block's column fragment. Its four MFMAs (hi, hi, lo, lo
      // of the two 16-k halves) are spread over two turns, so that two chains
      // alternate, and the block sums are scaled in the turn after, beside the MFMAs
      // of the next two tiles
#pragma unroll
      for (int j = 0; j < TPS; j++) {
        const int b = j / NF, c = j % NF;
        const int j1 = (j + TPS - 1) % TPS, j2 = (j + TPS - 2) % TPS;  // the tile before, and the one before it
        if (c == 0) {
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const u32x4* r = a[b % RA];
            u32x4 hv, lv;
            if (PK) {
              hv = r[e];
              lv = r[2 + e];
            } else {
              split8(__builtin_bit_cast(f32x4, r[2 * e]), __builtin_bit_cast(f32x4, r[2 * e + 1]), hv, lv);
            }
            h[e] = __builtin_bit_cast(bf16x8, hv);
            l[e] = __builtin_bit_cast(bf16x8, lv);
          }
        }
        wread(j + 1, j + 1 < TPS ? buf : nbuf, (j + 1) / NF % NB, (j + 1) % NF);
        const bool head = c == 0;  // the tile before is of the block before
        p[j % 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h[0], w[j % 3][0], zero, 0, 0, 0);
        p[j1 % 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(head ? lp[0] : l[0], w[j1 % 3][0], p[j1 % 3], 0, 0, 0);
        p[j % 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h[1], w[j % 3][1], p[j % 3], 0, 0, 0);
        p[j1 % 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(head ? lp[1] : l[1], w[j1 % 3][1], p[j1 % 3], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 16; e++) acc[j2 % NF][e] = fmaf(ws[j2 % 4], p[j2 % 3][e], acc[j2 % NF][e]);
        if (c == 0) aload((b + RA - 1) % RA, s * NB + b + RA - 1);
        if (c == NF - 1) {
          lp[0] = l[0];
          lp[1] = l[1];
        }
        if (PK) {
#pragma unroll
          for (int e = 0; e < 4; e++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      buf = nbuf;
    }
    {
      constexpr int j1 = TPS - 1, j2 = TPS - 2;
      p[j1 % 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lp[0], w[j1 % 3][0], p[j1 % 3], 0, 0, 0);
      p[j1 % 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lp[1], w[j1 % 3][1], p[j1 % 3], 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 16; e++) acc[j2 % NF][e] = fmaf(ws[j2 % 4], p[j2 % 3][e], acc[j2 % NF][e]);
#pragma unroll
      for (int e = 0; e < 16; e++) acc[j1 % NF][e] = fmaf(ws[j1 % 4], p[j1 % 3][e], acc[j1 % NF][e]);
    }
  }

#pragma unroll
  for (int c = 0; c < NF; c++) {
    const int n = n0 + 32 * c + l32;
    if (n >= N) continue;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int m = m0 + 8 * (e >> 2) + 4 * g + (e & 3);
      if (m >= M) continue;
      if (y_dtype == RQ_F32)
        static_cast<float*>(y)[(int64_t)m * N + n] = acc[c][e];
      else
        static_cast<uint16_t*>(y)[(int64_t)m * N + n] = (uint16_t)f32_to_bf16_bits(acc[c][e]);
    }
  }
}

template <int FMT, typename ST, int XT, bool PK, int NF, int RA>
static hipError_t launch_rs_t(const MatmulArgs& a, const void* x, void* y, int64_t m, hipEvent_t begin,
                           hipEvent_t done) {
  constexpr int BM = 128, BN = 32 * NF;
  const int64_t tiles_m = (m + BM - 1) / BM, tiles_n = (a.n + BN - 1) / BN;
  if (tiles_m * tiles_n > INT32_MAX) return hipErrorInvalidValue;
  const int64_t bytes = std::min<int64_t>(PK ? packed_bytes(XT, m, a.k) : m * a.k * 4, UINT32_MAX);
  hipExtLaunchKernelGGL((gemm_blk_rs_kernel<FMT, ST, XT, PK, NF, RA>), dim3((unsigned)(tiles_m * tiles_n)), dim3(512), 0,
                        a.stream, begin, done, 0, a.q, static_cast<const ST*>(a.scales), x, y, (int)m, (int)a.k,
                        (int)a.n, (int)a.npad, a.y_dtype, (int)tiles_m, (uint32_t)bytes);
  return hipGetLastError();
}

template <int FMT, typename ST, int XT, bool PK, int MF, int NF, int WM, int KG, bool WIDE = false>
static hipError_t launch_t(const MatmulArgs& a, const void* x, void* y, int64_t m, hipEvent_t begin,
                           hipEvent_t done) {
  constexpr int BM = 32 * MF * WM, BN = 32 * NF;
  const int64_t tiles_m = (m + BM - 1) / BM, tiles_n = (a.n + BN - 1) / BN;
  if (tiles_m * tiles_n > INT32_MAX) return hipErrorInvalidValue;
  const int64_t bytes = std::min<int64_t>(PK ? packed_bytes(XT, m, a.k) : m * a.k * 4, UINT32_MAX);
  hipExtLaunchKernelGGL((gemm_blk_kernel<FMT, ST, XT, PK, WIDE, MF, NF, WM, KG>), dim3((unsigned)(tiles_m * tiles_n)),
                        dim3(64 * WM * KG), 0, a.stream, begin, done, 0, a.q, static_cast<const ST*>(a.scales), x, y,
                        (int)m, (int)a.k, (int)a.n, (int)a.npad, a.y_dtype, (int)tiles_m, (uint32_t)bytes);
  return hipGetLastError();
}

namespace {

// The tiles. Time of a call, fitted to an MI355X with c = workgroups per CU
// (rounded up): K-blocks / kg x max(one_ns, c block_ns) + c round_ns. Measured,
// us a call with the packing pass, Q8_0, f32 y:
//                        32x32  64x32  128x64  128x96  128x192
//   11008 x 4096  m = 32  22.8   31.3    53.0    45.1    73.6
//                 m = 64  33.7   35.1    53.6    45.8    73.6
//                 m = 256 99.1   86.9    65.6    54.6    77.8
//                 m = 333 136    127     93.3    93.8    79.4
//                 m = 512 222    164     105     102     94.5
//   4096 x 4096   m = 256 45.8   38.1    55.3    48.2    76.8
//                 m = 768 190    108     70.9    99.2    80.3
// The kernel before these (one 128 x 128 tile, both operands converted in every
// workgroup, two barriers per 32-block) took 275 us at m = 333, 11008 x 4096
// (Q4_0).
struct BlkTile {
  int bm, bn, kg, one_ns, block_ns, round_ns;
};
constexpr BlkTile kF32Tiles[] = {{32, 32, 4, 310, 262, 0},
                                 {64, 32, 4, 500, 440, 0},
                                 {128, 64, 1, 360, 245, 0},
                                 {128, 96, 1, 315, 315, 4000},
                                 {128, 192, 1, 570, 570, 5000}};

// int8 activations, fitted alike. Measured, us a call with the packing pass, Q8_0,
// f32 y, against the kernel before (int8 MFMA, every int32 dot converted and
// scaled by the product of its two scales on the VALU; 32 x 64 to 64 x 128 tiles):
//                        before  32x32  128x64  128x128
//   11008 x 4096  m = 17   59.8   25.9    31.7    48.9
//                 m = 128  60.7   64      33.4    52
//                 m = 256  83.3  109      58.9    51.3
//                 m = 512 107.6  205      87.4    99.9
//                 m = 1024 227.5 429     170     150
//   4096 x 4096   m = 512  62.1   83.3    35.2    51.8
//   28672 x 2048  m = 512 141.5  306     115     111
constexpr BlkTile kI8Tiles[] = {{32, 32, 4, 340, 300, 0}, {128, 64, 1, 200, 200, 2500}, {128, 128, 1, 315, 315, 3500}};

int pick_tile(const BlkTile* table, int count, int64_t m, int64_t k, int64_t n, int cu_count) {
  int best = 0;
  int64_t best_cost = INT64_MAX;
  for (int i = 0; i < count; i++) {
    const BlkTile& t = table[i];
    const int64_t tiles = (m + t.bm - 1) / t.bm * ((n + t.bn - 1) / t.bn), c = (tiles + cu_count - 1) / cu_count;
    const int64_t cost = k / 32 * std::max<int64_t>(t.one_ns, c * t.block_ns) / t.kg + c * t.round_ns;
    if (cost < best_cost) best_cost = cost, best = i;
  }
  return best;
}

template <int FMT, typename ST, int XT, bool PK>
hipError_t launch_tile(int tile, const MatmulArgs& a, const void* x, void* y, int64_t m, hipEvent_t begin,
                           hipEvent_t done) {
  switch (tile) {
    case 0: return launch_t<FMT, ST, XT, PK, 1, 1, 1, 4>(a, x, y, m, begin, done);
    case 1: return launch_t<FMT, ST, XT, PK, 2, 1, 1, 4>(a, x, y, m, begin, done);
    case 2: return launch_t<FMT, ST, XT, PK, 1, 2, 4, 1>(a, x, y, m, begin, done);
    case 3: return launch_rs_t<FMT, ST, XT, PK, 3, 4>(a, x, y, m, begin, done);
    default: return launch_rs_t<FMT, ST, XT, PK, 6, 2>(a, x, y, m, begin, done);
  }
}

// Rows longer than this run the first tile with 64-bit addresses (WIDE): up to it the
// weights of the widest tile (192 columns, 16 B of Q8_0 codes per row and 16
// elements) and the least rows of packed int8 activations (32) stay within 32-bit
// offsets
constexpr int64_t kMaxK32 = (int64_t)1 << 24;
static_assert(192 * kMaxK32 <= UINT32_MAX && 32 * (2 * kMaxK32 + (kMaxK32 / 32 + 1) * 4) + 2048 <= UINT32_MAX,
              "32-bit offsets");

// Rows per launch: the packed copy within rq_qmatmul_noalloc's scratch, x within
// the 32-bit buffer offsets
int64_t chunk_rows(int64_t k, bool packed) {
  const int64_t rows = (packed ? (int64_t)RQ_NOALLOC_SCRATCH_MAX : (int64_t)UINT32_MAX) / (4 * k);
  return rows >= 256 ? rows / 256 * 256 : packed ? rows / 32 * 32 : std::max<int64_t>(rows, 1);
}

// int8: the packed copy within 64 MiB, at least 32 rows
int64_t i8_chunk_rows(int64_t k) {
  const int64_t rows = (int64_t)(64 << 20) / (2 * k + k / 8);
  return rows >= 256 ? rows / 256 * 256 : std::max<int64_t>(rows / 32 * 32, 32);
}

}  // namespace

size_t gemm_f32_pack_bytes(int64_t m, int64_t k) {
  return (size_t)(std::min((m + 31) / 32 * 32, chunk_rows(k, true)) * k * 4);
}

template <int FMT, typename ST>
static hipError_t launch_x(const MatmulArgs& a, int cu_count) {
  const bool pk = a.scratch != nullptr;
  if (a.k > kMaxK32)
    return launch_t<FMT, ST, RQ_F32, false, 1, 1, 1, 4, true>(a, a.x, a.y, a.m, a.ev_main[0], a.ev_main[1]);
  // of the whole call, whatever its chunks
  const int tile = pick_tile(kF32Tiles, 5, a.m, a.k, a.n, cu_count);
  const int64_t chunk = chunk_rows(a.k, pk);
  for (int64_t m0 = 0; m0 < a.m; m0 += chunk) {
    const int64_t m = std::min(chunk, a.m - m0);
    const float* x = static_cast<const float*>(a.x) + m0 * a.k;
    void* y = static_cast<uint8_t*>(a.y) + m0 * a.n * (a.y_dtype == RQ_F32 ? 4 : 2);
    const hipEvent_t done = m0 + chunk >= a.m ? a.ev_main[1] : nullptr;
    if (pk) {
      const int64_t blocks = (m + 31) / 32 * ((a.k / 32 + 1) / 2);
      hipExtLaunchKernelGGL(pack_x32_split_kernel, dim3((unsigned)blocks), dim3(256), 0, a.stream, nullptr,
                            m0 == 0 ? a.ev_main[0] : nullptr, 0, x, static_cast<uint16_t*>(a.scratch), (int)m,
                            (int)a.k);
      if (hipError_t e = hipGetLastError()) return e;
    }
    const hipError_t e = pk ? launch_tile<FMT, ST, RQ_F32, true>(tile, a, a.scratch, y, m, nullptr, done)
                            : launch_tile<FMT, ST, RQ_F32, false>(tile, a, x, y, m, m0 == 0 ? a.ev_main[0] : nullptr, done);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int FMT, typename ST>
static hipError_t launch_i8(const MatmulArgs& a, int cu_count) {
  const int64_t chunk = i8_chunk_rows(a.k), nb = a.k / 32;
  const int tile = a.k > kMaxK32 ? -1 : pick_tile(kI8Tiles, 3, a.m, a.k, a.n, cu_count);
  for (int64_t m0 = 0; m0 < a.m; m0 += chunk) {
    const int64_t m = std::min(chunk, a.m - m0);
    void* y = static_cast<uint8_t*>(a.y) + m0 * a.n * (a.y_dtype == RQ_F32 ? 4 : 2);
    const int64_t blocks = (m + 31) / 32 * ((nb + 1) / 2);
    hipExtLaunchKernelGGL(pack_x32_i8_kernel, dim3((unsigned)blocks), dim3(256), 0, a.stream, nullptr,
                          m0 == 0 ? a.ev_main[0] : nullptr, 0, static_cast<const int8_t*>(a.x) + m0 * a.k,
                          a.ops.act_scale + m0 * nb, static_cast<uint16_t*>(a.scratch), (int)m, (int)a.k);
    if (hipError_t e = hipGetLastError()) return e;
    const hipEvent_t done = m0 + chunk >= a.m ? a.ev_main[1] : nullptr;
    const hipError_t e =
        tile < 0    ? launch_t<FMT, ST, kXtI8, true, 1, 1, 1, 4, true>(a, a.scratch, y, m, nullptr, done)
        : tile == 0 ? launch_t<FMT, ST, kXtI8, true, 1, 1, 1, 4>(a, a.scratch, y, m, nullptr, done)
        : tile == 1 ? launch_rs_t<FMT, ST, kXtI8, true, 2, 4>(a, a.scratch, y, m, nullptr, done)
                    : launch_rs_t<FMT, ST, kXtI8, true, 4, 4>(a, a.scratch, y, m, nullptr, done);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

size_t gemm_i8_pack_bytes(int64_t m, int64_t k) {
  return (size_t)packed_bytes(kXtI8, std::min(m, i8_chunk_rows(k)), k);
}

hipError_t launch_gemm_i8(const MatmulArgs& a, int cu_count) {
  if (a.format == RQ_Q8_0) return launch_i8<RQ_Q8_0, float>(a, cu_count);
  if (a.scale_dtype == RQ_F16) return launch_i8<RQ_Q4_0, uint16_t>(a, cu_count);
  return launch_i8<RQ_Q4_0, float>(a, cu_count);
}

hipError_t launch_gemm(const MatmulArgs& a, int cu_count) {
  if (a.x_dtype != RQ_F32) return hipErrorInvalidValue;
  if (a.format == RQ_Q8_0) return launch_x<RQ_Q8_0, float>(a, cu_count);
  if (a.scale_dtype == RQ_F16) return launch_x<RQ_Q4_0, uint16_t>(a, cu_count);
  return launch_x<RQ_Q4_0, float>(a, cu_count);
}

}  // namespace rq
