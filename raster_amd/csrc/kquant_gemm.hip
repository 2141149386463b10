// kquant_gemm.hip — K-quant (Q4_K, Q6_K) GEMM on CDNA4 int8 MFMA, for more
// activation rows than the K-quant GEMV (kquant.hip) serves in a pass or two.
//
// y[t][o] = sum over super-blocks of 256 elements, with q8_K activations
// (quantize-act-q8k, raster/compiler/backend/cpu/quant.clj:158-176), of
//   Q4_K  d_act * (da * sum_j aq_j dot_j + db * sum_j bq_j bsum_j)
//   Q6_K  d_act * ds * sum_j sc_j (dot_j - 32 bsum_j)
// (qmatmul-q4k-dp4a! / qmatmul-q6k-dp4a!, raster/quant/kernels_k.clj:186-297).
// The sub-block scales are integers, so a super-block's sum is one: the kernel
// multiplies them into the codes and forms the whole 256-element sum exactly in
// int32, with one f32 scaling per output and super-block (the GEMV rounds once
// per sub-block). A scaled code needs up to 13 bits; it is carried as two int8
// digits, two MFMAs on the same activation fragment:
//   Q4_K  aq q = 8 (ah q) + (al q), aq = 8 ah + al <= 63: every digit <= 105
//         (weights with a larger aq keep the GEMV: Weight::kq_gemm)
//   Q6_K  sc (q - 32) = 256 h + l, l the signed low byte, |h| <= 16
// so v_mfma_i32_16x16x64_i8 runs at the cost per element of one bf16 MFMA. The
// Q4_K minimum term sum_j bq_j bsum_j is one 16x16x16 f16 MFMA per super-block
// and 16 x 16 outputs: bsum = 64 h + l, k slots 0..7 hold (64 bq_j, h_j) and
// 8..15 (bq_j, l_j); all exact in f16, the sum exact in f32.
#include <algorithm>

#include "rq_internal.h"

namespace rq {

namespace {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));

// one thread's share of a super-block: 16 codes of one weight row
template <int FMT>
struct KgRaw {
  u32x4 w;     // Q4_K: 8 bytes, elements 8 h + 0..7 and 16 + 8 h + 0..7 of sub-block j; Q6_K: the sub-block's 12 bytes
  uint32_t s;  // Q4_K: aq | bq << 8; Q6_K: sc
};

// four codes in the bytes of v times a factor of at most 7 (no carries between bytes)
__device__ __forceinline__ uint32_t kg_mul4(uint32_t v, u16x2 f) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, v) * f);
}

// Q6_K: sc (q - 32) of the four 6-bit codes in the bytes of d, as digits
// 256 h + l: hi and lo bytes
__device__ __forceinline__ void kg_q6(uint32_t d, i16x2 sc, i16x2 m32sc, uint32_t& hi, uint32_t& lo) {
  const i16x2 e = __builtin_bit_cast(i16x2, d & 0x00FF00FFu), o = __builtin_bit_cast(i16x2, (d >> 8) & 0x00FF00FFu);
  const i16x2 ve = e * sc + m32sc, vo = o * sc + m32sc;
  const i16x2 half = {128, 128};
  const uint32_t ue = __builtin_bit_cast(uint32_t, ve + half), uo = __builtin_bit_cast(uint32_t, vo + half);
  // v_perm byte selects: 0..3 of the second operand, 4..7 of the first
  lo = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, vo), __builtin_bit_cast(uint32_t, ve), 0x06020400u);
  hi = __builtin_amdgcn_perm(uo, ue, 0x07030501u);
}

}  // namespace

// Workgroup: WM x WN x KG waves; tile 16 MF WM rows x 16 NF WN columns, a wave
// 16 MF x 16 NF of it over the super-blocks s with s % KG = its kg (their sums
// are added in kg order at the end). All waves dequantize the next KG
// super-blocks' weights (16 codes per thread and task) into the other half of a
// double-buffered LDS ring while the current ones compute; one barrier per KG
// super-blocks. Activations go straight from xq (row-major, one 16-byte load
// per lane and fragment) into registers.
template <int FMT, bool PK, int MF, int NF, int WM, int WN, int KG>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WM * WN * KG, 64 * WM * WN * KG),
                          amdgpu_waves_per_eu(2))) void kquant_gemm_kernel(
    const uint8_t* __restrict__ wq, const void* __restrict__ sup, const void* __restrict__ subsc,
    const int8_t* __restrict__ xq, const float* __restrict__ xs, const int32_t* __restrict__ bsums,
    void* __restrict__ y, int M, int K, int N, int y_dtype, int tiles_m) {
  constexpr int T = 64 * WM * WN * KG;
  constexpr int BM = 16 * MF * WM, BN = 16 * NF * WN, C = NF * WN;
  constexpr int NT = BN * KG * 16 / T;  // dequantization tasks per thread and step
  static_assert(NT * T == BN * KG * 16 && BN * KG <= T && T % (16 * KG) == 0, "whole tasks");
  constexpr bool Q4 = FMT == RQ_Q4_K;
  // weight digits [buffer][kg][k-step of 64][high, low][16-column fragment][slot]
  struct Lds {
    u32x4 w[2][KG][4][2][C][64];
    float a[2][KG][BN];
    float b[2][Q4 ? KG : 1][Q4 ? BN : 4];
    _Float16 m[2][Q4 ? KG : 1][Q4 ? BN : 1][16];
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
  const int wm = wave % WM, wn = wave / WM % WN, kg = wave / (WM * WN);
  const int l16 = lane & 15, grp = lane >> 4;
  const int nsb = K / 256;
  const int n0 = tn * BN, m0 = tm * BM + wm * 16 * MF;

  // ---- dequantization tasks: thread tid takes tasks tid + T i: piece p =
  // task % 16 of super-block kg = task / 16 % KG of tile row task / 16 / KG
  // (rows past N reread the last one, super-blocks past the end the last one)
  const int p = tid & 15, tkg = (tid >> 4) % KG, trow = (tid >> 4) / KG;
  const int row_bytes = FMT == RQ_Q4_K ? K / 2 : K / 4 * 3;
  const uint32_t codes = (uint32_t)N * (uint32_t)row_bytes, nsub = (uint32_t)K / (FMT == RQ_Q4_K ? 32 : 16);
  constexpr uint32_t SS = FMT == RQ_Q4_K ? 2 : 1, SP = FMT == RQ_Q4_K ? 8 : 4;  // bytes per sub-block / super-block scale
  const __amdgpu_buffer_rsrc_t qr = buffer_rsrc(wq, codes), ur = buffer_rsrc(subsc, (uint32_t)N * nsub * SS),
                               pr = buffer_rsrc(sup, (uint32_t)N * (uint32_t)nsb * SP);
  uint32_t wo[NT], uo[NT];
#pragma unroll
  for (int i = 0; i < NT; i++) {
    const uint32_t o = (uint32_t)min(n0 + trow + T / 16 / KG * i, N - 1);
    wo[i] = o * (uint32_t)row_bytes + (uint32_t)(FMT == RQ_Q4_K ? 8 * p : 12 * p);
    uo[i] = FMT == RQ_Q4_K ? (o * nsub + (uint32_t)p / 2) * 2 : o * nsub + (uint32_t)p;
  }
  const int skg = tid % KG, srow = tid / KG;  // tid < BN KG: row srow's super-block scales
  const uint32_t po = (uint32_t)min(n0 + srow, N - 1) * (uint32_t)nsb * SP;
  KgRaw<FMT> raw[NT];
  u32x2 rs = {0u, 0u};
  auto wload = [&](int step) {
    const uint32_t s = (uint32_t)min(step * KG + tkg, nsb - 1);
#pragma unroll
    for (int i = 0; i < NT; i++) {
      if (Q4) {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(qr, (int)(wo[i] + s * 128), 0, 0));
        raw[i].w = u32x4{v[0], v[1], 0u, 0u};
        raw[i].s = __builtin_amdgcn_raw_buffer_load_b16(ur, (int)(uo[i] + s * 16), 0, 0);
      } else {
        const u32x3 v = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(qr, (int)(wo[i] + s * 192), 0, 0));
        raw[i].w = u32x4{v[0], v[1], v[2], 0u};
        raw[i].s = __builtin_amdgcn_raw_buffer_load_b8(ur, (int)(uo[i] + s * 16), 0, 0);
      }
    }
    if (tid < BN * KG) {
      const uint32_t sp = (uint32_t)min(step * KG + skg, nsb - 1);
      if (Q4)
        rs = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(pr, (int)(po + sp * 8), 0, 0));
      else
        rs[0] = __builtin_amdgcn_raw_buffer_load_b32(pr, (int)(po + sp * 4), 0, 0);
    }
  };
  auto wstore = [&](int b) {
#pragma unroll
    for (int i = 0; i < NT; i++) {
      const int r = trow + T / 16 / KG * i, c = r >> 4, n = r & 15;
      if (FMT == RQ_Q4_K) {
        // sub-block j's 8-byte half h: low nibbles are elements 8 h + 0..7,
        // high nibbles 16 + 8 h + 0..7: k-step j / 2, k groups 2 (j % 2) + 0, 1
        const int j = p >> 1, h = p & 1;
        const uint32_t aq = raw[i].s & 0xFFu;
        const uint16_t ah = (uint16_t)(aq >> 3), al = (uint16_t)(aq & 7u);
        const u16x2 fh = {ah, ah}, fl = {al, al};
        const u32x2 lo = {raw[i].w[0] & 0x0F0F0F0Fu, raw[i].w[1] & 0x0F0F0F0Fu};
        const u32x2 hi = {(raw[i].w[0] >> 4) & 0x0F0F0F0Fu, (raw[i].w[1] >> 4) & 0x0F0F0F0Fu};
        const int slot = (n ^ j) + 32 * (j & 1);
        u32x2* dh = reinterpret_cast<u32x2*>(&L.w[b][tkg][j >> 1][0][c][slot]) + h;
        u32x2* dl = reinterpret_cast<u32x2*>(&L.w[b][tkg][j >> 1][1][c][slot]) + h;
        dh[0] = u32x2{kg_mul4(lo[0], fh), kg_mul4(lo[1], fh)};
        dh[32] = u32x2{kg_mul4(hi[0], fh), kg_mul4(hi[1], fh)};  // 16 slots on: the next k group
        dl[0] = u32x2{kg_mul4(lo[0], fl), kg_mul4(lo[1], fl)};
        dl[32] = u32x2{kg_mul4(hi[0], fl), kg_mul4(hi[1], fl)};
        const int bq = (int)(int8_t)(raw[i].s >> 8);
        L.m[b][tkg][r][8 * h + j] = (_Float16)(h == 0 ? 64 * bq : bq);
      } else {
        const u32x4 q = u32x4{
            (raw[i].w[0] & 0x0F0F0F0Fu) | ((raw[i].w[2] & 0x03030303u) << 4),
            (raw[i].w[1] & 0x0F0F0F0Fu) | (((raw[i].w[2] >> 2) & 0x03030303u) << 4),
            ((raw[i].w[0] >> 4) & 0x0F0F0F0Fu) | (((raw[i].w[2] >> 4) & 0x03030303u) << 4),
            ((raw[i].w[1] >> 4) & 0x0F0F0F0Fu) | (((raw[i].w[2] >> 6) & 0x03030303u) << 4)};
        const int16_t sc = (int16_t)(int8_t)raw[i].s;
        const i16x2 s2 = {sc, sc}, m2 = {(int16_t)(-32 * sc), (int16_t)(-32 * sc)};
        u32x4 h, l;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          uint32_t hv, lv;
          kg_q6(q[e], s2, m2, hv, lv);
          h[e] = hv;
          l[e] = lv;
        }
        const int slot = (n ^ (p & 7)) + 16 * (p & 3);
        L.w[b][tkg][p >> 2][0][c][slot] = h;
        L.w[b][tkg][p >> 2][1][c][slot] = l;
      }
    }
    if (tid < BN * KG) {
      L.a[b][skg][srow] = __uint_as_float(rs[0]);
      if (Q4) L.b[b][skg][srow] = __uint_as_float(rs[1]);
    }
  };

  // ---- this wave's activation rows m0 + 16 f + lane % 16 (rows past M reread the last one)
  const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(xq, (uint32_t)M * (uint32_t)K),
                               dr = buffer_rsrc(xs, (uint32_t)M * (uint32_t)nsb * 4),
                               br = buffer_rsrc(bsums, (uint32_t)M * (uint32_t)nsb * 32);
  // fragment f's rows m0 + 16 f .. and the lane's row of it (rows past M reread the last one); packed
  // tiles (a whole call's rows in order) hold R = 16 rows, the last one what is left
  uint32_t xo[MF], xt[MF], dO[MF], ds[MF], bo[MF];
#pragma unroll
  for (int f = 0; f < MF; f++) {
    if (PK) {
      const uint32_t t16 = (uint32_t)min((m0 >> 4) + f, (M - 1) >> 4), R = min(16u, (uint32_t)M - 16 * t16);
      const uint32_t r = min((uint32_t)l16, R - 1);
      xo[f] = t16 * 16 * (uint32_t)K + ((uint32_t)grp * R + r) * 16;
      xt[f] = R * 64;
      dO[f] = (t16 * 16 * (uint32_t)nsb + r) * 4;
      ds[f] = R * 4;
      bo[f] = t16 * 16 * (uint32_t)nsb * 32 + ((uint32_t)grp * R + r) * 8;
    } else {
      const uint32_t row = (uint32_t)min(m0 + 16 * f + l16, M - 1) * (uint32_t)nsb;
      xo[f] = row * 256 + 16 * (uint32_t)grp;
      xt[f] = 64;
      dO[f] = row * 4;
      ds[f] = 4;
      bo[f] = row * 32 + 16 * ((uint32_t)grp & 1);
    }
  }
  i32x4 a[4][MF];  // a super-block's activation fragments, k-step t
  auto aload = [&](int sb, int t) {
    sb = min(sb, nsb - 1);
#pragma unroll
    for (int f = 0; f < MF; f++)
      a[t][f] = __builtin_bit_cast(
          i32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, (int)xo[f], (int)((uint32_t)(4 * sb + t) * xt[f]), 0));
  };

  f32x4 acc[MF][NF];
#pragma unroll
  for (int f = 0; f < MF; f++)
#pragma unroll
    for (int c = 0; c < NF; c++) acc[f][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const i32x4 zero = {0, 0, 0, 0};

  const int steps = (nsb + KG - 1) / KG;
  wload(0);
#pragma unroll
  for (int t = 0; t < 4; t++) aload(kg, t);
  wstore(0);
  wload(1);
  __syncthreads();
  for (int st = 0; st < steps; st++) {
    const int b = st & 1, s = st * KG + kg, sc = min(s, nsb - 1);
    float dact[MF];
    f16x4 av[MF];  // Q4_K: the rows' bsums as 64 h + l
    i32x4 bs[MF];
#pragma unroll
    for (int f = 0; f < MF; f++) {
      dact[f] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(dr, (int)dO[f], (int)((uint32_t)sc * ds[f]), 0));
      if (Q4 && PK)
        av[f] = __builtin_bit_cast(
            f16x4, __builtin_amdgcn_raw_buffer_load_b64(br, (int)bo[f], (int)((uint32_t)sc * ds[f] * 8), 0));
      else if (Q4)
        bs[f] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(br, (int)bo[f], sc * 32, 0));
    }
    // half of the waves dequantize before their MFMAs and half after, so that
    // the waves of a SIMD use the VALU and the matrix core at different times
    if (wave < WM * WN * KG / 2) {
      wstore(b ^ 1);
      wload(st + 2);
    }
    // the high digits' sum over the super-block, shifted, then the low digits'
    // on top; a fragment's registers take the next super-block's after its last use
    i32x4 d[MF][NF];
#pragma unroll
    for (int hl = 0; hl < 2; hl++) {
#pragma unroll
      for (int t = 0; t < 4; t++) {
#pragma unroll
        for (int c = 0; c < NF; c++) {
          const int sw = Q4 ? 2 * t + (grp >> 1) : 4 * (t & 1) + grp;
          const i32x4 w = __builtin_bit_cast(i32x4, L.w[b][kg][t][hl][wn * NF + c][(l16 ^ sw) + 16 * grp]);
#pragma unroll
          for (int f = 0; f < MF; f++)
            d[f][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                w, a[t][f], t > 0 ? d[f][c] : hl == 0 ? zero : d[f][c] << (Q4 ? 3 : 8), 0, 0, 0);
        }
        if (hl == 1) aload(s + KG, t);
      }
    }
    if (wave >= WM * WN * KG / 2) {
      wstore(b ^ 1);
      wload(st + 2);
    }
    if (Q4 && !PK) {
#pragma unroll
      for (int f = 0; f < MF; f++)
#pragma unroll
        for (int e = 0; e < 4; e++) av[f][e] = (_Float16)(grp < 2 ? bs[f][e] >> 6 : bs[f][e] & 63);
    }
    // ---- the super-block's scaling: lane holds y[row l16 of f][4 grp + e of c]
    if (KG == 1 || s < nsb) {
#pragma unroll
      for (int c = 0; c < NF; c++) {
        const int col = (wn * NF + c) * 16;
        const f32x4 sa = *reinterpret_cast<const f32x4*>(&L.a[b][kg][col + 4 * grp]);
        f32x4 sb = {0.0f, 0.0f, 0.0f, 0.0f};
        f16x4 bm = {0, 0, 0, 0};
        if (Q4) {
          sb = *reinterpret_cast<const f32x4*>(&L.b[b][kg][col + 4 * grp]);
          bm = *reinterpret_cast<const f16x4*>(&L.m[b][kg][col + l16][4 * grp]);
        }
#pragma unroll
        for (int f = 0; f < MF; f++) {
          if (Q4) {
            const f32x4 mn = __builtin_amdgcn_mfma_f32_16x16x16f16(bm, av[f], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; e++)
              acc[f][c][e] = fmaf(dact[f], fmaf(sb[e], mn[e], sa[e] * (float)d[f][c][e]), acc[f][c][e]);
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++) acc[f][c][e] = fmaf(dact[f], sa[e] * (float)d[f][c][e], acc[f][c][e]);
          }
        }
      }
    }
    __syncthreads();
  }

  if (KG > 1) {
    // the kg waves' sums through LDS, added in kg order
    f32x4* red = reinterpret_cast<f32x4*>(smem);
    constexpr int W = WM * WN * MF * NF * 64;
    const int at = (wave % (WM * WN)) * MF * NF * 64 + lane;
    if (kg > 0) {
#pragma unroll
      for (int f = 0; f < MF; f++)
#pragma unroll
        for (int c = 0; c < NF; c++) red[(kg - 1) * W + at + (f * NF + c) * 64] = acc[f][c];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 0; g < KG - 1; g++)
#pragma unroll
      for (int f = 0; f < MF; f++)
#pragma unroll
        for (int c = 0; c < NF; c++) acc[f][c] += red[g * W + at + (f * NF + c) * 64];
  }

  const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
#pragma unroll
  for (int f = 0; f < MF; f++) {
    const int m = m0 + 16 * f + l16;
    if (m >= M) continue;
#pragma unroll
    for (int c = 0; c < NF; c++) {
      const int n = n0 + (wn * NF + c) * 16 + 4 * grp;
      if (vec && n + 3 < N) {
        if (y_dtype == RQ_F32)
          *reinterpret_cast<f32x4*>(static_cast<float*>(y) + (int64_t)m * N + n) = acc[f][c];
        else
          *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(y) + (int64_t)m * N + n) =
              u32x2{pack2_bf16(acc[f][c][0], acc[f][c][1]), pack2_bf16(acc[f][c][2], acc[f][c][3])};
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (n + e >= N) break;
          if (y_dtype == RQ_F32)
            static_cast<float*>(y)[(int64_t)m * N + n + e] = acc[f][c][e];
          else
            static_cast<uint16_t*>(y)[(int64_t)m * N + n + e] = (uint16_t)f32_to_bf16_bits(acc[f][c][e]);
        }
      }
    }
  }
}

template <int FMT, bool PK, int MF, int NF, int WM, int WN, int KG>
static hipError_t launch_kg_t(const Weight& w, const int8_t* xq, const float* xs, const int32_t* bsums, void* y,
                              int y_dtype, int64_t m, hipStream_t stream) {
  constexpr int BN = 16 * NF * WN, BM = 16 * MF * WM, T = 64 * WM * WN * KG;
  const int64_t tiles_m = (m + BM - 1) / BM, tiles_n = (w.out + BN - 1) / BN;
  if (tiles_m * tiles_n > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((kquant_gemm_kernel<FMT, PK, MF, NF, WM, WN, KG>), dim3((unsigned)(tiles_m * tiles_n)), dim3(T), 0,
                     stream, w.q, w.scales, w.sub_scales, xq, xs, bsums, y, (int)m, (int)w.in, (int)w.out, y_dtype,
                     (int)tiles_m);
  return hipGetLastError();
}


namespace {

// The tiles, and per tile what the choice between them needs: rows, columns,
// super-blocks per step (KG), workgroups a CU holds (LDS), and the time of a
// step of a full round in ns (least squares over the calls below, MI355X).
// Measured, us per call with the quantizer, against the GEMV's passes (the
// route before, quantizer not counted), Q4_K / Q6_K:
//   11008 x 4096   m = 5    15.8 /  19.6 (16 x 16)    19.0 /   24.0
//                  m = 32   18.1 /  20.3 (32 x 16)    86.5 /  113.0
//                  m = 64   26.6 /  25.6 (64 x 64)   171.9 /  223.6
//                  m = 128  38.5 /  38.1 (128 x 64)  345.3 /  444.6
//                  m = 512  74.4 /  66.7 (256 x 96)  1396  /  1779
//   28672 x 8192   m = 256  179  /  190  (128 x 64)  2925  /  4248
//   3000 x 4096    m = 128  17.7 /  16.8 (64 x 32)    225  /   266
struct KgTile {
  int bm, bn, kg, per_cu, step_ns;
};
constexpr KgTile kKgTiles[] = {{16, 16, 4, 2, 1500}, {32, 16, 4, 2, 1850}, {64, 32, 4, 1, 3100}, {64, 64, 2, 1, 2650},
                               {128, 32, 2, 1, 2400}, {128, 64, 1, 2, 2750}, {256, 96, 1, 1, 3500}};

// The tile whose rounds of the CUs cost least: rounds x steps x step time (a
// round that leaves every CU one workgroup of two runs its steps in about 3/4
// of the time).
int pick_tile(int64_t m, int64_t n, int64_t nsb, int cu_count) {
  int best = 0;
  int64_t best_cost = INT64_MAX;
  for (int i = 0; i < (int)(sizeof(kKgTiles) / sizeof(kKgTiles[0])); i++) {
    const KgTile& t = kKgTiles[i];
    const int64_t tiles = (m + t.bm - 1) / t.bm * ((n + t.bn - 1) / t.bn), slots = (int64_t)cu_count * t.per_cu;
    const int64_t rounds = (tiles + slots - 1) / slots, steps = (nsb + t.kg - 1) / t.kg;
    const int64_t ns = tiles <= cu_count && t.per_cu > 1 ? t.step_ns * 3 / 4 : t.step_ns;
    const int64_t cost = rounds * steps * ns;
    if (cost < best_cost) best_cost = cost, best = i;
  }
  return best;
}

template <int FMT, bool PK>
hipError_t launch_kg(int tile, const Weight& w, const int8_t* xq, const float* xs, const int32_t* bsums, void* y,
                     int y_dtype, int64_t m, hipStream_t stream) {
  switch (tile) {  // MF, NF, WM, WN, KG
    case 0: return launch_kg_t<FMT, PK, 1, 1, 1, 1, 4>(w, xq, xs, bsums, y, y_dtype, m, stream);
    case 1: return launch_kg_t<FMT, PK, 2, 1, 1, 1, 4>(w, xq, xs, bsums, y, y_dtype, m, stream);
    case 2: return launch_kg_t<FMT, PK, 4, 1, 1, 2, 4>(w, xq, xs, bsums, y, y_dtype, m, stream);
    case 3: return launch_kg_t<FMT, PK, 4, 1, 1, 4, 2>(w, xq, xs, bsums, y, y_dtype, m, stream);
    case 4: return launch_kg_t<FMT, PK, 4, 1, 2, 2, 2>(w, xq, xs, bsums, y, y_dtype, m, stream);
    case 5: return launch_kg_t<FMT, PK, 4, 2, 2, 2, 1>(w, xq, xs, bsums, y, y_dtype, m, stream);
    default: return launch_kg_t<FMT, PK, 4, 3, 4, 2, 1>(w, xq, xs, bsums, y, y_dtype, m, stream);
  }
}

}  // namespace

// From five rows (the GEMV serves four in one pass over the weight: 9-16 us
// against this kernel's 12-15 at 14336 x 4096), codes within the 32-bit buffer
// offsets, and scales that the digits hold (kq_gemm).
bool kquant_gemm_takes(const Weight& w, int64_t m) {
  const int64_t row_bytes = w.format == RQ_Q4_K ? w.in / 2 : w.in / 4 * 3;
  return m > 4 && w.kq_gemm && w.out <= UINT32_MAX / row_bytes;
}

hipError_t launch_kquant_gemm(const Weight& w, const int8_t* xq, const float* xs, const int32_t* bsums, bool packed,
                              void* y, int y_dtype, int64_t m, int cu_count, hipStream_t stream) {
  const int64_t nsb = w.in / 256, sub = w.in / (w.format == RQ_Q4_K ? 32 : 16);
  // rows per launch within the 32-bit buffer offsets (a multiple of every tile's)
  const int64_t most = INT32_MAX / w.in / 256 * 256;
  for (int64_t t0 = 0; t0 < m; t0 += most) {
    const int64_t mt = std::min(most, m - t0);
    const int tile = pick_tile(mt, w.out, nsb, cu_count);
    const int8_t* q = xq + t0 * w.in;
    const float* s = xs + t0 * nsb;
    const int32_t* b = bsums + t0 * sub;
    void* yt = static_cast<uint8_t*>(y) + t0 * w.out * (y_dtype == RQ_F32 ? 4 : 2);
    const hipError_t e = w.format == RQ_Q4_K ? (packed ? launch_kg<RQ_Q4_K, true>(tile, w, q, s, b, yt, y_dtype, mt, stream)
                                                       : launch_kg<RQ_Q4_K, false>(tile, w, q, s, b, yt, y_dtype, mt, stream))
                                             : (packed ? launch_kg<RQ_Q6_K, true>(tile, w, q, s, b, yt, y_dtype, mt, stream)
                                                       : launch_kg<RQ_Q6_K, false>(tile, w, q, s, b, yt, y_dtype, mt, stream));
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace rq
