// kquant.hip — Raster's K-quant formats (Q4_K, Q6_K) on the device: the q8_K
// activation quantizer, the K-quant GEMV, and dequantization.
//
// Formats (raster/compiler/backend/cpu/quant.clj:78-280, Raster's own layout,
// each weight row its own 256-element super-blocks):
//   Q4_K  x = (da*aq)*q + (db*bq): nibbles q (w[k] low, w[k+16] high per
//         32-sub-block), per super-block f32 da / db, per sub-block 6-bit aq
//         (0..63) and bq (-32..31).
//   Q6_K  x = (ds*sc)*(q - 32): one byte q (0..63) per element, per
//         16-sub-block int8 sc, per super-block f32 ds.
// Resident form: the codes as Raster stores them (row-major), the super-block
// scales per (row, super-block) (Q4_K: da and db side by side), the sub-block
// scales per (row, sub-block) (Q4_K: aq and bq side by side).
//
// Activations are q8_K (quantize-act-q8k, quant.clj:158-176, and its GPU form
// quant-act-q8k-gpu!, raster/quant/kernels_k.clj:93-134): per 256-element
// super-block d = max|x| / 127 and int8 codes, plus per-sub-block sums bsums
// (32-element for Q4_K, 16 for Q6_K).
//
// The GEMV is the K dot of qmatmul-q4k-dp4a! / qmatmul-q6k-dp4a!
// (kernels_k.clj:186-297): per super-block
//   Q4_K  d_act * sum_j [(da*aq_j) * dot_j + (db*bq_j) * bsum_j]
//   Q6_K  ds * d_act * sum_j sc_j * (dot_j - 32 * bsum_j)
// with the sub-block dots exact in int32 (v_dot4 over packed bytes: nibbles
// and 6-bit codes are non-negative int8). The terms are added in f32 (Raster
// adds in double). HBM-bound on the codes: a wave takes kKqRows rows at a time,
// its lanes one sub-block each (16 code bytes, one load) strided by 64, the
// activations of up to 4 rows staged in LDS once per workgroup; a short f32 x is
// quantized there by the workgroup itself.
#include <algorithm>
#include <atomic>

#include "rq_internal.h"

namespace rq {

namespace {

constexpr int kKqThreads = 256;
constexpr int kKqWaves = 16;        // most waves of a workgroup
constexpr int kKqFusedMax = 12288;  // most elements of x quantized inside the GEMV (kquant_gemv_quantizes)
// weight rows a wave takes at a time (14336 x 4096, m = 1, cold, rows 1 / 2 /
// 4 / 8: Q4_K 12.1 / 10.3 / 11.3 / 12.7 us, Q6_K 15.7 / 12.5 / 13.8 / 14.4 us;
// m = 4 likewise best at 2)
constexpr int kKqRows = 2;

__device__ __forceinline__ float wave_sum64(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// The largest of the wave's values, in every lane: quads and half rows by DPP,
// then the rows by lane swaps.
__device__ __forceinline__ float wave_max64(float v) {
  v = max8(v);
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false)));  // row_ror:8
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
}

// quantize-act-q8k of one super-block by one wave, four elements per lane: the
// lane's codes as a word, d in every lane, and in the first lane of each SUB / 4
// the sum of the sub-block's codes.
template <int SUB>
__device__ __forceinline__ uint32_t quantize_q8k(const f32x4& v, double& d, int& sum) {
  const float a = wave_max64(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
  d = (double)a / 127.0;
  const double id = d == 0.0 ? 0.0 : 1.0 / d;
  uint32_t word = 0u;
  int s = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int q = java_round_clamp127((double)v[i] * id);
    word |= (uint32_t)(q & 0xFF) << (8 * i);
    s += q;
  }
  s += dpp_xor1(s);
  s += dpp_xor2(s);
  sum = SUB == 32 ? s + dpp_half_mirror(s) : s;
  return word;
}

}  // namespace

// ---- q8_K activation quantizer: one wave per 256-element super-block, four
// elements per lane; SUB-element sub-block sums over SUB/4 lanes.
template <int SUB>
__global__ __launch_bounds__(kKqThreads) void quantize_act_q8k_kernel(const float* __restrict__ x,
                                                                     int8_t* __restrict__ xq, float* __restrict__ xs,
                                                                     int32_t* __restrict__ bsums, int64_t nsb) {
  const int lane = threadIdx.x & 63;
  const int64_t sb = (int64_t)blockIdx.x * (kKqThreads / 64) + (threadIdx.x >> 6);
  const int64_t b = sb < nsb ? sb : nsb - 1;  // waves past the end reread the last one and store nothing
  const f32x4 v = *reinterpret_cast<const f32x4*>(x + b * 256 + lane * 4);
  double d;
  int s;
  const uint32_t word = quantize_q8k<SUB>(v, d, s);
  if (sb < nsb) {
    *reinterpret_cast<uint32_t*>(xq + b * 256 + lane * 4) = word;
    if (lane == 0) xs[b] = (float)d;
    if (lane % (SUB / 4) == 0) bsums[b * (256 / SUB) + lane / (SUB / 4)] = s;
  }
}

// The same codes in the operand order of the K-quant GEMM (kquant_gemm.hip):
// per 16-row tile (the last one R = m % 16 rows if that is not 0) and 64-element
// step one fragment, 16 bytes per (k group of 16, row); xs as [tile][super-block]
// [row]; for SUB 32 the block sums as the f16 digits 64 h + l of the minimum
// term's operand, 8 bytes per (slot group, row): slots 0..7 h, 8..15 l of the 8
// sub-blocks (SUB 16: not stored, the GEMM does not use them). The buffers have
// the sizes of the row-major form. A wave takes one super-block of 4 rows, 16
// elements per lane, so every store instruction writes runs of 64 bytes.
template <int SUB>
__global__ __launch_bounds__(kKqThreads) void quantize_act_q8k_packed_kernel(const float* __restrict__ x,
                                                                            int8_t* __restrict__ xq,
                                                                            float* __restrict__ xs,
                                                                            int32_t* __restrict__ bsums, int64_t M,
                                                                            int nsb) {
  const int lane = threadIdx.x & 63, ch = lane & 15;
  const int64_t wv = (int64_t)blockIdx.x * (kKqThreads / 64) + (threadIdx.x >> 6);
  const int64_t row = wv / nsb * 4 + (lane >> 4), sb = wv % nsb;
  const bool live = row < M;
  const float* src = x + ((live ? row : M - 1) * nsb + sb) * 256 + ch * 16;
  f32x4 v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = reinterpret_cast<const f32x4*>(src)[i];
  float a = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; i++)
    a = fmaxf(a, fmaxf(fmaxf(fabsf(v[i][0]), fabsf(v[i][1])), fmaxf(fabsf(v[i][2]), fabsf(v[i][3]))));
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) a = fmaxf(a, __shfl_xor(a, off, 64));
  const double d = (double)a / 127.0;
  const double id = d == 0.0 ? 0.0 : 1.0 / d;
  u32x4 w = {0u, 0u, 0u, 0u};
  int s = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int q = java_round_clamp127((double)v[i / 4][i % 4] * id);
    w[i / 4] |= (uint32_t)(q & 0xFF) << (8 * (i % 4));
    s += q;
  }
  if (SUB == 32) s += __shfl_xor(s, 1, 64);
  if (!live) return;
  const int64_t t16 = row >> 4, R = M - 16 * t16 < 16 ? M - 16 * t16 : 16, r = row & 15;
  *reinterpret_cast<u32x4*>(xq + t16 * 16 * nsb * 256 + (4 * sb + (ch >> 2)) * 64 * R + ((ch & 3) * R + r) * 16) = w;
  if (ch == 0) xs[t16 * 16 * nsb + sb * R + r] = (float)d;
  if (SUB == 32) {
    const int slot = (ch & 1) * 8 + (ch >> 1);  // even lanes h, odd lanes l
    reinterpret_cast<_Float16*>(bsums)[(t16 * 16 * nsb + sb * R) * 16 + ((slot >> 2) * R + r) * 4 + (slot & 3)] =
        (_Float16)((ch & 1) ? s & 63 : s >> 6);
  }
}

hipError_t launch_quantize_act_q8k_packed(const float* x, int64_t m, int64_t in, int sub, int8_t* xq, float* xs,
                                          int32_t* bsums, hipStream_t stream) {
  const int64_t waves = (m + 3) / 4 * (in / 256);
  if (waves == 0) return hipSuccess;
  const dim3 grid((unsigned)((waves + kKqThreads / 64 - 1) / (kKqThreads / 64)));
  if (sub == 32)
    hipLaunchKernelGGL((quantize_act_q8k_packed_kernel<32>), grid, dim3(kKqThreads), 0, stream, x, xq, xs, bsums, m,
                       (int)(in / 256));
  else
    hipLaunchKernelGGL((quantize_act_q8k_packed_kernel<16>), grid, dim3(kKqThreads), 0, stream, x, xq, xs, bsums, m,
                       (int)(in / 256));
  return hipGetLastError();
}

hipError_t launch_quantize_act_q8k(const float* x, int64_t m, int64_t in, int sub, int8_t* xq, float* xs,
                                   int32_t* bsums, hipStream_t stream) {
  const int64_t nsb = m * (in / 256);
  if (nsb == 0) return hipSuccess;
  const dim3 grid((unsigned)((nsb + kKqThreads / 64 - 1) / (kKqThreads / 64)));
  if (sub == 32)
    hipLaunchKernelGGL((quantize_act_q8k_kernel<32>), grid, dim3(kKqThreads), 0, stream, x, xq, xs, bsums, nsb);
  else
    hipLaunchKernelGGL((quantize_act_q8k_kernel<16>), grid, dim3(kKqThreads), 0, stream, x, xq, xs, bsums, nsb);
  return hipGetLastError();
}

// Q6_K codes on the device: each 16-code sub-block packed into 12 bytes.
// Bytes 0..7: byte j holds code j (low nibble) and code j + 8 (high nibble),
// their low 4 bits; bytes 8..11: byte j holds bits 4..5 of codes j, j + 4,
// j + 8, j + 12 in its bit pairs 0, 1, 2, 3. p0, p1, p2 are bytes 0..3, 4..7,
// 8..11 as little-endian words; the result holds codes 4 k .. 4 k + 3 as
// bytes in word k.
__device__ __forceinline__ u32x4 unpack_q6k(uint32_t p0, uint32_t p1, uint32_t p2) {
  return u32x4{(p0 & 0x0F0F0F0Fu) | ((p2 & 0x03030303u) << 4), (p1 & 0x0F0F0F0Fu) | (((p2 >> 2) & 0x03030303u) << 4),
               ((p0 >> 4) & 0x0F0F0F0Fu) | (((p2 >> 4) & 0x03030303u) << 4),
               ((p1 >> 4) & 0x0F0F0F0Fu) | (((p2 >> 6) & 0x03030303u) << 4)};
}

// ---- K-quant GEMV: y[t][o] for MT activation rows t. FMT RQ_Q4_K / RQ_Q6_K.
// LDS: xq[MT][K] codes, bsums[MT][K/SUB], xs[MT][K/256].
// XF: x is given as f32 and quantized while it is staged (xq and bsums unused,
// xs = x).
template <int FMT, int MT, bool XF, int D>
__global__ __launch_bounds__(64 * kKqWaves) void kquant_gemv_kernel(
    const uint8_t* __restrict__ wq, const void* __restrict__ sup, const void* __restrict__ subsc,
    const int8_t* __restrict__ xq, const float* __restrict__ xs, const int32_t* __restrict__ bsums,
    void* __restrict__ y, int M, int K, int N, int y_dtype) {
  constexpr int SUB = FMT == RQ_Q4_K ? 32 : 16;  // elements per sub-block (16 code bytes either way)
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int nsub = K / SUB, nsb = K / 256;
  int8_t* lx = reinterpret_cast<int8_t*>(smem);
  int32_t* lb = reinterpret_cast<int32_t*>(smem + MT * K);
  float* ls = reinterpret_cast<float*>(smem + MT * K + MT * nsub * 4);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // ---- this wave's work: row groups gi = 0 .. ng-1 (kKqRows rows from o0 =
  // kKqRows (gw + gi nwaves)), each swept in nit steps (lane: sub-block lane + 64 si). The
  // steps stream through a D-step register ring of raw code and scale bits
  // across row groups (steps padded to whole ring turns); nothing converts or
  // tests loaded bits before the step computes, and refills are unconditional
  // at clamped addresses, so the compiler keeps D steps of loads in flight.
  // D = 1 measured best (14336 x 4096, m = 1: Q4_K 11.7 / 12.2 / 13.5 /
  // 15.5 us and Q6_K 16.9 / 17.4 / 18.9 / 19.0 us at D = 1 .. 4; before this
  // stream, loading each step only when it was computed: 15.0 and 16.3 us).
  const int nthr = (int)blockDim.x;
  const int gw = XF ? wave * (int)gridDim.x + (int)blockIdx.x : (int)blockIdx.x * (nthr / 64) + wave;
  const int nwaves = (int)gridDim.x * (nthr / 64);
  const int ngrp = (N + kKqRows - 1) / kKqRows;
  const int ng = gw < ngrp ? (ngrp - 1 - gw) / nwaves + 1 : 0;
  const int nit = (nsub + 63) / 64, nitp = (nit + D - 1) / D * D;
  // code bytes per row: K / 2 (Q4_K nibbles), 3 K / 4 (Q6_K, 12 bytes per 16-code sub-block)
  const int64_t row_bytes = FMT == RQ_Q4_K ? K / 2 : K / 4 * 3;
  struct Slot {
    u32x4 w[kKqRows];
    uint32_t a[kKqRows], b[kKqRows], c[kKqRows];  // Q4_K: da, db bits, aq | bq << 8; Q6_K: ds bits, sc
  };
  Slot ring[D];
  auto load = [&](int slot, int gi, int si) {
    if (gi >= ng) {  // past the end: the last step again
      gi = ng - 1;
      si = nitp - 1;
    }
    const int o0 = (gw + gi * nwaves) * kKqRows;
    const int sb = min(lane + 64 * min(si, nit - 1), nsub - 1);
#pragma unroll
    for (int r = 0; r < kKqRows; r++) {
      const int o = min(o0 + r, N - 1);
      if (FMT == RQ_Q4_K) {
        ring[slot].w[r] = *reinterpret_cast<const u32x4*>(wq + (int64_t)o * row_bytes + sb * 16);
      } else {  // 12 bytes, unpacked when the step computes
        const uint32_t* p = reinterpret_cast<const uint32_t*>(wq + (int64_t)o * row_bytes + sb * 12);
        ring[slot].w[r] = u32x4{p[0], p[1], p[2], 0u};
      }
      if (FMT == RQ_Q4_K) {
        const u32x2 d2 = static_cast<const u32x2*>(sup)[(int64_t)o * nsb + sb / 8];
        ring[slot].a[r] = d2[0];
        ring[slot].b[r] = d2[1];
        ring[slot].c[r] = static_cast<const uint16_t*>(subsc)[(int64_t)o * nsub + sb];
      } else {
        ring[slot].a[r] = static_cast<const uint32_t*>(sup)[(int64_t)o * nsb + sb / 16];
        ring[slot].c[r] = (uint32_t)(uint8_t)static_cast<const int8_t*>(subsc)[(int64_t)o * nsub + sb];
      }
    }
  };
  int lg = 0, ls_ = 0;
  auto advance = [&](int& gi, int& si) {
    if (++si == nitp) {
      si = 0;
      ++gi;
    }
  };
  // XF: the wave's super-blocks of x, wave, wave + waves, ... of the M rows; the
  // first XJ go out before the weights, so that quantizing them waits for them
  // only (loads complete in order)
  constexpr int XJ = XF ? 2 : 1;
  f32x4 xv[XJ];
  const int nxb = M * nsb, xw = nthr / 64;
  auto load_x = [&](int b0) {
#pragma unroll
    for (int j = 0; j < XJ; j++) {
      const int b = min(b0 + j * xw, nxb - 1);
      xv[j] = *reinterpret_cast<const f32x4*>(xs + (int64_t)b * 256 + lane * 4);
    }
  };
  if (XF) {
    load_x(wave);
    __builtin_amdgcn_sched_barrier(0);
  }
  // the first weight loads go out before the activations are staged, so
  // their latency overlaps the staging (14336 x 4096, m = 1, cold: Q4_K
  // 11.65 -> 11.19 us; Q6_K unchanged at 16.9)
  if (ng > 0) {
#pragma unroll
    for (int i = 0; i < D; i++) {
      load(i, lg, ls_);
      advance(lg, ls_);
    }
  }

  // stage the activations (rows past M as zeros)
  if constexpr (XF) {
    __builtin_amdgcn_sched_barrier(0);
    for (int b0 = wave; b0 < nxb; b0 += XJ * xw) {
      if (b0 != wave) load_x(b0);
#pragma unroll
      for (int j = 0; j < XJ; j++) {
        const int b = b0 + j * xw;
        if (b >= nxb) break;  // wave-uniform
        double d;
        int sum;
        const uint32_t word = quantize_q8k<SUB>(xv[j], d, sum);
        reinterpret_cast<uint32_t*>(lx)[b * 64 + lane] = word;
        if (lane == 0) ls[b] = (float)d;
        if (lane % (SUB / 4) == 0) lb[b * (256 / SUB) + lane / (SUB / 4)] = sum;
      }
    }
    for (int b = nxb + wave; b < MT * nsb; b += xw) {
      reinterpret_cast<uint32_t*>(lx)[b * 64 + lane] = 0u;
      if (lane == 0) ls[b] = 0.0f;
      if (lane % (SUB / 4) == 0) lb[b * (256 / SUB) + lane / (SUB / 4)] = 0;
    }
  } else {
    for (int i = tid; i < MT * K / 16; i += nthr) {
      const int t = i / (K / 16);
      u32x4 v = u32x4{0u, 0u, 0u, 0u};
      if (t < M) v = reinterpret_cast<const u32x4*>(xq + (int64_t)t * K)[i % (K / 16)];
      reinterpret_cast<u32x4*>(lx)[i] = v;
    }
    for (int i = tid; i < MT * nsub; i += nthr) lb[i] = i / nsub < M ? bsums[(int64_t)i] : 0;
    for (int i = tid; i < MT * nsb; i += nthr) ls[i] = i / nsb < M ? xs[(int64_t)i] : 0.0f;
  }
  __syncthreads();
  if (ng == 0) return;  // wave-uniform; no barrier follows

  float acc[kKqRows][MT];
#pragma unroll
  for (int r = 0; r < kKqRows; r++)
#pragma unroll
    for (int t = 0; t < MT; t++) acc[r][t] = 0.0f;
  for (int gi = 0; gi < ng; gi++) {
    for (int si0 = 0; si0 < nitp; si0 += D) {
#pragma unroll
      for (int i = 0; i < D; i++) {
        const int si = si0 + i;
        const Slot cur = ring[i];
        load(i, lg, ls_);
        advance(lg, ls_);
        const int sraw = lane + 64 * si;
        if (si < nit) {  // wave-uniform: padding steps compute nothing
          const bool live = sraw < nsub;
          const int s = min(sraw, nsub - 1);
          float f0[kKqRows], f1[kKqRows];
#pragma unroll
          for (int r = 0; r < kKqRows; r++) {
            if (FMT == RQ_Q4_K) {
              f0[r] = __uint_as_float(cur.a[r]) * (float)(int)(cur.c[r] & 0xFFu);        // da * aq
              f1[r] = __uint_as_float(cur.b[r]) * (float)(int)(int8_t)(cur.c[r] >> 8);   // db * bq
            } else {
              f0[r] = __uint_as_float(cur.a[r]) * (float)(int)(int8_t)cur.c[r];          // ds * sc
              f1[r] = 0.0f;
            }
          }
          // Q6_K: the rows' 16 codes as bytes, unpacked once for all MT rows
          u32x4 cw[kKqRows];
#pragma unroll
          for (int r = 0; r < kKqRows; r++)
            cw[r] = FMT == RQ_Q6_K ? unpack_q6k(cur.w[r][0], cur.w[r][1], cur.w[r][2]) : cur.w[r];
#pragma unroll
          for (int t = 0; t < MT; t++) {
            const u32x4 xa = reinterpret_cast<const u32x4*>(lx + t * K)[s * SUB / 16];
            const int bs = lb[t * nsub + s];
            const float dact = ls[t * nsb + s * SUB / 256];
            if (FMT == RQ_Q4_K) {
              const u32x4 xb = reinterpret_cast<const u32x4*>(lx + t * K)[s * 2 + 1];
#pragma unroll
              for (int r = 0; r < kKqRows; r++) {
                int dp = 0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                  dp = __builtin_amdgcn_sdot4((int)(cur.w[r][k] & 0x0F0F0F0Fu), (int)xa[k], dp, false);
                  dp = __builtin_amdgcn_sdot4((int)((cur.w[r][k] >> 4) & 0x0F0F0F0Fu), (int)xb[k], dp, false);
                }
                const float v = fmaf(dact, f0[r] * (float)dp + f1[r] * (float)bs, acc[r][t]);
                acc[r][t] = live ? v : acc[r][t];
              }
            } else {
#pragma unroll
              for (int r = 0; r < kKqRows; r++) {
                int dp = 0;
#pragma unroll
                for (int k = 0; k < 4; k++) dp = __builtin_amdgcn_sdot4((int)cw[r][k], (int)xa[k], dp, false);
                const float v = fmaf(dact * f0[r], (float)(dp - 32 * bs), acc[r][t]);
                acc[r][t] = live ? v : acc[r][t];
              }
            }
          }
        }
      }
    }
    // ---- row group gi: sum the lanes, store
    const int o0 = (gw + gi * nwaves) * kKqRows;
#pragma unroll
    for (int r = 0; r < kKqRows; r++)
#pragma unroll
      for (int t = 0; t < MT; t++) {
        const float v = wave_sum64(acc[r][t]);
        acc[r][t] = 0.0f;
        const int o = o0 + r;
        if (lane == 0 && o < N && t < M) {
          if (y_dtype == RQ_F32)
            static_cast<float*>(y)[(int64_t)t * N + o] = v;
          else
            static_cast<uint16_t*>(y)[(int64_t)t * N + o] = (uint16_t)f32_to_bf16_bits(v);
        }
      }
  }
}
size_t kquant_gemv_lds(int format, int64_t k, int mt) {
  const int64_t sub = format == RQ_Q4_K ? 32 : 16;
  return (size_t)mt * (size_t)(k + 4 * (k / sub) + 4 * (k / 256));
}

template <int FMT, int MT, bool XF, int D = 1>
static hipError_t launch_kq_t(const Weight& w, const int8_t* xq, const float* xs, const int32_t* bsums, void* y,
                              int y_dtype, int64_t m, int cu_count, hipStream_t stream) {
  auto kernel = &kquant_gemv_kernel<FMT, MT, XF, D>;
  const size_t lds = kquant_gemv_lds(FMT, w.in, MT);
  if (lds > 65536) {
    static std::atomic<uint64_t> attr_set{0};
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return e;
    const uint64_t bit = uint64_t(1) << (dev & 63);
    if (!(attr_set.load(std::memory_order_acquire) & bit)) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 163840);
      if (e != hipSuccess) return e;
      attr_set.fetch_or(bit, std::memory_order_acq_rel);
    }
  }
  // m = 1 with quantized activations of a short row: a wave per row group in
  // workgroups of four, all launched at once (14336 x 4096, cold, Q4_K 12.3 and
  // Q6_K 15.0 us with the quantizer, against 12.8 / 15.3 with one workgroup per
  // CU). Otherwise at most one workgroup per CU, so that x is staged once per
  // CU, with as many waves as spread the row groups evenly over whole turns:
  // 28672 x 8192 m = 1 / 4 Q4_K 31.9 / 54.0 -> 30.5 / 40.7 us, Q6_K 43.2 / 79.7
  // -> 39.7 / 54.2; 4096 x 14336 m = 4 Q4_K 21.9 -> 19.0. XF: the waves that
  // quantizing x keeps busy, also where fewer have rows (1024 x 4096 m = 1 5.8
  // us with the waves that have rows, 4.7 with all).
  const int64_t groups = std::max<int64_t>((w.out + kKqRows - 1) / kKqRows, 1);
  int64_t waves = kKqThreads / 64, wg = (groups + waves - 1) / waves;
  if (XF || MT > 1 || w.in >= 8192) {
    const int64_t turns = (groups + cu_count * kKqWaves - 1) / (cu_count * kKqWaves);
    waves = std::max<int64_t>(waves, (groups + cu_count * turns - 1) / (cu_count * turns));
    if (XF) {
      waves = std::max<int64_t>(waves, std::min<int64_t>(kKqWaves, m * (w.in / 256)));
      wg = std::min<int64_t>(cu_count, groups);
    } else {
      wg = std::min<int64_t>(cu_count, (groups + waves - 1) / waves);
    }
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)wg), dim3((unsigned)(64 * waves)), (unsigned)lds, stream, w.q,
                     w.scales, w.sub_scales, xq, xs, bsums, y, (int)m, (int)w.in, (int)w.out, y_dtype);
  return hipGetLastError();
}

// XF: xs is the f32 x
template <bool XF>
static hipError_t launch_kquant_rows(const Weight& w, const int8_t* xq, const float* xs, const int32_t* bsums, void* y,
                                     int y_dtype, int64_t m, int cu_count, hipStream_t stream) {
  const int64_t nsub = w.in / (w.format == RQ_Q4_K ? 32 : 16), nsb = w.in / 256;
  const size_t ysz = y_dtype == RQ_F32 ? 4 : 2;
  // four activation rows per launch; two rows have an instance of their own
  // (14336 x 4096, Q4_K, with the quantizer: 17.6 us in the one for four, 14.5)
  for (int64_t t0 = 0; t0 < m; t0 += 4) {
    const int64_t mt = std::min<int64_t>(4, m - t0);
    const int8_t* xq_t = XF ? nullptr : xq + t0 * w.in;
    const float* xs_t = xs + t0 * (XF ? w.in : nsb);
    const int32_t* bs_t = XF ? nullptr : bsums + t0 * nsub;
    void* y_t = static_cast<uint8_t*>(y) + (size_t)(t0 * w.out) * ysz;
    hipError_t e;
    if (w.format == RQ_Q4_K)
      e = mt == 1   ? launch_kq_t<RQ_Q4_K, 1, XF>(w, xq_t, xs_t, bs_t, y_t, y_dtype, mt, cu_count, stream)
          : mt == 2 ? launch_kq_t<RQ_Q4_K, 2, XF>(w, xq_t, xs_t, bs_t, y_t, y_dtype, mt, cu_count, stream)
                    : launch_kq_t<RQ_Q4_K, 4, XF>(w, xq_t, xs_t, bs_t, y_t, y_dtype, mt, cu_count, stream);
    else
      e = mt == 1   ? launch_kq_t<RQ_Q6_K, 1, XF>(w, xq_t, xs_t, bs_t, y_t, y_dtype, mt, cu_count, stream)
          : mt == 2 ? launch_kq_t<RQ_Q6_K, 2, XF>(w, xq_t, xs_t, bs_t, y_t, y_dtype, mt, cu_count, stream)
                    : launch_kq_t<RQ_Q6_K, 4, XF>(w, xq_t, xs_t, bs_t, y_t, y_dtype, mt, cu_count, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_kquant_gemv(const Weight& w, const int8_t* xq, const float* xs, const int32_t* bsums, void* y,
                              int y_dtype, int64_t m, int cu_count, hipStream_t stream) {
  return launch_kquant_rows<false>(w, xq, xs, bsums, y, y_dtype, m, cu_count, stream);
}

// Every CU quantizes all of x, 0.08 us per 256 elements, against 1.5-2.5 us for
// the quantizer's own launch. Cold, in a graph, own launch / fused: Q4_K
// 14336 x 4096 m = 1 / 2 / 3 / 4 12.2 / 10.6, 14.7 / 13.2, 16.8 / 16.3,
// 17.2 / 17.1 us; 4096 x 4096 m = 1 / 3 / 4 7.7 / 5.9, 10.0 / 10.0, 10.2 / 11.0;
// 28672 x 8192 m = 1 / 2 31.2 / 28.6, 34.2 / 33.9; 2048 x 5632 m = 2 / 3 9.4 /
// 8.4, 11.5 / 11.3; 4096 x 14336 m = 1 13.1 / 13.4; 32000 x 2048 m = 4 20.6 /
// 19.4; Q6_K 14336 x 4096 m = 1 / 3 14.5 / 13.3, 19.5 / 18.9. The line is
// between 3 x 4096 and 1 x 14336. Workgroups read x while others store y, so a
// call whose y overlaps x keeps the quantizer's launch.
bool kquant_gemv_quantizes(const Weight& w, const float* x, const void* y, int y_dtype, int64_t m) {
  if (m > 4 || m * w.in > kKqFusedMax) return false;
  const uintptr_t x0 = (uintptr_t)x, x1 = x0 + (size_t)m * (size_t)w.in * 4;
  const uintptr_t y0 = (uintptr_t)y, y1 = y0 + (size_t)m * (size_t)w.out * (y_dtype == RQ_F32 ? 4 : 2);
  return y1 <= x0 || x1 <= y0;
}

hipError_t launch_kquant_gemv_f32(const Weight& w, const float* x, void* y, int y_dtype, int64_t m, int cu_count,
                                  hipStream_t stream) {
  return launch_kquant_rows<true>(w, nullptr, x, nullptr, y, y_dtype, m, cu_count, stream);
}

// ---- dequantization, bitwise as dequant-q4k / dequant-q6k (the products are
// exact in double, one rounding of the sum, one narrowing)
template <int FMT>
__global__ __launch_bounds__(256) void kquant_dequant_kernel(const uint8_t* __restrict__ wq,
                                                            const void* __restrict__ sup,
                                                            const void* __restrict__ subsc, float* __restrict__ out,
                                                            int64_t K, int64_t n) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  const int64_t o = e / K, k = e % K, nsb = K / 256;
  if (FMT == RQ_Q4_K) {
    const int64_t s = k / 32, j = k % 32;
    const uint32_t b = wq[o * (K / 2) + s * 16 + (j % 16)];
    const uint32_t q = j < 16 ? (b & 0xFu) : (b >> 4);
    const f32x2 d2 = static_cast<const f32x2*>(sup)[o * nsb + s / 8];
    const uint32_t ab = static_cast<const uint16_t*>(subsc)[o * (K / 32) + s];
    const double a1 = (double)d2[0] * (double)(int)(ab & 0xFFu);
    const double b1 = (double)d2[1] * (double)(int)(int8_t)(ab >> 8);
    out[e] = (float)(a1 * (double)q + b1);
  } else {
    const double a1 = (double)static_cast<const float*>(sup)[o * nsb + k / 256] *
                      (double)static_cast<const int8_t*>(subsc)[o * (K / 16) + k / 16];
    const int64_t s = k / 16, j = k % 16;
    const uint8_t* sbp = wq + o * (K / 4 * 3) + s * 12;
    const uint32_t lo = (sbp[j % 8] >> (j < 8 ? 0 : 4)) & 0xFu, hi = (sbp[8 + j % 4] >> (2 * (j / 4))) & 3u;
    out[e] = (float)(a1 * (double)((int)(lo | (hi << 4)) - 32));
  }
}

hipError_t launch_kquant_dequant(const Weight& w, float* out, hipStream_t stream) {
  const int64_t n = w.out * w.in;
  if ((n + 255) / 256 > INT32_MAX) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (w.format == RQ_Q4_K)
    hipLaunchKernelGGL((kquant_dequant_kernel<RQ_Q4_K>), grid, dim3(256), 0, stream, w.q, w.scales, w.sub_scales,
                       out, w.in, n);
  else
    hipLaunchKernelGGL((kquant_dequant_kernel<RQ_Q6_K>), grid, dim3(256), 0, stream, w.q, w.scales, w.sub_scales,
                       out, w.in, n);
  return hipGetLastError();
}

}  // namespace rq
