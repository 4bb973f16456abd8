// Quantize-on-append: encode 128-token codec pages of pre-RoPE keys and values
// straight into 16-token physical pages, gfx950 -- the recipe's page and the
// general page (include/bmx_k2b.h).
//
//   append_us_kernel     Us = M * basis32 (or the first page's SVD factor), fp16
//   append_codes_kernel  (recipe's page) two kinds of workgroup in one launch:
//                        R = M - Us16 * basis16^T with its per-channel RTN, and
//                        per (token, head) the value's fp16 norm and Lloyd codes
//   gen_kres_kernel, value_codes_kernel  the same two as launches of their own
//                        (general page; the values of spectral pages)
// Reference semantics: cache/packed_streaming.py:475-580 (page commit),
// cache/codecs.py:616-636, 677-695, 786-796 (codecs), quant/rtn.py:23-44 (RTN),
// quant/hadamard.py:12-33 (FWHT).  Element-wise steps follow the reference's
// operation order (divide, round-half-even, divide-then-multiply by sqrt(d)) and
// this file is built without floating-point contraction, so codes are identical
// to the reference's whenever the reduction results (Us, the norm) agree.

#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>

#include "k2b_common.h"
#include "k2b_general.h"

namespace bmx {

__device__ __forceinline__ uint8_t* append_page(const AppendKArgs& a, int slot) {
  return a.pages + clamp_page(a.page_ids[slot], a.n_pool) * (int64_t)a.L.bytes;
}

// 4x4 transpose between four registers and the four 16-lane rows of a wave:
// register e of row q in, register q of row e out.
__device__ __forceinline__ void transpose_rows(float (&x)[8], int at) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  uint32_t w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = __float_as_uint(x[at + e]);
  const u32x2 a = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false);   // odd rows of the first, even of the second
  const u32x2 b = __builtin_amdgcn_permlane16_swap(w[2], w[3], false, false);
  const u32x2 c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);   // upper half of the first, lower of the second
  const u32x2 d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
  x[at] = __uint_as_float(c[0]);
  x[at + 1] = __uint_as_float(d[0]);
  x[at + 2] = __uint_as_float(c[1]);
  x[at + 3] = __uint_as_float(d[1]);
}

// grid (16-token pages of the call, R / 16), block 256 = 4 waves.
// Us[t][r] = sum_c M[t][c] basis32[c][r] in fp32 (the reference's M @ V): wave w
// sums channels [w C/4, (w+1) C/4) in order, and the four partial sums are added
// in wave order.  The first codec page of a sequence takes its SVD factor instead.
// The wave's 16 tokens x 16 ranks go on v_mfma_f32_16x16x4_f32, which adds its 4
// products one after another, each as an fma: 64 instructions make the chain of
// 256 steps that a lane's own FMAs made (C 1024), with the same bits.  Its A
// operand is token lane & 15, channel 4 m + (lane >> 4) of step m: a lane loads 8
// channels of its token (16 bytes) at 8 (lane >> 4) of a 32-channel chunk, and two
// 4x4 transposes across the wave's rows put them in order.  Its B operand is one
// dword a lane, whole lines of basis32, straight from memory.
// Bound: the chain (a commit of one codec page has only 8 R / 16 workgroups) and
// the round trip before it: the loads of 8 chunks, a quarter of C 1024, are in
// flight at once, and there is no barrier before the sum over the waves.
// Measured at h_kv 8: 5.7 us for one codec page at R 32, 8.4 us for 63 at
// R 16; with FMAs on the VALU and the basis columns staged in LDS 10.8 and 16.3 us.
// kVec: rows 16-byte aligned; else the 8 channels are read one by one.
constexpr int kUsSets = 8;   // chunks of 32 channels in flight

template <bool kVec>
__global__ __launch_bounds__(256, 2) void append_us_kernel(const AppendKArgs a) {
  __shared__ float s_part[4][kPT][17];
  const int pg = blockIdx.x, rg = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int C = a.C, R = a.R, ld = a.log2d, d = 1 << ld;
  uint8_t* page = append_page(a, pg);
  uint16_t* us = reinterpret_cast<uint16_t*>(page + a.L.us);
  const int ot = tid >> 4, orank = 16 * rg + (tid & 15);     // the output of this thread
  const int oi = a.general ? ot * R + orank : us_half(R, ot, orank);
  if (a.us_first != nullptr && pg < 8) {
    us[oi] = float_to_half_bits(a.us_first[(pg * kPT + ot) * R + orank]);
    return;
  }
  const int n = lane & 15, q = lane >> 4;
  const int Q = C / 4, c0 = wave * Q;             // the wave's channels: a multiple of 8
  const int n32 = (Q + 31) / 32;                  // chunks, the last of 8, 16, 24 or 32 channels
  const uint16_t* row = a.k_pre + (int64_t)(pg * kPT + n) * a.kst;
  const float* bp = a.basis32 + (int64_t)(c0 + q) * R + 16 * rg + n;
  uint4 kx[kUsSets];
  float bx[kUsSets][8];
  auto load = [&](int s, int k) {   // chunk k; past the wave's channels: its last ones again, not used
    const int c = c0 + min(32 * k + 8 * q, Q - 8);
    const uint16_t* p = row + (int64_t)(c >> ld) * a.ksh + (c & (d - 1));
    if constexpr (kVec) {
      kx[s] = *reinterpret_cast<const uint4*>(p);
    } else {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = p[2 * i] | (uint32_t)p[2 * i + 1] << 16;
      kx[s] = make_uint4(w[0], w[1], w[2], w[3]);
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) bx[s][m] = bp[(int64_t)min(32 * k + 4 * m, Q - 4) * R];
  };
#pragma unroll
  for (int s = 0; s < kUsSets; ++s)
    if (s < n32) load(s, s);
  float4_t acc = {0.f, 0.f, 0.f, 0.f};   // tokens 4 q + i, rank 16 rg + n
  for (int k0 = 0; k0 < n32; k0 += kUsSets) {
#pragma unroll
    for (int s = 0; s < kUsSets; ++s) {
      const int k = k0 + s;
      if (k >= n32) break;
      const uint32_t w[4] = {kx[s].x, kx[s].y, kx[s].z, kx[s].w};
      float m[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) m[e] = (float)as_h2(w[e >> 1])[e & 1];
      transpose_rows(m, 0);   // channels 8 i + q
      transpose_rows(m, 4);   // channels 8 i + 4 + q
      const int steps = (Q - 32 * k) / 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (2 * i >= steps) break;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(m[i], bx[s][2 * i], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(m[4 + i], bx[s][2 * i + 1], acc, 0, 0, 0);
      }
      if (k + kUsSets < n32) load(s, k + kUsSets);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) s_part[wave][4 * q + i][n] = acc[i];
  __syncthreads();
  const int o = tid & 15;
  us[oi] = float_to_half_bits(((s_part[0][ot][o] + s_part[1][ot][o]) + s_part[2][ot][o]) + s_part[3][ot][o]);
}

// One residual group's tokens x one head's channels, 512 threads: a thread has
// one channel and PER tokens: L = sum_r Us16[t][r] basis16[c][r] (fp32, ranks in
// order), R = M - L; the channel's scale is max |R| over the group / qmax and its
// codes clamp(rint(R / scale), -qmax - 1, qmax).  VALU-bound.
// Recipe's page (64 tokens, 128 channels): L on v_mfma_f32_16x16x4_f32 as Us is
// (the same bits as the chain of FMAs), a wave for 16 channels; the page's Us and
// the basis rows are read as the decode kernels read them, 4 or 8 ranks a lane.
// General page: thread (channel j = tid % d, part tid / d) takes tokens part,
// part + 512/d, ...; its basis row stays in registers (fp16 pairs, exact) and a
// token's Us row is one LDS broadcast per 8 ranks.
template <int R, int PER>
struct ResidualLds {
  static constexpr int kNG = 16 * PER < 128 ? 16 * PER : 128;   // tokens of a group, at most
  uint16_t us[kNG * R];
  float amax[512];
  int8_t code[512 * PER + 4 * kNG];                             // [tokens][d + 4]
};

template <int R, int PER, bool kGeneral>
__device__ __forceinline__ void encode_residual(const AppendKArgs& a, ResidualLds<R, PER>& s, int gi, int h) {
  const int tid = threadIdx.x, ld = kGeneral ? a.log2d : 7, D = 1 << ld;
  const int NG = (512 * PER) >> ld, C = a.C;
  const int slot0 = gi * (NG / kPT);                 // first 16-token page slot of the group
  const int n = tid & 15, q = (tid >> 4) & 3;
  const int j = kGeneral ? tid & (D - 1) : 16 * (tid >> 6) + n, part = kGeneral ? tid >> ld : q;
  const int parts = kGeneral ? 512 >> ld : 4;
  auto tok = [&](int k) { return kGeneral ? part + parts * k : 16 * (k >> 2) + 4 * q + (k & 3); };
  const bool aligned = (reinterpret_cast<uintptr_t>(a.basis16) & 15) == 0;
  float res[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k)
    res[k] = half_bits_to_float(a.k_pre[h * a.ksh + (int64_t)(slot0 * kPT + tok(k)) * a.kst + j]);
  float amax = 0.f;
  if constexpr (kGeneral) {
    half8_t b[R / 8];                                  // the channel's basis row
    const uint16_t* bp = a.basis16 + (int64_t)(h * D + j) * R;
    if (aligned) {
#pragma unroll
      for (int i = 0; i < R / 8; ++i) b[i] = *reinterpret_cast<const half8_t*>(bp + 8 * i);
    } else {
#pragma unroll
      for (int i = 0; i < R; ++i) b[i / 8][i % 8] = __builtin_bit_cast(_Float16, bp[i]);
    }
    for (int e = tid; e < NG * R / 2; e += 512) {      // rank pairs (2 e' even: within one row)
      const int t = 2 * e / R, r = 2 * e % R;
      reinterpret_cast<uint32_t*>(s.us)[e] =
          *reinterpret_cast<const uint32_t*>(append_page(a, slot0 + t / kPT) + a.L.us + 2 * ((t % kPT) * R + r));
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const half8_t* u = reinterpret_cast<const half8_t*>(s.us + tok(k) * R);
      float L = 0.f;
#pragma unroll
      for (int i = 0; i < R / 8; ++i) {
        const half8_t uv = u[i];
#pragma unroll
        for (int e = 0; e < 8; ++e) L = __builtin_fmaf((float)uv[e], (float)b[i][e], L);
      }
      res[k] = res[k] - L;
      amax = fmaxf(amax, fabsf(res[k]));
    }
  } else {
    // lane (n, q): ranks KQ q .. + KQ - 1 of token (A) or channel (B) n; after the
    // transposes register i holds rank 4 i + q of the step that takes it
    constexpr int KQ = R / 4;
    typedef _Float16 hvec_t __attribute__((ext_vector_type(KQ)));
    auto in_order = [&](const hvec_t& x, float (&f)[8]) {
#pragma unroll
      for (int e = 0; e < KQ; ++e) f[e] = (float)x[e];
      transpose_rows(f, 0);
      if constexpr (KQ == 8) transpose_rows(f, 4);
    };
    auto step = [](const float (&f)[8], int m) { return KQ == 8 ? f[4 * (m & 1) + (m >> 1)] : f[m]; };
    hvec_t uh[PER / 4], bh;
#pragma unroll
    for (int k = 0; k < PER / 4; ++k)
      uh[k] = *reinterpret_cast<const hvec_t*>(append_page(a, slot0 + k) + a.L.us + (tid & 63) * (2 * KQ));
    const uint16_t* bp = a.basis16 + (int64_t)(h * D + j) * R + KQ * q;
    if (aligned) {
      bh = *reinterpret_cast<const hvec_t*>(bp);
    } else {
#pragma unroll
      for (int i = 0; i < KQ; ++i) bh[i] = __builtin_bit_cast(_Float16, bp[i]);
    }
    float bf[8], uf[8];
    in_order(bh, bf);
#pragma unroll
    for (int k = 0; k < PER / 4; ++k) {
      in_order(uh[k], uf);
      float4_t L = {0.f, 0.f, 0.f, 0.f};   // tokens 16 k + 4 q + i, the lane's channel
#pragma unroll
      for (int m = 0; m < R / 4; ++m) L = __builtin_amdgcn_mfma_f32_16x16x4f32(step(uf, m), step(bf, m), L, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        res[4 * k + i] = res[4 * k + i] - L[i];
        amax = fmaxf(amax, fabsf(res[4 * k + i]));
      }
    }
  }
  s.amax[(part << ld) + j] = amax;
  __syncthreads();
  float mx = s.amax[j];
  for (int p = 1; p < parts; ++p) mx = fmaxf(mx, s.amax[(p << ld) + j]);
  const int qmax = kGeneral ? (1 << (a.bits - 1)) - 1 : 3;
  const float scale = fmaxf(mx, 1e-12f) / (float)qmax;
  const float lo = (float)(-qmax - 1), hi = (float)qmax;
  // scale is at least 1e-12 / 7; only the rounding near half codes matters, so
  // tiny residuals need no exact quotient
  if (__all(scale < 3.0e38f)) {
    const float rs = 1.0f / scale;
#pragma unroll
    for (int k = 0; k < PER; ++k)
      s.code[tok(k) * (D + 4) + j] = (int8_t)fminf(fmaxf(rintf(div_by(res[k], scale, rs)), lo), hi);
  } else {
#pragma unroll
    for (int k = 0; k < PER; ++k)
      s.code[tok(k) * (D + 4) + j] = (int8_t)fminf(fmaxf(rintf(res[k] / scale), lo), hi);
  }
  if (part == 0) {
    const int f = kGeneral ? h * D + j : kscale_flat(h * D + j), per_slot = C / (NG / kPT);
    const int slot = f / per_slot;
    *reinterpret_cast<uint16_t*>(append_page(a, slot0 + slot) + a.L.kscale + (f - slot * per_slot) * 2) =
        float_to_half_bits(scale);
  }
  __syncthreads();
  if constexpr (kGeneral) {
    // KRES: 8 channels (4 bytes) of one token per item, offset-binary nibbles
    const int off = 1 << (a.bits - 1), l8 = ld - 3;
    for (int e = tid; e < NG << l8; e += 512) {
      const int t = e >> l8, j8 = e & ((1 << l8) - 1);
      uint32_t w = 0u;
#pragma unroll
      for (int i = 0; i < 8; ++i) w |= (uint32_t)(s.code[t * (D + 4) + 8 * j8 + i] + off) << (4 * i);
      *reinterpret_cast<uint32_t*>(append_page(a, slot0 + t / kPT) + a.L.kres + (h * kPT + t % kPT) * (D / 2) +
                                   4 * j8) = w;
    }
  } else if (tid < 256) {
    // thread -> (page pl, lane 16q+n); pair p = 4b+i is channels (j, j+64),
    // j = 16b + 4q + i, stored offset-binary
    const int pl = tid >> 6, lane = tid & 63, q = lane >> 4, n = lane & 15;
    const int8_t* c = s.code + (pl * kPT + n) * (kD + 4);
    uint32_t w[3] = {0u, 0u, 0u};
#pragma unroll
    for (int p = 0; p < 16; ++p) {
      const int jj = 16 * (p >> 2) + 4 * q + (p & 3);
      const uint32_t lo3 = (uint32_t)(c[jj] + 4), hi3 = (uint32_t)(c[jj + 64] + 4);
      if (p < 15) {
        w[p / 5] |= (lo3 << (3 * (p % 5))) | (hi3 << (16 + 3 * (p % 5)));
      } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) w[k] |= (((lo3 >> k) & 1u) << 15) | (((hi3 >> k) & 1u) << 31);
      }
    }
    uint32_t* dst = reinterpret_cast<uint32_t*>(append_page(a, slot0 + pl) + a.L.kres + h * 768 + lane * 12);
    dst[0] = w[0]; dst[1] = w[1]; dst[2] = w[2];
  }
}

// Eight tokens of one head, one wave: lane 8t + j holds channels 8i + j of
// token t.  The fp16 norm in the order torch's CPU 2-norm reduces a row (8
// strided FMA accumulators -- one per lane --, then those left to right, then a
// correctly rounded sqrt), the unit row times the signs, the FWHT's stages in
// the reference's order (channel bits 0..2 across the token's lanes by DPP, the
// others in registers), and each code as the count of thresholds the rotated
// value reaches (code_cuts: the values from which (x / sqrt(d)) * sqrt(d) > mid).
// No LDS and no barrier; VALU-bound, ~27 instructions a value.
template <int D>
__device__ __forceinline__ void encode_values(const AppendKArgs& a, int pg, int half, int h, bool recipe) {
  constexpr int NI = D / 8;
  const int lane = threadIdx.x & 63, j = lane & 7, tok = 8 * half + (lane >> 3);
  const int64_t row = h * a.vsh + (int64_t)(pg * kPT + tok) * a.vst + j;
  float x[NI];
  bool tiny = false;   // a nonzero value below 2^-100: div_by would not be exact
  if (a.v_dtype == BMX_K2B_F16) {
#pragma unroll
    for (int i = 0; i < NI; ++i) x[i] = half_bits_to_float(static_cast<const uint16_t*>(a.v)[row + 8 * i]);
  } else {
    if (a.v_dtype == BMX_K2B_BF16) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        x[i] = __uint_as_float((uint32_t)static_cast<const uint16_t*>(a.v)[row + 8 * i] << 16);
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) x[i] = static_cast<const float*>(a.v)[row + 8 * i];
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) tiny |= (x[i] != 0.f) & (fabsf(x[i]) < 0x1p-100f);
  }
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) acc = __builtin_fmaf(x[i], x[i], acc);
  // the 8 lanes' sums, left to right, in every lane of the token
  auto of_lane = [&](auto k) {   // lane k of each group of 8
    return __builtin_bit_cast(
        float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, acc), 0x18 | (decltype(k)::value << 5)));
  };
  const float s1 = of_lane(std::integral_constant<int, 1>{}), s2 = of_lane(std::integral_constant<int, 2>{}),
              s3 = of_lane(std::integral_constant<int, 3>{}), s4 = of_lane(std::integral_constant<int, 4>{}),
              s5 = of_lane(std::integral_constant<int, 5>{}), s6 = of_lane(std::integral_constant<int, 6>{}),
              s7 = of_lane(std::integral_constant<int, 7>{});
  float ss = of_lane(std::integral_constant<int, 0>{});
  ss = ((((((ss + s1) + s2) + s3) + s4) + s5) + s6) + s7;
  const uint16_t nb = float_to_half_bits(fmaxf(__builtin_sqrtf(ss), 1e-12f));
  const float nrm = half_bits_to_float(nb);
  uint8_t* page = append_page(a, __builtin_amdgcn_readfirstlane(pg));
  if (j == 0) *reinterpret_cast<uint16_t*>(page + a.L.vnorm + (h * kPT + tok) * 2) = nb;
  if (__all(nrm > 0.f && nrm < 65505.f && !tiny)) {
    const float r = 1.0f / nrm;
#pragma unroll
    for (int i = 0; i < NI; ++i) x[i] = div_by(x[i], nrm, r);
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i) x[i] = x[i] / nrm;
  }
#pragma unroll
  for (int i = 0; i < NI; ++i)   // channel 8i + j: byte i & 3 of sign word i >> 2
    x[i] = __uint_as_float(__float_as_uint(x[i]) ^ (((a.v_sign_bits[i >> 2] >> (8 * (i & 3) + j)) & 1u) << 31));
  // FWHT stages (c, c + hb): the upper lane's partner minus its own
  const float g1 = (j & 1) ? -1.f : 1.f, g2 = (j & 2) ? -1.f : 1.f, g4 = (j & 4) ? -1.f : 1.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) x[i] = __builtin_fmaf(g1, x[i], xor_row16<1>(x[i]));
#pragma unroll
  for (int i = 0; i < NI; ++i) x[i] = __builtin_fmaf(g2, x[i], xor_row16<2>(x[i]));
#pragma unroll
  for (int i = 0; i < NI; ++i) x[i] = __builtin_fmaf(g4, x[i], xor_row16<4>(x[i]));
#pragma unroll
  for (int hb = 1; hb < NI; hb <<= 1)
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (!(i & hb)) {
        const float u = x[i], w = x[i | hb];
        x[i] = u + w;
        x[i | hb] = u - w;
      }
  const float k0 = a.code_cuts[0], k1 = a.code_cuts[1], k2 = a.code_cuts[2];
  const int t4 = tok & 3, q = tok >> 2;
  uint32_t w[NI / 4];
#pragma unroll
  for (int k = 0; k < NI / 4; ++k) w[k] = 0u;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const uint32_t code = (uint32_t)(x[i] >= k0) + (uint32_t)(x[i] >= k1) + (uint32_t)(x[i] >= k2);
    // recipe's page: dword 2 (i & 1) + (b >> 2), channel block b = i >> 1, byte
    // b & 3; general page: dword i >> 2, byte i & 3
    if (D == 128 && recipe) w[2 * (i & 1) + (i >> 3)] |= code << (8 * ((i >> 1) & 3));
    else w[i >> 2] |= code << (8 * (i & 3));
  }
  // a byte holds the codes of 4 tokens: those of lanes ^ 8, ^ 16, ^ 24
#pragma unroll
  for (int k = 0; k < NI / 4; ++k) {
    uint32_t v = w[k] << (2 * t4);
    v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, true);   // row rotation by 8: lane ^ 8
    v |= (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x1F | (16 << 10));     // lane ^ 16
    w[k] = v;
  }
  if (D == 128 && recipe) {   // token t4's lane writes dword t4: lane 16q + m, m = 8 (t4 >> 1) + j, word t4 & 1
    const uint32_t lo = (t4 & 1) ? w[1] : w[0], hi = (t4 & 1) ? w[NI / 4 - 1] : w[NI >= 12 ? 2 : 0];
    *reinterpret_cast<uint32_t*>(page + a.L.vcode + h * 512 + (16 * q + 8 * (t4 >> 1) + j) * 8 + 4 * (t4 & 1)) =
        (t4 & 2) ? hi : lo;
  } else {                    // VCODE [h][4][d] bytes: token t4's lane writes bytes t4 of each dword
    uint8_t* dst = page + a.L.vcode + (h * 4 + q) * D + j;
#pragma unroll
    for (int k = 0; k < NI / 4; ++k) dst[8 * (4 * k + t4)] = (uint8_t)(w[k] >> (8 * t4));
  }
}

// The recipe's page: workgroups [0, 2 h n) encode the residual of one 64-token
// group of one head, the rest the values of 64 tokens of one head (8 waves x 8
// tokens).  One launch for both: a commit of one codec page has 16 workgroups
// of each, and they run side by side.  Measured at h_kv 8: 5.8 us for one codec
// page at R 32 and 18.9 us for 63 at R 16 (6.6 and 19.8 with the residual's
// product as FMAs); the two as kernels of their own, with
// both residual operands from LDS and the FWHT's stages through LDS with a
// barrier each, 21.7 + 7.5 and 27.1 + 27.1 us.
template <int R>
__global__ __launch_bounds__(512) void append_codes_kernel(const AppendKArgs a, int n_res) {
  __shared__ ResidualLds<R, 16> s;
  const int i = (int)blockIdx.x < n_res ? blockIdx.x : blockIdx.x - n_res;
  const int u = i / a.h_kv, h = i - u * a.h_kv;
  if ((int)blockIdx.x < n_res) {
    encode_residual<R, 16, false>(a, s, u, h);
  } else {
    const int wave = threadIdx.x >> 6;
    encode_values<128>(a, 4 * u + (wave >> 1), wave & 1, h, true);
  }
}

// grid (residual groups of the call, h_kv), block 512 (general page).
template <int R, int PER>
__global__ __launch_bounds__(512) void gen_kres_kernel(const AppendKArgs a) {
  __shared__ ResidualLds<R, PER> s;
  encode_residual<R, PER, true>(a, s, blockIdx.x, blockIdx.y);
}

// grid (16-token pages of the call, h_kv), block 128: a wave for 8 tokens.
template <int D>
__global__ __launch_bounds__(128) void value_codes_kernel(const AppendKArgs a) {
  encode_values<D>(a, blockIdx.x, threadIdx.x >> 6, blockIdx.y, !a.general);
}

// The smallest float x with (x / s) * s > mid, s = fl(sqrt(d)): the codes'
// test as one compare (both operations are monotonic in x).  NaN (no such x)
// where mid is not a number below infinity.
static float code_cut(float mid, float s) {
  if (!(mid < INFINITY)) return NAN;
  auto above = [&](float x) {
    volatile float q = x / s;
    volatile float r = q * s;
    return r > mid;
  };
  float x = std::max(mid, -3.0e38f);
  for (int i = 0; i < 64 && above(x); ++i) x = std::nextafterf(x, -INFINITY);
  for (int i = 0; i < 64 && !above(x); ++i) x = std::nextafterf(x, INFINITY);
  return x;
}

void set_code_cuts(AppendKArgs& k, const float codebook[4], int d) {
  const float s = std::sqrt((float)d);   // correctly rounded
  for (int i = 0; i < 3; ++i) k.code_cuts[i] = code_cut((codebook[i] + codebook[i + 1]) / 2.0f, s);
}

// The values alone, for pages whose layout has value sections only (the
// spectral key path keeps its keys in pages of its own).
hipError_t launch_k2b_values(const AppendKArgs& a, int n_pages16, int h_kv, hipStream_t st) {
  hipLaunchKernelGGL(value_codes_kernel<128>, dim3(n_pages16, h_kv), dim3(128), 0, st, a);
  return hipGetLastError();
}

static void launch_us(const AppendKArgs& k, int n_slots, hipStream_t st) {
  const bool vec = (reinterpret_cast<uintptr_t>(k.k_pre) & 15) == 0 && k.ksh % 8 == 0 && k.kst % 8 == 0;
  const dim3 grid(n_slots, k.R / 16);
  if (vec) hipLaunchKernelGGL(append_us_kernel<true>, grid, dim3(256), 0, st, k);
  else hipLaunchKernelGGL(append_us_kernel<false>, grid, dim3(256), 0, st, k);
}

template <int R>
static void launch_gen_kres(const AppendKArgs& k, int per, dim3 grid, hipStream_t st) {
  switch (per) {
    case 1: hipLaunchKernelGGL((gen_kres_kernel<R, 1>), grid, dim3(512), 0, st, k); break;
    case 2: hipLaunchKernelGGL((gen_kres_kernel<R, 2>), grid, dim3(512), 0, st, k); break;
    case 4: hipLaunchKernelGGL((gen_kres_kernel<R, 4>), grid, dim3(512), 0, st, k); break;
    case 8: hipLaunchKernelGGL((gen_kres_kernel<R, 8>), grid, dim3(512), 0, st, k); break;
    case 16: hipLaunchKernelGGL((gen_kres_kernel<R, 16>), grid, dim3(512), 0, st, k); break;
    default: hipLaunchKernelGGL((gen_kres_kernel<R, 32>), grid, dim3(512), 0, st, k); break;
  }
}

}  // namespace bmx

using namespace bmx;

static int afail(int code, const std::string& msg) {
  bmx_set_error(msg);
  return code;
}

extern "C" int bmx_k2b_append(const bmx_k2b_append_args* a, void* stream) {
  if (!a) return afail(BMX_E_INVALID, "bmx_k2b_append: args is NULL");
  const bmx_k2b_geom& g = a->geom;
  const Geo geo = Geo::from(g);
  if (g.h_kv < 1 || g.h_kv > 16) return afail(BMX_E_INVALID, "bmx_k2b_append: h_kv must be 1..16");
  if (!geo.general && g.rank != 16 && g.rank != 32)
    return afail(BMX_E_INVALID, "bmx_k2b_append: rank must be 16 or 32");
  if (geo.general && !geo.check().empty()) return afail(BMX_E_INVALID, "bmx_k2b_append: " + geo.check());
  if (a->n_codec_pages < 0) return afail(BMX_E_INVALID, "bmx_k2b_append: n_codec_pages < 0");
  if (a->n_codec_pages == 0) return BMX_OK;
  if (!a->k_pre || !a->v || !a->basis32 || !a->basis16 || !a->pages || !a->page_ids)
    return afail(BMX_E_INVALID, "bmx_k2b_append: null pointer argument");
  if (a->n_pool_pages < 1) return afail(BMX_E_INVALID, "bmx_k2b_append: n_pool_pages must be >= 1");
  if (reinterpret_cast<uintptr_t>(a->basis32) % 16 != 0)
    return afail(BMX_E_INVALID, "bmx_k2b_append: basis32 must be 16-byte aligned");
  if (a->v_dtype != BMX_K2B_F16 && a->v_dtype != BMX_K2B_F32 && a->v_dtype != BMX_K2B_BF16)
    return afail(BMX_E_INVALID, "bmx_k2b_append: v_dtype must be BMX_K2B_F16, _F32 or _BF16");
  AppendKArgs k{};
  k.h_kv = g.h_kv; k.R = geo.R; k.n_codec_pages = a->n_codec_pages;
  k.C = geo.C(); k.log2d = __builtin_ctz((unsigned)geo.d); k.bits = geo.bits; k.general = geo.general;
  k.k_pre = a->k_pre; k.ksh = a->k_stride_h; k.kst = a->k_stride_t;
  k.v = a->v; k.vsh = a->v_stride_h; k.vst = a->v_stride_t; k.v_dtype = a->v_dtype;
  k.basis32 = a->basis32; k.basis16 = a->basis16; k.us_first = a->us_first;
  k.pages = a->pages; k.page_ids = a->page_ids; k.n_pool = a->n_pool_pages;
  if (geo.general) {
    const GenLayout L = GenLayout::of(geo);
    k.L.us = L.us; k.L.vnorm = L.vnorm; k.L.kscale = L.kscale; k.L.kres = L.kres; k.L.vcode = L.vcode;
    k.L.bytes = L.bytes;
  } else {
    k.L = PageLayout::make(g.h_kv, g.rank);
  }
  for (int i = 0; i < 4; ++i) k.v_sign_bits[i] = a->v_sign_bits[i];
  set_code_cuts(k, a->codebook, geo.d);
  hipStream_t st = (hipStream_t)stream;
  const int slots = a->n_codec_pages * 8;
  launch_us(k, slots, st);
  if (!geo.general) {
    const int n_res = a->n_codec_pages * 2 * g.h_kv;   // workgroups of the residual, and as many of the values
    if (geo.R == 32) hipLaunchKernelGGL(append_codes_kernel<32>, dim3(2 * n_res), dim3(512), 0, st, k, n_res);
    else hipLaunchKernelGGL(append_codes_kernel<16>, dim3(2 * n_res), dim3(512), 0, st, k, n_res);
  } else {
    const dim3 kgrid(a->n_codec_pages * (kCodec / geo.group), geo.h), vgrid(slots, geo.h);
    const int per = geo.group * geo.d / 512;
    if (geo.R == 16) launch_gen_kres<16>(k, per, kgrid, st);
    else if (geo.R == 32) launch_gen_kres<32>(k, per, kgrid, st);
    else if (geo.R == 64) launch_gen_kres<64>(k, per, kgrid, st);
    else launch_gen_kres<128>(k, per, kgrid, st);
    if (geo.d == 32) hipLaunchKernelGGL(value_codes_kernel<32>, vgrid, dim3(128), 0, st, k);
    else if (geo.d == 64) hipLaunchKernelGGL(value_codes_kernel<64>, vgrid, dim3(128), 0, st, k);
    else hipLaunchKernelGGL(value_codes_kernel<128>, vgrid, dim3(128), 0, st, k);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return afail(BMX_E_HIP, std::string("bmx_k2b_append: launch: ") + hipGetErrorString(e));
  return BMX_OK;
}
