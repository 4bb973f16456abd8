// The k2b path on the general page (include/bmx_k2b.h): head_dim 32, 64 or
// 128, rank 16..128, residual group 16..128 tokens, 2..4-bit keys, gfx950.
//
// The read side (k2b_append.hip writes the pages):
//   gen_split_kernel one workgroup of 8 waves per (split, head block, sequence),
//                    a wave per KV head (or several per head when there are
//                    fewer heads than waves), 4 pages at a time: RoPE tables
//                    shared by the heads in LDS, keys rebuilt on MFMA (K^T =
//                    basis * Us^T), residual and rotation in registers, scores
//                    K^T Q^T on MFMA, online softmax, V^T P^T on MFMA in the
//                    rotated value domain, the inverse Hadamard at the end
//   combine_kernel   (decode_shared.h) merges the splits and the recent window
//   gen_dequant_kernel  dense keys and values of committed pages (prefill)
// Reference semantics: cache/packed_streaming.py:475-580 and 957-1060,
// cache/codecs.py:616-649, 677-695, 786-796, quant/rtn.py:23-44,
// quant/hadamard.py:12-33, cache/triton_dequant_attention.py:1232-1368.
// This file is built without floating-point contraction.

#include <algorithm>
#include <string>

#include "decode_shared.h"
#include "k2b_general.h"

namespace bmx {

// ---------------------------------------------------------------------------
// Dequant.  MFMA 16x16x16 f16 fragments (lane l = 16 qd + n): A holds
// A[n][4qd .. 4qd+3], B holds B[4qd .. 4qd+3][n], the result D[4qd + e][n].
//   K^T tile rt (channels 16rt ..): A = basis rows 16rt + n, ranks 16ks + 4qd ..
//     (LDS), B = Us[token n][16ks + 4qd ..] -> lane: K[16rt + 4qd + e][token n]
// RoPE pairs channels j and j + d/2: tiles rt and rt + d/32 of the same lane.
// ---------------------------------------------------------------------------
struct GenReadArgs {
  GenLayout L;
  const uint8_t* pages;
  const int32_t* page_table;   // [B][max_pages] or NULL: page b * max_pages + i
  int max_pages, n_pool;
  const uint16_t* basis;       // [C][R] fp16 (+ b * basis_stride)
  int64_t basis_stride;
  float inv_freq[64];
  float rope_scaling;
  float level[4];
  uint32_t v_sign_bits[4];
};

__device__ __forceinline__ const uint8_t* gen_read_page(const GenReadArgs& a, int b, int p) {
  const int32_t pid = a.page_table ? a.page_table[(int64_t)b * a.max_pages + p] : b * a.max_pages + p;
  return a.pages + clamp_page(pid, a.n_pool) * (int64_t)a.L.bytes;
}

// The lane's rebuilt keys of one page (before RoPE): kt[rt][e] = channel
// 16rt + 4qd + e of token n (head h).
template <int D, int R>
__device__ __forceinline__ void gen_keys(const GenReadArgs& a, const uint8_t* pg, const uint16_t* s_B, int b,
                                         int p, int h, int n, int qd, float4_t kt[D / 16]) {
  constexpr int NT = D / 16, NK = R / 16, LDB = R + 4;
  const GenLayout& L = a.L;
  half4_t us[NK];
#pragma unroll
  for (int ks = 0; ks < NK; ++ks)
    us[ks] = *reinterpret_cast<const half4_t*>(pg + L.us + (n * R + 16 * ks + 4 * qd) * 2);
  uint32_t kr[NT];
  half4_t sc[NT];
  const int p0 = p - p % L.slots;   // first page of the residual group
#pragma unroll
  for (int rt = 0; rt < NT; ++rt) {
    kr[rt] = *reinterpret_cast<const uint16_t*>(pg + L.kres + (h * kPT + n) * (D / 2) + (16 * rt + 4 * qd) / 2);
    const int c0 = h * D + 16 * rt + 4 * qd, slot = c0 / L.per_slot;
    const uint8_t* spg = slot == p - p0 ? pg : gen_read_page(a, b, p0 + slot);
    sc[rt] = *reinterpret_cast<const half4_t*>(spg + L.kscale + (c0 % L.per_slot) * 2);
  }
  const int off = 1 << (L.bits - 1);
#pragma unroll
  for (int rt = 0; rt < NT; ++rt) {
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      const half4_t bw = *reinterpret_cast<const half4_t*>(s_B + (16 * rt + n) * LDB + 16 * ks + 4 * qd);
      acc = __builtin_amdgcn_mfma_f32_16x16x16f16(bw, us[ks], acc, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      acc[e] = __builtin_fmaf((float)sc[rt][e], (float)((int)((kr[rt] >> (4 * e)) & 15u) - off), acc[e]);
    kt[rt] = acc;
  }
}

// RoPE of the lane's keys at position pos: mode 1 exact fp32 cos/sin, mode 2
// the fp16-rounded tables (cos and sin times rope_scaling, then fp16).
template <int D>
__device__ __forceinline__ void gen_rope(const GenReadArgs& a, float4_t kt[D / 16], int pos, int qd, int mode) {
  constexpr int NP = D / 32;
#pragma unroll
  for (int rt = 0; rt < NP; ++rt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float ang = (float)pos * a.inv_freq[16 * rt + 4 * qd + e];
      float sn, cs;
      sincosf(ang, &sn, &cs);
      cs = cs * a.rope_scaling;
      sn = sn * a.rope_scaling;
      if (mode == 2) {
        cs = (float)(_Float16)cs;
        sn = (float)(_Float16)sn;
      }
      const float x = kt[rt][e], y = kt[rt + NP][e];
      kt[rt][e] = x * cs - y * sn;
      kt[rt + NP][e] = y * cs + x * sn;
    }
}

// ---------------------------------------------------------------------------
// Decode.  Fragments of the 16x16x32 f16 MFMA (lane l = 16 qd + n): A holds
// A[n][8qd .. 8qd+7], B holds B[8qd .. 8qd+7][n], the result D[4qd + e][n].
//   K^T tile rt: A = the basis row of the channel that row n stands for, ranks
//     32ks + 8qd .., B = Us[token n][32ks + 8qd ..] -> lane: channel of row
//     4qd + e, token n.  Row 4qd + e of tile rt < d/32 stands for channel
//     qd d/8 + 4rt + e, of tile rt + d/32 for that channel + d/2: a lane's
//     channels are two runs of d/8, so its codes, scales and table entries are
//     contiguous, and both channels of a RoPE pair are in one lane
//   S^T = K^T Q^T: the keys as fp16 high and low parts (kh, kl), the queries
//     too (qh, ql): one product of (kh, kl) against (qh, qh) per tile and one of
//     (kh, kh') against (ql, ql') per tile pair: kl ql is below 2^-22
//     -> lane: score of token 4qd + e for query n
//   V^T P^T: A = the levels (fp16 high and low parts) of channel n d/16 + ct,
//     tokens 4qd .. 4qd+3 (one code byte through an LDS table), B = the lane's own
//     weight times norm as high and low parts: (lh, lh) against (ph, pl) per page
//     and (ll, ll') against (ph, ph') per page pair
//     -> lane: channel (4qd + e) d/16 + ct for query n
// A low part holds nothing below 2^-25, so weight times norm is not taken
// relative to the largest weight (as the weights' sum is): with small norms, or
// with all tokens under a sink, it would lose its bits.  The accumulator has a
// maximum of its own, a bound of score + log2(norm) -- a lane's largest score plus
// its largest norm --, and its operand fills fp16's range up to 2^14 of it: what
// lies up to 2^-24 below the bound keeps 2^-22 of itself.  Both maxima are whole
// numbers of base-2 scores, so rescaling by them is exact.  Error against float64
// at norms of 1e-4: 7e-4 with weight times norm relative to the largest weight,
// 2e-4 with the weight and level times norm as a pair each, 1e-6 now.
// G queries fill G of the 16 columns; pages are compacted SW columns apart (as
// k2b_decode_split_kernel does), so the softmax runs once per 16/SW pages.
//
// What bounds it: VALU issue and the fixed latency of two launches.  A page of
// one head takes ~135 VALU (residual 48, rotation 32, high and low parts 32)
// and, a quarter of its quad's softmax and products, ~45 more at d 64; the
// HBM floor of 32,640 tokens at d 64, rank 16, h_kv 8 is 2.6 us.  Measured there
// (G 4, 128-row window): split 17.5 + merge 4.3 us, 19.7 us a call; a workgroup
// per (split, head) with a page at a time per wave, the rotation remade per head
// and page (22 of them, f64 included, per RoPE pair) and a merge workgroup per
// query took 31.6 + 8.5 us, 37.4 us a call.  d 128, rank 64: 92 -> 37 us a call.
// ---------------------------------------------------------------------------
struct GenDecodeArgs {
  GenReadArgs r;
  int G, n_split, hpb, wph;        // workgroups of a sequence and head block, heads of a block, waves of a head
  int win_tiles, win_wgs;          // 16-token tiles of the window, workgroups a sequence has for them alone
  int div32;                       // (n_split + 1) * quads < 2^32
  float inv_per_slot;              // 1 / L.per_slot
  int b0;                          // the call's sequence that block z = 0 serves (the pointers start there)
  const void* q;
  int io_dtype;
  const int32_t* packed_len;
  int max_packed_len;
  float qscale;                    // sm_scale * log2(e): scores in base 2
  float* ws_acc;                   // [B][h][G][d/16][n_split wph][16] fp32 records (means over the split)
  float* ws_ml;                    // [B][h][G][n_split wph][2] (max, sum)
  float* ws_win;                   // [B][h][G][tail_cap] window scores, base 2
  const uint16_t* k_tail;
  int64_t ts_b, ts_h, ts_t;
  int tail_cap, tail_bf16;
  WinNew nw;
};

constexpr int kGenQuad = 4;        // pages a wave takes at a time
constexpr float kGenUp = 14.f;     // log2 of the largest weight times norm as an operand (fp16's largest is 2^16)
constexpr int kGenTables = 4;      // RoPE tables (64 positions each) in LDS
constexpr int kGenIds = 64;        // page ids held per lane vector
template <int D>
constexpr int gen_cs_row() { return D / 2 + 4; }   // dwords per position row of a table (rows 4 banks apart)
template <int D>
constexpr size_t gen_lds() { return (size_t)kGenTables * 64 * gen_cs_row<D>() * 4; }
// 8 waves a workgroup (2 per SIMD), or 4 where the basis and query fragments need
// more than the 256 registers that leaves a wave
constexpr int gen_waves(int D, int R) { return D == 128 || R == 128 ? 4 : 8; }

// N bytes at p (16, 8, 4 or 2) as dwords
template <int N>
struct GenBytes {
  uint32_t w[(N + 3) / 4];
  __device__ __forceinline__ void load(const uint8_t* p) {
    if constexpr (N == 16) {
      const uint4 v = *reinterpret_cast<const uint4*>(p);
      w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    } else if constexpr (N == 8) {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      w[0] = v.x; w[1] = v.y;
    } else if constexpr (N == 4) {
      w[0] = *reinterpret_cast<const uint32_t*>(p);
    } else {
      w[0] = *reinterpret_cast<const uint16_t*>(p);
    }
  }
};

__device__ __forceinline__ half2_t gen_half2(float x, float y) {   // one v_cvt_pk_f16_f32: to nearest
  typedef float f2_t __attribute__((ext_vector_type(2)));
  return __builtin_convertvector((f2_t{x, y}), half2_t);
}

// x and y as fp16 high parts and the fp16 low parts that remain, both to nearest
// (x = h + l to 2^-23 where l is normal).  m1: -1 in a register the compiler
// cannot see through, so that x - h reads the fp16 h in place (v_fma_mix_f32;
// exact), with no conversion instruction.
__device__ __forceinline__ void gen_split2(float x, float y, float m1, uint32_t& hi, uint32_t& lo) {
  const half2_t h = gen_half2(x, y);
  hi = as_u32(h);
  lo = as_u32(gen_half2(__builtin_fmaf((float)h[0], m1, x), __builtin_fmaf((float)h[1], m1, y)));
}

// One 16-token tile of one head's recent window against its G queries: S^T = K Q^T
// on MFMA (A: token n, channels 32c + 8qd ..; B: query n, the same channels; the
// lane gets tokens 4qd + e of query n).  The query row is scaled by a power of two
// so that its largest element is 2^13 .. 2^14, and split into rounded parts that
// carry it to fp32: two of fp16, or three of bf16 for a bf16 window; the sums are
// fp32, the later parts' apart, and scaled back: an output's error against float64
// 3e-7, 6e-7 with fp32 products.  Rows given apart are also stored into the window buffer.
// Bound: one load round trip, whatever G is.  Products on the VALU took the queries
// 2 or 4 at a time, a round trip each, at one or two waves a SIMD: 40 sequences of
// 128 tokens and 128 window rows, G 16: 16 heads, d 64, rank 128 150.4 -> 124.2 us a
// call, 8 heads, d 32, rank 16 51.5 -> 33.5.  Loading a wave's next tile ahead: the
// same to 2 %.
template <int D>
__device__ __forceinline__ void gen_window_tile(const GenDecodeArgs& a, int b, int h, int j, int n, int qd) {
  constexpr int NP = D / 16;   // 4-channel pieces of a lane: two of each 32 channels
  auto at = [](int k) { return 32 * (k >> 1) + 4 * (k & 1); };
  const int t = 16 * j + n, i_new = fresh_row(a.nw, t);
  const int64_t tb = (int64_t)b * a.ts_b + (int64_t)h * a.ts_h;
  const uint16_t* row = (i_new >= 0 ? a.nw.k + (int64_t)b * a.nw.sb + (int64_t)h * a.nw.sh + (int64_t)i_new * a.nw.st
                                    : a.k_tail + tb + (int64_t)(t < a.tail_cap ? t : 0) * a.ts_t) + 8 * qd;
  uint2 kw[NP];
#pragma unroll
  for (int k = 0; k < NP; ++k) kw[k] = *reinterpret_cast<const uint2*>(row + at(k));
  const int64_t r0 = ((int64_t)b * a.r.L.h + h) * a.G, q0 = (r0 + (n < a.G ? n : 0)) * D + 8 * qd;
  RawQ4 qr[NP];
  load_q4(a.q, a.io_dtype, [&](int k) { return q0 + at(k); }, qr);
  if (i_new >= 0) {
    uint16_t* dst = a.nw.k_dst + tb + (int64_t)t * a.ts_t + 8 * qd;
#pragma unroll
    for (int k = 0; k < NP; ++k) *reinterpret_cast<uint2*>(dst + at(k)) = kw[k];
  }
  float4_t x[NP];
  cvt_q4(qr, a.io_dtype, x);
  const float sc = n < a.G ? a.qscale : 0.f;
  float mx = 0.f;
#pragma unroll
  for (int k = 0; k < NP; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[k][e] *= sc;
      mx = fmaxf(mx, fabsf(x[k][e]));
    }
  mx = fmaxf(mx, __shfl_xor(mx, 16));
  mx = fmaxf(mx, __shfl_xor(mx, 32));
  const int up = 14 - __builtin_amdgcn_frexp_expf(mx);
  const bool bf = __builtin_amdgcn_readfirstlane(a.tail_bf16) != 0;
  float4_t s = {0.f, 0.f, 0.f, 0.f}, low = s;   // sums of the first parts, of the later ones
#pragma unroll
  for (int c = 0; c < NP / 2; ++c) {
    union { uint2 u[2]; half8_t h; bf16x8_t v; } kk = {{kw[2 * c], kw[2 * c + 1]}};
    float r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = __builtin_amdgcn_ldexpf(x[2 * c + (i >> 2)][i & 3], up);
    if (bf) {
#pragma unroll
      for (int part = 0; part < 3; ++part) {
        union { uint16_t w[8]; bf16x8_t v; } q;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t w = bf16_bits(r[i]);
          q.w[i] = (uint16_t)w;
          r[i] -= __uint_as_float(w << 16);
        }
        float4_t& sum = part ? low : s;
        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kk.v, q.v, sum, 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int part = 0; part < 2; ++part) {
        half8_t q;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          q[i] = (_Float16)r[i];
          r[i] -= (float)q[i];
        }
        float4_t& sum = part ? low : s;
        sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(kk.h, q, sum, 0, 0, 0);
      }
    }
  }
  // an infinite key makes its later parts' products infinite of either sign, or not
  // a number: the score is the first parts' infinity
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = fabsf(s[e]) == INFINITY ? s[e] : s[e] + low[e];
  if (n < a.G) {
    float* dst = a.ws_win + (r0 + n) * a.tail_cap;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (16 * j + 4 * qd + e < a.tail_cap) dst[16 * j + 4 * qd + e] = __builtin_amdgcn_ldexpf(s[e], -up);
  }
}

template <int D, int R, int SW>
__global__ __launch_bounds__(64 * gen_waves(D, R)) void gen_split_kernel(const GenDecodeArgs a) {
  constexpr int NWV = gen_waves(D, R), NT = D / 16, NP = NT / 2, NK = R >= 32 ? R / 32 : 1;
  constexpr int KQ = R >= 32 ? 8 : 4;            // ranks per lane of one K^T product
  constexpr int NSLOT = 16 / SW, NCR = kGenQuad / NSLOT;
  constexpr int RUN = D / 8;                     // channels of a lane's run
  constexpr int CSROW = gen_cs_row<D>();
  constexpr int PF = D == 128 ? 2 : 4;           // pages whose key data is in flight or in use
  typedef _Float16 hvec_t __attribute__((ext_vector_type(KQ)));
  extern __shared__ __attribute__((aligned(16))) uint32_t s_cs[];   // [tables][64][CSROW]: fp16 (cos, sin)
  // the 4 levels of a code byte (tokens 4a .. 4a + 3): fp16 high parts twice (the
  // product's operand as it is), low parts
  __shared__ uint4 s_lvh[256];
  __shared__ uint2 s_lvl[256];
  // the scalar arguments of the prologue requested at once: one round trip
  asm volatile("" ::"s"(a.r.pages), "s"(a.r.page_table), "s"(a.r.max_pages), "s"(a.r.n_pool), "s"(a.r.basis),
               "s"(a.r.basis_stride), "s"(a.r.rope_scaling), "s"(a.G), "s"(a.n_split), "s"(a.hpb), "s"(a.wph),
               "s"(a.div32), "s"(a.inv_per_slot), "s"(a.b0), "s"(a.q), "s"(a.io_dtype), "s"(a.packed_len),
               "s"(a.max_packed_len), "s"(a.qscale));
  asm volatile("" ::"s"(a.r.L.us), "s"(a.r.L.vnorm), "s"(a.r.L.kscale), "s"(a.r.L.kres), "s"(a.r.L.vcode),
               "s"(a.r.L.bytes), "s"(a.r.L.h), "s"(a.r.L.bits), "s"(a.r.L.slots), "s"(a.r.L.per_slot),
               "s"(a.r.level[0]), "s"(a.r.level[1]), "s"(a.r.level[2]), "s"(a.r.level[3]));
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int n = lane & 15, qd = lane >> 4;
  const GenLayout& L = a.r.L;
  const int split = blockIdx.x, b = blockIdx.z, G = a.G;
  // the window's (16-token tile, head) pairs, dealt over workgroups and waves:
  // over the sequence's own workgroups at their end, or over win_wgs more that do
  // nothing else
  auto window = [&](int wg, int n_x) {
    const int n_wg = n_x * gridDim.y, n_pairs = a.win_tiles * L.h;
    for (int p = wg + n_x * blockIdx.y + wave * n_wg; p < n_pairs; p += NWV * n_wg) {
      const int j = p / L.h;
      gen_window_tile<D>(a, b, p - j * L.h, j, n, qd);
    }
  };
  if (split >= a.n_split) {
    window(split - a.n_split, a.win_wgs);
    return;
  }
  const float freq = a.r.inv_freq[tid & (D / 2 - 1)];   // the RoPE frequency this thread makes table entries of
  const int len_raw = a.packed_len[b];
  const int sub = wave / a.hpb, h_own = blockIdx.y * a.hpb + wave % a.hpb;
  const bool active = sub < a.wph && h_own < L.h;
  const int h = active ? h_own : 0;
  // ---- the basis rows and the query, before anything waits for the length
  hvec_t bw[NT][NK];
  half8_t qhh[NT], qll[NP];                      // (qh, qh) of each tile, (ql, ql') of each tile pair
  RawQ4 qx[NT];
  if (a.max_packed_len > 0) {
    const uint16_t* basis = a.r.basis + (int64_t)b * a.r.basis_stride;
    auto row = [&](int rt) {
      return basis + (int64_t)(h * D + (n >> 2) * RUN + 4 * (rt % NP) + (n & 3) + (rt / NP) * (D / 2)) * R + KQ * qd;
    };
    if ((reinterpret_cast<uintptr_t>(basis) & 15) == 0) {
#pragma unroll
      for (int rt = 0; rt < NT; ++rt)
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) bw[rt][ks] = *reinterpret_cast<const hvec_t*>(row(rt) + 4 * KQ * ks);
    } else {
#pragma unroll
      for (int rt = 0; rt < NT; ++rt)
#pragma unroll
        for (int ks = 0; ks < NK; ++ks)
#pragma unroll
          for (int i = 0; i < KQ; ++i) bw[rt][ks][i] = __builtin_bit_cast(_Float16, row(rt)[4 * KQ * ks + i]);
    }
    const int64_t qrow = (((int64_t)b * L.h + h) * G + (n < G ? n : 0)) * D;
    load_q4(a.q, a.io_dtype, [&](int rt) { return qrow + RUN * qd + 4 * (rt % NP) + (rt / NP) * (D / 2); }, qx);
  }
  // the workgroup's quads, first of the host's bound of the length (so that the
  // first pages are requested without a wait for the device length)
  int n_pages, q0, q1;
  auto set_range = [&](int len) {
    n_pages = len / kPT;
    const int n_quads = (n_pages + kGenQuad - 1) / kGenQuad;
    if (a.div32) {   // every product fits 32 bits
      q0 = (int)((uint32_t)split * (uint32_t)n_quads / (uint32_t)a.n_split);
      q1 = (int)(((uint32_t)split + 1u) * (uint32_t)n_quads / (uint32_t)a.n_split);
    } else {
      q0 = (int)((int64_t)split * n_quads / a.n_split);
      q1 = (int)((int64_t)(split + 1) * n_quads / a.n_split);
    }
    q0 = __builtin_amdgcn_readfirstlane(q0);
    q1 = __builtin_amdgcn_readfirstlane(q1);
  };
  set_range(a.max_packed_len);

  // ---- page ids, 64 from an 8-page boundary at or before the wave's next quad
  // (a residual group of up to 128 tokens lies within 8 pages)
  int id_base = 0, idv = 0;
  auto load_ids = [&](int quad) {
    id_base = (kGenQuad * quad) & ~7;
    const int p = min(id_base + lane, max(a.r.max_pages - 1, 0));
    idv = a.r.page_table ? a.r.page_table[(int64_t)b * a.r.max_pages + p] : (b + a.b0) * a.r.max_pages + p;
    idv = (int)clamp_page(idv, a.r.n_pool);
  };
  auto page_of = [&](int p) -> const uint8_t* {   // uniform p
    return a.r.pages + (int64_t)__builtin_amdgcn_readlane(idv, p - id_base) * L.bytes;
  };
  auto page_of_lane = [&](int p) -> const uint8_t* {   // p per lane
    return a.r.pages + (int64_t)__shfl(idv, p - id_base) * L.bytes;
  };
  // ---- the lane's scales: channels h d + RUN qd .. and + d/2, in the page
  // slot of the residual group that holds them
  const int c_lo = h * D + RUN * qd, c_hi = c_lo + D / 2;
  const int slot_lo = (int)(((float)c_lo + 0.5f) * a.inv_per_slot), slot_hi = (int)(((float)c_hi + 0.5f) * a.inv_per_slot);
  const int off_lo = L.kscale + 2 * (c_lo - slot_lo * L.per_slot), off_hi = L.kscale + 2 * (c_hi - slot_hi * L.per_slot);
  const int kres_off = L.kres + (h * kPT + n) * (D / 2) + (RUN / 2) * qd, vcode_off = L.vcode + (h * 4 + qd) * D + NT * n;
  struct Key {
    hvec_t us[NK];
    GenBytes<RUN / 2> lo, hi;
    GenBytes<2 * RUN < 16 ? 2 * RUN : 16> slo[(2 * RUN + 15) / 16], shi[(2 * RUN + 15) / 16];
  };
  Key key[PF];
  GenBytes<NT> vc[kGenQuad];
  half4_t vn[NCR];
  auto last_page = [&](int p) { return min(p, n_pages - 1); };
  auto load_key = [&](Key& k, int p_any) {
    const int p = last_page(p_any), p0 = p & ~(L.slots - 1);
    const uint8_t* pg = page_of(p);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
      k.us[ks] = *reinterpret_cast<const hvec_t*>(pg + L.us + (n * R + 4 * KQ * ks + KQ * qd) * 2);
    k.lo.load(pg + kres_off);
    k.hi.load(pg + kres_off + D / 4);
    const uint8_t* gl = page_of_lane(p0 + slot_lo) + off_lo;
    const uint8_t* gh = page_of_lane(p0 + slot_hi) + off_hi;
#pragma unroll
    for (int i = 0; i < (2 * RUN + 15) / 16; ++i) {
      k.slo[i].load(gl + 16 * i);
      k.shi[i].load(gh + 16 * i);
    }
  };
  const int my_slot = NSLOT > 1 ? n / SW : 0;   // page slot of this lane after compaction
  auto load_values = [&](int quad) {
#pragma unroll
    for (int pp = 0; pp < kGenQuad; ++pp) vc[pp].load(page_of(last_page(kGenQuad * quad + pp)) + vcode_off);
#pragma unroll
    for (int r = 0; r < NCR; ++r)
      vn[r] = *reinterpret_cast<const half4_t*>(page_of_lane(last_page(kGenQuad * quad + r * NSLOT + my_slot)) +
                                                L.vnorm + (h * kPT + 4 * qd) * 2);
  };

  // ---- the wave's first quad in flight
  int qi;                                        // the wave's quads: q0 + sub, + wph, ...
  auto load_first = [&]() {
    qi = q0 + sub;
    if (active && qi < q1) {
      load_ids(qi);
#pragma unroll
      for (int i = 0; i < PF; ++i) load_key(key[i], kGenQuad * qi + i);
      load_values(qi);
    }
  };
  load_first();
  for (int i = tid; i < 256; i += 64 * NWV) {
    uint32_t hi[2] = {0u, 0u}, lo[2] = {0u, 0u};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float x = level4((i >> (2 * t)) & 3, a.r.level[0], a.r.level[1], a.r.level[2], a.r.level[3]);
      const _Float16 xh = (_Float16)x;
      hi[t >> 1] |= half_bits(xh) << (16 * (t & 1));
      lo[t >> 1] |= half_bits((_Float16)(x - (float)xh)) << (16 * (t & 1));
    }
    s_lvh[i] = make_uint4(hi[0], hi[1], hi[0], hi[1]);
    s_lvl[i] = make_uint2(lo[0], lo[1]);
  }
  {
    const float sc = n < G ? a.qscale : 0.f;
    float4_t qf[NT];
    cvt_q4(qx, a.io_dtype, qf);
#pragma unroll
    for (int rt = 0; rt < NT; ++rt) {
      const float4_t x = qf[rt] * sc;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const _Float16 xh = (_Float16)x[e];
        qhh[rt][e] = qhh[rt][4 + e] = xh;
        qll[rt % NP][4 * (rt / NP) + e] = (_Float16)(x[e] - (float)xh);
      }
    }
  }
  float4_t acc[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) acc[ct] = float4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;          // l_run: the weights' sum, relative to 2^m_run
  float z_run = -INFINITY, up = 0.f;             // acc: relative to 2^(z_run - kGenUp); up = 2^(m_run - z_run + kGenUp)
  const int len = __builtin_amdgcn_readfirstlane(min(max(len_raw, 0), a.max_packed_len));
  if (len != a.max_packed_len) {                 // a shorter sequence: its own quads
    set_range(len);
    load_first();
  }
  // nibble e of a half word: its mask, the exponent field of 2^(23 - 4e) and
  // that power plus the codes' offset (in registers: one AND-OR a code)
  uint32_t nib_m[4], nib_e[4];
  float nib_b[4], m1 = -1.0f, zero = -0.0f;   // m1, zero: see gen_split2
  asm volatile("" : "+s"(m1), "+s"(zero));
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    nib_m[e] = 15u << (4 * e);
    nib_e[e] = 0x4B000000u - (0x02000000u * e);
    nib_b[e] = (float)((8388608 >> (4 * e)) + (1 << (L.bits - 1)));
    asm volatile("" : "+v"(nib_m[e]));
    asm volatile("" : "+s"(nib_e[e]));
  }

  for (int qt = q0; qt < q1; qt += kGenTables) {
    const int nt = min(kGenTables, q1 - qt);
    if (qt != q0) __syncthreads();               // every wave is done with the previous tables
    // (cos, sin) of HF's fp32 angle fl(pos * inv_freq) from its fraction of a
    // revolution (the product scaled by 1/2pi in double, its fraction rounded
    // to fp32) and the hardware sin/cos of revolutions, ~1e-6 absolute, times
    // rope_scaling, rounded to fp16: the reference's shared tables
    {
      const int j = tid & (D / 2 - 1);
      for (int p = tid / (D / 2); p < 64 * nt; p += 64 * NWV / (D / 2)) {
        const float ang = (float)(64 * qt + p) * freq;
        const double rev = (double)ang * 0.15915494309189535;
        const float fr = (float)(rev - floor(rev));
        const half2_t v = {(_Float16)fp32_rounded(__builtin_amdgcn_cosf(fr) * a.r.rope_scaling),
                           (_Float16)fp32_rounded(__builtin_amdgcn_sinf(fr) * a.r.rope_scaling)};
        s_cs[p * CSROW + j] = as_u32(v);
      }
    }
    __syncthreads();
    if (!active) continue;
    for (; qi < qt + nt; qi += a.wph) {
      const int qn = qi + a.wph;                 // the wave's next quad
      const bool more = qn < q1;
      const int p0 = kGenQuad * qi;
      float4_t st[kGenQuad];
#pragma unroll
      for (int pp = 0; pp < kGenQuad; ++pp) {
        Key& k = key[pp % PF];
        float4_t kt[NT];
        const float4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
          kt[rt] = z;
#pragma unroll
          for (int ks = 0; ks < NK; ++ks) {
            if constexpr (R >= 32) kt[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bw[rt][ks], k.us[ks], kt[rt], 0, 0, 0);
            else kt[rt] = __builtin_amdgcn_mfma_f32_16x16x16f16(bw[rt][ks], k.us[ks], kt[rt], 0, 0, 0);
          }
        }
        // residual code times scale: the nibble at bit 4k of a half word under
        // the exponent of 2^(23 - 4k) reads as 2^(23 - 4k) + code, exactly
#pragma unroll
        for (int rt = 0; rt < NT; ++rt)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * (rt % NP) + e;     // position in the run
            const uint32_t w = rt < NP ? k.lo.w[i / 8] : k.hi.w[i / 8];
            const uint32_t sw = rt < NP ? k.slo[i / 8].w[(i % 8) / 2] : k.shi[i / 8].w[(i % 8) / 2];
            const float c = __uint_as_float(((i % 8 < 4 ? w : w >> 16) & nib_m[e]) | nib_e[e]) - nib_b[e];
            kt[rt][e] = __builtin_fmaf((float)as_h2(sw)[i & 1], c, kt[rt][e]);
          }
        // RoPE and the high and low parts, a tile pair at a time
        const uint32_t* cs = s_cs + ((qi - qt) * 64 + pp * kPT + n) * CSROW + RUN * qd;
        float4_t s = z;
#pragma unroll
        for (int rt = 0; rt < NP; ++rt) {
          const uint4 cv = *reinterpret_cast<const uint4*>(cs + 4 * rt);
          const uint32_t cw[4] = {cv.x, cv.y, cv.z, cv.w};
          float xr[4], yr[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const half2_t c2 = as_h2(cw[e]);
            const float x = kt[rt][e], y = kt[rt + NP][e];
            xr[e] = __builtin_fmaf(-y, (float)c2[1], __builtin_fmaf(x, (float)c2[0], zero));
            yr[e] = __builtin_fmaf(x, (float)c2[1], __builtin_fmaf(y, (float)c2[0], zero));
          }
          union { uint32_t w[4]; half8_t v; } kx, ky, kh;
          gen_split2(xr[0], xr[1], m1, kx.w[0], kx.w[2]);
          gen_split2(xr[2], xr[3], m1, kx.w[1], kx.w[3]);
          gen_split2(yr[0], yr[1], m1, ky.w[0], ky.w[2]);
          gen_split2(yr[2], yr[3], m1, ky.w[1], ky.w[3]);
          kh.w[0] = kx.w[0]; kh.w[1] = kx.w[1]; kh.w[2] = ky.w[0]; kh.w[3] = ky.w[1];
          s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kx.v, qhh[rt], s, 0, 0, 0);
          s = __builtin_amdgcn_mfma_f32_16x16x32_f16(ky.v, qhh[rt + NP], s, 0, 0, 0);
          s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh.v, qll[rt], s, 0, 0, 0);
        }
        if (p0 + pp >= n_pages) s = float4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        st[pp] = s;
        // the page's registers take the page PF further on
        const int quad_n = pp + PF < kGenQuad ? qi : qn, p_n = kGenQuad * quad_n + (pp + PF) % kGenQuad;
        if (quad_n == qi || more) {
          if (quad_n != qi && kGenQuad * qn + kGenQuad > id_base + kGenIds) load_ids(qn);
          load_key(k, p_n);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // ---- compaction: page r NSLOT + s to columns [s SW, (s + 1) SW)
      float4_t cr[NCR];
#pragma unroll
      for (int r = 0; r < NCR; ++r) {
        cr[r] = st[r * NSLOT];
        if constexpr (NSLOT == 4) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            cr[r][i] = dpp<kRowShr + 4, 0x2>(cr[r][i], st[r * NSLOT + 1][i]);
            cr[r][i] = dpp<kRowShr + 8, 0x4>(cr[r][i], st[r * NSLOT + 2][i]);
            cr[r][i] = dpp<kRowShr + 12, 0x8>(cr[r][i], st[r * NSLOT + 3][i]);
          }
        } else if constexpr (NSLOT == 2) {
#pragma unroll
          for (int i = 0; i < 4; ++i) cr[r][i] = dpp<kRowShr + 8, 0xC>(cr[r][i], st[r * NSLOT + 1][i]);
        }
      }
      // ---- online softmax (two running maxima per query, sums rescaled only when
      // one of them grows); z_run stays within 64 of m_run where every norm is 0
      float mx = -INFINITY;
      half4_t vm = vn[0];
#pragma unroll
      for (int r = 0; r < NCR; ++r) {
        mx = fmaxf(mx, fmaxf(fmaxf(cr[r][0], cr[r][1]), fmaxf(cr[r][2], cr[r][3])));
        vm = __builtin_elementwise_max(vm, vn[r]);
      }
      const half2_t vm2 = __builtin_elementwise_max(half2_t{vm[0], vm[1]}, half2_t{vm[2], vm[3]});
      const float mz = mx + __builtin_amdgcn_logf(fmaxf((float)vm2[0], (float)vm2[1]));
      if (__any(mx > m_run || mz > z_run)) {
        auto of_query = [](float x) {
          if constexpr (NSLOT == 4) x = fmaxf(x, dpp_row<kRowRor + 4>(x));
          if constexpr (NSLOT >= 2) x = fmaxf(x, dpp_row<kRowRor + 8>(x));
          x = fmaxf(x, __shfl_xor(x, 16));
          return ceilf(fmaxf(x, __shfl_xor(x, 32)));
        };
        const float m_new = fmaxf(m_run, of_query(mx));
        const float z_new = fmaxf(fmaxf(z_run, of_query(mz)), m_new - 64.f);
        const float beta = __builtin_amdgcn_exp2f(z_run - z_new);
        l_run *= __builtin_amdgcn_exp2f(m_run - m_new);
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) acc[ct] *= beta;
        m_run = m_new;
        z_run = z_new;
        up = __builtin_amdgcn_exp2f(m_run - z_run + kGenUp);
      }
      uint2 ph[NCR], pl[NCR];
#pragma unroll
      for (int r = 0; r < NCR; ++r) {
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(cr[r][i] - m_run);
          l_run += p;
          x[i] = p * ((float)vn[r][i] * up);
        }
        gen_split2(x[0], x[1], m1, ph[r].x, pl[r].x);
        gen_split2(x[2], x[3], m1, ph[r].y, pl[r].y);
      }
      // ---- V^T P^T, two pages at a time
#pragma unroll
      for (int u = 0; u < kGenQuad / 2; ++u) {
        const int pa = 2 * u, pb = 2 * u + 1;
        const bool on_a = NSLOT == 1 || my_slot == pa % NSLOT, on_b = NSLOT == 1 || my_slot == pb % NSLOT;
        const uint2 z2 = make_uint2(0u, 0u);
        const uint2 ha = on_a ? ph[pa / NSLOT] : z2, la = on_a ? pl[pa / NSLOT] : z2;
        const uint2 hb = on_b ? ph[pb / NSLOT] : z2, lb = on_b ? pl[pb / NSLOT] : z2;
        union U { uint4 e; half8_t v; };
        U ba, bb, bl;
        ba.e = make_uint4(ha.x, ha.y, la.x, la.y);
        bb.e = make_uint4(hb.x, hb.y, lb.x, lb.y);
        bl.e = make_uint4(ha.x, ha.y, hb.x, hb.y);
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) {
          const uint32_t ia = (vc[pa].w[ct / 4] >> (8 * (ct % 4))) & 0xFFu;
          const uint32_t ib = (vc[pb].w[ct / 4] >> (8 * (ct % 4))) & 0xFFu;
          U ua, ub, ul;
          ua.e = s_lvh[ia];
          ub.e = s_lvh[ib];
          const uint2 xa = s_lvl[ia], xb = s_lvl[ib];
          ul.e = make_uint4(xa.x, xa.y, xb.x, xb.y);
          acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ua.v, ba.v, acc[ct], 0, 0, 0);
          acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ub.v, bb.v, acc[ct], 0, 0, 0);
          acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ul.v, bl.v, acc[ct], 0, 0, 0);
        }
      }
      if (more) load_values(qn);
    }
  }

  if (a.win_wgs == 0) window(split, a.n_split);
  if (!active) return;
  // ---- fold the page slots, then the inverse Hadamard of channel
  // (4qd + e) NT + ct: ct and e in registers, qd across the rows; signs, 1/d
  if constexpr (NSLOT == 4) {
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[ct][i] += dpp_row<kRowRor + 4>(acc[ct][i]);
    l_run += dpp_row<kRowRor + 4>(l_run);
  }
  if constexpr (NSLOT >= 2) {
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[ct][i] += dpp_row<kRowRor + 8>(acc[ct][i]);
    l_run += dpp_row<kRowRor + 8>(l_run);
  }
  l_run += __shfl_xor(l_run, 16);
  l_run += __shfl_xor(l_run, 32);
#pragma unroll
  for (int hb = 1; hb < NT; hb <<= 1)
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
      if (!(ct & hb)) {
        const float4_t u = acc[ct], w = acc[ct | hb];
        acc[ct] = u + w;
        acc[ct | hb] = u - w;
      }
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
#pragma unroll
    for (int hb = 1; hb < 4; hb <<= 1)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!(e & hb)) {
          const float u = acc[ct][e], w = acc[ct][e | hb];
          acc[ct][e] = u + w;
          acc[ct][e | hb] = u - w;
        }
#pragma unroll
    for (int rb = 1; rb < 4; rb <<= 1)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float o = __shfl_xor(acc[ct][e], 16 * rb);
        acc[ct][e] = (qd & rb) ? o - acc[ct][e] : acc[ct][e] + o;
      }
  }
  if (n >= G) return;
  const float inv = l_run > 0.f ? __builtin_amdgcn_exp2f(z_run - m_run - kGenUp) / ((float)D * l_run) : 0.f;
  const int S = a.n_split * a.wph, slot = split * a.wph + sub;
  const int64_t row = ((int64_t)b * L.h + h) * G + n;
  float* rec = a.ws_acc + row * D * S + slot * 16;   // chunk k at + 16 k S
#pragma unroll
  for (int i = 0; i < D / 4; i += 4) {               // channels qd d/4 + i .. + 3
    float4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = acc[(i + e) % NT][(i + e) / NT] * inv;
    const int c = qd * (D / 4) + i;
    const uint32_t sg = a.r.v_sign_bits[c >> 5] >> (c & 31);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (sg >> e) & 1u ? -o[e] : o[e];
    *reinterpret_cast<float4_t*>(rec + (int64_t)(c >> 4) * 16 * S + (c & 15)) = o;
  }
  if (qd == 0) *reinterpret_cast<float2*>(a.ws_ml + (row * S + slot) * 2) = make_float2(m_run, l_run);
}

// Dense keys and values of committed pages: grid (pages, h_kv), block 64.
struct GenDequantArgs {
  GenReadArgs r;
  int apply_rope, pos0, out_dtype;
  int64_t out_rows;
  void* k_out;
  void* v_out;
};

template <int D, int R>
__global__ __launch_bounds__(64) void gen_dequant_kernel(const GenDequantArgs a) {
  constexpr int NT = D / 16, LDB = R + 4;
  const int p = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, n = lane & 15, qd = lane >> 4;
  const GenLayout& L = a.r.L;
  __shared__ __align__(16) uint16_t s_B[D * LDB];
  __shared__ float s_v[kPT][D + 1];
  const uint16_t* basis = a.r.basis + (int64_t)(h * D) * R;
  for (int e = lane; e < D * R; e += 64) s_B[(e / R) * LDB + e % R] = basis[e];
  __syncthreads();
  const uint8_t* pg = gen_read_page(a.r, 0, p);
  float4_t kt[NT];
  gen_keys<D, R>(a.r, pg, s_B, 0, p, h, n, qd, kt);
  if (a.apply_rope) gen_rope<D>(a.r, kt, a.pos0 + p * kPT + n, qd, a.apply_rope);
  const int64_t krow = ((int64_t)h * a.out_rows + p * kPT + n) * D;
#pragma unroll
  for (int rt = 0; rt < NT; ++rt)
#pragma unroll
    for (int e = 0; e < 4; ++e) store_elem(a.k_out, krow + 16 * rt + 4 * qd + e, kt[rt][e], a.out_dtype);
  // values: fwht(level / sqrt(d)) * signs * norm, per token
  const float sqrt_d = __builtin_sqrtf((float)D);
  for (int e = lane; e < kPT * D; e += 64) {
    const int t = e / D, c = e % D;
    const uint32_t code = (pg[L.vcode + (h * 4 + t / 4) * D + c] >> (2 * (t % 4))) & 3u;
    s_v[t][c] = a.r.level[code] / sqrt_d;
  }
  __syncthreads();
  for (int hb = 1; hb < D; hb <<= 1) {
    for (int e = lane; e < kPT * D / 2; e += 64) {
      const int t = e / (D / 2), i = e % (D / 2), i0 = (i / hb) * 2 * hb + (i % hb);
      const float u = s_v[t][i0], v = s_v[t][i0 + hb];
      s_v[t][i0] = u + v;
      s_v[t][i0 + hb] = u - v;
    }
    __syncthreads();
  }
  for (int e = lane; e < kPT * D; e += 64) {
    const int t = e / D, c = e % D;
    float v = s_v[t][c] / sqrt_d;
    if (sign_neg(a.r.v_sign_bits, c)) v = -v;
    v = v * half_bits_to_float(*reinterpret_cast<const uint16_t*>(pg + L.vnorm + (h * kPT + t) * 2));
    store_elem(a.v_out, ((int64_t)h * a.out_rows + p * kPT + t) * D + c, v, a.out_dtype);
  }
}

}  // namespace bmx

// ---------------------------------------------------------------------------
// Host side: argument checks, launches.
// ---------------------------------------------------------------------------
using namespace bmx;

static int gfail(int code, const std::string& msg) {
  bmx_set_error(msg);
  return code;
}

namespace {

// the (d, R) instance of a kernel template: d in {32, 64, 128}, R in {16, 32, 64, 128}
#define BMX_GEN_DISPATCH(D_, R_, CALL)                                    \
  switch ((D_) * 1000 + (R_)) {                                          \
    case 32016: CALL(32, 16); break;  case 32032: CALL(32, 32); break;    \
    case 32064: CALL(32, 64); break;  case 32128: CALL(32, 128); break;   \
    case 64016: CALL(64, 16); break;  case 64032: CALL(64, 32); break;    \
    case 64064: CALL(64, 64); break;  case 64128: CALL(64, 128); break;   \
    case 128016: CALL(128, 16); break; case 128032: CALL(128, 32); break; \
    case 128064: CALL(128, 64); break; case 128128: CALL(128, 128); break; \
    default: break;                                                      \
  }

void fill_read(GenReadArgs& r, const Geo& g) {
  r.L = GenLayout::of(g);
}

// The decode grid of a sequence: n_split workgroups (its 4-page quads dealt
// evenly) x head blocks of hpb heads, wph waves per head.  One workgroup per CU
// over the batch, or as many as split_tokens asks for; a wave per head, or several
// where there are fewer heads than waves, each with its own partial slot.  A range
// of fewer splits than CUs spreads its heads over more blocks (a wave alone on its
// SIMD takes a quad in about half the time), and where CUs are still idle the
// window's pairs get workgroups of their own (d 64, 2,048 tokens and a 128-row
// window: 17.1 us a call with neither, 15.8 with the window apart, 12.6 with both),
// 4 pairs each if there is room, unless a wave would have more of them there than
// behind the quads.
// With split_tokens 512 and the heads of 2,048 tokens (d 64, rank 32, h_kv 8, G 4) on
// one workgroup a split 48.9 us, spread 19.5.  The sequences are launched `chunk`
// at a time, so that the workspace stays within kGenWorkspace whatever the batch;
// one sequence needs 12.8 MB at most (16 heads x 16 queries, d 128, a 4,096-row
// window), unless split_tokens asks for more splits than fit: it gets those that do.
constexpr size_t kGenWorkspace = 24u << 20;

struct GenPlan {
  int chunk, n_split, hpb, blocks, wph, win_wgs;
  size_t bytes;
  int slots() const { return n_split * wph; }
};

GenPlan gen_plan(const bmx_k2b_decode_args* a, const Geo& g) {
  GenPlan p;
  const int nw = gen_waves(g.d, g.R), cus = bmx_device_cu_count();
  const int quads = std::max(1, (a->max_packed_len / kPT + kGenQuad - 1) / kGenQuad);
  // at most so many splits (with split_tokens: exactly)
  const int most = a->split_tokens > 0
                       ? std::max(1, std::min(quads, (a->max_packed_len + a->split_tokens - 1) / a->split_tokens))
                       : quads;
  // the window's bound: a bound call's plan holds at any length
  const int pairs = (a->tail_cap + 15) / 16 * g.h;
  p.chunk = a->batch;
  for (;; p.chunk = (p.chunk + 1) / 2) {
    p.blocks = (g.h + nw - 1) / nw;
    const int win_most = a->split_tokens > 0 ? 0 : (pairs + nw - 1) / nw;   // room kept for the window
    while (2 * p.blocks <= g.h && (int64_t)p.chunk * (2 * p.blocks * (int64_t)most + win_most) <= cus)
      p.blocks *= 2;
    p.hpb = (g.h + p.blocks - 1) / p.blocks;
    const int per_seq = cus / (p.chunk * p.blocks);
    p.n_split = a->split_tokens > 0 ? most : std::max(1, std::min(per_seq, most));
    p.wph = std::max(1, std::min(nw / p.hpb, (quads + p.n_split - 1) / p.n_split));
    if (p.chunk == 1) {
      const int fit = ((int)(kGenWorkspace / (sizeof(float) * g.h * g.G)) - a->tail_cap) / (g.d + 2);   // >= 157
      if (p.slots() > fit) {
        p.wph = 1;
        p.n_split = std::min(p.n_split, fit);
      }
    }
    p.win_wgs = std::max(0, std::min(per_seq - p.n_split, (pairs + 4 * p.blocks - 1) / (4 * p.blocks)));
    auto rounds = [&](int wgs) { return (pairs + wgs * p.blocks * nw - 1) / (wgs * p.blocks * nw); };
    if (p.win_wgs > 0 && rounds(p.win_wgs) > rounds(p.n_split)) p.win_wgs = 0;
    p.bytes = (size_t)p.chunk * g.h * g.G * ((size_t)p.slots() * (g.d + 2) + a->tail_cap) * sizeof(float);
    if (p.chunk == 1 || p.bytes <= kGenWorkspace) return p;
  }
}

}  // namespace

namespace bmx {

size_t gen_decode_workspace(const bmx_k2b_decode_args* a) { return gen_plan(a, Geo::from(a->geom)).bytes; }

std::string gen_decode_check(const bmx_k2b_decode_args* a) {
  const Geo g = Geo::from(a->geom);
  const std::string why = g.check();
  if (!why.empty()) return why;
  if (g.G < 1 || g.G > 16) return "n_q_groups must be 1..16";
  if (a->max_packed_len % g.group != 0) return "max_packed_len must be a multiple of k_group";
  return "";
}

template <int D, int R>
static hipError_t gen_launch_split(const GenDecodeArgs& k, dim3 grid, hipStream_t st) {
  auto go = [&](auto sw) {
    constexpr int SW = decltype(sw)::value;
    const hipError_t e = bmx_ensure_dynamic_lds((const void*)gen_split_kernel<D, R, SW>, gen_lds<D>());
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((gen_split_kernel<D, R, SW>), grid, dim3(64 * gen_waves(D, R)), gen_lds<D>(), st, k);
    return hipGetLastError();
  };
  if (k.G <= 4) return go(std::integral_constant<int, 4>{});
  if (k.G <= 8) return go(std::integral_constant<int, 8>{});
  return go(std::integral_constant<int, 16>{});
}

int gen_decode(const bmx_k2b_decode_args* a, hipStream_t st, void* ws, size_t ws_cap, const std::string& name) {
  const Geo g = Geo::from(a->geom);
  const GenPlan p = gen_plan(a, g);
  if (!ws || ws_cap < p.bytes)
    return gfail(BMX_E_WORKSPACE, name + ": workspace missing or smaller than bmx_k2b_decode_workspace_bytes()");
  GenDecodeArgs k{};
  fill_read(k.r, g);
  k.r.pages = a->pages; k.r.max_pages = a->max_pages;
  k.r.n_pool = a->n_pool_pages > 0 ? a->n_pool_pages : 1;
  k.r.basis_stride = a->basis_stride;
  for (int j = 0; j < 64; ++j) k.r.inv_freq[j] = a->inv_freq[j];
  k.r.rope_scaling = a->rope_scaling;
  for (int j = 0; j < 4; ++j) { k.r.level[j] = a->codebook[j]; k.r.v_sign_bits[j] = a->v_sign_bits[j]; }
  k.G = g.G; k.n_split = p.n_split; k.hpb = p.hpb; k.wph = p.wph;
  k.win_tiles = ((a->tail_len ? a->tail_cap : a->tail_len_value) + 15) / 16;
  k.win_wgs = p.win_wgs;
  k.div32 = ((uint64_t)p.n_split + 1) * (a->max_packed_len / 64 + 1) < (1ull << 32);
  k.inv_per_slot = 1.0f / (float)k.r.L.per_slot;
  k.io_dtype = a->io_dtype;
  k.max_packed_len = a->max_packed_len;
  k.qscale = a->sm_scale * 1.4426950408889634f;
  const int hg = g.h * g.G;
  const size_t recs = (size_t)p.chunk * hg * p.slots();
  k.ws_acc = (float*)ws;
  k.ws_ml = k.ws_acc + recs * g.d;
  k.ws_win = k.ws_ml + recs * 2;
  k.ts_b = a->tail_stride_b; k.ts_h = a->tail_stride_h; k.ts_t = a->tail_stride_t;
  k.tail_cap = a->tail_cap; k.tail_bf16 = a->tail_dtype == BMX_K2B_TAIL_BF16;
  k.nw.sb = a->new_stride_b; k.nw.sh = a->new_stride_h; k.nw.st = a->new_stride_t;
  k.nw.n = a->n_new;
  k.nw.T = a->tail_len ? -1 : a->tail_len_value;
  CombineKArgs c{};
  c.h_kv = g.h; c.G = g.G; c.max_splits = p.slots(); c.tail_cap = a->tail_cap;
  c.io_dtype = a->io_dtype;
  c.ws_acc = k.ws_acc; c.ws_ml = k.ws_ml; c.ws_win = k.ws_win;
  c.ts_b = k.ts_b; c.ts_h = k.ts_h; c.ts_t = k.ts_t; c.tail_bf16 = k.tail_bf16;
  c.packed_scale = 1.0f;
  c.max_packed_len = a->max_packed_len;
  const int64_t io_bytes = a->io_dtype == BMX_K2B_IO_F32 ? 4 : 2;
  for (int b0 = 0; b0 < a->batch; b0 += p.chunk) {
    const int nb = std::min(p.chunk, a->batch - b0);
    auto at = [&](const uint16_t* x, int64_t stride) { return x ? x + b0 * stride : nullptr; };
    k.b0 = b0;
    k.r.page_table = a->page_table ? a->page_table + (int64_t)b0 * a->max_pages : nullptr;
    k.r.basis = at(a->basis, a->basis_stride);
    k.q = (const char*)a->q + b0 * (int64_t)hg * g.d * io_bytes;
    c.out = (char*)a->out + b0 * (int64_t)hg * g.d * io_bytes;
    k.packed_len = c.packed_len = a->packed_len + b0;
    k.k_tail = at(a->k_tail, a->tail_stride_b);
    c.v_tail = at(a->v_tail, a->tail_stride_b);
    c.tail_len = a->tail_len ? a->tail_len + b0 : nullptr;
    k.nw.k = at(a->new_k, a->new_stride_b);
    k.nw.v = at(a->new_v, a->new_stride_b);
    k.nw.k_dst = const_cast<uint16_t*>(k.k_tail);
    k.nw.v_dst = const_cast<uint16_t*>(c.v_tail);
    c.nw = k.nw;
    const dim3 grid(p.n_split + p.win_wgs, p.blocks, nb);
    hipError_t e = hipSuccess;
#define BMX_GEN_SPLIT(D_, R_) e = gen_launch_split<D_, R_>(k, grid, st)
    BMX_GEN_DISPATCH(g.d, g.R, BMX_GEN_SPLIT)
#undef BMX_GEN_SPLIT
    if (e != hipSuccess) return gfail(BMX_E_HIP, name + ": split kernel launch: " + hipGetErrorString(e));
    if (a->split_end_event) {
      e = hipEventRecord((hipEvent_t)a->split_end_event, st);
      if (e != hipSuccess) return gfail(BMX_E_HIP, name + ": hipEventRecord: " + hipGetErrorString(e));
    }
    if (g.d == 32) launch_combine<false, 32, float>(c, hg, nb, st);
    else if (g.d == 64) launch_combine<false, 64, float>(c, hg, nb, st);
    else launch_combine<false, 128, float>(c, hg, nb, st);
    e = hipGetLastError();
    if (e != hipSuccess) return gfail(BMX_E_HIP, name + ": merge kernel launch: " + hipGetErrorString(e));
  }
  return BMX_OK;
}

int gen_dequant(const bmx_k2b_dequant_args* a, hipStream_t st) {
  const Geo g = Geo::from(a->geom);
  const std::string why = g.check();
  if (!why.empty()) return gfail(BMX_E_INVALID, "bmx_k2b_dequant: " + why);
  if (a->n_tokens % g.group != 0)
    return gfail(BMX_E_INVALID, "bmx_k2b_dequant: n_tokens must be a multiple of k_group");
  GenDequantArgs k{};
  fill_read(k.r, g);
  k.r.pages = a->pages; k.r.page_table = a->page_table; k.r.max_pages = 0; k.r.n_pool = a->n_pool_pages;
  k.r.basis = a->basis; k.r.basis_stride = 0;
  for (int j = 0; j < 64; ++j) k.r.inv_freq[j] = a->inv_freq[j];
  k.r.rope_scaling = a->rope_scaling;
  for (int j = 0; j < 4; ++j) { k.r.level[j] = a->codebook[j]; k.r.v_sign_bits[j] = a->v_sign_bits[j]; }
  k.apply_rope = a->apply_rope; k.pos0 = a->pos0; k.out_dtype = a->out_dtype;
  k.out_rows = a->out_rows ? a->out_rows : a->n_tokens;
  k.k_out = a->k_out; k.v_out = a->v_out;
  const dim3 grid(a->n_tokens / kPT, g.h);
#define BMX_GEN_DQ(D_, R_) hipLaunchKernelGGL((gen_dequant_kernel<D_, R_>), grid, dim3(64), 0, st, k)
  BMX_GEN_DISPATCH(g.d, g.R, BMX_GEN_DQ)
#undef BMX_GEN_DQ
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gfail(BMX_E_HIP, std::string("bmx_k2b_dequant: launch: ") + hipGetErrorString(e));
  return BMX_OK;
}

}  // namespace bmx
