// Untied lm_head GEMV (gfx950): logits[b][j] = sum_k h[b][k] * W[row_j][k], f32, for a table W of
// V rows of H = 2048 in Q6_K (the shipped artifact's output.weight), Q8_0 or bf16, over all rows
// (dense) or a list of row ids (gather). This is prototype/lm_head/lm_head_kernels.h:474-512
// (lmh_dot_batch: one row's dot for up to LMH_MAX_BATCH = 8 hidden vectors) on the path
// lm_head.hip:51 launches, with the Q6_K width the prototype defers (prototype/lm_head/results.md:341-343).
//
// HBM-bound: every table byte is read once (bf16: once per 4 tokens), 1680 B per row in Q6_K (417 MB at
// V = 248320), 2176 B in Q8_0, 4096 B in bf16. Q6_K / Q8_0: the int8 kernel below, but
// for one token of a short list. Layout of the work of the others:
//   * one row per wave; each lane owns a fixed set of 32 element positions of every row, so its
//     slice of the hidden vectors (32 floats per token) stays in registers for the whole sweep;
//   * Q6_K / Q8_0 rows (2-byte-aligned blocks of 210 / 34 B) are staged into LDS by the block with
//     coalesced 16-byte loads, 8 rows per iteration, double buffered (the next iteration's loads
//     are in flight while the current rows are decoded); lanes then read their bytes from LDS as
//     aligned dwords and realign them with v_alignbyte;
//   * bf16 rows are read straight from HBM, 64 lanes x 16 B contiguous per load, two rows in
//     flight per wave.
// Arithmetic: the block's integer quants are accumulated against h (the quant as an exact small
// float), and the block scale multiplies the partial sum: sum_i h_i (s q_i) = s sum_i h_i q_i, a
// re-association of the reference's f32 dot, which the reference's own band covers
// (prototype/lm_head/gate.py:214-240: gamma_{2K-1} sum |h_k w_k| when products are inexact).
#include "common.h"
#include "lds_dma.h"
#include "moe_internal.h"

namespace moe {
namespace lmh {

constexpr int kH = 2048;                 // the lane mapping covers 64 lanes x 32 positions
constexpr int kThreads = 256;            // 4 waves
constexpr int kPad = 16;                 // LDS slack after the last row (the Q8_0 window overreads 6 B)
// Rows per wave per block iteration of the staged formats: small iterations (less LDS) let four blocks
// share a CU
constexpr int kRowsPerWave = 2, kRows = 4 * kRowsPerWave;

template <int FMT> struct Staged;
template <> struct Staged<MOE_FMT_Q6_K> {
  static constexpr int kRowB = kH / 256 * 210;                      // 1680
};
template <> struct Staged<MOE_FMT_Q8_0> {
  static constexpr int kRowB = kH / 32 * 34;                        // 2176
};

template <int XDT>
__device__ __forceinline__ float load_h(const void* h, size_t i) {
  if (XDT == MOE_DT_F32) return reinterpret_cast<const float*>(h)[i];
  return bf16_to_f32(reinterpret_cast<const uint16_t*>(h)[i]);
}

// byte b of v as a float (one v_cvt_f32_ubyteN)
__device__ __forceinline__ float cvt_b(uint32_t v, int b) { return (float)((v >> (8 * b)) & 0xFFu); }

// the table row of output j: j itself, or ids[j] (-1 when that id is outside [0, V))
template <int GATHER>
__device__ __forceinline__ long long row_of(const int32_t* ids, long long j, long long V) {
  if (!GATHER) return j;
  const int id = ids[j];
  return (id >= 0 && (long long)id < V) ? (long long)id : -1;
}

// Lane L's 32 positions: Q6_K: super-block sb = L >> 3, half g, 16-element run j and nibble
// parity k2 (element 128g + 32k + l of the super-block, k in {k2, k2 + 2}, l in [16j, 16j + 16):
// tools/gguf_reader.py:299-322 addresses it as ql[64g + 32(k & 1) + l] nibble k >> 1,
// qh[32g + l] bits 2k, sc[8g + 2k + (l >> 4)]); Q8_0: block L (elements 32L .. 32L + 31).
template <int FMT>
__device__ __forceinline__ int pos_of(int lane, int i) {
  if (FMT == MOE_FMT_Q6_K) {
    const int sb = lane >> 3, g = (lane >> 2) & 1, j = (lane >> 1) & 1, k2 = lane & 1;
    return 256 * sb + 128 * g + 32 * k2 + 16 * j + (i & 15) + ((i >> 4) << 6);
  }
  return 32 * lane + i;
}

template <int FMT, int XDT, int GATHER>
__global__ __launch_bounds__(kThreads) void k_lm_head_staged(const void* __restrict__ h,
                                                             const uint8_t* __restrict__ w,
                                                             long long V,
                                                             const int32_t* __restrict__ ids,
                                                             long long n_rows,
                                                             float* __restrict__ out) {
  constexpr int kRowB = Staged<FMT>::kRowB;
  constexpr int kChunks = kRowB / 16;                               // 105 / 136 per row
  constexpr int kBuf = kRows * kRowB + kPad;
  constexpr int kLoads = (kRows * kChunks + kThreads - 1) / kThreads;
  __shared__ __attribute__((aligned(16))) uint8_t smem[2][kBuf];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;

  // this lane's slice of the hidden vector, and its sums (the quant offsets below)
  float hv[32], hs[2] = {};
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    hv[i] = load_h<XDT>(h, pos_of<FMT>(lane, i));
    hs[(FMT == MOE_FMT_Q6_K) ? (i >> 4) : 0] += hv[i];
  }

  const long long n_it = (n_rows + kRows - 1) / kRows;
  uint4 reg[kLoads];
  long long it = blockIdx.x;
  auto load = [&](long long it_) {
    const long long r0 = it_ * kRows;
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
      const int c = t + kThreads * q;
      const int r = c / kChunks;
      reg[q] = make_uint4(0u, 0u, 0u, 0u);
      if (c < kRows * kChunks && r0 + r < n_rows) {
        const long long row = row_of<GATHER>(ids, r0 + r, V);
        if (row >= 0)
          reg[q] = *reinterpret_cast<const uint4*>(w + (size_t)row * kRowB + 16 * (c - r * kChunks));
      }
    }
  };
  auto stage = [&](uint8_t* buf) {
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
      const int c = t + kThreads * q;
      if (c < kRows * kChunks) *reinterpret_cast<uint4*>(buf + 16 * c) = reg[q];
    }
  };
  if (it < n_it) load(it);
  int cur = 0;
  for (; it < n_it; it += gridDim.x) {
    stage(smem[cur]);
    __syncthreads();
    if (it + gridDim.x < n_it) load(it + gridDim.x);
    const uint32_t* L32 = reinterpret_cast<const uint32_t*>(smem[cur]);
#pragma unroll 1
    for (int rr = 0; rr < kRowsPerWave; ++rr) {
      const int r = kRowsPerWave * wave + rr;
      const long long j = it * kRows + r;
      if (j >= n_rows) break;
      float part;
      if (FMT == MOE_FMT_Q6_K) {
        const int sb = lane >> 3, g = (lane >> 2) & 1, jj = (lane >> 1) & 1, k2 = lane & 1;
        const int sbb = r * kRowB + 210 * sb;                       // 2-byte aligned
        const int s = (sbb & 3) * 8;                                // bit shift 0 or 16
        const int oql = (sbb + 64 * g + 32 * k2 + 16 * jj) >> 2;    // dword index, same offset
        const int oqh = (sbb + 128 + 32 * g + 16 * jj) >> 2;
        uint32_t ql[5], qh[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) { ql[i] = L32[oql + i]; qh[i] = L32[oqh + i]; }
        const int osc = sbb + 192 + 8 * g + 2 * k2 + jj;
        const uint32_t sw0 = L32[osc >> 2], sw1 = L32[(osc >> 2) + 1];
        const int ssh = (osc & 3) * 8;
        const float sc_lo = (float)(int8_t)(sw0 >> ssh), sc_hi = (float)(int8_t)(sw1 >> ssh);
        const int od = sbb + 208;
        const float d = f16_to_f32((L32[od >> 2] >> ((od & 3) * 8)) & 0xFFFFu);
        float alo = 0.0f, ahi = 0.0f;
        const uint32_t shl = 4u - 2u * (uint32_t)k2, shr = 2u * (uint32_t)k2;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const uint32_t wq = __builtin_amdgcn_alignbyte(ql[m + 1], ql[m], s >> 3);
          const uint32_t wh = __builtin_amdgcn_alignbyte(qh[m + 1], qh[m], s >> 3);
          const uint32_t lo = (wq & 0x0F0F0F0Fu) | ((wh << shl) & 0x30303030u);
          const uint32_t hi = ((wq >> 4) & 0x0F0F0F0Fu) | ((wh >> shr) & 0x30303030u);
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) {
            const float ql_ = cvt_b(lo, bb), qh_ = cvt_b(hi, bb);
            alo = fmaf(hv[4 * m + bb], ql_, alo);
            ahi = fmaf(hv[16 + 4 * m + bb], qh_, ahi);
          }
        }
        const float dlo = d * sc_lo, dhi = d * sc_hi;               // exact (<= 19 bits)
        part = dlo * fmaf(-32.0f, hs[0], alo) + dhi * fmaf(-32.0f, hs[1], ahi);
      } else {
        const int off = r * kRowB + 34 * lane;                      // 2-byte aligned
        const int ow = off >> 2, s = off & 3;                       // s = 0 or 2
        uint32_t q[10];
#pragma unroll
        for (int i = 0; i < 10; ++i) q[i] = L32[ow + i];
        const float d = f16_to_f32((q[0] >> (8 * s)) & 0xFFFFu);
        const int qb = (s + 2) >> 2, qs = (s + 2) & 3;              // quants start at byte s + 2
        float a = 0.0f;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          const uint32_t lo_w = qb ? q[m + 1] : q[m], hi_w = qb ? q[m + 2] : q[m + 1];
          // int8 q + 128 as an unsigned byte: the sign bit flipped
          const uint32_t x = __builtin_amdgcn_alignbyte(hi_w, lo_w, qs) ^ 0x80808080u;
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) a = fmaf(hv[4 * m + bb], cvt_b(x, bb), a);
        }
        part = d * fmaf(-128.0f, hs[0], a);
      }
      const bool valid = row_of<GATHER>(ids, j, V) >= 0;
      const float v = wave_sum_f32(part);
      if (lane == 0) out[j] = valid ? v : __builtin_nanf("");
    }
    cur ^= 1;
  }
}

// ---- Q6_K / Q8_0 rows on the int8 matrix cores -----------------------------------
// The f32 dots above pay an FMA per element and token: from 2 tokens they no longer keep up with HBM, and
// more than four would take a second pass over the table. Here the hidden vectors are fixed-point numbers, four
// int8 digits of a token (30 bits under the largest of its 256-element slice) as MFMA rows beside the
// others', and the quants go into the MFMA as the bytes they are: the sums over a scale's 16 or 32 elements
// are exact integers, Q6_K's whole super-block (scales are integers too) as well. Only the final scaling and
// the sum over the eight super-blocks round: error against 64 bits (2-norm, standard normal f32 hidden
// vectors) 5.9e-8 in Q6_K, 7.6e-8 in Q8_0, where the f32 dots had 1.9e-7 and 3.1e-7.
// V = 248320, us, f32 dots -> now (1, 2, 4, 8 tokens): Q6_K 85, 120, 160, 312 -> 77, 80, 82, 118 (417 MB:
// 5.4 TB/s at 1); Q8_0 95, 111, 152, 300 -> 93, 94, 96, 113 (540 MB: 5.8 TB/s at 1). Up to four tokens
// HBM-bound; above, the second row group's MFMAs and scalings count. Short lists: the digits are a fixed
// 3 us (the rule for one token in launch_quant; two tokens, 64 rows: 6.8 -> 7.3 and 7.7 -> 6.2).
//   * block of 8 waves, persistent, 16 table rows an iteration; wave w owns elements 256 w .. of every row
//     (a Q6_K super-block, eight Q8_0 blocks); rows go straight to LDS, two buffers, one barrier;
//   * MFMA row 4 b + i is digit i of token b (row group r: tokens 4 r ..), so lane n + 16 g holds table row n's
//     four digit sums of token 4 r + g and combines them alone;
//   * the waves' f32 sums meet in LDS and are added in wave order an iteration later.
typedef int i32x4_t __attribute__((ext_vector_type(4)));

constexpr int kMW = 8;
constexpr int kMRows = 16;

template <int FMT> struct MStage {
  static constexpr int kRowB = Staged<FMT>::kRowB;
  // LDS row stride: 36 dwords past a multiple of the 64 banks, so 16 rows' dwords spread over them
  static constexpr int kStride = FMT == MOE_FMT_Q6_K ? kRowB : kRowB + 16;
  static constexpr int kPieces = (kMRows * kStride + 1023) / 1024;      // of 64 lanes x 16 bytes
  static constexpr int kBuf = 1024 * kPieces;
  static_assert(kMRows * kStride + 4 <= kBuf, "reads go up to a dword past the last row");
};

__device__ __forceinline__ i32x4_t mfma_i8(uint2 a, uint2 b) {
  return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(((uint64_t)a.y << 32) | a.x), (long)(((uint64_t)b.y << 32) | b.x),
                                               (i32x4_t){}, 0, 0, 0);
}
// over the lanes m, m + 16, m + 32, m + 48
__device__ __forceinline__ float max_g(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ int sum_g(int v) {
  const auto a = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
  v = (int)(a[0] + a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
  return (int)(b[0] + b[1]);
}
// the power of two that takes |x| <= mx to at most 127 (2^24 + 2^16 + 2^8 + 1), the largest four balanced int8
// digits hold: the exponent to 30, one less when mx's mantissa passes 2139062143 / 2^30
__device__ __forceinline__ int fix_up(float mx) {
  const uint32_t u = __float_as_uint(mx);
  const int e = max((int)(u >> 23), 1) - 127;
  return 30 - e - ((u & 0x7FFFFFu) > 0x7EFEFEu ? 1 : 0);
}
template <int XDT>
__device__ __forceinline__ void load_h4(const void* h, size_t i, float* v) {   // h is element aligned only
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = load_h<XDT>(h, i + k);
}

// R row groups of four tokens (B <= 4 R)
template <int FMT, int R, int XDT, int GATHER>
__global__ __launch_bounds__(64 * kMW, 4) void k_lm_head_i8(const void* __restrict__ h, int B,
                                                            const uint8_t* __restrict__ w, long long V,
                                                            const int32_t* __restrict__ ids, long long n_rows,
                                                            float* __restrict__ out) {
  using S = MStage<FMT>;
  constexpr bool Q6 = FMT == MOE_FMT_Q6_K;
  __shared__ __attribute__((aligned(16))) uint8_t smem[2][S::kBuf];
  __shared__ float part[2][kMW][R][64];
  const int t = threadIdx.x, lane = t & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);

  const long long n_it = (n_rows + kMRows - 1) / kMRows;
  auto load = [&](long long it_, const uint8_t* buf) {
    const long long r0 = it_ * kMRows;
    const uint32_t lds = dma::lds_addr(buf);
#pragma unroll
    for (int q = 0; q < (S::kPieces + kMW - 1) / kMW; ++q) {
      const int piece = wave + kMW * q;
      if (piece >= S::kPieces) break;
      const uint32_t u = 64 * piece + lane, row = min(u / (S::kStride / 16), kMRows - 1u);
      const uint32_t at = min(16 * (u - row * (S::kStride / 16)), S::kRowB - 16u);   // in the row; the gap: anything
      // (rows past the end and rows that no id names: any row's bytes)
      if constexpr (!GATHER) {
        const uint32_t last = (uint32_t)min((long long)kMRows, n_rows - r0) - 1u;
        dma::load16(min(row, last) * S::kRowB + at, w + (size_t)r0 * S::kRowB, lds + 1024 * piece);
      } else {
        const long long id = row_of<GATHER>(ids, min(r0 + row, n_rows - 1), V);
        dma::load16(w + (size_t)max(id, 0LL) * S::kRowB + at, lds + 1024 * piece);
      }
    }
  };

  long long it = blockIdx.x;
  if (it < n_it) load(it, smem[0]);

  // Digit fragments. Q8_0: a[r][j] = block j, elements 32 j + 8 g .. + 7. Q6_K: a[r][q] = elements 4 g .. + 3 of
  // groups (kk) and (kk + 2) of 16, q = 4 g2 + 2 half + kk, group 8 g2 + 2 k + half = elements
  // 128 g2 + 32 k + 16 half ..
  uint2 a[R][8];
  uint2 xh[Q6 ? R : 1], xl[Q6 ? R : 1];   // sums of the digits of groups 8 (g & 1) .. + 7, / 64 and % 64, as K slots
  int up[R];                          // of token 4 r + g
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int tok = min(4 * r + (m >> 2), B - 1);
    asm volatile("" : "+v"(tok));   // after the digits of the group before: one group's 64 values at a time
    const int i = m & 3;
    const size_t h0 = (size_t)tok * kH + 256 * wave;
    // the lane's 64 elements: 8 runs of 8 (Q8_0), 16 of 4 (Q6_K); with its g neighbours the whole slice
    float hv[64];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if constexpr (Q6) {
        const int e = 128 * (q >> 2) + 16 * ((q >> 1) & 1) + 32 * (q & 1) + 4 * g;
        load_h4<XDT>(h, h0 + e, hv + 8 * q);
        load_h4<XDT>(h, h0 + e + 64, hv + 8 * q + 4);
      } else {
        load_h4<XDT>(h, h0 + 32 * q + 8 * g, hv + 8 * q);
        load_h4<XDT>(h, h0 + 32 * q + 8 * g + 4, hv + 8 * q + 4);
      }
    }
    float mx = 0.0f;
    bool bad = false;
#pragma unroll
    for (int e = 0; e < 64; ++e) {
      const float v = fabsf(hv[e]);
      bad |= !(v <= 3.402823466e38f);
      mx = fmaxf(mx, v);
    }
    mx = max_g(bad ? __builtin_inff() : mx);
    const bool nan = mx > 3.402823466e38f;   // infinities and NaN: the token's outputs are NaN
    const int u = fix_up(mx);
    up[r] = __shfl(nan ? 1 << 20 : u, 4 * g);
    // digit i of the lane's elements 4 c .. (NaN, inf: any integers): with 128 added to every digit the digits
    // are the number's bytes
    const uint32_t sel = 0x01010101u * (3 - i) + 0x0400u;
    auto dig4 = [&](int c) {
      uint32_t n[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        n[k] = (uint32_t)(int)rintf(__builtin_amdgcn_ldexpf(hv[4 * c + k], u)) + 0x80808080u;
      const uint32_t lo = __builtin_amdgcn_perm(n[1], n[0], sel), hi = __builtin_amdgcn_perm(n[3], n[2], sel);
      return __builtin_amdgcn_perm(hi, lo, 0x05040100u) ^ 0x80808080u;
    };
    if constexpr (Q6) {
      uint32_t hb[4] = {}, lb[4] = {};      // bytes of groups 0 .. 15
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int g2 = q >> 2, half = (q >> 1) & 1, kk = q & 1;
        a[r][q] = make_uint2(dig4(2 * q), dig4(2 * q + 1));
        // both groups' sums over the four lanes, |.| <= 2048, in one word
        const int x2 = sum_g(__builtin_amdgcn_sdot4((int)a[r][q].x, 0x01010101, 0, false) +
                             (__builtin_amdgcn_sdot4((int)a[r][q].y, 0x01010101, 0, false) << 16));
#pragma unroll
        for (int u2 = 0; u2 < 2; ++u2) {
          const int j = 8 * g2 + 2 * (kk + 2 * u2) + half;
          const int x = u2 ? (x2 - (int)(int16_t)x2) >> 16 : (int)(int16_t)x2;
          const int lo = ((x + 32) & 63) - 32;
          hb[j >> 2] |= ((uint32_t)((x - lo) >> 6) & 255u) << (8 * (j & 3));
          lb[j >> 2] |= ((uint32_t)lo & 255u) << (8 * (j & 3));
        }
      }
      const bool odd = g & 1, use = g < 2;
      xh[r] = use ? make_uint2(odd ? hb[2] : hb[0], odd ? hb[3] : hb[1]) : make_uint2(0u, 0u);
      xl[r] = use ? make_uint2(odd ? lb[2] : lb[0], odd ? lb[3] : lb[1]) : make_uint2(0u, 0u);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) a[r][j] = make_uint2(dig4(2 * j), dig4(2 * j + 1));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(a[r][j].x), "+v"(a[r][j].y));
  }

  __builtin_amdgcn_sched_barrier(0);

  // sums of an earlier iteration's partials: thread 16 b + n: token b, row n
  auto reduce = [&](long long it_, int buf) {
    if (t < 16 * B) {
      const int n = t & 15, b = t >> 4;
      const long long j = it_ * kMRows + n;
      if (j < n_rows) {
        const float* p = &part[buf][0][b >> 2][n + 16 * (b & 3)];
        auto w2 = [&](int q) { return p[q * R * 64] + p[(q + 1) * R * 64]; };
        const float s = (w2(0) + w2(2)) + (w2(4) + w2(6));
        out[(size_t)b * n_rows + j] = row_of<GATHER>(ids, j, V) >= 0 ? s : __builtin_nanf("");
      }
    }
  };

  int cur = 0;
  long long prev = -1;
  for (; it < n_it; it += gridDim.x) {
    dma::wait_vm<0>();
    __syncthreads();
    if (it + gridDim.x < n_it) load(it + gridDim.x, smem[cur ^ 1]);
    __builtin_amdgcn_sched_barrier(0);
    if (prev >= 0) reduce(prev, cur ^ 1);
    const uint8_t* row = smem[cur] + m * S::kStride;
    float fin[R];
    if constexpr (Q6) {
      const uint8_t* sb = row + 210 * wave;                          // 2-byte aligned, by the wave's parity
      const int sh = 2 * (wave & 1);
      const uint32_t* L = reinterpret_cast<const uint32_t*>(sb - sh);
      auto at = [&](int dw) { return __builtin_amdgcn_alignbyte(L[dw + 1], L[dw], sh); };   // bytes 4 dw .. of the block
      uint32_t sc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) sc[i] = at(48 + i);
      const float d = f16_to_f32(at(52) & 0xFFFFu);
      int acc[R][4] = {};
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int g2 = q >> 2, half = (q >> 1) & 1, kk = q & 1;
        const uint32_t wh = at(32 + 8 * g2 + 4 * half + g), wq = at(16 * g2 + 8 * kk + 4 * half + g);
        const uint32_t v[2] = {(wq & 0x0F0F0F0Fu) | ((wh << (4 - 2 * kk)) & 0x30303030u),
                               ((wq >> 4) & 0x0F0F0F0Fu) | ((wh >> (2 * kk)) & 0x30303030u)};
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int j = 8 * g2 + 2 * (kk + 2 * u) + half;
          const int s = (int)(int8_t)(sc[j >> 2] >> (8 * (j & 3)));
          const uint2 b = u ? make_uint2(0u, v[1]) : make_uint2(v[0], 0u);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const i32x4_t x = mfma_i8(a[r][q], b);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][i] += __mul24(x[i], s);
          }
        }
        // (the sums now, not gathered at the end with 128 products kept: both row groups would not fit)
        if constexpr (R > 1) {
#pragma unroll
          for (int r = 0; r < R; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(acc[r][i]));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // the quants went in as q + 32: -32 sum_j sc_j X_j
      const uint2 scv = (g & 1) ? make_uint2(sc[2], sc[3]) : make_uint2(sc[0], sc[1]);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const i32x4_t ch = mfma_i8(xh[r], scv), cl = mfma_i8(xl[r], scv);
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = (float)(acc[r][i] - 32 * (64 * ch[i] + cl[i]));
        fin[r] = d * fmaf(f[0], 16777216.0f, fmaf(f[1], 65536.0f, fmaf(f[2], 256.0f, f[3])));
      }
    } else {
      const uint32_t* L = reinterpret_cast<const uint32_t*>(row + 272 * wave);
      float acc[R][4] = {};
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const uint32_t* P = L + 17 * p;                               // a pair of 34-byte blocks
        const float dd[2] = {f16_to_f32(P[0] & 0xFFFFu), f16_to_f32(P[8] >> 16)};
        const uint32_t e0 = P[2 * g], e1 = P[2 * g + 1], e2 = P[2 * g + 2];
        const uint2 q[2] = {make_uint2(__builtin_amdgcn_alignbyte(e1, e0, 2), __builtin_amdgcn_alignbyte(e2, e1, 2)),
                            make_uint2(P[9 + 2 * g], P[10 + 2 * g])};
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const i32x4_t x = mfma_i8(a[r][2 * p + u], q[u]);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][i] = fmaf(dd[u], (float)x[i], acc[r][i]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < R; ++r) 
        fin[r] = fmaf(acc[r][0], 16777216.0f, fmaf(acc[r][1], 65536.0f, fmaf(acc[r][2], 256.0f, acc[r][3])));
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      part[cur][wave][r][lane] = up[r] == 1 << 20 ? __builtin_nanf("") : ldexpf(fin[r], -up[r]);
    prev = it;
    cur ^= 1;
  }
  __syncthreads();
  if (prev >= 0) reduce(prev, cur ^ 1);
}

template <int NB, int XDT, int GATHER>
__global__ __launch_bounds__(kThreads) void k_lm_head_bf16(const void* __restrict__ h,
                                                           const uint16_t* __restrict__ w,
                                                           long long V,
                                                           const int32_t* __restrict__ ids,
                                                           long long n_rows,
                                                           float* __restrict__ out) {
  const int t = threadIdx.x, lane = t & 63;
  // lane L: elements 512c + 8L .. +8 (c = 0..3): every load is 64 lanes x 16 B contiguous
  float hv[NB][32];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < 32; ++i) hv[b][i] = load_h<XDT>(h, (size_t)b * kH + 512 * (i >> 3) + 8 * lane + (i & 7));
  const long long gw = (long long)blockIdx.x * (kThreads / 64) + (t >> 6);
  const long long nw = (long long)gridDim.x * (kThreads / 64);
  for (long long j0 = gw; j0 < n_rows; j0 += 2 * nw) {
    uint4 v[2][4];
    long long rows[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const long long j = j0 + u * nw;
      rows[u] = j < n_rows ? row_of<GATHER>(ids, j, V) : -1;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        v[u][c] = rows[u] >= 0 ? *reinterpret_cast<const uint4*>(w + (size_t)rows[u] * kH + 512 * c + 8 * lane)
                               : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const long long j = j0 + u * nw;
      if (j >= n_rows) break;
      float a[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) a[b] = 0.0f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t ww[4] = {v[u][c].x, v[u][c].y, v[u][c].z, v[u][c].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float wf = bf16_to_f32((e & 1) ? (ww[e >> 1] >> 16) : (ww[e >> 1] & 0xFFFFu));
#pragma unroll
          for (int b = 0; b < NB; ++b) a[b] = fmaf(hv[b][8 * c + e], wf, a[b]);
        }
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const float s = wave_sum_f32(a[b]);
        if (lane == b) out[(size_t)b * n_rows + j] = rows[u] >= 0 ? s : __builtin_nanf("");
      }
    }
  }
}

}  // namespace lmh
}  // namespace moe

using namespace moe;

namespace {

int cu_count() {
  static int ncu = -1;
  if (ncu < 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      ncu = 256;
  }
  return ncu;
}

template <int FMT, int XDT>
void launch_staged(const void* h, const uint8_t* w, long long V, const int32_t* ids, long long n, float* out,
                   hipStream_t st) {
  const long long n_it = (n + lmh::kRows - 1) / lmh::kRows, cap = 4LL * cu_count();
  auto k = ids ? lmh::k_lm_head_staged<FMT, XDT, 1> : lmh::k_lm_head_staged<FMT, XDT, 0>;
  hipLaunchKernelGGL(k, dim3((unsigned)(n_it < cap ? n_it : cap)), dim3(lmh::kThreads), 0, st, h, w, V, ids, n, out);
}

template <int FMT, int R, int XDT>
void launch_i8(const void* h, int B, const uint8_t* w, long long V, const int32_t* ids, long long n, float* out,
               hipStream_t st) {
  const long long n_it = (n + lmh::kMRows - 1) / lmh::kMRows, cap = 2LL * cu_count();
  auto k = ids ? lmh::k_lm_head_i8<FMT, R, XDT, 1> : lmh::k_lm_head_i8<FMT, R, XDT, 0>;
  hipLaunchKernelGGL(k, dim3((unsigned)(n_it < cap ? n_it : cap)), dim3(64 * lmh::kMW), 0, st, h, B, w, V, ids, n, out);
}

template <int FMT, int XDT>
void launch_quant(const void* h, int B, const uint8_t* w, long long V, const int32_t* ids, long long n, float* out,
                  hipStream_t st) {
  // One token of a short list: the lighter start-up counts (gather from 32768 rows in the last-level cache, us,
  // staged against int8: 64 rows Q6_K 4.1, 7.5, Q8_0 4.5, 6.2; 4096 rows 5.4, 8.0 and 6.1, 6.6; 16384 rows 11.7,
  // 15.5 and 13.9, 13.4). The whole table from HBM: 85, 77 and 95, 93.
  constexpr long long kStagedRows = FMT == MOE_FMT_Q6_K ? 65536 : 12288;
  if (B == 1 && n <= kStagedRows) launch_staged<FMT, XDT>(h, w, V, ids, n, out, st);
  else if (B <= 4) launch_i8<FMT, 1, XDT>(h, B, w, V, ids, n, out, st);
  else launch_i8<FMT, 2, XDT>(h, B, w, V, ids, n, out, st);
}

template <int NB, int XDT, int GATHER>
void launch_bf16(const void* h, const uint8_t* w, long long V, const int32_t* ids, long long n,
                 float* out, hipStream_t st) {
  const long long waves = (n + 1) / 2;
  const long long want = (waves + 3) / 4, cap = 8LL * cu_count();
  hipLaunchKernelGGL((lmh::k_lm_head_bf16<NB, XDT, GATHER>), dim3((unsigned)(want < cap ? want : cap)),
                     dim3(lmh::kThreads), 0, st, h, reinterpret_cast<const uint16_t*>(w), V, ids, n, out);
}

template <int XDT, int GATHER>
void launch_nb(int nb, const void* h, const uint8_t* w, long long V, const int32_t* ids, long long n, float* out,
               hipStream_t st) {
  switch (nb) {
    case 1: launch_bf16<1, XDT, GATHER>(h, w, V, ids, n, out, st); break;
    case 2: launch_bf16<2, XDT, GATHER>(h, w, V, ids, n, out, st); break;
    case 3: launch_bf16<3, XDT, GATHER>(h, w, V, ids, n, out, st); break;
    default: launch_bf16<4, XDT, GATHER>(h, w, V, ids, n, out, st); break;
  }
}

}  // namespace

bool moe_lm_head_supported(int H, int fmt) {
  return H == lmh::kH && (fmt == MOE_FMT_Q6_K || fmt == MOE_FMT_Q8_0 || fmt == MOE_FMT_BF16);
}

int moe_launch_lm_head(const void* h, int h_dtype, int B, const void* w, int fmt, long long V,
                       const int32_t* row_ids, long long n_rows, float* logits, hipStream_t st) {
  const uint8_t* wb = reinterpret_cast<const uint8_t*>(w);
  const size_t hstride = (size_t)lmh::kH * (h_dtype == MOE_DT_F32 ? 4 : 2);
  if (fmt != MOE_FMT_BF16) {
    const bool f32 = h_dtype == MOE_DT_F32;
    auto k = fmt == MOE_FMT_Q6_K ? (f32 ? launch_quant<MOE_FMT_Q6_K, MOE_DT_F32> : launch_quant<MOE_FMT_Q6_K, MOE_DT_BF16>)
                                 : (f32 ? launch_quant<MOE_FMT_Q8_0, MOE_DT_F32> : launch_quant<MOE_FMT_Q8_0, MOE_DT_BF16>);
    k(h, B, wb, V, row_ids, n_rows, logits, st);
    return moe_check_launch("lm_head");
  }
  // tokens in passes of up to four (each pass reads the table once)
  for (int b0 = 0; b0 < B; b0 += 4) {
    const int nb = B - b0 < 4 ? B - b0 : 4;
    const void* hp = reinterpret_cast<const uint8_t*>(h) + (size_t)b0 * hstride;
    float* op = logits + (size_t)b0 * n_rows;
    if (h_dtype == MOE_DT_F32) {
      if (row_ids) launch_nb<MOE_DT_F32, 1>(nb, hp, wb, V, row_ids, n_rows, op, st);
      else launch_nb<MOE_DT_F32, 0>(nb, hp, wb, V, nullptr, n_rows, op, st);
    } else {
      if (row_ids) launch_nb<MOE_DT_BF16, 1>(nb, hp, wb, V, row_ids, n_rows, op, st);
      else launch_nb<MOE_DT_BF16, 0>(nb, hp, wb, V, nullptr, n_rows, op, st);
    }
    const int rc = moe_check_launch("lm_head");
    if (rc != MOE_OK) return rc;
  }
  return MOE_OK;
}
