// Grouped GEMM of the routed experts for few rows per expert (small batches, prompts up to about a
// thousand tokens): Q4_K gate_up, Q4_K / Q5_K down (gfx950, v_mfma_f32_16x16x32_f16).
//
// With few (token, slot) rows per expert the work is the weights: read each once, decode each once.
// Every wave streams its own weight rows, one super-block (256 of K) of 32 rows at a time: whole
// 16-byte units in address order (4.5 or 5.5 KB, five or six loads, held in registers while the
// super-block before is decoded), then through the wave's own LDS, from which a lane reads the
// header and nibbles of its column: lane n + 16 g the bytes 8 g .. 8 g + 7 of each 32-byte group of
// column n. (Lanes loading their own pieces from memory touched 16 lines per instruction and
// fetched each header four times: gate_up at 64 tokens, 222 experts, 67 us, against 58 so.)
//
// The nibbles go into the MFMA as whole numbers, one mask per pair: a nibble in bits 0-3 of a 16-bit
// half is the f16 subnormal q 2^-24, in bits 4-7 it is q 2^-20, and gfx950's f16 MFMA takes
// subnormals as they are. A sub-block's 32 products are summed alone and scaled by sc_j in f32, a
// super-block's sum by d; the mins are one MFMA per super-block on the sub-block sums of x:
//   sum_k x_k w_k = d sum_j sc_j (sum_k x_k q_k) - dmin sum_j m_j X_j,   X_j = sum of x over sub-block j,
// with X_j / 32 held as an f16 pair (high and low part, 22 bits) and m_j again a subnormal. Nothing of
// the weights is rounded, where gemm4.hip rounds each to f16: 2.9e-4 from the 64-bit expert rows
// instead of 1.2e-3. The price is four f32 FMAs per 16 x 32 sub-block and 16 rows (half the issue
// time of packed 16-bit instructions on this chip: 2 cycles a wave against 4), so it pays for one or
// two row groups and the 160-row kernels keep the larger tiles.
// A dword's pairs come out in byte order (0, 2), (1, 3); the activations are put in the same K order.
//
// The MFMA's 16-deep form is not used for the mins: with its result as the first addend of a
// 32-deep MFMA three instructions later, that MFMA read it before it was written.
//
// Measured at the model's sizes, uniform routing (us; before: gemm6.hip / gemm4.hip for gate_up and
// Q4_K down, gemm3.hip for Q5_K down):
//   tokens                16          64          256         512         1024
//   gate_up (302 MB all)  42 -> 30    85 -> 57    90 -> 71    108 -> 79   114 -> 119
//   Q5_K down (184 MB)    79 -> 22    139 -> 41   160 -> 47   162 -> 53   169 -> 74
// The weights' rate at 256 tokens is 4.3 (gate_up) and 3.9 TB/s; with every item on one expert
// (weights in L2) the same grids take 55 and 36 us, so decode and HBM overlap but not fully.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "moe_internal.h"
#include "lds_dma.h"
#include "shared_small.h"

namespace moe {
namespace g8 {

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kXcd = 8;
constexpr int kGuWaves = 8, kDnWaves = 4;
constexpr int kFrag = 8192;            // LDS bytes of 16 rows x 256 of K (eight 1 KB fragments)
constexpr int kSum = 512 + 16;         // LDS bytes of the sub-block sums of 16 rows, and 16 zero bytes

template <int FMT>
constexpr int sb_bytes() { return FMT == MOE_FMT_Q4_K ? 144 : 176; }
template <int FMT>
constexpr int qs_off() { return FMT == MOE_FMT_Q4_K ? 16 : 48; }
// one super-block's activations of R row groups
template <int R>
constexpr int slot_bytes() { return R * (kFrag + kSum); }

// one super-block of the wave's 32 weight rows, row after row, in 16-byte units
template <int FMT>
constexpr int wbuf_bytes() { return 32 * sb_bytes<FMT>(); }
template <int FMT>
constexpr int raw_loads() { return (32 * sb_bytes<FMT>() + 1023) / 1024; }   // 5 (Q4_K), 6 (Q5_K)

// base is wave-uniform; the offset passes through an empty asm so that its widening stays beside
// the load, which then takes the scalar base + 32-bit offset form (no 64-bit lane address)
__device__ __forceinline__ uint4 ld16(const uint8_t* base, uint32_t off) {
  asm volatile("" : "+v"(off));
  return *reinterpret_cast<const uint4*>(base + off);
}

__device__ __forceinline__ f16x2_t as_h2(uint32_t v) { return __builtin_bit_cast(f16x2_t, v); }

// eight weights of sub-block J as f16 bit patterns, subnormals q 2^-24 (J even, low nibbles) or q 2^-20
// (J odd, high nibbles where they are), from two nibble dwords and (Q5_K) the fifth bits
template <int FMT, int J>
__device__ __forceinline__ uint4 frag(uint2 w, uint2 h) {
  constexpr uint32_t mask = (J & 1) ? 0x00F000F0u : 0x000F000Fu;
  uint32_t p[4] = {w.x & mask, (w.x >> 8) & mask, w.y & mask, (w.y >> 8) & mask};
  if constexpr (FMT == MOE_FMT_Q5_K) {
    // bit J of each byte of h to the nibble's bit 4
    constexpr int to = (J & 1) ? 8 : 4;
    constexpr uint32_t fm = (J & 1) ? 0x01000100u : 0x00100010u;
    auto at = [](uint32_t v, int from) { return from < to ? v << (to - from) : v >> (from - to); };
    p[0] = (at(h.x, J) & fm) | p[0];
    p[1] = (at(h.x, J + 8) & fm) | p[1];
    p[2] = (at(h.y, J) & fm) | p[2];
    p[3] = (at(h.y, J + 8) & fm) | p[3];
  }
  return make_uint4(p[0], p[1], p[2], p[3]);
}

__device__ __forceinline__ f32x4_t mfma32(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
// LDS byte of lane l's 16 bytes of sub-block s's fragment, row group 0 (rows spread over the banks
// for the staging writes; a fragment read covers its kilobyte whatever the order)
__device__ __forceinline__ int frag_at(int s, int m, int g) { return s * 1024 + g * 256 + ((m ^ (g & 1) ^ (2 * (s & 3))) << 4); }

// One super-block of 32 weight rows: the raw rows in wb (row m of column group c at (16 c + m) rows),
// the activations' fragments from fa(r, s) and sums from fx(r); out(c, r, d', n', part, mins): the
// super-block's sums are d' part + n' mins.
template <int R, int FMT, class FA, class FX, class FO>
__device__ __forceinline__ void super_block_t(const uint8_t* wb, FA fa, FX fx, int m, int g, FO out) {
  constexpr int kC = 16 * sb_bytes<FMT>();
  const uint8_t* wr = wb + m * sb_bytes<FMT>();
  const uint8_t* wq = wr + 8 * g;
  uint4 hdr[2];
  uint2 qh[2];
  uint32_t sc[2][2];
  f32x4_t part[2][R];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    hdr[c] = *reinterpret_cast<const uint4*>(wr + c * kC);
    if constexpr (FMT == MOE_FMT_Q5_K) qh[c] = *reinterpret_cast<const uint2*>(wq + c * kC + 16);
    else qh[c] = make_uint2(0u, 0u);
    sc[c][0] = hdr[c].y & 0x3F3F3F3Fu;
    sc[c][1] = (hdr[c].w & 0x0F0F0F0Fu) | ((hdr[c].y >> 2) & 0x30303030u);
  }
  // sub-blocks 2 j (low nibbles) and 2 j + 1 (high)
  auto group = [&](auto J) {
    constexpr int j = decltype(J)::value;
    uint4 b[2][2];
    float s[2][2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const uint2 q = *reinterpret_cast<const uint2*>(wq + c * kC + qs_off<FMT>() + 32 * j);
      b[c][0] = frag<FMT, 2 * j>(q, qh[c]);
      b[c][1] = frag<FMT, 2 * j + 1>(q, qh[c]);
      const uint32_t w = sc[c][j >> 1] >> (16 * (j & 1));
      s[c][0] = (float)(w & 0xFFu);
      s[c][1] = (float)((w >> 8) & 0xFFu) * 0.0625f;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint4 a = fa(r, 2 * j + h);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const f32x4_t v = mfma32(a, b[c][h], (f32x4_t){});
#pragma unroll
          for (int i = 0; i < 4; ++i) part[c][r][i] = j == 0 && h == 0 ? s[c][h] * v[i] : fmaf(s[c][h], v[i], part[c][r][i]);
        }
      }
  };
  group(std::integral_constant<int, 0>{});
  group(std::integral_constant<int, 1>{});
  group(std::integral_constant<int, 2>{});
  group(std::integral_constant<int, 3>{});
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint4 h = hdr[c];
    // d 2^24; -dmin 2^24 32 (the mins are subnormals, the sums X_j / 32)
    const float d = f16_to_f32(h.x & 0xFFFFu) * 0x1p24f, nd = f16_to_f32(h.x >> 16) * -0x1p29f;
    const uint32_t m03 = h.z & 0x3F3F3F3Fu, m47 = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
    const uint4 bm = make_uint4(__builtin_amdgcn_perm(0u, m03, 0x0C010C00u), __builtin_amdgcn_perm(0u, m03, 0x0C030C02u),
                                __builtin_amdgcn_perm(0u, m47, 0x0C010C00u), __builtin_amdgcn_perm(0u, m47, 0x0C030C02u));
#pragma unroll
    for (int r = 0; r < R; ++r) out(c, r, d, nd, part[c][r], mfma32(fx(r), bm, (f32x4_t){}));
  }
}

// acc[c][r] += a super-block with the activations in LDS
template <int R, int FMT>
__device__ __forceinline__ void super_block(const uint8_t* wb, const uint8_t* slot, int m, int g,
                                            f32x4_t (&acc)[2][R]) {
  // K slots 8 g ..: high parts (g = 0), low parts (g = 1) of the eight sub-block sums, zeros
  const uint8_t* sums = slot + R * kFrag + (g < 2 ? m * 32 + g * 16 : 512);
  super_block_t<R, FMT>(
      wb, [&](int r, int s) { return *reinterpret_cast<const uint4*>(slot + r * kFrag + frag_at(s, m, g)); },
      [&](int r) { return *reinterpret_cast<const uint4*>(sums + r * kSum); }, m, g,
      [&](int c, int r, float d, float nd, f32x4_t part, f32x4_t mins) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c][r][i] = fmaf(nd, mins[i], fmaf(d, part[i], acc[c][r][i]));
      });
}
// acc[c][r] = a super-block with the activations in registers
template <int R, int FMT, class AR>
__device__ __forceinline__ void super_block_r(const uint8_t* wb, const AR& A, int m, int g,
                                            f32x4_t (&acc)[2][R]) {
  super_block_t<R, FMT>(
      wb, [&](int r, int s) { return A.f[r][s]; }, [&](int r) { return A.xs[r]; }, m, g,
      [&](int c, int r, float d, float nd, f32x4_t part, f32x4_t mins) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c][r][i] = fmaf(nd, mins[i], d * part[i]);
      });
}

// Staging of one super-block's activations by the block's 256 threads: thread t takes chunk t % 32
// (8 elements) of rows t / 32 + 8 p, p < 2 R.
template <int R>
struct Stage {
  uint4 v[2 * R];
};
template <int R>
__device__ __forceinline__ void stage_load(Stage<R>& s, const uint8_t* base, const uint32_t (&roff)[2 * R], int koff) {
#pragma unroll
  for (int p = 0; p < 2 * R; ++p) {
    uint32_t o = roff[p];
    asm volatile("" : "+v"(o));
    s.v[p] = *reinterpret_cast<const uint4*>(base + koff + o);
  }
}
// a + the two f16 of v (one v_fma_mix_f32 each: `one` is 1.0f the compiler cannot see)
__device__ __forceinline__ float add_h2(uint32_t v, float a, float one) {
  const f16x2_t h = as_h2(v);
  return fmaf((float)h[1], one, fmaf((float)h[0], one, a));
}
template <int R>
__device__ __forceinline__ void stage_store(const Stage<R>& s, uint8_t* slot) {
  const int t = threadIdx.x, row = t >> 5, sub = (t & 31) >> 2, cc = t & 3;
  float one = 1.0f;
  asm volatile("" : "+v"(one));
  const int at0 = frag_at(sub, row, cc);
  const int sum0 = R * kFrag + row * 32 + 2 * sub + 16 * (cc & 1);
#pragma unroll
  for (int p = 0; p < 2 * R; ++p) {
    const uint4 v = s.v[p];
    uint4 o;
    o.x = __builtin_amdgcn_perm(v.y, v.x, 0x05040100u);
    o.y = __builtin_amdgcn_perm(v.y, v.x, 0x07060302u);
    o.z = __builtin_amdgcn_perm(v.w, v.z, 0x05040100u);
    o.w = __builtin_amdgcn_perm(v.w, v.z, 0x07060302u);
    // rows 8 further: bit 3 of m
    *reinterpret_cast<uint4*>(slot + (p >> 1) * kFrag + (at0 ^ ((p & 1) << 7))) = o;
    float x = add_h2(v.x, add_h2(v.y, add_h2(v.z, add_h2(v.w, 0.0f, one), one), one), one);
    x += dpp_f32<0xB1>(x);
    x += dpp_f32<0x4E>(x);
    x *= 0.03125f;
    const _Float16 hi = (_Float16)x;
    const _Float16 lo = (_Float16)(x - (float)hi);
    if (cc < 2) *reinterpret_cast<_Float16*>(slot + (p >> 1) * kSum + sum0 + 256 * (p & 1)) = cc ? lo : hi;
  }
}

// the zero bytes of each row group's sums, in all slots
template <int R>
__device__ __forceinline__ void zero_pads(uint8_t* sm, int slots) {
  for (int i = threadIdx.x; i < 4 * R * slots; i += 64 * kDnWaves)
    *reinterpret_cast<uint32_t*>(sm + i / (4 * R) * slot_bytes<R>() + R * kFrag + (i / 4 % R) * kSum + 512 + 4 * (i & 3)) = 0u;
}

// A list of at most kFewTiles 16-row tiles (skewed routing, or a dozen tokens) leaves most CUs one block or
// none: its tiles are cut into kGuFine (gate_up) and kDnFine (down) times the slabs, the same sums. The count
// is known on the device only, so the kernels choose. Block us, coarse -> fine, Zipf routing: 64 tokens (66 tiles)
// 72.6 -> 66.1, 32 (43) 59.2 -> 54.9, 16 (28) 69.8 -> 60.6. At 96 tiles (16 tokens, uniform) even twice the slabs
// lose: 88 -> 91.
constexpr int kFewTiles = 80, kGuFine = 4, kDnFine = 2;
__device__ __forceinline__ bool few_tiles(const int32_t* __restrict__ tiles) { return tiles[0] <= kFewTiles; }

struct Item {
  int e, m0, rows, col;
};
// Block b: XCD x = b % 8, q = b / 8 -> slab q % ncol of tile 8 (q / ncol) + x. False past the list.
__device__ __forceinline__ bool get_item(const int32_t* __restrict__ tiles, const int32_t* __restrict__ offsets,
                                         int ncol, int bm, Item& it) {
  const int x = blockIdx.x % kXcd, q = blockIdx.x / kXcd;
  const int t = (q / ncol) * kXcd + x;
  if (t >= tiles[0]) return false;
  it.col = q % ncol;
  it.e = tiles[1 + 2 * t];
  it.m0 = tiles[2 + 2 * t];
  it.rows = min(bm, offsets[it.e + 1] - it.m0);
  return true;
}

// f(row groups of a tile of `rows` rows)
template <int RMAX, class F>
__device__ __forceinline__ void with_groups(int rows, F f) {
  if (RMAX == 1 || rows <= 16) return f(std::integral_constant<int, 1>{});
  if constexpr (RMAX > 1) return f(std::integral_constant<int, RMAX>{});
}

// ---- gate_up: wave w of 8 owns super-block w of K (H = 2048) ------------------------------------
// The tile's activations of that super-block stay in the wave's registers for the whole item, so
// nothing is staged and the eight waves together read whole weight rows. A step is 16 gate rows and
// the matching 16 up rows; the eight partial sums meet in LDS (double-buffered, one barrier a
// step) and half the block adds them in wave order while the other waves go on.
// the activations of a wave's super-block: fragment s of row group r, and the sub-block sums as an
// MFMA operand (K slots 8 g ..: high parts for g = 0, low parts for g = 1, zeros)
template <int R>
struct AReg {
  uint4 f[R][8];
  uint4 xs[R];
};

__device__ __forceinline__ float sum_g(float v) {   // over the lanes m, m + 16, m + 32, m + 48
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ uint32_t pack_h2(_Float16 a, _Float16 b) {
  return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
}

// row r of the group: 16 bytes of each sub-block at p + 64 s
template <int R>
__device__ __forceinline__ void load_a(AReg<R>& A, const uint8_t* const (&p)[R]) {
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int s = 0; s < 8; ++s) A.f[r][s] = *reinterpret_cast<const uint4*>(p[r] + 64 * s);
}
template <int R>
__device__ __forceinline__ void arrange_a(AReg<R>& A, int g) {
  float one = 1.0f;
  asm volatile("" : "+v"(one));
#pragma unroll
  for (int r = 0; r < R; ++r) {
    _Float16 h[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const uint4 v = A.f[r][s];
      float x = add_h2(v.x, add_h2(v.y, add_h2(v.z, add_h2(v.w, 0.0f, one), one), one), one);
      x = sum_g(x) * 0.03125f;
      const _Float16 hi = (_Float16)x, lo = (_Float16)(x - (float)hi);
      h[s] = g == 0 ? hi : g == 1 ? lo : (_Float16)0.0f;
      A.f[r][s] = make_uint4(__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.y, v.x, 0x07060302u),
                             __builtin_amdgcn_perm(v.w, v.z, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u));
    }
    A.xs[r] = make_uint4(pack_h2(h[0], h[1]), pack_h2(h[2], h[3]), pack_h2(h[4], h[5]), pack_h2(h[6], h[7]));
  }
}

template <int R>
__device__ __forceinline__ void gateup_item(const Item& it, const uint16_t* __restrict__ x16,
                                            const uint8_t* __restrict__ wg, const uint8_t* __restrict__ wu,
                                            size_t estride, const int32_t* __restrict__ sorted_pairs, int K,
                                            int H, int I, int nsteps, uint16_t* __restrict__ S, uint8_t* sm) {
  constexpr int FMT = MOE_FMT_Q4_K;
  const int t = threadIdx.x, lane = t & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t rowb = (uint32_t)(H / 256) * sb_bytes<FMT>();
  AReg<R> A;
  const uint8_t* ap[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t tok = (uint32_t)sorted_pairs[it.m0 + min(16 * r + m, it.rows - 1)] / (uint32_t)K;
    ap[r] = reinterpret_cast<const uint8_t*>(x16) + tok * (size_t)(H * 2) + wave * 512 + 16 * g;
  }
  // raw units (16 bytes) of the step's 16 gate rows, then its 16 up rows: 144 each, unit u = row
  // u / 9, piece u % 9. Loads 0, 1: gate units 0..127; 2, 3: up; 4: the last 16 of each (the upper
  // lanes repeat the lower ones)
  const size_t eoff = (size_t)it.e * estride + (size_t)(it.col * 16 * nsteps) * rowb + wave * sb_bytes<FMT>();
  const uint8_t *bg = wg + eoff, *bu = wu + eoff;
  uint32_t uo[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) uo[i] = (uint32_t)((64 * i + lane) / 9) * rowb + 16u * ((64 * i + lane) % 9);
  const int u4 = 128 + (lane & 15);
  const uint8_t* p4 = ((lane & 16) ? bu : bg) + (uint32_t)(u4 / 9) * rowb + 16u * (u4 % 9);
  uint8_t* wb = sm + wave * wbuf_bytes<FMT>();
  uint8_t* wst = wb + 16 * lane;
  uint8_t* wst4 = wb + ((lane & 16) ? 2304 : 0) + 16 * u4;
  uint4 raw[5];
  auto load_raw = [&]() {
    raw[0] = ld16(bg, uo[0]);
    raw[1] = ld16(bg, uo[1]);
    raw[2] = ld16(bu, uo[0]);
    raw[3] = ld16(bu, uo[1]);
    raw[4] = *reinterpret_cast<const uint4*>(p4);
    bg += 16 * rowb;
    bu += 16 * rowb;
    p4 += 16 * rowb;
  };
  auto store_raw = [&]() {
    *reinterpret_cast<uint4*>(wst) = raw[0];
    *reinterpret_cast<uint4*>(wst + 1024) = raw[1];
    *reinterpret_cast<uint4*>(wst + 2304) = raw[2];
    *reinterpret_cast<uint4*>(wst + 2304 + 1024) = raw[3];
    *reinterpret_cast<uint4*>(wst4) = raw[4];
  };
  // partial sums: [buffer][wave][r][c][lane] of 16 bytes
  uint8_t* red = sm + kGuWaves * wbuf_bytes<FMT>();
  constexpr int kPart = R * 2048, kBuf = kGuWaves * kPart;
  uint8_t* redw = red + wave * kPart + 16 * lane;
  const __amdgpu_buffer_rsrc_t rs = dma::rsrc(S + (size_t)it.m0 * I, it.rows * I * 2);
  // the element of a row group this thread adds up: row rr, column cc
  const int q = t & 255, rr = q >> 4, cc = q & 15;
  const int rdo = (cc + 16 * (rr >> 2)) * 16 + (rr & 3) * 4;
  const int so = (rr * I + it.col * 16 * nsteps + cc) * 2;
  load_a<R>(A, ap);
  load_raw();
  __builtin_amdgcn_sched_barrier(0);
  arrange_a<R>(A, g);
  for (int i = 0; i < nsteps; ++i) {
    // the wave's own rows: its LDS operations run in order
    store_raw();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (i + 1 < nsteps) load_raw();
    __builtin_amdgcn_sched_barrier(0);
    f32x4_t acc[2][R];
    super_block_r<R, FMT>(wb, A, m, g, acc);
    uint8_t* buf = redw + (i & 1) * kBuf;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < 2; ++c) *reinterpret_cast<f32x4_t*>(buf + r * 2048 + c * 1024) = acc[c][r];
    __syncthreads();
    // R = 1: the block's halves in turn; R = 2: one row group each
    if (R == 2 || (t >> 8) == (i & 1)) {
      const int r = R == 2 ? t >> 8 : 0;
      const uint8_t* rd = red + (i & 1) * kBuf + r * 2048 + rdo;
      float gv = 0.0f, uv = 0.0f;
#pragma unroll
      for (int w = 0; w < kGuWaves; ++w) {
        gv += *reinterpret_cast<const float*>(rd + w * kPart);
        uv += *reinterpret_cast<const float*>(rd + w * kPart + 1024);
      }
      float v = gv * __builtin_amdgcn_rcpf(1.0f + __expf(-gv)) * uv;
      v = fminf(fmaxf(v, -65504.0f), 65504.0f);
      __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (_Float16)v), rs, so + (16 * r * I + 16 * i) * 2, 0, 0);
    }
  }
}

// ---- down: 512 columns per block (few tiles: 256), passes of 128, wave w: 32 of each -------------
// The tile's whole rows (I of K) sit in LDS, staged once.
constexpr int kDownCols = 512, kPassCols = 32 * kDnWaves;
template <int R, int FMT, bool Y16>
__device__ __forceinline__ void down_item(const Item& it, const uint16_t* __restrict__ S,
                                          const uint8_t* __restrict__ wd, size_t estride, int H, int I,
                                          int cols, void* __restrict__ y, uint8_t* sm) {
  const int t = threadIdx.x, lane = t & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nsb = I / 256;
  const uint32_t rowb = (uint32_t)nsb * sb_bytes<FMT>();
  const uint8_t* sbase = reinterpret_cast<const uint8_t*>(S + (size_t)it.m0 * I);
  uint32_t roff[2 * R];
#pragma unroll
  for (int p = 0; p < 2 * R; ++p)
    roff[p] = (uint32_t)min((t >> 5) + 8 * p, it.rows - 1) * (uint32_t)I * 2u + 16u * (t & 31);
  // pass cb: columns it.col cols + 128 cb + 32 w + {0, 16} + m; raw unit u of a super-block: row
  // u / 9 (Q5_K: 11) of the wave's 32, the last load's upper lanes repeating the lower ones
  const uint8_t* b0 = wd + (size_t)it.e * estride + (size_t)(it.col * cols + 32 * wave) * rowb;
  constexpr int NL = raw_loads<FMT>(), kU = sb_bytes<FMT>() / 16;
  uint32_t uo[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int u = 64 * i + (i == NL - 1 ? lane & 31 : lane);
    uo[i] = (uint32_t)(u / kU) * rowb + 16u * (u % kU);
  }
  uint8_t* wb = sm + nsb * slot_bytes<R>() + wave * wbuf_bytes<FMT>();
  uint4 raw[NL];
  auto load_raw = [&](const uint8_t* base) {
#pragma unroll
    for (int i = 0; i < NL; ++i) raw[i] = ld16(base, uo[i]);
  };
  auto store_raw = [&]() {
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<uint4*>(wb + 1024 * i + 16 * (i == NL - 1 ? lane & 31 : lane)) = raw[i];
  };
  load_raw(b0);
  __builtin_amdgcn_sched_barrier(0);
  zero_pads<R>(sm, nsb);
  for (int sb = 0; sb < nsb; ++sb) {
    Stage<R> st;
    stage_load<R>(st, sbase, roff, sb * 512);
    stage_store<R>(st, sm + sb * slot_bytes<R>());
  }
  __syncthreads();
  constexpr int kB = Y16 ? 2 : 4;
  char* yb = reinterpret_cast<char*>(y) + (size_t)it.m0 * H * kB;
  const __amdgpu_buffer_rsrc_t rs = dma::rsrc(yb, it.rows * H * kB);
  const int lane_off = (4 * g * H + it.col * cols + 32 * wave + m) * kB;
  for (int cb = 0; cb < cols / kPassCols; ++cb) {
    f32x4_t acc[2][R];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[c][r] = (f32x4_t){};
    for (int sb = 0; sb < nsb; ++sb) {
      // the wave's own rows: its LDS operations run in order
      store_raw();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      // the next super-block: of these columns, or the first of the pass's next
      const bool row_end = sb + 1 == nsb;
      if (row_end) b0 += (size_t)kPassCols * rowb;
      if (!row_end || cb + 1 < cols / kPassCols) load_raw(b0 + (row_end ? 0 : (sb + 1) * sb_bytes<FMT>()));
      __builtin_amdgcn_sched_barrier(0);
      super_block<R, FMT>(wb, sm + sb * slot_bytes<R>(), m, g, acc);
    }
    const int off = lane_off + kPassCols * cb * kB;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          float v = acc[c][r][i];
          const int at = off + (16 * r + i) * H * kB + 16 * c * kB;
          if constexpr (Y16) {
            v = fminf(fmaxf(v, -65504.0f), 65504.0f);
            __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (_Float16)v), rs, at, 0, 0);
          } else {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rs, at, 0, 0);
          }
        }
  }
}

}  // namespace g8

extern __shared__ __attribute__((aligned(16))) uint8_t g8_lds[];   // the tile's activations

// S [P, I] f16 (sorted order) = SiLU(x16[token] . gate^T) * (x16[token] . up^T) per tile row
template <int RMAX>
__global__ __launch_bounds__(512, (RMAX == 1 ? 4 : 2)) void k_gemm8_gateup(
    const uint16_t* __restrict__ x16, const uint8_t* __restrict__ wg, const uint8_t* __restrict__ wu,
    size_t estride, const int32_t* __restrict__ tiles, const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ sorted_pairs, int K, int H, int I, int nsteps, uint16_t* __restrict__ S) {
  using namespace g8;
  Item it;
  if (RMAX == 1 && few_tiles(tiles)) nsteps /= kGuFine;
  if (!get_item(tiles, offsets, I / (16 * nsteps), 16 * RMAX, it)) return;
  with_groups<RMAX>(it.rows, [&](auto R) {
    gateup_item<decltype(R)::value>(it, x16, wg, wu, estride, sorted_pairs, K, H, I, nsteps, S, g8_lds);
  });
}

// y [P, H] (sorted order; f32, or f16 saturated when Y16) = S . down^T per tile row
template <int RMAX, int FMT, bool Y16>
__global__ __launch_bounds__(64 * g8::kDnWaves, (RMAX == 1 ? 4 : 3)) void k_gemm8_down(
    const uint16_t* __restrict__ S, const uint8_t* __restrict__ wd, size_t estride,
    const int32_t* __restrict__ tiles, const int32_t* __restrict__ offsets, int bm, int H, int I,
    void* __restrict__ y, MoeShJob sh) {
  using namespace g8;
  const int nr = (int)gridDim.x - sh.n;
  if ((int)blockIdx.x >= nr) {
    // the small-T shared expert's down: y = shared_raw
    const int b = (int)blockIdx.x - nr, nslab = sh.H / 32;
    float* red = reinterpret_cast<float*>(g8_lds);
    if (sh.fmt == MOE_FMT_Q8_0)
      shs::down_tile_q8<kDnWaves>(sh.S, reinterpret_cast<const uint8_t*>(sh.w0), sh.T, sh.H, sh.Is, b % nslab,
                                  (b / nslab) * 32, sh.y, red);
    else
      shs::down_tile<kDnWaves, 32>(sh.S, reinterpret_cast<const uint16_t*>(sh.w0), sh.T, sh.H, sh.Is, b % nslab,
                                   (b / nslab) * 32, sh.y, red);
    return;
  }
  Item it;
  const int cols = RMAX == 1 && few_tiles(tiles) ? kDownCols / kDnFine : kDownCols;
  if (!get_item(tiles, offsets, H / cols, bm, it)) return;
  // a taller tile (the list is another kernel's) in pieces
  for (int left = it.rows; left > 0; left -= 16 * RMAX, it.m0 += 16 * RMAX) {
    it.rows = min(left, 16 * RMAX);
    with_groups<RMAX>(it.rows, [&](auto R) { down_item<decltype(R)::value, FMT, Y16>(it, S, wd, estride, H, I, cols, y, g8_lds); });
    if (left > 16 * RMAX) __syncthreads();
  }
}

}  // namespace moe

using namespace moe;

// one block per (tile, slab): the tile list's capacity rounded up to whole groups of 8 tiles; enough too for
// a list of few tiles in `fine` times the slabs
static dim3 g8_grid(int max_tiles, int ncol, int fine) {
  static_assert(g8::kFewTiles % g8::kXcd == 0, "whole groups of 8 tiles");
  const int n = (max_tiles + g8::kXcd - 1) / g8::kXcd * g8::kXcd;
  return dim3((unsigned)(ncol * std::max(n, fine * std::min(n, g8::kFewTiles))));
}

bool moe_gemm8_gateup_supports(int fmt, int H, int I) {
  return fmt == MOE_FMT_Q4_K && H == 256 * g8::kGuWaves && I % 256 == 0;
}
// the tile's S rows stay in LDS whole: 32 rows of at most 1024
bool moe_gemm8_down_supports(int fmt, int H, int I) {
  return (fmt == MOE_FMT_Q4_K || fmt == MOE_FMT_Q5_K) && H % g8::kDownCols == 0 && I % 256 == 0 && I <= 1024;
}

int moe_launch_gemm8_gateup(const uint16_t* x16, const void* w_gate, const void* w_up, size_t expert_stride,
                            const int32_t* tiles, int max_tiles, int bm, const int32_t* offsets,
                            const int32_t* sorted_pairs, int K, int H, int I, uint16_t* S, hipStream_t st) {
  if (!moe_gemm8_gateup_supports(MOE_FMT_Q4_K, H, I) || (bm != 16 && bm != 32))
    return moe_set_error(MOE_E_UNSUPPORTED, "gemm8 gate_up needs H == 2048, I %% 256 == 0 and 16- or 32-row tiles");
  // steps (16 gate + 16 up rows) per block: 8 with 16-row tiles (two blocks on a CU), 16 with 32-row
  // tiles (one block on a CU, so the activations' load at its start is not covered by another):
  // 512 tokens 79 us, against 87 with 8
  const int ns = bm == 16 ? 8 : 16;
  const dim3 grid = g8_grid(max_tiles, I / (16 * ns), bm == 16 ? g8::kGuFine : 1);
  const size_t lds = g8::kGuWaves * (size_t)(g8::wbuf_bytes<MOE_FMT_Q4_K>() + 2 * 2048 * (bm / 16));
  const uint8_t *g = reinterpret_cast<const uint8_t*>(w_gate), *u = reinterpret_cast<const uint8_t*>(w_up);
  if (bm == 16)
    hipLaunchKernelGGL(k_gemm8_gateup<1>, grid, dim3(64 * g8::kGuWaves), lds, st, x16, g, u, expert_stride, tiles,
                       offsets, sorted_pairs, K, H, I, ns, S);
  else
    hipLaunchKernelGGL(k_gemm8_gateup<2>, grid, dim3(64 * g8::kGuWaves), lds, st, x16, g, u, expert_stride, tiles,
                       offsets, sorted_pairs, K, H, I, ns, S);
  return moe_check_launch("gemm8_gateup");
}

template <int RMAX, int FMT>
static void g8_down(bool y16, dim3 grid, hipStream_t st, const uint16_t* S, const uint8_t* w, size_t estride,
                    const int32_t* tiles, const int32_t* offsets, int bm, int H, int I, void* y, const MoeShJob& job) {
  size_t lds = (size_t)(I / 256) * g8::slot_bytes<RMAX>() + g8::kDnWaves * g8::wbuf_bytes<FMT>();
  if (job.n) lds = std::max(lds, shs::red_floats<g8::kDnWaves>() * sizeof(float));
  auto k = y16 ? k_gemm8_down<RMAX, FMT, true> : k_gemm8_down<RMAX, FMT, false>;
  hipLaunchKernelGGL(k, grid, dim3(64 * g8::kDnWaves), lds, st, S, w, estride, tiles, offsets, bm, H, I, y, job);
}

int moe_launch_gemm8_down(const uint16_t* S, const void* w_down, int fmt, size_t expert_stride,
                          const int32_t* tiles, int max_tiles, int bm, const int32_t* offsets, int H, int I,
                          void* y, int y16, hipStream_t st, const MoeShJob* sh) {
  if (!moe_gemm8_down_supports(fmt, H, I))
    return moe_set_error(MOE_E_UNSUPPORTED, "gemm8 down needs Q4_K or Q5_K, H %% 512 == 0, I %% 256 == 0 and I <= 1024");
  const MoeShJob job = sh ? *sh : MoeShJob{};
  if (job.n) {
    // the shared expert's down blocks: 32-column slabs, K split over 4 waves in 64-wide chunks
    if (job.H % 32 || job.Is % 256 || !job.S || !job.w0 || !job.y)
      return moe_set_error(MOE_E_UNSUPPORTED, "gemm8: shared-expert blocks need H %% 32 == 0, I_s %% 256 == 0 and every pointer");
    const int want = moe_shjob_down_blocks(job.T, job.H);
    if (job.n != want) return moe_set_error(MOE_E_ARG, "gemm8: %d shared-expert blocks given, %d needed", job.n, want);
  }
  const bool one = bm <= 16;
  dim3 grid = g8_grid(max_tiles, H / g8::kDownCols, one ? g8::kDnFine : 1);
  grid.x += (unsigned)job.n;
  const uint8_t* w = reinterpret_cast<const uint8_t*>(w_down);
  if (fmt == MOE_FMT_Q4_K)
    (one ? g8_down<1, MOE_FMT_Q4_K> : g8_down<2, MOE_FMT_Q4_K>)(y16, grid, st, S, w, expert_stride, tiles, offsets, bm, H, I, y, job);
  else
    (one ? g8_down<1, MOE_FMT_Q5_K> : g8_down<2, MOE_FMT_Q5_K>)(y16, grid, st, S, w, expert_stride, tiles, offsets, bm, H, I, y, job);
  return moe_check_launch("gemm8_down");
}
