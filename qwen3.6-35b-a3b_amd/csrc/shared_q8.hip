// The shared expert with Q8_0 weights (the artifact's ffn_*_shexp) on the matrix cores, 17 to 896 tokens: one
// block per (32- or 64-row token tile, narrow weight slab), K split over its waves (shared_small.h), the
// scalar gate and the routed GEMMs' f16 copy of x made by the gate/up launch. (Up to 256 tokens the
// block forward runs the same tiles inside the router and routed down launches.) The 3.3 MB of weights
// stay in L2; what bounds it is the weight pieces' loads (dwords at 2-byte block offsets), so from 257
// tokens on a block takes 64 rows per weight decoded. The 160-row kernels (gemm3.hip) fill few CUs at these
// sizes: gate_up + down 60 + 21 us at 257 to 1024 tokens there, 23 + 10 here at 257, 38 + 16 at 700.
#include "common.h"
#include "moe_internal.h"
#include "shared_small.h"

namespace moe {

template <int XDT, int RG>
__global__ __launch_bounds__(512) void k_sq8_gateup(const void* __restrict__ x, const uint8_t* __restrict__ wg,
                                                    const uint8_t* __restrict__ wu, const void* __restrict__ wsg,
                                                    int gdt, int T, int H, int Is, uint16_t* __restrict__ S,
                                                    float* __restrict__ gate_prob, uint16_t* __restrict__ x16) {
  __shared__ __attribute__((aligned(16))) float red[shs::red_q8_floats<8, RG>()];
  const int nblk = gridDim.x * gridDim.y, bid = blockIdx.y * gridDim.x + blockIdx.x;
  if (x16) {
    const size_t n8 = (size_t)T * H / 8;
    for (size_t i = (size_t)bid * 512 + threadIdx.x; i < n8; i += (size_t)nblk * 512) {
      shs::ARaw<XDT> r;
      shs::ld_a<XDT>(r, reinterpret_cast<const uint8_t*>(x) + i * (XDT == MOE_DT_F32 ? 32 : 16));
      reinterpret_cast<uint4*>(x16)[i] = shs::a_frag_f16<XDT>(r);
    }
  }
  shs::gateup_tile_q8<XDT, 8, RG>(x, wg, wu, T, H, Is, blockIdx.x, blockIdx.y * (16 * RG), S, red);
  if (gate_prob) shs::gate_rows<XDT>(x, wsg, gdt, T, H, gate_prob, bid * 8 + (int)(threadIdx.x >> 6), nblk * 8);
}

template <int RG>
__global__ __launch_bounds__(256) void k_sq8_down(const uint16_t* __restrict__ S, const uint8_t* __restrict__ wd,
                                                  int T, int H, int Is, float* __restrict__ y) {
  __shared__ __attribute__((aligned(16))) float red[shs::red_q8_floats<4, RG>()];
  shs::down_tile_q8<4, RG>(S, wd, T, H, Is, blockIdx.x, blockIdx.y * (16 * RG), y, red);
}

}  // namespace moe

using namespace moe;

// row groups of 16 tokens per block: four once that still gives each CU a block (gate_up at 512 tokens: 23 us,
// 31 with two; at 1024: 39, 56 with two)
static int sq8_groups(int T) { return T <= 256 ? 2 : 4; }

bool moe_sq8_supports(int H, int Is) { return H % 512 == 0 && Is % 256 == 0; }

int moe_launch_sq8_gateup(const void* x, int x_dtype, const void* w_gate, const void* w_up, const void* wsg,
                          int gate_dtype, int T, int H, int Is, uint16_t* S, float* gate_prob, uint16_t* x16,
                          hipStream_t st) {
  if (!moe_sq8_supports(H, Is)) return moe_set_error(MOE_E_UNSUPPORTED, "Q8_0 shared gate_up needs H %% 512 == 0, I_s %% 256 == 0");
  const int rg = sq8_groups(T);
  const dim3 grid(Is / 16, (T + 16 * rg - 1) / (16 * rg));
  const uint8_t *g = reinterpret_cast<const uint8_t*>(w_gate), *u = reinterpret_cast<const uint8_t*>(w_up);
  auto k = x_dtype == MOE_DT_BF16 ? (rg == 2 ? k_sq8_gateup<MOE_DT_BF16, 2> : k_sq8_gateup<MOE_DT_BF16, 4>)
                                  : (rg == 2 ? k_sq8_gateup<MOE_DT_F32, 2> : k_sq8_gateup<MOE_DT_F32, 4>);
  hipLaunchKernelGGL(k, grid, dim3(512), 0, st, x, g, u, wsg, gate_dtype, T, H, Is, S, gate_prob, x16);
  return moe_check_launch("sq8_gateup");
}

int moe_launch_sq8_down(const uint16_t* S, const void* w_down, int T, int H, int Is, float* y, hipStream_t st) {
  if (!moe_sq8_supports(H, Is)) return moe_set_error(MOE_E_UNSUPPORTED, "Q8_0 shared down needs H %% 512 == 0, I_s %% 256 == 0");
  const int rg = sq8_groups(T);
  hipLaunchKernelGGL(rg == 2 ? k_sq8_down<2> : k_sq8_down<4>, dim3(H / 32, (T + 16 * rg - 1) / (16 * rg)), dim3(256), 0, st,
                     S, reinterpret_cast<const uint8_t*>(w_down), T, H, Is, y);
  return moe_check_launch("sq8_down");
}
