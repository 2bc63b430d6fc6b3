// What the matrix-core kernels (mfma.hip, exact.hip) share: vector types, the
// deal of workgroups to XCDs, exact f16 operands from small integers, and the
// SwiGLU.
#pragma once
#include "common.hpp"
#include "expf_ref.h"

namespace biv {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int WAVE = 64;
constexpr int N_XCD = 8;

// (slot, row tile) of workgroup b of a grouped launch.  The units (the
// shared expert's slots, then the routed slots in use, row tiles fastest)
// go to the 8 XCDs in runs of RUN slots, run g to XCD g % 8 (workgroup
// ids go round-robin over the XCDs): an expert's consecutive slots, and
// every row tile of a slot, then share one XCD's L2, so that the expert's
// rows come from HBM about once, while runs from all over the dispatch
// order keep the XCDs' loads alike.  (Slots of the BF16 kernel hold up to
// 256 pairs, one expert each as a rule: runs of 1.)  The routed slots in
// use are counted in every used slot record.  False: no unit for this
// workgroup.
constexpr int SLOT_RUN = 4, SLOT_RUN_BF16 = 1;
template <int RUN, class Args> __device__ inline bool slot_unit(const Args &a, int b, int &u, int &rt)
{
    const int used = a.u_max > 0 ? min(a.dp.slots[0].used, a.u_max) : 0;
    const int n = (a.n_sh + used) * a.n_rt, run = RUN * a.n_rt;
    const int x = b % N_XCD, i = b / N_XCD;
    const int unit = (x + N_XCD * (i / run)) * run + i % run;
    if (unit >= n) return false;
    u = unit / a.n_rt;
    rt = unit % a.n_rt;
    return true;
}
// workgroups of a grouped launch over `slots` slots (an upper bound) of
// n_rt row tiles: every XCD's share of the runs
template <int RUN> inline unsigned slot_grid(int slots, int n_rt)
{
    const int runs = (slots + RUN - 1) / RUN;
    return (unsigned)(N_XCD * ((runs + N_XCD - 1) / N_XCD) * RUN * n_rt);
}

__device__ const uint64_t exp_tab[32] = BIV_EXPF_TAB_INIT;

// silu(g) * u (ops.rs:159-167) with the exp table in shared memory
__device__ inline float silu_mul_t(float g, float u, const uint64_t *tab)
{
    double r;
    uint64_t ki;
    const uint32_t i = biv_expf_reduce(-g, &r, &ki);
    const float ex = biv_expf_finish(-g, r, ki, tab[i]);
    return (g * (1.0f / (1.0f + ex))) * u;
}

// Four small integers as four exact f16 (two dwords).  Each byte u (0..255)
// becomes the f16 with bits 0x64uu, i.e. 1024 + u, and BIAS is taken off
// (exact: every value is an integer below 2048).  Signed int8 quants come
// in as q ^ 0x80 = q + 128 with BIAS 1152; nibbles 0..15 with BIAS 1024.
template <int BIAS> __device__ __forceinline__ uint2 bytes_to_f16x4(uint32_t u)
{
    const uint32_t r0 = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    const uint32_t r1 = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    const f16x2 bias = {(_Float16)BIAS, (_Float16)BIAS};
    const f16x2 h0 = __builtin_bit_cast(f16x2, r0) - bias, h1 = __builtin_bit_cast(f16x2, r1) - bias;
    return make_uint2(__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1));
}
__device__ __forceinline__ uint2 i8x4_to_f16x4(uint32_t q) { return bytes_to_f16x4<1152>(q ^ 0x80808080u); }

__device__ inline float f16_to_f32(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

} // namespace
} // namespace biv
