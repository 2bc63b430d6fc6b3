// Quantised matrices at prefill sizes, bit for bit in the x86 order, with the
// integer work on the matrix cores.
//
// biv's x86 dot_q8_0, dot_q4k and dot_q6k (engine/src/quant.rs:1368-1533)
// keep 16 f32 chains per row: chain (pi, l) takes the 32-element blocks b =
// pi, pi + 2, ... and for each the int32 of the block's word l (bytes 4l ..
// 4l + 3: a 4-element dot, Q6_K's times its sub-scale), fma(float(word dot),
// w_scale(b) * d_x(b), acc); then the chains are summed in a fixed tree, and
// Q4_K subtracts its mins term last.  The order is kept to the bit because
// gate/up outputs are quantised again, where a rounding difference moves a
// quant by a whole step.
//
// v_mfma_f32_16x16x4_4b_f16 multiplies four independent 16 x 4 by 4 x 16
// blocks, so with block w of a lane group holding word 4 hh + w of 16 input
// rows (A) and of 16 weight rows (B), its 4 x 16 x 16 results are exactly
// the 1024 word dots of one half (hh) of a 32-element block: no masked or
// padded operand.  Both operands hold the quants as f16 (exact integers),
// every product and partial sum is an integer below 2^24, so a result is the
// f32 the reference converts its int32 to.  Lane (lg, lc) = (lane / 16, lane
// % 16) supplies word lg of input row lc and of weight row lc, and receives,
// in register 4 w + r, word w of input row 4 lg + r and weight row lc: it ends
// up with all 16 chains of its 4 input rows and one weight row, and the tree
// runs within the lane.
//
// What bounds it: the chains' FMAs, one per word dot on the vector ALU (64
// cycles per 1024 word dots; an MFMA takes 32 and runs beside them: the pair
// alone measured 72 cycles).  Everything else is kept small against them: a
// wave holds one parity's chains of 16 rows of one matrix and up to 64 input
// rows, so a weight word is converted to f16 once for 64 input rows (10
// instructions per block and lane against 128 FMAs), and the activations are
// written as f16 once by the quantiser and arrive in LDS by DMA.
#include <type_traits>

#include "common.hpp"
#include "layout.hpp"
#include "lds_dma.hpp"
#include "mfma_ops.hpp"

namespace biv {
namespace {

constexpr int EX_WAVES = 4;
constexpr int EX_NTH = 64 * EX_WAVES;
constexpr int EX_KC = 256; // elements of a chunk: a group of 8 blocks, 4 of each parity

__device__ __forceinline__ f16x4 as_f16x4(const uint2 &v) { return __builtin_bit_cast(f16x4, v); }

// The weights of parity pi of one group (256 elements: blocks pi + 2 j, j =
// 0..3) of a row, as lane lg sees them: words lg and 4 + lg of every block.
// operand(j, hh) is word 4 hh + lg of block pi + 2 j as four exact f16;
// wscale() the f32 scale of block pi + 2 lg as the reference forms it.  (pi
// is uniform over the wave.)
// ALL: the scales of the four blocks in every lane (scale(j, pi)).
template <int TY, bool ALL = false> struct ExW;

// Q8_0 (chain layout: unit 16 g + 8 pi + w holds word w of blocks 8 g + pi +
// 2 j, j = 0..3); scale f16(d)
template <bool ALL> struct ExW<T_Q8_0, ALL> {
    uint4 q[2];
    std::conditional_t<ALL, uint2, uint16_t> s;
    __device__ __forceinline__ void load(const DevMat &M, size_t row, int K, int g, int lg, int pi)
    {
        const uint4 *p = reinterpret_cast<const uint4 *>(M.q + row * K) + 16 * g + 8 * pi + lg;
        q[0] = p[0];
        q[1] = p[4];
        const uint16_t *ps = reinterpret_cast<const uint16_t *>(M.s + row * (K / 16)) + pi * (K / 64) + 4 * g;
        if constexpr (ALL) s = *reinterpret_cast<const uint2 *>(ps);
        else s = ps[lg];
    }
    __device__ __forceinline__ f16x4 operand(int j, int hh, int) const { return as_f16x4(i8x4_to_f16x4(q[hh][j])); }
    __device__ __forceinline__ float wscale(int lg, int) const
    {
        if constexpr (ALL) return f16_to_f32((uint32_t)(((uint64_t)s.y << 32 | s.x) >> (16 * lg)) & 0xFFFF);
        else return f16_to_f32(s);
    }
    __device__ __forceinline__ float scale(int j, int) const
    {
        const uint32_t h2 = j < 2 ? s.x : s.y;
        return f16_to_f32((j & 1) ? h2 >> 16 : h2 & 0xFFFF);
    }
};

// Q4_K (chain layout: unit 8 g + w holds word w of the four sub-block pairs
// of super-block g, low nibbles the even sub-block, high the odd); scale d *
// sc of the sub-block, the mins apart
template <bool ALL> struct ExW<T_Q4K, ALL> {
    uint4 q[2];
    uint4 hd; // d, dmin, the 12 scale bytes
    __device__ __forceinline__ void load(const DevMat &M, size_t row, int K, int g, int lg, int)
    {
        const uint4 *p = reinterpret_cast<const uint4 *>(M.q + row * (K / 2)) + 8 * g + lg;
        q[0] = p[0];
        q[1] = p[4];
        hd = reinterpret_cast<const uint4 *>(M.s)[row * (K / 256) + g];
    }
    __device__ __forceinline__ f16x4 operand(int j, int hh, int pi) const
    {
        return as_f16x4(bytes_to_f16x4<1024>((q[hh][j] >> (4 * pi)) & 0x0F0F0F0Fu));
    }
    // the 6-bit scales (or mins) of sub-blocks 0..3 and 4..7, a byte each
    __device__ __forceinline__ uint32_t six(int min, int upper) const
    {
        const uint32_t a = min ? hd.z : hd.y;
        if (!upper) return a & 0x3F3F3F3Fu;
        return ((min ? hd.w >> 4 : hd.w) & 0x0F0F0F0Fu) | ((a >> 2) & 0x30303030u);
    }
    __device__ __forceinline__ float wscale(int lg, int pi) const
    {
        const uint64_t sc = (uint64_t)six(0, 1) << 32 | six(0, 0);
        return f16_to_f32(hd.x & 0xFFFF) * (float)((uint32_t)(sc >> (8 * (2 * lg + pi))) & 0xFF);
    }
    __device__ __forceinline__ float scale(int j, int pi) const
    {
        return f16_to_f32(hd.x & 0xFFFF) * (float)((six(0, j >> 1) >> (8 * (2 * (j & 1) + pi))) & 0xFF);
    }
    __device__ __forceinline__ float dmin() const { return f16_to_f32(hd.x >> 16); }
};

// Q6_K (chain layout: unit (qq / 4) * 16 + 8 pi + w holds the ql words of
// halves qq .. qq + 3, unit (qq / 4) * 8 + w after them their qh words; qq =
// 2 super-block + half); chain pi's step j reads quarter pi + 2 (j & 1) of
// half j >> 1.  The word's sub-scale goes into the operand: (q - 32) * sc as
// (q - 32) * 16 (sc >> 4) plus (q - 32) * (sc & 15), both exact in f16, in
// two MFMAs whose sum is the exact integer.  Scale d.
template <bool ALL> struct ExW<T_Q6K, ALL> {
    uint2 ql[2], qh[2];
    uint32_t sc[2]; // [hh], a byte per step
    uint16_t d;
    __device__ __forceinline__ void load(const DevMat &M, size_t row, int K, int g, int lg, int pi)
    {
        const uint8_t *base = M.q + row * (K / 256) * 192;
        const uint8_t *pl = base + 256 * (g >> 1) + 8 * (g & 1) + 16 * (8 * pi + lg);
        const uint8_t *ph = base + (K / 256) * 128 + 128 * (g >> 1) + 8 * (g & 1) + 16 * lg;
        const uint8_t *ps = M.s + row * (K / 16) + 2 * pi * (K / 64) + 4 * g;
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            ql[hh] = *reinterpret_cast<const uint2 *>(pl + 64 * hh);
            qh[hh] = *reinterpret_cast<const uint2 *>(ph + 64 * hh);
            sc[hh] = *reinterpret_cast<const uint32_t *>(ps + hh * (K / 64));
        }
        d = reinterpret_cast<const uint16_t *>(M.d)[row * (K / 256) + g];
    }
    __device__ __forceinline__ void operands(int j, int hh, int pi, f16x4 &hi, f16x4 &lo) const
    {
        const uint32_t lw = j < 2 ? ql[hh].x : ql[hh].y, hw = j < 2 ? qh[hh].x : qh[hh].y;
        const uint32_t u = ((lw >> (4 * (j & 1))) & 0x0F0F0F0Fu) | (((hw >> (4 * (j & 1) + 2 * pi)) & 0x03030303u) << 4);
        const f16x4 v = as_f16x4(bytes_to_f16x4<1056>(u)); // q - 32
        const int s = (int)(int8_t)(sc[hh] >> (8 * j));
        const _Float16 sh = (_Float16)(s & ~15), sl = (_Float16)(s & 15);
        hi = v * sh;
        lo = v * sl;
    }
    __device__ __forceinline__ float wscale(int, int) const { return f16_to_f32(d); }
};

// LDS of a workgroup that holds NT 16-row input tiles, two chunks: a
// chunk's activations (a row's 512 bytes as 32 16-byte pieces, piece p of row
// r at p ^ (r & 15): 16 lanes reading one piece of 16 rows then fall in 64
// banks), block scales (and Q4_K's block sums) [block][input row]
template <int TY, int NT> struct ExLds {
    static constexpr int ROWS = 16 * NT;
    static constexpr int X = ROWS * 2 * EX_KC;
    static constexpr int S = 8 * ROWS * 4;
    static constexpr int BUF = X + S * (TY == T_Q4K ? 2 : 1);
    // the epilogue's exchange: half of each wave's tiles, 32 chains of a lane each
    static constexpr int EX = EX_WAVES * ((NT + 1) / 2) * 32 * 64 * 4;
    static constexpr int BYTES = 2 * BUF > EX ? 2 * BUF : EX;
};
template <int TY, int NT> constexpr int ex_halves() { return TY == T_Q8_0 && NT > 2 ? 2 : 1; }
// waves per SIMD the registers allow (the 64-row instances at all 256, with 1
// of Q8_0, 11 of Q4_K and 5 of Q6_K spilled)
template <int TY, int NT> constexpr int ex_waves() { return NT > 2 ? 2 : NT == 1 ? 4 : TY == T_Q8_0 ? 3 : 2; }

// out[t][r] = row_r . x_t over rows of any multiple of 512 elements (dense
// FFN): GATEUP silu(gate_r . x_t) * (up_r . x_t).  A workgroup takes up to 16
// NTM input rows and 16 output rows of gate and up (waves: gate, up x the two
// parities), or 32 output rows (two 16-row tiles x the two parities); input
// tiles past the count are left out.  K advances in chunks of 256, the
// next one on its way (activations by DMA, weights to registers) while this
// one is computed.  Workgroups of one
// block of rows are consecutive on one XCD, so its weights come from HBM once
// and from that L2 for the other input rows.
template <int TY, bool GATEUP, int NTM>
__global__ __launch_bounds__(EX_NTH) __attribute__((amdgpu_waves_per_eu(ex_waves<TY, NTM>()))) void k_exact(ExactArgs a)
{
    using W = ExW<TY>;
    using L = ExLds<TY, NTM>;
    constexpr bool Q4 = TY == T_Q4K;
    constexpr int ROWS_WG = GATEUP ? 16 : 32;
    __shared__ __align__(16) uint8_t lds[L::BYTES];
    __shared__ uint32_t roff[L::ROWS]; // bytes from the tile's first activation row
    __shared__ uint64_t tab[GATEUP ? 32 : 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lg = lane >> 4, lc = lane & 15;
    // (row block, input tile) of this workgroup: input tiles fastest, row
    // block rb on XCD rb % 8
    const int n_tt = (a.T + L::ROWS - 1) / L::ROWS, x = blockIdx.x % N_XCD, i0 = blockIdx.x / N_XCD;
    const int rb = (i0 / n_tt) * N_XCD + x, t0 = (i0 % n_tt) * L::ROWS;
    const int rows = a.a.rows, K = a.K;
    if (rb * ROWS_WG >= rows) return;
    const int cnt = min(L::ROWS, a.T - t0);
    // rows past the count repeat the last one (their results are not stored)
    if (tid < L::ROWS) roff[tid] = (uint32_t)min(tid, cnt - 1) * (uint32_t)(2 * K);
    if (GATEUP && tid < 32) tab[tid] = exp_tab[tid];
    const uint8_t *xh = reinterpret_cast<const uint8_t *>(a.xh) + (size_t)t0 * K * 2;
    const uint8_t *xd = reinterpret_cast<const uint8_t *>(a.xd) + (size_t)t0 * (K / 8);
    const uint8_t *xs = reinterpret_cast<const uint8_t *>(a.xs) + (size_t)t0 * (K / 8);
    const int pi = wave & 1, m = wave >> 1; // parity; up (GATEUP) or the row tile
    const DevMat &M = GATEUP && m ? a.b : a.a;
    const int orow = rb * ROWS_WG + (GATEUP ? 0 : 16 * m) + lc;
    const int nc = K / EX_KC;
    const unsigned lds0 = lds_addr(lds);
    __syncthreads();

    auto run = [&](auto nt_c) {
        constexpr int NT = decltype(nt_c)::value;
        // this wave's share of chunk c's DMAs: activations two rows an
        // instruction, then 64 scales an instruction ([block][row]; waves
        // past the 8 blocks repeat them)
        constexpr int ND = 8 * NT / EX_WAVES, BPI = 64 / L::ROWS;
        constexpr int NS = (8 / BPI + EX_WAVES - 1) / EX_WAVES;
        auto issue = [&](int c, unsigned buf) { // buf: LDS address
#pragma unroll
            for (int q = 0; q < ND; q++) {
                const int r2 = EX_WAVES * q + wave, r = 2 * r2 + (lane >> 5);
                lds_dma16_off(xh + 512 * c, roff[r] + 16 * ((lane & 31) ^ (r & 15)), buf + 1024 * r2);
            }
#pragma unroll
            for (int q = 0; q < NS; q++) {
                const int bi = (EX_WAVES * q + wave) % (8 / BPI), b = bi * BPI + lane / L::ROWS;
                const uint32_t o = roff[lane % L::ROWS] / 16 + 4 * b;
                lds_dma4_off(xd + 32 * c, o, buf + L::X + 256 * bi);
                if (Q4) lds_dma4_off(xs + 32 * c, o, buf + L::X + L::S + 256 * bi);
            }
        };
        W w[2];
        issue(0, lds0);
        w[0].load(M, orow, K, 0, lg, pi);
        constexpr int TH = (NT + 1) / 2;
        float acc[NT][4][8], mins[TH][4];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                mins[t / 2][r] = 0.0f;
#pragma unroll
                for (int l = 0; l < 8; l++) acc[t][r][l] = 0.0f;
            }
        const f32x16 z = {};
        // the lane's row (lc of a tile); piece 4 b + lg of it is words lg and 4 + lg of block b
        const int xo = lc * 512;
        auto compute = [&](const W &w, const uint8_t *buf) {
            if constexpr (Q4) {
                // mins += dmin * (m_a * s_a + m_b * s_b) over the sub-block
                // pairs in order; the products m * s (rounded once, as
                // written) by k = 1 f32 MFMAs, four sub-blocks in one.  The
                // even tiles' in parity 0's waves, the odd tiles' in parity 1's.
                const float dm = w.dmin();
#pragma unroll
                for (int hf = 0; hf < 2; hf++) {
                    const float mv = (float)((w.six(1, hf) >> (8 * lg)) & 0xFF);
#pragma unroll
                    for (int t2 = 0; t2 < TH; t2++) {
                        // (past the last tile: its values again, unused)
                        const float sv = *reinterpret_cast<const float *>(
                            buf + L::X + L::S + ((4 * hf + lg) * L::ROWS + 16 * min(2 * t2 + pi, NT - 1) + lc) * 4);
                        const f32x16 p = __builtin_amdgcn_mfma_f32_16x16x1f32(sv, mv, z, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            mins[t2][r] = mins[t2][r] + dm * (p[r] + p[4 + r]);
                            mins[t2][r] = mins[t2][r] + dm * (p[8 + r] + p[12 + r]);
                        }
                    }
                }
            }
            // The words' halves hh in passes of NH: the weight operands of a
            // pass once for all tiles (K-quants, whose operands or mins take
            // more registers, one half at a time).
            constexpr int NH = ex_halves<TY, NTM>();
            const float dw = w.wscale(lg, pi);
#pragma unroll
            for (int h0 = 0; h0 < 2; h0 += NH) {
                f16x4 b0[4][NH], b1[4][NH];
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int h = 0; h < NH; h++) {
                        if constexpr (TY == T_Q6K) w.operands(j, h0 + h, pi, b0[j][h], b1[j][h]);
                        else b0[j][h] = w.operand(j, h0 + h, pi);
                    }
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    // w_scale * d_x of four blocks, the rounded product the
                    // reference forms, in one k = 1 f32 MFMA: register 4 j + r
                    // is block 2 j + pi of input row 4 lg + r and the lane's
                    // weight row
                    float dx = *reinterpret_cast<const float *>(buf + L::X + ((2 * lg + pi) * L::ROWS + 16 * t + lc) * 4);
                    // (formed again in each pass rather than kept: registers)
                    if (NH == 1) asm volatile("" : "+v"(dx));
                    const f32x16 s = __builtin_amdgcn_mfma_f32_16x16x1f32(dx, dw, z, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const uint8_t *xp = buf + xo + 8192 * t + 16 * ((4 * (2 * j + pi) + lg) ^ lc);
                        f16x4 xa[NH];
                        if constexpr (NH == 2) {
                            const f16x8 v = *reinterpret_cast<const f16x8 *>(xp);
                            xa[0] = __builtin_shufflevector(v, v, 0, 1, 2, 3);
                            xa[NH - 1] = __builtin_shufflevector(v, v, 4, 5, 6, 7);
                        } else {
                            xa[0] = *reinterpret_cast<const f16x4 *>(xp + 8 * h0);
                        }
#pragma unroll
                        for (int h = 0; h < NH; h++) {
                            const int hh = h0 + h;
                            f32x16 d = __builtin_amdgcn_mfma_f32_16x16x4f16(xa[h], b0[j][h], z, 0, 0, 0);
                            if constexpr (TY == T_Q6K) d = __builtin_amdgcn_mfma_f32_16x16x4f16(xa[h], b1[j][h], d, 0, 0, 0);
#pragma unroll
                            for (int l = 0; l < 4; l++)
#pragma unroll
                                for (int r = 0; r < 4; r++)
                                    acc[t][r][4 * hh + l] = __builtin_fmaf(d[4 * l + r], s[4 * j + r], acc[t][r][4 * hh + l]);
                        }
                    }
                }
            }
        };
        // (nc is even; past the end the last chunk is fetched again, unused,
        // so that the loop body has no branch)
        for (int c0 = 0; c0 < nc; c0 += 2)
#pragma unroll
            for (int d = 0; d < 2; d++) {
                // chunk c0 + d is in, in every wave; and every wave is done
                // with the chunk before it, whose buffer the next one takes
                __builtin_amdgcn_sched_barrier(0);
                wait_vm<0>();
                rm_barrier();
                const int cn = min(c0 + d + 1, nc - 1);
                issue(cn, lds0 + (1 - d) * L::BUF);
                w[1 - d].load(M, orow, K, cn, lg, pi);
                __builtin_amdgcn_sched_barrier(0);
                compute(w[d], lds + d * L::BUF);
            }
        wait_vm<0>();
        // The reference's tree: chains pi, then l 4, 2 and 1 apart.  The
        // parities' waves swap tiles through LDS (the chunks' buffers, free
        // after the barrier): parity 0 finishes the even tiles, 1 the odd.
        float4 *ex = reinterpret_cast<float4 *>(lds);
        __syncthreads();
        auto give = [&](auto p_c) {
            constexpr int P = decltype(p_c)::value;
#pragma unroll
            for (int t2 = 0; t2 < TH; t2++)
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        const int t = 2 * t2 + 1 - P;
                        if (t < NT)
                            ex[((wave * TH + t2) * 8 + 2 * r + q) * 64 + lane] =
                                make_float4(acc[t < NT ? t : 0][r][4 * q], acc[t < NT ? t : 0][r][4 * q + 1],
                                            acc[t < NT ? t : 0][r][4 * q + 2], acc[t < NT ? t : 0][r][4 * q + 3]);
                    }
        };
        if (pi) give(std::integral_constant<int, 1>());
        else give(std::integral_constant<int, 0>());
        __syncthreads();
        float y[TH][4];
        auto take = [&](auto p_c) {
            constexpr int P = decltype(p_c)::value;
#pragma unroll
            for (int t2 = 0; t2 < TH; t2++) {
                const int t = 2 * t2 + P;
                if (t >= NT) continue;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float4 o0 = ex[(((wave ^ 1) * TH + t2) * 8 + 2 * r) * 64 + lane];
                    const float4 o1 = ex[(((wave ^ 1) * TH + t2) * 8 + 2 * r + 1) * 64 + lane];
                    const float *c = acc[t < NT ? t : 0][r];
                    const float v0 = (c[0] + o0.x) + (c[4] + o1.x), v1 = (c[1] + o0.y) + (c[5] + o1.y);
                    const float v2 = (c[2] + o0.z) + (c[6] + o1.z), v3 = (c[3] + o0.w) + (c[7] + o1.w);
                    y[t2][r] = (v0 + v2) + (v1 + v3);
                    if (Q4) y[t2][r] = y[t2][r] - mins[t2][r];
                }
            }
        };
        if (pi) take(std::integral_constant<int, 1>());
        else take(std::integral_constant<int, 0>());
        // input row t0 + 16 t + 4 lg + r, output row orow
        auto store = [&](int t, int r, float v) {
            const int i = 16 * t + 4 * lg + r;
            if (i >= cnt) return;
            float *o = a.out + (size_t)(t0 + i) * rows + orow;
            *o = (!GATEUP && a.add) ? *o + v : v;
        };
        if constexpr (!GATEUP) {
#pragma unroll
            for (int t2 = 0; t2 < TH; t2++)
                if (2 * t2 + pi < NT)
#pragma unroll
                    for (int r = 0; r < 4; r++) store(2 * t2 + pi, r, y[t2][r]);
        } else {
            // gate and up meet: the gate waves finish rows r = 0, 1 of each
            // four, the up waves r = 2, 3
            float2 *ex2 = reinterpret_cast<float2 *>(lds);
            __syncthreads();
#pragma unroll
            for (int t2 = 0; t2 < TH; t2++)
                if (2 * t2 + pi < NT)
                    ex2[(wave * TH + t2) * 64 + lane] =
                        m ? make_float2(y[t2][0], y[t2][1]) : make_float2(y[t2][2], y[t2][3]);
            __syncthreads();
#pragma unroll
            for (int t2 = 0; t2 < TH; t2++) {
                if (2 * t2 + pi >= NT) continue;
                const float2 o = ex2[((wave ^ 2) * TH + t2) * 64 + lane];
                const float g0 = m ? o.x : y[t2][0], g1 = m ? o.y : y[t2][1];
                const float u0 = m ? y[t2][2] : o.x, u1 = m ? y[t2][3] : o.y;
                store(2 * t2 + pi, 2 * m, silu_mul_t(g0, u0, tab));
                store(2 * t2 + pi, 2 * m + 1, silu_mul_t(g1, u1, tab));
            }
        }
    };
    // the tiles that hold rows (uniform over the workgroup)
    const int nt = (cnt + 15) / 16;
    if constexpr (NTM >= 4) {
        if (nt == 4) return run(std::integral_constant<int, 4>());
        if (nt == 3) return run(std::integral_constant<int, 3>());
    }
    if constexpr (NTM >= 2)
        if (nt == 2) return run(std::integral_constant<int, 2>());
    run(std::integral_constant<int, 1>());
}

// ---------------------------------------------------------------------------
// The experts' gate/up at prefill sizes (Q8_0, Q4_K), the same sums over a
// slot of up to 16 pairs.
//
// Here the weights are met by one slot only and come from HBM, so what counts
// besides the chains' FMAs is that their loads run far ahead: a workgroup
// stages its pairs' whole rows once (f16, 64 KB at K = 2048, by DMA), and
// after that one barrier its waves run free, each streaming 16 rows of gate
// and the same 16 of up with the next group's loads in flight in registers
// (three of four steps ahead, a step being one matrix and one parity of 256
// elements; Q4_K, whose bytes hold both parities, two of four).  A wave holds
// both matrices' chains of the 16 pairs (128 accumulators), so the tree and
// the SwiGLU need no exchange between lanes.
//
// DUMP: the instance that writes the integer block dots, for the taps only (it
// spills 530 to 730 VGPRs; the f32 chains that matter are the other's, which
// the block's outputs test).
constexpr int GS_WAVES = 4;
constexpr int GS_NTH = 64 * GS_WAVES;
constexpr int GS_ROWS = MFMA_Q8_TILE;       // pairs of a slot
constexpr int GS_ROWS_WG = 16 * GS_WAVES;   // output rows of a workgroup
static_assert(GS_ROWS == 16, "one tile of pairs");

template <int TY, int K, bool DUMP>
__global__ __launch_bounds__(GS_NTH) __attribute__((amdgpu_waves_per_eu(DUMP ? 1 : 2))) void k_gu_slot(MvArgs a)
{
    using W = ExW<TY, true>;
    constexpr bool Q4 = TY == T_Q4K;
    constexpr int NB = K / 32, NG = K / EX_KC;
    constexpr int X = GS_ROWS * 2 * K, S = NB * GS_ROWS * 4;
    // a pair's row as 16-byte pieces, piece p of row r at p ^ r (low four
    // bits): 16 lanes reading one piece of 16 rows fall in 64 banks; then the
    // block scales (and Q4_K's block sums) [block][pair]
    __shared__ __align__(16) uint8_t lds[X + S * (Q4 ? 2 : 1)];
    __shared__ uint64_t tab[32]; // expf's table, for the SwiGLU
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lg = lane >> 4, lc = lane & 15;
    int u, rt;
    if (!slot_unit<SLOT_RUN>(a, blockIdx.x, u, rt)) return;
    const bool shared = u < a.n_sh;
    int e = 0, beg, cnt, tok0 = 0;
    if (shared) {
        tok0 = u * a.sh_chunk;
        beg = a.P + tok0;
        cnt = min(a.sh_chunk, a.T - tok0);
    } else {
        const Slot &sl = a.dp.slots[u - a.n_sh];
        cnt = __builtin_amdgcn_readfirstlane(sl.cnt);
        if (cnt == 0) return;
        e = __builtin_amdgcn_readfirstlane(sl.expert);
        beg = __builtin_amdgcn_readfirstlane(sl.beg);
    }
    if (tid < 32) tab[tid] = exp_tab[tid];
    const DevMat Mg = shared ? a.sa : a.a, Mu = shared ? a.sb : a.b;
    const int rows = Mg.rows, orow = rt * GS_ROWS_WG + 16 * wave + lc;
    const size_t wrow = (size_t)e * rows + orow;
    // lane lc's pair (past the count the last one)
    const int ti = min(lc, cnt - 1), tok = shared ? tok0 + ti : a.dp.pair_tok[beg + ti];
    // the weights of steps: w[mat][pi] of a 256-element group (Q4_K: both
    // parities in pi 0).  (Two groups a turn for Q4_K, loads three steps
    // ahead, double the loop's code, which narrow rows run through once:
    // 512-wide layers 41 against 38 us.)
    constexpr int NP = Q4 ? 1 : 2;
    W w[2][NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
        w[0][p].load(Mg, wrow, K, 0, lg, p);
        w[1][p].load(Mu, wrow, K, 0, lg, p);
    }
    {
        const unsigned lds0 = lds_addr(lds);
        const uint8_t *xh = reinterpret_cast<const uint8_t *>(a.xq);
        // rows past the count stay as they are (their results are not stored)
#pragma unroll
        for (int q = 0; q < GS_ROWS / GS_WAVES; q++) {
            const int r = GS_WAVES * q + wave;
            if (r >= cnt) break; // uniform over the wave
            const uint8_t *src = xh + (size_t)(uint32_t)__builtin_amdgcn_readlane(tok, r) * (2 * K);
#pragma unroll
            for (int i = 0; i < K / 512; i++)
                lds_dma16_off(src, 16 * ((64 * i + lane) ^ r), lds0 + r * 2 * K + 1024 * i);
        }
        const size_t so = (size_t)tok * NB + lg; // four blocks of 16 pairs an instruction
#pragma unroll
        for (int q = 0; q < NB / 4 / GS_WAVES; q++) {
            const int b4 = GS_WAVES * q + wave;
            lds_dma4_at(a.xd + so + 4 * b4, lds0 + X + 256 * b4);
            if (Q4) lds_dma4_at(a.xs + so + 4 * b4, lds0 + X + S + 256 * b4);
        }
    }
    wait_vm<0>();
    __syncthreads();
    const f32x16 z = {};
    const f32x4 z4 = {};
    const std::integral_constant<int, 0> c0;
    const std::integral_constant<int, 1> c1;
    auto at = [&](int o) { return reinterpret_cast<const float *>(lds + o); };
    // The steps of every group in turn, each matrix's (and for Q8_0 parity's)
    // followed by the load of the same of the next group (past the end the
    // last one again, unused: no branch in the loop); advance() ends a group.
    auto walk = [&](auto step, auto advance) {
        // the group count as a value the compiler cannot see through (a.T is
        // never negative): a loop of one or two turns it would lay out flat,
        // the turns' loads and chains overlapped past the registers
        const int ng = NG + (a.T < 0 ? 2 : 0);
#pragma unroll 1
        for (int g = 0; g < ng; g++) {
            const int gn = min(g + 1, NG - 1);
            step(w[0][0], g, c0, c0);
            if constexpr (Q4) step(w[0][0], g, c0, c1);
            w[0][0].load(Mg, wrow, K, gn, lg, 0);
            step(w[1][0], g, c1, c0);
            if constexpr (Q4) step(w[1][0], g, c1, c1);
            w[1][0].load(Mu, wrow, K, gn, lg, 0);
            if constexpr (!Q4) {
                step(w[0][NP - 1], g, c0, c1);
                w[0][NP - 1].load(Mg, wrow, K, gn, lg, 1);
                step(w[1][NP - 1], g, c1, c1);
                w[1][NP - 1].load(Mu, wrow, K, gn, lg, 1);
            }
            advance();
        }
    };
    auto dump = [&](int m, int row, int b, int v) { // the block dots, for the taps
        int32_t *d = m ? a.dump_b : a.dump_a;
        if (d && row < cnt) d[((size_t)(beg + row) * rows + orow) * NB + b] = v;
    };
    // Slots of more than 8 pairs: 16-row tiles.
    auto run16 = [&]() {
        float acc[2][4][2][8], mins[2][4]; // [matrix][row][parity][word]
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                mins[m][r] = 0.0f;
#pragma unroll
                for (int l = 0; l < 8; l++) acc[m][r][0][l] = acc[m][r][1][l] = 0.0f;
            }
        // byte offsets in LDS, 512 a group: the lane's pieces of blocks 2 j +
        // pi (j & 1; j >> 1 is 256 bytes on), its block scale and block sum
        int xo[2][2], dlo = X + 128 * lg + 4 * lc, slo = X + S + 64 * lg + 4 * lc;
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int p = 0; p < 2; p++) xo[j][p] = lc * 2 * K + 16 * ((8 * j + 4 * p + lg) ^ lc);
        auto step = [&](const W &wm, int g, auto m_c, auto pi_c) {
            constexpr int m = decltype(m_c)::value, pi = decltype(pi_c)::value;
            if constexpr (Q4) if constexpr (pi == 0) {
                // mins += dmin * (m_a * s_a + m_b * s_b) over the sub-block
                // pairs in order; four products m * s (rounded once, as
                // written) in one k = 1 f32 MFMA
                const float dm = wm.dmin();
#pragma unroll
                for (int hf = 0; hf < 2; hf++) {
                    const float mv = (float)((wm.six(1, hf) >> (8 * lg)) & 0xFF);
                    const f32x16 p = __builtin_amdgcn_mfma_f32_16x16x1f32(*at(slo + 256 * hf), mv, z, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        mins[m][r] = mins[m][r] + dm * (p[r] + p[4 + r]);
                        mins[m][r] = mins[m][r] + dm * (p[8 + r] + p[12 + r]);
                    }
                }
            }
            // w_scale * d_x of blocks 2 j + pi in registers 4 j + r
            const f32x16 s = __builtin_amdgcn_mfma_f32_16x16x1f32(*at(dlo + 64 * pi), wm.wscale(lg, pi), z, 0, 0, 0);
            // (the second matrix's step reads the activations again: kept
            // from the first they take 16 registers)
            asm volatile("" : "+v"(xo[0][pi]), "+v"(xo[1][pi]));
            // Unit u = 2 j + hh: its MFMA is issued before the FMAs of the
            // unit before it, which cover its latency (kernel alone: Q8_0 at
            // 512 tokens 231 -> 219 us, Q4_K at 2048 644 -> 615).  LDS reads,
            // weight loads and scalar work may cross the scheduling barriers.
            constexpr int LOADS = 0x124; // SALU, VMEM reads, LDS reads
            f16x8 xa[4];
#pragma unroll
            for (int j = 0; j < 4; j++) xa[j] = *reinterpret_cast<const f16x8 *>(lds + xo[j & 1][pi] + 256 * (j >> 1));
            auto dots = [&](int u) {
                const f16x8 v = xa[u >> 1];
                const f16x4 x4 = u & 1 ? __builtin_shufflevector(v, v, 4, 5, 6, 7) : __builtin_shufflevector(v, v, 0, 1, 2, 3);
                return __builtin_amdgcn_mfma_f32_16x16x4f16(x4, wm.operand(u >> 1, u & 1, pi), z, 0, 0, 0);
            };
            f32x16 dn = dots(0);
            int bdot[4] = {0, 0, 0, 0}; // (DUMP)
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const f32x16 d = dn;
                if (u < 7) dn = dots(u + 1);
                __builtin_amdgcn_sched_barrier(LOADS);
#pragma unroll
                for (int l = 0; l < 4; l++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        acc[m][r][pi][4 * (u & 1) + l] =
                            __builtin_fmaf(d[4 * l + r], s[4 * (u >> 1) + r], acc[m][r][pi][4 * (u & 1) + l]);
                if (DUMP)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        bdot[r] = (u & 1 ? bdot[r] : 0) + (int)d[r] + (int)d[4 + r] + (int)d[8 + r] + (int)d[12 + r];
                        if (u & 1) dump(m, 4 * lg + r, 8 * g + 2 * (u >> 1) + pi, bdot[r]);
                    }
                __builtin_amdgcn_sched_barrier(LOADS);
            }
            __builtin_amdgcn_sched_barrier(0); // (steps one by one: registers)
        };
        walk(step, [&]() {
            xo[0][0] += 512;
            xo[0][1] += 512;
            xo[1][0] += 512;
            xo[1][1] += 512;
            dlo += 512;
            slo += 512;
        });
        // the reference's tree (chains pi, then l 4, 2 and 1 apart), the
        // mins, and silu(gate) * up
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float y[2];
#pragma unroll
            for (int m = 0; m < 2; m++) {
                float v[4];
#pragma unroll
                for (int l = 0; l < 4; l++)
                    v[l] = (acc[m][r][0][l] + acc[m][r][1][l]) + (acc[m][r][0][l + 4] + acc[m][r][1][l + 4]);
                y[m] = (v[0] + v[2]) + (v[1] + v[3]);
                if (Q4) y[m] = y[m] - mins[m][r];
            }
            o[r] = silu_mul_t(y[0], y[1], tab);
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (4 * lg + r < cnt) a.out[(size_t)(beg + 4 * lg + r) * rows + orow] = o[r];
    };
    // Slots of up to 8 pairs, in NQ groups of 4 rows (v_mfma_f32_4x4x4_16b_f16,
    // whose 16 blocks are the words lg of 16 weight rows): lane (lg, lc) gets
    // word lg of a group's row r and weight row lc in register r, so it holds
    // the chains of words lg and 4 + lg, and the tree over lg runs across
    // lanes 16 and 32 apart.
    auto run4 = [&](auto nq_c) {
        constexpr int NQ = decltype(nq_c)::value;
        float acc[2][NQ][2][2][4], mins[2][NQ][4]; // [matrix][group][parity][half][row]
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int q = 0; q < NQ; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    mins[m][q][r] = 0.0f;
#pragma unroll
                    for (int h = 0; h < 2; h++) acc[m][q][0][h][r] = acc[m][q][1][h][r] = 0.0f;
                }
        const int row = lane & 3; // the lane's row of each group, as an operand
        int xo[NQ][2][2], dlo = X + 4 * row;
#pragma unroll
        for (int q = 0; q < NQ; q++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int p = 0; p < 2; p++)
                    xo[q][j][p] = (4 * q + row) * 2 * K + 16 * ((8 * j + 4 * p + lg) ^ (4 * q + row));
        auto step = [&](const W &wm, int g, auto m_c, auto pi_c) {
            constexpr int m = decltype(m_c)::value, pi = decltype(pi_c)::value;
            if constexpr (Q4) if constexpr (pi == 0) {
                const float dm = wm.dmin();
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float mv[2];
#pragma unroll
                    for (int o = 0; o < 2; o++) mv[o] = (float)((wm.six(1, j >> 1) >> (8 * (2 * (j & 1) + o))) & 0xFF);
#pragma unroll
                    for (int q = 0; q < NQ; q++) {
                        f32x4 p[2];
#pragma unroll
                        for (int o = 0; o < 2; o++)
                            p[o] = __builtin_amdgcn_mfma_f32_4x4x1f32(*at(dlo + S + 64 * (2 * j + o) + 16 * q), mv[o], z4, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) mins[m][q][r] = mins[m][q][r] + dm * (p[0][r] + p[1][r]);
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float dw = wm.scale(j, pi);
                f32x4 s[NQ];
                f16x8 xa[NQ];
                int bdot[NQ][4] = {}; // (DUMP)
#pragma unroll
                for (int q = 0; q < NQ; q++) {
                    s[q] = __builtin_amdgcn_mfma_f32_4x4x1f32(*at(dlo + 64 * (2 * j + pi) + 16 * q), dw, z4, 0, 0, 0);
                    xa[q] = *reinterpret_cast<const f16x8 *>(lds + xo[q][j & 1][pi] + 256 * (j >> 1));
                }
#pragma unroll
                for (int hh = 0; hh < 2; hh++) {
                    const f16x4 b = wm.operand(j, hh, pi);
#pragma unroll
                    for (int q = 0; q < NQ; q++) {
                        const f16x4 x4 = hh ? __builtin_shufflevector(xa[q], xa[q], 4, 5, 6, 7)
                                            : __builtin_shufflevector(xa[q], xa[q], 0, 1, 2, 3);
                        const f32x4 d = __builtin_amdgcn_mfma_f32_4x4x4f16(x4, b, z4, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            acc[m][q][pi][hh][r] = __builtin_fmaf(d[r], s[q][r], acc[m][q][pi][hh][r]);
                            if (DUMP) bdot[q][r] += (int)d[r];
                        }
                    }
                }
                if (DUMP)
#pragma unroll
                    for (int q = 0; q < NQ; q++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            int v = bdot[q][r]; // of the lane's words: the four lanes' sum
                            v += __shfl_xor(v, 16);
                            v += __shfl_xor(v, 32);
                            if (lg == 0) dump(m, 4 * q + r, 8 * g + 2 * j + pi, v);
                        }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        walk(step, [&]() {
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                xo[q][0][0] += 512;
                xo[q][0][1] += 512;
                xo[q][1][0] += 512;
                xo[q][1][1] += 512;
            }
            dlo += 512;
        });
        // the tree, in every lane; lane lg then finishes row lg of each group
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            float y[2];
#pragma unroll
            for (int m = 0; m < 2; m++) {
                float t[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float v = (acc[m][q][0][0][r] + acc[m][q][1][0][r]) + (acc[m][q][0][1][r] + acc[m][q][1][1][r]);
                    v = v + __shfl_xor(v, 32); // v0 + v2, v1 + v3
                    t[r] = v + __shfl_xor(v, 16);
                    if (Q4) t[r] = t[r] - mins[m][q][r];
                }
                y[m] = lg == 0 ? t[0] : lg == 1 ? t[1] : lg == 2 ? t[2] : t[3];
            }
            const float o = silu_mul_t(y[0], y[1], tab);
            if (4 * q + lg < cnt) a.out[(size_t)(beg + 4 * q + lg) * rows + orow] = o;
        }
    };
    // (uniform over the workgroup.  Everything is in already: the waits here
    // tell the compiler so, whose merged view of the paths would otherwise
    // make each turn of a loop wait for every load in flight.)
    if (cnt > 8) {
        wait_vm<0>();
        run16();
    } else if (cnt > 4) {
        wait_vm<0>();
        run4(std::integral_constant<int, 2>());
    } else {
        wait_vm<0>();
        run4(std::integral_constant<int, 1>());
    }
}

} // namespace

constexpr int N_CU = 256;

// workgroups of a launch with 16 NTM input rows each
template <bool GATEUP, int NTM> static size_t exact_grid(const ExactArgs &a)
{
    constexpr int ROWS_WG = GATEUP ? 16 : 32, TT = 16 * NTM;
    const int n_rb = (a.a.rows + ROWS_WG - 1) / ROWS_WG, n_tt = (a.T + TT - 1) / TT;
    return (size_t)((n_rb + N_XCD - 1) / N_XCD) * N_XCD * n_tt;
}

template <int TY, bool GATEUP, int NTM> static hipError_t launch_exact_n(const ExactArgs &a, hipStream_t st)
{
    const size_t grid = exact_grid<GATEUP, NTM>(a);
    if (grid > INT32_MAX) return hipErrorInvalidValue;
    k_exact<TY, GATEUP, NTM><<<(unsigned)grid, EX_NTH, 0, st>>>(a);
    return hipGetLastError();
}

template <int TY, bool GATEUP> static hipError_t launch_exact_t(const ExactArgs &a, hipStream_t st)
{
    if (a.T <= 16) return launch_exact_n<TY, GATEUP, 1>(a, st);
    // 64 input rows a workgroup convert a weight half as often, 32 leave a
    // smaller last round of workgroups: whichever takes less by the rounds of
    // resident workgroups (two per CU; three of 32-row Q8_0) and a round's
    // time (down 4096 x 12288, us: Q8_0 160 against 132, Q4_K and Q6_K 249
    // against 146).  Q8_0 gate/up 12288 x 4096 at T = 96 157 against 131, at
    // T = 128 164 against 172; down at T = 384 277 against 258, at T = 512 348
    // against 396.
    constexpr size_t PER2 = N_CU * (TY == T_Q8_0 ? 3 : 2), PER4 = N_CU * 2;
    const size_t r4 = (exact_grid<GATEUP, 4>(a) + PER4 - 1) / PER4, r2 = (exact_grid<GATEUP, 2>(a) + PER2 - 1) / PER2;
    if (a.T <= 32 || r2 * (TY == T_Q8_0 ? 10 : 7) < r4 * 12) return launch_exact_n<TY, GATEUP, 2>(a, st);
    return launch_exact_n<TY, GATEUP, 4>(a, st);
}

hipError_t launch_exact(const ExactArgs &a, int gateup, hipStream_t st)
{
    if (a.T <= 0) return hipSuccess;
    if (a.K % (2 * EX_KC) || a.a.rows % 32 || (size_t)a.K * 128 > UINT32_MAX || a.a.cols != a.K ||
        (gateup && (a.b.ty != a.a.ty || a.b.cols != a.K || a.b.rows != a.a.rows)))
        return hipErrorInvalidValue;
#define BIV_EX_CASE(TY)                                                                                         \
    if (a.a.ty == TY) return gateup ? launch_exact_t<TY, true>(a, st) : launch_exact_t<TY, false>(a, st);
    BIV_EX_CASE(T_Q8_0)
    BIV_EX_CASE(T_Q4K)
    BIV_EX_CASE(T_Q6K)
#undef BIV_EX_CASE
    return hipErrorInvalidValue;
}

static hipError_t launch_gu_t(MvArgs a, int routed, int shared, hipStream_t st)
{
    const DevMat &M = routed ? a.a : a.sa;
    if (!routed) a.u_max = 0;
    a.n_sh = shared ? (a.T + a.sh_chunk - 1) / a.sh_chunk : 0;
    const int slots = a.u_max + a.n_sh;
    if (slots == 0) return hipSuccess;
    if (a.sh_chunk > GS_ROWS || M.rows % GS_ROWS_WG) return hipErrorInvalidValue;
    a.n_rt = M.rows / GS_ROWS_WG;
    const dim3 grid(slot_grid<SLOT_RUN>(slots, a.n_rt));
    const bool dump = a.dump_a || a.dump_b;
#define BIV_GU_CASE(TY, KK)                                                                                     \
    if (M.ty == TY && M.cols == KK) {                                                                           \
        if (dump)                                                                                               \
            k_gu_slot<TY, KK, true><<<grid, GS_NTH, 0, st>>>(a);                                                 \
        else                                                                                                    \
            k_gu_slot<TY, KK, false><<<grid, GS_NTH, 0, st>>>(a);                                                \
        return hipGetLastError();                                                                               \
    }
    BIV_GU_CASE(T_Q8_0, 2048)
    BIV_GU_CASE(T_Q8_0, 1024)
    BIV_GU_CASE(T_Q8_0, 512)
    BIV_GU_CASE(T_Q4K, 2048)
    BIV_GU_CASE(T_Q4K, 1024)
    BIV_GU_CASE(T_Q4K, 512)
#undef BIV_GU_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_mfma_gateup_exact(const MvArgs &a, hipStream_t st)
{
    // routed and shared in one launch when they share a type and shape
    const bool has_shared = a.sa.q != nullptr;
    if (a.a.ty != a.b.ty || (has_shared && a.sa.ty != a.sb.ty)) return hipErrorInvalidValue;
    if (has_shared && a.sa.ty == a.a.ty && a.sa.cols == a.a.cols && a.sa.rows == a.a.rows)
        return launch_gu_t(a, 1, 1, st);
    hipError_t err = launch_gu_t(a, 1, 0, st);
    if (err != hipSuccess || !has_shared) return err;
    return launch_gu_t(a, 0, 1, st);
}

} // namespace biv
