// BF16 experts at prefill sizes on the matrix cores (gfx950 MFMA).
//
// biv's dot_bf16 (engine/src/quant.rs:1228-1256) multiplies bf16 weights by
// f32 activations in f32 FMA chains.  Here the activations are split into
// two bf16 halves, x = hi + lo + r with |r| <= 2^-17 |x| (hi = x rounded to
// bf16, lo = x - hi rounded to bf16), and each product w * hi and w * lo is
// exact in f32; v_mfma_f32_32x32x16_bf16 sums them in f32.  Only the order of
// the sums differs from the reference (bit-identical results come from the
// chain kernels in kernels.hip, which run decode sizes).
//
// Operand order: a 16-byte chunk c of a row holds the 8 elements
// 128 (c / 16) + 16 m + (c % 16), m = 0..7: the BF16 weight layout of
// layout.hpp (bf16_elem), so a lane's MFMA operand is one 16-byte load of the
// weights and one of each activation half.
#include <type_traits>

#include "common.hpp"
#include "layout.hpp"
#include "mfma_ops.hpp"

namespace biv {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ inline bf16x8 as_bf16x8(const uint4 &v) { return __builtin_bit_cast(bf16x8, v); }

// hi / lo bf16 halves of rows x [rows][K] in the chunk order above:
// xh[r][c] and xl[r][c] are 16-byte chunks.  One thread per chunk.
__global__ __launch_bounds__(256) void k_split_bf16(const float *__restrict__ x, int rows, int K,
                                                    uint4 *__restrict__ xh, uint4 *__restrict__ xl)
{
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nc = K / 8;
    if (idx >= (size_t)rows * nc) return;
    const size_t r = idx / nc;
    const int c = (int)(idx % nc), g = c / 16, L = c % 16;
    uint32_t h[8], lo[8];
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const float v = x[r * K + 128 * g + 16 * m + L];
        bf16_split(v, &h[m], &lo[m]);
    }
    xh[idx] = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
    xl[idx] = make_uint4(lo[0] | lo[1] << 16, lo[2] | lo[3] << 16, lo[4] | lo[5] << 16, lo[6] | lo[7] << 16);
}

// Grouped GEMM over the slots of the dispatch (the shared expert's first):
// a workgroup takes a whole slot (up to TOK_TILE pairs) and ROW_TILE output
// rows; wave (wt, wr) of the 4 x 2 grid takes 64 pairs x 64 rows of each of
// gate and up (gate/up) or 64 pairs x 128 rows (down), as 32 x 32 blocks, and
// skips the blocks of pairs past the slot's count.
// gate/up: each block has a gate and an up accumulator and the SwiGLU is
// formed in the epilogue.
//
// The row tiles of a slot go to one XCD (slot_unit): the slot's activation
// rows come from HBM once per slot and from that XCD's L2 after, and every
// expert's weights are read once per slot.
//
// K advances in stages of 32 (4 chunks, 64 bytes of a row).  A stage's tiles
// go straight from global memory into LDS (global_load_lds) into a ring of
// three buffers: the loads of the next two stages are in flight while the
// waves run this stage's MFMAs from LDS.  LDS layouts: A [half][pair][4], B
// [row][4], chunk c of row r in slot 4 r + (c ^ ((r >> 2) & 3)): the 64 lanes
// of a load write 64 consecutive slots, 4 lanes reading one row's 64
// contiguous bytes, and the swizzle keeps a fragment read (consecutive rows,
// one chunk) free of bank conflicts.
constexpr int NWT = 4;              // waves along the pairs
constexpr int NWR = 2;              // waves along the rows
constexpr int TOK_TILE = 64 * NWT;  // pairs of a workgroup
constexpr int NTH = 64 * NWT * NWR; // threads of a workgroup
constexpr int SK = 4;               // chunks per stage
static_assert(TOK_TILE == MFMA_TOK_TILE, "slot size");

template <int K, bool GATEUP>
__global__ __launch_bounds__(NTH) __attribute__((amdgpu_waves_per_eu(2, 8))) void k_mfma_bf16(MfArgs a)
{
    constexpr int NC = K / 8;          // chunks per row
    constexpr int NS = NC / SK;        // stages
    constexpr int NB = GATEUP ? 2 : 1; // weight matrices
    constexpr int RB = 4 / NB;         // 32-row blocks of a wave, per matrix
    constexpr int ROW_TILE = 32 * RB * NWR; // output rows of a workgroup
    constexpr int BR = ROW_TILE * NB;  // weight rows of a tile
    constexpr int A_SLOTS = 2 * SK * TOK_TILE, B_SLOTS = SK * BR;
    static_assert(A_SLOTS % NTH == 0 && B_SLOTS % NTH == 0, "tile shapes");
    // separate arrays: the compiler then tells the buffers a DMA writes apart
    // (one array would make it wait for every DMA before each LDS read)
    __shared__ uint4 sA0[A_SLOTS], sA1[A_SLOTS], sA2[A_SLOTS], sB0[B_SLOTS], sB1[B_SLOTS], sB2[B_SLOTS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 31, kg = lane >> 5;
    // the two waves of a SIMD (waves w and w + 4) take pairs 64 apart x 2
    const int wt = wave >> 1, wr = wave & 1;
    // workgroup -> (slot, row tile): ids b with one b % 8 are one XCD's
    int u, rt;
    if (!slot_unit<SLOT_RUN_BF16>(a, blockIdx.x, u, rt)) return;
    const bool shared = u < a.n_sh;
    int e = 0, beg, cnt, tok0 = 0;
    if (shared) {
        tok0 = u * a.sh_chunk;
        beg = a.P + tok0;
        cnt = min(a.sh_chunk, a.T - tok0);
    } else {
        const Slot sl = a.dp.slots[u - a.n_sh];
        if (sl.cnt == 0) return; // uniform over the workgroup
        e = sl.expert;
        beg = sl.beg;
        cnt = sl.cnt;
    }
    const DevMat &Ma = shared ? a.sa : a.a;
    const int rows = Ma.rows;
    const int r0 = rt * ROW_TILE;
    // this wave's 32-pair blocks that hold pairs of the slot
    const bool live0 = wt * 64 < cnt, live1 = wt * 64 + 32 < cnt;
    // this thread's load slots: slot tid + NTH q is row (tid + NTH q) / 4,
    // position tid % 4 (the chunk it loads is swizzled by the row); pairs
    // past the count load the slot's last pair (unused)
    constexpr int RQ = NTH / SK; // rows a pass of the threads covers
    const int p = tid % SK;
    const uint4 *srcA[2 * TOK_TILE / RQ];
    int swA[2 * TOK_TILE / RQ];
#pragma unroll
    for (int q = 0; q < 2 * TOK_TILE / RQ; q++) { // A rows: (half, pair)
        const int tr = (tid + NTH * q) / SK, hl = tr / TOK_TILE, tt = tr % TOK_TILE;
        const int ti = min(tt, cnt - 1);
        const size_t ar = GATEUP ? (size_t)(shared ? tok0 + ti : a.dp.pair_tok[beg + ti]) : (size_t)(beg + ti);
        srcA[q] = (hl ? a.xl : a.xh) + ar * NC;
        swA[q] = p ^ ((tt >> 2) & 3);
    }
    const uint4 *srcB[BR / RQ];
    int swB[BR / RQ];
#pragma unroll
    for (int q = 0; q < BR / RQ; q++) { // B rows: gate rows, then up rows
        const int br = (tid + NTH * q) / SK;
        const uint8_t *base = (GATEUP && br >= ROW_TILE) ? (shared ? a.sb.q : a.b.q) : Ma.q;
        srcB[q] = reinterpret_cast<const uint4 *>(base + ((size_t)e * rows + r0 + br % ROW_TILE) * K * 2);
        swB[q] = p ^ ((br >> 2) & 3);
    }
    auto lds_load = [](const uint4 *src, uint4 *dst_wave) {
        __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void *)dst_wave, 16, 0, 0);
    };
    // A load q of a thread covers pairs 128 (q & 1) .. + 127 of half q >> 1
    // (for every wave alike): a slot of at most 128 pairs (HALF) leaves out
    // the odd ones, which would only load its last pair again.  (Leaving out
    // each wave's loads that hold no pair of the slot, down to all of them,
    // measured no faster.)
    static_assert(A_SLOTS / NTH == 4 && NTH / SK == 128, "A loads by pair halves");
    auto issue = [&](int s, uint4 *sA, uint4 *sB, auto half_c) {
        constexpr bool HALF = decltype(half_c)::value;
#pragma unroll
        for (int q = 0; q < A_SLOTS / NTH; q++)
            if (!HALF || !(q & 1)) lds_load(srcA[q] + s * SK + swA[q], sA + NTH * q + 64 * wave);
#pragma unroll
        for (int q = 0; q < B_SLOTS / NTH; q++) lds_load(srcB[q] + s * SK + swB[q], sB + NTH * q + 64 * wave);
    };
    auto slot_of = [](int r, int c) { return SK * r + (c ^ ((r >> 2) & 3)); };
    f32x16 acc[2][RB][NB];
#pragma unroll
    for (int tb = 0; tb < 2; tb++)
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int q = 0; q < NB; q++)
#pragma unroll
                for (int j = 0; j < 16; j++) acc[tb][rb][q][j] = 0.0f;
    auto compute = [&](const uint4 *sA, const uint4 *sB) {
#pragma unroll
        for (int ks = 0; ks < SK / 2; ks++) {
            const int c = 2 * ks + kg;
            uint4 xa[2][2], wb[RB][NB];
#pragma unroll
            for (int tb = 0; tb < 2; tb++)
#pragma unroll
                for (int hl = 0; hl < 2; hl++)
                    if (tb ? live1 : live0) xa[tb][hl] = sA[slot_of(hl * TOK_TILE + wt * 64 + tb * 32 + li, c)];
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int q = 0; q < NB; q++) wb[rb][q] = sB[slot_of(q * ROW_TILE + wr * 32 * RB + rb * 32 + li, c)];
            // the halves outermost: consecutive MFMAs feed different
            // accumulators (an MFMA on the accumulator just written waits)
#pragma unroll
            for (int hl = 0; hl < 2; hl++)
#pragma unroll
                for (int tb = 0; tb < 2; tb++)
                    if (tb ? live1 : live0)
#pragma unroll
                    for (int rb = 0; rb < RB; rb++)
#pragma unroll
                        for (int q = 0; q < NB; q++)
                            acc[tb][rb][q] = GATEUP ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                                          as_bf16x8(wb[rb][q]), as_bf16x8(xa[tb][hl]), acc[tb][rb][q], 0, 0, 0)
                                                    : __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                                          as_bf16x8(xa[tb][hl]), as_bf16x8(wb[rb][q]), acc[tb][rb][q], 0, 0, 0);
        }
    };
    // three buffers, loads two stages ahead: stage s is in buffer s % 3
    auto run = [&](auto half_c) {
        constexpr bool HALF = decltype(half_c)::value;
        // loads of a stage, per thread
        constexpr int NLD = (HALF ? A_SLOTS / NTH / 2 : A_SLOTS / NTH) + B_SLOTS / NTH;
        // s_waitcnt immediates: vmcnt <= NLD (or 0) and lgkmcnt 0 (this
        // wave's LDS reads of the buffer the next loads overwrite are done)
        constexpr int WAIT_ONE_STAGE = (NLD & 15) | ((NLD >> 4) << 14) | (7 << 4);
        constexpr int WAIT_NONE_LEFT = 7 << 4;
        auto step = [&](int s, const uint4 *__restrict__ cA, const uint4 *__restrict__ cB, uint4 *__restrict__ nA,
                        uint4 *__restrict__ nB) {
            // this thread's loads of stage s are in (stage s + 1's may be in
            // flight); after the barrier every thread's are, and every wave
            // is done with stage s - 1, whose buffer stage s + 2 takes
            if (s + 1 < NS) __builtin_amdgcn_s_waitcnt(WAIT_ONE_STAGE);
            else __builtin_amdgcn_s_waitcnt(WAIT_NONE_LEFT);
            // a raw s_barrier (the compiler's barrier would wait for every
            // load) between compiler fences, so no LDS access moves across it
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (s + 2 < NS) issue(s + 2, nA, nB, half_c);
            compute(cA, cB);
        };
        issue(0, sA0, sB0, half_c);
        if (NS > 1) issue(1, sA1, sB1, half_c);
        int s = 0;
        for (; s + 3 <= NS; s += 3) {
            step(s, sA0, sB0, sA2, sB2);
            step(s + 1, sA1, sB1, sA0, sB0);
            step(s + 2, sA2, sB2, sA1, sB1);
        }
        if (s < NS) step(s, sA0, sB0, sA2, sB2);
        if (s + 1 < NS) step(s + 1, sA1, sB1, sA0, sB0);
    };
    // uniform over the workgroup (compute reads only the pairs below cnt)
    if (cnt <= TOK_TILE / 2) run(std::true_type());
    else run(std::false_type());
    // the exp table in LDS for the SwiGLU
    __shared__ uint64_t tab[GATEUP ? 32 : 1];
    if (GATEUP) {
        if (tid < 32) tab[tid] = exp_tab[tid];
        __syncthreads(); // (also: every wave is done with the ring)
    }
    // D of a 32 x 32 block.  gate/up (weights as A, the pairs as B): lane
    // (li, kg), registers 4 q .. 4 q + 3: weight rows 8 q + 4 kg .. 8 q + 4 kg
    // + 3 of the block, pair li: four consecutive outputs, one 16-byte store.
    // down (the pairs as A): register j is pair 8 (j / 4) + 4 kg + j % 4,
    // weight row li: a half wave stores 32 consecutive outputs (down's large
    // output keeps whole 128-byte segments that way; 16-byte stores across 32
    // rows measured slower)
    if constexpr (GATEUP) if (a.xo_h) {
        // the intermediate's bf16 hi / lo halves in the chunk order, as
        // k_split_bf16 forms them: the tile's SwiGLU values [pair][row]
        // through LDS (the ring's buffers, PA pairs' rows in each A buffer
        // and PB in each B buffer, EP floats apart), then 16-byte chunks:
        // this row tile is elements 128 rt .. 128 rt + 127 of each row, so
        // chunk 16 rt + L holds its rows 16 m + L
        constexpr int EP = 136, PA = A_SLOTS * 4 / EP, PB = B_SLOTS * 4 / EP;
        static_assert(ROW_TILE == 128, "one 128-element span per row tile");
        static_assert(3 * (PA + PB) >= TOK_TILE, "the tile fits in the ring");
        auto trow = [&](int p) -> float * {
            if (p < 3 * PA) {
                const int i = p / PA;
                return reinterpret_cast<float *>(i == 0 ? sA0 : i == 1 ? sA1 : sA2) + (p - PA * i) * EP;
            }
            const int i = (p - 3 * PA) / PB;
            return reinterpret_cast<float *>(i == 0 ? sB0 : i == 1 ? sB1 : sB2) + (p - 3 * PA - PB * i) * EP;
        };
#pragma unroll
        for (int tb = 0; tb < 2; tb++)
            if (tb ? live1 : live0)
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        float4 v;
                        v.x = silu_mul_t(acc[tb][rb][0][4 * q], acc[tb][rb][NB - 1][4 * q], tab);
                        v.y = silu_mul_t(acc[tb][rb][0][4 * q + 1], acc[tb][rb][NB - 1][4 * q + 1], tab);
                        v.z = silu_mul_t(acc[tb][rb][0][4 * q + 2], acc[tb][rb][NB - 1][4 * q + 2], tab);
                        v.w = silu_mul_t(acc[tb][rb][0][4 * q + 3], acc[tb][rb][NB - 1][4 * q + 3], tab);
                        *reinterpret_cast<float4 *>(trow(wt * 64 + tb * 32 + li) + wr * 32 * RB + rb * 32 + 8 * q +
                                                    4 * kg) = v;
                    }
        __syncthreads();
        const int nc = rows / 8;
        for (int x = tid; x < cnt * 16; x += NTH) {
            const int p = x >> 4, L = x & 15;
            uint32_t h[8], lo[8];
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const float v = trow(p)[16 * m + L];
                bf16_split(v, &h[m], &lo[m]);
            }
            const size_t c = (size_t)(beg + p) * nc + 16 * rt + L;
            a.xo_h[c] = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
            a.xo_l[c] = make_uint4(lo[0] | lo[1] << 16, lo[2] | lo[3] << 16, lo[4] | lo[5] << 16, lo[6] | lo[7] << 16);
        }
        return;
    }
    if constexpr (GATEUP) {
#pragma unroll
        for (int tb = 0; tb < 2; tb++) {
            const int ti = wt * 64 + tb * 32 + li;
            if (ti < cnt)
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int row = r0 + wr * 32 * RB + rb * 32 + 8 * q + 4 * kg;
                        float4 v;
                        v.x = silu_mul_t(acc[tb][rb][0][4 * q], acc[tb][rb][NB - 1][4 * q], tab);
                        v.y = silu_mul_t(acc[tb][rb][0][4 * q + 1], acc[tb][rb][NB - 1][4 * q + 1], tab);
                        v.z = silu_mul_t(acc[tb][rb][0][4 * q + 2], acc[tb][rb][NB - 1][4 * q + 2], tab);
                        v.w = silu_mul_t(acc[tb][rb][0][4 * q + 3], acc[tb][rb][NB - 1][4 * q + 3], tab);
                        *reinterpret_cast<float4 *>(a.out + (size_t)(beg + ti) * rows + row) = v;
                    }
        }
    } else {
        // pair ti's row starts (beg + ti) * rows floats in: one 64-bit base
        // per pair block and 32-bit offsets (j / 4) * 8 rows + (j % 4) rows,
        // not a 64-bit multiply per store
        const int r1 = rows, r8 = 8 * rows;
#pragma unroll
        for (int tb = 0; tb < 2; tb++) {
            const int t0 = wt * 64 + tb * 32 + 4 * kg;
            float *ob = a.out + (size_t)(beg + t0) * rows + r0 + wr * 32 * RB + li;
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    const int dt = (j / 4) * 8 + (j % 4);
                    if (t0 + dt < cnt) ob[(j / 4) * r8 + (j % 4) * r1 + rb * 32] = acc[tb][rb][0][j];
                }
        }
    }
}


// ---------------------------------------------------------------------------
// Q8_0 down matrices at prefill sizes on the int8 matrix cores.
//
// biv's dot_q8_0 (quant.rs:599-607, x86 1368-1382) sums, per row and input
// row, f16(d_w) * d_x * idot over the 32-element blocks, idot the exact int32
// dot of the block's int8 quants.  v_mfma_i32_16x16x32_i8 computes exactly
// those int32 block dots for 16 rows x 16 pairs at once (one block per
// instruction, so the dots stay apart); the scaling and the sum over blocks
// run in f32 on the vector ALU, in an order of their own.  Only the down
// matrices run here: their outputs go straight to the combine, so the other
// order moves them by rounding only.  gate/up outputs are quantised again
// (the down input), where a rounding difference can move a quant by one
// step; gate/up therefore keeps the x86 order (the chain kernels).
//
// Operands: a block's 32 quants as lanes (x, kq) see them, kq = 0..3 taking
// bytes 8 kq .. 8 kq + 7, for weights and activations alike.  In the chain
// layout (layout.hpp) the 16-byte unit 16 g + 8 pi + w of a row holds word w
// of the blocks 8 g + pi + 2 j, j = 0..3, so lane kq loads units 2 kq and
// 2 kq + 1 of each parity (32 contiguous bytes) and finds its 8 bytes of
// block j in word j of the two.
//
// A workgroup takes a slot (up to QT pairs, staged in LDS: quants and block
// scales) and QW waves of QR rows each; a wave streams its rows' blocks from
// HBM half a group (4 blocks of each row) ahead.  D of an MFMA: lane (n, kq)
// holds row n, pairs 4 kq .. 4 kq + 3 of the 16-pair tile.
constexpr int QW = 8;            // waves of a workgroup
constexpr int QT = MFMA_Q8_TILE; // pairs of a slot
constexpr int NTT = QT / 16;     // 16-pair tiles of a slot
constexpr int QNTH = QW * 64;
constexpr int QRT = 2;           // 16-row tiles of a wave
constexpr int Q_ROWS_WG = QW * 16 * QRT;

template <int K, bool DUMP>
__global__ __launch_bounds__(QNTH) void k_q8_down_mfma(MvArgs a)
{
    constexpr int RT = QRT;
    constexpr int NG = K / 256; // groups of 8 blocks
    constexpr int NB = K / 32;
    constexpr int XSTR = K / 16 + 1; // staged quant row: 16-byte units (+1 against bank conflicts)
    constexpr int DSTR = QT + 4;     // staged scales [block][pair], floats
    __shared__ uint4 xq_s[QT * XSTR];
    __shared__ float xd_s[NB * DSTR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, kq = lane >> 4;
    int u, rt;
    if (!slot_unit<SLOT_RUN>(a, blockIdx.x, u, rt)) return;
    const bool shared = u < a.n_sh;
    int e = 0, beg, cnt;
    if (shared) {
        const int tok0 = u * a.sh_chunk;
        beg = a.P + tok0;
        cnt = min(a.sh_chunk, a.T - tok0);
    } else {
        const Slot sl = a.dp.slots[u - a.n_sh];
        if (sl.cnt == 0) return; // uniform over the workgroup
        e = sl.expert;
        beg = sl.beg;
        cnt = sl.cnt;
    }
    const DevMat &M = shared ? a.sa : a.a;
    const int rows = M.rows;
    // the weight rows of this lane: row n of each 16-row tile
    const int rw0 = rt * Q_ROWS_WG + wave * 16 * RT;
    const uint4 *wq[RT];
    const uint2 *wsc[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const size_t row = (size_t)e * rows + rw0 + 16 * r + n;
        wq[r] = reinterpret_cast<const uint4 *>(M.q + row * K) + 2 * kq;
        wsc[r] = reinterpret_cast<const uint2 *>(M.s + row * NB * 2);
    }
    // half-group h = (g, pi)'s weights: per tile two units of quants and 4
    // f16 scales (blocks 8 g + pi + 2 j)
    struct Half {
        uint4 q[RT][2];
        uint2 s[RT];
    };
    auto load = [&](int h, Half &w) {
        const int g = h >> 1, pi = h & 1;
#pragma unroll
        for (int r = 0; r < RT; r++) {
            w.q[r][0] = wq[r][16 * g + 8 * pi];
            w.q[r][1] = wq[r][16 * g + 8 * pi + 1];
            w.s[r] = wsc[r][(pi * (K / 64) + 4 * g) / 4];
        }
    };
    Half w0, w1;
    load(0, w0); // the first weights go out before the staging waits
    // stage the slot's input rows: quants (chain layout, row stride XSTR
    // units) and block scales transposed to [block][pair]; pairs past the
    // count repeat the last one (their results are not stored)
    {
        constexpr int UPR = K / 16; // units per row
        static_assert((QT * UPR) % QNTH == 0, "staging shape");
#pragma unroll
        for (int it = 0; it < QT * UPR / QNTH; it++) {
            const int idx = tid + QNTH * it, i = idx / UPR, c = idx % UPR;
            const size_t ar = beg + min(i, cnt - 1);
            xq_s[i * XSTR + c] = reinterpret_cast<const uint4 *>(a.xq + ar * K)[c];
        }
        for (int idx = tid; idx < QT * NB; idx += QNTH) {
            const int i = idx / NB, bs = idx % NB;
            const size_t ar = beg + min(i, cnt - 1);
            const int b = 2 * (bs % (K / 64)) + bs / (K / 64); // lay::q8_scale's inverse
            xd_s[b * DSTR + i] = a.xd[ar * NB + bs];
        }
    }
    __syncthreads();
    float acc[NTT][RT][4];
#pragma unroll
    for (int t = 0; t < NTT; t++)
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[t][r][j] = 0.0f;
    auto compute = [&](int h, const Half &w) {
        const int g = h >> 1, pi = h & 1;
#pragma unroll
        for (int t = 0; t < NTT; t++) {
            if (16 * t >= cnt) break; // uniform: no pairs in this tile
            // this lane's activation units of the half-group
            const uint4 *xr = xq_s + (16 * t + n) * XSTR + 16 * g + 8 * pi + 2 * kq;
            const uint4 x0 = xr[0], x1 = xr[1];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int b = 8 * g + pi + 2 * j;
                const float4 dx = *reinterpret_cast<const float4 *>(xd_s + b * DSTR + 16 * t + 4 * kq);
                const long xo = (long)((uint64_t)x0[j] | (uint64_t)x1[j] << 32);
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    const uint32_t h2 = j < 2 ? w.s[r].x : w.s[r].y;
                    const float dw = f16_to_f32((j & 1) ? h2 >> 16 : h2 & 0xFFFF);
                    const long wo = (long)((uint64_t)w.q[r][0][j] | (uint64_t)w.q[r][1][j] << 32);
                    const i32x4 z = {0, 0, 0, 0};
                    const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(xo, wo, z, 0, 0, 0);
                    acc[t][r][0] = __builtin_fmaf((float)d[0], dx.x * dw, acc[t][r][0]);
                    acc[t][r][1] = __builtin_fmaf((float)d[1], dx.y * dw, acc[t][r][1]);
                    acc[t][r][2] = __builtin_fmaf((float)d[2], dx.z * dw, acc[t][r][2]);
                    acc[t][r][3] = __builtin_fmaf((float)d[3], dx.w * dw, acc[t][r][3]);
                    if (DUMP && a.dump_a) { // the block dots, for the taps
#pragma unroll
                        for (int jj = 0; jj < 4; jj++) {
                            const int i = 16 * t + 4 * kq + jj;
                            if (i < cnt) a.dump_a[((size_t)(beg + i) * rows + rw0 + 16 * r + n) * NB + b] = d[jj];
                        }
                    }
                }
                // keep each block's MFMA results short-lived (registers for
                // more waves rather than for MFMAs in flight)
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // two half-groups per turn, loads one ahead
    for (int h = 0; h < 2 * NG; h += 2) {
        load(h + 1, w1);
        compute(h, w0);
        if (h + 2 < 2 * NG) load(h + 2, w0);
        compute(h + 1, w1);
    }
    // pair 16 t + 4 kq + j of the slot, row rw0 + 16 r + n
#pragma unroll
    for (int t = 0; t < NTT; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int i = 16 * t + 4 * kq + j;
            if (i < cnt) {
#pragma unroll
                for (int r = 0; r < RT; r++) a.out[(size_t)(beg + i) * rows + rw0 + 16 * r + n] = acc[t][r][j];
            }
        }
}


// ---------------------------------------------------------------------------
// Q6_K down matrices at prefill sizes on the int8 matrix cores.
//
// biv's dot_q6k (quant.rs:651-686, x86 1475-1533) weighs each 16-element
// half of a 32-element block by its own int8 sub-scale: isum = sc_0 *
// dot16_0 + sc_1 * dot16_1 (exact int32), then d * d_x * isum.  Here
// v_mfma_i32_16x16x32_i8 takes A = one block of 8 input rows, each twice:
// A row 2 t + hh keeps only half hh of input row t (lanes kq = 2 hh, 2 hh + 1
// hold that half's bytes); B = the block of 16 weight rows as q - 32.  D row
// 2 t + hh, column n is dot16_hh of input row t and weight row n, exactly,
// and lane (n, kq) holds both halves of input rows 2 kq and 2 kq + 1: isum
// in integers, then the f32 scaling; the sum over blocks runs in an order of
// its own (down's outputs only meet the combine): d_x * isum summed over a
// super-block's eight blocks, times its d once.
//
// Weights (chain layout, layout.hpp): per 512 elements (four halves qq of a
// row) the ql units 16 (qq / 4) + 8 pi + w hold ql word w of quarters pi and
// pi + 2 of each half, the qh units 8 (qq / 4) + w qh word w; lane kq loads
// words 2 kq and 2 kq + 1, i.e. bytes 8 kq .. 8 kq + 7 of every block.
template <int K, bool DUMP>
__global__ __launch_bounds__(QNTH) void k_q6k_down_mfma(MvArgs a)
{
    constexpr int RT = QRT;
    constexpr int NB = K / 32;
    constexpr int NQ = K / 512;      // groups of four halves
    constexpr int XSTR = K / 16 + 1; // staged quant row: 16-byte units (+1 against bank conflicts)
    constexpr int DSTR = QT + 4;     // staged scales [block][pair], floats
    static_assert(K % 512 == 0 && QT % 8 == 0, "shapes");
    __shared__ uint4 xq_s[(QT + 1) * XSTR]; // the slot's rows, then a row of zeros
    __shared__ float xd_s[NB * DSTR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, kq = lane >> 4;
    int u, rt;
    if (!slot_unit<SLOT_RUN>(a, blockIdx.x, u, rt)) return;
    const bool shared = u < a.n_sh;
    int e = 0, beg, cnt;
    if (shared) {
        const int tok0 = u * a.sh_chunk;
        beg = a.P + tok0;
        cnt = min(a.sh_chunk, a.T - tok0);
    } else {
        const Slot sl = a.dp.slots[u - a.n_sh];
        if (sl.cnt == 0) return; // uniform over the workgroup
        e = sl.expert;
        beg = sl.beg;
        cnt = sl.cnt;
    }
    const DevMat &M = shared ? a.sa : a.a;
    const int rows = M.rows;
    const int rw0 = rt * Q_ROWS_WG + wave * 16 * RT;
    // this lane's weight words of group gq, per row tile
    uint4 ql[RT][2][2], qh[RT][2];
    int4 scv[RT][2];
    float dsb[RT][2];
    auto load_group = [&](int gq) {
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const size_t row = (size_t)e * rows + rw0 + 16 * r + n;
            const uint8_t *base = M.q + row * (K / 256) * 192;
            const uint4 *pl = reinterpret_cast<const uint4 *>(base);
            const uint4 *ph = reinterpret_cast<const uint4 *>(base + (K / 256) * 128);
#pragma unroll
            for (int pi = 0; pi < 2; pi++)
#pragma unroll
                for (int w = 0; w < 2; w++) ql[r][pi][w] = pl[16 * gq + 8 * pi + 2 * kq + w];
#pragma unroll
            for (int w = 0; w < 2; w++) qh[r][w] = ph[8 * gq + 2 * kq + w];
            // sub-scales of the group's 16 blocks: [pi][hsel] runs of K / 64
            const int8_t *sc = reinterpret_cast<const int8_t *>(M.s + row * (K / 16));
#pragma unroll
            for (int c = 0; c < 2; c++) {
                // scv[r][c]: bytes [pi = c][hsel = 0 / 1][s = 8 gq .. + 7] as two int2 halves
                const uint2 s0 = *reinterpret_cast<const uint2 *>(sc + (2 * c + 0) * (K / 64) + 8 * gq);
                const uint2 s1 = *reinterpret_cast<const uint2 *>(sc + (2 * c + 1) * (K / 64) + 8 * gq);
                scv[r][c] = make_int4((int)s0.x, (int)s0.y, (int)s1.x, (int)s1.y);
            }
            const uint16_t *dp = reinterpret_cast<const uint16_t *>(M.d + row * (K / 256) * 2);
            dsb[r][0] = f16_to_f32(dp[2 * gq]);
            dsb[r][1] = f16_to_f32(dp[2 * gq + 1]);
        }
    };
    // the first group's weights go out before the staging waits
    load_group(0);
    // stage the slot's input rows (as the Q8_0 down kernel)
    {
        constexpr int UPR = K / 16;
        for (int idx = tid; idx < QT * UPR; idx += QNTH) {
            const int i = idx / UPR, c = idx % UPR;
            const size_t ar = beg + min(i, cnt - 1);
            xq_s[i * XSTR + c] = reinterpret_cast<const uint4 *>(a.xq + ar * K)[c];
        }
        for (int c = tid; c < XSTR; c += QNTH) xq_s[QT * XSTR + c] = make_uint4(0u, 0u, 0u, 0u);
        for (int idx = tid; idx < QT * NB; idx += QNTH) {
            const int i = idx / NB, bs = idx % NB;
            const size_t ar = beg + min(i, cnt - 1);
            const int b = 2 * (bs % (K / 64)) + bs / (K / 64); // lay::q8_scale's inverse
            xd_s[b * DSTR + i] = a.xd[ar * NB + bs];
        }
    }
    __syncthreads();
    // A row 2 t + hh keeps only half hh, bytes 16 hh .. 16 hh + 15: lanes
    // kq = 2 hh and 2 hh + 1 read them, the other lanes the row of zeros
    // (no masking per block)
    const bool keep = (n & 1) == (kq >> 1);
    const int at = n >> 1; // A row's input row within the 8-row group
    const uint4 *const xrow = keep ? xq_s + at * XSTR : xq_s + QT * XSTR;
    const int xtstr = keep ? 8 * XSTR : 0; // from one 8-row group to the next
    // acc: the sum over super-blocks of d * (the super-block's sum over its
    // blocks of d_x * isum, in asb)
    float acc[QT / 8][RT][2], asb[QT / 8][RT][2];
#pragma unroll
    for (int t = 0; t < QT / 8; t++)
#pragma unroll
        for (int r = 0; r < RT; r++) acc[t][r][0] = acc[t][r][1] = 0.0f;
    for (int gq = 0; gq < NQ; gq++) {
        if (gq > 0) load_group(gq);
#pragma unroll
        for (int bl = 0; bl < 16; bl++) { // block b = 16 gq + bl: half qq = 4 gq + bl / 4, quarter k = bl % 4
            const int qq = bl >> 2, k = bl & 3, pi = k & 1, hi = k >> 1;
            const int b = 16 * gq + bl;
            const int s2 = 2 * (4 * gq + qq) + hi; // the sub-scale step of (pi, hsel)
            // B: q - 32 of words 2 kq, 2 kq + 1 of block b, per row tile
            long wo[RT];
            int sc0[RT], sc1[RT];
#pragma unroll
            for (int r = 0; r < RT; r++) {
                uint32_t wv[2];
#pragma unroll
                for (int w = 0; w < 2; w++) {
                    // each byte's high bits 2 k, 2 k + 1 of qh moved to bits 4, 5
                    const uint32_t lo = (ql[r][pi][w][qq] >> (4 * hi)) & 0x0F0F0F0Fu;
                    const uint32_t qv = qh[r][w][qq];
                    const uint32_t hs = k <= 2 ? qv << (4 - 2 * k) : qv >> (2 * k - 4);
                    const uint32_t x = (hs & 0x30303030u) | lo;
                    // bytewise q - 32: q + 96 carries out of no byte, and
                    // flipping bit 7 then subtracts 128 mod 256
                    wv[w] = (x + 0x60606060u) ^ 0x80808080u;
                }
                wo[r] = (long)((uint64_t)wv[0] | (uint64_t)wv[1] << 32);
                const int sidx = s2 - 8 * gq; // 0..7 within the group's run
                const int4 sv = scv[r][pi];
                const uint32_t w0 = sidx < 4 ? (uint32_t)sv.x : (uint32_t)sv.y;
                const uint32_t w1 = sidx < 4 ? (uint32_t)sv.z : (uint32_t)sv.w;
                sc0[r] = (int)(int8_t)((w0 >> (8 * (sidx & 3))) & 0xFF);
                sc1[r] = (int)(int8_t)((w1 >> (8 * (sidx & 3))) & 0xFF);
            }
            // the activations' block b: chain layout unit 16 g + 8 pi + w, word j
            const int g = b >> 3, xpi = b & 1, j = (b >> 1) & 3;
#pragma unroll
            for (int t = 0; t < QT / 8; t++) {
                if (8 * t >= cnt) break; // uniform
                const uint4 *xr = xrow + t * xtstr + 16 * g + 8 * xpi + 2 * kq;
                const uint32_t lo = xr[0][j], hi2 = xr[1][j];
                const long xo = (long)((uint64_t)lo | (uint64_t)hi2 << 32);
                const float2 dx = *reinterpret_cast<const float2 *>(xd_s + b * DSTR + 8 * t + 2 * kq);
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    const i32x4 z = {0, 0, 0, 0};
                    const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(xo, wo[r], z, 0, 0, 0);
                    // 24-bit products (full rate; |dot16| <= 16 * 128 * 32,
                    // sub-scales int8): the same integers as 32-bit ones
                    const int is0 = __mul24(sc0[r], d[0]) + __mul24(sc1[r], d[1]);
                    const int is1 = __mul24(sc0[r], d[2]) + __mul24(sc1[r], d[3]);
                    asb[t][r][0] = (bl & 7) ? __builtin_fmaf((float)is0, dx.x, asb[t][r][0]) : (float)is0 * dx.x;
                    asb[t][r][1] = (bl & 7) ? __builtin_fmaf((float)is1, dx.y, asb[t][r][1]) : (float)is1 * dx.y;
                    if ((bl & 7) == 7) {
                        const float dd = dsb[r][qq >> 1];
                        acc[t][r][0] = __builtin_fmaf(dd, asb[t][r][0], acc[t][r][0]);
                        acc[t][r][1] = __builtin_fmaf(dd, asb[t][r][1], acc[t][r][1]);
                    }
                    if (DUMP && a.dump_a) { // the block int32s, for the taps
                        const int i0 = 8 * t + 2 * kq, row = rw0 + 16 * r + n;
                        if (i0 < cnt) a.dump_a[((size_t)(beg + i0) * rows + row) * NB + b] = is0;
                        if (i0 + 1 < cnt) a.dump_a[((size_t)(beg + i0 + 1) * rows + row) * NB + b] = is1;
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // input rows 8 t + 2 kq + c, row rw0 + 16 r + n
#pragma unroll
    for (int t = 0; t < QT / 8; t++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int i = 8 * t + 2 * kq + c;
            if (i < cnt) {
#pragma unroll
                for (int r = 0; r < RT; r++) a.out[(size_t)(beg + i) * rows + rw0 + 16 * r + n] = acc[t][r][c];
            }
        }
}

} // namespace

hipError_t launch_split_bf16(const float *x, int rows, int K, void *xh, void *xl, hipStream_t st)
{
    const size_t n = (size_t)rows * (K / 8);
    if (n == 0) return hipSuccess;
    k_split_bf16<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(x, rows, K, static_cast<uint4 *>(xh),
                                                                static_cast<uint4 *>(xl));
    return hipGetLastError();
}

template <bool GATEUP> hipError_t launch_mfma_t(MfArgs a, int routed, int shared, hipStream_t st)
{
    const DevMat &M = routed ? a.a : a.sa;
    if (!routed) a.u_max = 0;
    a.n_sh = shared ? (a.T + a.sh_chunk - 1) / a.sh_chunk : 0;
    const int slots = a.u_max + a.n_sh;
    if (slots == 0) return hipSuccess;
    const int row_tile = 32 * NWR * (GATEUP ? 2 : 4);
    if (M.rows % row_tile) return hipErrorInvalidValue;
    if (a.chunk > TOK_TILE || a.sh_chunk > TOK_TILE) return hipErrorInvalidValue;
    a.n_rt = M.rows / row_tile;
    const dim3 grid(slot_grid<SLOT_RUN_BF16>(slots, a.n_rt));
#define BIV_MF_CASE(KK)                                                                                         \
    if (M.cols == KK) {                                                                                         \
        k_mfma_bf16<KK, GATEUP><<<grid, NTH, 0, st>>>(a);                                                       \
        return hipGetLastError();                                                                               \
    }
    BIV_MF_CASE(2048)
    BIV_MF_CASE(1024)
    BIV_MF_CASE(512)
#undef BIV_MF_CASE
    return hipErrorInvalidValue;
}

template <bool GATEUP> hipError_t launch_mfma(const MfArgs &a, hipStream_t st)
{
    // every matrix BF16 (the caller checks); routed and shared in one launch
    // when they share a shape
    const bool has_shared = a.sa.q != nullptr;
    if (has_shared && a.sa.cols == a.a.cols && a.sa.rows == a.a.rows) return launch_mfma_t<GATEUP>(a, 1, 1, st);
    hipError_t err = launch_mfma_t<GATEUP>(a, 1, 0, st);
    if (err != hipSuccess || !has_shared) return err;
    return launch_mfma_t<GATEUP>(a, 0, 1, st);
}

hipError_t launch_mfma_gateup(const MfArgs &a, hipStream_t st) { return launch_mfma<true>(a, st); }
hipError_t launch_mfma_down(const MfArgs &a, hipStream_t st) { return launch_mfma<false>(a, st); }


hipError_t launch_q8_down_t(MvArgs a, int routed, int shared, hipStream_t st)
{
    const DevMat &M = routed ? a.a : a.sa;
    if (!routed) a.u_max = 0;
    a.n_sh = shared ? (a.T + a.sh_chunk - 1) / a.sh_chunk : 0;
    const int slots = a.u_max + a.n_sh;
    if (slots == 0) return hipSuccess;
    if (a.sh_chunk > QT || M.rows % Q_ROWS_WG) return hipErrorInvalidValue;
    a.n_rt = M.rows / Q_ROWS_WG;
    const dim3 grid(slot_grid<SLOT_RUN>(slots, a.n_rt));
#define BIV_Q8_CASE(KK)                                                                                         \
    if (M.cols == KK) {                                                                                         \
        if (a.dump_a)                                                                                           \
            k_q8_down_mfma<KK, true><<<grid, QNTH, 0, st>>>(a);                                                 \
        else                                                                                                    \
            k_q8_down_mfma<KK, false><<<grid, QNTH, 0, st>>>(a);                                                \
        return hipGetLastError();                                                                               \
    }
    if (M.ty == T_Q8_0) {
        BIV_Q8_CASE(2048)
        BIV_Q8_CASE(1024)
        BIV_Q8_CASE(512)
    }
#undef BIV_Q8_CASE
#define BIV_Q6_CASE(KK)                                                                                         \
    if (M.cols == KK) {                                                                                         \
        if (a.dump_a)                                                                                           \
            k_q6k_down_mfma<KK, true><<<grid, QNTH, 0, st>>>(a);                                                \
        else                                                                                                    \
            k_q6k_down_mfma<KK, false><<<grid, QNTH, 0, st>>>(a);                                               \
        return hipGetLastError();                                                                               \
    }
    if (M.ty == T_Q6K) {
        BIV_Q6_CASE(2048)
        BIV_Q6_CASE(1024)
        BIV_Q6_CASE(512)
    }
#undef BIV_Q6_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_q8_mfma_down(const MvArgs &a, hipStream_t st)
{
    const bool has_shared = a.sa.q != nullptr;
    if (has_shared && a.sa.ty == a.a.ty && a.sa.cols == a.a.cols && a.sa.rows == a.a.rows)
        return launch_q8_down_t(a, 1, 1, st);
    hipError_t err = launch_q8_down_t(a, 1, 0, st);
    if (err != hipSuccess || !has_shared) return err;
    return launch_q8_down_t(a, 0, 1, st);
}

} // namespace biv
