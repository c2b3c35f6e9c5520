// gdn_prefill_model.hip -- the many-row matmul and the causal attention of
// the hybrid model's prefill (include/kai_gdn_hybrid.h) for gfx950.
//
// Prefill GEMM: y[m][n] = scale[n] sum_k x[m][k] Wq[n][k] for M rows (a
// whole prompt), on the same pre-tiled int8 weights as the decode GEMM
// (gdn_model.hip, w8f_tile_kernel) -- the M > 1 counterpart of the
// reference e2e loop's gemm_int8_neon (gdn_e2e_decode.c:606-612).  Persistent
// blocks of 64, 128 or 256 rows x 256 channels (w8t_kernel), k in steps of
// 64, 32x32x16 fp16 MFMA (the larger MFMA shape delivers about 1.5 times the
// 16x16x32 rate on gfx950); both operands reach LDS by DMA, the weights as
// int8, widened to fp16 (exactly) on their way into the MFMA.  The weight is
// the A operand, so a lane's accumulators hold runs of 4 consecutive channels
// of one row, and the interleaved gate/up rows put each gate channel and its
// up channel in the same lane.  Few rows leave most CUs without a tile: their
// k-steps are split over blocks (w8t_choose).
//
// Prefill attention: Qwen3_5Attention's causal softmax(q k^T / 16) v with
// the sigmoid output gate (modeling_qwen3_5.py:629-701), GQA, head dim 256,
// on the model's fp16 KV cache.  Block (64 positions, kv head), 8 waves: wave
// w takes query head kv * rep + (w % 4) at positions +32 (w / 4) .. +31, as
// two 16-query tiles, and walks the keys in blocks of 64 shared through LDS
// (K and a transposed copy of V, both moved by DMA).  Scores on fp16 MFMA
// 16x16x32 as S^T = K q^T (A = the 16-key x 32-dim fragment, which is one
// contiguous 1 KB of the tiled K cache; B = the tile's queries), online
// softmax in exp2 per query column, then O^T = V^T P^T with P taken from the
// score registers as the B operand (the 8 keys a lane holds, 4g .. 4g+3 and
// 16 + 4g .. 16 + 4g+3, permute the k index of both operands alike).  Each K
// and V fragment read from LDS feeds both query tiles.
#include <algorithm>
#include <climits>

#include "gdn_common.h"
#include "gdn_internal.h"

namespace gdn {
namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int kPBN = 256;                       // channels per block
constexpr int kPScratch = 512;                  // epilogue scratch, floats per wave (2 KB)
constexpr size_t kPPartWave = 2 * 16 * 64;      // floats of a wave's split partial per row tile

// LDS index (halves) of the 16-byte piece `piece` of activation row `row`
GDN_DEV int dswz(int row, int piece) { return row * 64 + ((piece ^ ((row >> 1) & 7)) << 3); }
// wait until at most N vector memory operations of this wave are outstanding
template <int N> GDN_DEV void wait_vm() { __builtin_amdgcn_s_waitcnt((N & 15) | 0x0F70 | ((N >> 4) << 14)); }
// LDS DMA: lane l's 16 bytes at base + off[l] go to lds + 16 l (lds uniform).
// Written as asm so that the compiler does not count it against the LDS reads
// of the other ring slots (it would wait for every DMA before them); the
// kernel's own wait_vm and barriers order it.  The compiler does not see that
// the asm reads base in a vector memory operation, which takes five wait
// states after a readfirstlane: base is derived by scalar arithmetic from what
// dma_bases returned.  (With the wait states in here the GEMM is 3% slower.)
GDN_DEV void dma16(const void *base, uint32_t off, uint32_t lds) {
    __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base)
                     : "memory", "m0");
}
template <typename A, typename B> GDN_DEV void dma_bases(const A *&a, const B *&b) {
    __asm__ volatile("s_nop 4" : "+s"(a), "+s"(b));
}
GDN_DEV int scalar(int x) { return __builtin_amdgcn_readfirstlane(x); }
GDN_DEV uint32_t lds_addr(const void *p) { return (uint32_t)(uintptr_t)(const lds_void_t *)p; }
// barrier that waits for this wave's LDS operations only (not for its DMA)
GDN_DEV void lds_bar() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), as a builtin: the compiler drops its own waits for what it covers
    __asm__ volatile("s_barrier" ::: "memory");
}
// silu(y) * up in fp32, the decode GEMM's arithmetic.  Of gate|up's time at
// 20000 rows (1592 us) it is 4%; a hardware exp2 and reciprocal without
// expf's reduction and the division take 1532 us and are off by up to 22 ulp
// (this form 2.7), NaN where y is infinite.
GDN_DEV float silu_mul(float y, float up) { return y / (1.0f + expf(-y)) * up; }

// Epilogues of a wave's 32 IT rows x 64 channels (per row tile two 32x32
// accumulator tiles; lane l holds, for q = 0..3, channels 32 jt + 8 q + 4 (l
// / 32) .. +3 of row l % 32).  Each tile crosses the wave's scratch, so that
// a row is stored as 128 contiguous bytes (SwiGLU: 64): stored from the
// accumulators, every store instruction would touch 32 rows with 32 (16)
// bytes each.  kW8tAdd is kW8Segments with one segment and a residual; its
// loads run one row tile ahead of the stores (vector memory operations
// complete in order, so a load behind a store would wait for it).
enum W8tMode : int { kW8tSegments = 0, kW8tAdd = 1, kW8tSwiGLU = 2 };
template <int IT, int MODE>
GDN_DEV void w8t_epilogue(const f32x16_t (&acc)[IT][2], float *scratch, int row0, int nc,
                          const float *__restrict__ scale, int M, int N, const W8Out &out) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, h2 = lane >> 5;
    if constexpr (MODE == kW8tSwiGLU) {
        // 16-channel groups: 8 gate channels (q even), then their 8 up channels (q + 1)
        f32x4_t sg[2][2], su[2][2];
#pragma unroll
        for (int jt = 0; jt < 2; ++jt)
#pragma unroll
            for (int q2 = 0; q2 < 2; ++q2) {
                const int n = nc + 32 * jt + 16 * q2 + 4 * h2;
                sg[jt][q2] = *reinterpret_cast<const f32x4_t *>(scale + n);
                su[jt][q2] = *reinterpret_cast<const f32x4_t *>(scale + n + 8);
            }
#pragma unroll
        for (int it = 0; it < IT; ++it) {
#pragma unroll
            for (int jt = 0; jt < 2; ++jt)
#pragma unroll
                for (int q2 = 0; q2 < 2; ++q2) {
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        o[e] = silu_mul(acc[it][jt][8 * q2 + e] * sg[jt][q2][e],
                                        acc[it][jt][8 * q2 + 4 + e] * su[jt][q2][e]);
                    // a row's 32 outputs are four 16-byte pieces: piece 2 jt + q2, half h2
                    const int slot = (2 * jt + q2) ^ ((l32 >> 2) & 3);
                    *reinterpret_cast<uint2 *>(scratch + l32 * 16 + slot * 4 + 2 * h2) =
                        make_uint2((uint32_t)f32_to_f16_rne(o[0]) | ((uint32_t)f32_to_f16_rne(o[1]) << 16),
                                   (uint32_t)f32_to_f16_rne(o[2]) | ((uint32_t)f32_to_f16_rne(o[3]) << 16));
                }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int rr = 16 * i + (lane >> 2), pc = lane & 3, row = row0 + 32 * it + rr;
                const u32x4_t v = *reinterpret_cast<const u32x4_t *>(scratch + rr * 16 + ((pc ^ ((rr >> 2) & 3)) << 2));
                if (row < M) *reinterpret_cast<u32x4_t *>(out.x16 + (size_t)row * (N / 2) + nc / 2 + 8 * pc) = v;
            }
        }
    } else {
        const int pc = lane & 7;  // the lane's four channels (of each 32) on the way out
        f32x4_t sc[2];
        float *dst[2];
        int ld[2];
        bool ok[2];  // channels past the last segment: padding
#pragma unroll
        for (int jt = 0; jt < 2; ++jt) {
            const int n = nc + 32 * jt + 4 * pc;
            sc[jt] = *reinterpret_cast<const f32x4_t *>(scale + n);
            ok[jt] = n < out.seg[out.nseg - 1].n_end;
            int nb = 0;
            dst[jt] = out.seg[0].dst;
            ld[jt] = out.seg[0].ld;
            if constexpr (MODE == kW8tSegments) {
#pragma unroll
                for (int qq = 1; qq < kW8MaxSegs; ++qq)
                    if (qq < out.nseg && n >= out.seg[qq - 1].n_end) {
                        nb = out.seg[qq - 1].n_end;
                        dst[jt] = out.seg[qq].dst;
                        ld[jt] = out.seg[qq].ld;
                    }
            }
            dst[jt] += n - nb;
        }
        // the residual of row tile it (rows past M and padding read an
        // element in bounds, never stored); it may be in place: each element
        // is read and written by one lane
        f32x4_t res[2][8];
        auto load_res = [&](int it) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int jt = j >> 2, row = min(row0 + 32 * it + 8 * (j & 3) + (lane >> 3), M - 1);
                res[it & 1][j] = *reinterpret_cast<const f32x4_t *>(
                    out.add_in + (size_t)row * out.add_ld + (ok[jt] ? nc + 32 * jt + 4 * pc : 0));
            }
        };
        if constexpr (MODE == kW8tAdd) load_res(0);
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            if constexpr (MODE == kW8tAdd)
                if (it + 1 < IT) load_res(it + 1);
#pragma unroll
            for (int jt = 0; jt < 2; ++jt)
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    if ((l32 >> 4) == half)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            *reinterpret_cast<f32x4_t *>(scratch + (l32 & 15) * 32 + (((2 * q + h2) ^ (l32 & 7)) << 2)) =
                                f32x4_t{acc[it][jt][4 * q], acc[it][jt][4 * q + 1], acc[it][jt][4 * q + 2],
                                        acc[it][jt][4 * q + 3]};
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const int rr = 8 * i + (lane >> 3), row = row0 + 32 * it + 16 * half + rr;
                        f32x4_t y =
                            *reinterpret_cast<const f32x4_t *>(scratch + rr * 32 + ((pc ^ (rr & 7)) << 2)) * sc[jt];
                        if constexpr (MODE == kW8tAdd) y = res[it & 1][4 * jt + 2 * half + i] + y;
                        // pinned ahead of the branch: a load that is waited for only inside it would
                        // leave the compiler a wait for every DMA at the head of the main loop
                        __asm__ volatile("" : "+v"(y));
                        if (row < M && ok[jt]) *reinterpret_cast<f32x4_t *>(dst[jt] + (size_t)row * ld[jt]) = y;
                    }
                }
        }
    }
}

// The launch's work units: below `full`, unit u is one output tile over all
// of K; from there, part (u - full) % S of the k-steps of tile full +
// (u - full) / S, its sums going to `part` unscaled for w8t_reduce_kernel.
// Blocks take units blockIdx, blockIdx + grid, ...; unit u runs on XCD u % 8
// (blocks are handed out round robin; the grid is 256, or, below 256 units,
// the unit count, and then no block takes a second one).
struct W8tPlan {
    int tiles_m, tiles_n, full, S, units, grid;
};
// First k-step of part sp of S.
GDN_DEV int w8t_part(int ksteps, int sp, int S) { return ksteps / S * sp + min(sp, ksteps % S); }
// Tile index of a unit -> (row block, channel block).  Each XCD takes a
// contiguous range of the whole tiles, four row blocks at a time, so that
// the tiles its CUs work on at once share activation and weight tiles in
// its L2.  S splits of a tile go to different XCDs, the same k-range of
// neighbouring tiles to the same one.
GDN_DEV void w8t_tile(const W8tPlan &p, int t, int &tm, int &tn) {
    const int n = p.full / 8;
    if (t < 8 * n) t = (t % 8) * n + t / 8;
    const int per = 4 * p.tiles_n, gi = t / per, r = t - gi * per;
    const int h = min(4, p.tiles_m - gi * 4);
    tn = r / h;
    tm = gi * 4 + r - tn * h;
}

// Block 64 IT rows x 256 channels (IT = 4, 2, 1), 8 waves as 2 x 4 (32 IT
// rows x 64 channels each: IT x 2 tiles of 32x32x16 fp16 MFMA), persistent
// over its units.  Both operands of a 64-k step reach LDS by DMA (1 KB per
// wave instruction): the activation rows and the four 4 KB weight tiles of
// the block's channel groups, copied as they lie, into a ring of three
// steps; the DMA runs two steps ahead, across unit boundaries.  An
// activation row is 128 B; its 16-byte piece p sits in slot p ^ ((row / 2) %
// 8), so that the 16 rows a quarter-wave reads cover all 64 banks.  The
// weights are widened to fp16 from LDS.  Lane l of a 32-channel MFMA tile
// reads, from 16-row weight tile 2 jt + (l % 32) / 16, row l % 16 and the
// 16-byte pieces g' = l / 32 and l / 32 + 2 of the 64-k step (k 16 g' ..
// +15); MFMA kk (4 per step) takes 8 of them: k = 32 (kk / 2) + 16 (l / 32)
// + 8 (kk % 2) .. +7, and the activation (B) lanes read the same k.
//
// What bounds it: at 256 rows the MFMA pipes under the chip's power limit
// (zero operands run the 4B down matrix at 20000 rows in 616 us, random ones
// in 845: the clock drops to 1.7 GHz), below that the latency of a step's
// load half.  At 20000 rows against the kernel with one block per tile and a
// store from the accumulators: gate|up 1842 -> 1616 us (fp32 out, 1168
// TFLOP/s), in 1274 -> 1100, down 935 -> 753 (with the split last round; 845
// without), out 451 -> 360; at 333 rows, down 106 -> 33 us (83 without the
// split over k).  hipBLASLt's fp16 GEMM on the same shapes: 1515, 974, 822.
//
// Schedule, IT = 4: the waves of wave row 0 (one per SIMD) and of wave row 1
// (the other one of each SIMD) run half a phase apart.  A phase is 32 k: first
// its LDS reads, the weights' widening and the DMA requests ("load"), then
// its 4 IT MFMAs ("multiply"), with a barrier after each half, so that on
// every SIMD one wave multiplies while the other loads.  Ring safety, group
// 0 half a phase ahead: the DMA of step s + 2 goes into the slot of step
// s - 1, issued by group 0 in its load of (s, 0), one barrier after group
// 1's load of (s - 1, 1) waited for its LDS reads; and every wave waits for
// its own part of step s + 1 at the end of its load of (s, 1), which for
// group 1 is one barrier before group 0's load of (s + 1, 0).
// IT < 4: a phase's 4 IT MFMAs do not cover another wave's load half (0.83
// us a step at IT = 2 that way, 0.69 this way), so each wave reads and widens
// a phase ahead between its own MFMAs, with one barrier per step: the slot of
// step s - 1 was last read before step s - 1's barrier, and the barrier of
// step s follows every wave's wait for its part of step s + 1.  The ring is 4
// (IT = 2) or 6 steps deep, what LDS holds.
template <int IT, int MODE>
__device__ __forceinline__ void w8t_body(const uint16_t *__restrict__ X, int ldx, const int8_t *__restrict__ W,
                                         const float *__restrict__ scale, int M, int N, int K, const W8tPlan &plan,
                                         float *__restrict__ part, const W8Out &out) {
    constexpr int BM = 64 * IT;
    constexpr int kRing = IT == 4 ? 3 : IT == 2 ? 4 : 6;  // steps of LDS (144, 128, 144 KB)
    __shared__ __align__(16) uint16_t xs[kRing * BM * 64];
    __shared__ __align__(16) int8_t ws[kRing * 4 * 4096];
    __shared__ __align__(16) float scratch[8 * kPScratch];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 2, wn = wave & 3;  // waves w and w + 4 share a SIMD: one of each wave row
    const int l32 = lane & 31, h2 = lane >> 5;
    const int ksteps = K / 64;
    // a unit's tile and k-steps
    struct Unit {
        int m0, n0, s0, s1;
    };
    auto unit_of = [&](int u) {
        const bool split = u >= plan.full;
        const int v = u - plan.full;
        const int sp = split ? v % plan.S : 0;
        int tm, tn;
        w8t_tile(plan, split ? plan.full + v / plan.S : u, tm, tn);
        return Unit{tm * BM, tn * kPBN, split ? w8t_part(ksteps, sp, plan.S) : 0,
                    split ? w8t_part(ksteps, sp + 1, plan.S) : ksteps};
    };

    // ---- the DMA's cursor: the next step of unit du -------------------------
    // activations: instruction i of wave w moves rows 8 (IT w + i) .. +7
    // (rows past M read row M - 1, never stored); weights: wave w moves
    // kilobytes 2w and 2w + 1 of the block's four 4 KB group tiles (group
    // w / 2, absent groups re-read group 0)
    int du = blockIdx.x, left;  // steps of unit du not requested yet, the next one included
    const uint16_t *xnext;
    const int8_t *wnext;
    uint32_t xoff[IT];
    const uint32_t loff = lane * 16;
    auto dma_unit = [&]() {
        const Unit t = unit_of(du);
        left = scalar(t.s1 - t.s0);
        const int wg = t.n0 / 64 + (wave >> 1) < N / 64 ? t.n0 / 64 + (wave >> 1) : 0;
        const int r0 = min(t.m0 + 8 * IT * wave, M - 1);  // the wave's first row
        xnext = X + (size_t)scalar(r0) * ldx + (size_t)scalar(t.s0) * 64;
        wnext = W + ((size_t)scalar(wg) * ksteps + scalar(t.s0)) * 4096 + (2 * wave & 3) * 1024;
        dma_bases(xnext, wnext);
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int row = 8 * i + (lane >> 3);  // of the wave's 8 IT
            const int piece = (lane & 7) ^ (((8 * IT * wave + row) >> 1) & 7);
            xoff[i] = ((uint32_t)min(row, M - 1 - r0) * (uint32_t)ldx + piece * 8) * 2;
        }
    };
    const uint32_t xl = lds_addr(xs) + (uint32_t)(IT * wave) * 1024, wl = lds_addr(ws) + (uint32_t)(2 * wave) * 1024;
    auto dma_x = [&](int slot) {
#pragma unroll
        for (int i = 0; i < IT; ++i) dma16(xnext, xoff[i], xl + (uint32_t)(slot * (BM * 128) + i * 1024));
    };
    auto dma_w = [&](int slot) {
#pragma unroll
        for (int i = 0; i < 2; ++i) dma16(wnext + i * 1024, loff, wl + (uint32_t)(slot * 16384 + i * 1024));
    };
    auto dma_advance = [&]() {
        if (left > 1) {
            --left;
            xnext += 64;
            wnext += 4096;
        } else if (du + plan.grid < plan.units) {
            du += plan.grid;
            dma_unit();
        }  // past the last unit its last step is read again (in bounds, never used)
    };

    f32x16_t acc[IT][2];
    // MFMA operands of a phase (32 k, two 16-k MFMA groups)
    struct Frags {
        u32x4_t raw[2];
        f16x8_t a[2][2], bx[2][IT];
    };
    const int woff = wn * 4096 + (l32 >> 4) * 1024 + (16 * h2 + (l32 & 15)) * 16;
    auto lds_read = [&](Frags &f, int phase, int slot) {
        const int8_t *wb = ws + slot * 16384 + woff + phase * 512;
        const uint16_t *xb = xs + slot * (BM * 64);
#pragma unroll
        for (int jt = 0; jt < 2; ++jt) f.raw[jt] = *reinterpret_cast<const u32x4_t *>(wb + jt * 2048);
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
            for (int it = 0; it < IT; ++it)
                f.bx[k2][it] = *reinterpret_cast<const f16x8_t *>(
                    &xb[dswz(32 * IT * wm + 32 * it + l32, 4 * phase + 2 * h2 + k2)]);
        __builtin_amdgcn_sched_barrier(0);  // every read requested before anything waits for one
    };
    auto widen = [&](Frags &f) {
#pragma unroll
        for (int jt = 0; jt < 2; ++jt) i8x16_to_f16(f.raw[jt], f.a[jt][0], f.a[jt][1]);
    };
    auto mult = [&](const Frags &f) {
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
            for (int jt = 0; jt < 2; ++jt)
#pragma unroll
                for (int it = 0; it < IT; ++it)
                    acc[it][jt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[jt][k2], f.bx[k2][it], acc[it][jt], 0, 0, 0);
    };
    // IT = 4: the load half (reads already requested) and the multiply half of a phase
    auto half_phases = [&](Frags &f) {
        widen(f);
        __builtin_amdgcn_sched_barrier(0);  // the widening belongs to the load half
        lds_bar();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
        mult(f);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        lds_bar();
    };
    // IT < 4: a phase's multiplies, the next phase's weights widened between them
    auto mult_widen = [&](const Frags &f, Frags &next) {
        mult(f);
        widen(next);
        // the first MFMAs cover the reads, then the widening goes between the rest
        __builtin_amdgcn_sched_group_barrier(0x008, IT, 0);
#pragma unroll
        for (int i = 0; i < 3 * IT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x002, (40 + 3 * IT - 1) / (3 * IT), 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
    };

    dma_unit();
#pragma unroll
    for (int i = 0; i < kRing - 1; ++i) {
        dma_x(i);
        dma_w(i);
        dma_advance();
    }
    wait_vm<(kRing - 2) * (IT + 2)>();  // the first step landed
    lds_bar();
    Frags fa, fb;
    int slot = 0, fill = kRing - 1;  // ring slots of the step multiplied and of the last step requested
    if constexpr (IT == 4) {
        if (wm == 1) lds_bar();  // half a phase behind
    } else {
        lds_read(fa, 0, 0);
        widen(fa);
    }
    for (int u = blockIdx.x; u < plan.units; u += plan.grid) {
        const Unit t = unit_of(u);
#pragma unroll
        for (int it = 0; it < IT; ++it)
#pragma unroll
            for (int jt = 0; jt < 2; ++jt)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[it][jt][e] = 0.f;
        for (int n = t.s1 - t.s0; n > 0; --n) {
            const int nslot = slot == kRing - 1 ? 0 : slot + 1;
            if constexpr (IT == 4) {
                lds_read(fa, 0, slot);
                dma_x(fill);
                half_phases(fa);
                lds_read(fa, 1, slot);
                dma_w(fill);
                dma_advance();
                wait_vm<(kRing - 2) * (IT + 2)>();
                half_phases(fa);
            } else {
                lds_read(fb, 1, slot);
                dma_x(fill);
                dma_w(fill);
                dma_advance();
                mult_widen(fa, fb);
                wait_vm<(kRing - 2) * (IT + 2)>();
                lds_bar();  // the step's reads are done, the next step's tiles are there
                lds_read(fa, 0, nslot);
                mult_widen(fb, fa);
            }
            fill = slot;
            slot = nslot;
        }
        if (u >= plan.full) {
            float *pp = part + ((size_t)(u - plan.full) * 8 + wave) * (IT * kPPartWave) + lane * 4;
#pragma unroll
            for (int it = 0; it < IT; ++it)
#pragma unroll
                for (int jt = 0; jt < 2; ++jt)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<f32x4_t *>(pp + ((it * 2 + jt) * 4 + q) * 256) = f32x4_t{
                            acc[it][jt][4 * q], acc[it][jt][4 * q + 1], acc[it][jt][4 * q + 2], acc[it][jt][4 * q + 3]};
        } else if (t.n0 / 64 + wn < N / 64) {
            w8t_epilogue<IT, MODE>(acc, scratch + wave * kPScratch, t.m0 + 32 * IT * wm, t.n0 + 64 * wn, scale, M, N,
                                   out);
        }
    }
    if constexpr (IT == 4)
        if (wm == 0) lds_bar();
    wait_vm<0>();  // no DMA in flight into LDS the block gives back
}

template <int IT, int MODE>
__global__ __launch_bounds__(512, 1) void w8t_kernel(const uint16_t *__restrict__ X, int ldx,
                                                     const int8_t *__restrict__ W, const float *__restrict__ scale,
                                                     int M, int N, int K, W8tPlan plan, float *__restrict__ part,
                                                     W8Out out) {
    w8t_body<IT, MODE>(X, ldx, W, scale, M, N, K, plan, part, out);
}

// Sums the S parts of every split tile in part order and runs the tile's
// epilogue, with the multiplying kernel's wave and lane mapping: one wave per
// block (split tile, 8 it + wave), so that the few tiles of a small problem
// spread over the chip (with eight waves a block, 30 tiles of 128 rows in 8
// parts took 8.6 us; 60 tiles of 64 rows in 4 parts take 5.4), kParts parts' loads in flight together.
template <int IT, int MODE>
__global__ __launch_bounds__(64) void w8t_reduce_kernel(const float *__restrict__ part,
                                                        const float *__restrict__ scale, int M, int N,
                                                        W8tPlan plan, W8Out out) {
    constexpr int kParts = 4;
    __shared__ __align__(16) float scratch[kPScratch];
    const int lane = threadIdx.x;
    const int wave = blockIdx.y & 7, it = blockIdx.y >> 3;
    const int wm = wave >> 2, wn = wave & 3;
    int tm, tn;
    w8t_tile(plan, plan.full + blockIdx.x, tm, tn);
    const int nc = tn * kPBN + 64 * wn, row0 = tm * 64 * IT + 32 * (IT * wm + it);
    if (nc >= N || row0 >= M) return;
    const float *pp =
        part + ((size_t)blockIdx.x * plan.S * 8 + wave) * (IT * kPPartWave) + it * kPPartWave + lane * 4;
    f32x16_t acc[1][2];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[0][jt][e] = 0.f;
    for (int s0 = 0; s0 < plan.S; s0 += kParts) {
        f32x4_t y[kParts][8];
#pragma unroll
        for (int s = 0; s < kParts; ++s)
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (s0 + s < plan.S)
                    y[s][q] = *reinterpret_cast<const f32x4_t *>(pp + (size_t)(s0 + s) * 8 * (IT * kPPartWave) + q * 256);
#pragma unroll
        for (int s = 0; s < kParts; ++s)
            if (s0 + s < plan.S)
#pragma unroll
                for (int q = 0; q < 8; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[0][q >> 2][4 * (q & 3) + e] += y[s][q][e];
    }
    w8t_epilogue<1, MODE>(acc, scratch, row0, nc, scale, M, N, out);
}

// ---- causal prefill attention ------------------------------------------------

constexpr int kApQ = 64;       // positions per block
constexpr int kApK = 64;       // keys per step
constexpr int kApD = 256;      // head dim

// V^T tile in LDS: [256 dims][64 keys], 128 bytes per dim row, the 16-byte
// piece c of row d in slot c ^ (d % 8): a fragment read (16 rows x 32
// bytes) then covers every bank twice, the minimum.
GDN_DEV int vt_slot(int d, int c) { return d * kApK + ((c ^ (d & 7)) << 3); }

// Block (64 positions, kv head), 8 waves: wave w takes query head
// kv * rep + (w % 4) at positions +32 (w / 4) .. +31, as two 16-query tiles
// that share every K and V fragment the wave reads from LDS (two MFMAs per
// fragment read, against one with a tile per wave: the LDS reads bounded
// that form).  K (the cache's tiled layout, 32 KB per step, contiguous) and
// V^T (from the transposed copy) reach LDS by DMA, double buffered.  The DMA
// is dma16's: as a builtin on one two-slot array the compiler waited for the
// next step's tiles before this step's first LDS read, and so did queries
// still in flight at the loop (20000 positions: 4.39 -> 4.12 ms a layer, 0.80
// PFLOP/s counting the causal half).  What bounds it now: two waves per SIMD
// whose LDS reads, MFMAs and softmax hide each other only in part (running
// the two position halves half a phase apart, as the GEMM does, took 4.26).
constexpr int kApT = 2;  // query tiles per wave
constexpr int kApThreads = 512;

__global__ __launch_bounds__(kApThreads) void attn_prefill_kernel(
    const uint16_t *__restrict__ q16, const uint16_t *__restrict__ Kc, const uint16_t *__restrict__ vT,
    const float *__restrict__ gate, int gate_row, uint16_t *__restrict__ out16, int T, int Hq, int Hkv, int Tmax,
    int Tv, float sc_log2) {
    __shared__ __align__(16) uint16_t ks[2][kApK * kApD];  // tiled as in the cache
    __shared__ __align__(16) uint16_t vs[2][kApD * kApK];  // [dim][key], swizzled pieces
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: the DMA addresses stay in SGPRs
    const int g = lane >> 4, r = lane & 15;
    const int qb = (int)gridDim.x - 1 - (int)blockIdx.x;  // longest blocks first
    const int kv = blockIdx.y;
    const int rep = Hq / Hkv;
    {  // sequence blockIdx.z of the launch
        const size_t z = blockIdx.z;
        q16 += z * T * Hq * kApD;
        out16 += z * T * Hq * kApD;
        gate += z * T * gate_row;
        Kc += z * Hkv * Tmax * kApD;
        vT += z * Hkv * kApD * Tv;
    }
    const bool live = (wave & 3) < rep;                   // wave-uniform
    const int h = kv * rep + min(wave & 3, rep - 1);
    int qpos[kApT];
#pragma unroll
    for (int qt = 0; qt < kApT; ++qt) qpos[qt] = qb * kApQ + 32 * (wave >> 2) + 16 * qt + r;  // B column r

    // the wave's queries as B operands: dims 32 j + 8 g .. +7 of query r
    f16x8_t qf[kApT][8];
#pragma unroll
    for (int qt = 0; qt < kApT; ++qt) {
        const uint16_t *qp = q16 + ((size_t)min(qpos[qt], T - 1) * Hq + h) * kApD + 8 * g;
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[qt][j] = *reinterpret_cast<const f16x8_t *>(qp + 32 * j);
    }
    f32x4_t o[kApT][16];  // O^T per tile: dims 16 dt + 4 g + e of query r
#pragma unroll
    for (int qt = 0; qt < kApT; ++qt)
#pragma unroll
        for (int dt = 0; dt < 16; ++dt) o[qt][dt] = zero4();
    // running max (log2 units, all lanes of column r agree) and partial sum, per tile
    float m[kApT], l[kApT];
#pragma unroll
    for (int qt = 0; qt < kApT; ++qt) {
        m[qt] = -INFINITY;
        l[qt] = 0.f;
    }

    const int kend = min(T, qb * kApQ + kApQ);
    const int nkb = (kend + kApK - 1) / kApK;
    const uint16_t *kbase = Kc + (size_t)kv * Tmax * kApD;
    const uint16_t *vbase = vT + (size_t)kv * kApD * Tv;
    // DMA of step kb into buffer b: wave w moves K kilobytes 4w .. 4w+3 (of
    // 16-key group w / 2: a group past the cache rows reads the last group
    // instead, its keys are masked, every key >= T lies after every query)
    // and V^T rows 32 w .. 32 w + 31 (8 per instruction)
    // per-lane parts of the DMA addresses (loop-invariant): K chunk lane of a
    // kilobyte; V^T row lane / 8 of an 8-row group (whose first row is a
    // multiple of 8, so the row's swizzle is (lane / 8) % 8), piece lane % 8
    const uint32_t koff = lane * 16, voff = 2u * ((lane >> 3) * (uint32_t)Tv + 8 * ((lane & 7) ^ (lane >> 3)));
    const uint32_t kl = lds_addr(ks) + 4096u * wave, vl = lds_addr(vs) + 4096u * wave;
    auto dma = [&](int kb, int b) {
        const int t0 = min(kb * kApK + 16 * (wave >> 1), Tmax - 16);
        const uint16_t *kp = kbase + (size_t)t0 * kApD + (4 * (wave & 1)) * 512;
        const uint16_t *vp = vbase + (size_t)(32 * wave) * Tv + kb * kApK;
        dma_bases(kp, vp);
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16(kp + i * 512, koff, kl + 32768u * b + 1024u * i);
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16(vp + (size_t)(8 * i) * Tv, voff, vl + 32768u * b + 1024u * i);
    };
    // One step: the 64 keys of buffer b as two halves of 32, each an online
    // softmax update (scores, P, then P V), so that one half's scores and P
    // fragments are live at a time (registers).
    auto step = [&](int b, int kb) {
        if (!live) return;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            // S^T tiles: keys kb * 64 + 32 half + 16 kh + 4 g + e, query r of tile qt
            f32x4_t s[kApT][2];
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) {
                const int kt = 2 * half + kh;
#pragma unroll
                for (int qt = 0; qt < kApT; ++qt) s[qt][kh] = zero4();
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const f16x8_t kf = *reinterpret_cast<const f16x8_t *>(&ks[b][kt * 4096 + j * 512 + lane * 8]);
#pragma unroll
                    for (int qt = 0; qt < kApT; ++qt)
                        s[qt][kh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[qt][j], s[qt][kh], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);  // one key tile's fragments in flight at a time
            }
            f16x8_t pb[kApT];  // P^T fragments: keys 32 half + {4g .. 4g+3, 16 + 4g .. 16 + 4g+3}
#pragma unroll
            for (int qt = 0; qt < kApT; ++qt) {
                float mx = m[qt];
#pragma unroll
                for (int kh = 0; kh < 2; ++kh)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int key = kb * kApK + 32 * half + 16 * kh + 4 * g + e;
                        const float v = key <= qpos[qt] ? s[qt][kh][e] * sc_log2 : -INFINITY;
                        s[qt][kh][e] = v;
                        mx = fmaxf(mx, v);
                    }
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                mx = fmaxf(mx, __shfl_xor(mx, 32));
                // the first half of the first step holds key 0, which precedes
                // every query: mx is finite from then on (a later fully
                // masked half leaves m and alpha = 1 unchanged)
                const float alpha = __builtin_amdgcn_exp2f(m[qt] - mx);
                m[qt] = mx;
                // once the running maxima settle, alpha is 1 in every lane: skip
                // the 64 multiplies of O (x * 1 = x, so the result is the same)
                if (__ballot(alpha != 1.0f)) {
                    l[qt] *= alpha;
#pragma unroll
                    for (int dt = 0; dt < 16; ++dt) o[qt][dt] *= alpha;
                }
#pragma unroll
                for (int kh = 0; kh < 2; ++kh)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float p = __builtin_amdgcn_exp2f(s[qt][kh][e] - mx);
                        l[qt] += p;
                        pb[qt][kh * 4 + e] = (_Float16)p;
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
            // per-lane V^T offsets of this half, recomputed here (a few VALU
            // operations) rather than kept live across the step: row r, keys
            // 32 half + 4 g .. +3 (piece 4 half + g / 2, half g % 2) and 16
            // keys further (piece + 2); row 16 dt + r adds 1024 dt
            int vlo, vhi;
            {
                int ln = lane;
                __asm__ volatile("" : "+v"(ln));
                const int gg = ln >> 4, rr = ln & 15;
                vlo = vt_slot(rr, 4 * half + (gg >> 1)) + 4 * (gg & 1);
                vhi = vt_slot(rr, 4 * half + 2 + (gg >> 1)) + 4 * (gg & 1);
            }
#pragma unroll
            for (int dt = 0; dt < 16; ++dt) {
                const uint16_t *vb = &vs[b][1024 * dt];  // rows 16 dt + r keep their swizzle (16 dt % 8 = 0)
                const u32x2_t lo = *reinterpret_cast<const u32x2_t *>(vb + vlo);
                const u32x2_t hi = *reinterpret_cast<const u32x2_t *>(vb + vhi);
                const f16x8_t a = __builtin_bit_cast(f16x8_t, u32x4_t{lo[0], lo[1], hi[0], hi[1]});
#pragma unroll
                for (int qt = 0; qt < kApT; ++qt)
                    o[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, pb[qt], o[qt][dt], 0, 0, 0);
                if ((dt & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // four V fragments in flight
            }
        }
    };

    dma(0, 0);
    wait_vm<0>();
    lds_bar();
    // the queries land here: waited for at their first use, every step would
    // wait for its own prefetch
#pragma unroll
    for (int qt = 0; qt < kApT; ++qt)
#pragma unroll
        for (int j = 0; j < 8; ++j) __asm__ volatile("" : "+v"(qf[qt][j]));
    for (int kb = 0; kb < nkb; ++kb) {
        if (kb + 1 < nkb) dma(kb + 1, (kb + 1) & 1);  // into the buffer step kb - 1 read
        step(kb & 1, kb);
        wait_vm<0>();
        lds_bar();
    }
    if (!live) return;
#pragma unroll
    for (int qt = 0; qt < kApT; ++qt) {
        // lanes of one query column agree on qpos, so the shuffles stay within active lanes
        if (qpos[qt] >= T) continue;
        float lt = l[qt];
        lt += __shfl_xor(lt, 16);
        lt += __shfl_xor(lt, 32);
        const float inv = 1.0f / lt;
        const float *gp = gate + (size_t)qpos[qt] * gate_row + (size_t)h * 512;
        uint16_t *op = out16 + ((size_t)qpos[qt] * Hq + h) * kApD;
#pragma unroll
        for (int dt = 0; dt < 16; ++dt) {
            const int d = 16 * dt + 4 * g;
            const f32x4_t gt = *reinterpret_cast<const f32x4_t *>(gp + d);
            uint32_t hv[2];
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                const float a = (o[qt][dt][e] * inv) * (1.0f / (1.0f + expf(-gt[e])));
                const float b = (o[qt][dt][e + 1] * inv) * (1.0f / (1.0f + expf(-gt[e + 1])));
                hv[e / 2] = (uint32_t)f32_to_f16_rne(a) | ((uint32_t)f32_to_f16_rne(b) << 16);
            }
            *reinterpret_cast<uint2 *>(op + d) = make_uint2(hv[0], hv[1]);
        }
    }
}

}  // namespace

long long w8p_max_rows() { return 65535LL * 256; }

namespace {

constexpr int kW8tBlocks = 256;              // one block per CU
constexpr int kW8tMaxSplits = 8;
constexpr int kW8tMinSteps = 4;              // k-steps of a split part at least
constexpr int kW8tTailRows = 4096;           // rows from which only the last round's tiles are split
constexpr size_t kW8tPartBytes = 384u << 20; // partial sums of one launch at most

struct W8tChoice {
    int it = 1;
    W8tPlan plan{};
    size_t need = 0;  // bytes of partials with which the same split is chosen (any row tile fits them)
};

// A plan counts in int: its units are at most kW8tMaxSplits per 64 x 256 tile.
bool w8t_counts_fit(int M, int N) {
    return M <= w8p_max_rows() && ((M + 63LL) / 64) * ((N + kPBN - 1LL) / kPBN) <= INT_MAX / kW8tMaxSplits;
}
// Rows that the 32-bit offsets of a wave's DMA reach (its last 16-byte piece
// lies 112 bytes into a 64-k step); a wave of a 64 IT-row tile takes 8 IT.
long long w8t_wave_rows(int ldx) { return ((1LL << 32) - 113) / (2LL * ldx) + 1; }
W8tPlan w8t_plan(int M, int N, int it, int S, bool tail) {
    W8tPlan p{};
    p.tiles_m = (M + 64 * it - 1) / (64 * it);
    p.tiles_n = (N + kPBN - 1) / kPBN;
    const int tiles = p.tiles_m * p.tiles_n;
    p.full = S == 1 ? tiles : tail ? tiles / kW8tBlocks * kW8tBlocks : 0;
    p.S = S;
    p.units = p.full + (tiles - p.full) * S;
    p.grid = std::min(p.units, kW8tBlocks);
    return p;
}
size_t w8t_part_bytes(const W8tPlan &p, int it) {
    return (size_t)(p.units - p.full) * 8 * it * kPPartWave * sizeof(float);
}
// Modelled time (us) of a plan, from sweeps over the 4B matrices at 64 to
// 20000 rows: a 64-k step of a block takes 1.05 / 0.68 / 0.54 us (IT = 4, 2,
// 1) with few blocks on the chip and 1.5 / 0.92 / 0.65 us with all 256 (the
// power limit lowers the clock), a tile's epilogue about IT us, a split
// launch its second kernel and its partial sums written and read at about
// 4.5 TB/s.  The model ranks the measured plans as they measured within 10%.
double w8t_cost(const W8tPlan &p, int it, int ksteps) {
    const int i = it == 4 ? 2 : it - 1;
    const double few[3] = {0.54, 0.68, 1.05}, all[3] = {0.65, 0.92, 1.5};
    const double load = (double)p.grid / kW8tBlocks, step = few[i] + (all[i] - few[i]) * load;
    const int split_units = p.units - p.full;
    const int rounds = (p.full + kW8tBlocks - 1) / kW8tBlocks;
    double t = rounds * (ksteps * step + it);
    if (split_units > 0) {
        const int parts = (split_units + kW8tBlocks - 1) / kW8tBlocks;
        t += parts * ((ksteps + p.S - 1) / p.S * step + it) + 3.0 + 2.0 * w8t_part_bytes(p, it) / 4.5e6;
    }
    return t;
}
// The row tile (64 IT) and the k-splits of M rows made of sequences of
// `seq_rows` rows each, at most max_rows together.  The split decides the
// order of a sum, so it is chosen without M (a sequence's result does not
// depend on how many sequences it is batched with).  Its price: a group whose
// tiles fill the chip still writes and sums the parts that one of its
// sequences alone wants (16 prompts of 200 rows through the 4B model 31 ms,
// modelled 25 without; one after another, each as its own launch, 172).
// Below kW8tTailRows every tile is split alike, the row tile does not change a
// bit, and it is chosen for M.  From there (where a launch holds one sequence)
// only the tiles left over after the whole rounds of 256 are split: the row
// tile decides which rows those are, and it is the one that the split was
// chosen with.
W8tChoice w8t_choose(int M, int seq_rows, int max_rows, int N, int K, int ldx, size_t part_limit) {
    const int ksteps = K / 64;
    const bool tail = seq_rows >= kW8tTailRows;
    part_limit = std::min(part_limit, kW8tPartBytes);
    const auto it_fits = [&](int it) { return std::min(8 * it, M) <= w8t_wave_rows(ldx); };
    int S = 1;
    size_t need = 0;
    double best = 1e30;
    for (int s = 1; s <= kW8tMaxSplits && (s == 1 || ksteps / s >= kW8tMinSteps); ++s)
        for (int it = 1; it <= 4; it *= 2) {
            if (!it_fits(it)) continue;
            // 256-row tiles bound the padded rows of every IT
            const W8tPlan worst = w8t_plan(tail ? seq_rows : max_rows, N, tail ? it : 4, s, tail);
            if (s > 1 && w8t_part_bytes(worst, tail ? it : 4) > part_limit) continue;
            const double c = w8t_cost(w8t_plan(seq_rows, N, it, s, tail), it, ksteps);
            if (c < best) {
                best = c;
                S = s;
                need = s > 1 ? w8t_part_bytes(worst, tail ? it : 4) : 0;
            }
        }
    W8tChoice r;
    best = 1e30;
    for (int it = 1; it <= 4; it *= 2) {
        if (!it_fits(it)) continue;
        const W8tPlan p = w8t_plan(M, N, it, S, tail);
        const size_t pb = w8t_part_bytes(p, it);
        const double c = w8t_cost(p, it, ksteps);
        if (pb <= part_limit && c < best) {
            best = c;
            r = W8tChoice{it, p, need};
        }
    }
    return r;
}

template <int IT, int MODE>
hipError_t w8t_run(const uint16_t *x, int ldx, const int8_t *W, const float *scale, int M, int N, int K,
                   const W8tPlan &p, float *part, const W8Out &out, hipStream_t st) {
    w8t_kernel<IT, MODE><<<p.grid, 512, 0, st>>>(x, ldx, W, scale, M, N, K, p, part, out);
    const int split = p.tiles_m * p.tiles_n - p.full;
    if (split > 0) w8t_reduce_kernel<IT, MODE><<<dim3(split, 8 * IT), 64, 0, st>>>(part, scale, M, N, p, out);
    return hipGetLastError();
}
template <int MODE>
hipError_t w8t_run_it(const W8tChoice &c, const uint16_t *x, int ldx, const int8_t *W, const float *scale, int M, int N,
                      int K, float *part, const W8Out &out, hipStream_t st) {
    if (c.it == 4) return w8t_run<4, MODE>(x, ldx, W, scale, M, N, K, c.plan, part, out, st);
    if (c.it == 2) return w8t_run<2, MODE>(x, ldx, W, scale, M, N, K, c.plan, part, out, st);
    return w8t_run<1, MODE>(x, ldx, W, scale, M, N, K, c.plan, part, out, st);
}

}  // namespace

size_t w8p_part_bytes(int seq_rows, int max_rows, int N, int K) {
    if (!w8t_counts_fit(max_rows, N)) return 0;  // no such launch
    if (const int reach = (int)std::min(8LL, w8t_wave_rows(K)); reach < std::min(8, max_rows)) seq_rows = max_rows = reach;
    return w8t_choose(max_rows, seq_rows, max_rows, N, K, K, kW8tPartBytes).need;
}

hipError_t launch_w8p(const uint16_t *x, int ldx, const int8_t *W, const float *scale, int M, int seq_rows,
                      int max_rows, int N, int K, const W8Out &out, float *part, size_t part_bytes, hipStream_t st) {
    if (M <= 0) return hipSuccess;
    if (N <= 0 || N % 64 || K <= 0 || K % 64 || ldx < K || ldx % 8 || (uintptr_t)x % 16 || seq_rows <= 0 || seq_rows > M || max_rows < M || !w8t_counts_fit(max_rows, N) || (uintptr_t)part % 16 ||
        (out.mode != kW8Segments && out.mode != kW8SwiGLU) || (out.mode == kW8SwiGLU && (N % 16 || !out.x16)) ||
        (out.mode == kW8Segments && (out.nseg < 1 || out.nseg > kW8MaxSegs)) ||
        (out.add_in && (out.mode != kW8Segments || out.nseg != 1)))
        return hipErrorInvalidValue;
    // rows of more than 306 million values: as many at a time as a wave reaches
    if (const long long reach = w8t_wave_rows(ldx); reach < std::min(8, M)) {
        for (int m = 0; m < M; m += (int)reach) {
            const int n = std::min((int)reach, M - m);
            W8Out o = out;
            for (W8Seg &sg : o.seg)
                if (sg.dst) sg.dst += (size_t)m * sg.ld;
            if (o.x16) o.x16 += (size_t)m * (N / 2);
            if (o.add_in) o.add_in += (size_t)m * o.add_ld;
            const hipError_t e = launch_w8p(x + (size_t)m * ldx, ldx, W, scale, n, n, n, N, K, o, part, part_bytes, st);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    const W8tChoice c = w8t_choose(M, seq_rows, max_rows, N, K, ldx, part ? part_bytes : 0);
    if (out.mode == kW8SwiGLU) return w8t_run_it<kW8tSwiGLU>(c, x, ldx, W, scale, M, N, K, part, out, st);
    if (out.add_in) return w8t_run_it<kW8tAdd>(c, x, ldx, W, scale, M, N, K, part, out, st);
    return w8t_run_it<kW8tSegments>(c, x, ldx, W, scale, M, N, K, part, out, st);
}

hipError_t launch_attn_prefill(const uint16_t *q16, const uint16_t *Kc, const uint16_t *vT, const float *gate,
                               int gate_row, uint16_t *out16, int nseq, int T, int Hq, int Hkv, int Tmax,
                               int Tv, float scaling, hipStream_t st) {
    if (T <= 0 || nseq <= 0) return hipSuccess;
    if (Hkv <= 0 || Hq % Hkv || Hq / Hkv > 4 || Tmax % 16 || Tmax < T || Tv % kApK || Tv < T)
        return hipErrorInvalidValue;
    const float sc_log2 = scaling * 1.4426950408889634f;
    attn_prefill_kernel<<<dim3((unsigned)((T + kApQ - 1) / kApQ), (unsigned)Hkv, (unsigned)nseq), kApThreads, 0, st>>>(
        q16, Kc, vT, gate, gate_row, out16, T, Hq, Hkv, Tmax, Tv, sc_log2);
    return hipGetLastError();
}

}  // namespace gdn
