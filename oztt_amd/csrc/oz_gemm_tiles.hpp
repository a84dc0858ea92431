// Products of few or short tiles: the INT8 products of oz_gemm.hip in smaller tiles, for launches whose
// 256 x 256 tiles would leave compute units idle or spend more time on filling and draining a tile
// than on its K steps. The same operands (OZ_BLOCK tiles), the same exact int32 sums.
#pragma once
#include "oz2_modular.hpp"
#include "oz_gemm_common.hpp"

namespace ozg {

// Output modes of the INT8 product kernels. PRODUCTS: C[b] = A[b] Bt[b]^T as int32. DIGITS: the same
// products reduced in the epilogue to the CRT digit for modulus b ((C mod m_b) y_b mod m_b, from
// dc.m/y[b]; a digit 0 may be stored as m_b, oz2::mod_mul_f64), C as uint8. DIAG (scheme I):
// C[d] = sum_{i <= d} A[i] Bt[d-i]^T as int32 for the diagonals d < nbatch, the d+1 slice pairs
// concatenated along K in one accumulation.
enum GemmMode { PRODUCTS = 0, DIGITS = 1, DIAG = 2 };

// Workgroup -> (batch, tile row, tile column). Digits: each XCD takes a contiguous range of the
// batch-major sequence (tile_of), whole moduli where there are few tiles. Diagonals differ up to p-fold
// in length: batch by batch over all XCDs, the longest first, or the XCD that got the last diagonals
// would run several times as long as the first (1024^2 x 8192, 8 slices: 566 against 378 us).
template <int MODE>
__device__ __forceinline__ void small_tile_of(int w, int tiles_m, int tiles_n, int nbatch, int& batch, int& tm, int& tn) {
    if constexpr (MODE != DIAG) {
        tile_of(w, tiles_m, tiles_n, nbatch, batch, tm, tn);
    } else {
        tile_of_lockstep(w, tiles_m, tiles_n, nbatch, batch, tm, tn);
        batch = nbatch - 1 - batch;
    }
    // wave-uniform, but the divisions run on the VALU
    batch = __builtin_amdgcn_readfirstlane(batch);
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
}

// Byte offset, inside a 1 KB OZ_BLOCK block, of the 16 bytes that lane l brings to
// v_mfma_i32_16x16x64_i8: row l % 16, chunk l / 16.
__device__ __forceinline__ int fragment16_offset(int lane) {
    const int r = lane & 15, c = lane >> 4;
    return 64 * r + 16 * (c ^ (((r >> 1) ^ (r >> 2)) & 3));
}

// Sums staged in LDS, row-major in rows of 16 TJ ints whose 16-int groups are swizzled by bits 2..3 of
// the row, so that the four rows that one accumulator register holds fall on different banks.
template <int TJ>
__device__ __forceinline__ int staged_group(int row, int group) {
    constexpr int XM = TJ >= 4 ? 3 : TJ - 1;
    return row * 16 * TJ + ((16 * group) ^ (16 * ((row >> 2) & XM)));
}

// 16 staged sums at src -> 16 digits at dst.
__device__ __forceinline__ void store_digits16(const int32_t* src, uint8_t* dst, double yr, double md) {
    int32_t v[16];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const v4i x = *reinterpret_cast<const v4i*>(src + 4 * k);
#pragma unroll
        for (int q = 0; q < 4; q++) v[4 * k + q] = x[q];
    }
    uint32_t w[4];
    oz2::mod_mul_f64_x16(v, yr, md, w);
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(u32x4{w[0], w[1], w[2], w[3]}, reinterpret_cast<u32x4*>(dst));
}

// Few tiles, long K: a tile of 16 TI x 16 TJ per workgroup, its K steps dealt out to KW waves, which sum
// their int32 accumulators in LDS at the end (exact, any order). A wave owns the whole tile, so there is
// nothing to share between the waves and no barrier in the loop: an OZ_BLOCK block is one MFMA operand,
// and the wave reads its TI + TJ blocks of a K step straight into registers, P steps ahead, one
// coalesced 1 KB load each. Bound by those loads (a tile of 64 x 64 reads 8 KB for 16 MFMAs, about half
// of what the matrix cores could take from L2), so it serves where the 256 x 256 tiles (or, for the
// diagonals, the all-diagonals kernel's 64 x 64) are too few for the chip. 256 x 256 x 32768, 16 moduli
// (256 tiles): 255.6 -> 50.6 us launch after launch, 290 -> 78 in a pass (the planes in no cache yet);
// 256 x 256 x 2048, 8 diagonals: 141 -> 16.5 us.
template <int MODE, int TI, int TJ, int KW, int P>
__global__ void __launch_bounds__(64 * KW) gemm_i8_ksplit_kernel(const int8_t* __restrict__ A,
                                                                 const int8_t* __restrict__ Bt, void* __restrict__ C,
                                                                 int K, int ldc, long long sA, long long sB,
                                                                 long long sC, int tiles_m, int tiles_n, int nbatch,
                                                                 oz2::DigitConsts dc) {
    constexpr int TM = 16 * TI, TN = 16 * TJ;
    __shared__ __attribute__((aligned(1024))) int32_t sums[TM * TN];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int e = threadIdx.x; e < TM * TN / 4; e += 64 * KW) reinterpret_cast<v4i*>(sums)[e] = v4i{0, 0, 0, 0};
    int batch, tm, tn;
    small_tile_of<MODE>(blockIdx.x, tiles_m, tiles_n, nbatch, batch, tm, tn);
    const int nk = K / BK;
    const int nst = MODE == DIAG ? (batch + 1) * nk : nk;  // K steps of this tile
    const long long band = (long long)nk * 1024;
    const int foff = fragment16_offset(lane);
    const int8_t* Ab = A + (MODE == DIAG ? 0 : batch * sA) + (long long)tm * TI * band + foff;
    const int8_t* Bb = Bt + batch * sB + (long long)tn * TJ * band + foff;
    v4i acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = v4i{0, 0, 0, 0};
    // This wave's steps are wave, wave + KW, ... (`mine` of them, possibly none). DIAG: step st is block
    // lk = st % nk of pair st / nk (A plane i, B plane batch - i), kept as running offsets.
    const int mine = (nst - wave + KW - 1) / KW;
    int at = 0, lk = wave;
    long long oA = 0, oB = 0;
    auto wrap = [&]() {
        if constexpr (MODE == DIAG)
            while (lk >= nk) {
                lk -= nk;
                oA += sA;
                oB -= sB;
            }
    };
    wrap();
    v4i a[P][TI], b[P][TJ];
    auto load = [&](int p) {
        if (at < mine) {
            const int8_t* pa = Ab + oA + (long long)lk * 1024;
            const int8_t* pb = Bb + oB + (long long)lk * 1024;
#pragma unroll
            for (int i = 0; i < TI; i++) a[p][i] = *reinterpret_cast<const v4i*>(pa + (long long)i * band);
#pragma unroll
            for (int j = 0; j < TJ; j++) b[p][j] = *reinterpret_cast<const v4i*>(pb + (long long)j * band);
        }
        at++;
        lk += KW;
        wrap();
    };
    auto multiply = [&](int p) {
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[p][i], b[p][j], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int p = 0; p < P; p++) load(p);
    int kt = 0;
    for (; kt + P <= mine; kt += P) {
#pragma unroll
        for (int p = 0; p < P; p++) {
            multiply(p);
            load(p);
        }
    }
#pragma unroll
    for (int p = 0; p < P - 1; p++)
        if (kt + p < mine) multiply(p);
    __syncthreads();  // the zeros
    const int r = lane & 15, c = lane >> 4;
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                atomicAdd(&sums[staged_group<TJ>(16 * i + 4 * c + q, j) + r], acc[i][j][q]);
    __syncthreads();
    const long long c0 = batch * sC + (long long)tm * TM * ldc + tn * TN;
    if constexpr (MODE == DIGITS) {
        const uint32_t m = dc.m[batch];
        const double md = (double)m, yr = (double)dc.y[batch] / md;
        uint8_t* Cb = static_cast<uint8_t*>(C) + c0;
        for (int e = threadIdx.x; e < TM * TJ; e += 64 * KW)
            store_digits16(sums + staged_group<TJ>(e / TJ, e % TJ), Cb + (long long)(e / TJ) * ldc + 16 * (e % TJ), yr, md);
    } else {
        int32_t* Cb = static_cast<int32_t*>(C) + c0;
        for (int e = threadIdx.x; e < TM * TN; e += 64 * KW) {
            const int row = e / TN, col = e % TN;
            __builtin_nontemporal_store(sums[staged_group<TJ>(row, col >> 4) + (col & 15)],
                                        &Cb[(long long)row * ldc + col]);
        }
    }
}

// Short K, or tiles that fill the chip unevenly: WM x WN waves, each 16 TI x 16 TJ, share the operands of
// a K step through a ring of NSTG LDS stages (direct global->LDS copies, NSTG - 1 steps ahead, as in
// oz_gemm.hip). Two or three workgroups fit a CU (LDS and registers), so one fills its ring or writes its
// digits while another multiplies; a 256 x 256 tile is alone on its CU and pays 10 us for both. Per K step
// the smaller tiles move more bytes through L2 (128 x 128: twice those of 256 x 256 per product), so
// from K of about 1500 on the large tile is the faster one wherever it fills the chip. 4096 x 4096 x 256,
// 15 moduli: 177 -> 160 us (256 x 128); 512^3, 16 moduli: 12.9 -> 6.9 us (128 x 128); 256 x 256 x 128:
// 9.6 -> 3.4 us (64 x 64).
template <int MODE, int TI, int TJ, int WM, int WN, int NSTG>
__global__ void __launch_bounds__(64 * WM * WN, 2) gemm_i8_tile_kernel(const int8_t* __restrict__ A,
                                                                       const int8_t* __restrict__ Bt,
                                                                       void* __restrict__ C, int K, int ldc,
                                                                       long long sA, long long sB, long long sC,
                                                                       int tiles_m, int tiles_n, int nbatch,
                                                                       oz2::DigitConsts dc) {
    constexpr int W = WM * WN, BA = TI * WM, BB = TJ * WN;  // waves; 1 KB blocks of a stage
    constexpr int LA = BA / W, LB = BB / W, LD = LA + LB;   // copies per wave and stage
    static_assert(LA * W == BA && LB * W == BB, "whole blocks per wave");
    constexpr int STG = (BA + BB) * 1024;
    constexpr int TM = 16 * BA, TN = 16 * BB;
    __shared__ __attribute__((aligned(1024))) int8_t lds[NSTG * STG];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int batch, tm, tn;
    small_tile_of<MODE>(blockIdx.x, tiles_m, tiles_n, nbatch, batch, tm, tn);
    const int nk = K / BK;
    const int nst = MODE == DIAG ? (batch + 1) * nk : nk;
    const long long band = (long long)nk * 1024;
    const int8_t* Ab = A + (MODE == DIAG ? 0 : batch * sA) + (long long)tm * BA * band;
    const int8_t* Bb = Bt + batch * sB + (long long)tn * BB * band;
    const unsigned lane16 = 16u * lane;
    // The step to load next, as in oz_gemm.hip: running offsets, the last step again past the end, so
    // that every step issues the same copies and the wait counts never change.
    int lk = 0, lcount = 0;
    long long oA = 0, oB = 0;
    auto next_stage = [&]() {
        const int adv = lcount < nst - 1;
        lcount += adv;
        oA += adv ? 1024 : 0;
        oB += adv ? 1024 : 0;
        if constexpr (MODE == DIAG) {
            lk += adv;
            const int wrap = lk == nk;
            lk = wrap ? 0 : lk;
            oA += wrap ? sA - band : 0;
            oB -= wrap ? sB + band : 0;
        }
    };
    auto issue = [&](int buf) {
#pragma unroll
        for (int j = 0; j < LA; j++) {
            const int q = W * j + wave;
            lds_copy_block(Ab + ((long long)q * band + oA), lds + buf * STG + q * 1024, lane16);
        }
#pragma unroll
        for (int j = 0; j < LB; j++) {
            const int q = W * j + wave;
            lds_copy_block(Bb + ((long long)q * band + oB), lds + buf * STG + (BA + q) * 1024, lane16);
        }
    };
    const int wm = wave / WN, wn = wave % WN;
    const int r = lane & 15, c = lane >> 4;
    const int foff = fragment16_offset(lane);
    v4i acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < NSTG - 1; s++) {
        issue(s);
        next_stage();
    }
    // Step kt: its stage has landed (all but the last NSTG - 2 stages' copies are complete) and every wave
    // has read step kt - 1's (its fragments entered MFMAs before the barrier), whose buffer is refilled.
    int buf = 0, fill = NSTG - 1;
    for (int kt = 0; kt < nst; kt++) {
        wait_vmcnt_lgkm0<LD * (NSTG - 2)>();
        stage_barrier();
        issue(fill);
        next_stage();
        v4i fa[TI], fb[TJ];
#pragma unroll
        for (int i = 0; i < TI; i++) fa[i] = *reinterpret_cast<const v4i*>(lds + buf * STG + (wm * TI + i) * 1024 + foff);
#pragma unroll
        for (int j = 0; j < TJ; j++) fb[j] = *reinterpret_cast<const v4i*>(lds + buf * STG + (BA + wn * TJ + j) * 1024 + foff);
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
        buf = buf + 1 == NSTG ? 0 : buf + 1;
        fill = fill + 1 == NSTG ? 0 : fill + 1;
    }
    wait_vmcnt<0>();  // drain the clamped tail copies before the ring is reused or the workgroup ends
    const long long c0 = batch * sC + (long long)(tm * TM + wm * 16 * TI) * ldc + tn * TN + wn * 16 * TJ;
    if constexpr (MODE == DIGITS) {
        const uint32_t m = dc.m[batch];
        const double md = (double)m, yr = (double)dc.y[batch] / md;
        uint8_t* Cb = static_cast<uint8_t*>(C) + c0;
        __syncthreads();
        // each wave stages its sums in its share of the ring, RI bands of 16 rows at a time
        constexpr int ROOM = NSTG * STG / W / 4;
        constexpr int RI = TI * TJ * 256 <= ROOM ? TI : TI / 2;
        static_assert(RI >= 1 && RI * TJ * 256 <= ROOM && TI % RI == 0 && RI * TJ % 4 == 0, "staging room");
        int32_t* tile = reinterpret_cast<int32_t*>(lds) + wave * ROOM;
#pragma unroll
        for (int h = 0; h < TI / RI; h++) {
#pragma unroll
            for (int i = 0; i < RI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        tile[staged_group<TJ>(16 * i + 4 * c + q, j) + r] = acc[h * RI + i][j][q];
#pragma unroll
            for (int t = 0; t < RI * TJ / 4; t++) {
                const int e = 64 * t + lane;
                store_digits16(tile + staged_group<TJ>(e / TJ, e % TJ),
                               Cb + (long long)(16 * RI * h + e / TJ) * ldc + 16 * (e % TJ), yr, md);
            }
        }
    } else {
        int32_t* Cb = static_cast<int32_t*>(C) + c0;
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    __builtin_nontemporal_store(acc[i][j][q], &Cb[(long long)(16 * i + 4 * c + q) * ldc + 16 * j + r]);
    }
}

// Scheme I, all diagonals of a 64 x 64 tile in one workgroup: the P slices of 64 rows of A and of 64
// columns of B are brought in once per K step (8 P KB) and serve all P (P + 1)/2 pairs, where a tile per
// diagonal brings every pair's two slices by itself. With 8 slices that is 0.11 KB per MFMA from L2, as
// little as the 256 x 256 tile needs, at a sixteenth of its area: the chip is full from 1024 x 1024 on,
// and every tile is equally long. 4 waves of 32 x 32, 4 P accumulators each; two stages of 8 P KB; the
// fragments of the next step are read while this one multiplies, and the copies that refill the ring go
// out in the first half of the step (they land at its end: spread over the whole step, the last ones
// made every step wait, 185 against 158 us for 256 x 256 x 8192). At 1024^2 x 8192, 8 slices: 566 -> 238
// us, 2.6 POP/s, the rate at which the matrix cores meet the power limit.
template <int P, bool EVEN>
__global__ void __launch_bounds__(256, 1) gemm_i8_diagonals_kernel(const int8_t* __restrict__ A,
                                                                   const int8_t* __restrict__ Bt,
                                                                   int32_t* __restrict__ C, int K, int ldc,
                                                                   long long sA, long long sB, long long sC,
                                                                   int tiles_m, int tiles_n) {
    constexpr int STG = 8 * P * 1024;
    __shared__ __attribute__((aligned(1024))) int8_t lds[2 * STG];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int one, tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, 1, one, tm, tn);
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
    const int nst = K / BK;
    const long long band = (long long)nst * 1024;
    const int8_t* Ab = A + (long long)(tm * 4 + wave) * band;
    const int8_t* Bb = Bt + (long long)(tn * 4 + wave) * band;
    const unsigned lane16 = 16u * lane;
    // copy t of this wave: its 16-row band of A's slice t (t < P) or B's slice t - P, K step st
    auto issue = [&](int buf, int t, int st) {
        const int8_t* g = t < P ? Ab + (long long)t * sA : Bb + (long long)(t - P) * sB;
        lds_copy_block(g + (long long)st * 1024, lds + buf * STG + (4 * t + wave) * 1024, lane16);
    };
    const int wm = wave >> 1, wn = wave & 1;
    const int r = lane & 15, c = lane >> 4;
    const int foff = fragment16_offset(lane);
    v4i acc[P][2][2];
#pragma unroll
    for (int d = 0; d < P; d++)
#pragma unroll
        for (int q = 0; q < 4; q++) acc[d][q >> 1][q & 1] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int t = 0; t < 2 * P; t++) issue(s, t, min(s, nst - 1));
    // fragment t of A (op 0) or B (op 1): half t % 2 of this wave's 32 rows of slice t / 2
    v4i fa[2 * P], fb[2 * P], ga[2 * P], gb[2 * P];
    auto rd = [&](int buf, int op, int t) -> v4i {
        return *reinterpret_cast<const v4i*>(lds + buf * STG + (4 * (op * P + (t >> 1)) + 2 * (op ? wn : wm) + (t & 1)) * 1024 + foff);
    };
    wait_vmcnt<2 * P>();
    stage_barrier();
#pragma unroll
    for (int t = 0; t < 2 * P; t++) {
        fa[t] = rd(0, 0, t);
        fb[t] = rd(0, 1, t);
    }
    // One K step: the pairs (i, j), i + j < P, by max(i, j), so that the first ones need the first slices;
    // 4 P fragment reads spread over all MFMAs, 2 P copies over the first half.
    auto substep = [&](v4i* xa, v4i* xb, v4i* ya, v4i* yb, int rbuf, int lbuf, int lst) {
        constexpr int NM = 2 * P * (P + 1);  // MFMAs
        int n = 0, reads = 0, copies = 0;
#pragma unroll
        for (int m = 0; m < P; m++)
#pragma unroll
            for (int k = 0; k <= 2 * m; k++) {
                const int i = k <= m ? m : 2 * m - k, j = k <= m ? k : m;
                if (i + j >= P) continue;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    v4i& s = acc[i + j][q >> 1][q & 1];
                    s = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[2 * i + (q >> 1)], xb[2 * j + (q & 1)], s, 0, 0, 0);
                    if (reads < 4 * P && n * 4 * P >= reads * NM) {
                        const int t = reads >> 1;
                        if (reads & 1) yb[t] = rd(rbuf, 1, t);
                        else ya[t] = rd(rbuf, 0, t);
                        reads++;
                    }
                    if (copies < 2 * P && n * 4 * P >= copies * NM + P) {
                        issue(lbuf, (copies & 1) ? P + (copies >> 1) : (copies >> 1), lst);
                        copies++;
                    }
                    n++;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
    };
    int kt = 0;
    for (; kt + 1 < nst; kt += 2) {
        wait_vmcnt_lgkm0<0>();
        stage_barrier();
        substep(fa, fb, ga, gb, 1, 0, min(kt + 2, nst - 1));
        wait_vmcnt_lgkm0<0>();
        stage_barrier();
        substep(ga, gb, fa, fb, 0, 1, min(kt + 3, nst - 1));
    }
    if constexpr (!EVEN) {
        if (kt < nst) {
            wait_vmcnt_lgkm0<0>();
            stage_barrier();
            substep(fa, fb, ga, gb, 1, 0, nst - 1);
        }
    }
    wait_vmcnt<0>();  // drain the clamped tail copies before the workgroup ends
    int32_t* Cb = C + (long long)(tm * 64 + wm * 32) * ldc + tn * 64 + wn * 32;
#pragma unroll
    for (int d = 0; d < P; d++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    __builtin_nontemporal_store(acc[d][i][j][q],
                                                &Cb[d * sC + (long long)(16 * i + 4 * c + q) * ldc + 16 * j + r]);
}

}  // namespace ozg
