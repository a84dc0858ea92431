// The residue generator of Scheme II INT8 for the kernels that write blocked residue planes
// (oz2_split.hip: operands whose deltas are known; oz2_prep.hip: deltas and planes in one pass), and its
// constants. Files that include this header are compiled as oz2_residue.hpp states.
#pragma once
#include "oz2_residue.hpp"

namespace {

// Generator of the blocked splitter (oz_tf32.hpp) for residues, E elements per lane: the state of
// an element is A' in balanced base-256 bytes and its residue modulo the even modulus, if the set
// has one (from the reference's sequence on the digits); plane s is the residue modulo m_s. The
// generator runs the planes itself: the even modulus, the odd moduli below 17 (byte dot products and
// one FP32 reduction, oz2_residue.hpp), then the odd moduli from 17 up four at a time, with their dot
// products on the matrix cores and the integer remainder step on the VALU.
//
// Matrix-core dot products for nd = 3 (8 balanced bytes per element; v_mfma_i32_16x16x64_i8, operand
// layout as in oz_gemm.hip: lane l holds row l%16 of the first operand and column l%16 of the second,
// K bytes 16(l/16)..+15 of each; output register r of lane l is row 4(l/16) + r, column l%16). The
// second operand of lane l is the bytes of two of its own elements, e in its low 8 bytes and e' in its
// high 8. Row i = 4g + r of the first operand holds, in K chunk g only, the byte weights w_p of modulus
// p = r%2 of a pair of moduli (symmetric residues of 256^j) over the half h = r/2 of the chunk, and zero
// elsewhere. So D[4g + r][j] = dinit_p + w_p . (half h of the second operand of lane 16g + j), and
// output register r of lane l is the dot product of lane l's element (e for r < 2, e' above) with
// modulus p: every lane gets the four sums of its own two elements and two moduli, 8 MFMAs per pair of
// moduli for its 16 elements (E = 16) in place of 2 v_dot4 per element and modulus. The sums are exact
// integers, the same as the v_dot4 chain's. For nd = 4 and 5 (12 and 16 bytes) the v_dot4 chain stays.
typedef int v4i_t __attribute__((ext_vector_type(4)));

template <int ND, int E = 16>
struct ResidueGen {
    static constexpr bool kDrivesPlanes = true;
    using Far = FarElements;
    static constexpr int W = balanced_words<ND>();
    SplitConsts k;
    struct State {
        uint32_t a[W];
        int even;
    };
    // PROCEDURE: nd = 3 too through the binary32 digits.
    template <bool PROCEDURE = ND != 3>
    __device__ __forceinline__ void load(State& st, double x, int32_t d, Far& far) const {
        float dig[ND];
        if constexpr (!PROCEDURE) {
            far.add(split_integer3(x, d, st.a, dig), d);
        } else {
            make_digits<ND>(x, d, dig);
            balanced_bytes<ND>(dig, st.a);
        }
        // (here and without a branch, held by the empty asm: sunk to its plane, as the compiler would have it, it
        // keeps every element's digits live that far, 110 registers and more; a set without an even modulus
        // computes a residue that no plane takes)
        st.even = residue<ND>(dig, k, max(k.even, 0));
        if constexpr (ND == 3)
            asm volatile("" : "+v"(st.even), "+v"(st.a[0]), "+v"(st.a[1]));
        else
            asm volatile("" : "+v"(st.even));
    }
    // After a lane's E elements: where a wave has some that are Far, all go through the procedure, out of line, and are
    // read again for it by again(e, x, d) (kept for this, the elements would take 20 registers more).
    template <class AGAIN>
    __device__ __forceinline__ void redo(State* st, const Far& far, AGAIN again) const {
        if constexpr (ND == 3)
            if (__builtin_expect(__ballot(far.any()) != 0, 0)) {
                Far same;
#pragma unroll
                for (int e = 0; e < E; e++) {
                    double x;
                    int32_t d;
                    again(e, x, d);
                    load<true>(st[e], x, d, same);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
    }
    // x = r + (m-1)/2 in the low byte: adding 128 - (m-1)/2 keeps every byte in [1, 255] (no carry
    // into the next one), and xor 0x80 then subtracts 128 from each (two's complement bytes)
    template <class EMIT>
    __device__ __forceinline__ void emit_odd(EMIT& emit, int s, const uint32_t* pk) const {
        const uint32_t badd = k.badd[s];
        uint32_t w[E / 4];
#pragma unroll
        for (int c = 0; c < E / 4; c++) w[c] = (pk[c] + badd) ^ 0x80808080u;
        emit(s, w);
    }
    template <class EMIT>
    __device__ __forceinline__ void run(State* st, EMIT&& emit) const {
        uint32_t w[E / 4];
        if (k.even >= 0) {
#pragma unroll
            for (int c = 0; c < E / 4; c++) w[c] = pack4(st[4 * c].even, st[4 * c + 1].even, st[4 * c + 2].even, st[4 * c + 3].even);
            emit(k.even, w);
        }
        for (int i = 0; i < k.nsmall; i++) {
            const int s = k.small[i];
            int v[E];
#pragma unroll
            for (int e = 0; e < E; e++) v[e] = (int)residue_odd<W>(st[e].a, k.w[s], k.m[s], k.rinv[s]);
#pragma unroll
            for (int c = 0; c < E / 4; c++) w[c] = pack4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
            emit(s, w);
        }
        if constexpr (W == 2) {
            const int lane = threadIdx.x & 63, r = lane & 3;
            const bool on = (lane >> 4) == ((lane & 15) >> 2);
            for (int g = 0; g < k.npair; g++) {
                const int s0 = __builtin_amdgcn_readfirstlane(k.pair[g][0]);
                const int s1 = __builtin_amdgcn_readfirstlane(k.pair[g][1]);
                const uint32_t w00 = __builtin_amdgcn_readfirstlane(k.w[s0][0]), w01 = __builtin_amdgcn_readfirstlane(k.w[s0][1]);
                const uint32_t w10 = __builtin_amdgcn_readfirstlane(k.w[s1][0]), w11 = __builtin_amdgcn_readfirstlane(k.w[s1][1]);
                const uint32_t lo = (r & 1) ? w10 : w00, hi = (r & 1) ? w11 : w01;
                const bool h = (r >> 1) != 0;
                const v4i_t wa = {on && !h ? (int)lo : 0, on && !h ? (int)hi : 0, on && h ? (int)lo : 0, on && h ? (int)hi : 0};
                const int d0 = k.dinit[s0], d1 = k.dinit[s1];
                const v4i_t c0 = {d0, d1, d0, d1};
                const uint32_t mg0 = k.magic[s0], mg1 = k.magic[s1];
                const int mn0 = k.mneg[s0], mn1 = k.mneg[s1];
                uint32_t pk0[E / 4], pk1[E / 4];
#pragma unroll
                for (int c = 0; c < E / 4; c++) {
                    int x0[4], x1[4];
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        const State& ea = st[4 * c + 2 * t];
                        const State& eb = st[4 * c + 2 * t + 1];
                        const v4i_t b = {(int)ea.a[0], (int)ea.a[1], (int)eb.a[0], (int)eb.a[1]};
                        const v4i_t u = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa, b, c0, 0, 0, 0);
                        x0[2 * t] = reduce_odd_int<W>(u[0], mg0, mn0);
                        x1[2 * t] = reduce_odd_int<W>(u[1], mg1, mn1);
                        x0[2 * t + 1] = reduce_odd_int<W>(u[2], mg0, mn0);
                        x1[2 * t + 1] = reduce_odd_int<W>(u[3], mg1, mn1);
                    }
                    pk0[c] = pack4(x0[0], x0[1], x0[2], x0[3]);
                    pk1[c] = pack4(x1[0], x1[1], x1[2], x1[3]);
                }
                emit_odd(emit, s0, pk0);
                if (s1 != s0) emit_odd(emit, s1, pk1);
            }
        } else {
            for (int g = 0; g < k.npair; g++)
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const int s = k.pair[g][p];
                    if (p == 1 && s == k.pair[g][0]) break;
                    uint32_t a[E][W];
#pragma unroll
                    for (int e = 0; e < E; e++)
#pragma unroll
                        for (int i = 0; i < W; i++) a[e][i] = st[e].a[i];
                    int v[E];
                    residues_odd_int<W, E>(a, k.w[s], k.dinit[s], k.magic[s], k.mneg[s], v);
                    uint32_t pk[E / 4];
#pragma unroll
                    for (int c = 0; c < E / 4; c++) pk[c] = pack4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
                    emit_odd(emit, s, pk);
                }
        }
    }
};

// ---- Pieces of an OZ_BLOCK block ------------------------------------------------------------
// A wave's share of a 1 KB block with E elements per lane (E = 4, 8 or 16): piece q of 16 / E. Rows of A
// (ROWS): rows 16 br + q E + e of column 64 kb + lane. Columns of B: K indices k0 + e of column
// 16 br + lane / 4, with k0 = 64 kb + 4 E q + E (lane & 3).
template <int E>
__device__ __forceinline__ int piece_k0(int kb, int q, int lane) {
    return kb * 64 + q * 4 * E + E * (lane & 3);
}

// The piece of X (rows x cols, ld); zeros outside, addresses clamped into X.
template <int E, bool ROWS>
__device__ __forceinline__ void load_piece(const double* __restrict__ X, int rows, int cols, int ld, int br, int kb, int q,
                                           int lane, double* x) {
    const int r0 = ROWS ? br * 16 + q * E : piece_k0<E>(kb, q, lane);
    const int col = ROWS ? kb * 64 + lane : br * 16 + (lane >> 2);
    const int cc = min(col, cols - 1);
#pragma unroll
    for (int e = 0; e < E; e++) {
        const double v = X[(size_t)min(r0 + e, rows - 1) * ld + cc];
        x[e] = r0 + e < rows && col < cols ? v : 0.0;
    }
}

// Element e of it, with no address kept since (the lane is taken afresh).
template <int E, bool ROWS>
__device__ __forceinline__ double piece_element(const double* __restrict__ X, int rows, int cols, int ld, int br, int kb,
                                                int q, int e) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int r = (ROWS ? br * 16 + q * E : piece_k0<E>(kb, q, lane)) + e;
    const int col = ROWS ? kb * 64 + lane : br * 16 + (lane >> 2);
    const double v = X[(size_t)min(r, rows - 1) * ld + min(col, cols - 1)];
    return r < rows && col < cols ? v : 0.0;
}

// E bytes (E / 4 words) to p: a whole block's lane piece non-temporally (as oz_tf32.hpp), shorter ones as
// ordinary stores (several waves fill a line, which the L2 joins).
template <int E>
__device__ __forceinline__ void store_piece(uint8_t* p, const uint32_t* w) {
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    if constexpr (E == 4)
        *reinterpret_cast<uint32_t*>(p) = w[0];
    else if constexpr (E == 8)
        *reinterpret_cast<u32x2*>(p) = u32x2{w[0], w[1]};
    else
        __builtin_nontemporal_store(u32x4{w[0], w[1], w[2], w[3]}, reinterpret_cast<u32x4*>(p));
}

// All planes of the piece from its states; img: 64 E bytes of LDS private to the wave (ROWS: a plane's byte
// columns in, contiguous pieces out; the LDS operations of a wave are in order).
template <int ND, int E, bool ROWS>
__device__ __forceinline__ void emit_piece(const ResidueGen<ND, E>& gen, typename ResidueGen<ND, E>::State* st,
                                           uint8_t* __restrict__ planes, long long stride, int br, int kblocks, int kb,
                                           int q, int lane, uint8_t* img) {
    uint8_t* blk = planes + ((long long)br * kblocks + kb) * 1024;
    if constexpr (ROWS) {
        uint8_t* out = blk + q * E * 64 + E * lane;
        const int part = 16 * (lane >> 4), byte = lane & 15;
        gen.run(st, [&](int p, const uint32_t* w) {
#pragma unroll
            for (int e = 0; e < E; e++)
                img[64 * e + (part ^ (16 * block_swizzle(q * E + e))) + byte] = (uint8_t)(w[e >> 2] >> (8 * (e & 3)));
            uint32_t v[E / 4];
#pragma unroll
            for (int i = 0; i < E / 4; i++) v[i] = reinterpret_cast<const uint32_t*>(img + E * lane)[i];
            store_piece<E>(out + (long long)p * stride, v);
        });
    } else {
        const int rr = lane >> 2, k0 = piece_k0<E>(kb, q, lane);
        uint8_t* out = blk + rr * 64 + 16 * (((k0 & 63) >> 4) ^ block_swizzle(rr)) + (k0 & 15);
        gen.run(st, [&](int p, const uint32_t* w) { store_piece<E>(out + (long long)p * stride, w); });
    }
}

int check_moduli(oz_dev* dev, const oz2_moduli_dev* mo) {
    if (!mo || mo->S < 1 || mo->S > OZ2_MAXS || mo->nd < 3 || mo->nd > 5)
        return oz::fail(dev, OZ_ERR_ARG, "oz2_split_int8: invalid moduli descriptor");
    for (int s = 0; s < mo->S; s++)
        if (!(mo->m[s] >= 2.0f && mo->m[s] <= 255.0f))
            return oz::fail(dev, OZ_ERR_ARG, "oz2_split_int8: modulus %g outside the INT8 range", (double)mo->m[s]);
    return OZ_OK;
}

// Kernel constants of a moduli descriptor (oz2_residue.hpp); *evens counts the even moduli.
SplitConsts split_consts(const oz2_moduli_dev* mo, int* evens) {
    SplitConsts k{};
    k.even = -1;
    *evens = 0;
    for (int s = 0; s < mo->S; s++) {
        k.m[s] = mo->m[s];
        k.rinv[s] = mo->rinv[s];
        for (int j = 0; j < 4; j++) k.c[j][s] = mo->c[j][s];
        // symmetric residues of 256^j modulo m, four to a word (signed bytes)
        const int m = (int)mo->m[s];
        if (m % 2 == 1 && m >= 17) {
            const int U = mo->nd == 3 ? 18 : 19, sh = 24 - U, h = (m - 1) / 2;
            const long long half = 1ll << (U - 1);
            k.dinit[s] = (int)((half + m - 1) / m * m + h);
            k.magic[s] = (uint32_t)(((1ull << (32 - sh)) + m - 1) / m);
            k.badd[s] = (uint32_t)(128 - h) * 0x01010101u;
            k.mneg[s] = (1 << 24) - m;
        }
        if (m % 2 == 0) {
            k.even = s;
            (*evens)++;
        } else if (m < 17) {
            k.small[k.nsmall++] = s;
        } else if (k.npair && k.pair[k.npair - 1][1] < 0) {
            k.pair[k.npair - 1][1] = s;
        } else {
            k.pair[k.npair][0] = s;
            k.pair[k.npair++][1] = -1;
        }
        int p = 1;  // 256^j mod m
        for (int i = 0; i < 4; i++) {
            uint32_t word = 0;
            for (int j = 0; j < 4; j++) {
                const int sym = p > m / 2 ? p - m : p;
                word |= (uint32_t)(sym & 0xFF) << (8 * j);
                p = p * 256 % m;
            }
            k.w[s][i] = word;
        }
    }
    if (k.npair && k.pair[k.npair - 1][1] < 0)  // a last single modulus is paired with itself (stored once)
        k.pair[k.npair - 1][1] = k.pair[k.npair - 1][0];
    return k;
}

}  // namespace
