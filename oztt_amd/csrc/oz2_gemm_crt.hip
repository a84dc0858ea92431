// Scheme II INT8 products and reconstruction in one kernel, for short inner dimensions and small results.
//
// Semantics: oz2_gemm_digits followed by oz2_crt_digits_f64 (A9-A11): for every output element the exact
// products C_s of the S residue planes, the integer C' in (floor(M/2) - M, floor(M/2)] congruent to every
// C_s modulo m_s, and C' * 2^(eA_i + eB_j - 2b) rounded once to nearest-even. The results are the same bit
// for bit, C' being exact in both.
//
// What it saves: at K = 256 the digits of a 4096 x 4096 product (15 x 16 MB) are as many bytes as
// everything else together, written and read back, and a 256 x 256 tile spends more time on filling its
// ring and on its digits than on its 4 K steps. Here a workgroup computes its tile for all moduli, one
// after another, in one software pipeline that never drains, and adds every modulus's sums straight to the
// CRT accumulator in registers:
//     V = sum_s C_s W_s,   W_s = y_s Q_s < M  (so V == C' modulo M),
// in L limbs of w bits held as exact doubles, w such that S max|C_s| 2^w <= 2^52: one conversion and L
// FMAs per element and modulus, in place of a digit (four FP64 operations, packing, LDS, a store), a load
// and its L accumulations. t = rint(V / M) is now up to S max|C_s| and its estimate good to 2^-20.6 (w >= 24; the
// threshold of the exact comparison, delta, is 2^-20); the rest of the finish is that of oz2_crt.hip.
//
// It is bound by the FP64 pipe (L + 1 operations per element and modulus, about 110 for the finish) while
// the products ride along on the matrix cores, at the price of small tiles: a wave's 32 x 32 sums need
// 32 L registers of limbs. So it pays while K is short; oz2_pass.hip holds the rule and the times.
#include "oz2_gemm_crt.hpp"

#include <algorithm>
#include <cmath>

#include "oz_gemm_tiles.hpp"

namespace {

using namespace ozg;

template <int L>
struct FusedCrt {
    int S, b, shift;
    double radix;   // 2^w
    double carry;   // 2^-w
    double invM;
    double delta;
    double W[OZ2_MAXS][L];
    double Mw[L], Mhalf[L], Mrest[L];
    double pow[L];  // 2^(w l)
};

// Carries of limbs 0..L-2 into [0, 2^w); the top limb keeps the sign. Exact: integers of at most 2^53.
template <int L>
__device__ __forceinline__ void normalize(double* x, const FusedCrt<L>& a) {
#pragma unroll
    for (int l = 0; l + 1 < L; l++) {
        const double c = __builtin_floor(x[l] * a.carry);
        x[l] = __builtin_fma(-c, a.radix, x[l]);
        x[l + 1] += c;
    }
}

template <int L>
__device__ __forceinline__ int limb_sign(const double* x) {
    if (x[L - 1] != 0.0) return x[L - 1] > 0.0 ? 1 : -1;
    bool nz = false;
#pragma unroll
    for (int l = 0; l + 1 < L; l++) nz |= x[l] != 0.0;
    return nz ? 1 : 0;
}

// x = V in limbs of at most 2^52 -> C' 2^e2 rounded to nearest-even; the steps of oz2_crt.hip's crt_finish
// and magnitude40 for limbs of any width (the cascade's argument holds for every w: a stage that rounds
// has an ulp of at least twice its term's unit, and all terms below are together less than that unit).
template <int L>
__device__ __forceinline__ double finish(double* x, const FusedCrt<L>& a, int e2) {
    double vd = x[L - 1];
#pragma unroll
    for (int l = L - 2; l >= 0; l--) vd = __builtin_fma(vd, a.radix, x[l]);
    const double q = vd * a.invM;
    const double t = __builtin_rint(q);
#pragma unroll
    for (int l = 0; l < L; l++) x[l] = __builtin_fma(-t, a.Mw[l], x[l]);
    bool neg = q - t < 0.0;
    if (__builtin_fabs(q - t) > 0.5 - a.delta) {
        // the estimate may pick the wrong neighbour: compare C' with floor(M/2) exactly
        normalize<L>(x, a);
        double y[L];
#pragma unroll
        for (int l = 0; l < L; l++) y[l] = x[l] - a.Mhalf[l];
        normalize<L>(y, a);
        if (limb_sign<L>(y) > 0) {
#pragma unroll
            for (int l = 0; l < L; l++) x[l] -= a.Mw[l];
            normalize<L>(x, a);
        } else {
#pragma unroll
            for (int l = 0; l < L; l++) y[l] = x[l] + a.Mrest[l];
            normalize<L>(y, a);
            if (limb_sign<L>(y) <= 0) {
#pragma unroll
                for (int l = 0; l < L; l++) x[l] += a.Mw[l];
                normalize<L>(x, a);
            }
        }
        neg = x[L - 1] < 0.0;
    }
    const int sm = neg ? (int)0x80000000u : 0;
#pragma unroll
    for (int l = 0; l < L; l++) x[l] = __hiloint2double(__double2hiint(x[l]) ^ sm, __double2loint(x[l]));
    normalize<L>(x, a);
    if (x[L - 1] < 0.0) {  // |C'| so small that the estimate's sign was wrong
#pragma unroll
        for (int l = 0; l < L; l++) x[l] = -x[l];
        normalize<L>(x, a);
        neg = !neg;
    }
    double T[L], e[L];
#pragma unroll
    for (int j = 0; j < L; j++) T[j] = x[L - 1 - j] * a.pow[L - 1 - j];
    double s = T[0];
#pragma unroll
    for (int j = 1; j < L; j++) {
        const double sn = s + T[j];
        e[j] = T[j] - (sn - s);
        s = sn;
    }
    const double h = __hiloint2double((__double2hiint(s) & 0x7FF00000) - (53 << 20), 0);  // half an ulp
    bool fix = false, below = false;
#pragma unroll
    for (int j = L - 1; j >= 1; j--) {
        fix = fix | (below & (e[j] == h));
        below = below | (T[j] != 0.0);
    }
    const double r0 = fix ? __builtin_fma(2.0, h, s) : s;
    const int ex = ((__double2hiint(r0) >> 20) & 0x7FF) - 1023 + e2;
    double r = __builtin_ldexp(r0, e2);
    r = ex < -1022 ? 0.0 : r;  // (only by a b far from any plan's: e2 >= -252 - 2 b, and C' = 0 for smaller maxima)
    r = neg ? -r : r;
    return r0 == 0.0 ? 0.0 : r;
}

// A workgroup of 2 x 2 waves computes a 64 x 64 tile, 32 x 32 per wave; two workgroups share a CU. The K
// steps of all moduli run one after another through a ring of NSTG stages of 8 KB, NSTG - 1 steps ahead.
// A step is bound by those copies, 34 bytes per clock and CU (4096 x 4096: 26 us per 64 of K, 15 moduli;
// a ring of 4 stages 29 us). Larger tiles per wave would halve them but need the limbs of 32 elements per
// lane in accumulation registers, which FP64 operations cannot read (1.5 times slower).
template <int L>
__global__ void __launch_bounds__(256, 2) gemm_crt_kernel(
    const int8_t* __restrict__ A, const int8_t* __restrict__ Bt, int K, long long sA, long long sB, int tiles_m,
    int tiles_n, FusedCrt<L> a, const int32_t* __restrict__ dA, const int32_t* __restrict__ dB, int M, int N,
    double* __restrict__ out, int ldo, uint32_t* __restrict__ fsrc, uint32_t* __restrict__ fdst) {
    if (blockIdx.x == 0 && threadIdx.x < 2) {  // the pass's range flags (crt_digits_kernel's move_flags)
        fdst[threadIdx.x] = fsrc[threadIdx.x];
        fsrc[threadIdx.x] = 0u;
    }
    constexpr int TI = 2, TJ = 2, NSTG = 6;
    constexpr int BA = 2 * TI, BB = 2 * TJ;  // 1 KB blocks of a stage
    constexpr int TM = 16 * BA, TN = 16 * BB;
    constexpr int STG = (BA + BB) * 1024;
    constexpr int LD = (BA + BB) / 4;        // copies per wave and stage
    __shared__ __attribute__((aligned(1024))) int8_t ring[NSTG * STG];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int one, tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, 1, one, tm, tn);
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
    const int nk = K / BK;
    const long long band = (long long)nk * 1024;
    const int8_t* Ab = A + (long long)tm * BA * band;
    const int8_t* Bb = Bt + (long long)tn * BB * band;
    const unsigned lane16 = 16u * lane;
    const int total = a.S * nk;
    // the step to load next is block lk of its modulus; past the end the last one again
    int lk = 0, lcount = 0;
    long long oA = 0, oB = 0;
    auto next_stage = [&]() {
        const int adv = lcount < total - 1;
        lcount += adv;
        lk += adv;
        oA += adv ? 1024 : 0;
        oB += adv ? 1024 : 0;
        const int wrap = lk == nk;
        lk = wrap ? 0 : lk;
        oA += wrap ? sA - band : 0;
        oB += wrap ? sB - band : 0;
    };
    auto issue = [&](int buf) {
#pragma unroll
        for (int j = 0; j < LD; j++) {
            const int q = 4 * j + wave;
            const int8_t* p = q < BA ? Ab + ((long long)q * band + oA) : Bb + ((long long)(q - BA) * band + oB);
            lds_copy_block(p, ring + buf * STG + q * 1024, lane16);
        }
    };
    const int wm = wave >> 1, wn = wave & 1;
    const int r = lane & 15, c = lane >> 4;
    const int foff = fragment16_offset(lane);
    v4i acc[TI][TJ];
    double x[TI][TJ][4][L];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            acc[i][j] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int l = 0; l < L; l++) x[i][j][q][l] = 0.0;
        }
#pragma unroll
    for (int s = 0; s < NSTG; s++) {
        issue(s);
        next_stage();
    }
    v4i xa[TI], xb[TJ], ya[TI], yb[TJ];
    auto read = [&](v4i* pa, v4i* pb, int buf) {
#pragma unroll
        for (int i = 0; i < TI; i++) pa[i] = *reinterpret_cast<const v4i*>(ring + buf * STG + (wm * TI + i) * 1024 + foff);
#pragma unroll
        for (int j = 0; j < TJ; j++) pb[j] = *reinterpret_cast<const v4i*>(ring + buf * STG + (BA + wn * TJ + j) * 1024 + foff);
    };
    wait_vmcnt<LD * (NSTG - 1)>();
    stage_barrier();
    read(xa, xb, 0);
    // Step u multiplies the fragments pa, pb read one step earlier and reads the next step's: stage u + 1 has
    // landed (all but NSTG - 2 stages' copies are complete) and this wave's reads of stage u are done, so
    // after the barrier stage u's buffer is refilled.
    int buf = 0, kk = 0, s = 0;
    auto step = [&](v4i* pa, v4i* pb, v4i* na, v4i* nb) {
        wait_vmcnt_lgkm0<LD * (NSTG - 2)>();
        stage_barrier();
        issue(__builtin_amdgcn_readfirstlane(buf));
        next_stage();
        buf = buf + 1 == NSTG ? 0 : buf + 1;
        read(na, nb, buf);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(pa[i], pb[j], acc[i][j], 0, 0, 0);
        if (++kk < nk) return;
        kk = 0;  // this modulus is done: its sums times W_s into the limbs
        double w[L];
#pragma unroll
        for (int l = 0; l < L; l++) w[l] = a.W[s][l];
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const double v = (double)acc[i][j][q];
#pragma unroll
                    for (int l = 0; l < L; l++) x[i][j][q][l] = __builtin_fma(v, w[l], x[i][j][q][l]);
                }
                acc[i][j] = v4i{0, 0, 0, 0};
            }
        s++;
    };
    int u = 0;
    for (; u + 1 < total; u += 2) {
        step(xa, xb, ya, yb);
        step(ya, yb, xa, xb);
    }
    if (u < total) step(xa, xb, ya, yb);
    wait_vmcnt<0>();  // drain the clamped tail copies before the workgroup ends
    const int gi = 2 * a.shift - 2 * a.b;
#pragma unroll
    for (int j = 0; j < TJ; j++) {
        const int col = tn * TN + (wn * TJ + j) * 16 + r;
        const int eb = col < N ? gi - dB[col] : 0;
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int row = tm * TM + (wm * TI + i) * 16 + 4 * c + q;
                const int ea = row < M ? dA[row] : 0;
                const double v = finish<L>(x[i][j][q], a, eb - ea);
                if (row < M && col < N) __builtin_nontemporal_store(v, &out[(long long)row * ldo + col]);
            }
    }
}

// w bits of the 8 little-endian words from bit at on, as a double.
double bits_at(const uint32_t* words, int at, int w) {
    uint64_t v = 0;
    for (int k = 0; k < 3; k++) {
        const int word = at / 32 + k, sh = 32 * k - at % 32;
        if (word >= 8) break;
        v |= sh >= 0 ? (sh < 64 ? (uint64_t)words[word] << sh : 0) : (uint64_t)words[word] >> -sh;
    }
    return (double)(v & ((1ull << w) - 1));
}

int bit_length(uint64_t v) { return v ? 64 - __builtin_clzll(v) : 0; }

template <int L>
void constants(const oz2_crt_dev* crt, int w, FusedCrt<L>& a) {
    a.S = crt->S;
    a.b = crt->b;
    a.shift = crt->shift;
    a.radix = std::ldexp(1.0, w);
    a.carry = std::ldexp(1.0, -w);
    uint32_t half[8], rest[8];
    uint32_t r = 0, borrow = 0;
    for (int k = 7; k >= 0; k--) {
        const uint64_t cur = ((uint64_t)r << 32) | crt->Mw[k];
        half[k] = (uint32_t)(cur >> 1);
        r = (uint32_t)(cur & 1u);
    }
    for (int k = 0; k < 8; k++) {
        const uint64_t d = (uint64_t)crt->Mw[k] - half[k] - borrow;
        rest[k] = (uint32_t)d;
        borrow = (uint32_t)(d >> 63);
    }
    double Md = 0.0;
    for (int k = 7; k >= 0; k--) Md = Md * 4294967296.0 + (double)crt->Mw[k];
    a.invM = 1.0 / Md;
    a.delta = 0x1p-20 + 2.0 / Md;
    for (int l = 0; l < L; l++) {
        a.Mw[l] = bits_at(crt->Mw, w * l, w);
        a.Mhalf[l] = bits_at(half, w * l, w);
        a.Mrest[l] = bits_at(rest, w * l, w);
        a.pow[l] = std::ldexp(1.0, w * l);
    }
    for (int s = 0; s < crt->S; s++) {
        uint32_t W[8];
        uint64_t carry = 0;
        for (int k = 0; k < 8; k++) {
            const uint64_t p = (uint64_t)crt->Q[s][k] * crt->y[s] + carry;
            W[k] = (uint32_t)p;
            carry = p >> 32;
        }
        for (int l = 0; l < L; l++) a.W[s][l] = bits_at(W, w * l, w);
    }
}

// M = prod m_s, Q_s m_s = M for every modulus, and S M within the nw words of the accumulator (the descriptor is the
// caller's: what is not so goes to the general route, where oz2_crt_digits_f64 refuses it).
bool consistent(const oz2_crt_dev* crt) {
    if (crt->nw < 3 || crt->nw > 8) return false;
    uint32_t M[9] = {1};
    for (int s = 0; s < crt->S; s++) {
        uint64_t carry = 0;
        for (int k = 0; k < 9; k++) {
            const uint64_t p = (uint64_t)M[k] * crt->m[s] + carry;
            M[k] = (uint32_t)p;
            carry = p >> 32;
        }
    }
    for (int k = 0; k < 8; k++)
        if (M[k] != crt->Mw[k]) return false;
    if (M[8]) return false;
    uint64_t over = 0;
    for (int k = 0; k < 8; k++) {
        const uint64_t p = (uint64_t)M[k] * (uint64_t)crt->S + over;
        if (k >= crt->nw && (uint32_t)p) return false;
        over = p >> 32;
    }
    if (over) return false;
    for (int s = 0; s < crt->S; s++) {
        uint64_t carry = 0;
        for (int k = 0; k < 8; k++) {
            const uint64_t p = (uint64_t)crt->Q[s][k] * crt->m[s] + carry;
            if ((uint32_t)p != M[k]) return false;
            carry = p >> 32;
        }
        if (carry) return false;
    }
    return true;
}

template <int L>
int launch(oz_dev* dev, const oz::FusedArgs& f, int w) {
    FusedCrt<L> a{};
    constants<L>(f.crt, w, a);
    const int tm = (f.M + 63) / 64, tn = (f.N + 63) / 64;
    oz::launch_product(dev, gemm_crt_kernel<L>, dim3((unsigned)(tm * tn)), dim3(256), f.A, f.Bt, f.K, f.sA, f.sB, tm, tn,
                       a, f.dA, f.dB, f.M, f.N, f.out, f.ldo, f.fsrc, f.fdst);
    return oz::launch_check(dev, "gemm_crt_kernel");
}

}  // namespace

namespace oz {

// Limb width and count: S max|C_s| 2^w <= 2^52 with |C_s| <= K 127^2, and L w bits for M. w >= 24, so that the
// quotient V / M < 2^28 is good to 2^-20.6 (at most 2 L + 8 roundings on the way, each within 2^-53 of 2^28) and
// finish settles every neighbour that delta, 2^-20, leaves open: with w = 18 (10 moduli, K = 65536) it is off by more.
bool fused_limbs(const oz2_crt_dev* crt, int K, int* width, int* limbs) {
    const int w = 52 - bit_length((uint64_t)crt->S * K * 127 * 127);
    int bits = 0;
    for (int k = 7; k >= 0 && !bits; k--)
        if (crt->Mw[k]) bits = 32 * k + 32 - __builtin_clz(crt->Mw[k]);
    if (w < 24 || !bits) return false;
    const int L = std::max(4, (bits + w - 1) / w);
    *width = w;
    *limbs = L;
    return L <= 6 && consistent(crt);
}

int launch_fused(oz_dev* dev, const FusedArgs& f) {
    int w = 0, L = 0;
    if (!fused_limbs(f.crt, f.K, &w, &L)) return fail(dev, OZ_ERR_ARG, "gemm_crt: the moduli do not fit the limbs");
    switch (L) {
    case 4: return launch<4>(dev, f, w);
    case 5: return launch<5>(dev, f, w);
    default: return launch<6>(dev, f, w);
    }
}

}  // namespace oz
