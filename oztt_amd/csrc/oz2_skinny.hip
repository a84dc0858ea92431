// Scheme II INT8 for a matrix on at most 64 columns: the residues of A are multiplied as they are made.
//
// Semantics: oz2_split_int8 of A, then oz2_gemm_digits with B's residue planes: the CRT digits
// k_s = (C_s y_s) mod m_s of the products, in one or two parts by the halves of K, whose digits add up.
//
// MI355X design. With N <= 64 the passes over memory are the time: at 8192 x 64 x 8192 A's 16 residue planes
// (1 GB) are written in 302 us and read back in 225, beside reading A itself (0.5 GB). Here the planes never
// exist. A workgroup of 8 waves takes 64 rows of A; per 64-wide K block
//   - its threads read the 64 x 64 elements (16 bytes of 8 lanes join to 128), make A' of each in balanced
//     bytes once and put it into LDS (32 KB, granules of two elements swizzled by the row);
//   - waves w and w + 4 take 16 rows each and half of the moduli each: a lane reads 16 consecutive A' of one
//     row, which are the bytes that lane brings to v_mfma_i32_16x16x64_i8, so the packed residues of a
//     modulus go straight into the MFMAs of the 64 columns, whose sums of all K stay in registers (128 per
//     lane, two waves per SIMD: with all moduli in one wave, one per SIMD, every latency showed, 1.9x slower);
//   - B's blocks (4 S KB per K block, 64 rows of planes) come into LDS once for the 8 waves, a block ahead.
// A's residues may be any representatives (the products are reduced), so the even modulus goes the way of the
// odd ones, whatever the planes' sequence makes of a tie, and a small modulus that of a multiple. A workgroup that met
// an element without a place in the bytes (its row has a range flag) puts the planes' own residues in its place at the
// end, so that flagged rows come out as the stages give them too.
// Bound by the VALU work of the residues (54% busy) and, for A's 64 KB rows, by the memory channels: without the
// reads of A the pass takes 88 us less, without B's copies 46, without the residues' VALU work 29.
// Whole pass, us, with planes -> here: 8192 x 64 x 8192: 645 -> 405; 8192 x 1 x 8192: 632 -> 413; 12288 x 64 x
// 4096: 499 -> 393; 16384 x 32 x 2048: 357 -> 239; 6144 x 64 x 1024 (192 workgroups): 95 -> 77.
#include "oz2_gemm_crt.hpp"
#include "oz2_pass.hpp"
#include "oz2_residue_gen.hpp"
#include "oz_gemm_tiles.hpp"

namespace {

using namespace ozg;

constexpr int kMaxS = 16;
constexpr int kBuf = kMaxS * 4096;             // a K block of B's planes

// Constants of a modulus m (128 <= m <= 255, h = m / 2; for a smaller modulus of the set, m is its largest multiple
// up to 255: the residues are representatives). With u = dot + 2 h + 2 L m (one MFMA) and
// v = u + dot = 2 (dot + h + L m) (a second one on top), q = floor(v magic / 2^32), magic = ceil(2^31 / m) < 2^24,
// is floor((dot + h) / m) + L exactly (v < 2^20, so the excess of magic adds less than 2^-12 < 1 / m), and
// u - q m = r + (2 h + L m) with r = dot + h mod m - h the symmetric residue. L m >= 2^17 > |dot| is chosen with
// 2 h + L m = 0 mod 256: the low byte of u - q m is r. So a residue takes two VALU instructions (24-bit multiply
// high and multiply-add) and its share of the packing, 2.75 against the 4.25 of reduce_odd_int with its shift
// and its offset, and the matrix cores, idle otherwise, make v. Both parities of m: for even m, h + h = m.
// m = 128 has no such magic (2^24): with 0, q = 0 and the byte is u's own, congruent to dot modulo 128 since 256 is a
// multiple of it, at most 128 in magnitude beside B's 64. tests/test_narrow_constants.py checks every m and every dot.
struct SkinnyConsts {
    uint32_t w[kMaxS][2], magic[kMaxS];
    int init[kMaxS], mneg[kMaxS];
    int even;  // the even modulus of the set or -1, with the constants of its sequence on the digits (residue_f)
    float m, rinv, c0, c1;
};

// Whether any of some elements has |x 2^d| >= 2^22 or is an infinity or NaN, by the upper words of split_integer3 (the
// integer part stands 12 bits below it). A' of the others fits its 8 bytes, |A'| < 2^63, and every residue of it is that
// of its digits; from 2^23 on the bytes are A' modulo 2^64, which is another residue for the even modulus. The scale
// leaves at most 2^(b - 40) <= 2^20 unless a range flag is raised for the row, wherever in the row its reason stands.
struct BeyondBytes {
    uint32_t top = 0;
    __device__ __forceinline__ void add(uint32_t T) { top = max(top, T - (0x41F80000u - 0x400u)); }
    __device__ __forceinline__ bool any() const { return top >= 0x800u; }
};

__device__ __forceinline__ int residue_byte(int u, int v, uint32_t magic, int mneg) {
    const uint32_t q = (uint32_t)(((unsigned long long)((uint32_t)v & 0xFFFFFFu) * (magic & 0xFFFFFFu)) >> 32);
    int x;  // u - q m modulo 2^24 (mneg = 2^24 - m)
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(x) : "v"(q), "s"(mneg), "v"(u));
    return x;
}

// P pairs of moduli per wave.
template <int P>
__global__ void __launch_bounds__(512) skinny_kernel(const double* __restrict__ A, int M, int K, int lda,
                                                     const int32_t* __restrict__ dA, const int8_t* __restrict__ pB, int nk,
                                                     long long sB, uint8_t* __restrict__ D, int ldd, long long sD, int groups,
                                                     int part_steps, int S, int wide, SkinnyConsts k, oz2::DigitConsts dc) {
    __shared__ __attribute__((aligned(1024))) int8_t lds[2 * kBuf];
    __shared__ v4i states[64 * 32];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = wave >> 2, band = wave & 3;
    const int part = __builtin_amdgcn_readfirstlane((int)blockIdx.x / groups);
    const int row0 = ((int)blockIdx.x - part * groups) * 64;
    const int st0 = part * part_steps, steps = min(nk, st0 + part_steps) - st0;
    // The K blocks in turn from one that differs by XCD (the last one again past the end): rows a power of two
    // apart would have all workgroups read the same memory channels at once, while those of one XCD should
    // read B's blocks together.
    const int turn = (int)(blockIdx.x % 8) * steps / 8;
    auto block = [&](int i) {
        const int b = min(i, steps - 1) + turn;
        return st0 + (b >= steps ? b - steps : b);
    };
    const int r = lane & 15, c = lane >> 4;
    const unsigned lane16 = 16u * lane;
    const int foff = fragment16_offset(lane);
    // this thread's elements: 2 lq + 16 j, + 1 (j = 0..3) of row lrow of the K block
    const int lrow = threadIdx.x >> 3, lq = threadIdx.x & 7;
    const int row = min(row0 + lrow, M - 1);
    const bool live = row0 + lrow < M;
    const double* a = A + (size_t)row * lda + 2 * lq;
    const int32_t delta = dA[row];
    // block `band` of this half's share of the planes of K block st
    auto issue = [&](int buf, int st) {
        for (int s = half; s < S; s += 2)
            lds_copy_block(pB + ((long long)s * sB + ((long long)band * nk + st) * 1024),
                           lds + __builtin_amdgcn_readfirstlane(buf * kBuf + (s * 4 + band) * 1024), lane16);
    };
    auto load = [&](double* x, int st) {
        const int k0 = st * 64;
        if (k0 + 64 <= K) {
            if (wide) {
                typedef double f64x2 __attribute__((ext_vector_type(2)));
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const f64x2 v = *reinterpret_cast<const f64x2*>(a + k0 + 16 * j);
                    x[2 * j] = v[0];
                    x[2 * j + 1] = v[1];
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = a[k0 + 16 * (e >> 1) + (e & 1)];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int kk = k0 + 16 * (e >> 1) + (e & 1);
                const double v = a[min(kk, K - 1 - 2 * lq)];
                x[e] = kk + 2 * lq < K ? v : 0.0;
            }
        }
    };
    BeyondBytes far;  // over all elements of this thread
    auto convert = [&](const double* x, v4i* g) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t a0[2], a1[2];
            float dig[3];
            far.add(split_integer3(live ? x[2 * j] : 0.0, delta, a0, dig));
            far.add(split_integer3(live ? x[2 * j + 1] : 0.0, delta, a1, dig));
            g[j] = v4i{(int)a0[0], (int)a0[1], (int)a1[0], (int)a1[1]};
        }
    };
    // granule g of a row at (g ^ row % 16): a wave's reads of 16 rows fall on all banks
    auto put = [&](const v4i* g) {
#pragma unroll
        for (int j = 0; j < 4; j++) states[32 * lrow + ((lq + 8 * j) ^ (lrow & 15))] = g[j];
    };
    // this wave's pairs of moduli: (s0 + 2 g, s0 + 2 g + 1); those from S on repeat the last modulus (no branches,
    // so that the compiler overlaps one pair's matrix products with the next one's residues) and are not stored
    const int s0 = half * 2 * P;
    // rows of the weights of a pair (ResidueGen, oz2_residue_gen.hpp): the lane's modulus and half
    const bool on = (lane >> 4) == ((lane & 15) >> 2), upper = (lane & 2) != 0;
    uint32_t w0[P], w1[P];
#pragma unroll
    for (int g = 0; g < P; g++) {
        const int s = s0 + 2 * g;
        const uint32_t x = (lane & 1) ? k.w[s + 1][0] : k.w[s][0], y = (lane & 1) ? k.w[s + 1][1] : k.w[s][1];
        w0[g] = on ? x : 0u;
        w1[g] = on ? y : 0u;
    }
    v4i acc[2 * P][4];
#pragma unroll
    for (int i = 0; i < 2 * P; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = v4i{0, 0, 0, 0};
    double x[8];
    v4i made[4];
    load(x, block(0));
    issue(0, block(0));
    convert(x, made);
    put(made);
    load(x, block(1));
    for (int i = 0; i < steps; i++) {
        const int buf = i & 1;
        // this block's A' and copies, the next block's elements; the last block's reads
        wait_vmcnt_lgkm0<0>();
        stage_barrier();
        v4i e[8];
#pragma unroll
        for (int j = 0; j < 8; j++) e[j] = states[32 * (16 * band + r) + ((8 * c + j) ^ r)];
        convert(x, made);
        wait_vmcnt_lgkm0<0>();
        stage_barrier();  // A' of this block is read
        put(made);
        issue(buf ^ 1, block(i + 1));
        load(x, block(i + 2));
        const int8_t* frag = lds + buf * kBuf + foff;
#pragma unroll
        for (int g = 0; g < P; g++) {
            const int s = s0 + 2 * g, f = min(s, S - 1), t = min(s + 1, S - 1);
            const v4i wa = {upper ? 0 : (int)w0[g], upper ? 0 : (int)w1[g], upper ? (int)w0[g] : 0, upper ? (int)w1[g] : 0};
            const int d0 = k.init[s], d1 = k.init[s + 1];
            const v4i init = {d0, d1, d0, d1};
            uint32_t p0[4], p1[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                int x0[4], x1[4];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const v4i u = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa, e[2 * q + h], init, 0, 0, 0);
                    const v4i v = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa, e[2 * q + h], u, 0, 0, 0);
                    x0[2 * h] = residue_byte(u[0], v[0], k.magic[s], k.mneg[s]);
                    x1[2 * h] = residue_byte(u[1], v[1], k.magic[s + 1], k.mneg[s + 1]);
                    x0[2 * h + 1] = residue_byte(u[2], v[2], k.magic[s], k.mneg[s]);
                    x1[2 * h + 1] = residue_byte(u[3], v[3], k.magic[s + 1], k.mneg[s + 1]);
                }
                p0[q] = pack4(x0[0], x0[1], x0[2], x0[3]);
                p1[q] = pack4(x1[0], x1[1], x1[2], x1[3]);
            }
            const v4i f0 = {(int)p0[0], (int)p0[1], (int)p0[2], (int)p0[3]};
            const v4i f1 = {(int)p1[0], (int)p1[1], (int)p1[2], (int)p1[3]};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4i b0 = *reinterpret_cast<const v4i*>(frag + f * 4096 + j * 1024);
                const v4i b1 = *reinterpret_cast<const v4i*>(frag + t * 4096 + j * 1024);
                acc[2 * g][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f0, b0, acc[2 * g][j], 0, 0, 0);
                acc[2 * g + 1][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f1, b1, acc[2 * g + 1][j], 0, 0, 0);
            }
        }
    }
    wait_vmcnt_lgkm0<0>();  // the last block's copies, issued twice
    __syncthreads();
    // Elements beyond their bytes (an operand with a range flag) are what the procedure makes of them, also in the even
    // modulus, whose sequence on the digits then is no residue of A'. A workgroup that met any goes over its elements
    // again, and in the K blocks that hold some it takes these elements' products back out of the sums and puts in
    // those of the planes' residues: of A' the same byte as above, by the same steps (every product is exact modulo
    // 2^32, so only the sums that stand at the end have to fit). 6272 x 64 x 1536, 16 moduli, three such elements:
    // 149 us (108 without any; 320 with every block of these rows computed again; 140 by the planes).
    int* seen = reinterpret_cast<int*>(states);
    if (lane == 0) seen[wave] = 0;
    if (far.any() || delta >= 541) seen[wave] = 1;
    __syncthreads();
    bool again = false;
#pragma unroll
    for (int i = 0; i < 8; i++) again |= seen[i] != 0;
    if (__builtin_expect(again, 0)) {
        // (the sums leave few registers: the lane's place is taken afresh)
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int lane = t & 63, lrow = t >> 3, lq = t & 7, row = min(row0 + lrow, M - 1);
        const bool live = row0 + lrow < M;
        const int32_t delta = dA[row];
        const int foff = fragment16_offset(lane);
        for (int i = 0; i < steps; i++) {
            auto element = [&](int e) {
                const int kk = (st0 + i) * 64 + 2 * lq + 16 * (e >> 1) + (e & 1);
                const double v = A[(size_t)row * lda + min(kk, K - 1)];
                return live && kk < K ? v : 0.0;
            };
            uint32_t mine = 0;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                uint32_t a[2];
                float dig[3];
                BeyondBytes f;
                f.add(split_integer3(element(e), delta, a, dig));
                mine |= (f.any() || delta >= 541 ? 1u : 0u) << e;
            }
            // the votes of two blocks in turn: those of this one are read before the next barrier
            int* vote = seen + 8 + 8 * (i & 1);
            const bool any = __ballot(mine != 0) != 0;
            if (lane == 0) vote[wave] = any;
            __syncthreads();
            int votes = 0;
#pragma unroll
            for (int w = 0; w < 8; w++) votes |= vote[w];
            if (!__builtin_amdgcn_readfirstlane(votes)) continue;
            for (int q = t; q < 256 * S; q += 512) {
                reinterpret_cast<v4i*>(lds)[q] = v4i{0, 0, 0, 0};
                reinterpret_cast<v4i*>(lds + kBuf)[q] = v4i{0, 0, 0, 0};
            }
            __syncthreads();
            for (; mine; mine &= mine - 1) {
                const int e = __builtin_ctz(mine);
                const double v = element(e);
                uint32_t taken[2], a[2];
                float dig[3];
                split_integer3(v, delta, taken, dig);
                make_digits<3>(v, delta, dig);
                balanced_bytes<3>(dig, a);
                int8_t* at = lds + 64 * lrow + 2 * lq + 16 * (e >> 1) + (e & 1);
                for (int s = 0; s < S; s++) {
                    const int dot = __builtin_amdgcn_sdot4((int)taken[1], (int)k.w[s][1],
                                                           __builtin_amdgcn_sdot4((int)taken[0], (int)k.w[s][0], 0, false), false);
                    const int u = dot + k.init[s];
                    const float m = (float)((1 << 24) - k.mneg[s]);
                    at[kBuf + 4096 * s] = (int8_t)residue_byte(u, u + dot, k.magic[s], k.mneg[s]);
                    at[4096 * s] = (int8_t)(int)(s == k.even ? residue_f<3>(dig, k.m, k.rinv, k.c0, k.c1, 0.0f, 0.0f)
                                                             : residue_odd<2>(a, k.w[s], m, 1.0f / m));
                }
            }
            __syncthreads();
#pragma unroll
            for (int g = 0; g < 2 * P; g++) {
                const int s = min(s0 + g, S - 1);
                const int8_t* at = lds + 4096 * s + 64 * (16 * band + (lane & 15)) + 16 * (lane >> 4);
                const v4i in = *reinterpret_cast<const v4i*>(at), out = *reinterpret_cast<const v4i*>(at + kBuf);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4i b = *reinterpret_cast<const v4i*>(pB + ((long long)s * sB + ((long long)j * nk + st0 + i) * 1024 + foff));
                    const v4i less = __builtin_amdgcn_mfma_i32_16x16x64_i8(out, b, -acc[g][j], 0, 0, 0);
                    acc[g][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(in, b, -less, 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    // digits through 4 KB of the ring per wave (its LDS operations are in order), 16 sums per lane and modulus
    int32_t* tile = reinterpret_cast<int32_t*>(lds) + wave * 1024;
#pragma unroll
    for (int i = 0; i < 2 * P; i++) {
        const int s = s0 + i;
        if (s < S) {
            const uint32_t m = dc.m[s];
            const double md = (double)m, yr = (double)dc.y[s] / md;
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) tile[staged_group<4>(4 * c + q, j) + r] = acc[i][j][q];
            store_digits16(tile + staged_group<4>(lane >> 2, lane & 3),
                           D + (long long)s * sD + (long long)(row0 + 16 * band + (lane >> 2)) * ldd + 64 * part +
                               16 * (lane & 3),
                           yr, md);
        }
    }
}

}  // namespace

namespace oz2pass {

// The parts of K (0: the kernel does not take the pass). It takes three digits and at most 16 moduli, and pays
// from where normalization and residues are no longer one launch (K > 512, oz2_prep.hip) and its workgroups, one
// per CU, fill the chip: with 192 of them (M = 6144, two parts) the pass takes 77 us against 95 at K = 1024. And from a
// number of moduli on, whose planes are what it saves while it makes A' and the matrix products of at least 8 (with
// planes -> here, 64 columns): 8192 x 1024 with 3 moduli 58 against 56 us, with 2 53 against 55, x 2048 89 against 87
// and 79 against 85; with three quarters of the CUs 6144 x 2048 with 6 94 -> 84, with 5 82 either way, with 4 79 against 82, 12288
// x 2048 with 5 136 against 145.
int skinny_parts(int cus, const oz2_moduli_dev* mo, int M, int N, int K) {
    int evens = 0;  // (more than one, and the planes are all of the sequence on the digits)
    for (int s = 0; s < mo->S; s++) evens += (int)mo->m[s] % 2 == 0;
    if (N > 64 || mo->nd != 3 || mo->S < 4 || mo->S > kMaxS || K < 1024 || evens > 1) return 0;
    const long long groups = (M + 63ll) / 64;
    for (int parts = 1; parts <= 2; parts++) {
        const long long w = groups * parts, rounds = (w + cus - 1) / cus;
        if (4 * w >= 3 * rounds * cus)  // at least three quarters of the CUs in every round
            return mo->S >= 6 || 10 * w >= 9 * rounds * cus ? parts : 0;
    }
    return 0;
}

NarrowModulus narrow_modulus(int m1) {
    const int m = 255 / m1 * m1, h = m / 2;
    NarrowModulus c{};
    int p = 1;  // 256^j mod m, symmetric
    for (int j = 0; j < 8; j++, p = p * 256 % m)
        c.w[j / 4] |= (uint32_t)((p > h ? p - m : p) & 0xFF) << (8 * (j % 4));
    int L = ((1 << 17) + m - 1) / m;
    while ((2 * h + L * m) % 256) L++;
    c.magic = m == 128 ? 0u : (uint32_t)(((1ull << 31) + m - 1) / m);
    c.init = 2 * h + 2 * L * m;
    c.mneg = (1 << 24) - m;
    return c;
}

int launch_skinny(oz_dev* dev, const double* A, int M, int K, int lda, const int32_t* dA, const int8_t* pB, int Kg,
                  uint8_t* D, int ldd, long long sD, int parts, const oz2_moduli_dev* mo, const oz2_crt_dev* crt) {
    SkinnyConsts k{};
    k.even = -1;
    for (int s = 0; s < mo->S; s++)
        if ((int)mo->m[s] % 2 == 0) {
            k.even = s;
            k.m = mo->m[s];
            k.rinv = mo->rinv[s];
            k.c0 = mo->c[0][s];
            k.c1 = mo->c[1][s];
        }
    for (int i = 0; i < kMaxS; i++) {
        const NarrowModulus c = narrow_modulus((int)mo->m[std::min(i, mo->S - 1)]);
        k.w[i][0] = c.w[0];
        k.w[i][1] = c.w[1];
        k.magic[i] = c.magic;
        k.init[i] = c.init;
        k.mneg[i] = c.mneg;
    }
    oz2::DigitConsts dc{};
    for (int s = 0; s < mo->S; s++) {
        dc.m[s] = crt->m[s];
        dc.y[s] = crt->y[s];
    }
    const int groups = (M + 63) / 64, nk = Kg / 64, part_steps = (nk + parts - 1) / parts;
    const int wide = lda % 2 == 0 && !((uintptr_t)A & 15);
    const auto launch = [&](auto kernel) {
        oz::launch_product(dev, kernel, dim3((unsigned)(groups * parts)), dim3(512), A, M, K, lda, dA, pB, nk, 64ll * Kg, D, ldd, sD,
                           groups, part_steps, mo->S, wide, k, dc);
    };
    mo->S <= 8 ? launch(skinny_kernel<2>) : mo->S <= 12 ? launch(skinny_kernel<3>) : launch(skinny_kernel<4>);
    return oz::launch_check(dev, "skinny_kernel");
}

}  // namespace oz2pass
