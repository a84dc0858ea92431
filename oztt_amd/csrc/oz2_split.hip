// A6-A8: Scheme II splitting of FP64 operands into int8 residue planes.
//
// Semantics (reference f64_tf.h:141-172 split_f64, slice_tf_core.h:67-76 tf_load_f64, digits.h:80-112
// oz2_make_digits, digits.h:165-179 oz2_residue, modslice_int8.cpp:60-95). The residues must equal
// the reference's bit for bit, and the reference defines them through a sequence of binary32
// operations: round-to-nearest-even, no fused multiply-add, denormal inputs and outputs flushed to
// zero. This file is compiled with -ffp-contract=off (no implicit contraction) and
// -fgpu-flush-denormals-to-zero (the kernels run with FP32 denormals flushed, the hardware
// equivalent of that rule). The signs of zeros may differ from the reference's model (its products
// with a zero factor are +0); a zero's sign never changes a digit or residue value.
//
// Per element x with exponent delta d:
//   1. x*2^d -> triple-float (hi, mid, lo) with integer operations on the FP64 words (exact);
//   2. nd digits: digit = rint(hi); hi -= digit; between digits the triple is multiplied by 2^20
//      and renormalized with two TwoSums and a FastTwoSum (only hi is ever rounded, so A' can be a
//      neighbour of the nearest integer; the reference documents |A'-X| <= 1);
//   3. per modulus: r = MR(d0 + MR(d1)*c0 + MR(d2)*c1) (nd = 3; 4/5 digits reduce in between),
//      MR(v) = v - rint(v*rinv)*m. Every product and sum there is an exact integer below 2^24
//      except the rounded v*rinv, so writing MR as rint + fma gives the same value.
//
// MI355X design. Layouts 2/3 (the GEMM's OZ_BLOCK tiles, the production path) run the blocked
// splitter of oz_tf32.hpp: one wave per 1 KB block, one contiguous 1 KB store per plane. Layouts 0/1
// (plain row-major planes): one thread per 4 elements along the contiguous dimension of the plane,
// so every store is a 32-bit word; layout 1 is transposed through LDS. The kernels are bound by
// their VALU work (about 12 operations per element and modulus), not by HBM.
#pragma clang fp contract(off)

#include "oz2_residue_gen.hpp"

namespace {

// Layout 0: planes[s][r][c], thread = 4 consecutive c of one row r; grid covers prow x pld.
template <int ND>
__global__ void __launch_bounds__(256) split_row_kernel(const double* __restrict__ X, int rows, int cols, int ld,
                                                        int mode, const int32_t* __restrict__ delta, SplitConsts k,
                                                        int S, uint32_t* __restrict__ planes, int prow, int pq,
                                                        long long pstride_words) {
    const long long q = (long long)blockIdx.x * 256 + threadIdx.x;  // word index within a plane
    if (q >= (long long)prow * pq) return;
    const int r = (int)(q / pq);
    const int c0 = (int)(q % pq) * 4;
    float dig[4][ND];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int c = c0 + e;
        if (r < rows && c < cols) {
            const int32_t d = mode == 0 ? delta[r] : delta[c];
            make_digits<ND>(X[(size_t)r * ld + c], d, dig[e]);
        } else {
#pragma unroll
            for (int j = 0; j < ND; j++) dig[e][j] = 0.0f;
        }
    }
    uint32_t* out = planes + q;
    for (int s = 0; s < S; s++)
        out[(long long)s * pstride_words] =
            pack4(residue<ND>(dig[0], k, s), residue<ND>(dig[1], k, s), residue<ND>(dig[2], k, s), residue<ND>(dig[3], k, s));
}

// Layout 1: planes[s][c][r] (transposed), tile of 64 columns x 64 rows per workgroup. Thread
// (cc = t%64, g = t/64) computes the 16 elements rows g*16..g*16+15 of column cc; the words go
// through LDS so that the stores are 64-byte row segments.
template <int ND>
__global__ void __launch_bounds__(256) split_tran_kernel(const double* __restrict__ X, int rows, int cols, int ld,
                                                         int mode, const int32_t* __restrict__ delta, SplitConsts k,
                                                         int S, uint32_t* __restrict__ planes, int pld_words,
                                                         long long pstride_words) {
    __shared__ uint32_t tile[64][17];  // [column][row word], padded against bank conflicts
    const int t = threadIdx.x;
    const int cc = t & 63, g = t >> 6;
    const int c = blockIdx.x * 64 + cc;  // column of X = row of the plane
    const int rbase = blockIdx.y * 64 + g * 16;
    float dig[16][ND];
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const int r = rbase + e;
        if (r < rows && c < cols) {
            const int32_t d = mode == 0 ? delta[r] : delta[c];
            make_digits<ND>(X[(size_t)r * ld + c], d, dig[e]);
        } else {
#pragma unroll
            for (int j = 0; j < ND; j++) dig[e][j] = 0.0f;
        }
    }
    // store phase mapping: thread -> plane row blockIdx.x*64 + t/4, words (t%4)*4 .. +4
    const int orow = blockIdx.x * 64 + (t >> 2);
    const int ow = blockIdx.y * 16 + (t & 3) * 4;
    for (int s = 0; s < S; s++) {
#pragma unroll
        for (int w = 0; w < 4; w++)
            tile[cc][g * 4 + w] = pack4(residue<ND>(dig[4 * w], k, s), residue<ND>(dig[4 * w + 1], k, s),
                                        residue<ND>(dig[4 * w + 2], k, s), residue<ND>(dig[4 * w + 3], k, s));
        __syncthreads();
        uint32_t* out = planes + (long long)s * pstride_words + (long long)orow * pld_words + ow;
        const uint4 v = make_uint4(tile[t >> 2][(t & 3) * 4], tile[t >> 2][(t & 3) * 4 + 1], tile[t >> 2][(t & 3) * 4 + 2],
                                   tile[t >> 2][(t & 3) * 4 + 3]);
        *reinterpret_cast<uint4*>(out) = v;
        __syncthreads();
    }
}

// The reference's sequence for every modulus (sets with more than one even modulus, which a
// pairwise coprime plan never has): the state is the nd digits.
template <int ND>
struct ResidueChainGen {
    SplitConsts k;
    struct State {
        float dig[ND];
    };
    __device__ __forceinline__ void load(State& st, double x, int32_t d) const { make_digits<ND>(x, d, st.dig); }
    __device__ __forceinline__ int plane(State& st, int s) const { return residue<ND>(st.dig, k, s); }
    OZ_PLANES_FROM_PLANE
};

template <int ND>
__global__ void digits_kernel(const double* __restrict__ X, int rows, int cols, int ld, int mode,
                              const int32_t* __restrict__ delta, float* __restrict__ out) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)rows * cols) return;
    const int r = (int)(i / cols), c = (int)(i % cols);
    float dig[ND];
    make_digits<ND>(X[(size_t)r * ld + c], mode == 0 ? delta[r] : delta[c], dig);
#pragma unroll
    for (int j = 0; j < ND; j++) out[i * ND + j] = dig[j];
}

template <class GEN>
int launch_blocked(oz_dev* dev, const double* X, int rows, int cols, int ld, int mode, const int32_t* delta,
                   const GEN& gen, int S, int8_t* planes, int layout, int pld, long long nblocks, long long pstride) {
    const int kblocks = pld / 64;
    const unsigned grid = oz::ceil_div(nblocks, 4);
    if (layout == 2)
        hipLaunchKernelGGL((split_block_kernel<GEN, false>), dim3(grid), dim3(256), 0, dev->stream, X, rows, cols, ld,
                           mode, delta, gen, S, reinterpret_cast<uint4*>(planes), kblocks, nblocks, pstride / 16);
    else
        hipLaunchKernelGGL((split_block_kernel<GEN, true>), dim3(grid), dim3(256), 0, dev->stream, X, rows, cols, ld,
                           mode, delta, gen, S, reinterpret_cast<uint4*>(planes), kblocks, nblocks, pstride / 16);
    return oz::launch_check(dev, "split_block_kernel");
}

template <int ND>
int launch_split(oz_dev* dev, const double* X, int rows, int cols, int ld, int mode, const int32_t* delta,
                 const SplitConsts& k, int S, int8_t* planes, int layout, int prow, int pld, long long pstride,
                 bool one_even) {
    if (layout == 0) {
        const int pq = pld / 4;
        const long long words = (long long)prow * pq;
        hipLaunchKernelGGL(split_row_kernel<ND>, dim3(oz::ceil_div(words, 256)), dim3(256), 0, dev->stream, X, rows,
                           cols, ld, mode, delta, k, S, reinterpret_cast<uint32_t*>(planes), prow, pq, pstride / 4);
        return oz::launch_check(dev, "split_row_kernel");
    }
    if (layout >= 2) {
        const long long nblocks = (long long)(prow / 16) * (pld / 64);
        if (one_even)
            return launch_blocked(dev, X, rows, cols, ld, mode, delta, ResidueGen<ND>{k}, S, planes, layout, pld,
                                  nblocks, pstride);
        return launch_blocked(dev, X, rows, cols, ld, mode, delta, ResidueChainGen<ND>{k}, S, planes, layout, pld,
                              nblocks, pstride);
    }
    // transposed: plane rows = columns of X (prow of them, multiple of 64); plane bytes = rows of X
    hipLaunchKernelGGL(split_tran_kernel<ND>, dim3(prow / 64, pld / 64), dim3(256), 0, dev->stream, X, rows, cols, ld,
                       mode, delta, k, S, reinterpret_cast<uint32_t*>(planes), pld / 4, pstride / 4);
    return oz::launch_check(dev, "split_tran_kernel");
}

// Both operands in pieces of 64 E elements per wave (the first ceil(nA / 4) workgroups split A): for
// operands of few blocks, where 16 elements per lane leave SIMDs idle and every wave's chain is long. The
// whole pass with 16 -> 4 elements per lane, us: 128 x 128 x 512 32.0 -> 27.1, 256 x 256 x 1024 34.0 ->
// 30.5, 1024^3 (2048 blocks) 58.2 -> 56.6; 2048 x 1024 x 1024 (3072 blocks) 90.2 against 93.7: every wave
// loads the constants and addresses of its moduli for a quarter of the elements.
template <int ND, int E>
__global__ void __launch_bounds__(256) split_pieces_kernel(const double* __restrict__ A, int M, int K, int lda,
                                                           const int32_t* __restrict__ dA, uint8_t* __restrict__ pA,
                                                           long long nA, long long sA, const double* __restrict__ B, int N,
                                                           int ldb, const int32_t* __restrict__ dB,
                                                           uint8_t* __restrict__ pB, long long nB, long long sB,
                                                           int kblocks, ResidueGen<ND, E> gen) {
    constexpr int Q = 16 / E;
    __shared__ __attribute__((aligned(16))) uint8_t image[4][64 * E];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long gA = (nA + 3) / 4;
    const bool rows = (long long)blockIdx.x < gA;
    const long long piece = ((long long)blockIdx.x - (rows ? 0 : gA)) * 4 + wave;
    if (piece >= (rows ? nA : nB)) return;
    const int q = (int)(piece % Q), br = (int)(piece / Q / kblocks), kb = (int)(piece / Q % kblocks);
    double x[E];
    typename ResidueGen<ND, E>::State st[E];
    FarElements far;
    if (rows) {
        int32_t d[E];
        load_piece<E, true>(A, M, K, lda, br, kb, q, lane, x);
#pragma unroll
        for (int e = 0; e < E; e++) d[e] = dA[min(br * 16 + q * E + e, M - 1)];
#pragma unroll
        for (int e = 0; e < E; e++) gen.load(st[e], x[e], d[e], far);
        gen.redo(st, far, [&](int e, double& v, int32_t& w) {
            v = piece_element<E, true>(A, M, K, lda, br, kb, q, e);
            w = dA[min(br * 16 + q * E + e, M - 1)];
        });
        emit_piece<ND, E, true>(gen, st, pA, sA, br, kblocks, kb, q, lane, image[wave]);
    } else {
        load_piece<E, false>(B, K, N, ldb, br, kb, q, lane, x);
        const int32_t d = dB[min(br * 16 + (lane >> 2), N - 1)];
#pragma unroll
        for (int e = 0; e < E; e++) gen.load(st[e], x[e], d, far);
        gen.redo(st, far, [&](int e, double& v, int32_t& w) {
            v = piece_element<E, false>(B, K, N, ldb, br, kb, q, e);
            w = d;
        });
        emit_piece<ND, E, false>(gen, st, pB, sB, br, kblocks, kb, q, lane, nullptr);
    }
}

template <int ND, int E>
int launch_pieces(oz_dev* dev, const double* A, int M, int K, int lda, const int32_t* dA, const double* B, int N, int ldb,
                  const int32_t* dB, const SplitConsts& k, int8_t* pA, int8_t* pB, int Mg, int Ng, int Kg) {
    const int kblocks = Kg / 64;
    const long long nA = (long long)(Mg / E) * kblocks, nB = (long long)(Ng / E) * kblocks;
    hipLaunchKernelGGL((split_pieces_kernel<ND, E>), dim3((unsigned)((nA + 3) / 4 + (nB + 3) / 4)), dim3(256), 0,
                       dev->stream, A, M, K, lda, dA, reinterpret_cast<uint8_t*>(pA), nA, (long long)Mg * Kg, B, N, ldb, dB,
                       reinterpret_cast<uint8_t*>(pB), nB, (long long)Ng * Kg, kblocks, ResidueGen<ND, E>{k});
    return oz::launch_check(dev, "split_pieces_kernel");
}

template <int ND>
int launch_pair(oz_dev* dev, const double* A, int M, int K, int lda, const int32_t* dA, const double* B, int N,
                int ldb, const int32_t* dB, const SplitConsts& k, int S, int8_t* pA, int8_t* pB, int Mg, int Ng,
                int Kg, bool one_even) {
    const int kblocks = Kg / 64;
    const long long nbA = (long long)(Mg / 16) * kblocks, nbB = (long long)(Ng / 16) * kblocks;
    const long long sA = (long long)Mg * Kg / 16, sB = (long long)Ng * Kg / 16;
    const long long grid = (nbA + 3) / 4 + (nbB + 3) / 4;
    if (grid > 0x7FFFFFFFll) return oz::fail(dev, OZ_ERR_ARG, "oz2_split_pair_int8: grid too large");
    auto* qA = reinterpret_cast<uint4*>(pA);
    auto* qB = reinterpret_cast<uint4*>(pB);
    // few blocks: four waves share one (2048 blocks are two waves per SIMD otherwise)
    if (one_even && nbA + nbB <= 8ll * dev->cus)
        return launch_pieces<ND, 4>(dev, A, M, K, lda, dA, B, N, ldb, dB, k, pA, pB, Mg, Ng, Kg);
    if (one_even)
        hipLaunchKernelGGL((split_pair_kernel<ResidueGen<ND>>), dim3((unsigned)grid), dim3(256), 0, dev->stream, A, M,
                           K, lda, dA, qA, nbA, sA, B, N, ldb, dB, qB, nbB, sB, kblocks, ResidueGen<ND>{k}, S);
    else
        hipLaunchKernelGGL((split_pair_kernel<ResidueChainGen<ND>>), dim3((unsigned)grid), dim3(256), 0, dev->stream,
                           A, M, K, lda, dA, qA, nbA, sA, B, N, ldb, dB, qB, nbB, sB, kblocks, ResidueChainGen<ND>{k},
                           S);
    return oz::launch_check(dev, "split_pair_kernel");
}

}  // namespace

extern "C" int oz2_split_int8(oz_dev* dev, const double* X, int rows, int cols, int ld, int mode,
                              const int32_t* delta, const oz2_moduli_dev* mo, int8_t* planes, int layout, int prow,
                              int pld, long long plane_stride) {
    if (int st = oz::use(dev)) return st;
    if (int st = check_moduli(dev, mo)) return st;
    if (!X || !delta || !planes || rows <= 0 || cols <= 0 || ld < cols || (mode != 0 && mode != 1) || layout < 0 ||
        layout > 3)
        return oz::fail(dev, OZ_ERR_ARG, "oz2_split_int8: invalid arguments");
    // The plane must hold the operand: layouts 0/2 rows x cols, layouts 1/3 cols x rows.
    const bool tran = layout == 1 || layout == 3;
    const int need_rows = tran ? cols : rows, need_ld = tran ? rows : cols;
    const bool blocked = layout >= 2;
    if (prow < need_rows || pld < need_ld || pld % 64 != 0 || (layout == 1 && prow % 64 != 0) ||
        (blocked && (prow % 16 != 0 || plane_stride % 1024 != 0)) || plane_stride < (long long)prow * pld ||
        plane_stride % 16 != 0 || ((uintptr_t)planes & 15u))
        return oz::fail(dev, OZ_ERR_ARG, "oz2_split_int8: plane geometry %dx%d (stride %lld) does not fit", prow, pld,
                        plane_stride);
    int evens = 0;
    const SplitConsts k = split_consts(mo, &evens);
    switch (mo->nd) {
    case 3:
        return launch_split<3>(dev, X, rows, cols, ld, mode, delta, k, mo->S, planes, layout, prow, pld, plane_stride,
                               evens <= 1);
    case 4:
        return launch_split<4>(dev, X, rows, cols, ld, mode, delta, k, mo->S, planes, layout, prow, pld, plane_stride,
                               evens <= 1);
    default:
        return launch_split<5>(dev, X, rows, cols, ld, mode, delta, k, mo->S, planes, layout, prow, pld, plane_stride,
                               evens <= 1);
    }
}

extern "C" int oz2_digits_f32(oz_dev* dev, const double* X, int rows, int cols, int ld, int mode,
                              const int32_t* delta, int nd, float* digits) {
    if (int st = oz::use(dev)) return st;
    if (!X || !delta || !digits || rows <= 0 || cols <= 0 || ld < cols || nd < 3 || nd > 5 || (mode != 0 && mode != 1))
        return oz::fail(dev, OZ_ERR_ARG, "oz2_digits_f32: invalid arguments");
    const unsigned grid = oz::ceil_div((long long)rows * cols, 256);
    if (nd == 3)
        hipLaunchKernelGGL(digits_kernel<3>, dim3(grid), dim3(256), 0, dev->stream, X, rows, cols, ld, mode, delta, digits);
    else if (nd == 4)
        hipLaunchKernelGGL(digits_kernel<4>, dim3(grid), dim3(256), 0, dev->stream, X, rows, cols, ld, mode, delta, digits);
    else
        hipLaunchKernelGGL(digits_kernel<5>, dim3(grid), dim3(256), 0, dev->stream, X, rows, cols, ld, mode, delta, digits);
    return oz::launch_check(dev, "digits_kernel");
}

extern "C" int oz2_split_pair_int8(oz_dev* dev, const double* A, int M, int K, int lda, const int32_t* dA,
                                   const double* B, int N, int ldb, const int32_t* dB, const oz2_moduli_dev* mo,
                                   int8_t* planesA, int8_t* planesB, int Mg, int Ng, int Kg) {
    if (int st = oz::use(dev)) return st;
    if (int st = check_moduli(dev, mo)) return st;
    if (!A || !B || !dA || !dB || !planesA || !planesB || M <= 0 || N <= 0 || K <= 0 || lda < K || ldb < N)
        return oz::fail(dev, OZ_ERR_ARG, "oz2_split_pair_int8: invalid arguments");
    if (Mg < M || Ng < N || Kg < K || Mg % 16 || Ng % 16 || Kg % 64 || ((uintptr_t)planesA & 15u) ||
        ((uintptr_t)planesB & 15u))
        return oz::fail(dev, OZ_ERR_ARG, "oz2_split_pair_int8: plane geometry %dx%d / %dx%d does not fit", Mg, Kg, Ng,
                        Kg);
    int evens = 0;
    const SplitConsts k = split_consts(mo, &evens);
    switch (mo->nd) {
    case 3: return launch_pair<3>(dev, A, M, K, lda, dA, B, N, ldb, dB, k, mo->S, planesA, planesB, Mg, Ng, Kg, evens <= 1);
    case 4: return launch_pair<4>(dev, A, M, K, lda, dA, B, N, ldb, dB, k, mo->S, planesA, planesB, Mg, Ng, Kg, evens <= 1);
    default: return launch_pair<5>(dev, A, M, K, lda, dA, B, N, ldb, dB, k, mo->S, planesA, planesB, Mg, Ng, Kg, evens <= 1);
    }
}
