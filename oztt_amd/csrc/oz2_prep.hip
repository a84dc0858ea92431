// Scheme II INT8, K <= 512: normalization (A5) and residue planes (A6-A8) of both operands in one launch.
//
// Semantics: oz_scale_pair_f64 (ceil mode 1) followed by oz2_split_pair_int8, the same deltas, flags and
// residues bit for bit (the same key, triple and residue functions).
//
// MI355X design: a workgroup takes one 16-row band of A (or 16 columns of B) over the whole of K and holds
// it in registers, so its maxima are known before it is split, it is read once, and one launch (and the
// wait for it) goes. A wave holds E rows (E consecutive K of a column) of a 64-wide K block, 64 E elements;
// the band takes (K/64)(16/E) waves, at most 16: E = 4 up to K = 256, 8 up to 512. Small operands are bound
// by the latency of one wave's chain (its elements one after another through digits and moduli: 14.6 us
// at 128^3 with 16 elements per lane), so E is the smallest that fits. The maxima meet in LDS (a DPP
// maximum over 16 lanes, then ds_max).
#include "oz2_pass.hpp"
#include "oz2_residue_gen.hpp"
#include "oz_scale_key.hpp"

namespace {

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false));
}

template <int ND, int E>
__global__ void __launch_bounds__(1024, 8) prep_kernel(const double* __restrict__ A, int M, int K, int lda,
                                                    int32_t* __restrict__ dA, uint8_t* __restrict__ pA, long long sA,
                                                    int bandsA, const double* __restrict__ B, int N, int ldb,
                                                    int32_t* __restrict__ dB, uint8_t* __restrict__ pB, long long sB,
                                                    int kblocks, int shift, uint32_t* __restrict__ flags,
                                                    ResidueGen<ND, E> gen) {
    constexpr int Q = 16 / E;  // waves per 1 KB block
    __shared__ uint32_t key[16];
    __shared__ int32_t delta[16];
    __shared__ __attribute__((aligned(16))) uint8_t image[16][64 * E];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int kb = wave / Q, q = wave % Q;
    if (t < 16) key[t] = 0;
    __syncthreads();
    const bool rows = (int)blockIdx.x < bandsA;  // a band of A
    const int br = rows ? (int)blockIdx.x : (int)blockIdx.x - bandsA;
    double x[E];
    if (rows) {
        load_piece<E, true>(A, M, K, lda, br, kb, q, lane, x);
#pragma unroll
        for (int e = 0; e < E; e++) {
            const uint32_t m = dpp_max<0x121>(dpp_max<0x122>(dpp_max<0x124>(dpp_max<0x128>(bf16_key<1>(x[e])))));
            if ((lane & 15) == 0) atomicMax(&key[q * E + e], m);
        }
    } else {
        load_piece<E, false>(B, K, N, ldb, br, kb, q, lane, x);
        uint32_t m = 0;
#pragma unroll
        for (int e = 0; e < E; e++) m = max(m, bf16_key<1>(x[e]));
        m = dpp_max<0x4E>(dpp_max<0xB1>(m));  // over the column's 4 lanes
        if ((lane & 3) == 0) atomicMax(&key[lane >> 2], m);
    }
    __syncthreads();
    if (t < 16) {
        uint32_t bad;
        const int i = br * 16 + t, d = key_delta(key[t], shift, bad);
        delta[t] = d;
        if (i < (rows ? M : N)) {
            (rows ? dA : dB)[i] = d;
            if (bad) atomicOr(&flags[rows ? 0 : 1], bad);
        }
    }
    __syncthreads();
    typename ResidueGen<ND, E>::State st[E];
    FarElements far;
    if (rows) {
#pragma unroll
        for (int e = 0; e < E; e++) {
            gen.load(st[e], x[e], delta[q * E + e], far);
            if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        gen.redo(st, far, [&](int e, double& v, int32_t& w) {
            v = piece_element<E, true>(A, M, K, lda, br, kb, q, e);
            w = delta[q * E + e];
        });
        emit_piece<ND, E, true>(gen, st, pA, sA, br, kblocks, kb, q, lane, image[wave]);
    } else {
        const int d = delta[lane >> 2];
#pragma unroll
        for (int e = 0; e < E; e++) {
            gen.load(st[e], x[e], d, far);
            if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        gen.redo(st, far, [&](int e, double& v, int32_t& w) {
            v = piece_element<E, false>(B, K, N, ldb, br, kb, q, e);
            w = d;
        });
        emit_piece<ND, E, false>(gen, st, pB, sB, br, kblocks, kb, q, lane, nullptr);
    }
}

template <int ND, int E>
int launch(oz_dev* dev, const oz2pass::PrepArgs& a, const SplitConsts& k) {
    const int kblocks = a.Kg / 64;
    const dim3 grid((unsigned)((a.Mt + a.Nt) / 16)), block((unsigned)(64 * kblocks * (16 / E)));
    hipLaunchKernelGGL((prep_kernel<ND, E>), grid, block, 0, dev->stream, a.A, a.M, a.K, a.lda, a.dA, a.pA, a.sA, a.Mt / 16,
                       a.B, a.N, a.ldb, a.dB, a.pB, a.sB, kblocks, a.shift, a.flags, ResidueGen<ND, E>{k});
    return oz::launch_check(dev, "prep_kernel");
}

}  // namespace

namespace oz2pass {

// K <= 256 with 4 elements per lane; up to 512 with 8 (nd = 3, whose registers leave room for two
// workgroups of 16 waves per CU), where the bands fill the chip. Separate launches -> this one, whole pass,
// us: 128^3 28.4 -> 20.4; 512 x 512 x 64 31 -> 24; 2048 x 2048 x 256 80 -> 75; 4096 x 4096 x 256 237 -> 226;
// 4096 x 4096 x 512 337 -> 305; 8192 x 8192 x 512 1195 -> 1126; 512^3 34.1 against 35.5; 8192 x 64 x 512
// 81.2 against 83.5. At K = 1024 16 elements per lane leave one workgroup per CU, nothing hides its loads,
// and 272 bands take two rounds: 79 against 102 (4096 x 256 x 1024).
bool prep_takes(int cus, const oz2_moduli_dev* mo, int M, int N, int Kg) {
    int evens = 0;
    for (int s = 0; s < mo->S; s++) evens += (int)mo->m[s] % 2 == 0;
    if (evens > 1) return false;
    return Kg <= 256 || (Kg <= 512 && mo->nd == 3 && M >= 256 && N >= 256 && ((long long)M + N) / 16 >= cus);
}

int launch_prep(oz_dev* dev, const PrepArgs& a, const oz2_moduli_dev* mo) {
    if (int st = check_moduli(dev, mo)) return st;
    int evens = 0;
    const SplitConsts k = split_consts(mo, &evens);
    if (a.Kg > 256) return launch<3, 8>(dev, a, k);
    return mo->nd == 3 ? launch<3, 4>(dev, a, k) : mo->nd == 4 ? launch<4, 4>(dev, a, k) : launch<5, 4>(dev, a, k);
}

}  // namespace oz2pass
