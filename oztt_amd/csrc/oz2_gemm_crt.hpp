// The last steps of Scheme II INT8 as the whole pass calls them: products and reconstruction in one kernel
// (oz2_gemm_crt.hip), or the reconstruction from digits (oz2_crt.hip).
#pragma once
#include "oz_internal.hpp"

namespace oz {

// The S residue planes of A (plane stride sA) and of B^T (sB) in OZ_BLOCK tiles, K a multiple of 64, rows
// padded with zeros to multiples of 64; C (M x N, ldo) as oz2_crt_digits_f64 gives it.
struct FusedArgs {
    const int8_t* A;
    const int8_t* Bt;
    int M, N, K;
    long long sA, sB;
    const oz2_crt_dev* crt;
    const int32_t* dA;
    const int32_t* dB;
    double* out;
    int ldo;
    uint32_t* fsrc;  // range flags moved to fdst and zeroed (two words)
    uint32_t* fdst;
};

// Whether the kernel takes these moduli at this K, and the width and number of its limbs.
bool fused_limbs(const oz2_crt_dev* crt, int K, int* width, int* limbs);
int launch_fused(oz_dev* dev, const FusedArgs& f);

// oz2_crt_digits_f64, which also moves the range flags of a whole pass from fsrc to fdst (two device words
// each) and zeroes fsrc for the next pass, so that no launch has to clear them. two (at most 16 moduli and
// 64 columns): the digits are the sums of two, 64 columns apart.
int crt_digits_moving_flags(oz_dev* dev, const uint8_t* D, int M, int N, int ldd, long long strideD,
                            const oz2_crt_dev* crt, const int32_t* dA, const int32_t* dB, double* out, int ldo,
                            uint32_t* fsrc, uint32_t* fdst, bool two = false);

}  // namespace oz
