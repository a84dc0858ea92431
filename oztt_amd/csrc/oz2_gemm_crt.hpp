// The fused products and reconstruction of Scheme II INT8 (oz2_gemm_crt.hip), as the whole pass calls it.
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
};

// Whether the kernel takes these moduli at this K, and the width and number of its limbs.
bool fused_limbs(const oz2_crt_dev* crt, int K, int* width, int* limbs);
int launch_fused(oz_dev* dev, const FusedArgs& f);

}  // namespace oz
