// The whole Scheme II INT8 device pass of oz2_pass.hip, shared by its entry points: the layout of
// its intermediates in a workspace, the checks of its arguments, and the pass itself.
#pragma once
#include "oz_internal.hpp"

namespace oz2pass {

// Byte offsets, inside the workspace, of the exponent deltas of A's rows and B's columns, the S
// residue planes of A (Mg x Kg) and of B^T (Ng x Kg) and the S digit planes (Mg x Ng); every region
// starts on a 256-byte boundary. Mg, Ng: M, N rounded up to 256; Kg: K rounded up to 64.
struct PassLayout {
    int Mg, Ng, Kg;
    size_t dA, dB, planesA, planesB, digits, total;
};

// The workspace of a pass of M x N x K with S moduli; false for shapes outside the kernels' index range.
bool pass_layout(int M, int N, int K, int S, PassLayout* L);

// The descriptors must describe one plan: the same moduli (INT8: 2..255) in both, the shift of the
// width b with nd digits, and int32 products that stay exact over K (|C_s| <= Kg 127^2 < 2^31).
// Returns a message or nullptr.
const char* check_plan(const oz2_moduli_dev* mo, const oz2_crt_dev* crt, int Kg);

// Pointers, extents and leading dimensions; returns a message or nullptr.
const char* check_args(const double* A, int lda, const double* B, int ldb, const double* C, int ldc, int M, int N,
                       int K, const uint32_t* flags);

// The pass on a workspace of L.total bytes at `work` (checked arguments), ordered on dev's stream.
int run_pass(oz_dev* dev, const double* A, int lda, const double* B, int ldb, double* C, int ldc, int M, int N, int K,
             const oz2_moduli_dev* mo, const oz2_crt_dev* crt, uint32_t* flags, uint8_t* work, const PassLayout& L);

// Deltas and residue planes of both operands in one launch (oz2_prep.hip): A's rows up to Mt and B's
// columns up to Nt (multiples of 16, zeros past M and N), K padded to Kg; plane strides sA, sB in bytes;
// flags are ORed into. prep_takes: the rule (short K, a pairwise coprime set).
struct PrepArgs {
    const double* A;
    int M, K, lda, Mt;
    int32_t* dA;
    uint8_t* pA;
    long long sA;
    const double* B;
    int N, ldb, Nt;
    int32_t* dB;
    uint8_t* pB;
    long long sB;
    int Kg, shift;
    uint32_t* flags;
};
bool prep_takes(int cus, const oz2_moduli_dev* mo, int M, int N, int Kg);
int launch_prep(oz_dev* dev, const PrepArgs& a, const oz2_moduli_dev* mo);

// A matrix on at most 64 columns (oz2_skinny.hip): the digits of A's products with B's residue planes (64 rows
// of Kg each, OZ_BLOCK tiles) without A's planes. Part p of K (of `parts`, the rule's answer, 0 for a pass it
// does not take) writes its digits to columns 64 p .. of D's rows; the parts' digits add up. Rows up to a
// multiple of 64 are written.
// The constants of modulus m1 in that kernel (oz2_skinny.hip, SkinnyConsts).
struct NarrowModulus {
    uint32_t w[2], magic;
    int init, mneg;
};
NarrowModulus narrow_modulus(int m1);
int skinny_parts(int cus, const oz2_moduli_dev* mo, int M, int N, int K);
int launch_skinny(oz_dev* dev, const double* A, int M, int K, int lda, const int32_t* dA, const int8_t* pB, int Kg,
                  uint8_t* D, int ldd, long long sD, int parts, const oz2_moduli_dev* mo, const oz2_crt_dev* crt);

// The way of a pass: the parts of K without A's planes (0: with planes), else normalization and residues in one
// launch or two, products and reconstruction in one kernel or two.
struct Route {
    int parts;
    bool prep, fused;
};
Route route_of(int cus, const oz2_moduli_dev* mo, const oz2_crt_dev* crt, int M, int N, int K);

}  // namespace oz2pass
