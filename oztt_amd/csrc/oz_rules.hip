// The rules of the dispatch and constants that they go with, for tests to ask (no GPU needed).
#include "oz2_gemm_crt.hpp"
#include "oz2_pass.hpp"

extern "C" int oz_rule_fused_limbs(const oz2_crt_dev* crt, int K, int* width, int* limbs) {
    return oz::fused_limbs(crt, K, width, limbs);
}

extern "C" void oz_rule_narrow_modulus(int m, oz2pass::NarrowModulus* out) { *out = oz2pass::narrow_modulus(m); }
