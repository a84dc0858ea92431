// The rules of the dispatch by themselves, for tests to ask which way a call goes (no GPU needed).
#include "oz2_gemm_crt.hpp"

extern "C" int oz_rule_fused_limbs(const oz2_crt_dev* crt, int K, int* width, int* limbs) {
    return oz::fused_limbs(crt, K, width, limbs);
}
