// The rules of the dispatch and constants that they go with, for tests to ask (no GPU needed).
#include "oz2_gemm_crt.hpp"
#include "oz_gemm_launch.hpp"
#include "oz2_pass.hpp"

extern "C" int oz_rule_fused_limbs(const oz2_crt_dev* crt, int K, int* width, int* limbs) {
    return oz::fused_limbs(crt, K, width, limbs);
}

extern "C" void oz_rule_narrow_modulus(int m, oz2pass::NarrowModulus* out) { *out = oz2pass::narrow_modulus(m); }

extern "C" int oz_rule_digit_tile(int cus, int M, int N, int K, int S) { return (int)oz::digit_tile(cus, M, N, K, S); }
extern "C" int oz_rule_diag_tile(int cus, int M, int N, int K, int p) { return (int)oz::diag_tile(cus, M, N, K, p); }
extern "C" int oz_rule_tile_ranges(int cus, int M, int N, int K, int batch) { return oz::tile_ranges(cus, M, N, K, batch); }
extern "C" int oz_rule_strip_chunks(int cus, int M, int N, int K) {
    int rows;
    return oz::strip_chunks(cus, M, N, K, &rows);
}
// 4 parts + 2 fused + prep
extern "C" int oz_rule_pass(int cus, const oz2_moduli_dev* mo, const oz2_crt_dev* crt, int M, int N, int K) {
    const oz2pass::Route r = oz2pass::route_of(cus, mo, crt, M, N, K);
    return 4 * r.parts + 2 * r.fused + r.prep;
}
