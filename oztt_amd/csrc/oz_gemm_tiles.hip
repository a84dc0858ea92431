// The rules that send a product launch to the smaller tiles of oz_gemm_tiles.hpp.
#include "oz_gemm_tiles.hpp"

#include "oz_gemm_launch.hpp"

namespace {

using namespace ozg;

template <int MODE, int TI, int TJ, int KW, int P>
int launch_ksplit(oz_dev* dev, const oz::ProductArgs& a) {
    const int tm = a.M / (16 * TI), tn = a.N / (16 * TJ);
    oz::launch_product(dev, gemm_i8_ksplit_kernel<MODE, TI, TJ, KW, P>, dim3((unsigned)(tm * tn * a.batch)), dim3(64 * KW),
                       a.A, a.Bt, a.C, a.K, a.ldc, a.sA, a.sB, a.sC, tm, tn, a.batch, a.dc);
    return oz::launch_check(dev, "gemm_i8_ksplit_kernel");
}

template <int MODE, int TI, int TJ, int WM, int WN, int NSTG>
int launch_tile(oz_dev* dev, const oz::ProductArgs& a) {
    const int tm = a.M / (16 * TI * WM), tn = a.N / (16 * TJ * WN);
    oz::launch_product(dev, gemm_i8_tile_kernel<MODE, TI, TJ, WM, WN, NSTG>, dim3((unsigned)(tm * tn * a.batch)),
                       dim3(64 * WM * WN), a.A, a.Bt, a.C, a.K, a.ldc, a.sA, a.sB, a.sC, tm, tn, a.batch, a.dc);
    return oz::launch_check(dev, "gemm_i8_tile_kernel");
}

template <int P>
int launch_diagonals(oz_dev* dev, const oz::ProductArgs& a) {
    const int tm = a.M / 64, tn = a.N / 64;
    const dim3 grid((unsigned)(tm * tn)), block(256);
    int32_t* C = static_cast<int32_t*>(a.C);
    if ((a.K / BK) % 2 == 0)
        oz::launch_product(dev, gemm_i8_diagonals_kernel<P, true>, grid, block, a.A, a.Bt, C, a.K, a.ldc, a.sA, a.sB, a.sC, tm, tn);
    else
        oz::launch_product(dev, gemm_i8_diagonals_kernel<P, false>, grid, block, a.A, a.Bt, C, a.K, a.ldc, a.sA, a.sB, a.sC, tm, tn);
    return oz::launch_check(dev, "gemm_i8_diagonals_kernel");
}

}  // namespace

namespace oz {

// The measured times (us, 16 moduli, one launch after another) behind the lines, 256 x 256 tiles first:
//   64 x 64 tiles in all    K <= 512             longer K
//   256 (256 x 256)         12.5 -> 4.3 (K 512)  40.1 -> 9.3 (4096), 255.6 -> 50.6 (32768)
//   512 (512 x 256)         12.7 -> 5.3          40.5 -> 16.1, 289 -> 133
//   1024 (512 x 512)        12.9 -> 6.9          41.7 -> 23.5, 289 -> 191
//   2304 (768 x 768)        13.6 -> 12.0         27.7 -> 26.1 (2048); 83.9 against 83.3 (8192)
//   3072 (1024 x 768)       13.9 -> 12.6         19.0 -> 17.5 (1024); with the planes not yet in a cache, as in
//                                                a pass, 25.8 against 28.2 (1536)
//   4096 (1024 x 1024, one  12.1 -> 11.9 (192);  20.0 against 20.8 (1024)
//     256 x 256 tile per CU)  14.6 either way
//   6144 (1536 x 1024)      29.0 -> 21.1         63.8 -> 49.4 (2048), 109 -> 89.4, 233 -> 194 (8192)
//   16384 (2048 x 2048)     56.7 -> 51.0         76.7 -> 74.5 (1024); 231 against 262 (4096)
//   36864 (3072 x 3072)     129 -> 112           188 -> 183 (1024)
// and with other numbers of moduli, where 256 x 256 tiles fill more than three quarters of their rounds and K is long:
//   6400 (1280^2, 16)       78 against 85 (3072), 185 against 211 (8192)
//   6272 (1792^2, 8)        97 against 108 (4096), 178 against 202 (8192)
DigitTile digit_tile(int cus, int M, int N, int K, int S) {
    const long long t64 = (long long)(M / 64) * (N / 64) * S, t256 = t64 / 16;
    if (cus <= 0 || t256 > (1 << 28)) return DigitTile::Tile256;
    if (t64 <= 2ll * cus) return K <= 512 ? DigitTile::Tile64 : t64 <= cus ? DigitTile::Split8 : DigitTile::Split4;
    if (t64 <= 12ll * cus)
        return t64 <= 6ll * cus || K <= (t64 <= 9ll * cus ? 2048 : 1024) ? DigitTile::Tile128 : DigitTile::Tile256;
    const long long rounds = (t256 + cus - 1) / cus;  // of the 256 x 256 tiles over the CUs
    if (rounds == 1) return K < 512 ? DigitTile::Tile256x128 : DigitTile::Tile256;
    return K <= 1024 || 4 * t256 <= 3 * rounds * cus ? DigitTile::Tile256x128 : DigitTile::Tile256;
}

int launch_digit_tile(oz_dev* dev, DigitTile tile, const ProductArgs& a) {
    switch (tile) {
    case DigitTile::Tile64: return launch_tile<DIGITS, 2, 2, 2, 2, 4>(dev, a);
    case DigitTile::Split8: return launch_ksplit<DIGITS, 4, 4, 8, 2>(dev, a);
    case DigitTile::Split4: return launch_ksplit<DIGITS, 4, 4, 4, 3>(dev, a);
    case DigitTile::Tile128: return launch_tile<DIGITS, 4, 4, 2, 2, 3>(dev, a);
    default: return launch_tile<DIGITS, 4, 4, 4, 2, 3>(dev, a);
    }
}

// Times (us, 8 slices), 256 x 256 tiles first, by the 64 x 64 tiles of one diagonal:
//   16 (256 x 256)     40.8 -> 6.1 (K 512), 140.8 -> 16.7 (2048), 537 -> 62 (8192): 32 x 32, K split
//   64 (512 x 512)     12.3 -> 5.2 (64), 42 -> 12.4 (512), 143 -> 29.8, 541 -> 106 (all diagonals: 163)
//   256 (1024 x 1024)  22.8 -> 13.2 (192), 45.7 -> 25 (512), 156 -> 61 (2048), 566 -> 238 (8192)
//   512 (2048 x 1024)  59.8 -> 40.5 (512), 102 -> 69 (1024), 193 -> 125 (2048), 678 -> 494 (8192)
//   1024 (2048 x 2048) 54.1 -> 43.5 (192), 77.7 -> 74.9 (512); 139 against 141 (1024)
//   4096 (4096 x 4096) 204.6 -> 167.6 (192); 347 against 370 (512); 1742 against 1776 (4096)
// With p slices the 256 x 256 tiles take n p (p + 1) / 2 steps of K (n tiles per diagonal) on `cus` CUs and at least
// the p of the longest diagonal: `fill` of that is work. 128 x 128 tiles (times second) cost more per step and less
// per tile, so they lose where the large ones fill their time or are long:
//   fill .55-.6   1280^2, 11 slices: 21.1 against 27.5 (128), 811 against 863 (8192), 206 in place of 215 (2048)
//   fill .65-.7   1280^2, 13 slices: 26.0 against 31.1 (128), 510 against 603 (4096), 1008 against 1311 (8192)
//   fill .63-.95  1536^2, 8: 24.3 against 29.5 (192); 2048 x 1536, 7: 28.8 against 33.1 (256); 2304^2, 5: 38.9 against
//                 41.6 (384); but 2048^2, 6: 33.7 against 32.5 (192)
//   fill .72-1.0  2048 x 1024, 13: 81 against 89 (512), 1057 against 1494 (8192); 256 x 8192, 13: 1248 against 1783
//   long tiles    3584^2 x 384: 339 against 375 (12 slices), 545 against 627 (16); 180 either way with 8
DiagTile diag_tile(int cus, int M, int N, int K, int p) {
    const long long t64 = (long long)(M / 64) * (N / 64), t256 = t64 / 16;
    const bool all = p >= 5 && p <= 9;  // the slices for which the all-diagonals kernel is built
    if (cus <= 0 || t64 * p > (1 << 28)) return DiagTile::Tile256;
    if (16 * t64 <= cus) return DiagTile::Split32;
    if (2 * t64 < cus) return K <= 128 ? DiagTile::Tile64 : DiagTile::Split64;
    const int nk = K / BK;
    const double fill = 0.5 * (double)t256 * (p + 1) / cus;
    if (t64 <= 2ll * cus) {
        if (all && K >= (t64 <= cus ? 512 : 2048)) return DiagTile::All;
        const bool two = t64 == 2ll * cus;  // (2048 x 1024 x 128: 128 x 128 tiles up to 13% faster, 12 slices)
        const double least = nk < 2 || (two && nk < 3) ? 2.0 : nk < 5 ? (two ? 0.62 : 0.54) : nk < 8 ? (two ? 0.62 : 0.72) :
                             nk < 32 ? 0.72 : nk < 64 ? 0.65 : 0.57;
        return fill >= least && fill <= (nk < 8 ? 1.0 : 1.1) ? DiagTile::Tile256 : DiagTile::Tile128;
    }
    if (K > 384) return DiagTile::Tile256;
    // up to one and a half rounds of large tiles, which the shorter diagonals fill
    if (fill >= 0.62 && fill <= (p == 3 ? 1.2 : 1.0) && t256 * p > cus && p > 2 && (nk >= 3 || (nk == 2 && p >= 8)))
        return DiagTile::Tile256;
    return nk * (p + 1) > (t64 > 7ll * cus ? 60 : 96) ? DiagTile::Tile256 : DiagTile::Tile128;
}

int launch_diag_tile(oz_dev* dev, DiagTile tile, const ProductArgs& a) {
    switch (tile) {
    case DiagTile::Split32: return launch_ksplit<DIAG, 2, 2, 4, 3>(dev, a);
    case DiagTile::Split64: return launch_ksplit<DIAG, 4, 4, 8, 2>(dev, a);
    case DiagTile::Tile64: return launch_tile<DIAG, 2, 2, 2, 2, 4>(dev, a);
    case DiagTile::All:
        switch (a.batch) {
        case 5: return launch_diagonals<5>(dev, a);
        case 6: return launch_diagonals<6>(dev, a);
        case 7: return launch_diagonals<7>(dev, a);
        case 8: return launch_diagonals<8>(dev, a);
        case 9: return launch_diagonals<9>(dev, a);
        }
        [[fallthrough]];
    default: return launch_tile<DIAG, 4, 4, 2, 2, 3>(dev, a);
    }
}

}  // namespace oz
