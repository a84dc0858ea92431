// Which tiles a launch of INT8 products runs in: the 256 x 256 kernel of oz_gemm.hip or one of the smaller
// tiles of oz_gemm_tiles.hip, by a rule on the sizes.
#pragma once
#include "oz2_modular.hpp"
#include "oz_internal.hpp"

namespace oz {

// A launch of INT8 products as the kernels take it (oz_gemm_i8): M and N multiples of 256, K of 64.
struct ProductArgs {
    const int8_t* A;
    const int8_t* Bt;
    void* C;
    int M, N, K, batch, ldc;
    long long sA, sB, sC;
    oz2::DigitConsts dc;
};

// The order of the 256 x 256 tiles of products of equal length (oz_gemm.hip).
bool tile_ranges(int cus, int M, int N, int K, int batch);

enum class DigitTile { Tile256, Tile256x128, Tile128, Tile64, Split4, Split8 };
DigitTile digit_tile(int cus, int M, int N, int K, int S);
int launch_digit_tile(oz_dev* dev, DigitTile tile, const ProductArgs& a);  // not Tile256

enum class DiagTile { Tile256, All, Tile128, Tile64, Split64, Split32 };
DiagTile diag_tile(int cus, int M, int N, int K, int p);
int launch_diag_tile(oz_dev* dev, DiagTile tile, const ProductArgs& a);  // not Tile256

}  // namespace oz
