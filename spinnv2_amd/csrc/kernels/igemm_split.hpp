// The implicit GEMM on bf16 parts (conv_split.hip): its kernel, instantiated
// there for the tiles listed here.
#pragma once

#include "igemm.hpp"

namespace spk::kern {

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int WPE, int MODE>
__global__ void __launch_bounds__(64 * WAVES_M * WAVES_N, WPE - (BM == 128 && MODE == kModeKvec)) conv_split_f32(IgemmArgs a);

// Packs weights w[M][K] (device) for BM x BK tiles into out, m_tiles * k_tiles *
// BM * BK * 6 bytes.
int pack_split(hipStream_t st, const float *w, int M, int K, int BM, int BK, int m_tiles, int k_tiles, void *out);

// T(BM, BN, BK, waves along M, along N, waves per SIMD the registers are
// held to, rate of the tile relative to the fp32 MFMA peak).  128 rows
// amortize the splitting of the activations best and are held to the 168
// registers that leave room for three waves, except a Gemm's, which need 172
// (ResNet stage-3 layers at batch 64: 3x3 101 us, 1x1 reduce 48 us, against 130
// and 61 us for 64 rows); 64 rows are for layers of at most 64 outputs and for
// few columns (56x56 3x3 at 64 channels: 100 us against 164), and run 4 to 10%
// faster held to 128 registers; 32 rows for the thinnest layers.
// Larger tiles lose what they save in loads and splits to fewer waves a CU:
// 256x64 with eight waves 106 us against 108 on the 3x3 layer but 72 against
// 62 on the 1x1 expand, 128x128 with 256 registers 218 and 92.
#define SPK_SPLIT_TILES(T) T(128, 64, 32, 4, 1, 3, 1.25) T(64, 64, 32, 2, 2, 4, 1.1) T(32, 128, 32, 1, 4, 1, 0.9)

#define SPK_SPLIT_EXTERN(BM, BN, BK, WM, WN, WPE, EFF)                                                \
    extern template __global__ void conv_split_f32<BM, BN, BK, WM, WN, WPE, kModePlain>(IgemmArgs);   \
    extern template __global__ void conv_split_f32<BM, BN, BK, WM, WN, WPE, kModeKvec>(IgemmArgs);    \
    extern template __global__ void conv_split_f32<BM, BN, BK, WM, WN, WPE, kModeChk>(IgemmArgs);
#ifndef SPK_SPLIT_DEFINE
SPK_SPLIT_TILES(SPK_SPLIT_EXTERN)
#endif

}  // namespace spk::kern
