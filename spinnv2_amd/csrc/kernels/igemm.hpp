// What the implicit-GEMM conv kernels share: their arguments and the epilogue
// of a tile held as 32x32 MFMA accumulator blocks.
#pragma once

#include "common.hpp"

namespace spk::kern {

// gfx9 buffer resource word 3 (raw, untyped loads); loads whose offset is at
// or beyond num_records return 0.
constexpr int kBufferWord3 = 0x00020000;
// byte offset that is out of range for every B source (they are shorter:
// plan_igemm_f32, kMaxViewBytes), and still does not wrap when a valid offset is
// added to it
constexpr int kOobOffset = 0x7fff0000;

// Tiles of out-of-range entries that a k -> offset table (and a tap table) has
// past the last one: conv_split_f32 reads offsets three tiles ahead, the others
// two.
constexpr int kTilesPastK = 3;

struct IgemmArgs {
    const float *__restrict__ x;     // B-operand source: NCHW input, zero-padded when the conv pads
    const float *__restrict__ wp;    // [m_tiles][k_tiles] BM x BK tiles in MFMA fragment order
    const int *__restrict__ koff;    // [Kpad + kTilesPastK * BK] byte offset of k = (c, kh, kw) in x, kOobOffset past K
    const float *__restrict__ bias;  // [M] or null
    const float *__restrict__ res;   // like y, or null
    float *__restrict__ y;
    float *__restrict__ ws;          // split-K partials [splitk][M][ws_ld], column n at n - ws_n0
    int ws_n0, ws_ld;                // first column with partials, columns per partial row
    int dp_tiles, rem_split;         // hybrid: whole tiles first; rem_split slices per split tile
    int x_bytes;                     // extent of x for the bounds-checked loads
    int y_bytes;                     // extent of y (and of the residual)
    int ws_bytes;                    // extent of the split-K partials
    int Wp;                          // row pitch of x (padded width)
    int M, OW, OHW, Ntot;
    int sh, sw;
    int x_img_stride;                // elements between images in x
    int y_img_stride;                // elements between images in y and the residual
    int y_cstride;                   // elements between channels in y (OHW unless y is a view)
    int m_tiles, k_tiles, kt_per_split;
    int act;
    float alpha;
    // handoff: also store the output into the consuming conv's zero-padded
    // input (NCHW, Hp x Wp planes); y may then be null (no other reader)
    float *__restrict__ yp;
    int yp_bytes, yp_Wp, yp_pt, yp_pl, yp_plane;
    int yp_m0, yp_C;  // the handed-off channels: m0 .. m0 + C - 1 of y, the target's channels 0 .. C - 1
    // skinny kernel: k = tap * sk_C + c (a tap's channels consecutive);
    // channel c of a tap is c * sk_cstride elements past channel 0, tap
    // (kh, kw) = (tap / sk_KW, tap % sk_KW) kh * sk_tap_h + kw * sk_tap_w
    // elements past tap 0
    int sk_C, sk_cstride, sk_KW, sk_tap_h, sk_tap_w;
    // implicit padding (kModeChk): per-k tap table of koff's size ((kh*dh) <<
    // 16 | kw*dw, 0x7fff7fff past K), the unpadded input's extent and the padding
    const int *__restrict__ ktap;
    int chk_H, chk_W, chk_ph, chk_pw;
    int chk_KH, chk_KW, chk_dh, chk_dw;  // conv_split_f32: its ktap entry is bits kh and 16 + kw, all ones past K
    int th_steps;  // thin kernel: K / 4 MFMA steps (k' = tap * sk_C + c)
    // row-window kernel: the input window's geometry (GatherGeom's win_*)
    int win_KH, win_len, win_shift, win_owb, win_OH, win_dw;
};

// How the B operand is read (see conv_igemm_f32): taps of a padded input, four
// k at a time, or bounds-checked taps of the unpadded input.
constexpr int kModePlain = 0, kModeKvec = 1, kModeChk = 2;

// Four consecutive outputs from v[r], `left` of which are inside the tensor,
// at byte offset `off` (out of range past the last column): one 16-byte store
// when they are all in or all out (quads).
template <typename Block>
__device__ __forceinline__ void store_rows(const Block &v, int r, __amdgpu_buffer_rsrc_t rs, int off, int left,
                                           bool quads) {
    if (quads) {
        const uintx4 o = {__float_as_uint(v[r]), __float_as_uint(v[r + 1]), __float_as_uint(v[r + 2]),
                          __float_as_uint(v[r + 3])};
        __builtin_amdgcn_raw_buffer_store_b128(o, rs, left > 0 ? off : kPastTensor, 0, 0);
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[r + e]), rs, e < left ? off + 4 * e : kPastTensor, 0,
                                                  0);
    }
}

// Epilogue of one BM x BN tile held as TM x TN accumulator blocks of BS x BS
// outputs per wave (wave wm, wn of the tile): split-K partials, or alpha,
// bias, residual and activation in registers, then y and / or the handoff
// target.  A lane holds one column of a block (lane % BS) and, of a 32x32
// block, rows 8*(r/4) + 4*(lane/32) + (r%4) for r = 0..15, of a 16x16 block
// rows 4*(lane/16) + r for r = 0..3.
// ROWS: one pixel per image (a Gemm), so that a lane's groups of four rows are
// four consecutive outputs: 16-byte accesses where M is a multiple of 4, and
// split-K partials ordered [slice][n][m].  (Dword stores M * 4 bytes apart
// touched a line per lane.)
template <int BM, int BN, int BS, int TM, int TN, bool ROWS, typename Block>
__device__ __forceinline__ void igemm_epilogue(const IgemmArgs &a, const Block (&acc)[TM][TN], int mt, int nt, int wm,
                                               int wn, int lane, bool part, int slice) {
    constexpr int NR = BS * BS / 64;
    constexpr int JG = BS == 32 ? 1 : TN;  // blocks whose loads are in flight together: 16 values
    static_assert(BS == 32 || BS == 16, "MFMA shapes");
    const int row = lane & (BS - 1);
    const int rsub = 4 * (lane / BS);
    // Output offsets are 32-bit (tensors < 2 GiB); rows past M and columns
    // past N get an out-of-range offset, so the buffer stores drop them.
    int obase[TN];  // byte offset of (row 0, this lane's column) in y / res / ws
    int mrow[TM];   // first row of this lane in block i
#pragma unroll
    for (int i = 0; i < TM; i++) mrow[i] = mt * BM + (wm * TM + i) * BS + rsub;
    if (part) {
        // split-K partials: ws[slice][m][n - ws_n0], rows of ws_ld columns
        const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
            a.ws, static_cast<short>(0), a.ws_bytes, kBufferWord3);
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = nt * BN + (wn * TN + j) * BS + row;
            obase[j] = n >= a.Ntot ? kPastTensor
                       : ROWS      ? (slice * a.ws_ld + n - a.ws_n0) * a.M * 4
                                   : (slice * a.M * a.ws_ld + n - a.ws_n0) * 4;
        }
        if constexpr (ROWS) {
            const bool quads = (a.M & 3) == 0;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int q = 0; q < NR / 4; q++) {
                        const int m = mrow[i] + 8 * q;
                        store_rows(acc[i][j], 4 * q, wrs, obase[j] + m * 4, a.M - m, quads);
                    }
            return;
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const int m = mrow[i] + 8 * (r >> 2) + (r & 3);
                    const int off = m < a.M ? obase[j] + m * a.ws_ld * 4 : kPastTensor;
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][j][r]), wrs, off, 0, 0);
                }
        return;  // splitk_epilogue sums the partials
    }
    const int ohw4 = a.OHW * 4;        // the residual's channel stride (natural layout)
    const int ycs4 = a.y_cstride * 4;  // y's
    const int plane4 = a.yp_plane * 4;
    int pbase[TN];  // handoff target: this lane's pixel in the padded planes
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = nt * BN + (wn * TN + j) * BS + row;
        const int img = n / a.OHW;
        const int sp = n - img * a.OHW;
        const int oh = sp / a.OW;
        const int ow = sp - oh * a.OW;
        obase[j] = n < a.Ntot ? (img * a.y_img_stride + sp) * 4 : kPastTensor;
        pbase[j] = n < a.Ntot ? (img * a.yp_C * a.yp_plane + (oh + a.yp_pt) * a.yp_Wp + ow + a.yp_pl) * 4 : kPastTensor;
    }
    float *const any = a.y ? a.y : a.yp;
    const __amdgpu_buffer_rsrc_t yrs =
        __builtin_amdgcn_make_buffer_rsrc(any, static_cast<short>(0), a.y ? a.y_bytes : 0, kBufferWord3);
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
        a.yp ? a.yp : any, static_cast<short>(0), a.yp ? a.yp_bytes : 0, kBufferWord3);
    const __amdgpu_buffer_rsrc_t rrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.res ? a.res : any), static_cast<short>(0), a.res ? a.y_bytes : 0, kBufferWord3);
    const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.bias ? a.bias : any), static_cast<short>(0), a.bias ? a.M * 4 : 0, kBufferWord3);
    // JG blocks at a time: their bias and residual loads are all in flight
    // before the first use
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
        for (int j0 = 0; j0 < TN; j0 += JG) {
            Block v[JG];
#pragma unroll
            for (int j = 0; j < JG; j++) {
                v[j] = acc[i][j0 + j];
                if (a.alpha != 1.0f) v[j] *= a.alpha;
            }
            if (a.bias) {
                Block bv;
#pragma unroll
                for (int r = 0; r < NR; r++)
                    bv[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                          brs, (mrow[i] + 8 * (r >> 2) + (r & 3)) * 4, 0, 0));
#pragma unroll
                for (int j = 0; j < JG; j++) v[j] += bv;
            }
            if constexpr (ROWS) {
                const bool quads = (a.M & 3) == 0;
                if (a.res) {
#pragma unroll
                    for (int j = 0; j < JG; j++)
#pragma unroll
                        for (int r = 0; r < NR; r++) {
                            const int m = mrow[i] + 8 * (r >> 2) + (r & 3);
                            v[j][r] += __builtin_bit_cast(
                                float, __builtin_amdgcn_raw_buffer_load_b32(
                                           rrs, m < a.M ? obase[j0 + j] + m * 4 : kPastTensor, 0, 0));
                        }
                }
#pragma unroll
                for (int j = 0; j < JG; j++) {
#pragma unroll
                    for (int r = 0; r < NR; r++) v[j][r] = apply_act(v[j][r], a.act);
#pragma unroll
                    for (int q = 0; q < NR / 4; q++) {
                        const int m = mrow[i] + 8 * q;
                        store_rows(v[j], 4 * q, yrs, obase[j0 + j] + m * 4, a.M - m, quads);
                    }
                }
                continue;
            }
            if (a.res) {
                Block rv[JG];
#pragma unroll
                for (int j = 0; j < JG; j++)
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        const int m = mrow[i] + 8 * (r >> 2) + (r & 3);
                        rv[j][r] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(
                                       rrs, m < a.M ? obase[j0 + j] + m * ohw4 : kPastTensor, 0, 0));
                    }
#pragma unroll
                for (int j = 0; j < JG; j++) v[j] += rv[j];
            }
#pragma unroll
            for (int j = 0; j < JG; j++) {
                if (a.act == 1) {
#pragma unroll
                    for (int r = 0; r < NR; r++) v[j][r] = v[j][r] > 0.0f ? v[j][r] : 0.0f;
                } else if (a.act == 2) {
#pragma unroll
                    for (int r = 0; r < NR; r++) v[j][r] = apply_act(v[j][r], 2);
                }
            }
            if (a.yp) {
#pragma unroll
                for (int j = 0; j < JG; j++)
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        const unsigned mc = static_cast<unsigned>(mrow[i] + 8 * (r >> 2) + (r & 3) - a.yp_m0);
                        __builtin_amdgcn_raw_buffer_store_b32(
                            __float_as_uint(v[j][r]), prs,
                            mc < static_cast<unsigned>(a.yp_C) ? pbase[j0 + j] + static_cast<int>(mc) * plane4
                                                               : kPastTensor,
                            0, 0);
                    }
            }
            if (a.y) {
#pragma unroll
                for (int j = 0; j < JG; j++)
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        const int m = mrow[i] + 8 * (r >> 2) + (r & 3);
                        // __float_as_uint takes the element by value (a bit
                        // cast applied to a vector element reads element 0)
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[j][r]), yrs,
                                                              m < a.M ? obase[j0 + j] + m * ycs4 : kPastTensor, 0, 0);
                    }
            }
        }
    }
}

}  // namespace spk::kern
