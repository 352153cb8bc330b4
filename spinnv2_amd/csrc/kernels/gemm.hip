// Gemm and MatMul.
//
// Gemm (reference runtime/kernels/reference/mm/gemm.c:3-33):
//   Y[r][n] = alpha * sum_k A'[r][k] * B'[k][n] + C[n]
// where A' / B' are A / B transposed when trans_a / trans_b are set, and beta
// is not applied (the x86 reference ignores it too).  On the device this is
// the fp32 MFMA implicit GEMM of a 1x1 convolution over an [rows, K, 1, 1]
// input: the GEMM's M is the output feature dimension, its N the rows.  B is
// constant weight data, transposed into [n][k] panels at prepare time;
// trans_a only changes the k-offset table and the per-row stride.
//
// MatMul (reference mm/matmul.c:3-49): batched, numpy-broadcast leading
// dimensions; one thread per output element, k inner, lanes along n.
#include <cstdlib>
#include <cstring>
#include <vector>

#include "conv.hpp"
#include "kernels.hpp"
#include "parts.hpp"

namespace spk::kern {

int plan_igemm_gemm(hipStream_t st, const ConvGeom &g, const float *w_host, int k_stride, ConvPlan *plan);
int run_igemm_f32(Spkv2Context *ctx, const ConvPlan *p, const float *x, const float *bias, const float *res, float *y,
                  float alpha);
std::string igemm_name(const ConvPlan *p);

namespace {

struct GemmPlan {
    ConvPlan conv;
    int rows, K, Nout;
    int trans_a;
    float alpha;
    int x_stride;
    // at most four rows of A (a classifier at batch 1-4), A not transposed,
    // K a multiple of 4: the matrix-vector kernel over these weights, W[n][k]
    // row-major (device); null otherwise
    float *wrow;
};

void gemm_plan_free(void *p) {
    GemmPlan *g = static_cast<GemmPlan *>(p);
    if (!g) return;
    if (g->conv.wpack) (void)hipFree(g->conv.wpack);
    if (g->conv.ktab) (void)hipFree(g->conv.ktab);
    if (g->wrow) (void)hipFree(g->wrow);
    delete g;
}

// Matrix-vector form of a Gemm with R <= 4 rows of A: y[r][n] = alpha *
// sum_k A[r][k] W[n][k] + c[n].  One wave per output n reads row n of W in
// 16-byte pieces (lane l takes k = 4 (l + 64 j) .. + 3, j = 0, 1, ...), all
// of a lane's pieces in flight together with the matching pieces of the R
// rows of A; each lane sums its products in k order, then the 64 lane sums
// are added in a fixed butterfly.  Bound by the HBM reads of W (4 K bytes per
// output), where the 16 x 16 MFMA tiles leave most CUs idle and each tile's
// k chain serial.
template <int R>
__global__ void __launch_bounds__(256) gemv_f32(const float *__restrict__ W, const float *__restrict__ A,
                                                const float *__restrict__ c, float *__restrict__ Y, int K, int Nout,
                                                float alpha) {
    const int lane = threadIdx.x & 63;
    const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (n >= Nout) return;  // the whole wave (n is per wave)
    const floatx4 *w4 = reinterpret_cast<const floatx4 *>(W + static_cast<size_t>(n) * K);
    const floatx4 *a4 = reinterpret_cast<const floatx4 *>(A);
    const int K4 = K / 4;
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
    constexpr int U = 8;  // pieces per lane in flight
    for (int j0 = lane; j0 < K4; j0 += 64 * U) {
        floatx4 wv[U], av[U][R];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = j0 + 64 * u;
            const bool ok = j < K4;
            wv[u] = ok ? w4[j] : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < R; r++) av[u][r] = ok ? a4[r * K4 + j] : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[r] = fmaf(wv[u][e], av[u][r][e], acc[r]);
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) acc[r] += __shfl_xor(acc[r], off, 64);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < R; r++) Y[static_cast<size_t>(r) * Nout + n] = alpha * acc[r] + (c ? c[n] : 0.0f);
    }
}

// Batched MatMul y[b] = A[a(b)] x B[b(b)] (reference kernels/reference/mm/
// matmul.c:3-49: numpy broadcasting of the leading dims, K from A's last
// dim, no transposes).  One workgroup computes a 64x64 tile of one batch:
// 4 waves in a 2x2 grid, each a 32x32 block on v_mfma_f32_32x32x2f32.  k
// tiles of 16 are staged through LDS k-contiguous for both operands (B is
// transposed on the way in), double-buffered with the next tile's global
// loads in flight during the MFMAs.
struct MatmulArgs {
    const float *__restrict__ a;
    const float *__restrict__ b;
    float *__restrict__ y;
    int M, N, K;
    int yrank, arank, brank;
    int yshape[8], ashape[8], bshape[8];
};

constexpr int kMmTile = 64, kMmBK = 16, kMmLd = kMmBK + 1;

// Matrix indices into a and b of batch z of y (numpy broadcasting: a
// leading dim of 1 repeats).
__device__ __forceinline__ void matmul_batch(const MatmulArgs &p, int z, size_t *ab, size_t *bb) {
    int coords[8] = {0};
    int t = z;
    for (int d = p.yrank - 3; d >= 0; d--) {
        coords[d] = t % p.yshape[d];
        t /= p.yshape[d];
    }
    *ab = 0;
    *bb = 0;
    for (int d = 0; d + 2 < p.arank; d++) {
        const int yd = p.yrank - p.arank + d;
        *ab = *ab * p.ashape[d] + (p.ashape[d] == 1 || yd < 0 ? 0 : coords[yd]);
    }
    for (int d = 0; d + 2 < p.brank; d++) {
        const int yd = p.yrank - p.brank + d;
        *bb = *bb * p.bshape[d] + (p.bshape[d] == 1 || yd < 0 ? 0 : coords[yd]);
    }
}

__global__ void __launch_bounds__(256) matmul_mfma(MatmulArgs p) {
    __shared__ float As[2][kMmTile * kMmLd];
    __shared__ float Bs[2][kMmTile * kMmLd];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * kMmTile, n0 = blockIdx.x * kMmTile;
    size_t ab = 0, bb = 0;
    matmul_batch(p, blockIdx.z, &ab, &bb);
    const size_t M = p.M, N = p.N, K = p.K;
    const float *A = p.a + ab * M * K;
    const float *B = p.b + bb * K * N;
    float *Y = p.y + static_cast<size_t>(blockIdx.z) * M * N;

    const int ar = tid >> 2, ak = (tid & 3) * 4;   // A tile: row, 4 k's
    const int bk = tid >> 4, bn = (tid & 15) * 4;  // B tile: k, 4 columns
    float ra[4], rb[4];
    auto load = [&](int k0) {
        const int gm = m0 + ar;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int gk = k0 + ak + i;
            ra[i] = gm < p.M && gk < p.K ? A[static_cast<size_t>(gm) * K + gk] : 0.0f;
        }
        const int gk = k0 + bk;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int gn = n0 + bn + i;
            rb[i] = gk < p.K && gn < p.N ? B[static_cast<size_t>(gk) * N + gn] : 0.0f;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            As[buf][ar * kMmLd + ak + i] = ra[i];
            Bs[buf][(bn + i) * kMmLd + bk] = rb[i];
        }
    };

    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    const int ktiles = (p.K + kMmBK - 1) / kMmBK;
    const int row = lane & 31, kh = lane >> 5;
    load(0);
    store(0);
    __syncthreads();
    for (int kt = 0; kt < ktiles; kt++) {
        const int buf = kt & 1;
        if (kt + 1 < ktiles) load((kt + 1) * kMmBK);
#pragma unroll
        for (int s = 0; s < kMmBK / 2; s++) {
            // lanes 0-31 supply k = 2s, lanes 32-63 k = 2s+1, for A and B alike
            const float av = As[buf][(wm * 32 + row) * kMmLd + 2 * s + kh];
            const float bv = Bs[buf][(wn * 32 + row) * kMmLd + 2 * s + kh];
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc, 0, 0, 0);
        }
        if (kt + 1 < ktiles) store(buf ^ 1);  // that buffer was last read before the previous barrier
        __syncthreads();
    }
    // accumulator layout: column lane & 31, rows 8*(r/4) + 4*(lane/32) + r%4
    const int col = n0 + wn * 32 + row;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int m = m0 + wm * 32 + 8 * (r >> 2) + 4 * kh + (r & 3);
        if (m < p.M && col < p.N) Y[static_cast<size_t>(m) * N + col] = acc[r];
    }
}

// Batched MatMul on bf16 parts (parts.hpp, conv_split.hip): one BM x 64 tile
// per workgroup, BK k at a time, both operands split on their way into LDS
// (pieces of 8 k of one row or column), two tiles of loads in flight.
//   BM = 32, BK = 64: waves 0 and 1 sum the two column halves over the first
//   32 k of every tile, waves 2 and 3 over the others, and the two halves are
//   added through LDS at the end.  For long k on few tiles (attention at small
//   batches), a chain of K / 64 steps bound by their latency.
//   BM = 64, BK = 32: four waves side by side, for the others.
// TA / TB: the operand is stored transposed (A [K][M], B [N][K]), so that a
// Transpose in front of it need not run.  Sixteen attention products at 20x20:
// [400 x 32] x [32 x 400] 8.9 us behind its Transpose's 3 before, 8.9 alone
// now, [64 x 400] x [400 x 400] 19 us behind a Transpose's 8.2, now 8.7; one
// 2048^3 product 364 us on the fp32 tiles, now 143.
constexpr int kPtN = 64, kPtPad = 2;

// One operand's BK-k tile of R rows (columns of B) in registers: R * BK / 256
// elements a thread, all loads in flight.  KCONT: k is contiguous, `ld` apart
// by row (QUADS: K is a multiple of 4, so that a lane's four k are all in or all
// out); otherwise rows are contiguous, `ld` apart by k.
template <int R, int BK, bool KCONT, bool QUADS>
struct PartTile {
    static constexpr int N = R * BK / 256;
    static constexpr int LPR = BK / 4;       // KCONT: lanes a row
    static constexpr int RPP = 256 / LPR;    // KCONT: rows a pass
    static_assert(R % RPP == 0 || !KCONT, "whole passes");
    static_assert(N % 8 == 0, "whole pieces");
    float v[N];

    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int ld, int r0, int rows, int k0, int K, int tid) {
        constexpr int kOob = 0x7fff0000;
        if constexpr (KCONT) {
            const int k = k0 + tid % LPR * 4;
#pragma unroll
            for (int p = 0; p < R / RPP; p++) {
                const int r = r0 + tid / LPR + RPP * p;
                const int off = r < rows ? (r * ld + k) * 4 : kOob;
                if constexpr (QUADS) {
                    const floatx4 q = __builtin_bit_cast(
                        floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, k < K ? off : kOob, 0, 0));
#pragma unroll
                    for (int e = 0; e < 4; e++) v[4 * p + e] = q[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        v[4 * p + e] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(rs, k + e < K ? off + 4 * e : kOob, 0, 0));
                }
            }
        } else {
            const int r = r0 + tid % R, g = tid / R * N;
#pragma unroll
            for (int j = 0; j < N; j++) {
                const int k = k0 + g + j;
                v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                     rs, r < rows && k < K ? (k * ld + r) * 4 : kOob, 0, 0));
            }
        }
    }
    // pieces [part][k group][row]
    __device__ __forceinline__ void store(uintx4 (*lds)[BK / 8][R + kPtPad], int tid) const {
        if constexpr (KCONT) {
            const int g = tid % LPR >> 1, half = tid & 1;
#pragma unroll
            for (int p = 0; p < R / RPP; p++) {
                unsigned h[2], m[2], l[2];
                split_pair(v[4 * p], v[4 * p + 1], h[0], m[0], l[0]);
                split_pair(v[4 * p + 2], v[4 * p + 3], h[1], m[1], l[1]);
                const int r = tid / LPR + RPP * p;
                reinterpret_cast<uintx2 *>(&lds[0][g][r])[half] = uintx2{h[0], h[1]};
                reinterpret_cast<uintx2 *>(&lds[1][g][r])[half] = uintx2{m[0], m[1]};
                reinterpret_cast<uintx2 *>(&lds[2][g][r])[half] = uintx2{l[0], l[1]};
            }
        } else {
#pragma unroll
            for (int g8 = 0; g8 < N / 8; g8++) {
                uintx4 h, m, l;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    unsigned hv, mv, lv;
                    split_pair(v[8 * g8 + 2 * e], v[8 * g8 + 2 * e + 1], hv, mv, lv);
                    h[e] = hv;
                    m[e] = mv;
                    l[e] = lv;
                }
                const int g = tid / R * (N / 8) + g8, r = tid % R;
                lds[0][g][r] = h;
                lds[1][g][r] = m;
                lds[2][g][r] = l;
            }
        }
    }
};

template <int BM, bool TA, bool TB, bool QUADS>
__global__ void __launch_bounds__(256) matmul_parts(MatmulArgs p) {
    constexpr int BK = BM == 32 ? 64 : 32;
    __shared__ __attribute__((aligned(16))) uintx4 As[2][3][BK / 8][BM + kPtPad];
    __shared__ __attribute__((aligned(16))) uintx4 Bs[2][3][BK / 8][kPtN + kPtPad];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 31, half = lane >> 5;
    const int wn = wave & 1;
    const int wk = BM == 32 ? wave >> 1 : 0, wm = BM == 32 ? 0 : wave >> 1;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * kPtN;
    size_t ab = 0, bb = 0;
    matmul_batch(p, blockIdx.z, &ab, &bb);
    const float *A = p.a + ab * p.M * p.K;
    const float *B = p.b + bb * p.K * p.N;
    float *Y = p.y + static_cast<size_t>(blockIdx.z) * p.M * p.N;
    const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A), static_cast<short>(0),
                                                                         p.M * p.K * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), static_cast<short>(0),
                                                                         p.K * p.N * 4, 0x00020000);
    PartTile<BM, BK, !TA, QUADS> a0, a1;
    PartTile<kPtN, BK, TB, QUADS> b0, b1;
    const int lda = TA ? p.M : p.K, ldb = TB ? p.K : p.N;
    const int tiles = (p.K + BK - 1) / BK;

    floatx16 acc, sml;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = sml[r] = 0.0f;
    // tiles past the last load zeros without a memory access
    auto load = [&](int t, PartTile<BM, BK, !TA, QUADS> &at, PartTile<kPtN, BK, TB, QUADS> &bt) __attribute__((always_inline)) {
        at.load(ars, lda, m0, p.M, t * BK, p.K, tid);
        bt.load(brs, ldb, n0, p.N, t * BK, p.K, tid);
    };
    auto step = [&](int t, int buf, const PartTile<BM, BK, !TA, QUADS> &an, const PartTile<kPtN, BK, TB, QUADS> &bn,
                    PartTile<BM, BK, !TA, QUADS> &af, PartTile<kPtN, BK, TB, QUADS> &bf) __attribute__((always_inline)) {
        load(t + 2, af, bf);
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int g = 4 * wk + 2 * q + half;
            bf16x8 a[3], b[3];
#pragma unroll
            for (int s = 0; s < 3; s++) {
                a[s] = __builtin_bit_cast(bf16x8, As[buf][s][g][wm * 32 + row]);
                b[s] = __builtin_bit_cast(bf16x8, Bs[buf][s][g][wn * 32 + row]);
            }
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
            sml = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], sml, 0, 0, 0);
            sml = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], sml, 0, 0, 0);
            sml = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], sml, 0, 0, 0);
            sml = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], sml, 0, 0, 0);
            sml = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], sml, 0, 0, 0);
        }
        an.store(As[buf ^ 1], tid);
        bn.store(Bs[buf ^ 1], tid);
        __syncthreads();
    };
    load(0, a0, b0);
    load(1, a1, b1);
    a0.store(As[0], tid);
    b0.store(Bs[0], tid);
    __syncthreads();
    for (int t = 0; t < tiles; t += 2) {
        step(t, 0, a1, b1, a0, b0);
        if (t + 1 < tiles) step(t + 1, 1, a0, b0, a1, b1);
    }
    acc = (acc + sml) * kPartsUnscale;
    if constexpr (BM == 32) {
        // the second k half's sums, 16 floats a lane, through LDS
        floatx4 *red = reinterpret_cast<floatx4 *>(&As[0][0][0][0]);
        static_assert(sizeof(As) >= 2 * 64 * 16 * 4, "room for two waves' sums");
        if (wk == 1) {
#pragma unroll
            for (int q = 0; q < 4; q++)
                red[(wn * 4 + q) * 64 + lane] = floatx4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
        }
        __syncthreads();
        if (wk == 1) return;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const floatx4 v = red[(wn * 4 + q) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; e++) acc[4 * q + e] += v[e];
        }
    }
    // outputs that parts cannot give: the wave's block again without them
    unsigned odd = 0;
#pragma unroll
    for (int r = 0; r < 16; r++) odd |= static_cast<unsigned>(parts_unfit(acc[r])) << r;
    const int n = n0 + wn * 32 + row;
    if (__ballot(odd != 0)) {
        auto operand = [&](__amdgpu_buffer_rsrc_t rs, int ld, bool kcont, int at, int count, int k,
                           float (&v)[8]) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int kk = k + 8 * half + e;
                const int off = (kcont ? at * ld + kk : kk * ld + at) * 4;
                v[e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(rs, at < count && kk < p.K ? off : 0x7fff0000, 0, 0));
            }
        };
        const floatx16 plain = block_sum_f32(
            0, p.K,
            [&](int k, float (&v)[8]) __attribute__((always_inline)) {
                operand(ars, lda, !TA, m0 + wm * 32 + row, p.M, k, v);
            },
            [&](int k, float (&v)[8]) __attribute__((always_inline)) { operand(brs, ldb, TB, n, p.N, k, v); });
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = odd >> r & 1 ? plain[r] : acc[r];
    }
    // accumulator layout: column lane & 31, rows 8*(r/4) + 4*(lane/32) + r%4
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int m = m0 + wm * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
        if (m < p.M && n < p.N) Y[static_cast<size_t>(m) * p.N + n] = acc[r];
    }
}

// Batched MatMul for grids too small to fill the GPU with 64x64 tiles (the
// PSA attention products at batch 1): one 32x32 tile per workgroup, its k
// range cut into four contiguous quarters (whole groups of 8 k), one per
// wave.  Each wave accumulates the whole tile over its quarter on
// v_mfma_f32_32x32x2f32 with its operands loaded straight into registers,
// four groups of loads in flight (lanes 0-31 take k = 8g + t and lanes 32-63
// k = 8g + 4 + t for MFMA step t of group g, for A and B alike, so every k
// is summed once); the four partial tiles are then summed through LDS in
// wave order, so the result does not depend on timing.
__global__ void __launch_bounds__(256) matmul_ksplit(MatmulArgs p) {
    __shared__ float red[4][1024];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 31, half = lane >> 5;
    const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
    size_t ab = 0, bb = 0;
    matmul_batch(p, blockIdx.z, &ab, &bb);
    const size_t M = p.M, N = p.N, K = p.K;
    const float *A = p.a + ab * M * K;
    const float *B = p.b + bb * K * N;
    float *Y = p.y + static_cast<size_t>(blockIdx.z) * M * N;
    const int groups = (p.K + 7) / 8;
    const int per = (groups + 3) / 4;
    const int g0 = wave * per, g1 = min(g0 + per, groups);
    const int am = m0 + row, bn = n0 + row;
    const bool arow = am < p.M, bcol = bn < p.N;
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    for (int gi = g0; gi < g1; gi += 4) {
        float av[4][4], bv[4][4];
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int k = (gi + u) * 8 + 4 * half + t;
                const bool ok = gi + u < g1 && k < p.K;
                av[u][t] = ok && arow ? A[static_cast<size_t>(am) * K + k] : 0.0f;
                bv[u][t] = ok && bcol ? B[static_cast<size_t>(k) * N + bn] : 0.0f;
            }
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int t = 0; t < 4; t++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[u][t], bv[u][t], acc, 0, 0, 0);
    }
    // accumulator layout: column lane & 31, rows 8*(r/4) + 4*(lane/32) + r%4
#pragma unroll
    for (int r = 0; r < 16; r++) red[wave][(8 * (r >> 2) + 4 * half + (r & 3)) * 32 + row] = acc[r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int e = tid * 4 + i;
        const int m = m0 + (e >> 5), n = n0 + (e & 31);
        const float v = ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
        if (m < p.M && n < p.N) Y[static_cast<size_t>(m) * N + n] = v;
    }
}

}  // namespace

int gemm_prepare(Spkv2Context *ctx, const Spkv2NodeRecord *node, size_t *ws) {
    void **slot = &ctx->plans[node->id];
    if (*slot) {
        const ConvPlan &p = static_cast<GemmPlan *>(*slot)->conv;
        *ws = p.ws_in_scratch ? 0 : p.workspace;
        return 0;
    }
    Spkv2AttrRecord attr;
    if (int rc = spkv2_ctx_get_attr(ctx, node, &attr)) return rc;
    if (node->input_count < 2 || node->output_count < 1) return -11;
    const Spkv2TensorRecord *ar = rec(ctx, node->inputs[0]), *br = rec(ctx, node->inputs[1]);
    if (ar->rank != 2 || br->rank != 2) return -11;
    if (ar->dtype != SPKV2_DTYPE_FP32 || br->dtype != SPKV2_DTYPE_FP32) return SPKV2_E_UNSUPPORTED;
    const float *bh = reinterpret_cast<const float *>(host_weight_data(ctx, node->inputs[1]));
    if (!bh) return SPKV2_E_UNSUPPORTED;  // B produced at run time
    GemmPlan *gp = new GemmPlan();
    memset(gp, 0, sizeof(*gp));
    *slot = gp;
    ctx->plan_dtors[node->id] = gemm_plan_free;
    gp->rows = attr.trans_a ? ar->shape[1] : ar->shape[0];
    gp->K = attr.trans_a ? ar->shape[0] : ar->shape[1];
    gp->Nout = attr.trans_b ? br->shape[0] : br->shape[1];
    gp->trans_a = attr.trans_a;
    gp->alpha = attr.alpha;
    // weight matrix of the 1x1 conv: W[n][k] = B'[k][n]
    std::vector<float> w(static_cast<size_t>(gp->Nout) * gp->K);
    for (int n = 0; n < gp->Nout; n++)
        for (int k = 0; k < gp->K; k++)
            w[static_cast<size_t>(n) * gp->K + k] =
                attr.trans_b ? bh[static_cast<size_t>(n) * gp->K + k] : bh[static_cast<size_t>(k) * gp->Nout + n];
    ConvGeom g{};
    g.N = gp->rows;
    g.C = gp->K;
    g.H = g.W = 1;
    g.M = gp->Nout;
    g.KH = g.KW = g.OH = g.OW = 1;
    g.sh = g.sw = g.dh = g.dw = 1;
    g.group = 1;
    g.has_bias = node->input_count > 2;
    g.x_elems = static_cast<int64_t>(gp->rows) * gp->K;
    g.y_elems = static_cast<int64_t>(gp->rows) * gp->Nout;
    // byte offsets inside the kernels are 32-bit signed
    if (g.x_elems * 4 >= (int64_t(1) << 31) || g.y_elems * 4 >= (int64_t(1) << 31)) return SPKV2_E_UNSUPPORTED;
    gp->conv.g = g;
    // (also the fallback of the matrix-vector kernel: an A not 16-byte aligned)
    if (int rc = plan_igemm_gemm(ctx->stream, g, w.data(), attr.trans_a ? gp->rows : 1, &gp->conv)) return rc;
    // a forced tile configuration (SPKV2_CONV_CFG) keeps the tiles
    if (gp->rows >= 1 && gp->rows <= 4 && !attr.trans_a && gp->K % 4 == 0 && !getenv("SPKV2_CONV_CFG")) {
        const size_t wb = w.size() * sizeof(float);
        if (hipMalloc(reinterpret_cast<void **>(&gp->wrow), wb) != hipSuccess) {
            (void)hipGetLastError();
            gp->wrow = nullptr;
        } else if (hipMemcpy(gp->wrow, w.data(), wb, hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipFree(gp->wrow);
            gp->wrow = nullptr;
        }
    }
    set_kernel_name(ctx, node, gp->wrow ? "gemm:gemv_f32<" + std::to_string(gp->rows) + ">"
                                        : "gemm:" + igemm_name(&gp->conv));
    *ws = claim_spec_scratch(ctx, node, &gp->conv);
    return 0;
}

int run_igemm_f32_strided(Spkv2Context *ctx, const ConvPlan *p, const float *x, const float *bias, float *y,
                          float alpha, int x_img_stride);

int gemm_run(Spkv2Context *ctx, const Spkv2NodeRecord *node, void *) {
    if (ctx->plan_dtors[node->id] != gemm_plan_free) return SPKV2_E_UNSUPPORTED;  // not prepared as a Gemm
    GemmPlan *gp = static_cast<GemmPlan *>(ctx->plans[node->id]);
    if (!gp) return SPKV2_E_UNSUPPORTED;
    const float *a = dptr<const float>(ctx, node->inputs[0]);
    const float *c = node->input_count > 2 ? dptr<const float>(ctx, node->inputs[2]) : nullptr;
    float *y = dptr<float>(ctx, node->outputs[0]);
    if (gp->wrow && (reinterpret_cast<uintptr_t>(a) & 15) == 0) {
        const dim3 grid(static_cast<unsigned>((gp->Nout + 3) / 4));
        switch (gp->rows) {
            case 1: gemv_f32<1><<<grid, 256, 0, ctx->stream>>>(gp->wrow, a, c, y, gp->K, gp->Nout, gp->alpha); break;
            case 2: gemv_f32<2><<<grid, 256, 0, ctx->stream>>>(gp->wrow, a, c, y, gp->K, gp->Nout, gp->alpha); break;
            case 3: gemv_f32<3><<<grid, 256, 0, ctx->stream>>>(gp->wrow, a, c, y, gp->K, gp->Nout, gp->alpha); break;
            default: gemv_f32<4><<<grid, 256, 0, ctx->stream>>>(gp->wrow, a, c, y, gp->K, gp->Nout, gp->alpha); break;
        }
        return launch_status("gemv_f32");
    }
    // A is [rows][K] (one "image" of K channels per row), or [K][rows] with trans_a
    return run_igemm_f32_strided(ctx, &gp->conv, a, c, y, gp->alpha, gp->trans_a ? 1 : gp->K);
}

int matmul_run(Spkv2Context *ctx, const Spkv2NodeRecord *node, void *) {
    const Spkv2TensorRecord *ar = rec(ctx, node->inputs[0]), *br = rec(ctx, node->inputs[1]),
                            *yr = rec(ctx, node->outputs[0]);
    if (ar->rank < 2 || br->rank < 2 || yr->rank < 2 || ar->rank > 8 || br->rank > 8 || yr->rank > 8) return -11;
    if (ar->dtype != SPKV2_DTYPE_FP32 || br->dtype != SPKV2_DTYPE_FP32) return SPKV2_E_UNSUPPORTED;
    const uint64_t M = yr->shape[yr->rank - 2], N = yr->shape[yr->rank - 1], K = ar->shape[ar->rank - 1];
    // operands must hold what the loops read (the reference trusts the records)
    if (ar->shape[ar->rank - 2] != M || br->shape[br->rank - 2] != K || br->shape[br->rank - 1] != N) return -11;
    const uint64_t total = elem_count(yr);
    if (total == 0) return 0;
    const uint64_t batch = total / (M * N);
    for (int d = 0; d + 2 < yr->rank; d++) {
        const int da = d - (yr->rank - ar->rank), db = d - (yr->rank - br->rank);
        if (da >= 0 && ar->shape[da] != 1 && ar->shape[da] != yr->shape[d]) return -11;
        if (db >= 0 && br->shape[db] != 1 && br->shape[db] != yr->shape[d]) return -11;
    }
    if (M > 0x7fffffffULL || N > 0x7fffffffULL || K > 0x7fffffffULL) return SPKV2_E_UNSUPPORTED;
    const uint64_t mt = (M + kMmTile - 1) / kMmTile, nt = (N + kMmTile - 1) / kMmTile;
    if (mt > 65535 || batch > 65535 || nt > 0x7fffffffULL) return SPKV2_E_UNSUPPORTED;
    // on the fp32 matrix cores: 64x64 tiles for fewer than half the CUs: 32x32
    // tiles with k split over the waves instead (measured on the PSA attention
    // products: 14 tiles at batch 1 27 -> 15 us of node time; 224 tiles at
    // batch 16 the 64x64 kernel is faster);
    // SPKV2_MATMUL_KSPLIT=0 / 1 forces either
    const uint64_t mt32 = (M + 31) / 32, nt32 = (N + 31) / 32;
    bool ksplit = mt * nt * batch < 128 && mt32 <= 65535;
    if (const char *e = getenv("SPKV2_MATMUL_KSPLIT")) ksplit = e[0] == '1' ? mt32 <= 65535 : false;
    MatmulArgs p{};
    p.a = dptr<const float>(ctx, node->inputs[0]);
    p.b = dptr<const float>(ctx, node->inputs[1]);
    p.y = dptr<float>(ctx, node->outputs[0]);
    p.M = static_cast<int>(M);
    p.N = static_cast<int>(N);
    p.K = static_cast<int>(K);
    p.yrank = yr->rank;
    p.arank = ar->rank;
    p.brank = br->rank;
    for (int i = 0; i < 8; i++) {
        p.yshape[i] = static_cast<int>(yr->shape[i]);
        p.ashape[i] = static_cast<int>(ar->shape[i]);
        p.bshape[i] = static_cast<int>(br->shape[i]);
    }
    bool trans[2] = {false, false};
    for (int slot = 0; slot < 2; slot++) {
        const size_t at = 2 * static_cast<size_t>(node->id) + slot;
        if (at >= ctx->matmul_src.size() || !ctx->matmul_src[at] || !handoffs_live(ctx)) continue;
        trans[slot] = true;
        (slot ? p.b : p.a) = dptr<const float>(ctx, ctx->matmul_src[at] - 1);
    }
    // (the parts kernel's offsets into one matrix are 31-bit)
    const uint64_t limit = 0x7fff0000ULL / 4;
    // 32 rows and k over the waves where k is long and the 64-row tiles would
    // leave CUs idle (one 512^3 product, 64 tiles: 12.0 us against 13.7; eight
    // of them, 512 tiles: 33 against 22); few tiles without a Transpose to
    // save stay on the fp32 tiles, k split, whose loads go straight to
    // registers (four 128^3 products: 3.6 us against 5.5)
    const uint64_t tiles64 = ((M + 63) / 64) * ((N + 63) / 64) * batch;
    const bool small = K > 64 && tiles64 < 256;
    const int bm = small ? 32 : 64;
    const uint64_t mt_pt = (M + bm - 1) / bm, nt_pt = (N + kPtN - 1) / kPtN;
    const bool parts_fit = K >= kPartsMinK && M * K < limit && K * N < limit && mt_pt <= 65535;
    const bool reads_transposed = node->id < ctx->matmul_parts.size() && ctx->matmul_parts[node->id];
    const bool parts = (tiles64 >= 64 || reads_transposed) && !getenv("SPKV2_MATMUL_KSPLIT");
    if (parts_fit && (parts || trans[0] || trans[1])) {
        set_kernel_name(ctx, node, "matmul_parts<" + std::to_string(bm) + "x64" + (trans[0] ? ",ta" : "") +
                                       (trans[1] ? ",tb" : "") + ">");
        using Kernel = void (*)(MatmulArgs);
#define PARTS_TILE(BM, Q)                                                                    \
    {{matmul_parts<BM, false, false, Q>, matmul_parts<BM, false, true, Q>},                  \
     {matmul_parts<BM, true, false, Q>, matmul_parts<BM, true, true, Q>}}
        const Kernel kernels[2][2][2][2] = {{PARTS_TILE(64, false), PARTS_TILE(32, false)},
                                            {PARTS_TILE(64, true), PARTS_TILE(32, true)}};
#undef PARTS_TILE
        hipLaunchKernelGGL(kernels[K % 4 == 0][small][trans[0]][trans[1]],
                           dim3(static_cast<unsigned>(nt_pt), static_cast<unsigned>(mt_pt),
                                static_cast<unsigned>(batch)),
                           dim3(256), 0, ctx->stream, p);
        return launch_status("matmul");
    }
    if (trans[0] || trans[1]) return SPKV2_E_UNSUPPORTED;  // not set up that way
    if (ksplit) {
        set_kernel_name(ctx, node, "matmul_ksplit_f32<32x32>");
        hipLaunchKernelGGL(matmul_ksplit, dim3(static_cast<unsigned>(nt32), static_cast<unsigned>(mt32),
                                               static_cast<unsigned>(batch)),
                           dim3(256), 0, ctx->stream, p);
        return launch_status("matmul");
    }
    set_kernel_name(ctx, node, "matmul_mfma_f32<64x64x16>");
    hipLaunchKernelGGL(matmul_mfma, dim3(static_cast<unsigned>(nt), static_cast<unsigned>(mt),
                                         static_cast<unsigned>(batch)),
                       dim3(256), 0, ctx->stream, p);
    return launch_status("matmul");
}

}  // namespace spk::kern
