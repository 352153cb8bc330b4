// fp32 implicit GEMM on the bf16 matrix cores (conv_split_f32), for the layers
// large enough to be bound by the fp32 ones.
//
// A float is the sum of three bf16 parts (8 + 8 + 8 significant bits), and a
// product of two floats the sum of nine products of parts, each exact in
// float32.  The six largest are computed, on v_mfma_f32_32x32x16_bf16, which
// runs 16 times as many operations a cycle as v_mfma_f32_32x32x2_f32: 2.7
// times the fp32 rate at the clocks' limit, though at this load the chip
// holds the matrix cores to about 1.5 PFLOP/s, 1.6 times what the fp32 ones
// reach.  The three products left out are below 2^-24 of the whole together
// (2^-25, 2^-25 and 2^-34).  The split and the six products are those of Henry,
// Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype
// For Higher-Precision Computations" (ARITH 2019).
//
// Precision: against 64-bit sums of N(0, 1) data the relative error is 5e-8
// at K = 64, 8.5e-8 at 256 and 2.9e-7 at 2304, where the fp32 MFMA's is
// 1.4e-7, 2.7e-7 and 8.7e-7: sixteen products are summed before a rounding
// instead of two, and the five smaller products have an accumulator of their
// own (in one accumulator all six would round at the sum's size: 7.3e-7 at
// 2304).  The parts are of operands scaled by 2^24, which makes them exact for
// the smallest floats too (parts.hpp).  Infinities, NaN and overflows of scaled
// operands or sums are summed again in float32 multiply-adds (below).
//
// What bounds it: per 128 x 64 x 32 step a workgroup runs 768 cycles of MFMA
// a SIMD, loads 24 KB of weights (fragment order, straight to registers) and
// 8 KB of activations, which it splits (6.5 VALU operations an element) into
// 12 KB of LDS pieces that every wave reads.  Timed on a 14x14 3x3 layer, 256
// channels, batch 64 (14.8 GFLOP, 392 tiles on 256 CUs): 101 us; without the
// activations' loads 90, without splitting them 84, without the weights'
// loads 75; the fp32 tiles take 117 us.
#define SPK_SPLIT_DEFINE
#include "igemm_split.hpp"
#include "parts.hpp"

namespace spk::kern {

namespace {

// BM x BK tiles [m_tiles][k_tiles], each [BM/32][BK/16][3 parts][64 lanes][8]
// bf16: lane l of a 32x32x16 step holds row l & 31, k = 8 * (l >> 5) + 0..7 of
// one part of 2^24 w.  One thread per lane and step; ragged edges are zeros.
constexpr unsigned kRawWeight = 0x7f80;  // bf16 infinity, no part of a finite weight
__global__ void __launch_bounds__(256) pack_split_kernel(const float *__restrict__ w, int M, int K, int blocks, int steps,
                                                         int k_tiles, unsigned pieces, uintx4 *__restrict__ out) {
    const unsigned id = blockIdx.x * 256u + threadIdx.x;
    if (id >= pieces) return;
    const unsigned at = id / 64, lane = id & 63;
    const unsigned step = at % steps, kt = at / (blocks * steps) % k_tiles;
    const int m = static_cast<int>((at / (k_tiles * blocks * steps) * blocks + at / steps % blocks) * 32 + lane % 32);
    const int k = static_cast<int>((kt * steps + step) * 16 + lane / 32 * 8);
    unsigned part[3][8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float raw = m < M && k + j < K ? w[static_cast<size_t>(m) * K + k + j] : 0.0f;
        float v = raw * kPartsScale;
        if (!(__builtin_fabsf(v) < __builtin_inff())) {
            // 2^104 and above, infinite or NaN: an infinite part, which makes
            // every sum it enters one that is summed again, from the weight's
            // own bits in the other two
            part[0][j] = kRawWeight;
            part[1][j] = __float_as_uint(raw) >> 16;
            part[2][j] = __float_as_uint(raw) & 0xffffu;
            continue;
        }
#pragma unroll
        for (int p = 0; p < 3; p++) {
            // to nearest; the largest floats are cut, so that none becomes infinite
            const unsigned u = __float_as_uint(v);
            const unsigned h = (u & 0x7fffffffu) >= 0x7f7f8000u ? u : u + 0x7fffu + (u >> 16 & 1);
            part[p][j] = h >> 16;
            v -= __uint_as_float(h & 0xffff0000u);
        }
    }
#pragma unroll
    for (int p = 0; p < 3; p++) {
        uintx4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = part[p][2 * e] | part[p][2 * e + 1] << 16;
        out[(static_cast<size_t>(at) * 3 + p) * 64 + lane] = o;
    }
}

// Implicit padding: bit kh of the result is set when tap row kh of the column
// whose tap (0, 0) is at (ih, iw) lies inside the input, bit 16 + kw when tap
// column kw does.  The table holds bits kh and 16 + kw for each k, so an
// element's check is one and, one compare.
__device__ __forceinline__ unsigned tap_mask(const IgemmArgs &a, int ih, int iw) {
    unsigned v = 0;
    for (int t = 0; t < a.chk_KH; t++)
        v |= static_cast<unsigned>(static_cast<unsigned>(ih + t * a.chk_dh) < static_cast<unsigned>(a.chk_H)) << t;
    for (int t = 0; t < a.chk_KW; t++)
        v |= static_cast<unsigned>(static_cast<unsigned>(iw + t * a.chk_dw) < static_cast<unsigned>(a.chk_W))
             << (16 + t);
    return v;
}

}  // namespace

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int WPE, int MODE>
__global__ void __launch_bounds__(64 * WAVES_M * WAVES_N, WPE - (BM == 128 && MODE == kModeKvec)) conv_split_f32(IgemmArgs a) {
    constexpr int NT = 64 * WAVES_M * WAVES_N;
    constexpr int TM = BM / (32 * WAVES_M);
    constexpr int TN = BN / (32 * WAVES_N);
    constexpr int Q = BK / 16;           // MFMA k steps per k-tile
    constexpr int KG = BK / 8;           // 16-byte k groups per plane and column
    constexpr int KPT = BK * BN / NT;    // B elements per thread per k-tile
    constexpr int GPT = KPT / 8;         // k groups per thread
    // B is a matrix of rows (a Gemm's A): eight lanes read the 32 k of a row,
    // four each, where lane-per-column loads would touch a line per lane
    constexpr bool ROWMAJOR = MODE == kModeKvec;
    constexpr int RPP = NT / 8;          // rows per pass of the workgroup
    constexpr int PAD = ROWMAJOR ? 4 : 0;  // keeps its 8-byte LDS writes off each other's banks
    static_assert(BK == 32 && (!ROWMAJOR || BN % RPP == 0), "row-major pass");
    static_assert(TM >= 1 && TN >= 1 && KPT % 8 == 0 && BN >= 64 && NT % BN == 0, "tile shape");

    // [buffer][plane][k group][column] 16-byte pieces: a thread writes the
    // pieces of its column, a wave reads 32 columns of two groups, both
    // contiguous across lanes (no bank conflicts without padding)
    __shared__ __attribute__((aligned(16))) uintx4 Bs[2][3][KG][BN + PAD];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WAVES_N;
    const int wn = wave % WAVES_N;

    // tiles, split-K slices and the hybrid schedule as in conv_igemm_f32
    int bid = blockIdx.x;
    int slice = blockIdx.y;
    bool part = a.ws != nullptr;
    if (a.dp_tiles > 0) {
        if (bid < a.dp_tiles) {
            if ((a.dp_tiles & 7) == 0) bid = (bid & 7) * (a.dp_tiles >> 3) + (bid >> 3);
            part = false;
        } else {
            const int r = bid - a.dp_tiles;
            bid = a.dp_tiles + r / a.rem_split;
            slice = r - (r / a.rem_split) * a.rem_split;
        }
    } else {
        const int nb = gridDim.x;
        if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
    }
    const int mt = bid % a.m_tiles;
    const int nt = bid / a.m_tiles;
    const int kt0 = part ? slice * a.kt_per_split : 0;
    const int kt1 = part ? min(kt0 + a.kt_per_split, a.k_tiles) : a.k_tiles;
    if (kt0 >= kt1) return;  // empty split-K slice

    const int bcol = tid % BN;
    const int bgrp = __builtin_amdgcn_readfirstlane(tid / BN);  // wave-uniform: BN >= 64
    const int row = lane & 31;
    const int half = lane >> 5;

    // kModeChk: tap (0, 0) of a column may lie up to `before` bytes ahead of
    // the input; offsets count from there, so that none is negative (no load
    // goes there: its taps are not valid)
    const int before = MODE == kModeChk ? (a.chk_ph * a.Wp + a.chk_pw) * 4 : 0;
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char *>(reinterpret_cast<const char *>(a.x) - before), static_cast<short>(0), a.x_bytes + before,
        kBufferWord3);
    int col = kOobOffset;
    unsigned valid = 0;  // kModeChk: the column's taps inside the input
    {
        const int n = nt * BN + bcol;
        if (n < a.Ntot) {
            const int img = n / a.OHW;
            const int sp = n - img * a.OHW;
            const int oh = sp / a.OW;
            const int ow = sp - oh * a.OW;
            // from `before` ahead of the input, tap (0, 0) is at row oh * sh
            col = (img * a.x_img_stride + oh * a.sh * a.Wp + ow * a.sw) * 4;
            if constexpr (MODE == kModeChk) valid = tap_mask(a, oh * a.sh - a.chk_ph, ow * a.sw - a.chk_pw);
        }
    }

    // row-major B: this lane's first k of a tile, and its rows
    const int K = a.sk_C;
    const int rk = (tid & 7) * 4;
    int rowoff[ROWMAJOR ? BN / RPP : 1];
    if constexpr (ROWMAJOR) {
#pragma unroll
        for (int p = 0; p < BN / RPP; p++) {
            const int n = nt * BN + (tid >> 3) + p * RPP;
            rowoff[p] = n < a.Ntot ? n * a.x_img_stride * 4 : kOobOffset;
        }
    }

    // A: [m_tile][k_tile][32-row block][k step][part][lane] 16-byte pieces
    const bf16x8 *const wbase = reinterpret_cast<const bf16x8 *>(a.wp) +
                                (static_cast<size_t>(mt) * a.k_tiles * (BM / 32) + wm * TM) * (Q * 3 * 64) + lane;
    bf16x8 a0[TM][Q][3], a1[TM][Q][3];
    float br0[KPT], br1[KPT];

    auto load_a = [&](int kt, bf16x8 (&ax)[TM][Q][3]) __attribute__((always_inline)) {
        const bf16x8 *src = wbase + static_cast<size_t>(min(kt, a.k_tiles - 1)) * ((BM / 32) * Q * 3 * 64);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int q = 0; q < Q; q++)
#pragma unroll
                for (int p = 0; p < 3; p++) ax[i][q][p] = src[((i * Q + q) * 3 + p) * 64];
    };
    // The k offsets are read one tile ahead of the loads that use them (the
    // table goes kTilesPastK tiles past K), in two sets taken
    // in turn: a scalar load in flight makes every wait for LDS wait for it
    // too, so it is issued ahead of the step's vector loads, which cover it
    // (72 to 100 channels, stride 2, at 75x57, batch 5 33.2 -> 30.8 us; it also
    // freed registers, and the checked 128- and 32-row tiles a third wave).
    struct Offsets {
        int ko[KPT];
        unsigned tap[MODE == kModeChk ? KPT : 1];
    } o0, o1;
    auto load_ko = [&](int kt, Offsets &o) __attribute__((always_inline)) {
        if constexpr (ROWMAJOR) return;
#pragma unroll
        for (int j = 0; j < KPT; j++) {
            o.ko[j] = a.koff[kt * BK + bgrp * KPT + j];
            if constexpr (MODE == kModeChk) o.tap[j] = static_cast<unsigned>(a.ktap[kt * BK + bgrp * KPT + j]);
        }
    };
    auto load_b = [&](int kt, float (&br)[KPT], const Offsets &o) __attribute__((always_inline)) {
        if constexpr (ROWMAJOR) {
            // the quad of the last tile that K cuts is read from K - 4 on
            // and shifted into place when it is split (store_b)
            const int k4 = min(kt * BK + rk, K - 4) * 4;
#pragma unroll
            for (int p = 0; p < BN / RPP; p++) {
                const floatx4 v =
                    __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xrs, rowoff[p] + k4, 0, 0));
                br[4 * p] = v[0];
                br[4 * p + 1] = v[1];
                br[4 * p + 2] = v[2];
                br[4 * p + 3] = v[3];
            }
            return;
        } else if constexpr (MODE == kModeChk) {
#pragma unroll
            for (int j = 0; j < KPT; j++)
                br[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                      xrs, (valid & o.tap[j]) == o.tap[j] ? col : kOobOffset, o.ko[j], 0));
        } else {
#pragma unroll
            for (int j = 0; j < KPT; j++)
                br[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, col, o.ko[j], 0));
        }
    };
    auto store_b = [&](int kt, int buf, const float (&br)[KPT]) __attribute__((always_inline)) {
        if constexpr (ROWMAJOR) {
            float v[KPT];
#pragma unroll
            for (int j = 0; j < KPT; j++) v[j] = br[j];
            if ((kt + 1) * BK > K) {
                const int shift = kt * BK + rk - min(kt * BK + rk, K - 4);
#pragma unroll
                for (int p = 0; p < BN / RPP; p++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float t = 0.0f;  // past K
#pragma unroll
                        for (int f = e; f < 4; f++) t = f == e + shift ? br[4 * p + f] : t;
                        v[4 * p + e] = t;
                    }
            }
#pragma unroll
            for (int p = 0; p < BN / RPP; p++) {
                unsigned h[2], m[2], l[2];
                split_pair(v[4 * p], v[4 * p + 1], h[0], m[0], l[0]);
                split_pair(v[4 * p + 2], v[4 * p + 3], h[1], m[1], l[1]);
                uintx4 *at = &Bs[buf][0][rk / 8][(tid >> 3) + p * RPP];
                const int q = rk / 4 & 1;
                reinterpret_cast<uintx2 *>(at)[q] = uintx2{h[0], h[1]};
                reinterpret_cast<uintx2 *>(at + KG * (BN + PAD))[q] = uintx2{m[0], m[1]};
                reinterpret_cast<uintx2 *>(at + 2 * KG * (BN + PAD))[q] = uintx2{l[0], l[1]};
            }
            return;
        }
#pragma unroll
        for (int g = 0; g < GPT; g++) {
            uintx4 h, m, l;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                unsigned hv, mv, lv;
                split_pair(br[g * 8 + 2 * e], br[g * 8 + 2 * e + 1], hv, mv, lv);
                h[e] = hv;
                m[e] = mv;
                l[e] = lv;
            }
            Bs[buf][0][bgrp * GPT + g][bcol] = h;
            Bs[buf][1][bgrp * GPT + g][bcol] = m;
            Bs[buf][2][bgrp * GPT + g][bcol] = l;
        }
    };

    floatx16 acc[TM][TN], sml[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = sml[i][j][r] = 0.0f;

    auto frag_b = [&](int buf, int q, int p, bf16x8 (&bf)[TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; j++)
            bf[j] = __builtin_bit_cast(bf16x8, Bs[buf][p][2 * q + half][(wn * TN + j) * 32 + row]);
    };
    // one product of parts over the wave's blocks
    auto mma = [&](const bf16x8 (&ax)[TM][Q][3], int q, int pa, const bf16x8 (&bf)[TN],
                   floatx16 (&c)[TM][TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
                c[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ax[i][q][pa], bf[j], c[i][j], 0, 0, 0);
    };
    // The five products of 2^-8 and below keep a sum of their own: added one
    // by one to the large one each would round at its size.
    auto compute = [&](int buf, const bf16x8 (&ac)[TM][Q][3], const bf16x8 (&first)[TN],
                       auto &&between) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < Q; q++) {
            bf16x8 bh[TN], bm[TN], bl[TN];
            if (q == 0) {
#pragma unroll
                for (int j = 0; j < TN; j++) bh[j] = first[j];
            } else {
                frag_b(buf, q, 0, bh);
            }
            frag_b(buf, q, 1, bm);
            frag_b(buf, q, 2, bl);
            mma(ac, q, 0, bh, acc);
            mma(ac, q, 2, bh, sml);
            if (q == 0) between();
            mma(ac, q, 1, bh, sml);
            mma(ac, q, 1, bm, sml);
            mma(ac, q, 0, bm, sml);
            mma(ac, q, 0, bl, sml);
        }
    };
    auto step = [&](int kt, int buf, const bf16x8 (&ac)[TM][Q][3], bf16x8 (&an)[TM][Q][3], const float (&bnx)[KPT],
                    float (&bfree)[KPT], const Offsets &oc, Offsets &on) __attribute__((always_inline)) {
        bf16x8 first[TN];
        load_ko(kt + 3, on);
        frag_b(buf, 0, 0, first);
        __builtin_amdgcn_sched_barrier(0);
        load_b(kt + 2, bfree, oc);
        load_a(kt + 1, an);
        __builtin_amdgcn_sched_barrier(0);
        compute(buf, ac, first, [&]() __attribute__((always_inline)) { store_b(kt + 1, buf ^ 1, bnx); });
        __syncthreads();
    };

    load_ko(kt0, o0);
    load_ko(kt0 + 1, o1);
    load_b(kt0, br0, o0);
    load_b(kt0 + 1, br1, o1);
    load_ko(kt0 + 2, o0);
    load_a(kt0, a0);
    store_b(kt0, 0, br0);
    __syncthreads();
    int kt = kt0;
    // tiles past kt1 are loaded and ignored, which keeps the loop free of
    // data-dependent branches
    for (; kt + 1 < kt1; kt += 2) {
        step(kt, 0, a0, a1, br1, br0, o0, o1);
        step(kt + 1, 1, a1, a0, br0, br1, o1, o0);
    }
    if (kt < kt1) {
        bf16x8 first[TN];
        frag_b(0, 0, 0, first);
        compute(0, a0, first, []() {});
    }

    // A wave's block with an output that parts cannot give (parts_unfit) is
    // summed again without them, from the same packed weights.
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            acc[i][j] = (acc[i][j] + sml[i][j]) * kPartsUnscale;
            unsigned odd = 0;
#pragma unroll
            for (int r = 0; r < 16; r++) odd |= static_cast<unsigned>(parts_unfit(acc[i][j][r])) << r;
            if (!__ballot(odd != 0)) continue;
            const int n = nt * BN + (wn * TN + j) * 32 + row;
            const int img = n / a.OHW, sp = n - img * a.OHW, oh = sp / a.OW, ow = sp - oh * a.OW;
            const unsigned ncol = n < a.Ntot ? (img * a.x_img_stride + oh * a.sh * a.Wp + ow * a.sw) * 4 : kOobOffset;
            const unsigned taps = MODE == kModeChk && n < a.Ntot
                                      ? tap_mask(a, oh * a.sh - a.chk_ph, ow * a.sw - a.chk_pw)
                                      : 0u;
            auto weights = [&](int k, float (&v)[8]) __attribute__((always_inline)) {
                const int kt = min(k / BK, a.k_tiles - 1), q = k / 16 % Q;
                const uintx4 *src = reinterpret_cast<const uintx4 *>(wbase) +
                                    (static_cast<size_t>(kt) * (BM / 32) * Q + i * Q + q) * 3 * 64;
                const uintx4 h = src[0], m = src[64], l = src[128];
                auto whole = [](unsigned hi, unsigned mid, unsigned lo) __attribute__((always_inline)) {
                    const float sum = __uint_as_float(hi) + (__uint_as_float(mid) + __uint_as_float(lo));
                    return hi == kRawWeight << 16 ? __uint_as_float(mid | lo >> 16) : sum * (1.0f / kPartsScale);
                };
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[2 * e] = whole(h[e] << 16, m[e] << 16, l[e] << 16);
                    v[2 * e + 1] = whole(h[e] & 0xffff0000u, m[e] & 0xffff0000u, l[e] & 0xffff0000u);
                }
            };
            auto inputs = [&](int k, float (&v)[8]) __attribute__((always_inline)) {
                int ko[8], tap[8];
                const intx4 *kp = reinterpret_cast<const intx4 *>(a.koff + k + 8 * half);
                const intx4 *tp = reinterpret_cast<const intx4 *>(a.ktap + k + 8 * half);
#pragma unroll
                for (int e = 0; e < 8; e++) ko[e] = kp[e / 4][e % 4];
                if constexpr (MODE == kModeChk) {
#pragma unroll
                    for (int e = 0; e < 8; e++) tap[e] = tp[e / 4][e % 4];
                }
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    unsigned off = ncol + static_cast<unsigned>(ko[e]);  // neither wraps
                    if constexpr (MODE == kModeChk) off = (taps & tap[e]) == static_cast<unsigned>(tap[e]) ? off : kOobOffset;
                    v[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, off, 0, 0));
                }
            };
            const floatx16 plain = block_sum_f32(kt0 * BK, kt1 * BK, weights, inputs);
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = odd >> r & 1 ? plain[r] : acc[i][j][r];
        }
    igemm_epilogue<BM, BN, 32, TM, TN, ROWMAJOR>(a, acc, mt, nt, wm, wn, lane, part, slice);
}

int pack_split(hipStream_t st, const float *w, int M, int K, int BM, int BK, int m_tiles, int k_tiles, void *out) {
    const size_t pieces = static_cast<size_t>(m_tiles) * k_tiles * (BM / 32) * (BK / 16) * 64;
    if (pieces >= (size_t(1) << 31)) return SPKV2_E_UNSUPPORTED;
    hipLaunchKernelGGL(pack_split_kernel, dim3(blocks_for(pieces, 256)), dim3(256), 0, st, w, M, K, BM / 32, BK / 16,
                       k_tiles, static_cast<unsigned>(pieces), static_cast<uintx4 *>(out));
    return launch_status("pack_split");
}

#define SPLIT(BM, BN, BK, WM, WN, WPE, EFF)                                                  \
    template __global__ void conv_split_f32<BM, BN, BK, WM, WN, WPE, kModePlain>(IgemmArgs); \
    template __global__ void conv_split_f32<BM, BN, BK, WM, WN, WPE, kModeKvec>(IgemmArgs);  \
    template __global__ void conv_split_f32<BM, BN, BK, WM, WN, WPE, kModeChk>(IgemmArgs);
SPK_SPLIT_TILES(SPLIT)
#undef SPLIT

}  // namespace spk::kern
