// W8A8 GEMM for few rows (short requests, the last layer's picked rows; M <= 384): one round of small tiles
// whose waves split K, 16-bit outputs, v_mfma_i32_16x16x64_i8.
//
// What bounds these launches is the feed of the CUs that have a tile, not the matrix cores: a tile streams
// (BM + BN) rows x K bytes at 40 .. 55 bytes per ns and CU (80 with the weights in the last-level cache), and the
// 128-row and larger tiles of the other kernels leave most CUs idle there (128 x 2560 x 9728: 16 tiles of
// 128 x 160).  So tiles are as small as one round allows (thin_pick), and where such a tile has fewer fragments
// than waves, WK of the 4 to 8 waves take their own 128 bytes of every slab and the int32 partial sums meet in LDS at
// the end (exact in any order: same bits as every other schedule; no workspace, no second workgroup).  NS stages
// of LDS hold the slabs in flight, up to 150 KiB per workgroup.
// Measured on MI355X, weights cold in the caches (24 copies in turn), us, what QLinear ran before (K = 9728: split
// along K) -> this kernel:
//   M x N x K                8 rows         64 rows        128 rows       256 rows
//   2560 x 9728 + residual   21.2 ->  8.2   24.0 -> 14.0   27.0 -> 19.0   27.4 -> 24.4
//   2560 x 4096 + residual   13.0 ->  4.4   13.3 ->  5.7   14.2 ->  7.4   14.4 ->  9.3
//   6144 x 2560              19.5 ->  5.9   19.8 ->  8.6   23.6 -> 10.3   21.6 -> 13.2
//   12352 x 2560             20.1 ->  8.6   20.7 -> 11.8   24.5 -> 15.3   23.3 -> 19.2
//   19456 x 2560 SiLU        15.3 -> 14.0   17.8 -> 16.1   19.9 -> 19.4   (29.7: no tile at 193 .. 256 rows)
// Tried without gain: fragments loaded straight to registers (16 rows x 64 bytes per load: 64 clocks each in
// the address unit, 16 bytes per clock), a wave that touches the weights ahead of the DMA (they are already as
// deep in flight as the feed takes them), and a different K start per tile.
#include "gemm_i8_common.h"

namespace {

constexpr int kSub = 128;    // K bytes of one wave's share of a slab: whole cache lines

// A BM x BN tile (SiLU: BN / 2 outputs wide, BN / 2 gate rows and the matching up rows) on WK x WM x WN waves:
// WK of them split each slab's K, the others the tile; NS LDS stages of one slab (WK x 128 bytes of K) each.
template <int BM_, int BN_, int WK_, int WM_, int WN_, int NS_>
struct TCfg {
    static constexpr int BM = BM_, BN = BN_, WK = WK_, WM = WM_, WN = WN_, NS = NS_;
    static constexpr int kWaves = WK * WM * WN;
    static constexpr int MT = BM / 16 / WM, NT = BN / 16 / WN;
    static constexpr int kRows = BM + BN;
    static constexpr int kStage = kRows * kSub * WK;
    static constexpr int kDma = kRows / 8 * WK / kWaves; // 1 KiB DMA instructions a wave issues per slab
    static constexpr int kRed = WK > 1 ? WK * BM * BN * 4 : 0;
    static constexpr int kSmem = NS * kStage > kRed ? NS * kStage : kRed;
    static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0 && kRows / 8 * WK % kWaves == 0, "split");
    static_assert(kSmem <= 160 * 1024 && NS >= 2 && (NS - 1) * kDma < 64, "LDS, vmcnt");
};

// The fragments of one slab: NX row blocks at x0 / x1 (k-steps 0 / 1) and NW at w0 / w1, 2048 bytes (16 rows)
// apart, read and waited for in one asm block (the compiler's own LDS loads would wait for the LDS DMA in flight).
template <int NX, int NW>
MICA_DEVICE void read_frags(v4i (&x)[2][NX], v4i (&w)[2][NW], uint32_t x0, uint32_t x1, uint32_t w0, uint32_t w1);
#define MICA_RD(o, a, i) "ds_read_b128 %" #o ", %[" #a "] offset:2048*" #i "\n\t"
template <>
MICA_DEVICE void read_frags<1, 1>(v4i (&x)[2][1], v4i (&w)[2][1], uint32_t x0, uint32_t x1, uint32_t w0,
                                  uint32_t w1) {
    asm volatile(MICA_RD(0, x0, 0) MICA_RD(1, w0, 0)
                 MICA_RD(2, x1, 0) MICA_RD(3, w1, 0)
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(w[0][0]), "=&v"(x[1][0]), "=&v"(w[1][0])
                 : [x0] "v"(x0), [x1] "v"(x1), [w0] "v"(w0), [w1] "v"(w1));
}
template <>
MICA_DEVICE void read_frags<1, 2>(v4i (&x)[2][1], v4i (&w)[2][2], uint32_t x0, uint32_t x1, uint32_t w0,
                                  uint32_t w1) {
    asm volatile(MICA_RD(0, x0, 0) MICA_RD(1, w0, 0) MICA_RD(2, w0, 1)
                 MICA_RD(3, x1, 0) MICA_RD(4, w1, 0) MICA_RD(5, w1, 1)
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[1][0]), "=&v"(w[1][0]),
                   "=&v"(w[1][1])
                 : [x0] "v"(x0), [x1] "v"(x1), [w0] "v"(w0), [w1] "v"(w1));
}
template <>
MICA_DEVICE void read_frags<1, 4>(v4i (&x)[2][1], v4i (&w)[2][4], uint32_t x0, uint32_t x1, uint32_t w0,
                                  uint32_t w1) {
    asm volatile(MICA_RD(0, x0, 0) MICA_RD(1, w0, 0) MICA_RD(2, w0, 1) MICA_RD(3, w0, 2)
                 MICA_RD(4, w0, 3)
                 MICA_RD(5, x1, 0) MICA_RD(6, w1, 0) MICA_RD(7, w1, 1) MICA_RD(8, w1, 2)
                 MICA_RD(9, w1, 3)
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[0][3]),
                   "=&v"(x[1][0]), "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(w[1][2]), "=&v"(w[1][3])
                 : [x0] "v"(x0), [x1] "v"(x1), [w0] "v"(w0), [w1] "v"(w1));
}
template <>
MICA_DEVICE void read_frags<2, 2>(v4i (&x)[2][2], v4i (&w)[2][2], uint32_t x0, uint32_t x1, uint32_t w0,
                                  uint32_t w1) {
    asm volatile(MICA_RD(0, x0, 0) MICA_RD(1, x0, 1) MICA_RD(2, w0, 0) MICA_RD(3, w0, 1)
                 MICA_RD(4, x1, 0) MICA_RD(5, x1, 1) MICA_RD(6, w1, 0) MICA_RD(7, w1, 1)
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[1][0]),
                   "=&v"(x[1][1]), "=&v"(w[1][0]), "=&v"(w[1][1])
                 : [x0] "v"(x0), [x1] "v"(x1), [w0] "v"(w0), [w1] "v"(w1));
}
template <>
MICA_DEVICE void read_frags<2, 4>(v4i (&x)[2][2], v4i (&w)[2][4], uint32_t x0, uint32_t x1, uint32_t w0,
                                  uint32_t w1) {
    asm volatile(MICA_RD(0, x0, 0) MICA_RD(1, x0, 1) MICA_RD(2, w0, 0) MICA_RD(3, w0, 1)
                 MICA_RD(4, w0, 2) MICA_RD(5, w0, 3)
                 MICA_RD(6, x1, 0) MICA_RD(7, x1, 1) MICA_RD(8, w1, 0) MICA_RD(9, w1, 1)
                 MICA_RD(10, w1, 2) MICA_RD(11, w1, 3)
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(w[0][2]),
                   "=&v"(w[0][3]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(w[1][0]), "=&v"(w[1][1]),
                   "=&v"(w[1][2]), "=&v"(w[1][3])
                 : [x0] "v"(x0), [x1] "v"(x1), [w0] "v"(w0), [w1] "v"(w1));
}
template <>
MICA_DEVICE void read_frags<5, 2>(v4i (&x)[2][5], v4i (&w)[2][2], uint32_t x0, uint32_t x1, uint32_t w0,
                                  uint32_t w1) {
    asm volatile(MICA_RD(0, x0, 0) MICA_RD(1, x0, 1) MICA_RD(2, x0, 2) MICA_RD(3, x0, 3)
                 MICA_RD(4, x0, 4) MICA_RD(5, w0, 0) MICA_RD(6, w0, 1)
                 MICA_RD(7, x1, 0) MICA_RD(8, x1, 1) MICA_RD(9, x1, 2) MICA_RD(10, x1, 3)
                 MICA_RD(11, x1, 4) MICA_RD(12, w1, 0) MICA_RD(13, w1, 1)
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(x[0][3]), "=&v"(x[0][4]),
                   "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[1][2]),
                   "=&v"(x[1][3]), "=&v"(x[1][4]), "=&v"(w[1][0]), "=&v"(w[1][1])
                 : [x0] "v"(x0), [x1] "v"(x1), [w0] "v"(w0), [w1] "v"(w1));
}
template <>
MICA_DEVICE void read_frags<6, 2>(v4i (&x)[2][6], v4i (&w)[2][2], uint32_t x0, uint32_t x1, uint32_t w0,
                                  uint32_t w1) {
    asm volatile(MICA_RD(0, x0, 0) MICA_RD(1, x0, 1) MICA_RD(2, x0, 2) MICA_RD(3, x0, 3)
                 MICA_RD(4, x0, 4) MICA_RD(5, x0, 5) MICA_RD(6, w0, 0) MICA_RD(7, w0, 1)
                 MICA_RD(8, x1, 0) MICA_RD(9, x1, 1) MICA_RD(10, x1, 2) MICA_RD(11, x1, 3)
                 MICA_RD(12, x1, 4) MICA_RD(13, x1, 5) MICA_RD(14, w1, 0) MICA_RD(15, w1, 1)
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(x[0][3]), "=&v"(x[0][4]),
                   "=&v"(x[0][5]), "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]),
                   "=&v"(x[1][2]), "=&v"(x[1][3]), "=&v"(x[1][4]), "=&v"(x[1][5]), "=&v"(w[1][0]),
                   "=&v"(w[1][1])
                 : [x0] "v"(x0), [x1] "v"(x1), [w0] "v"(w0), [w1] "v"(w1));
}
#undef MICA_RD

template <class C, int EPI, int OUT, bool HAS_BIAS, bool HAS_RES>
MICA_DEVICE void thin_tile(const GemmParams &p, int8_t *smem) {
    constexpr bool kSilu = EPI == MICA_EPI_SILU_MUL;
    constexpr int MT = C::MT, NT = C::NT, NS = C::NS, kDma = C::kDma;
    static_assert(!kSilu || NT % 2 == 0, "gate / up pairs");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wk = wave / (C::WM * C::WN), wm = wave / C::WN % C::WM, wn = wave % C::WN;
    const int nt = p.tiles_m * p.tiles_n;
    const int per = nt / kXcds, rem = nt % kXcds;
    const int x = blockIdx.x % kXcds, local = blockIdx.x / kXcds;
    const int t = x * per + (x < rem ? x : rem) + local;
    const int tm = t % p.tiles_m, tn = t / p.tiles_m;
    const int m0 = tm * C::BM;
    const int r16 = lane & 15, kq = lane >> 4;

    // first weight row of the tile's 16-row block f (SiLU: a wave's NT blocks are NT / 2 gate, then NT / 2 up)
    auto brow = [&](int f) {
        if (!kSilu) return tn * C::BN + 16 * f;
        const int w = f / NT, j = f % NT;
        const int c = tn * (C::BN / 2) + (w * (NT / 2) + j % (NT / 2)) * 16;
        return (c >> 6) * 128 + (c & 63) + (j >= NT / 2 ? 64 : 0);
    };
    // DMA instruction d of this wave: 8 rows of sub-slab g; lane l takes chunk (l % 8) ^ (l / 8) of row l / 8
    int voff[kDma];
    const int lrow = lane >> 3, lcol = ((lane & 7) ^ lrow) << 4;
#pragma unroll
    for (int d = 0; d < kDma; ++d) {
        const int q = wave * kDma + d, g = q / (C::kRows / 8), r = q % (C::kRows / 8) * 8;
        if (r < C::BM) voff[d] = (m0 + r + lrow) * p.lda + g * kSub + lcol;
        else voff[d] = (brow((r - C::BM) / 16) + (r - C::BM) % 16 + lrow) * p.ldb + g * kSub + lcol;
    }
    constexpr int kSlabK = kSub * C::WK;
    const int nk = p.K / kSlabK;
    auto dma = [&](int slab, int stage) {
        const bool on = slab < nk;
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)p.A, 0, on ? p.M * p.lda : 0, kBufferFlags);
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)p.B, 0, on ? p.N * p.ldb : 0, kBufferFlags);
#pragma unroll
        for (int d = 0; d < kDma; ++d) {
            const int q = wave * kDma + d, r = q % (C::kRows / 8) * 8;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r < C::BM ? ra : rb, (lds_void *)(smem + stage * C::kStage + q * 1024),
                                                     16, voff[d], slab * kSlabK, 0, 0);
        }
    };
    v4i acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) int8_t *)smem;
    uint32_t xa[2], wa[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int pos = ((4 * s + kq) ^ (r16 & 7)) << 4;
        xa[s] = lds0 + (wk * C::kRows + wm * MT * 16 + r16) * kSub + pos;
        wa[s] = lds0 + (wk * C::kRows + C::BM + wn * NT * 16 + r16) * kSub + pos;
    }
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) dma(s, s);
    int stage = 0, into = NS - 1;
    for (int k = 0; k < nk; ++k) {
        wait_vmcnt<(NS - 2) * kDma>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        v4i fx[2][MT], fw[2][NT];
        const uint32_t so = stage * C::kStage;
        read_frags<MT, NT>(fx, fw, xa[0] + so, xa[1] + so, wa[0] + so, wa[1] + so);
        auto mma = [&](int s) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[s][j], fx[s][i], acc[i][j], 0, 0, 0);
        };
        mma(0);
        __builtin_amdgcn_sched_barrier(0);
        dma(k + NS - 1, into);
        __builtin_amdgcn_sched_barrier(0);
        mma(1);
        into = stage;
        stage = stage + 1 == NS ? 0 : stage + 1;
    }
    const int nout = kSilu ? p.N / 2 : p.N;
    constexpr int kOutN = kSilu ? NT / 2 : NT;
    // 4 consecutive output columns n .. n + 3 of row m from the sums s (SiLU: gate s, up s2)
    auto put = [&](int m, int n, v4i s, v4i s2) {
        if (m >= p.M || n >= nout) return;
        const int valid = nout - n < 4 ? nout - n : 4;
        const float sa = p.sa[m];
        const int nb = kSilu ? (n >> 6) * 128 + (n & 63) : n;
        float y[4], rv[4];
        if (HAS_RES) load4_res<OUT>(p.res, (long)m * p.ldr + n, rv, valid, p.vec_ok);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = q < valid ? nb + q : nb;
            y[q] = ((float)s[q] * sa) * p.sb[c];
            if (HAS_BIAS) y[q] = y[q] + p.bias[c];
            if (kSilu) {
                const float uv = round_bf16(((float)s2[q] * sa) * p.sb[c + 64]);
                y[q] = silu_bf16(round_bf16(y[q])) * uv;
            }
            if (HAS_RES) y[q] = to_out_precision<OUT>(y[q]) + rv[q];
        }
        store4<OUT>(p.C, (long)m * p.ldc + n, y, valid, p.vec_ok);
    };
    if constexpr (C::WK == 1) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < kOutN; ++j)
                put(m0 + (wm * MT + i) * 16 + r16, tn * (kOutN * C::WN * 16) + (wn * kOutN + j) * 16 + 4 * kq, acc[i][j],
                    kSilu ? acc[i][j + NT / 2] : acc[i][j]);
    } else {
        constexpr int kF = (C::BM / 16) * (C::BN / 16); // fragments of the tile, [row block][wn][j]
        v4i *red = (v4i *)smem;
        wait_vmcnt<0>();
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                red[(wk * kF + (wm * MT + i) * (C::WN * NT) + wn * NT + j) * 64 + lane] = acc[i][j];
        __syncthreads();
        auto sum = [&](int f) {
            v4i s = red[f * 64 + lane];
#pragma unroll
            for (int w = 1; w < C::WK; ++w) s += red[(w * kF + f) * 64 + lane];
            return s;
        };
        for (int f = wave; f < (C::BM / 16) * kOutN * C::WN; f += C::kWaves) {
            const int i = f / (kOutN * C::WN), b = f % (kOutN * C::WN), w = b / kOutN, j = b % kOutN;
            const int fr = i * (C::WN * NT) + w * NT + j;
            const v4i s = sum(fr);
            put(m0 + i * 16 + r16, (tn * kOutN * C::WN + b) * 16 + 4 * kq, s, kSilu ? sum(fr + NT / 2) : s);
        }
    }
}

template <class C, int EPI, int OUT, bool HAS_BIAS, bool HAS_RES>
__global__ __launch_bounds__(64 * C::kWaves) void gemm_i8_thin_kernel(GemmParams p) {
    extern __shared__ __align__(1024) int8_t smem[];
    thin_tile<C, EPI, OUT, HAS_BIAS, HAS_RES>(p, smem);
}

template <class C, int EPI, int OUT>
int thin_launch_tile(GemmParams p, bool has_bias, bool has_res, hipStream_t st) {
    constexpr bool kSilu = EPI == MICA_EPI_SILU_MUL;
    const int nout = kSilu ? p.N / 2 : p.N, bn = kSilu ? C::BN / 2 : C::BN;
    p.tiles_m = (p.M + C::BM - 1) / C::BM;
    p.tiles_n = (nout + bn - 1) / bn;
    dim3 grid(p.tiles_m * p.tiles_n), block(64 * C::kWaves);
#define MICA_T(B_, R_) hipLaunchKernelGGL((gemm_i8_thin_kernel<C, EPI, OUT, B_, R_>), grid, block, C::kSmem, st, p)
    if constexpr (kSilu) {
        MICA_T(false, false);
    } else {
        if (has_bias && has_res) MICA_T(true, true);
        else if (has_bias) MICA_T(true, false);
        else if (has_res) MICA_T(false, true);
        else MICA_T(false, false);
    }
#undef MICA_T
    return mica_err(hipGetLastError());
}


template <class C, int EPI>
int thin_launch_out(const GemmParams &p, int out_dtype, bool has_bias, bool has_res, hipStream_t st) {
    if (EPI == MICA_EPI_SILU_MUL || out_dtype == MICA_BF16)
        return thin_launch_tile<C, EPI, MICA_BF16>(p, has_bias, has_res, st);
    if constexpr (EPI == MICA_EPI_SCALE) return thin_launch_tile<C, EPI, MICA_FP16>(p, has_bias, has_res, st);
    return MICA_MISS_DTYPE;
}

// A launch by tile, in the order thin_pick prefers at equal cost (the faster of each pair, measured at N = 2560 and
// 10240); the 16-column tile has no gate / up pair.
typedef int (*thin_fn)(const GemmParams &, int, bool, bool, hipStream_t);
struct ThinTile {
    int bm, bn, wk;
    thin_fn scale, silu;
};
template <class C, bool SILU = true>
constexpr ThinTile thin_entry() {
    if constexpr (SILU)
        return ThinTile{C::BM, C::BN, C::WK, thin_launch_out<C, MICA_EPI_SCALE>, thin_launch_out<C, MICA_EPI_SILU_MUL>};
    else
        return ThinTile{C::BM, C::BN, C::WK, thin_launch_out<C, MICA_EPI_SCALE>, nullptr};
}
// (SiLU only: half the columns of a tile are outputs there, so a round holds wider tiles; for the plain epilogue
// 131 x 12352 x 2560 took 19.4 us on 80 x 160 tiles against 15.6 on 128 x 128)
template <class C>
constexpr ThinTile thin_silu() {
    return ThinTile{C::BM, C::BN, C::WK, nullptr, thin_launch_out<C, MICA_EPI_SILU_MUL>};
}
const ThinTile kThinTiles[] = {
    thin_entry<TCfg<16, 16, 4, 1, 1, 8>, false>(), thin_entry<TCfg<16, 32, 4, 1, 1, 6>>(),
    thin_entry<TCfg<16, 64, 4, 1, 2, 3>>(),        thin_entry<TCfg<32, 32, 4, 2, 1, 4>>(),
    thin_entry<TCfg<64, 32, 4, 2, 1, 3>>(),        thin_entry<TCfg<32, 64, 4, 1, 2, 3>>(),
    thin_entry<TCfg<64, 64, 2, 2, 2, 4>>(),        thin_entry<TCfg<32, 128, 2, 2, 2, 3>>(),
    thin_entry<TCfg<128, 64, 1, 4, 2, 5>>(),       thin_entry<TCfg<64, 128, 1, 2, 4, 5>>(),
    thin_entry<TCfg<128, 128, 1, 4, 2, 4>>(),      thin_silu<TCfg<80, 160, 1, 1, 5, 5>>(),
    thin_silu<TCfg<96, 192, 1, 1, 6, 4>>(),
};

// The tile that streams the fewest bytes per CU among those that cover the output in one round (128 x 128 with SiLU:
// or in two, the second three quarters full) and whose waves' K shares divide K; none past 384 rows or 1.25 MB a
// round.  The large tiles (128 x 128, and SiLU's own 80 x 160 and 96 x 192) have lines of their own:
//   plain: K >= 1536 (1152 where the kernels of 256-byte K steps don't serve K), and where the AGPR kernel covers the
//     output in one round of 128 x 160 tiles (gemm_i8.hip) at most 128 rows and K >= 2560;
//   SiLU: K >= 2048 (2560 past two rows of tiles), its own two at most two rows of tiles, and where the AGPR kernel
//     covers the output in one round of 128 x 128 tiles at most 128 rows.
// Measured against what would run instead, the split along K included (us, other / this; cold: 24 copies of the weights
// in turn, as in a model; warm: the same weights again, which stay in the caches).  Cold: 384 x 6144 x 2560 21.4 /
// 17.7, 384 x 2560 x 9728 28.8 / 24.2, 8192 x 1024 at 40 rows 9.7 / 5.3, SiLU x 19456 x 2560 at 131 rows 24.9 / 19.1,
// 192 27.3 / 22.6, 300 37.0 / 29.6 (two rounds).  Past the lines, cold, then warm:
//   512 x 6144 x 2560 16.5 / 18.7 cold (rows), 512 x 2560 x 9728 28.9 / 35 (bytes, 128 x 64 tiles), 384 x 12352 x 2560
//   19.6 / 33.9 (1.1 rounds), SiLU 224 x 24576 x 4096 42.7 / 47.8 (1.5);
//   plain 128 x 128, K: 321 x 6144 x 1024 7.9 / 9.1, 6.7 / 9.1; 256 x 10240 x 1024 8.4 / 9.3, 6.9 / 9.1; 257 x 8192 x
//   512 6.0 / 7.7, 5.4 / 7.4; on the other side 257 x 8192 x 1536 12.9 / 11.5, 8.3 / 11.1 and 256 x 12288 x 1280 13.0 /
//   12.1, 8.2 / 10.4 (K = 1280 at 257 x 8192: 9.3 / 10.2);
//   plain 128 x 128, one AGPR round: 257 x 10240 x 2560 16.3 / 16.3, 12.7 / 15.6; 257 x 9728 x 3584 18.6 / 20.9, 16.4 /
//   20.3; 128 x 32768 x 2048 18.2 / 19.3, 14.6 / 16.8; on the other side 128 x 19456 x 4096 30.4 / 28.3, 17.9 / 20.5;
//   SiLU: 131 x 12288 x 1024 9.0 / 10.3 cold (K; 11.8 in two rounds of 32 x 128); one AGPR round: 129 x 16384 x 2304
//   13.6 / 15.5, 12.4 / 14.3; 160 x 12288 x 2560 15.6 / 18.7, 12.3 / 15.2; 384 x 6144 x 3072 19.0 / 18.2, 12.5 / 15.6
//   (at most 128 rows: 128 x 19456 x 2560 19.8 / 19.2, 13.6 / 15.9).  K = 2048 to 2432 in two rounds past two rows of
//   tiles, which the line leaves out, would gain: 257 x 19456 x 2304 33.8 / 27.1.
// Cold decides: a model's weights are read once a pass.  Inside the lines the tiles of 128 x 128 are up to 20 % faster
// cold and up to 24 % slower warm (321 x 6144 x 2560 19.8 / 16.4, 11.2 / 14.6): the larger tiles of the other kernels
// read fewer bytes, this one has more of them in flight.
const ThinTile *thin_pick(int M, long long N, int K, bool silu, int cus) {
    const ThinTile *best = nullptr;
    long long best_bytes = 0;
    if (M > 384) return nullptr;
    const long long nout = silu ? N / 2 : N, rows128 = (M + 127) / 128;
    const long long tiles256 = (M + 255) / 256 * ((N + 255) / 256);
    const bool agpr_round = K % 256 == 0 && nout % 8 == 0 &&
                            (silu ? rows128 * (N / 128) <= cus
                                  : 4 * tiles256 > cus && 2 * tiles256 <= cus && rows128 * ((N + 159) / 160) <= cus);
    for (const ThinTile &t : kThinTiles) {
        if ((silu ? t.silu : t.scale) == nullptr || K % (kSub * t.wk) != 0) continue;
        const long long bn = silu ? t.bn / 2 : t.bn;
        const long long rows = (M + t.bm - 1) / t.bm, tiles = rows * ((nout + bn - 1) / bn);
        const bool large = t.bm + t.bn >= 240;
        if (large && silu && (K < (rows > 2 ? 2560 : 2048) || (t.scale == nullptr && rows > 2) || (agpr_round && M > 128)))
            continue;
        if (large && !silu && (K < (K % 256 == 0 ? 1536 : 1152) || (agpr_round && (M > 128 || K < 2560)))) continue;
        const bool two = large && silu && 4 * tiles >= 7 * cus && tiles <= 2 * cus;
        if (tiles > cus && !two) continue;
        const long long bytes = (long long)((M < t.bm ? M : t.bm) + t.bn) * K;
        if (bytes > 1250 * 1000) continue;
        if (best == nullptr || bytes * (two ? 2 : 1) < best_bytes) {
            best = &t;
            best_bytes = bytes * (two ? 2 : 1);
        }
    }
    return best;
}

}  // namespace

extern "C" int mica_mm_i8_few_rows_tile(int M, int N, int K, int epilogue, int cus, int *tile) {
    if (M < 0 || N <= 0 || K <= 0 || K % 16 != 0 || cus < 0 || tile == nullptr) return -1;
    if (epilogue != MICA_EPI_SCALE && (epilogue != MICA_EPI_SILU_MUL || N % 128 != 0)) return -1;
    const ThinTile *t = M > 0 ? thin_pick(M, N, K, epilogue == MICA_EPI_SILU_MUL, cus) : nullptr;
    if (t == nullptr) return 0;
    tile[0] = t->bm, tile[1] = t->bn, tile[2] = t->wk;
    return 1;
}

bool mica_gemm::thin_launch(const GemmParams &p, int epilogue, int out_dtype, int cus, bool has_bias, bool has_res,
                            hipStream_t st, int *rc) {
    const bool silu = epilogue == MICA_EPI_SILU_MUL;
    const ThinTile *t = thin_pick(p.M, p.N, p.K, silu, cus);
    if (t == nullptr) return false;
    *rc = (silu ? t->silu : t->scale)(p, out_dtype, has_bias, has_res, st);
    return true;
}
