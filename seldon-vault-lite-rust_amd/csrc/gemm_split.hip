// FP32-accurate GEMM on the F16 matrix cores: C = epilogue(A[M,K] . W[N,K]^T)
// with both operands held as pairs of halves (split rows, dev_common.hpp).
//
// Every product of two operands x = xh + xl, y = yh + yl is taken as xh.yh in
// one FP32 accumulator and xl.yh + xh.yl in a second: three F16 MFMAs. xh and
// yh carry the leading 11 bits of the scaled values and xl, yl the next 11 (of
// values within 2^-16 of their scale's top, dev_common.hpp), so the dropped xl.yl is below 2^-22 of the product, and an MFMA of 32 k
// rounds its accumulator 4 times (once per 8 products, probed) where the FP32
// MFMA chain rounds 32 times. Against 64-bit sums of normal inputs the result
// is off by 0.95e-7 / 1.9e-7 / 4.2e-7 (K = 64 / 768 / 4096, relative 2-norm)
// with a mean of -3e-9, the FP32 MFMA chain by 1.4e-7 / 5.0e-7 / 1.14e-6 with
// 3e-9. The mixed products have an accumulator of their own because the MFMA
// drops the bits of small addends downwards: in one accumulator the sums were
// off by 3.0e-7 with a mean of -1.6e-8, which averaging rows does not remove
// (2304-key attention: the image embeddings were twice as far from 64 bits).
//
// What bounds it: the F16 matrix pipes deliver 1230 TFLOP/s to a register-only
// loop of 16x16x32 MFMAs, i.e. 410 TFLOP/s of FP32 products, against 145 for
// FP32 MFMAs (32x32x16 MFMAs reach 1560, but their fragments cost registers
// and the same tiles ran 0-7 % slower on them); a split row takes the bytes of
// the FP32 row (4 per element), so HBM and LDS traffic per product are
// unchanged. At 18688 x 2304 x 768 the kernel runs at 357 TFLOP/s (185 us)
// against 142 (463 us) for the FP32 MFMA kernel; 128 x 768 x 768 with weights
// from HBM takes 5.8 against 7.0 us.
//
// Structure: WMW x WNW waves; K advances in slices of KB 32-k blocks that go
// from HBM/L2 straight into LDS (buffer_load ... lds) through NS stages, one
// barrier per slice. Rows lie unpadded in LDS, their 16-byte chunks
// XOR-swizzled by row on the way in, so fragment reads are conflict-free.
// Every tile shape issues the three products of a 32-k block in the same
// order per output, so a row's result depends neither on the tile chosen nor
// on its place in the batch.
//
// W is the first operand, so lane l holds row l % 16 of a 16x16 output block
// and its four columns 4 (l / 16) .. + 3. Two neighbouring blocks give it
// columns 4c .. 4c + 3 and 16 + 4c .. 16 + 4c + 3 (c = l / 16) of a 32-column
// group: chunk c of a split row, so an output that feeds another GEMM is split
// and stored 16 bytes at a time. Paired weights (gate / up) are interleaved in
// 16-row blocks, so neighbouring blocks hold x and y of the same outputs.
#include <algorithm>
#include <type_traits>

#include "dev_common.hpp"
#include "svl_internal.hpp"

namespace svl {

// Outputs that only another GEMM reads: stored as split rows.
template <int EPI>
constexpr bool split_output() {
    return EPI == EPI_GEGLU || EPI == EPI_GELU_MUL;
}

// Stores `lim` (<= 4) consecutive floats of a row.
__device__ __forceinline__ void store_run(float *p, const f32x4 &v, int lim, bool vec) {
    if (vec && lim >= 4) {
        *(f32x4 *)p = v;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r < lim) p[r] = v[r];
    }
}

template <int BM, int BN, int KB, int EPI, int MINB, int NS, int WMW, int WNW, bool RASTER>
__global__ __launch_bounds__(64 * WMW * WNW, MINB) void gemm_split(GemmArgs p, int tiles_m,
                                                                   int tiles_n) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NW = WMW * WNW;
    constexpr int WTM = BM / WMW, WTN = BN / WNW;  // wave tile
    constexpr int TM = WTM / 16, TN = WTN / 16;    // 16x16 output blocks per wave
    constexpr int BK = 32 * KB;                    // floats (4 bytes) per row of a slice
    constexpr int CPR = BK / 4;                    // 16-byte chunks per row
    constexpr int RPK = 64 / CPR;                  // rows per 1 KB DMA instruction
    constexpr int RPL = BK >= 64 ? 1 : 2;
    constexpr int SWZ = CPR < 16 ? CPR : 16;
    constexpr int A_CH = BM / RPK / NW, W_CH = BN / RPK / NW;  // DMA instructions per wave
    // the narrowest wave tile (one 16-column run per lane) has no pairs
    constexpr bool NARROW = WTN == 16;
    constexpr bool PAIRED = EPI == EPI_GEGLU;
    static_assert(!NARROW || !PAIRED, "paired epilogues take 32-column wave tiles");
    static_assert(WTM % 16 == 0 && (WTN % 32 == 0 || NARROW) && A_CH >= 1 && W_CH >= 1 &&
                      A_CH * RPK * NW == BM && W_CH * RPK * NW == BN,
                  "tile shape");
    static_assert(NS >= 2 && NS <= 4 && (NS - 2) * (A_CH + W_CH) < 64, "pipeline depth");
    constexpr bool SOUT = split_output<EPI>();
    // one LDS object per stage, addressed with compile-time stage indices, so
    // the compiler sees that the DMA filling one stage never aliases the
    // fragment reads of another
    __shared__ float As0[BM * BK], As1[BM * BK], As2[NS > 2 ? BM * BK : 4], As3[NS > 3 ? BM * BK : 4];
    __shared__ float Ws0[BN * BK], Ws1[BN * BK], Ws2[NS > 2 ? BN * BK : 4], Ws3[NS > 3 ? BN * BK : 4];
    auto stage_a = [&](auto st) -> float * {
        constexpr int i = decltype(st)::value;
        if constexpr (i == 0) return As0;
        else if constexpr (i == 1) return As1;
        else if constexpr (i == 2) return As2;
        else return As3;
    };
    auto stage_w = [&](auto st) -> float * {
        constexpr int i = decltype(st)::value;
        if constexpr (i == 0) return Ws0;
        else if constexpr (i == 1) return Ws1;
        else if constexpr (i == 2) return Ws2;
        else return Ws3;
    };

    // hardware hands workgroup b to XCD b % 8: each XCD runs a contiguous
    // range of the tile list
    const int ntiles = tiles_m * tiles_n;
    const int bid = blockIdx.x;
    const int xcd = bid & 7, local = bid >> 3;
    const int q8 = ntiles >> 3, r8 = ntiles & 7;
    const int tile = xcd * q8 + min(xcd, r8) + local;
    int tm, tn;
    if constexpr (RASTER) {
        // groups of SPLIT_RASTER_M M blocks, M fastest, every second group's
        // N blocks in reverse: the tiles in flight on an XCD share a few W
        // panels and A blocks
        const int gsize = SPLIT_RASTER_M * tiles_n, grp = tile / gsize,
                  first = grp * SPLIT_RASTER_M;
        const int gm = min(SPLIT_RASTER_M, tiles_m - first), in = tile - grp * gsize;
        tm = uniform(first + in % gm);
        tn = uniform(grp & 1 ? tiles_n - 1 - in / gm : in / gm);
    } else {
        tm = uniform(tile / tiles_n);
        tn = tile - tm * tiles_n;
    }
    const int m0 = tm * BM, n0 = tn * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int wm = wave / WNW, wn = wave % WNW;
    const int lr = lane & 15, lc = lane >> 4;  // fragment row and chunk of this lane
    const int M = p.M, N = p.N;

    // operand windows: reads past the last valid row return zero
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (void *)uniform(p.A + (int64_t)m0 * p.lda), (short)0,
        uniform((int)(min(BM, M - m0) * p.lda * 4)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void *)uniform(p.W + (int64_t)n0 * p.ldw), (short)0,
        uniform((int)(min(BN, N - n0) * p.ldw * 4)), 0x00020000);
    int a_off[A_CH], w_off[W_CH];
#pragma unroll
    for (int q = 0; q < A_CH; ++q) {
        const int row = (wave * A_CH + q) * RPK + lane / CPR;
        const int c = (lane % CPR) ^ ((row / RPL) % SWZ);
        a_off[q] = (row * (int)p.lda + 4 * c) * 4;
    }
#pragma unroll
    for (int q = 0; q < W_CH; ++q) {
        const int row = (wave * W_CH + q) * RPK + lane / CPR;
        const int c = (lane % CPR) ^ ((row / RPL) % SWZ);
        w_off[q] = (row * (int)p.ldw + 4 * c) * 4;
    }
    // DMA instruction q of the slice at k0: A for q < A_CH, else W
    auto issue_one = [&](auto st, int k0, int q) {
        float *as = stage_a(st);
        float *ws = stage_w(st);
        if (q < A_CH) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                ra, (__attribute__((address_space(3))) void *)&as[(wave * A_CH + q) * 256], 16,
                a_off[q], k0 * 4, 0, 0);
        } else {
            const int r = q - A_CH;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rw, (__attribute__((address_space(3))) void *)&ws[(wave * W_CH + r) * 256], 16,
                w_off[r], k0 * 4, 0, 0);
        }
    };
    constexpr int NDMA = A_CH + W_CH;
    auto issue = [&](auto st, int k0) {
#pragma unroll
        for (int q = 0; q < NDMA; ++q) issue_one(st, k0, q);
    };

    // Epilogue operands, ahead of the K loop: the descale of each column run
    // (columns col(j) .. + 3 of block j) and of each row, and EPI_GELU_MUL's
    // per-layer inputs.
    const int mw = m0 + wm * WTM, nw = n0 + wn * WTN;
    auto col = [&](int j) { return nw + 16 * j + 4 * lc; };
    f32x4 wd[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = col(j);
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (n + 3 < N) {
            v = *(const f32x4 *)(p.wd + n);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) v[r] = p.wd[n + r];
        }
        wd[j] = v;
    }
    float rs[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = mw + 16 * i + lr;
        rs[i] = p.rs && m < M ? p.rs[m] : 1.f;
    }
    f32x4 aux[EPI == EPI_GELU_MUL ? TM : 1][EPI == EPI_GELU_MUL ? TN : 1];
    if constexpr (EPI == EPI_GELU_MUL) {
        const bool vec = (p.ldaux & 3) == 0 && ((uintptr_t)p.aux & 15) == 0;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = mw + 16 * i + lr;
            const float *row = p.aux + (int64_t)(m < M ? m : 0) * p.ldaux;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = col(j);
                f32x4 v = {0.f, 0.f, 0.f, 0.f};
                if (vec && n + 3 < N) {
                    v = *(const f32x4 *)(row + n);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n + r < N) v[r] = row[n + r];
                }
                aux[i][j] = v;
            }
        }
    }

    // high products, and the two mixed ones
    f32x4 acc[TM][TN], acl[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = acl[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // 16-row blocks start at multiples of 16, so a row's swizzle depends on
    // the lane's row only
    const int sw = (lr / RPL) % SWZ;
    const int nk = p.K / BK;
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    if (0 < nk) issue(S0{}, 0);
    if constexpr (NS > 2) if (1 < nk) issue(S1{}, BK);
    if constexpr (NS > 3) if (2 < nk) issue(S2{}, 2 * BK);
    auto step = [&](int kt, auto st) {
        constexpr int cur = decltype(st)::value;
        // this wave's DMA of slice kt has landed (at most the NS - 2 later
        // slices are in flight), then every wave's; slice kt - 1 is no longer
        // read
        if (kt + NS - 2 < nk) wait_vmcnt<(NS - 2) * NDMA>();
        else wait_vmcnt<0>();
        __syncthreads();
        using NEXT = std::integral_constant<int, (cur + NS - 1) % NS>;
        const bool refill = kt + NS - 1 < nk;
        const float *as = stage_a(st) + (wm * WTM + lr) * BK;
        const float *ws = stage_w(st) + (wn * WTN + lr) * BK;
        // MFMA rounds of a slice: KB blocks x 3 products; the next slice's DMA
        // instructions go one by one behind the rounds of the first half
        constexpr int NR = KB * 3, HALF = (NR + 1) / 2;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            f16x8 ah[TM], al[TM], bh[TN], bl[TN];
            const int ph = 4 * ((kb * 8 + lc) ^ sw), pl = 4 * ((kb * 8 + lc + 4) ^ sw);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                ah[i] = *(const f16x8 *)(as + i * 16 * BK + ph);
                al[i] = *(const f16x8 *)(as + i * 16 * BK + pl);
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                bh[j] = *(const f16x8 *)(ws + j * 16 * BK + ph);
                bl[j] = *(const f16x8 *)(ws + j * 16 * BK + pl);
            }
#pragma unroll
            for (int t = 0; t < 3; ++t) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        f32x4 &to = t == 1 ? acc[i][j] : acl[i][j];
                        to = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            t == 2 ? bl[j] : bh[j], t == 0 ? al[i] : ah[i], to, 0, 0, 0);
                    }
                if (refill) {
#pragma unroll
                    for (int q = 0; q < NDMA; ++q)
                        if (q * HALF / NDMA == kb * 3 + t) issue_one(NEXT{}, (kt + NS - 1) * BK, q);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    for (int kt = 0; kt < nk; kt += NS) {
        step(kt, S0{});
        if (kt + 1 < nk) step(kt + 1, S1{});
        if constexpr (NS > 2) if (kt + 2 < nk) step(kt + 2, S2{});
        if constexpr (NS > 3) if (kt + 3 < nk) step(kt + 3, S3{});
    }

    // ---- epilogue ----
    // column limit of C; vector stores need aligned rows
    const int limit = PAIRED ? p.n_out : N;
    const bool vec = (p.ldc & 3) == 0 && ((uintptr_t)p.C & 15) == 0;
    auto value = [&](int i, int j) { return (acc[i][j] + acl[i][j]) * rs[i] * wd[j]; };
    constexpr int NBLK = NARROW ? 1 : WTN / 32;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = mw + 16 * i + lr;
        if (m >= M) continue;
        float *crow = p.C + (int64_t)m * p.ldc;
        const float row_scale = 1.f / rs[i];  // of a GELU_MUL output (a power of two)
        if constexpr (PAIRED) {
#pragma unroll
            for (int b = 0; b < NBLK; ++b) {
                const f32x4 x = value(i, 2 * b), y = value(i, 2 * b + 1);
                f32x4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = gelu_tanh(x[r]) * y[r];
                const int n = nw / 2 + 16 * b + 4 * lc;  // output columns n .. n + 3
                if (n < limit) split_store4(crow, n, o);
            }
        } else {
            // block j with its epilogue applied, columns col(j) .. + 3
            auto out = [&](int j) {
                f32x4 v = value(i, j);
                if constexpr (EPI == EPI_GELU_MUL) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        v[r] = gelu_tanh(v[r]) * aux[i][j][r] * row_scale;
                }
                return v;
            };
            if constexpr (!SOUT) {
#pragma unroll
                for (int j = 0; j < TN; ++j) store_run(crow + col(j), out(j), limit - col(j), vec);
            } else if constexpr (NARROW) {
                if (col(0) < limit) split_store4(crow, col(0), out(0));
            } else {
#pragma unroll
                for (int b = 0; b < NBLK; ++b)
                    if (nw + 32 * b < limit)
                        split_store8(crow, nw + 32 * b, lc, out(2 * b), out(2 * b + 1));
            }
        }
    }
#endif
}

// The grouped tile order (RASTER) is taken by outputs of 1280 columns or
// more: 18688 x 2304 x 768 187.1 -> 185.4 us, 6230 x 2304 x 768 72.5 -> 69.7
// us, and one-row launches, whose weights come from HBM, fetch each W panel on
// one XCD (512 x 2304 x 768 16.6 -> 13.6 us). Narrower outputs keep N fastest
// (6230 x 768 x 768 26.5 against 27.2 us, 3000 x 1024 x 4096 75.7 against 79.4).
constexpr int SPLIT_RASTER_MIN_N = 1280;

template <int BM, int BN, int KB, int EPI, int MINB, int NS, int WMW, int WNW>
static hipError_t launch_split_tile(const GemmArgs &a, hipStream_t s) {
    const int tm = (a.M + BM - 1) / BM, tn = (a.N + BN - 1) / BN;
    if (a.N >= SPLIT_RASTER_MIN_N)
        hipLaunchKernelGGL((gemm_split<BM, BN, KB, EPI, MINB, NS, WMW, WNW, true>), dim3(tm * tn),
                           dim3(64 * WMW * WNW), 0, s, a, tm, tn);
    else
        hipLaunchKernelGGL((gemm_split<BM, BN, KB, EPI, MINB, NS, WMW, WNW, false>), dim3(tm * tn),
                           dim3(64 * WMW * WNW), 0, s, a, tm, tn);
    return hipGetLastError();
}

// Tile choice. Every tile gives the same bits, so only time matters (us,
// weights from HBM below 2000 rows):
//  * Grids of at most one small tile per CU are a chain of memory round
//    trips: the smallest tiles with the deepest slices. 32x16 tiles, three
//    1 KB-row slices in flight (128 x 768 x 768: 5.8 us, against 7.5 for
//    32x32 tiles of two waves and 6.1 for 32x32x256 of four), then 32x32
//    (128 x 1280 x 768: 6.2), then 64x64 with 128-wide slices and eight waves
//    (1040 x 768 x 768: 10.1 against 12.9 for four waves).
//  * Up to two 64x64 tiles per CU: 64-wide slices, two workgroups per CU (1040 x
//    1280 x 768: 13.3 against 16.5).
//  * Larger grids: the least work on the busiest CU, ceil(tiles / 256) times
//    the tile's area over its measured rate: 128x128 (two per CU; a count of
//    one runs alone on its CU and an odd count leaves half of it idle) 1,
//    64x128 with the four waves side by side (three per CU) 0.87, 64x64 (four
//    per CU) 0.72, ties to the larger. 18688 x 2304 x 768: 186 us on 128x128,
//    197 on 64x128; 6230 x 768 x 768: 26.5 on 64x128, 28.4 on 128x64, 29.4 on
//    128x128; 3000 x 1024 x 1024: 22.2 on 64x64, 25.0 on 64x128.
// 256x128, 128x256 and 256x256 tiles (one workgroup per CU) were within 3 % or
// slower on every shape swept.
template <int EPI>
static hipError_t launch_split_auto(const GemmArgs &a, hipStream_t s) {
    auto tiles = [&](int bm, int bn) {
        return (int64_t)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
    };
    constexpr bool PAIRED = EPI == EPI_GEGLU;
    const bool k128 = a.K % 128 == 0;
    if (tiles(64, 64) <= 256 && k128) {
        if constexpr (!PAIRED)
            if (tiles(32, 16) <= 256) {
                if (a.K % 256 == 0) return launch_split_tile<32, 16, 8, EPI, 1, 3, 2, 1>(a, s);
                return launch_split_tile<32, 16, 4, EPI, 1, 4, 2, 1>(a, s);
            }
        if (tiles(32, 32) <= 256) {
            if constexpr (PAIRED) {
                if (a.K % 256 == 0) return launch_split_tile<32, 32, 8, EPI, 1, 2, 2, 1>(a, s);
            } else {
                if (a.K % 256 == 0) return launch_split_tile<32, 32, 8, EPI, 1, 2, 2, 2>(a, s);
                return launch_split_tile<32, 32, 4, EPI, 1, 3, 2, 2>(a, s);
            }
        }
        if constexpr (PAIRED) {
            if (tiles(64, 32) <= 256) return launch_split_tile<64, 32, 4, EPI, 1, 3, 4, 1>(a, s);
        } else if (tiles(32, 32) <= 512) {
            return launch_split_tile<32, 32, 4, EPI, 2, 2, 2, 2>(a, s);
        }
        return launch_split_tile<64, 64, 4, EPI, 1, 2, 4, 2>(a, s);
    }
    if (tiles(64, 64) <= 512 && a.K % 64 == 0)
        return launch_split_tile<64, 64, 2, EPI, 2, 2, 2, 2>(a, s);
    auto per_cu = [&](int bm, int bn) { return (double)((tiles(bm, bn) + 255) / 256); };
    const double n128 = per_cu(128, 128);
    const double c128 = (n128 < 2 ? 1.25 : (int)n128 % 2 ? n128 + 0.5 : n128) * (128.0 * 128.0);
    const double c64128 = per_cu(64, 128) * (64.0 * 128.0) / 0.87;
    const double c64 = per_cu(64, 64) * (64.0 * 64.0) / 0.72;
    if (c64 < c128 && c64 < c64128) return launch_split_tile<64, 64, 1, EPI, 4, 2, 2, 2>(a, s);
    if (c64128 < c128) return launch_split_tile<64, 128, 1, EPI, 3, 2, 1, 4>(a, s);
    return launch_split_tile<128, 128, 1, EPI, 2, 2, 2, 2>(a, s);
}

hipError_t launch_gemm_split(const GemmArgs &a, hipStream_t s) {
    if (a.M <= 0 || a.N <= 0) return hipSuccess;
    // buffer offsets are 32-bit: an operand window must stay below 2 GiB
    if (!a.wd || a.K % 32 || a.lda % 4 || a.ldw % 4 || (uintptr_t)a.A % 16 ||
        (uintptr_t)a.W % 16 || (uintptr_t)a.wd % 16 ||
        (int64_t)128 * std::max(a.lda, a.ldw) * 4 >= INT32_MAX)
        return hipErrorInvalidValue;
    switch (a.epi) {
        case EPI_STORE: return launch_split_auto<EPI_STORE>(a, s);
        case EPI_GEGLU: return launch_split_auto<EPI_GEGLU>(a, s);
        case EPI_GELU_MUL: return launch_split_auto<EPI_GELU_MUL>(a, s);
    }
    return hipErrorInvalidValue;
}

// ---- split rows -----------------------------------------------------------------

// One wave per row of w [rows, K], in place: the row times `cols`, scaled by the
// power of two that brings its largest magnitude into [2^13, 2^14). A wave
// reads the 256 values of a pass before it stores their blocks.
//
// A value scaled to 2^-2 or more keeps 22 bits; below that its low half ends in
// the half's denormals, 2^-25 being its error whatever its size. The flag is
// raised where that holds for more than a quarter of a row's nonzero values (a
// spread of 2^16 between most of the row and its largest value; a few small
// values beside many large ones lose nothing a sum would show), or where the
// largest lies outside what the scale's range brings there.
__global__ __launch_bounds__(256) void split_rows_kernel(float *w, int64_t rows, int K,
                                                         const float *__restrict__ cols, float also,
                                                         const float *__restrict__ row_mul,
                                                         float *__restrict__ descale, int *flag) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    float *wr = w + row * K;
    float mx = 0.f;
    bool finite = true;
    for (int k = lane; k < K; k += 64) {
        const float v = cols ? wr[k] * cols[k] : wr[k];
        finite = finite && isfinite(v);
        mx = fmaxf(mx, fabsf(v));
    }
    mx = wave_max(mx);
    const float sc = split_scale_of(mx);
    int small = 0, some = 0;
    for (int k = 4 * lane; k < K; k += 256) {
        f32x4 v = *(const f32x4 *)(wr + k);
        if (cols) v = v * *(const f32x4 *)(cols + k);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[r] *= sc;
            some += v[r] != 0.f;
            small += v[r] != 0.f && fabsf(v[r]) < 0.25f;
        }
        split_store4(wr, k, v);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        some += __shfl_xor(some, o);
        small += __shfl_xor(small, o);
    }
    const bool scaled = mx == 0.f || (mx * sc >= 8192.f && mx * sc < 16384.f);
    if (!finite || !scaled || 4 * small > some) raise_flag(flag, 1);
    if (lane == 0) descale[row] = (row_mul ? also * row_mul[row] : also) / sc;
}

// One wave per row; the squares are summed in double (no overflow or underflow
// of the floats' range).
__global__ __launch_bounds__(256) void row_bounds_kernel(const float *__restrict__ x, int64_t rows,
                                                         int K, const float *__restrict__ w,
                                                         float *__restrict__ out) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    double s = 0.0;
    for (int k = lane; k < K; k += 64) {
        const double v = (double)x[row * K + k] * (w ? (double)w[k] : 1.0);
        s += v * v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) out[row] = (float)(sqrt(s * (double)K) * 1.0005);
}

hipError_t launch_row_bounds(const float *x, int64_t rows, int K, const float *w, float *out,
                             hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(row_bounds_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, x,
                       rows, K, w, out);
    return hipGetLastError();
}

hipError_t launch_split_rows(float *w, int64_t rows, int K, const float *cols, float also,
                             const float *row_mul, float *descale, int *flag, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (K % 32 || (uintptr_t)w % 16 || (uintptr_t)cols % 16) return hipErrorInvalidValue;
    hipLaunchKernelGGL(split_rows_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, w, rows,
                       K, cols, also, row_mul, descale, flag);
    return hipGetLastError();
}

}  // namespace svl
