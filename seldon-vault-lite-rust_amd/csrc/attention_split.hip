// Attention on split operands (dev_common.hpp): the same packed ragged rows,
// work items, masks and online softmax as attn16_kernel (attention.hip), with
// Q, K and V held as pairs of halves and every product taken as three F16
// MFMAs. The Q/K/V norm kernels store split head rows in place; queries carry
// scale * log2(e), so scores come out in log2 units times 1 / qk_descale.
//
// What bounds it: the F16 matrix pipes run a product 2.7 times faster than the
// FP32 MFMA does (gemm_split.hip), so the wave's LDS fragment reads (64 KB of
// K and V per 16 queries and 32 keys at head_dim 256, 2/3 of the matrix time),
// the softmax's vector work and the barriers now weigh as much as the MFMAs.
//
// Per 32-key step (KT keys per tile):
//  * S^T = K . Q^T: the scores' partial sums over 64 dims (two MFMA chains,
//    high products and mixed products, added) fold as a binary tree, whether
//    one wave runs them all (DS = 1) or DS waves of a 16-query group run
//    their dims and meet through LDS; every wave of a group then holds the
//    same bits and runs the same softmax, so a row's result does not depend
//    on the variant its launch takes.
//  * P = 2^(s - m + 6), below 2^14 (the lazily moved reference m is at most 8
//    below a row's maximum), is split in registers: lane (q, g) holds keys
//    4g .. 4g + 3 and 16 + 4g .. 16 + 4g + 3, chunk g of the pair format. Its
//    last bit is 2^-24 of the half range, 2^-30 of the largest probability.
//  * O^T += V^T . P^T: V rows stay row-major in LDS and are read transposed
//    (ds_read_b64_tr_b16: a 16-lane group reads four keys x 16 dims, lane i
//    receiving dim i of each key), four reads per 16-dim tile and 32 keys. A
//    tile's 16 dims are both halves of two chunks, and the V rows' chunks are
//    swizzled so that the four keys of a group lie in different quarters of
//    the banks (with the first halves of four chunks and the K rows' swizzle,
//    conflicts took 36 % of the kernel's cycles, now 13 %). The
//    mixed products run in an accumulator of their own from zero each tile and
//    are added by the vector unit (the MFMA drops small addends' bits
//    downwards, which a sum over thousands of positive weights would keep).
//
// K and V tiles have one LDS buffer each (64 KB per workgroup at head_dim 256,
// two workgroups per CU): V(t) is loaded while the scores of tile t run, K(t+1)
// while the softmax and P.V of tile t run; two barriers per tile.
#include <type_traits>

#include "dev_common.hpp"
#include "svl_internal.hpp"

namespace svl {

typedef __fp16 fp16x4_raw __attribute__((vector_size(8)));

// Chunk swizzle of key r's V row.
__device__ __forceinline__ int v_swizzle(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// Four keys x 16 dims read transposed: `p` is this lane's 8-byte piece (key
// (lane % 16) / 4 of the group's four, piece lane % 4 of its 16 dims); the
// result holds element lane % 16 of the four keys' pieces.
__device__ __forceinline__ f16x4 read_transposed(const char *p) {
    const fp16x4_raw v = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
        (__attribute__((address_space(3))) fp16x4_raw *)p);
    return __builtin_bit_cast(f16x4, v);
}

// Pairwise fold of N (a power of two) values read by at(i).
template <int N, class F>
__device__ __forceinline__ f32x4 fold_tree(F &&at) {
    f32x4 t[N];
#pragma unroll
    for (int i = 0; i < N; ++i) t[i] = at(i);
#pragma unroll
    for (int w = 1; w < N; w *= 2)
#pragma unroll
        for (int i = 0; i < N; i += 2 * w) t[i] = t[i] + t[i + w];
    return t[0];
}

template <int HD, int WAVES, int DS, int KT, int MINB>
__global__ __launch_bounds__(64 * WAVES, MINB) void attn_split_kernel(AttnArgs p, int xcd_chunks) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int HDW = HD / DS;              // head dims per wave
    constexpr int NB = HDW / 32;              // 32-dim blocks per wave
    constexpr int NP = HDW / 64;              // partial sums per wave (64 dims each)
    constexpr int NT = HDW / 16;              // 16-dim output tiles per wave
    constexpr int NKB = KT / 16;              // 16-key blocks per tile
    constexpr int VPW = 16 * WAVES / DS;      // query vectors per workgroup
    constexpr int SPLIT = 128 / VPW;          // workgroups per 128-vector work item
    constexpr int NDMA = KT * HD / 256 / WAVES;  // 1 KB DMA instructions per operand and wave
    static_assert(HD % (64 * DS) == 0 && (NP & (NP - 1)) == 0 && (DS & (DS - 1)) == 0, "partial sums");
    static_assert(WAVES % DS == 0 && 128 % VPW == 0, "vector groups");
    static_assert(KT % 32 == 0 && NDMA >= 1 && (KT * HD / 256) % WAVES == 0, "key tile");
    __shared__ float Ks[KT * HD];
    __shared__ float Vs[KT * HD];
    __shared__ f32x4 Sx[DS > 1 ? WAVES * NKB * 64 : 1];  // the waves' partial scores

    const int wg = xcd_chunks ? xcd_chunk((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
    const AttnTile tile = p.tiles[wg / SPLIT];
    const int G = p.nh / p.nkv;
    const int lane = threadIdx.x & 63, wave = uniform((int)threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int dpart = DS > 1 ? wave % DS : 0, group = wave / DS;
    const int nvec = tile.len * G;
    const int vbase = tile.qv0 + (wg % SPLIT) * VPW;
    if (vbase >= nvec) return;   // the whole workgroup: a part past the row's vectors
    const int v = vbase + group * 16 + l16;
    const bool vvalid = v < nvec;
    const int vq = vvalid ? v : nvec - 1;
    const int qpos = vq / G;
    const int qhead = tile.kvh * G + (vq - qpos * G);

    // query fragments: chunk g of each 32-dim block, high and low halves
    const float *qrow = p.q + (int64_t)(tile.tok0 + qpos) * p.ldq + qhead * HD + dpart * HDW;
    f16x8 qh[NB], ql[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        qh[b] = *(const f16x8 *)(qrow + 32 * b + 4 * g);
        ql[b] = *(const f16x8 *)(qrow + 32 * b + 16 + 4 * g);
    }

    f32x4 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_ref = -INFINITY, l_run = 0.f;
    const float descale = p.qk_descale;

    const int v_last = min(vbase + VPW, nvec) - 1;
    const int p_lo = vbase / G, p_hi = v_last / G;
    int k_lo = 0, k_hi = tile.len - 1;
    if (p.window >= 0) {
        k_lo = max(0, p_lo - p.window);
        k_hi = min(tile.len - 1, p_hi + p.window);
    }
    const int k_first = (k_lo / KT) * KT;
    const int n_tiles = (k_hi - k_first) / KT + 1;

    // Buffer windows over this row's keys of this KV head; keys past the row
    // end fall outside them and read as zero. The rows' 16-byte chunks are
    // XOR-swizzled by key % 16 (V: v_swizzle of it) on the way into LDS.
    const int ldk = (int)p.ldk, ldv = (int)p.ldv;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(p.k + (int64_t)tile.tok0 * p.ldk + tile.kvh * HD), (short)0,
        ((tile.len - 1) * ldk + HD) * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(p.v + (int64_t)tile.tok0 * p.ldv + tile.kvh * HD), (short)0,
        ((tile.len - 1) * ldv + HD) * 4, 0x00020000);
    int koff[NDMA], voff[NDMA];
#pragma unroll
    for (int q = 0; q < NDMA; ++q) {
        const int e = (wave * NDMA + q) * 256 + 4 * lane;
        const int r = e / HD, slot = (e % HD) / 4;
        koff[q] = (r * ldk + 4 * (slot ^ (r & 15))) * 4;
        voff[q] = (r * ldv + 4 * (slot ^ v_swizzle(r & 15))) * 4;
    }
    auto issue_k = [&](int k0) {
#pragma unroll
        for (int q = 0; q < NDMA; ++q)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rk, (__attribute__((address_space(3))) void *)&Ks[(wave * NDMA + q) * 256], 16,
                koff[q] + k0 * ldk * 4, 0, 0, 0);
    };
    auto issue_v = [&](int k0) {
#pragma unroll
        for (int q = 0; q < NDMA; ++q)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rv, (__attribute__((address_space(3))) void *)&Vs[(wave * NDMA + q) * 256], 16,
                voff[q] + k0 * ldv * 4, 0, 0, 0);
    };

    issue_k(k_first);
    wait_vmcnt<0>();
    __syncthreads();
    // Fragment addresses: the swizzles move a chunk within its group of 16, so
    // block b reads at the address of its parity plus a constant (an address
    // per block would take 48 registers and spill).
    const char *ks[2][2], *vs[2][2][2];  // [block parity][tile of the block][high, low]
    {
        const int c0 = dpart * (HDW / 4);  // first 16-byte chunk of the wave's dims
        const int kr = 4 * g + (l16 >> 2), j = l16 & 3, vz = v_swizzle(kr);
#pragma unroll
        for (int pb = 0; pb < 2; ++pb)
#pragma unroll
            for (int hl = 0; hl < 2; ++hl) {
                ks[pb][hl] = (const char *)(Ks + l16 * HD) +
                             16 * (c0 + ((8 * pb + 4 * hl + g) ^ l16));
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    vs[pb][e][hl] = (const char *)(Vs + kr * HD) + (j & 1) * 8 +
                                    16 * (c0 + ((8 * pb + 4 * hl + 2 * e + (j >> 1)) ^ vz));
            }
    }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int it = 0; it < n_tiles; ++it) {
        const int k0 = k_first + it * KT;
        issue_v(k0);  // every wave is past P.V of tile it - 1

        // S^T for keys 16 kb + 4 g + r (register r of block kb), query l16
        f32x4 s[NKB];
        {
            f32x4 part[NP][NKB];
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                f32x4 hh[NKB], mx[NKB];
#pragma unroll
                for (int b = 2 * q; b < 2 * q + 2; ++b) {
                    const int at = 128 * (b & ~1);
                    f16x8 kh[NKB], kl[NKB];
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) {
                        kh[kb] = *(const f16x8 *)(ks[b & 1][0] + at + kb * 64 * HD);
                        kl[kb] = *(const f16x8 *)(ks[b & 1][1] + at + kb * 64 * HD);
                    }
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb)
                        mx[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            kh[kb], ql[b], b == 2 * q ? zero : mx[kb], 0, 0, 0);
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb)
                        hh[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            kh[kb], qh[b], b == 2 * q ? zero : hh[kb], 0, 0, 0);
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb)
                        mx[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl[kb], qh[b], mx[kb], 0, 0, 0);
                }
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb) part[q][kb] = hh[kb] + mx[kb];
            }
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
                s[kb] = fold_tree<NP>([&](int i) { return part[i][kb]; });
        }
        if constexpr (DS > 1) {
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb) Sx[(wave * NKB + kb) * 64 + lane] = s[kb];
        }
        wait_vmcnt<0>();   // this wave's part of V(it) has landed
        __syncthreads();   // ... and every wave's; no wave reads K(it) any more
        if (it + 1 < n_tiles) issue_k(k0 + KT);
        if constexpr (DS > 1) {
            const int w0 = group * DS;
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
                s[kb] = fold_tree<DS>([&](int i) { return Sx[((w0 + i) * NKB + kb) * 64 + lane]; });
        }

        // masks only on the row-tail tile and on tiles that cross a
        // sliding-window edge of some query of the block
        const bool tail = k0 + KT > tile.len;
        const bool edge = p.window >= 0 && (k0 < p_hi - p.window || k0 + KT - 1 > p_lo + p.window);
        if (tail || edge) {
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = k0 + kb * 16 + 4 * g + r;
                    const int dist = qpos > key ? qpos - key : key - qpos;
                    const bool ok = (key < tile.len) & ((p.window < 0) | (dist <= p.window));
                    s[kb][r] = ok ? s[kb][r] : -INFINITY;
                }
        }
        float tmax = s[0][0];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, s[kb][r]);
        tmax = fold_xor16_32_max(tmax) * descale;
        // lazy rescale: the reference only moves when a query's max grows by
        // more than RESCALE_LOG2
        const bool grow = tmax > m_ref + RESCALE_LOG2;
        if (__ballot(grow)) {
            const float m_new = grow ? tmax : m_ref;
            const float alpha = m_ref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_ref - m_new);
            l_run *= alpha;
#pragma unroll
            for (int t = 0; t < NT; ++t) o[t] = o[t] * alpha;
            m_ref = m_new;
        }
        const float base = ATTN_P_LOG2 - m_ref;
        f16x8 ph[KT / 32], pl[KT / 32];
        float psum = 0.f;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
            f32x4 pr;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pr[r] = s[kb][r] == -INFINITY
                            ? 0.f
                            : __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], descale, base));
                psum += pr[r];
            }
            f16x4 hi, lo;
            split4(pr, hi, lo);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                ph[kb / 2][4 * (kb & 1) + r] = hi[r];
                pl[kb / 2][4 * (kb & 1) + r] = lo[r];
            }
        }
        l_run += fold_xor16_32_sum(psum);

        // O^T += V^T P^T: tile t = 2 b + e takes chunks 2e and 2e + 1 of 32-dim
        // block b, whose row 4 q .. 4 q + 3 (register r of lane group q) is
        // dims 32 b + 8 e + 4 (q / 2) + 16 (q % 2) + r
        {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int b = t >> 1;
                const char *ph0 = vs[b & 1][t & 1][0] + 128 * (b & ~1);
                const char *pl0 = vs[b & 1][t & 1][1] + 128 * (b & ~1);
                f32x4 mx = zero;
#pragma unroll
                for (int u = 0; u < KT / 32; ++u) {
                    const int k0b = 128 * u * HD, k1b = k0b + 64 * HD;  // keys 32 u and 32 u + 16
                    const f16x8 vh = __builtin_shufflevector(
                        read_transposed(ph0 + k0b), read_transposed(ph0 + k1b), 0, 1, 2, 3, 4, 5, 6, 7);
                    const f16x8 vl = __builtin_shufflevector(
                        read_transposed(pl0 + k0b), read_transposed(pl0 + k1b), 0, 1, 2, 3, 4, 5, 6, 7);
                    mx = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, ph[u], mx, 0, 0, 0);
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ph[u], o[t], 0, 0, 0);
                    mx = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, pl[u], mx, 0, 0, 0);
                }
                o[t] = o[t] + mx;
            }
        }
        wait_vmcnt<0>();   // this wave's part of K(it + 1) has landed
        __syncthreads();   // ... and every wave's; no wave reads V(it) or Sx any more
    }

    if (vvalid) {
        const float inv = p.out_scale * p.v_descale / l_run;
        float *orow = p.out + (int64_t)(tile.tok0 + qpos) * p.ldo;
        const int ocol = qhead * HD + dpart * HDW;
        bool ok = isfinite(inv);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const f32x4 y = o[t] * inv;
            ok = ok && finite4(y);
            split_store4(orow, ocol + 32 * (t >> 1) + 8 * (t & 1) + 4 * (g >> 1) + 16 * (g & 1), y);
        }
        if (!ok) raise_flag(p.flag, FLAG_NONFINITE);
    }
#endif
}

template <int HD, int WAVES, int DS, int KT, int MINB>
static hipError_t launch_attn_split(const AttnArgs &a, hipStream_t s) {
    constexpr int SPLIT = 128 * DS / (16 * WAVES);
    const int chunks = a.window >= 0 && a.shortest > a.window + 1;
    hipLaunchKernelGGL((attn_split_kernel<HD, WAVES, DS, KT, MINB>),
                       dim3((unsigned)(SPLIT * a.n_tiles)), dim3(64 * WAVES), 0, s, a, chunks);
    return hipGetLastError();
}

bool attention_takes_split(int hd, int64_t ld, int64_t max_len) {
    return get_attention_path() == ATTN_PATH_AUTO && (hd == 64 || hd == 256 || hd == 512) &&
           (max_len + 64) * std::max(ld, (int64_t)hd) * 4 < INT32_MAX;
}

// Up to 64 work items (a few rows of a few hundred tokens), every 16-query
// group takes HD / 64 waves, which fill at most the 512 two-per-CU slots once;
// larger grids run 64 queries per workgroup.
hipError_t launch_attention_split(const AttnArgs &a, hipStream_t s) {
    if (a.tokens <= 0 || a.n_tiles <= 0) return hipSuccess;
    if (!(a.out_scale > 0.f)) return hipErrorInvalidValue;
    const bool small = 8 * (int64_t)a.n_tiles <= 512;
    switch (a.hd) {
        case 64:
            if (2 * (int64_t)a.n_tiles >= 256) return launch_attn_split<64, 4, 1, 64, 3>(a, s);
            if (4 * (int64_t)a.n_tiles >= 256) return launch_attn_split<64, 2, 1, 64, 1>(a, s);
            return launch_attn_split<64, 1, 1, 64, 1>(a, s);
        case 256:
            if (small) return launch_attn_split<256, 4, 4, 32, 1>(a, s);
            return launch_attn_split<256, 4, 1, 32, 2>(a, s);
        case 512:
            if (small) return launch_attn_split<512, 8, 8, 32, 1>(a, s);
            return launch_attn_split<512, 8, 2, 32, 1>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace svl
