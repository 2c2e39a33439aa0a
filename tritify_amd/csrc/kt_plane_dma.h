// The 3 x 3 digit-plane product (12-trit operands, the planes of kt_hip_pack_planes) fed by LDS DMA: the same sums,
// epilogue and split-k hand-off as plane_gemm_kernel, for the shapes plane_dma_shape picks.
//
// What bounds it: nine int8 MFMAs per 32 x 32 x 32 block. Staged through registers one k-tile ahead behind a barrier a
// tile, the general kernel waits on memory: 9 bytes a clock and CU where the L2 gives several times that. Here every
// operand byte goes from memory to a ring of NS stages by DMA, NS - 1 k-tiles ahead, the DMAs are issued between the
// MFMAs, and the epilogue stores through a descriptor over the tile's rows (one add per output, no 64-bit address or
// branch; 7 us of the 57 at 4096 x 1792 were that code). A CTA of 4 waves leaves room for two per CU, so one's
// epilogue runs under the other's products. Measured (us, general kernel -> this):
//   4096 x 1792, k 448    57.2 -> 44.3   64 x 128 tiles (8.9 a k-tile at first, 3.07 in the steady state: 2.75 POPS;
//                                        the 58.7 MB of sums alone take 12)
//   4096 x 448, k 1792    50.7 -> 36.9   64 x 64
//   512 x 4864, k 896     36.4 -> 28.4   64 x 64
//   256 x 1152, k 896     16.3 ->  8.4   32 x 64
//   256 x 896, k 4864             25     32 x 64, k over 2 CTAs (29.0 whole)
//   64 x 2816, k 2048     22.5 -> 15.2   32 x 64
// 128 x 128 tiles (8 waves, one CTA per CU) measured 47.5, 43.9 and 27.1 on the first three, 8 waves over the two
// halves of each k-tile of a 64 x 128 tile 62.2, 38.0 and 38.0: a CTA alone on its CU hides neither end of its tile.
#pragma once

#include "kt_w12_core.h"

namespace kt {

// CTA = WM x WN x KW waves: WM row tiles of 32, WN column blocks of 32 WTN, and KW = 2 (WTN = 1) gives each half of the
// waves one k32 half of every k-tile (their sums meet in LDS at the end).
template <int WM_, int WN_, int WTN_, int KW_, int NS_>
struct PlaneTile {
    static constexpr int WM = WM_, WN = WN_, WTN = WTN_, KW = KW_, NS = NS_;
    static constexpr int W = WM * WN * KW, NT = 64 * W, BM = 32 * WM, BN = 32 * WN * WTN;
    // DMA units of 16 rows x 64 bytes of one plane, A's planes first; a stage holds them in this order
    static constexpr int UA = 3 * BM / 16, UNITS = 3 * (BM + BN) / 16;
    static constexpr int UPW = UNITS / W, REM = UNITS % W;  // whole units per wave; the rest as one half unit per wave
    static constexpr int ND = UPW + (REM ? 1 : 0);          // DMAs per wave and k-tile, the same on every wave
    static constexpr int STAGE = 1024 * UNITS, LDS = NS * STAGE;
    static_assert(REM == 0 || REM * 2 == W, "the units left over make one half unit per wave");
    static_assert(KW == 1 || (WTN == 1 && LDS >= NT * 16 * 4), "the exchange of the k halves fits the ring");
    static_assert(NS >= 2 && ND * (NS - 2) <= 63, "vmcnt holds the DMAs of NS - 2 later tiles");
};
typedef PlaneTile<2, 2, 2, 1, 2> PlaneTile128;  // 64 x 128
typedef PlaneTile<2, 2, 1, 1, 3> PlaneTile64;   // 64 x 64
typedef PlaneTile<1, 2, 1, 2, 4> PlaneTile32;   // 32 x 64
static_assert(PlaneTile128::LDS == 73728 && PlaneTile64::LDS == 73728 && PlaneTile32::LDS == 73728, "two CTAs per CU");

template <class C>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void plane_dma_kernel(
    const int8_t* __restrict__ xa, const int8_t* __restrict__ wb, int64_t* __restrict__ y, int M, int N, int kp, int k0,
    int k1, int accumulate, int drop_top, const int64_t* __restrict__ ql_bias, QlState* ql_all,
    unsigned* __restrict__ tile_cnt, QlSeg seg) {
    constexpr int BM = C::BM, BN = C::BN, WTN = C::WTN, NS = C::NS, KW = C::KW, ND = C::ND, W = C::W;
    extern __shared__ __attribute__((aligned(16))) int8_t ring[];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // numbered as plane_gemm_kernel's tiles: a contiguous run per XCD, row tile fastest
    const int kw = KW == 2 ? w & 1 : 0, wt = KW == 2 ? w >> 1 : w, wn = wt % C::WN, wm = wt / C::WN;
    const int tiles_n = (N + BN - 1) / BN, tiles_m = (int)gridDim.x / tiles_n;
    const int nt = (int)gridDim.x, q8 = nt >> 3, r8 = nt & 7, xcd = (int)blockIdx.x & 7;
    const int t = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + ((int)blockIdx.x >> 3);
    const int m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
    QlState* ql = ql_all ? ql_all + ql_seg_of(seg, n0) : nullptr;  // this tile's call
    const size_t xplane = (size_t)M * kp, wplane = (size_t)N * kp;

    // this CTA's run of k-tiles: [kb, kb + 64 nk), nk >= 1 by the launcher's choice of gridDim.y
    const int nk_all = (k1 - k0) / 64, per = (nk_all + (int)gridDim.y - 1) / (int)gridDim.y;
    const int kb = k0 + (int)blockIdx.y * per * 64;
    const int nk = nk_all - (int)blockIdx.y * per < per ? nk_all - (int)blockIdx.y * per : per;

    // DMA unit u: lane l lands at row l / 4 of its 16 rows, chunk position l % 4, and fetches chunk (l % 4) ^ swz(row).
    // Rows past the matrix are past the descriptor and read as zero.
    auto unit_rsrc = [&](int u) {
        const bool isa = u < C::UA;
        const int ub = isa ? u : u - C::UA, p = isa ? ub / (BM / 16) : ub / (BN / 16);
        const int r0 = isa ? m0 + 16 * (ub % (BM / 16)) : n0 + 16 * (ub % (BN / 16)), left = (isa ? M : N) - r0;
        const int rows = left < 0 ? 0 : (left < 16 ? left : 16);
        const uint64_t b = reinterpret_cast<uint64_t>(isa ? xa + p * xplane : wb + p * wplane) +
                           (rows > 0 ? (uint64_t)r0 * (uint64_t)kp : 0);
        // the descriptor in scalar registers: left to itself the compiler forms it in vector ones and wraps every DMA
        // in a readfirstlane loop
        const uint32_t bl = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
        const uint32_t bh = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
        return make_rsrc(reinterpret_cast<const void*>(((uint64_t)bh << 32) | bl),
                         (uint32_t)__builtin_amdgcn_readfirstlane(rows * kp));
    };
    __amdgpu_buffer_rsrc_t rs[ND];
#pragma unroll
    for (int i = 0; i < C::UPW; i++) rs[i] = unit_rsrc(w + W * i);
    const uint32_t vo = (uint32_t)(lane >> 2) * (uint32_t)kp + 16u * ((lane & 3) ^ ((lane >> 4) & 3));
    uint32_t vh = 0;
    if constexpr (C::REM != 0) {  // half unit: rows 8 h .. 8 h + 7, lanes 0 .. 31
        rs[ND - 1] = unit_rsrc(W * C::UPW + (w >> 1));
        const int r = 8 * (w & 1) + ((lane & 31) >> 2);
        vh = (uint32_t)r * (uint32_t)kp + 16u * ((lane & 3) ^ ((r >> 2) & 3));
    }
    auto issue = [&](int st, int kt) {  // k-tile kt (past the end: the last once more, never consumed) into stage st
        const uint32_t ko = (uint32_t)(kb + 64 * (kt < nk ? kt : nk - 1));
        int8_t* s = ring + st * C::STAGE;
#pragma unroll
        for (int i = 0; i < C::UPW; i++) dma16(rs[i], s + 1024 * (w + W * i), vo, ko);
        if constexpr (C::REM != 0)
            if (lane < 32) dma16(rs[ND - 1], s + 1024 * (W * C::UPW) + 512 * w, vh, ko);
    };
    // the next tile has landed once at most the DMAs of the NS - 2 tiles after it are outstanding, and every wave's
    // reads of the last one are done: after the barrier its stage takes the tile NS further on
    auto wait_tile = [&]() {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(ND * (NS - 2)) : "memory");
    };
    struct Frag {
        v4i a[3], b[3][WTN];
    };
    auto load = [&](int st, int ks, Frag& f) {
        const int8_t* s = ring + st * C::STAGE;
#pragma unroll
        for (int p = 0; p < 3; p++) {
            f.a[p] = lds_read16(s + p * BM * 64, lds_off<4>(32 * wm + (lane & 31), 2 * ks + half));
#pragma unroll
            for (int j = 0; j < WTN; j++)
                f.b[p][j] = lds_read16(s + 3 * BM * 64 + p * BN * 64,
                                       lds_off<4>(32 * (WTN * wn + j) + (lane & 31), 2 * ks + half));
        }
    };
    v16i acc[5][WTN];
#pragma unroll
    for (int g = 0; g < 5; g++)
#pragma unroll
        for (int j = 0; j < WTN; j++) acc[g][j] = v16i{};
    auto mma = [&](const Frag& f) {
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int q = 0; q < 3; q++)
#pragma unroll
                for (int j = 0; j < WTN; j++) acc[p + q][j] = mfma32(f.a[p], f.b[q][j], acc[p + q][j]);
    };
    constexpr int MPD = 9 * WTN / ND;  // MFMAs per DMA of a step
    auto mix = [&]() {
        if constexpr (MPD >= 1)
#pragma unroll
            for (int q = 0; q < ND; q++) {
                __builtin_amdgcn_sched_group_barrier(0x008, MPD, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < NS - 1; i++) issue(i, i);
    wait_tile();
    issue(NS - 1, NS - 1);
    // ping-pong: the fragments of the next half (KW = 1) or tile (KW = 2) are read under the MFMAs of the last
    Frag f0, f1;
    if constexpr (KW == 1) {
        load(0, 0, f0);
        load(0, 1, f1);
        int cs = 0;  // kt % NS
        for (int kt = 0; kt < nk; kt++) {
            const int ns = cs + 1 == NS ? 0 : cs + 1;
            mma(f0);
            wait_tile();
            load(ns, 0, f0);
            __builtin_amdgcn_sched_barrier(0);
            issue(cs, kt + NS);
            mma(f1);
            mix();
            load(ns, 1, f1);
            cs = ns;
        }
    } else {
        load(0, kw, f0);
        int cs = 0;
        for (int kt = 0; kt < nk; kt += 2) {
            int ns = cs + 1 == NS ? 0 : cs + 1;
            wait_tile();
            load(ns, kw, f1);
            __builtin_amdgcn_sched_barrier(0);
            issue(cs, kt + NS);
            mma(f0);
            mix();
            cs = ns;
            if (kt + 1 < nk) {
                ns = cs + 1 == NS ? 0 : cs + 1;
                wait_tile();
                load(ns, kw, f0);
                __builtin_amdgcn_sched_barrier(0);
                issue(cs, kt + 1 + NS);
                mma(f1);
                mix();
                cs = ns;
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the ring is free

    // outputs of the wave: index o = 16 j + r; with KW == 2 (WTN = 1) wave kw keeps half kw of them
    constexpr int NO = 16 * WTN / KW;
    auto val = [&](int j, int r) {
        uint64_t v = 0;
#pragma unroll
        for (int g = 0; g < 5; g++)
            if (!(drop_top && g == 4)) v += (uint64_t)(int64_t)acc[g][j][r] << (8 * g);
        return v;
    };
    uint64_t f[NO];
    if constexpr (KW == 1) {
#pragma unroll
        for (int o = 0; o < NO; o++) f[o] = val(o >> 4, o & 15);
    } else {
        uint64_t* ex = reinterpret_cast<uint64_t*>(ring);
#pragma unroll
        for (int o = 0; o < NO; o++) {
            const uint64_t v0 = val(0, o), v1 = val(0, o + NO);
            f[o] = kw ? v1 : v0;
            ex[(w * NO + o) * 64 + lane] = kw ? v0 : v1;
        }
        __syncthreads();
#pragma unroll
        for (int o = 0; o < NO; o++) f[o] += ex[((w ^ 1) * NO + o) * 64 + lane];
    }
    const int ob = KW == 2 ? kw * NO : 0;  // this wave's first output
    // the tile's rows of y as a buffer: rows past M fall past its end, columns past N get an offset past every buffer
    const int rows_y = M - m0 < BM ? M - m0 : BM;
    const __amdgpu_buffer_rsrc_t rY = make_rsrc(y + (size_t)m0 * N, (uint32_t)rows_y * (uint32_t)N * 8u);
    const bool badd = ql && ql_bias && ql->mode == 0;
    uint32_t vy[WTN];  // the byte offset of output row 0 of each column block
    uint64_t bc[WTN];
#pragma unroll
    for (int j = 0; j < WTN; j++) {
        const int n = n0 + 32 * (WTN * wn + j) + (lane & 31);
        vy[j] = n < N ? (uint32_t)(32 * wm + 4 * half) * (uint32_t)N * 8u + (uint32_t)n * 8u : KT_OOB;
        bc[j] = badd && n < N ? (uint64_t)scale_apply(ql->f_mant, ql->f_shift, ql_bias[n]) : 0;
    }
    auto at = [&](int o) {  // byte offset of output o; a column past N stays past the end (its rows' offsets saturate)
        const int r = (ob + o) & 15;
        const uint32_t b = vy[o >> 4];
        return b == KT_OOB ? KT_OOB : b + (uint32_t)(8 * (r >> 2) + (r & 3)) * (uint32_t)N * 8u;
    };
    auto bias_of = [&](int o) { return bc[o >> 4]; };
    int64_t lmax = 0;
    auto raise = [&](uint64_t v) {
        const int64_t a = (int64_t)v < 0 ? (int64_t)(0 - v) : (int64_t)v;  // i64::abs, wrapping
        lmax = a > lmax ? a : lmax;
    };
    if (gridDim.y > 1) {  // partial sums into y; the tile's last CTA goes on (the hand-off of plane_gemm_kernel)
        auto valid = [&](int o, size_t& i) {
            const int r = (ob + o) & 15, m = m0 + 32 * wm + 8 * (r >> 2) + 4 * half + (r & 3);
            const int n = n0 + 32 * (WTN * wn + (o >> 4)) + (lane & 31);
            i = (size_t)m * N + n;
            return m < M && n < N;
        };
        size_t i;
#pragma unroll
        for (int o = 0; o < NO; o++)
            if (valid(o, i)) atomicAdd(reinterpret_cast<unsigned long long*>(y + i), (unsigned long long)f[o]);
        if (!split_last(&tile_cnt[blockIdx.x])) return;
#pragma unroll
        for (int o = 0; o < NO; o++)
            if (valid(o, i)) {
                const uint64_t b = bias_of(o);
                uint64_t v = __hip_atomic_load(reinterpret_cast<uint64_t*>(y + i), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                v += b;
                raise(v);
                if (b != 0) y[i] = (int64_t)v;
            }
    } else {
        if (accumulate) {
#pragma unroll
            for (int o = 0; o < NO; o++) {
                const v2i p = bload8(rY, at(o), 0);
                f[o] += ((uint64_t)(uint32_t)p.y << 32) | (uint32_t)p.x;
            }
        }
        if (ql) {
            const bool row_ok = rows_y == BM;
#pragma unroll
            for (int o = 0; o < NO; o++) {
                f[o] += bias_of(o);
                const int r = (ob + o) & 15;
                // rows and columns past the matrix hold a bias at most: not outputs
                if (at(o) != KT_OOB && (row_ok || 32 * wm + 8 * (r >> 2) + 4 * half + (r & 3) < rows_y)) raise(f[o]);
            }
        }
#pragma unroll
        for (int o = 0; o < NO; o++)
            __builtin_amdgcn_raw_buffer_store_b64(v2i{(int)(uint32_t)f[o], (int)(uint32_t)(f[o] >> 32)}, rY, at(o), 0,
                                                  0);
    }
    if (ql) {  // the CTA's largest |result| into the call's maximum
        __shared__ int64_t s_max[W];
        lmax = wave_max_i64(lmax);
        if (lane == 0) s_max[w] = lmax;
        __syncthreads();
        if (tid == 0) {
            int64_t b = s_max[0];
            for (int q = 1; q < W; q++) b = s_max[q] > b ? s_max[q] : b;
            if (b > 0) ql_raise_ymax(ql, b);
        }
    }
}

}  // namespace kt
