// The reference decoder's own layers on the device, at the reference's integer semantics: activations are i32 codes
// at the 2^28 level with one kt-int Scale per tensor (a kt_hip_qscale record in device memory), every op closes
// with requant_dyn to that level by its own largest magnitude, and scales compose with kt-int's integer Scale
// arithmetic (kt_scale_dev.h). With kt_hip_quant_linear for every projection they run DecoderModel::decode_step
// (crates/01-engine/kt-core/src/model.rs:290-294, 338-353) with no host round trip:
//
//   rd_embed           Embedding::lookup of a token read from device memory              (layers.rs:1127-1140)
//   rd_rmsnorm         RmsNorm::forward_int                                                (layers.rs:392-434)
//   rd_add             add, the residual add                                               (layers.rs:121-136)
//   rd_swiglu          SwiGluMlp::forward_int between the gate/up and down products       (layers.rs:615-637)
//   rd_attention_step  Attention::decode_step between the q/k/v and o products:           (attention.rs:358-458)
//                      RoPE, the KV cache append with per-step scales, the integer-code
//                      softmax at a common score scale, the heads brought to one scale
//   rd_argmax          argmax_codes, the greedy choice, with an optional per-step record  (generate.rs:48-56)
//   rd_gelu            apply_gelu, SAM's GELU by its CodeLut (many CTAs: a whole image's  (kt-model-vision/src/
//                      tokens)                                                             nonlin.rs:30-45)
//
// Each kernel is one CTA of 1024 threads (one token's tensors are at most a few thousand values); the Scale
// arithmetic of a tensor runs in one thread, the per-element work in all of them. The offline tables
// (CodeLut::build, the RoPE Scales, Scale::from_f64) are built on the host with the C library's f64 functions, as
// the reference builds them with its platform's.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <type_traits>

#include "kt_dpp.h"
#include "kt_kernels.h"
#include "kt_scale_dev.h"
#include "kt_w12_core.h"

namespace kt {

namespace {

constexpr int RD_THREADS = 1024;
constexpr int RD_WAVES = RD_THREADS / 64;
constexpr int RD_MAX_ROWS = 1024;  // RMSNorm rows in one call (one factor per thread)
constexpr int RD_PV_GROUP = 8;     // P.V by kv head for groups of up to this many q heads
constexpr int64_t ACT_LEVELS = 1LL << 28;

}  // namespace

// A QuantLinear output left as its exact sums by the one-row product (kt_hip_quant_linear_multi_sums), as the op
// reading it next takes it: the output's sums, its call's state (max |x|, c, mode) and where its record goes (or
// null). That op applies requant_dyn (layers.rs:33-39, 321-327) as ql_requant_kernel would: ymax = max |sum| over
// the output (i64::abs, wrapping, as the product's own maximum); codes requant_dyn(sum, 2^28, ymax) when the mode is
// 0 and ymax > 0, else zeros (x all zero, or c zero; the path carries no bias); the Scale from_ratio(ymax, 2^28) * c.
struct RqSums {
    const int64_t* acc;
    const QlState* st;
    kt_hip_qscale* rec;
};

// The arguments of rd_attention_step_kernel (kt_hip_ref_attention_step).
struct RdAttn {
    const int32_t *q, *k, *v;
    const kt_hip_qscale *qs, *ks, *vs;
    const int32_t* pos;
    int nh, nkv, hd, max_seq;
    int32_t *kc, *vc;                  // [max_seq][nkv * hd]
    kt_hip_sscale *kscale, *vscale;    // [max_seq]
    const kt_hip_sscale *cos, *sin;    // [max_seq][hd / 2]
    int64_t isq_mant;
    int32_t isq_shift;
    const int64_t* exp_codes;
    kt_hip_codelut exp;
    int32_t* o;
    kt_hip_qscale* os;
    unsigned char* ws;                 // the heads kernels' workspace (rd_heads_layout), or null: the one-CTA kernel
    int hb;                            // the one-CTA kernel: heads whose scores LDS holds at once
    int sums;                          // the heads kernels: q, k, v as the product's sums (qsum, ksum, vsum)
    RqSums qsum, ksum, vsum;
};

// Attention::forward_int over a sequence (prefill): the inputs, the tables and the workspace parts.
struct RdPrefill {
    const int32_t *q, *k, *v;          // T x nh*hd, T x nkv*hd, T x nkv*hd
    const kt_hip_qscale *qs, *ks, *vs;
    int T, nh, nkv, hd;
    const kt_hip_sscale *cos, *sin;    // [max_seq][hd / 2]
    int64_t isq_mant;
    int32_t isq_shift;
    const int64_t* exp_codes;
    kt_hip_codelut exp;
    int32_t *qd, *kd;                  // rotated q and k
    int64_t* hout;                     // [T][nh][hd]: the sums of numerator * v
    int64_t* hmax;                     // [T][nh]: each (row, head)'s largest |sum of numerator * v|
    Sc* fac;                           // [T][nh]: each (row, head)'s scale
    uint64_t* gmax;                    // the largest |output| at the common scale
    Sc* common;
    int32_t* o;                        // T x nh*hd
    kt_hip_qscale* os;
};

namespace {

__device__ inline Sc rec_sc(const kt_hip_qscale* r) { return Sc{r->mant, r->shift}; }
__device__ inline void put_rec(kt_hip_qscale* r, Sc s) {
    kt_hip_qscale o{};
    o.mant = s.mant, o.shift = s.shift;
    *r = o;
}
__device__ inline int64_t iabs(int64_t v) { return v < 0 ? (int64_t)(0 - (uint64_t)v) : v; }
// |v|, INT64_MAX for INT64_MIN
__device__ inline int64_t magnitude(int64_t v) { return v == INT64_MIN ? INT64_MAX : iabs(v); }
__device__ inline int64_t wmul(int64_t a, int64_t b) { return (int64_t)((uint64_t)a * (uint64_t)b); }
__device__ inline int64_t wadd(int64_t a, int64_t b) { return (int64_t)((uint64_t)a + (uint64_t)b); }

// Lane 0's value as a wave-uniform one (scalar registers). The one-thread Scale chains run in all lanes of wave 0 on
// such values, so their integer arithmetic is scalar and their branches are uniform, rather than per-lane code under
// a one-lane exec mask.
__device__ inline int64_t uni64(int64_t v) { return (int64_t)lane64((uint64_t)v, 0); }
__device__ inline Sc uni(Sc s) { return Sc{uni64(s.mant), __builtin_amdgcn_readlane(s.shift, 0)}; }
__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }
// Block-wide reductions over the CTA's 1024 threads; every thread gets the result: each wave's result to LDS, one
// barrier, the 16 of them reduced in row 0 of every wave.
__device__ int64_t block_max_i64(int64_t v, int64_t* red) {
    v = wave_max_i64(v);
    const int lane = threadIdx.x & 63;
    if (lane == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = (int64_t)lane64((uint64_t)row_max_i64(lane < RD_WAVES ? red[lane] : INT64_MIN), 0);
    __syncthreads();
    return v;
}
// The same reductions for CTAs of 256 threads (4 waves).
__device__ int64_t block_max_4w(int64_t v, int64_t* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int64_t u = __shfl_xor(v, o, 64);
        v = u > v ? u : v;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
    for (int w = 1; w < 4; w++) v = red[w] > v ? red[w] : v;
    __syncthreads();
    return v;
}
__device__ int64_t block_sum_4w(int64_t v, int64_t* red) {  // wrapping
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = wadd(v, __shfl_xor(v, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
    for (int w = 1; w < 4; w++) v = wadd(v, red[w]);
    __syncthreads();
    return v;
}

// Block maxima of two or three values at once (one pair of barriers); red holds 3 x RD_WAVES values.
template <int K>
__device__ void block_max_k(int64_t (&v)[K], int64_t* red) {
#pragma unroll
    for (int k = 0; k < K; k++) {
        v[k] = wave_max_i64(v[k]);
        if ((threadIdx.x & 63) == 0) red[k * RD_WAVES + (threadIdx.x >> 6)] = v[k];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < K; k++)
        v[k] = (int64_t)lane64((uint64_t)row_max_i64(lane < RD_WAVES ? red[k * RD_WAVES + lane] : INT64_MIN), 0);
    __syncthreads();
}

// requant_dyn of a sums output (RqSums): whether its codes are live, the Scale, the record as ql_requant_kernel
// writes it.
__device__ inline bool rqs_live(const QlState* st, int64_t ymax) { return st->mode == 0 && ymax > 0; }
__device__ inline Sc rqs_scale(const QlState* st, int64_t ymax) {
    return rqs_live(st, ymax) ? sc_mul(from_ratio((u128)(uint64_t)ymax, (u128)ACT_LEVELS), Sc{st->c_mant, st->c_shift})
                              : Sc{0, 0};
}
// rqs_scale with the state's fields read as wave-uniform values (wave 0's scalar chains)
__device__ inline Sc rqs_scale_u(const QlState* st, int64_t ymax) {
    const int mode = __builtin_amdgcn_readfirstlane(st->mode);
    const Sc c = uni(Sc{st->c_mant, st->c_shift});
    return mode == 0 && ymax > 0 ? sc_mul(from_ratio((u128)(uint64_t)ymax, (u128)ACT_LEVELS), c) : Sc{0, 0};
}
__device__ inline void rqs_record(const RqSums& r, int64_t ymax, Sc s) {
    if (!r.rec) return;
    kt_hip_qscale o{};
    o.xmax = r.st->xmax;
    if (rqs_live(r.st, ymax)) o.mant = s.mant, o.shift = s.shift, o.ymax = ymax;
    *r.rec = o;
}

// The engine's largest-scale fold (|a, b| if b.ge(a) { b } else { a } from Scale::ZERO, in sequence order) as a
// parallel reduction: of equal values the one latest in the sequence wins, as in the fold. idx < 0: no element.
struct ScIdx {
    Sc s;
    int idx;
};
__device__ inline ScIdx sc_pick(ScIdx a, ScIdx b) {
    if (a.idx < 0) return b;
    if (b.idx < 0) return a;
    const bool ab = sc_ge(a.s, b.s), ba = sc_ge(b.s, a.s);
    if (ab && ba) return a.idx > b.idx ? a : b;
    return ba ? b : a;
}
// The fold's total order as a key of three words per item: each Scale normalized exactly to m * 2^e with m's top bit
// set (e = -shift - clz(mant) lies in [-2^31 - 63, 2^31], stored as e + 2^40 > 0), so comparing values (sc_ge) is
// comparing (e, m) as integers, and the index breaks ties (the fold's later-wins rule). The third word holds the
// index above the item's clz, which the order then ignores (indices are distinct) and from which the winner's own
// (mant, shift) comes back exactly: mant = m >> clz, shift = -e - clz. A dead item (idx < 0 or a zero Scale) is the
// key (0, 0, 0), below every live one.
struct FoldKey {
    uint64_t e, m, i;
};
__device__ inline FoldKey fold_key(const ScIdx& v) {
    const bool live = v.idx >= 0 && v.s.mant != 0;
    const uint64_t a = (uint64_t)v.s.mant;
    const int lz = live ? __builtin_clzll(a) : 0;
    return live ? FoldKey{(uint64_t)(-(int64_t)v.s.shift - lz + (1LL << 40)), a << lz,
                          ((uint64_t)(uint32_t)v.idx << 6) | (uint64_t)lz}
                : FoldKey{0, 0, 0};
}
__device__ inline ScIdx fold_item(const FoldKey& k) {
    if (k.e == 0) return ScIdx{Sc{0, 0}, -1};
    const int lz = (int)(k.i & 63);
    return ScIdx{Sc{(int64_t)(k.m >> lz), (int32_t)(-((int64_t)k.e - (1LL << 40)) - lz)}, (int)(k.i >> 6)};
}
__device__ inline bool fold_gt(const FoldKey& x, const FoldKey& y) {
    return x.e != y.e ? x.e > y.e : (x.m != y.m ? x.m > y.m : x.i > y.i);
}
template <int CTRL>
__device__ inline void fold_dpp(FoldKey& k) {
    const FoldKey u{dpp64<CTRL>(k.e), dpp64<CTRL>(k.m), dpp64<CTRL>(k.i)};
    if (fold_gt(u, k)) k = u;
}
__device__ inline void fold_row(FoldKey& k) {
    fold_dpp<DPP_XOR1>(k);
    fold_dpp<DPP_XOR2>(k);
    fold_dpp<DPP_HALF_MIRROR>(k);
    fold_dpp<DPP_MIRROR>(k);
}
__device__ inline FoldKey fold_lane(const FoldKey& k, int l) { return FoldKey{lane64(k.e, l), lane64(k.m, l), lane64(k.i, l)}; }
// The engine's fold over K sequences at once, one item per thread for each, in two halves: each wave's largest key by
// DPP steps into red (at least 3 K RD_WAVES words), ending with a barrier; then, on any whole wave, sequence q's
// winner (its own Scale and index) out of the waves' keys. A wave without a live item writes dead keys at once, and a
// caller lets only the waves that use a winner form it: four waves a SIMD would otherwise repeat those steps.
template <int K>
__device__ void fold_waves(const ScIdx (&v)[K], ScIdx* red) {
    uint64_t* r64 = reinterpret_cast<uint64_t*>(red);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    FoldKey k[K] = {};
    bool live = false;
#pragma unroll
    for (int q = 0; q < K; q++) live = live || v[q].idx >= 0;
    if (__ballot(live) != 0) {  // uniform
#pragma unroll
        for (int q = 0; q < K; q++) {
            k[q] = fold_key(v[q]);
            fold_row(k[q]);
            FoldKey b = fold_lane(k[q], 0);
#pragma unroll
            for (int l = 16; l < 64; l += 16) {
                const FoldKey c = fold_lane(k[q], l);
                if (fold_gt(c, b)) b = c;
            }
            k[q] = b;
        }
    }
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < K; q++) {
            uint64_t* d = r64 + (q * RD_WAVES + w) * 3;
            d[0] = k[q].e, d[1] = k[q].m, d[2] = k[q].i;
        }
    __syncthreads();
}
__device__ inline ScIdx fold_winner(int q, const ScIdx* red) {
    const uint64_t* r64 = reinterpret_cast<const uint64_t*>(red);
    const int lane = threadIdx.x & 63;
    FoldKey b{0, 0, 0};
    if (lane < RD_WAVES) {
        const uint64_t* d = r64 + (q * RD_WAVES + lane) * 3;
        b = FoldKey{d[0], d[1], d[2]};
    }
    fold_row(b);
    return fold_item(fold_lane(b, 0));
}
// Both halves, the winners in every thread. Ends with a barrier.
template <int K>
__device__ void block_fold_max_k(ScIdx (&v)[K], ScIdx* red) {
    fold_waves<K>(v, red);
#pragma unroll
    for (int q = 0; q < K; q++) v[q] = fold_winner(q, red);
    __syncthreads();
}
// n: how many leading threads hold items (the rest hold idx -1); every thread of the CTA calls it. Ends with a
// barrier.
__device__ ScIdx block_fold_max(ScIdx v, ScIdx* red, int n) {
    (void)n;
    ScIdx a[1] = {v};
    block_fold_max_k<1>(a, red);
    return a[0];
}

// CodeLut::index / code_at (kt-int/src/lib.rs:382-395) with the call's factor m = scale * inv_step.
__device__ inline int64_t lut_index(Sc m, int64_t data, int64_t lo_index) { return sc_apply(m, data) - lo_index; }
// the same for an i32 code, in 64-bit arithmetic where sc_apply32 allows
__device__ inline int64_t lut_index32(Sc m, int32_t data, int64_t lo_index) { return sc_apply32(m, data) - lo_index; }
__device__ inline int64_t lut_code(const int64_t* codes, int n, int64_t idx) {
    return codes[idx < 0 ? 0 : (idx > n - 1 ? n - 1 : idx)];
}

}  // namespace

// Embedding::lookup (layers.rs:1127-1140): y = the token's code row at the table's scale. A token outside
// [0, vocab) gives zeros at Scale::ZERO (the reference panics there; a kernel must not read out of bounds).
__global__ __launch_bounds__(RD_THREADS) void rd_embed_kernel(const int32_t* __restrict__ emb, int64_t e_mant,
                                                              int32_t e_shift, const int32_t* __restrict__ token,
                                                              int vocab, int dim, int32_t* __restrict__ y,
                                                              kt_hip_qscale* __restrict__ ys) {
    const int t = *token;
    const bool ok = t >= 0 && t < vocab;
    for (int i = threadIdx.x; i < dim; i += RD_THREADS) y[i] = ok ? emb[(size_t)t * dim + i] : 0;
    if (threadIdx.x == 0) put_rec(ys, ok ? Sc{e_mant, e_shift} : Sc{0, 0});
}

// RmsNorm::forward_int of one row held in registers (NV values per thread, value i = threadIdx.x + RD_THREADS * k,
// dim <= RD_THREADS * NV; gv the gammas likewise): the exact sum of squares reduced across the CTA, the row factor
// c = xs * rsqrt(mean_sq + eps) * gs by thread 0 (only thread 0 reads xs), the products brought to c and
// requantized by their largest magnitude. The same integers as rd_rmsnorm_kernel's general path for one row.
template <int NV>
__device__ void rd_norm_row(int32_t (&xv)[NV], const int32_t (&gv)[NV], int dim, Sc xs, Sc gs, Sc eps,
                            int32_t* __restrict__ y, kt_hip_qscale* __restrict__ ys, int64_t* red) {
    __shared__ uint64_t sq2[RD_WAVES][2];
    __shared__ Sc cf[2];  // c and its factor over itself
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint64_t hi = 0, lo = 0;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        if ((int)threadIdx.x + RD_THREADS * k >= dim) xv[k] = 0;
        const int64_t v = xv[k];
        const uint64_t sq = (uint64_t)(v * v), t = lo + sq;
        hi += t < lo, lo = t;
    }
    add128_row(hi, lo);
    {  // the four rows' sums
        u128 w = 0;
#pragma unroll
        for (int l = 0; l < 64; l += 16) w += ((u128)lane64(hi, l) << 64) | lane64(lo, l);
        hi = (uint64_t)(w >> 64), lo = (uint64_t)w;
    }
    if (lane == 0) sq2[wave][0] = hi, sq2[wave][1] = lo;
    __syncthreads();
    const int wv = wave_id();
    Sc cc{0, 0};  // wave 0: the row factor (uniform)
    if (wv == 0) {  // the 16 waves' sums (lane q < 16 reads wave q's), then the row factor's chain on scalars
        uint64_t h2 = lane < RD_WAVES ? sq2[lane][0] : 0, l2 = lane < RD_WAVES ? sq2[lane][1] : 0;
        add128_row(h2, l2);
        const u128 ss = ((u128)lane64(h2, 0) << 64) | lane64(l2, 0);
        const Sc xu = uni(xs);
        const Sc mean_sq = sc_mul(sc_mul(from_ratio(ss, (u128)dim), xu), xu);
        const Sc denom = sc_add(mean_sq, eps);
        const Sc inv = denom.mant == 0 ? Sc{0, 0} : sc_rsqrt(denom);
        cc = sc_mul(sc_mul(xu, inv), gs);  // the largest of one row's factors is that factor
        const Sc f = cc.mant != 0 ? sc_mul(cc, sc_recip(cc)) : Sc{0, 0};
        if (lane == 0) cf[0] = cc, cf[1] = f;
    }
    __syncthreads();
    const Sc f0 = cf[1];
    if (wv != 0) cc = cf[0];
    int64_t hv[NV];
    int64_t m = 0;
#pragma unroll
    for (int k = 0; k < NV; k++) {  // values past dim stay 0 (whole waves skip the 128-bit products)
        hv[k] = 0;
        if (cc.mant != 0 && (int)threadIdx.x + RD_THREADS * k < dim)
            hv[k] = sc_apply(f0, (int64_t)xv[k] * (int64_t)gv[k]);
        m = iabs(hv[k]) > m ? iabs(hv[k]) : m;
    }
    const int64_t gmax = block_max_i64(m, red);
    const RqDen rd_gmax = rq_den(gmax);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int i = threadIdx.x + RD_THREADS * k;
        if (i < dim) y[i] = gmax == 0 ? 0 : rq_apply(rd_gmax, hv[k]);
    }
    if (wv == 0) {
        const Sc r = gmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), cc);
        if (lane == 0) put_rec(ys, r);
    }
}

// RmsNorm::forward_int (layers.rs:392-434) over `rows` rows of `dim`: per row the exact sum of squares, its
// mean-square Scale plus eps, the integer inverse square root, the row factor c_r = xs * inv * gs; the products
// x_i * g_i brought to the largest c_r and requantized by the largest magnitude.
__global__ __launch_bounds__(RD_THREADS) void rd_rmsnorm_kernel(const int32_t* __restrict__ x, int rows, int dim,
                                                                const kt_hip_qscale* __restrict__ xs_rec,
                                                                const int32_t* __restrict__ g, int64_t g_mant,
                                                                int32_t g_shift, int64_t e_mant, int32_t e_shift,
                                                                int32_t* __restrict__ y,
                                                                kt_hip_qscale* __restrict__ ys) {
    __shared__ int64_t red[RD_WAVES];
    __shared__ Sc crow[RD_MAX_ROWS], frow[RD_MAX_ROWS];
    __shared__ ScIdx redsc[RD_THREADS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const Sc xs = rec_sc(xs_rec), gs{g_mant, g_shift}, eps{e_mant, e_shift};
    constexpr int RD_NV = 8;
    if (rows == 1 && dim <= RD_THREADS * RD_NV) {
        // one row (the decode step): its values and gammas loaded once by every thread, all in flight together
        int32_t xv[RD_NV], gv[RD_NV];
#pragma unroll
        for (int k = 0; k < RD_NV; k++) {
            const int i = threadIdx.x + RD_THREADS * k, ic = i < dim ? i : dim - 1;
            xv[k] = x[ic], gv[k] = g[ic];
        }
        rd_norm_row<RD_NV>(xv, gv, dim, xs, gs, eps, y, ys, red);
        return;
    }
    // each row's exact sum of squares by one wave, its factor c_r = xs * rsqrt(mean_sq + eps) * gs by that wave's
    // first lane (the rows' Scale arithmetic runs side by side)
    for (int r = wave; r < rows; r += RD_WAVES) {
        uint64_t hi = 0, lo = 0;  // the u128 sum as two words: squares below 2^62, at most 2^26 of them per lane
        for (int i = lane; i < dim; i += 64) {
            const int64_t v = x[(size_t)r * dim + i];
            const uint64_t sq = (uint64_t)(v * v), t = lo + sq;
            hi += t < lo, lo = t;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const uint64_t ohi = __shfl_xor(hi, o, 64), olo = __shfl_xor(lo, o, 64), t = lo + olo;
            hi += ohi + (t < lo), lo = t;
        }
        if (lane == 0) {
            const u128 ss = ((u128)hi << 64) | lo;
            const Sc mean_sq = sc_mul(sc_mul(from_ratio(ss, (u128)dim), xs), xs);
            const Sc denom = sc_add(mean_sq, eps);
            const Sc inv = denom.mant == 0 ? Sc{0, 0} : sc_rsqrt(denom);
            crow[r] = sc_mul(sc_mul(xs, inv), gs);
        }
    }
    __syncthreads();
    // the largest row factor by the engine's fold (of equal values the latest row's), then each row's share of it
    ScIdx best{Sc{0, 0}, -1};
    for (int r = threadIdx.x; r < rows; r += RD_THREADS) best = sc_pick(best, ScIdx{crow[r], r});
    const Sc cc = block_fold_max(best, redsc, rows).s;
    if (cc.mant != 0) {
        const Sc cinv = sc_recip(cc);  // every thread: one Scale reciprocal, no extra barrier
        for (int r = threadIdx.x; r < rows; r += RD_THREADS) frow[r] = sc_mul(crow[r], cinv);
    }
    __syncthreads();
    const int n = rows * dim;
    int64_t m = 0;
    if (cc.mant != 0)
        for (int i = threadIdx.x; i < n; i += RD_THREADS) {
            const int64_t v = sc_apply(frow[i / dim], (int64_t)x[i] * (int64_t)g[i % dim]);
            m = iabs(v) > m ? iabs(v) : m;
        }
    const int64_t gmax = block_max_i64(m, red);
    const RqDen rd_gmax = rq_den(gmax);
    for (int i = threadIdx.x; i < n; i += RD_THREADS)
        y[i] = gmax == 0 ? 0 : rq_apply(rd_gmax, sc_apply(frow[i / dim], (int64_t)x[i] * (int64_t)g[i % dim]));
    if (threadIdx.x == 0)
        put_rec(ys, gmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), cc));
}

// add (layers.rs:121-136): both to the larger scale, summed, requantized. y may alias a or b.
__global__ __launch_bounds__(RD_THREADS) void rd_add_kernel(const int32_t* a, const kt_hip_qscale* as_rec,
                                                            const int32_t* b, const kt_hip_qscale* bs_rec, int n,
                                                            int32_t* y, kt_hip_qscale* ys) {
    __shared__ int64_t red[RD_WAVES];
    __shared__ Sc par[3];  // common, fa, fb
    // up to RD_AV values per thread held in registers, their loads issued before the Scale work of thread 0 so that
    // the two overlap; longer tensors read a and b twice
    constexpr int RD_AV = 4;
    const bool held = n <= RD_THREADS * RD_AV;
    int32_t av[RD_AV], bv[RD_AV];
    if (held) {
#pragma unroll
        for (int k = 0; k < RD_AV; k++) {
            const int i = threadIdx.x + RD_THREADS * k, ic = i < n ? i : n - 1;
            av[k] = a[ic], bv[k] = b[ic];
        }
    }
    if (threadIdx.x == 0) {
        const Sc as = rec_sc(as_rec), bs = rec_sc(bs_rec);
        const Sc common = sc_ge(as, bs) ? as : bs;
        par[0] = common;
        if (common.mant != 0) {
            const Sc cinv = sc_recip(common);
            par[1] = sc_mul(as, cinv), par[2] = sc_mul(bs, cinv);
        }
    }
    __syncthreads();
    const Sc common = par[0], fa = par[1], fb = par[2];
    int64_t m = 0, hv[RD_AV];
    if (held) {
#pragma unroll
        for (int k = 0; k < RD_AV; k++) {  // values past n stay 0 (whole waves skip them)
            hv[k] = 0;
            if (common.mant != 0 && (int)threadIdx.x + RD_THREADS * k < n)
                hv[k] = wadd(sc_apply32(fa, av[k]), sc_apply32(fb, bv[k]));
            m = iabs(hv[k]) > m ? iabs(hv[k]) : m;
        }
    } else if (common.mant != 0) {
        for (int i = threadIdx.x; i < n; i += RD_THREADS) {
            const int64_t v = wadd(sc_apply32(fa, a[i]), sc_apply32(fb, b[i]));
            m = iabs(v) > m ? iabs(v) : m;
        }
    }
    const int64_t gmax = block_max_i64(m, red);  // every read of a, b, and their records, is done past here
    const RqDen rd_gmax = rq_den(gmax);
    if (held) {
#pragma unroll
        for (int k = 0; k < RD_AV; k++) {
            const int i = threadIdx.x + RD_THREADS * k;
            if (i < n) y[i] = gmax == 0 ? 0 : rq_apply(rd_gmax, hv[k]);
        }
    } else {
        for (int i = threadIdx.x; i < n; i += RD_THREADS)
            y[i] = gmax == 0 ? 0 : rq_apply(rd_gmax, wadd(sc_apply32(fa, a[i]), sc_apply32(fb, b[i])));
    }
    if (threadIdx.x == 0)
        put_rec(ys, gmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), common));
}

// add (layers.rs:121-136) and then RmsNorm::forward_int (layers.rs:392-434) of the sum, for one row of
// n <= RD_THREADS * RD_AN values: the decode step's residual add followed by the next norm (model.rs:338-353), one
// launch where the two kernels took two. y = add(a, b) with its record ys (y may alias a or b), then h = the norm of
// y from the codes still in registers and the Scale thread 0 formed for ys. The same integers as rd_add_kernel and
// rd_rmsnorm_kernel in sequence. SUMS: b is a QuantLinear's sums (bsum), its requant_dyn and record formed here
// first, as ql_requant_kernel would.
// NV: the values a thread holds, 1 or RD_AN: the values past n cost what the others do (a row of 896 in 4 a
// thread: 13.0 us, in 1: 10.4).
constexpr int RD_AN = 4;
template <bool SUMS, int NV>
__global__ __launch_bounds__(RD_THREADS) void rd_add_norm_kernel(const int32_t* a, const kt_hip_qscale* as_rec,
                                                                 const int32_t* b, const kt_hip_qscale* bs_rec,
                                                                 RqSums bsum, int n, int32_t* y, kt_hip_qscale* ys,
                                                                 const int32_t* __restrict__ g, int64_t g_mant,
                                                                 int32_t g_shift, int64_t e_mant, int32_t e_shift,
                                                                 int32_t* __restrict__ h,
                                                                 kt_hip_qscale* __restrict__ hs) {
    __shared__ int64_t red[RD_WAVES];
    __shared__ Sc par[3];  // common, fa, fb
    int32_t av[NV], bv[NV], gv[NV];
    int64_t bacc[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int i = threadIdx.x + RD_THREADS * k, ic = i < n ? i : n - 1;
        av[k] = a[ic], gv[k] = g[ic];
        if constexpr (SUMS) bacc[k] = bsum.acc[ic];
        else bv[k] = b[ic];
    }
    int64_t bmax = 0;
    if constexpr (SUMS) {  // b's maximum (the values past n repeat value n - 1), codes and Scale
#pragma unroll
        for (int k = 0; k < NV; k++) bmax = iabs(bacc[k]) > bmax ? iabs(bacc[k]) : bmax;
        bmax = block_max_i64(bmax, red);
        const bool live = rqs_live(bsum.st, bmax);
        const RqDen d = rq_den(bmax);
#pragma unroll
        for (int k = 0; k < NV; k++) bv[k] = live ? rq_apply(d, bacc[k]) : 0;
    }
    const int wv = wave_id(), lane = threadIdx.x & 63;
    Sc common{0, 0};  // wave 0: the common Scale (uniform)
    if (wv == 0) {  // the Scale chain on scalars
        Sc bs;
        if constexpr (SUMS) {
            bs = rqs_scale_u(bsum.st, bmax);
            if (lane == 0) rqs_record(bsum, bmax, bs);
        } else {
            bs = uni(rec_sc(bs_rec));
        }
        const Sc as = uni(rec_sc(as_rec));
        common = sc_ge(as, bs) ? as : bs;
        Sc fa{0, 0}, fb{0, 0};
        if (common.mant != 0) {
            const Sc cinv = sc_recip(common);
            fa = sc_mul(as, cinv), fb = sc_mul(bs, cinv);
        }
        if (lane == 0) par[0] = common, par[1] = fa, par[2] = fb;
    }
    __syncthreads();
    const Sc fa = par[1], fb = par[2];
    if (wv != 0) common = par[0];
    int64_t m = 0, hv[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        hv[k] = 0;
        if (common.mant != 0 && (int)threadIdx.x + RD_THREADS * k < n)
            hv[k] = wadd(sc_apply32(fa, av[k]), sc_apply32(fb, bv[k]));
        m = iabs(hv[k]) > m ? iabs(hv[k]) : m;
    }
    const int64_t gmax = block_max_i64(m, red);  // every read of a and b is done past here
    const RqDen rd_gmax = rq_den(gmax);
    int32_t yv[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int i = threadIdx.x + RD_THREADS * k;
        yv[k] = gmax == 0 ? 0 : rq_apply(rd_gmax, hv[k]);
        if (i < n) y[i] = yv[k];
    }
    Sc xs{0, 0};  // the sum's Scale: wave 0 writes the record and carries it into the norm
    if (wv == 0) {
        xs = gmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), common);
        if (lane == 0) put_rec(ys, xs);
    }
    rd_norm_row<NV>(yv, gv, n, xs, Sc{g_mant, g_shift}, Sc{e_mant, e_shift}, h, hs, red);
}

// SwiGluMlp::forward_int's activation (layers.rs:615-637): h = silu_code(g) * u, the SiLU code from the CodeLut at
// g's scale (0 below the table, the identity tail g * gs / code_scale above it), requantized at code_scale * us.
// One CTA per row: row r's n values with its own records gs_rec[r], us_rec[r], hs[r] (rows = 1: one tensor).
// SUMS (one row, n <= RD_THREADS * RD_VPT): g and u are QuantLinear sums (gsum, usum), their requant_dyn and records
// formed here first, as ql_requant_kernel would.
template <bool SUMS>
__global__ __launch_bounds__(RD_THREADS) void rd_swiglu_kernel(const int32_t* __restrict__ g,
                                                               const kt_hip_qscale* __restrict__ gs_rec,
                                                               const int32_t* __restrict__ u,
                                                               const kt_hip_qscale* __restrict__ us_rec, RqSums gsum,
                                                               RqSums usum, int n, const int64_t* __restrict__ codes,
                                                               kt_hip_codelut L, int32_t* __restrict__ h,
                                                               kt_hip_qscale* __restrict__ hs) {
    __shared__ int64_t red[3 * RD_WAVES];
    if constexpr (!SUMS) {
        const int64_t r = blockIdx.x;
        g += r * n, u += r * n, h += r * n, gs_rec += r, us_rec += r, hs += r;
    }
    // up to RD_VPT values per thread formed once and held in registers, their loads issued before thread 0's Scale
    // work so that the two overlap (the table reads follow the factors); longer rows form each value twice
    constexpr int RD_VPT = 8;
    const bool held = SUMS || n <= RD_THREADS * RD_VPT;
    int32_t gd[RD_VPT], ud[RD_VPT];
    int64_t gmax = 0, umax = 0;
    if constexpr (SUMS) {  // the sums, their maxima (the values past n repeat value n - 1), codes and Scales
        int64_t ga[RD_VPT], ua[RD_VPT];
#pragma unroll
        for (int i = 0; i < RD_VPT; i++) {
            const int k = threadIdx.x + RD_THREADS * i, kk = k < n ? k : n - 1;
            ga[i] = gsum.acc[kk], ua[i] = usum.acc[kk];
        }
        int64_t mx[2] = {0, 0};
#pragma unroll
        for (int i = 0; i < RD_VPT; i++) {
            mx[0] = iabs(ga[i]) > mx[0] ? iabs(ga[i]) : mx[0];
            mx[1] = iabs(ua[i]) > mx[1] ? iabs(ua[i]) : mx[1];
        }
        block_max_k<2>(mx, red);
        gmax = mx[0], umax = mx[1];
        const bool lg = rqs_live(gsum.st, gmax), lu = rqs_live(usum.st, umax);
        const RqDen dg = rq_den(gmax), du = rq_den(umax);
#pragma unroll
        for (int i = 0; i < RD_VPT; i++) {
            gd[i] = lg ? rq_apply(dg, ga[i]) : 0;
            ud[i] = lu ? rq_apply(du, ua[i]) : 0;
        }
    } else if (held) {
#pragma unroll
        for (int i = 0; i < RD_VPT; i++) {
            const int k = threadIdx.x + RD_THREADS * i, kk = k < n ? k : n - 1;
            gd[i] = g[kk], ud[i] = u[kk];
        }
    }
    __shared__ Sc par[3];  // index factor, identity factor, h scale
    const Sc cs{L.code_mant, L.code_shift};
    if (threadIdx.x == 0) {  // g's factors (and with SUMS its Scale and record first)
        Sc gs;
        if constexpr (SUMS) {
            gs = rqs_scale(gsum.st, gmax);
            rqs_record(gsum, gmax, gs);
        } else {
            gs = rec_sc(gs_rec);
        }
        par[0] = sc_mul(gs, Sc{L.inv_mant, L.inv_shift});
        par[1] = sc_mul(gs, sc_recip(cs));
    }
    if (threadIdx.x == 64) {  // u's side, in another wave
        Sc us;
        if constexpr (SUMS) {
            us = rqs_scale(usum.st, umax);
            rqs_record(usum, umax, us);
        } else {
            us = rec_sc(us_rec);
        }
        par[2] = sc_mul(cs, us);
    }
    __syncthreads();
    const Sc mi = par[0], idf = par[1], hsc = par[2];
    auto act = [&](int k) -> int64_t {
        const int32_t gk = g[k];
        const int64_t idx = lut_index32(mi, gk, L.lo_index);
        const int64_t code = idx < 0 ? 0 : (idx >= L.n ? sc_apply32(idf, gk) : lut_code(codes, L.n, idx));
        return wmul(code, u[k]);
    };
    int64_t hv[RD_VPT];
    int64_t m = 0;
    if (held) {
#pragma unroll
        for (int i = 0; i < RD_VPT; i++) {  // values past n stay 0 (whole waves skip them)
            hv[i] = 0;
            if ((int)threadIdx.x + RD_THREADS * i < n) {
                const int64_t idx = lut_index32(mi, gd[i], L.lo_index);
                const int64_t code = idx < 0 ? 0 : (idx >= L.n ? sc_apply32(idf, gd[i]) : lut_code(codes, L.n, idx));
                hv[i] = wmul(code, ud[i]);
            }
            m = iabs(hv[i]) > m ? iabs(hv[i]) : m;
        }
    } else {
        for (int k = threadIdx.x; k < n; k += RD_THREADS) {
            const int64_t a = iabs(act(k));
            m = a > m ? a : m;
        }
    }
    const int64_t hmax = block_max_i64(m, red);
    const RqDen rd_hmax = rq_den(hmax);
    if (held) {
#pragma unroll
        for (int i = 0; i < RD_VPT; i++) {
            const int k = threadIdx.x + RD_THREADS * i;
            if (k < n) h[k] = hmax == 0 ? 0 : rq_apply(rd_hmax, hv[i]);
        }
    } else {
        for (int k = threadIdx.x; k < n; k += RD_THREADS) h[k] = hmax == 0 ? 0 : rq_apply(rd_hmax, act(k));
    }
    if (threadIdx.x == 0)
        put_rec(hs, hmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)hmax, (u128)ACT_LEVELS), hsc));
}

// The same activation of one row with g and u as sums, spread over the chip and left at its products for the down
// projection (ql_skinny_kernel's HV form), whose CTAs requantize them: a CTA of 256 threads takes 256 values, the maxima
// of g and u from the product's slots (one per CTA of 8 columns there) rather than from all the sums, and writes its
// values' products, their largest magnitude (part[blockIdx.x]) and, CTA 0, the Scale they are at and g's and u's records.
// One CTA for the row (above) forms two requantizations, a table read and a third requantization of 5 values a thread on
// one CU: 13.8 us and 8.7 for the down product at 4864 values; here 5.6 and 9.1, the step of 2 layers 236 -> 220.
constexpr int RD_SPLIT = 256;
__global__ __launch_bounds__(RD_SPLIT) void rd_swiglu_split_kernel(RqSums gsum, RqSums usum,
                                                                   const int64_t* __restrict__ gpart,
                                                                   const int64_t* __restrict__ upart, int nparts, int n,
                                                                   const int64_t* __restrict__ codes, kt_hip_codelut L,
                                                                   int64_t* __restrict__ hv, int64_t* __restrict__ part,
                                                                   kt_hip_qscale* __restrict__ scale) {
    constexpr int NW = RD_SPLIT / 64;
    __shared__ int64_t red[2][NW], hred[NW];
    __shared__ Sc par[3];  // index factor, identity factor, h scale
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
    const int i = (int)blockIdx.x * RD_SPLIT + tid, ii = i < n ? i : n - 1;
    const int64_t ga = gsum.acc[ii], ua = usum.acc[ii];
    int64_t gmax = 0, umax = 0;  // the slots hold no negative value
    for (int q = tid; q < nparts; q += RD_SPLIT) {
        gmax = gpart[q] > gmax ? gpart[q] : gmax;
        umax = upart[q] > umax ? upart[q] : umax;
    }
    gmax = wave_max_i64(gmax), umax = wave_max_i64(umax);
    if (lane == 0) red[0][wv] = gmax, red[1][wv] = umax;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; w++) {
        gmax = red[0][w] > gmax ? red[0][w] : gmax;
        umax = red[1][w] > umax ? red[1][w] : umax;
    }
    const Sc cs{L.code_mant, L.code_shift};
    if (wv == 0) {  // g's factors (its Scale first)
        const Sc gs = rqs_scale_u(gsum.st, uni64(gmax));
        const Sc mi = sc_mul(gs, Sc{L.inv_mant, L.inv_shift}), idf = sc_mul(gs, sc_recip(cs));
        if (lane == 0) {
            par[0] = mi, par[1] = idf;
            if (blockIdx.x == 0) rqs_record(gsum, gmax, gs);
        }
    } else if (wv == 1) {  // u's side
        const Sc us = rqs_scale_u(usum.st, uni64(umax));
        const Sc hs = sc_mul(cs, us);
        if (lane == 0) {
            par[2] = hs;
            if (blockIdx.x == 0) rqs_record(usum, umax, us), put_rec(scale, hs);
        }
    }
    const int32_t gd = rqs_live(gsum.st, gmax) ? rq_apply(rq_den(gmax), ga) : 0;
    const int32_t ud = rqs_live(usum.st, umax) ? rq_apply(rq_den(umax), ua) : 0;
    __syncthreads();
    int64_t h = 0;
    if (i < n) {
        const int64_t idx = lut_index32(par[0], gd, L.lo_index);
        h = wmul(idx < 0 ? 0 : (idx >= L.n ? sc_apply32(par[1], gd) : lut_code(codes, L.n, idx)), ud);
        hv[i] = h;
    }
    const int64_t m = wave_max_i64(iabs(h));
    if (lane == 0) hred[wv] = m;
    __syncthreads();
    if (tid == 0) {
        int64_t b = 0;  // as the one-CTA kernel's maximum: from 0
#pragma unroll
        for (int w = 0; w < NW; w++) b = hred[w] > b ? hred[w] : b;
        part[blockIdx.x] = b;
    }
}

// apply_gelu (kt-model-vision/src/nonlin.rs:30-45): each code through the GELU CodeLut at x's scale (0 below the
// table, the identity factor xs / code_scale above it), cast to i32, the output at the table's code scale with no
// requantization. Grid-stride over n; each CTA forms the two factors from the record.
__global__ __launch_bounds__(RD_THREADS) void rd_gelu_kernel(const int32_t* __restrict__ x,
                                                             const kt_hip_qscale* __restrict__ xs_rec, int64_t n,
                                                             const int64_t* __restrict__ codes, kt_hip_codelut L,
                                                             int32_t* __restrict__ y,
                                                             kt_hip_qscale* __restrict__ ys) {
    __shared__ Sc par[2];  // index factor, identity factor
    const Sc cs{L.code_mant, L.code_shift};
    if (threadIdx.x == 0) {
        const Sc xs = rec_sc(xs_rec);
        par[0] = sc_mul(xs, Sc{L.inv_mant, L.inv_shift});
        par[1] = sc_mul(xs, sc_recip(cs));
    }
    __syncthreads();
    const Sc mi = par[0], idf = par[1];
    const int64_t step = (int64_t)gridDim.x * RD_THREADS;
    for (int64_t i = (int64_t)blockIdx.x * RD_THREADS + threadIdx.x; i < n; i += step) {
        const int32_t d = x[i];
        const int64_t idx = lut_index32(mi, d, L.lo_index);
        const int64_t code = idx < 0 ? 0 : (idx >= L.n ? sc_apply32(idf, d) : lut_code(codes, L.n, idx));
        y[i] = (int32_t)code;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) put_rec(ys, cs);
}

// Attention::decode_step between its projections (attention.rs:358-458), at the position *pos:
//  1. RoPE (rope_int, attention.rs:222-246) of every q head into LDS and every k head into the cache row pos; v
//     into its cache row; this step's k and v scales into the per-step scale arrays;
//  2. v_ref = the largest v scale over the steps 0..pos, vf_j = vs_j / v_ref; the score scales
//     s_j = qs * ks_j * inv_sqrt, s_ref = the largest, f_j = s_j / s_ref;
//  3. per head: score_j = f_j.apply(q . k_j), ec_j = exp_code(score_j - max score) at s_ref (0 below the table),
//     sumc = sum ec_j, out_d = sum_j ec_j * vf_j.apply(v_jd), scale_h = v_ref / sumc;
//  4. the heads brought to the largest scale_h and requantized: o and its record.
// LDS: the per-step arrays (score and v factors, 32 B per cached position; hb heads' scores, 8 B per position each)
// for max_seq positions, then the head outputs and the rotated q (12 B per q value).
struct RdAttnShared {
    int64_t red[RD_WAVES];
    ScIdx redsc[RD_THREADS];
    Sc par[4];  // v_ref, s_ref, lut factor, common
    Sc hsc[64];
    Sc inv2[2];
    int64_t hsum[KT_REF_MAX_HEADS];
};

__device__ __forceinline__ void rd_attention_core(const RdAttn& a, unsigned char* lds, RdAttnShared& sh_,
                                                  int pos, int hb) {
    int64_t* red = sh_.red;
    ScIdx* redsc = sh_.redsc;
    Sc* par = sh_.par;
    Sc* hsc = sh_.hsc;
    const int tid = threadIdx.x, hd = a.hd, half = hd / 2, nh = a.nh, nkv = a.nkv, group = nh / nkv;
    const int kstride = nkv * hd, qstride = nh * hd;
    const int steps = pos + 1, rows = a.max_seq;  // rows: the per-step arrays' length
    Sc* F = reinterpret_cast<Sc*>(lds);  // score factors, per step
    Sc* VF = F + rows;                   // v factors, per step
    int64_t* S = reinterpret_cast<int64_t*>(VF + rows);   // scores, then exp codes: [hb][rows]
    int64_t* HO = S + (size_t)hb * rows;                  // head outputs, qstride
    int32_t* QD = reinterpret_cast<int32_t*>(HO + qstride);  // rotated q, qstride

    // 1. RoPE and the cache append
    auto rot = [&](const int32_t* src, int32_t* dst, int heads) {
        for (int i = tid; i < heads * half; i += RD_THREADS) {
            const int hh = i / half, j = i - hh * half;
            const kt_hip_sscale c = a.cos[(size_t)pos * half + j], s = a.sin[(size_t)pos * half + j];
            const int32_t av = src[hh * hd + j], bv = src[hh * hd + j + half];
            const Sc cm{c.mant, c.shift}, sm{s.mant, s.shift};
            dst[hh * hd + j] = (int32_t)(c.sign * sc_apply32(cm, av) - s.sign * sc_apply32(sm, bv));
            dst[hh * hd + j + half] = (int32_t)(c.sign * sc_apply32(cm, bv) + s.sign * sc_apply32(sm, av));
        }
    };
    rot(a.q, QD, nh);
    rot(a.k, a.kc + (size_t)pos * kstride, nkv);
    for (int i = tid; i < kstride; i += RD_THREADS) a.vc[(size_t)pos * kstride + i] = a.v[i];
    const Sc qs = rec_sc(a.qs), isq{a.isq_mant, a.isq_shift};
    if (tid == 0) {
        a.kscale[pos] = kt_hip_sscale{a.ks->mant, a.ks->shift, 1};
        a.vscale[pos] = kt_hip_sscale{a.vs->mant, a.vs->shift, 1};
    }
    __syncthreads();  // the cache row and both scales of this step are visible to the whole CTA past here

    // 2. v_ref and s_ref
    ScIdx bv{Sc{0, 0}, -1}, bs{Sc{0, 0}, -1};
    for (int j = tid; j < steps; j += RD_THREADS) {
        const Sc vj{a.vscale[j].mant, a.vscale[j].shift}, kj{a.kscale[j].mant, a.kscale[j].shift};
        const Sc sj = sc_mul(sc_mul(qs, kj), isq);
        F[j] = sj;
        bv = sc_pick(bv, ScIdx{vj, j});
        bs = sc_pick(bs, ScIdx{sj, j});
    }
    {
        ScIdx two[2] = {bv, bs};
        block_fold_max_k<2>(two, redsc);
        bv = two[0], bs = two[1];
    }
    if (tid == 0) {
        par[0] = bv.s, par[1] = bs.s;
        par[2] = bs.s.mant ? sc_mul(bs.s, Sc{a.exp.inv_mant, a.exp.inv_shift}) : Sc{0, 0};
    }
    __syncthreads();
    const Sc v_ref = par[0], s_ref = par[1], lm = par[2];
    if (v_ref.mant != 0 || s_ref.mant != 0) {
        Sc* inv2 = sh_.inv2;
        if (tid == 0) inv2[0] = v_ref.mant ? sc_recip(v_ref) : Sc{0, 0};  // the two reciprocals in two waves
        if (tid == 64) inv2[1] = s_ref.mant ? sc_recip(s_ref) : Sc{0, 0};
        __syncthreads();
        for (int j = tid; j < steps; j += RD_THREADS) {
            VF[j] = v_ref.mant ? sc_mul(Sc{a.vscale[j].mant, a.vscale[j].shift}, inv2[0]) : Sc{0, 0};
            if (s_ref.mant) F[j] = sc_mul(F[j], inv2[1]);
        }
    } else {
        for (int j = tid; j < steps; j += RD_THREADS) VF[j] = Sc{0, 0};
    }
    __syncthreads();

    // 3. the heads, hb at a time: the scores by one wave per (head, cached row) with the lanes across head_dim, the
    //    integer softmax by one wave per head, P.V by one thread per (head, dim). Sums wrap as i64 (any order gives
    //    the reference's integers).
    const int lane = tid & 63, wave = tid >> 6;
    int64_t* hsum = sh_.hsum;
    for (int h0 = 0; h0 < nh; h0 += hb) {
        const int hn = nh - h0 < hb ? nh - h0 : hb;
        if (s_ref.mant == 0) {  // every head skipped (the reference's `continue`)
            for (int i = tid; i < hn * hd; i += RD_THREADS) HO[h0 * hd + i] = 0;
            if (tid < hn) hsc[h0 + tid] = Sc{0, 0};
            continue;
        }
        const int items = hn * steps;
        // (16-byte loads: rows of a multiple of 32 values, q and the cache at 16-byte aligned addresses)
        const bool vec = hd % 32 == 0 && (((size_t)((const char*)QD - (const char*)lds)) & 15) == 0 &&
                         (reinterpret_cast<uintptr_t>(a.kc) & 15) == 0;
        if (vec) {
            // one thread per (head, cached row): the whole dot from 16-byte loads, 32 values of k in flight at a time
            for (int it = tid; it < items; it += RD_THREADS) {
                const int h = it / steps, j = it - h * steps, kv = (h0 + h) / group;
                const int4* kr = reinterpret_cast<const int4*>(a.kc + (size_t)j * kstride + kv * hd);
                const int4* qh = reinterpret_cast<const int4*>(QD + (h0 + h) * hd);
                int64_t dot = 0;
                for (int e4 = 0; e4 < hd / 4; e4 += 8) {
                    int4 kk[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) kk[u] = kr[e4 + u];
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        const int4 qq = qh[e4 + u];
                        dot = wadd(dot, (int64_t)qq.x * kk[u].x + (int64_t)qq.y * kk[u].y);  // each below 2^63
                        dot = wadd(dot, (int64_t)qq.z * kk[u].z + (int64_t)qq.w * kk[u].w);
                    }
                }
                S[(size_t)h * rows + j] = sc_apply(F[j], dot);
            }
        } else {
        // RD_SU items per wave at a time, every cached k row of them loaded before the first product (an item past
        // the end re-reads the last one and is dropped)
        constexpr int RD_SU = 8;
        for (int it0 = wave; it0 < items; it0 += RD_WAVES * RD_SU) {
            int64_t dot[RD_SU];
            int hh[RD_SU], jj[RD_SU];
#pragma unroll
            for (int u = 0; u < RD_SU; u++) {
                const int it = it0 + u * RD_WAVES, itc = it < items ? it : items - 1;
                hh[u] = itc / steps, jj[u] = itc - hh[u] * steps, dot[u] = 0;
            }
            for (int e = lane; e < hd; e += 64) {
                int32_t kk[RD_SU];
#pragma unroll
                for (int u = 0; u < RD_SU; u++)
                    kk[u] = a.kc[(size_t)jj[u] * kstride + ((h0 + hh[u]) / group) * hd + e];
#pragma unroll
                for (int u = 0; u < RD_SU; u++) dot[u] = wadd(dot[u], wmul(QD[(h0 + hh[u]) * hd + e], kk[u]));
            }
#pragma unroll
            for (int u = 0; u < RD_SU; u++) {
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) dot[u] = wadd(dot[u], __shfl_xor(dot[u], o, 64));
            }
            if (lane < RD_SU) {  // lane u stores item u (every lane holds every item's full sum)
                int64_t d = dot[0];
#pragma unroll
                for (int u = 1; u < RD_SU; u++) d = lane == u ? dot[u] : d;
                const int it = it0 + lane * RD_WAVES;
                const int h = it / steps, j = it - h * steps;
                if (it < items) S[(size_t)h * rows + j] = sc_apply(F[j], d);
            }
        }
        }
        __syncthreads();
        for (int h = wave; h < hn; h += RD_WAVES) {
            int64_t* sh = S + (size_t)h * rows;
            int64_t m = INT64_MIN;
            for (int j = lane; j < steps; j += 64) m = sh[j] > m ? sh[j] : m;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const int64_t u = __shfl_xor(m, o, 64);
                m = u > m ? u : m;
            }
            int64_t sum = 0;
            for (int j = lane; j < steps; j += 64) {
                const int64_t idx = lut_index(lm, (int64_t)((uint64_t)sh[j] - (uint64_t)m), a.exp.lo_index);
                sh[j] = idx < 0 ? 0 : lut_code(a.exp_codes, a.exp.n, idx);
                sum += sh[j];
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) sum = wadd(sum, __shfl_xor(sum, o, 64));
            if (lane == 0) {
                hsum[h] = sum;
                hsc[h0 + h] = sum <= 0 ? Sc{0, 0} : sc_mul(v_ref, from_ratio(1, (u128)(uint64_t)sum));
            }
        }
        __syncthreads();
        if (group <= RD_PV_GROUP) {
            // P.V by kv head: v_jd scaled once for the heads that share it (vf_j.apply(v_jd) is the same for every
            // head of a group), each wave one (kv head, slice of the steps) with its lanes across head_dim, the
            // heads' products summed into HO by LDS atomics (wrapping i64 sums: any order gives the same integers)
            for (int i = tid; i < hn * hd; i += RD_THREADS) HO[h0 * hd + i] = 0;
            __syncthreads();
            const int kv0 = h0 / group, nkvb = (h0 + hn - 1) / group - kv0 + 1;
            const int jp = RD_WAVES / nkvb > 1 ? RD_WAVES / nkvb : 1, tasks = nkvb * jp;
            for (int t = wave; t < tasks; t += RD_WAVES) {
                const int kv = kv0 + t / jp, js = t - (t / jp) * jp;
                const int hs = kv * group > h0 ? kv * group : h0;
                const int he = (kv + 1) * group < h0 + hn ? (kv + 1) * group : h0 + hn;  // heads [hs, he)
                for (int dd = lane; dd < hd; dd += 64) {
                    int64_t acc[RD_PV_GROUP];
#pragma unroll
                    for (int g = 0; g < RD_PV_GROUP; g++) acc[g] = 0;
                    const int32_t* vcol = a.vc + kv * hd + dd;
                    constexpr int RD_PU = 4;  // cached v values loaded before their products
                    for (int j0 = js; j0 < steps; j0 += RD_PU * jp) {
                        int32_t vv[RD_PU];
#pragma unroll
                        for (int u = 0; u < RD_PU; u++) {
                            const int j = j0 + u * jp < steps ? j0 + u * jp : steps - 1;
                            vv[u] = vcol[(size_t)j * kstride];
                        }
#pragma unroll
                        for (int u = 0; u < RD_PU; u++) {
                            const int j = j0 + u * jp;
                            if (j >= steps) break;
                            const int64_t sv = sc_apply32(VF[j], vv[u]);
#pragma unroll
                            for (int g = 0; g < RD_PV_GROUP; g++)
                                if (hs + g < he) acc[g] = wadd(acc[g], wmul(S[(size_t)(hs + g - h0) * rows + j], sv));
                        }
                    }
#pragma unroll
                    for (int g = 0; g < RD_PV_GROUP; g++)
                        if (hs + g < he && acc[g] != 0)
                            atomicAdd(reinterpret_cast<unsigned long long*>(&HO[(hs + g) * hd + dd]),
                                      (unsigned long long)acc[g]);
                }
            }
            __syncthreads();
            for (int i = tid; i < hn * hd; i += RD_THREADS)  // a head with no numerators: zeros
                if (hsum[i / hd] <= 0) HO[h0 * hd + i] = 0;
        } else {
            for (int it = tid; it < hn * hd; it += RD_THREADS) {
                const int h = it / hd, dd = it - h * hd, kv = (h0 + h) / group;
                int64_t acc = 0;
                if (hsum[h] > 0) {
                    const int64_t* sh = S + (size_t)h * rows;
                    const int32_t* vcol = a.vc + kv * hd + dd;
                    // RD_PU cached v values loaded before their products (a step past the end re-reads the last one
                    // and is dropped)
                    constexpr int RD_PU = 8;
                    for (int j0 = 0; j0 < steps; j0 += RD_PU) {
                        int32_t vv[RD_PU];
#pragma unroll
                        for (int u = 0; u < RD_PU; u++) {
                            const int j = j0 + u < steps ? j0 + u : steps - 1;
                            vv[u] = vcol[(size_t)j * kstride];
                        }
#pragma unroll
                        for (int u = 0; u < RD_PU; u++)
                            if (j0 + u < steps) acc = wadd(acc, wmul(sh[j0 + u], sc_apply32(VF[j0 + u], vv[u])));
                    }
                }
                HO[(h0 + h) * hd + dd] = acc;
            }
        }
        __syncthreads();  // S and hsum are reused by the next batch
    }

    // 4. one scale for the concatenated heads: the heads' largest by the engine's fold, then every thread its own
    //    reciprocal and its elements' head factors (no serial step)
    const Sc common = block_fold_max(tid < nh ? ScIdx{hsc[tid], tid} : ScIdx{Sc{0, 0}, -1}, redsc, nh).s;
    int64_t m = 0;
    if (common.mant != 0) {
        const Sc cinv = sc_recip(common);
        for (int i = tid; i < qstride; i += RD_THREADS) {
            HO[i] = sc_apply(sc_mul(hsc[i / hd], cinv), HO[i]);
            m = iabs(HO[i]) > m ? iabs(HO[i]) : m;
        }
    }
    const int64_t gmax = block_max_i64(m, red);
    const RqDen rd_gmax = rq_den(gmax);
    for (int i = tid; i < qstride; i += RD_THREADS) a.o[i] = gmax == 0 ? 0 : rq_apply(rd_gmax, HO[i]);
    if (tid == 0)
        put_rec(a.os, gmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), common));
}

// One CTA for every head: hb heads' scores at a time in LDS (a.hb >= 1).
__global__ __launch_bounds__(RD_THREADS) void rd_attention_step_kernel(RdAttn a) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ RdAttnShared sh_;
    const int pos = *a.pos;
    if (pos < 0 || pos >= a.max_seq) {  // outside the tables: zeros (the reference asserts here)
        for (int i = threadIdx.x; i < a.nh * a.hd; i += RD_THREADS) a.o[i] = 0;
        if (threadIdx.x == 0) put_rec(a.os, Sc{0, 0});
        return;
    }
    rd_attention_core(a, lds, sh_, pos, a.hb);
}

// Attention::decode_step between its projections with L.parts CTAs per q head, for caches of any length up to
// max_seq (kt_hip_ref_attention_step_ws): the cache reads, the per-step Scale work and P.V spread over nh * parts CUs
// instead of one. rd_attention_heads_kernel (CTA h * parts + part): RoPE of q_h and of this step's k (part 0 of the
// first head of each kv group appends the step's k and v rows to the cache, part 0 of head 0 the step's scales; row
// pos is taken from the inputs by every CTA, so no CTA reads what another writes in the same launch); every step's
// score factor f_j = s_j / s_ref and v factor vf_j = vs_j / v_ref, its head's scores, maximum and integer softmax
// numerators (the same integers in every CTA of the head); P.V over its share of the steps (P.V's 64-bit products
// are the step's largest cost, so they are what the parts divide); its part of the head's sums, and (part 0) the
// head's scale v_ref / sumc, into the workspace. rd_attention_combine_kernel (one CTA, the next launch): each head's
// parts added (wrapping, exact in any order), the heads at their largest scale, requantized -- step 4 of the one-CTA
// kernel.
struct RdHeadsLayout {
    size_t ho, hsc, arr, arr_stride;  // byte offsets: head output parts, head scales, per-CTA step arrays (and stride)
    int parts;                        // CTAs per head: each sums P.V over its share of the steps
};
__host__ __device__ inline size_t rd_round256(size_t v) { return (v + 255) / 256 * 256; }
__host__ __device__ inline RdHeadsLayout rd_heads_layout(int max_seq, int nh, int hd) {
    RdHeadsLayout L;
    L.parts = 128 / nh < 1 ? 1 : (128 / nh > 8 ? 8 : 128 / nh);  // 8 CTAs per head at the Qwen shape (112 CTAs)
    L.ho = 0;
    L.hsc = rd_round256((size_t)nh * L.parts * hd * sizeof(int64_t));
    L.arr = L.hsc + rd_round256((size_t)nh * sizeof(Sc));
    L.arr_stride = rd_round256((size_t)max_seq * (2 * sizeof(Sc) + sizeof(int64_t)));
    return L;
}

// cached v values (and their steps' numerators and factors) loaded before the products; RD_PV_W: the v values a lane
// of the wave-uniform P.V path has in flight
constexpr int RD_PV_U = 8, RD_PV_W = 16;
// The heads kernel's dynamic LDS when its per-step arrays stay in LDS (max_seq up to about 2,400 at head_dim 64; the
// static part is about 13 KB).
constexpr size_t RD_HEADS_LDS = 96 * 1024;

// GA: the per-step arrays in the workspace (caches longer than LDS holds), else in LDS after q and k. SUMS: q, k and v
// are the q / k / v product's sums (a.qsum, a.ksum, a.vsum): every CTA takes their maxima over the whole outputs,
// forms their Scales and the codes it reads as ql_requant_kernel would (CTA 0 writes the records).
// Bound by its chain of 64-bit Scale steps between barriers and the two round trips to the cache, not by bytes (14 / 2
// heads of 64 at 512 positions: 0.5 MB of cache). So every phase uses waves that the phase beside it leaves idle: RoPE
// a value a thread in the last waves, the v factors behind the numerators' waves, the Scale products a wave each; and
// the v rows are loaded before the softmax that weighs them (25.3 -> 20.8 us at 512 positions); the fold's winners are
// formed by the three waves that use them (20.8 -> 19.4).
template <bool GA, bool SUMS>
__global__ __launch_bounds__(RD_THREADS) void rd_attention_heads_kernel(RdAttn a, RdHeadsLayout L) {
    __shared__ int64_t red[3 * RD_WAVES];
    __shared__ Sc qkv_s[3];
    __shared__ ScIdx redsc[2 * RD_WAVES];
    __shared__ Sc par[4];  // v_ref, s_ref, lut factor, 1 / v_ref
    __shared__ Sc sinv_s;
    __shared__ int64_t PV[RD_THREADS];
    __shared__ int32_t VP[RD_THREADS];  // this step's v (hd <= RD_THREADS)
    extern __shared__ __align__(16) int32_t qk[];  // the rotated q_h (hd), then this step's rotated k (hd)
    const int P = L.parts, h = (int)blockIdx.x / P, part = (int)blockIdx.x % P;
    const int tid = threadIdx.x, hd = a.hd, half = hd / 2, nh = a.nh, nkv = a.nkv;
    const int group = nh / nkv, kv = h / group, kstride = nkv * hd;
    const int pos = *a.pos;
    // q, k and v: codes and Scales from the inputs, or requant_dyn of the sums
    int64_t ymax[3] = {0, 0, 0};
    if constexpr (SUMS) {
        for (int i = tid; i < nh * hd; i += RD_THREADS) ymax[0] = iabs(a.qsum.acc[i]) > ymax[0] ? iabs(a.qsum.acc[i]) : ymax[0];
        for (int i = tid; i < nkv * hd; i += RD_THREADS) {
            ymax[1] = iabs(a.ksum.acc[i]) > ymax[1] ? iabs(a.ksum.acc[i]) : ymax[1];
            ymax[2] = iabs(a.vsum.acc[i]) > ymax[2] ? iabs(a.vsum.acc[i]) : ymax[2];
        }
        block_max_k<3>(ymax, red);
        if ((tid & 63) == 0 && tid < 192) {  // the three Scale chains in three waves
            const RqSums& r = tid == 0 ? a.qsum : (tid == 64 ? a.ksum : a.vsum);
            const int64_t ym = ymax[tid >> 6];
            const Sc sc = rqs_scale(r.st, ym);
            qkv_s[tid >> 6] = sc;
            if (blockIdx.x == 0) rqs_record(r, ym, sc);
        }
        __syncthreads();
    }
    const Sc qs = SUMS ? qkv_s[0] : rec_sc(a.qs), ksp = SUMS ? qkv_s[1] : rec_sc(a.ks),
             vsp = SUMS ? qkv_s[2] : rec_sc(a.vs);
    unsigned char* ws = a.ws;
    int64_t* HO = reinterpret_cast<int64_t*>(ws + L.ho);
    Sc* HSC = reinterpret_cast<Sc*>(ws + L.hsc);
    if (pos < 0 || pos >= a.max_seq) {  // outside the tables: the combine writes zeros
        for (int d = tid; d < hd; d += RD_THREADS) HO[((size_t)h * P + part) * hd + d] = 0;
        if (tid == 0 && part == 0) HSC[h] = Sc{0, 0};
        return;
    }
    const int steps = pos + 1;
    int32_t* QD = qk;
    int32_t* KP = qk + hd;
    unsigned char* arr = GA ? ws + L.arr + ((size_t)h * P + part) * L.arr_stride
                            : reinterpret_cast<unsigned char*>(qk) + (size_t)rd_round256(2 * (size_t)hd * 4);
    Sc* F = reinterpret_cast<Sc*>(arr);                        // score factors, per step
    Sc* VF = F + a.max_seq;                                    // v factors, per step
    int64_t* S = reinterpret_cast<int64_t*>(VF + a.max_seq);   // scores, then exp codes

    // 1. RoPE (attention.rs:222-246) of q_h and of this step's k of kv head `kv`, this step's v, the cache append: a value
    //    a thread, from the last thread down, so that the waves of few steps' scales (2.) work beside them; read past
    //    the barriers of 2.
    const bool append = h == kv * group && part == 0;
    for (int t = RD_THREADS - 1 - tid; t < 3 * hd; t += RD_THREADS) {
        const int w = t / hd, i = t - w * hd;  // value i of q_h (w = 0), k (1) or v (2)
        const int j = i < half ? i : i - half, base = w == 0 ? h * hd : kv * hd;
        const int own = base + i, other = base + (i < half ? i + half : j);
        int32_t x, y = 0;
        if constexpr (SUMS) {
            const int64_t ym = w == 0 ? ymax[0] : (w == 1 ? ymax[1] : ymax[2]);
            const int64_t* acc = w == 0 ? a.qsum.acc : (w == 1 ? a.ksum.acc : a.vsum.acc);
            const bool live = w == 0 ? rqs_live(a.qsum.st, ymax[0])
                                     : (w == 1 ? rqs_live(a.ksum.st, ymax[1]) : rqs_live(a.vsum.st, ymax[2]));
            const RqDen dn = rq_den(ym);
            x = live ? rq_apply(dn, acc[own]) : 0;
            if (w != 2) y = live ? rq_apply(dn, acc[other]) : 0;
        } else {
            const int32_t* c = w == 0 ? a.q : (w == 1 ? a.k : a.v);
            x = c[own];
            if (w != 2) y = c[other];
        }
        if (w == 2) {
            VP[i] = x;
            if (append) a.vc[(size_t)pos * kstride + own] = x;
            continue;
        }
        const kt_hip_sscale c = a.cos[(size_t)pos * half + j], sn = a.sin[(size_t)pos * half + j];
        const int64_t cx = c.sign * sc_apply32(Sc{c.mant, c.shift}, x), sy = sn.sign * sc_apply32(Sc{sn.mant, sn.shift}, y);
        const int32_t r = (int32_t)(i < half ? cx - sy : cx + sy);
        qk[w * hd + i] = r;
        if (w == 1 && append) a.kc[(size_t)pos * kstride + own] = r;
    }
    if (h == 0 && part == 0 && tid == 0) {
        a.kscale[pos] = kt_hip_sscale{ksp.mant, ksp.shift, 1};
        a.vscale[pos] = kt_hip_sscale{vsp.mant, vsp.shift, 1};
    }

    // 2. every step's score scale s_j = qs * ks_j * inv_sqrt and v scale; their largest (the engine's fold)
    const Sc isq{a.isq_mant, a.isq_shift};
    ScIdx bv{Sc{0, 0}, -1}, bs{Sc{0, 0}, -1};
    for (int j = tid; j < steps; j += RD_THREADS) {
        const Sc kj = j == pos ? ksp : Sc{a.kscale[j].mant, a.kscale[j].shift};
        const Sc vj = j == pos ? vsp : Sc{a.vscale[j].mant, a.vscale[j].shift};
        const Sc sj = sc_mul(sc_mul(qs, kj), isq);
        F[j] = sj;
        VF[j] = vj;
        bv = sc_pick(bv, ScIdx{vj, j});
        bs = sc_pick(bs, ScIdx{sj, j});
    }
    fold_waves<2>({bv, bs}, redsc);
    const int wv = wave_id();  // the winners and what follows from each, a wave for each chain
    if (wv == 0) {
        const Sc v = fold_winner(0, redsc).s, r = v.mant ? sc_recip(v) : Sc{0, 0};
        if (tid == 0) par[0] = v, par[3] = r;
    } else if (wv == 1) {
        const Sc t = fold_winner(1, redsc).s, r = t.mant ? sc_recip(t) : Sc{0, 0};
        if (tid == 64) par[1] = t, sinv_s = r;
    } else if (wv == 2) {
        const Sc t = fold_winner(1, redsc).s, r = t.mant ? sc_mul(t, Sc{a.exp.inv_mant, a.exp.inv_shift}) : Sc{0, 0};
        if (tid == 128) par[2] = r;
    }
    __syncthreads();
    const Sc v_ref = par[0], s_ref = par[1], lm = par[2], vinv = par[3], sinv = sinv_s;
    if (s_ref.mant == 0) {  // the head is skipped (the reference's `continue`): zeros at Scale::ZERO
        for (int d = tid; d < hd; d += RD_THREADS) HO[((size_t)h * P + part) * hd + d] = 0;
        if (tid == 0 && part == 0) HSC[h] = Sc{0, 0};
        return;
    }

    // 3. scores: sp neighbouring lanes per cached step (16-byte loads of the cache row where it allows), so that few
    //    steps still use every wave and a lane's share of the row is one batch of loads
    const bool vec = hd % 4 == 0 && (reinterpret_cast<uintptr_t>(a.kc) & 15) == 0 && ((size_t)kstride * 4) % 16 == 0;
    const int sl = !vec || hd % 16 != 0 ? 0 : (steps <= RD_THREADS / 4 ? 2 : (steps <= RD_THREADS / 2 ? 1 : 0));
    const int sp = 1 << sl, sub = tid & (sp - 1);
    int64_t m = INT64_MIN;
    for (int j = tid >> sl; j < steps; j += RD_THREADS >> sl) {
        int64_t dot = 0;
        if (vec) {
            // 8 x 16 bytes of the cache row in flight at a time (16 spill registers)
            const int4* kr = reinterpret_cast<const int4*>(a.kc + (size_t)j * kstride + kv * hd);
            const int4 *kp = reinterpret_cast<const int4*>(KP), *qd = reinterpret_cast<const int4*>(QD);
            const int n4 = hd / 4;  // a multiple of sp
            for (int e0 = 0; e0 < n4; e0 += 8 * sp) {
                int4 kk[8];
                if (j != pos) {
#pragma unroll
                    for (int u = 0; u < 8; u++) kk[u] = e0 + u * sp < n4 ? kr[e0 + u * sp + sub] : int4{0, 0, 0, 0};
                } else {
#pragma unroll
                    for (int u = 0; u < 8; u++) kk[u] = e0 + u * sp < n4 ? kp[e0 + u * sp + sub] : int4{0, 0, 0, 0};
                }
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    if (e0 + u * sp >= n4) break;
                    const int4 q = qd[e0 + u * sp + sub];
                    dot = wadd(dot, (int64_t)q.x * kk[u].x + (int64_t)q.y * kk[u].y);  // each below 2^63
                    dot = wadd(dot, (int64_t)q.z * kk[u].z + (int64_t)q.w * kk[u].w);
                }
            }
            for (int o = 1; o < sp; o <<= 1) dot = wadd(dot, (int64_t)__shfl_xor((long long)dot, o));
        } else if (j == pos) {
            for (int d = 0; d < hd; d++) dot = wadd(dot, (int64_t)QD[d] * KP[d]);
        } else {
            const int32_t* kr = a.kc + (size_t)j * kstride + kv * hd;
            for (int d = 0; d < hd; d++) dot = wadd(dot, (int64_t)QD[d] * kr[d]);
        }
        const int64_t sc = sc_apply(sc_mul(F[j], sinv), dot);
        if (sub == 0) S[j] = sc;
        m = sc > m ? sc : m;
    }
    // the first v values of the wave-uniform P.V (5.) are on their way during the softmax (the row of this step is not
    // read: another CTA of this launch writes it)
    const int slices = RD_THREADS / hd, d = tid % hd, js = tid / hd, ST = P * slices;
    const int jw = __builtin_amdgcn_readfirstlane(js);
    const int32_t* vcol = a.vc + kv * hd + d;
    const bool wide = hd % 64 == 0 && jw < slices;
    int32_t v0[RD_PV_U];
#pragma unroll
    for (int u = 0; u < RD_PV_U; u++) {
        const int j = part * slices + jw + u * ST;
        v0[u] = 0;
        if (wide && j < pos) v0[u] = vcol[(size_t)j * kstride];
    }
    const int64_t dmax = block_max_i64(m, red);

    // 4. the integer-code softmax numerators and their sum
    int64_t sum = 0;
    for (int j = tid; j < steps; j += RD_THREADS) {
        const int64_t idx = lut_index(lm, (int64_t)((uint64_t)S[j] - (uint64_t)dmax), a.exp.lo_index);
        const int64_t ec = idx < 0 ? 0 : lut_code(a.exp_codes, a.exp.n, idx);
        S[j] = ec;
        sum += ec;
    }
    // the v factors, from the other end of the CTA's waves (of few steps: the waves that have no numerators)
    for (int j = (tid + RD_THREADS / 2) % RD_THREADS; j < steps; j += RD_THREADS)
        VF[j] = v_ref.mant ? sc_mul(VF[j], vinv) : Sc{0, 0};
    sum = (int64_t)wave_sum_u64((uint64_t)sum);
    if ((tid & 63) == 0) red[tid >> 6] = sum;
    __syncthreads();
    const int64_t sumc = (int64_t)lane64(row_sum_u64((tid & 63) < RD_WAVES ? (uint64_t)red[tid & 63] : 0), 0);
    if (sumc <= 0) {
        for (int d = tid; d < hd; d += RD_THREADS) HO[((size_t)h * P + part) * hd + d] = 0;
        if (tid == 0 && part == 0) HSC[h] = Sc{0, 0};
        return;
    }

    // 5. P.V: thread js * hd + d (hd <= RD_THREADS) sums the steps j = js (mod slices) of column d (wrapping i64:
    //    any order gives the reference's integers); the slices then add up in LDS
    const int32_t vpos = VP[d];  // this step's v (its cache row is written in this same launch)
    int64_t acc = 0;
    if (hd % 64 == 0) {
        // a wave is one slice: its step, numerator and v factor are the same on every lane, so they are read once
        // into scalar registers and Scale::apply's branches and shift amounts are scalar
        // The cached v rows come from HBM (the weight streams evicted them since the previous token): RD_PV_W of
        // them in flight per lane at a time, so that a few dependent round trips, not one per RD_PV_U steps, pay
        // for the whole column.
        // slice jw of this CTA's share: the steps j = part * slices + jw (mod P * slices)
        if (wide) {
            auto add = [&](int j, int32_t v) {  // j uniform
                if (j >= steps) return;
                const int64_t e = S[j];
                const Sc f = VF[j];
                const int64_t ec = ((int64_t)__builtin_amdgcn_readfirstlane((int)((uint64_t)e >> 32)) << 32) |
                                   (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)e);
                Sc vf;
                vf.mant = ((int64_t)__builtin_amdgcn_readfirstlane((int)((uint64_t)f.mant >> 32)) << 32) |
                          (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)f.mant);
                vf.shift = __builtin_amdgcn_readfirstlane(f.shift);
                acc = wadd(acc, wmul(ec, sc_apply32(vf, j == pos ? vpos : v)));
            };
            int j0 = part * slices + jw;
#pragma unroll
            for (int u = 0; u < RD_PV_U; u++) add(j0 + u * ST, v0[u]);
            for (j0 += RD_PV_U * ST; j0 < steps; j0 += RD_PV_W * ST) {
                int32_t vv[RD_PV_W];
#pragma unroll
                for (int u = 0; u < RD_PV_W; u++) {
                    vv[u] = 0;
                    if (j0 + u * ST < pos) vv[u] = vcol[(size_t)(j0 + u * ST) * kstride];
                }
#pragma unroll
                for (int u = 0; u < RD_PV_W; u++) add(j0 + u * ST, vv[u]);
            }
        }
    } else if (js < slices) {
        for (int j0 = part * slices + js; j0 < steps; j0 += RD_PV_U * ST) {
            int32_t vv[RD_PV_U];
            int64_t ec[RD_PV_U];
            Sc vf[RD_PV_U];
#pragma unroll
            for (int u = 0; u < RD_PV_U; u++) {  // a step past the end reads the last one and adds nothing
                const int j = j0 + u * ST < steps ? j0 + u * ST : steps - 1;
                vv[u] = j == pos ? vpos : vcol[(size_t)j * kstride];
                ec[u] = S[j];
                vf[u] = VF[j];
            }
#pragma unroll
            for (int u = 0; u < RD_PV_U; u++)
                if (j0 + u * ST < steps) acc = wadd(acc, wmul(ec[u], sc_apply32(vf[u], vv[u])));
        }
    }
    PV[tid] = acc;
    __syncthreads();
    for (int dd = tid; dd < hd; dd += RD_THREADS) {  // this CTA's part of the head's sums (the combine adds the parts)
        int64_t t = 0;
#pragma unroll 8
        for (int q = 0; q < slices; q++) t = wadd(t, PV[q * hd + dd]);
        HO[((size_t)h * P + part) * hd + dd] = t;
    }
    if (tid == 64 && part == 0) HSC[h] = sc_mul(v_ref, from_ratio(1, (u128)(uint64_t)sumc));
}

// Step 4 of Attention::decode_step over the heads kernel's outputs: the heads' largest scale by the engine's fold,
// each head brought to it, requant_dyn of the concatenation, the record.
// One wave forms the common Scale and its reciprocal (14 heads of 64: 7.2 -> 6.6 us; in every thread before).
constexpr int RD_CB = 2;  // head-output values a combine thread holds (nh * hd up to 2048); longer rows recompute
__global__ __launch_bounds__(RD_THREADS) void rd_attention_combine_kernel(RdAttn a, RdHeadsLayout L) {
    __shared__ int64_t red[RD_WAVES];
    __shared__ ScIdx redsc[2 * RD_WAVES];
    __shared__ Sc par[2];  // the common Scale, its reciprocal
    const int tid = threadIdx.x, hd = a.hd, nh = a.nh, qstride = nh * hd, P = L.parts;
    const int64_t* HOP = reinterpret_cast<const int64_t*>(a.ws + L.ho);
    const Sc* HSC = reinterpret_cast<const Sc*>(a.ws + L.hsc);
    // each head's sums: its CTAs' parts (at most 8) added, wrapping, in any order (the reference's integers); the
    // parts' loads all issued before the adds
    auto ho = [&](int i) {
        const int hh = i / hd, dd = i - hh * hd;
        const int64_t* p = HOP + (size_t)hh * P * hd + dd;
        int64_t t[8];
#pragma unroll
        for (int q = 0; q < 8; q++) t[q] = q < P ? p[(size_t)q * hd] : 0;
        int64_t s = 0;
#pragma unroll
        for (int q = 0; q < 8; q++) s = wadd(s, t[q]);
        return s;
    };
    // the sums of the values a thread holds are read before the heads' fold, so the two overlap
    const bool held = qstride <= RD_THREADS * RD_CB;
    int64_t hv[RD_CB];
#pragma unroll
    for (int k = 0; k < RD_CB; k++) {
        const int i = tid + RD_THREADS * k;
        hv[k] = held && i < qstride ? ho(i) : 0;
    }
    fold_waves<1>({tid < nh ? ScIdx{HSC[tid], tid} : ScIdx{Sc{0, 0}, -1}}, redsc);
    if (wave_id() == 0) {  // the common Scale and its reciprocal once, not on four waves of each SIMD
        const Sc c = fold_winner(0, redsc).s, r = c.mant != 0 ? sc_recip(c) : Sc{0, 0};
        if (tid == 0) par[0] = c, par[1] = r;
    }
    __syncthreads();
    const Sc common = par[0], cinv = par[1];
    int64_t m = 0;
    if (common.mant != 0) {
        if (held) {
#pragma unroll
            for (int k = 0; k < RD_CB; k++) {  // each value at the common scale, kept for the requant
                const int i = tid + RD_THREADS * k;
                if (i < qstride) hv[k] = sc_apply(sc_mul(HSC[i / hd], cinv), hv[k]);
                m = iabs(hv[k]) > m ? iabs(hv[k]) : m;
            }
        } else {
            for (int i = tid; i < qstride; i += RD_THREADS) {
                const int64_t v = sc_apply(sc_mul(HSC[i / hd], cinv), ho(i));
                m = iabs(v) > m ? iabs(v) : m;
            }
        }
    }
    const int64_t gmax = block_max_i64(m, red);
    const RqDen rd_gmax = rq_den(gmax);
    if (gmax == 0) {
        for (int i = tid; i < qstride; i += RD_THREADS) a.o[i] = 0;
    } else if (held) {
#pragma unroll
        for (int k = 0; k < RD_CB; k++) {
            const int i = tid + RD_THREADS * k;
            if (i < qstride) a.o[i] = rq_apply(rd_gmax, hv[k]);
        }
    } else {
        for (int i = tid; i < qstride; i += RD_THREADS) a.o[i] = rq_apply(rd_gmax, sc_apply(sc_mul(HSC[i / hd], cinv), ho(i)));
    }
    if (tid == 0)
        put_rec(a.os, gmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), common));
}

// The same ops over whole-sequence tensors on many CTAs (the batched forward's T-row tensors), two launches each: a
// grid pass takes the largest magnitude, a grid pass requantizes and writes the record. Integers identical to the
// one-CTA kernels.
//  - Every wave of add's and SwiGLU's first pass forms the tensor's Scales itself on wave-uniform values (two or three
//    Scale steps, under a microsecond): no one-CTA launch before the pass. CTA 0 leaves them for the second pass, since
//    y's record may overwrite an input's.
//  - A CTA's largest magnitude goes to its own slot of the workspace and the second pass takes the largest slot. An
//    atomic maximum on one word serialized (13 ns a CTA): SwiGLU's first pass at 256 x 4864 went from 28.3 (2,048
//    CTAs) to 10.1 us, the add's at 256 x 896 from 13.1 (896 CTAs) to 5.5 us.
//  - RMSNorm's first pass is a wave per row: the exact sum of squares, max |x g|, the row factor's Scale chain, all
//    rows side by side (8.3 us at 256 x 896; one CTA of 16 waves walking the rows took about 120). A factor f >= 0 keeps
//    order (Scale::apply rounds |v| monotonely, and f <= 1 so nothing wraps), so the tensor's largest magnitude is
//    the largest apply(f_row, max |x g| of the row): no pass over the values is needed for it.
constexpr int RS_PARTS = 512;        // the first pass's CTAs at most
constexpr int RS_FOLD_ROWS = 1024;   // RMSNorm rows that every CTA of the second pass folds itself
struct RdSeqWs {
    Sc par[4];               // add and SwiGLU: RsPar's three; RMSNorm past RS_FOLD_ROWS rows: the common Scale
    uint64_t gmax;           // those rows' largest magnitude
    int64_t part[RS_PARTS];  // the largest magnitude of each CTA of the first pass
    // then RMSNorm's rows: Sc crow[rows] (the row factor), int64_t pmax[rows] (the largest |x g| of the row)
};
__host__ __device__ inline Sc* rs_crow(RdSeqWs* w) { return reinterpret_cast<Sc*>(w + 1); }
__host__ __device__ inline int64_t* rs_pmax(RdSeqWs* w, int rows) { return reinterpret_cast<int64_t*>(rs_crow(w) + rows); }
enum { RS_ADD = 0, RS_SWIGLU = 1, RS_NORM = 2 };
struct RdSeq {
    int op;
    const int32_t *a, *b;  // add: a, b; SwiGLU: g, u; RMSNorm: x, gamma
    const kt_hip_qscale *as, *bs;
    int64_t n;             // values (rows * dim for RMSNorm)
    int rows, dim;
    int64_t g_mant, e_mant;
    int32_t g_shift, e_shift;
    const int64_t* codes;
    kt_hip_codelut lut;
    RdSeqWs* ws;
    int32_t* y;
    kt_hip_qscale* ys;
};

// add: common, fa, fb; SwiGLU (as is g's record, bs u's): index factor, identity factor, h scale.
struct RsPar {
    Sc p0, p1, p2;
};
template <int OP>
__device__ inline RsPar rs_params(const RdSeq& q, const kt_hip_qscale* as_rec, const kt_hip_qscale* bs_rec) {
    const Sc as = uni(rec_sc(as_rec)), bs = uni(rec_sc(bs_rec)), z{0, 0};
    if constexpr (OP == RS_ADD) {
        const Sc common = sc_ge(as, bs) ? as : bs;
        if (common.mant == 0) return RsPar{common, z, z};
        const Sc cinv = sc_recip(common);
        return RsPar{common, sc_mul(as, cinv), sc_mul(bs, cinv)};
    } else {
        const Sc cs{q.lut.code_mant, q.lut.code_shift};
        return RsPar{sc_mul(as, Sc{q.lut.inv_mant, q.lut.inv_shift}), sc_mul(as, sc_recip(cs)), sc_mul(cs, bs)};
    }
}
template <int OP>
__device__ inline int64_t rs_value(const RdSeq& q, const RsPar& p, int32_t a, int32_t b) {
    if constexpr (OP == RS_ADD) {
        return wadd(sc_apply32(p.p1, a), sc_apply32(p.p2, b));
    } else {
        const int64_t idx = lut_index32(p.p0, a, q.lut.lo_index);
        const int64_t code = idx < 0 ? 0 : (idx >= q.lut.n ? sc_apply32(p.p1, a) : lut_code(q.codes, q.lut.n, idx));
        return wmul(code, b);
    }
}
// whether the values are live (a zero common scale gives zeros)
template <int OP>
__device__ inline bool rs_live(const RsPar& p) { return OP == RS_SWIGLU || p.p0.mant != 0; }

// the largest of the first pass's slots, in every thread of a 256-thread CTA
__device__ inline int64_t rs_gmax(const RdSeqWs* w, int nparts, int64_t* red) {
    int64_t m = 0;
    for (int i = threadIdx.x; i < nparts; i += 256) m = max64(m, w->part[i]);
    return block_max_4w(m, red);
}

template <int OP>
__global__ __launch_bounds__(256) void rs_max_kernel(RdSeq q) {
    __shared__ int64_t red[4];
    const RsPar p = rs_params<OP>(q, q.as, q.bs);
    const int64_t step = (int64_t)gridDim.x * 256;
    int64_t m = 0;
    if (rs_live<OP>(p)) {
        for (int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x; i0 < q.n; i0 += 4 * step) {  // 4 loads in flight
            int32_t a[4], b[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int64_t i = i0 + u * step;
                a[u] = i < q.n ? q.a[i] : 0, b[u] = i < q.n ? q.b[i] : 0;  // zeros give a zero (add; silu * 0)
            }
#pragma unroll
            for (int u = 0; u < 4; u++) m = max64(m, iabs(rs_value<OP>(q, p, a[u], b[u])));
        }
    }
    m = block_max_4w(m, red);
    if (threadIdx.x == 0) q.ws->part[blockIdx.x] = m;
    // the record of y may be a's or b's (add in place): its reader takes the inputs' Scales from here
    if (blockIdx.x == 0 && threadIdx.x == 0) q.ws->par[0] = p.p0, q.ws->par[1] = p.p1, q.ws->par[2] = p.p2;
}

template <int OP>
__global__ __launch_bounds__(256) void rs_out_kernel(RdSeq q, int nparts) {
    __shared__ int64_t red[4];
    const RdSeqWs* w = q.ws;
    const RsPar p{w->par[0], w->par[1], w->par[2]};
    const int64_t gmax = rs_gmax(w, nparts, red);
    const RqDen rd_gmax = rq_den(gmax);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < q.n; i += (int64_t)gridDim.x * 256)
        q.y[i] = gmax == 0 ? 0 : rq_apply(rd_gmax, rs_value<OP>(q, p, q.a[i], q.b[i]));
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const Sc sc = OP == RS_SWIGLU ? p.p2 : p.p0;  // the tensor's scale before the requant
        put_rec(q.ys, gmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), sc));
    }
}

// RMSNorm's first pass: a wave per row.
__global__ __launch_bounds__(256) void rs_rows_kernel(RdSeq q) {
    const int lane = threadIdx.x & 63, r = (int)blockIdx.x * 4 + wave_id();
    if (r >= q.rows) return;  // the whole wave
    const int32_t* xr = q.a + (size_t)r * q.dim;
    uint64_t hi = 0, lo = 0;
    int64_t pm = 0;
    for (int i0 = lane; i0 < q.dim; i0 += 8 * 64) {  // 8 loads of each in flight
        int32_t x[8], g[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = i0 + 64 * u;
            x[u] = i < q.dim ? xr[i] : 0, g[u] = i < q.dim ? q.b[i] : 0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const uint64_t sq = (uint64_t)((int64_t)x[u] * x[u]), t = lo + sq;
            hi += t < lo, lo = t;
            pm = max64(pm, iabs((int64_t)x[u] * g[u]));
        }
    }
    add128_row(hi, lo);
    u128 ss = 0;
#pragma unroll
    for (int l = 0; l < 64; l += 16) ss += ((u128)lane64(hi, l) << 64) | lane64(lo, l);
    pm = wave_max_i64(pm);
    const Sc xs = uni(rec_sc(q.as)), gs{q.g_mant, q.g_shift}, eps{q.e_mant, q.e_shift};
    const Sc mean_sq = sc_mul(sc_mul(from_ratio(ss, (u128)q.dim), xs), xs);
    const Sc denom = sc_add(mean_sq, eps);
    const Sc cr = sc_mul(sc_mul(xs, denom.mant == 0 ? Sc{0, 0} : sc_rsqrt(denom)), gs);
    if (lane == 0) rs_crow(q.ws)[r] = cr, rs_pmax(q.ws, q.rows)[r] = pm;
}

// The largest of n Scales by the engine's fold over their order (of equal values the latest), and the largest
// magnitude at that scale of the groups they scale, pmax holding each group's largest |value| (INT64_MAX for a value of
// INT64_MIN); NT threads of the CTA. Below 2^62 a factor of at most 1 keeps the order of the magnitudes; past(r, factor)
// gives group r's largest from its values where they may wrap.
template <int NT, class Past>
__device__ inline void scale_fold(const Sc* scale, const int64_t* pmax, int n, uint64_t* redk, int64_t* red, Sc& cc,
                                  int64_t& gmax, Past past) {
    FoldKey k{0, 0, 0};
    for (int r = threadIdx.x; r < n; r += NT) {
        const FoldKey u = fold_key(ScIdx{scale[r], r});
        if (fold_gt(u, k)) k = u;
    }
    fold_row(k);
    const int lane = threadIdx.x & 63;
    if ((lane & 15) == 0) {
        uint64_t* d = redk + (threadIdx.x >> 4) * 3;
        d[0] = k.e, d[1] = k.m, d[2] = k.i;
    }
    __syncthreads();
    k = FoldKey{0, 0, 0};
    for (int i = lane & 15; i < NT / 16; i += 16) {  // the rows of 16 lanes' keys, in every row of every wave
        const uint64_t* d = redk + i * 3;
        const FoldKey u{d[0], d[1], d[2]};
        if (fold_gt(u, k)) k = u;
    }
    fold_row(k);
    cc = fold_item(fold_lane(k, 0)).s;
    int64_t m = 0;
    if (cc.mant != 0) {
        const Sc cinv = sc_recip(cc);
        for (int r = threadIdx.x; r < n; r += NT) {
            const Sc f = sc_mul(scale[r], cinv);
            m = max64(m, pmax[r] <= (int64_t)1 << 62 ? sc_apply(f, pmax[r]) : past(r, f));
        }
    }
    if constexpr (NT == 256) gmax = block_max_4w(m, red);
    else gmax = block_max_i64(m, red);
}
// RMSNorm's |x g| is at most 2^62.
__device__ inline int64_t rs_no_past(int, Sc) { return 0; }
// past RS_FOLD_ROWS rows: the fold by one CTA
__global__ __launch_bounds__(RD_THREADS) void rs_norm_fold_kernel(RdSeq q) {
    __shared__ uint64_t redk[3 * RD_THREADS / 16];
    __shared__ int64_t red[RD_WAVES];
    Sc cc;
    int64_t gmax;
    scale_fold<RD_THREADS>(rs_crow(q.ws), rs_pmax(q.ws, q.rows), q.rows, redk, red, cc, gmax, rs_no_past);
    if (threadIdx.x == 0) q.ws->par[0] = cc, q.ws->gmax = (uint64_t)gmax;
}
// RMSNorm's second pass: a CTA per row (grid-stride), FOLD: its CTAs fold the rows themselves.
template <bool FOLD>
__global__ __launch_bounds__(256) void rs_norm_out_kernel(RdSeq q) {
    __shared__ uint64_t redk[FOLD ? 3 * 256 / 16 : 1];
    __shared__ int64_t red[4];
    Sc cc;
    int64_t gmax;
    if constexpr (FOLD) scale_fold<256>(rs_crow(q.ws), rs_pmax(q.ws, q.rows), q.rows, redk, red, cc, gmax, rs_no_past);
    else cc = q.ws->par[0], gmax = (int64_t)q.ws->gmax;
    const RqDen rd_gmax = rq_den(gmax);
    const Sc cinv = cc.mant != 0 ? sc_recip(cc) : Sc{0, 0};
    for (int r = blockIdx.x; r < q.rows; r += gridDim.x) {
        const Sc f = gmax == 0 ? Sc{0, 0} : sc_mul(rs_crow(q.ws)[r], cinv);
        const size_t at = (size_t)r * q.dim;
        for (int i = threadIdx.x; i < q.dim; i += 256)
            q.y[at + i] = gmax == 0 ? 0 : rq_apply(rd_gmax, sc_apply(f, (int64_t)q.a[at + i] * (int64_t)q.b[i]));
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        put_rec(q.ys, gmax == 0 ? Sc{0, 0} : sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), cc));
}

// Embedding::lookup_seq (layers.rs:1138-1145): the code rows of T tokens at the table's scale (a token outside the
// vocabulary gives a zero row; the reference panics there).
__global__ __launch_bounds__(256) void rd_embed_seq_kernel(const int32_t* __restrict__ emb, int64_t e_mant,
                                                           int32_t e_shift, const int32_t* __restrict__ tokens,
                                                           int T, int vocab, int dim, int32_t* __restrict__ y,
                                                           kt_hip_qscale* __restrict__ ys) {
    const int64_t n = (int64_t)T * dim;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int t = tokens[i / dim];
        y[i] = t >= 0 && t < vocab ? emb[(int64_t)t * dim + i % dim] : 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) put_rec(ys, Sc{e_mant, e_shift});
}

// Attention::forward_int (attention.rs:467-598) in four launches:
//  rp_rope    q and k of row i rotated at position i (rope_int, attention.rs:208-229)
//  rp_head    per (head, row i): the causal dots j <= i (exact, wrapping i64) at the one score scale
//             q.scale * k.scale * inv_sqrt, the exp-CodeLut numerators of (dot - max), their sum, the sums of
//             numerator * v over the rows, their largest magnitude, the scale v.scale / sum
//  rp_fold    one CTA: the largest scale by the engine's fold over the [row][head] order, and the largest magnitude at
//             that scale, from each (row, head)'s largest sum (Scale::apply keeps order: scale_fold)
//  rp_out     the outputs brought to the common scale and requantized, and their record
__global__ __launch_bounds__(256) void rp_rope_kernel(RdPrefill a) {
    const int i = blockIdx.x, half = a.hd / 2, qw = a.nh * a.hd, kw = a.nkv * a.hd;
    for (int e = threadIdx.x; e < (a.nh + a.nkv) * half; e += 256) {
        const bool isk = e >= a.nh * half;
        const int hh = (isk ? e - a.nh * half : e) / half, j = (isk ? e - a.nh * half : e) % half;
        const int32_t* src = isk ? a.k + (size_t)i * kw : a.q + (size_t)i * qw;
        int32_t* dst = isk ? a.kd + (size_t)i * kw : a.qd + (size_t)i * qw;
        const kt_hip_sscale c = a.cos[(size_t)i * half + j], sn = a.sin[(size_t)i * half + j];
        const int32_t av = src[hh * a.hd + j], bv = src[hh * a.hd + j + half];
        const Sc cm{c.mant, c.shift}, sm{sn.mant, sn.shift};
        dst[hh * a.hd + j] = (int32_t)(c.sign * sc_apply32(cm, av) - sn.sign * sc_apply32(sm, bv));
        dst[hh * a.hd + j + half] = (int32_t)(c.sign * sc_apply32(cm, bv) + sn.sign * sc_apply32(sm, av));
    }
}

// The score table's index factor: q.scale * k.scale * inv_sqrt * inv_step.
__device__ inline Sc rp_index_factor(const RdPrefill& a) {
    const Sc s_score = sc_mul(sc_mul(uni(rec_sc(a.qs)), uni(rec_sc(a.ks))), Sc{a.isq_mant, a.isq_shift});
    return sc_mul(s_score, Sc{a.exp.inv_mant, a.exp.inv_shift});
}

// Head dimensions of 64 and 128: R rows of a head per CTA of 4 waves. The dots are 64-bit multiply-adds of one lane per
// cached row: the lane holds its k row in registers (16-byte loads) and meets each of the R q rows, whose values are
// wave-uniform and come through scalar registers; the waves take every fourth block of 64 cached rows. For the sums
// of numerator * v the lanes are the head's dimensions, a numerator is one LDS broadcast, and the waves take every
// fourth run of 8 rows. Bound by those multiply-adds (about half of the 28 us at 256 rows), R of them per k or v value
// read. 256 rows, 14 heads of 64: 41.6 -> 27.9 us against one row per CTA with a strided 4-byte k load per product
// (the whole op 69.4 -> 46.0; at 2048 rows 2045 -> 868).
template <int HD, int R>
__global__ __launch_bounds__(256) void rp_head_kernel(RdPrefill a) {
    typedef const __attribute__((address_space(4))) int32_t* const_i32;  // read through scalar loads
    constexpr int ND = HD / 64;
    extern __shared__ int64_t S[];  // [R][T]: the dots, then the numerators
    __shared__ int64_t red[R][4];
    __shared__ int64_t part[4][R][HD];
    const int T = a.T, nb = (T + R - 1) / R, h = (int)blockIdx.x / nb, kv = h / (a.nh / a.nkv), kw = a.nkv * HD;
    const int i0 = (nb - 1 - (int)blockIdx.x % nb) * R;  // the longest rows first
    const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
    const int nr = T - i0 < R ? T - i0 : R, jend = i0 + nr;  // rows of this CTA; cached rows any of them attends
    int64_t m[R];
#pragma unroll
    for (int r = 0; r < R; r++) m[r] = INT64_MIN;
    for (int t0 = 64 * w; t0 < jend; t0 += 256) {
        const int j = t0 + lane, jc = j < T ? j : T - 1;
        const v4i* kr = reinterpret_cast<const v4i*>(a.kd + (size_t)jc * kw + kv * HD);
        v4i k[HD / 4];
#pragma unroll
        for (int c = 0; c < HD / 4; c++) k[c] = kr[c];
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r >= nr) break;  // uniform
            const const_i32 q = (const_i32)(uint64_t)(a.qd + ((size_t)(i0 + r) * a.nh + h) * HD);
            int64_t dot = 0;
#pragma unroll
            for (int d = 0; d < HD; d++) dot = wadd(dot, (int64_t)q[d] * (int64_t)k[d >> 2][d & 3]);
            if (j <= i0 + r) {
                S[r * T + j] = dot;
                m[r] = max64(m[r], dot);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        m[r] = wave_max_i64(m[r]);
        if (lane == 0) red[r][w] = m[r];
    }
    const Sc lm = rp_index_factor(a);
    __syncthreads();
    int64_t sum[R], dmax[R];
    bool wide = false;  // a numerator past 31 bits (no table of 2^20 codes has one)
#pragma unroll
    for (int r = 0; r < R; r++) {
        dmax[r] = max64(max64(red[r][0], red[r][1]), max64(red[r][2], red[r][3]));
        sum[r] = 0;
    }
    for (int j = tid; j < jend; j += 256) {  // the rows' table reads in flight together
        int64_t c[R], idx[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const bool on = r < nr && j <= i0 + r;
            const int64_t dot = on ? S[r * T + j] : dmax[r];
            idx[r] = on ? lut_index(lm, (int64_t)((uint64_t)dot - (uint64_t)dmax[r]), a.exp.lo_index) : -1;
        }
#pragma unroll
        for (int r = 0; r < R; r++) c[r] = lut_code(a.exp_codes, a.exp.n, idx[r]);
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (idx[r] < 0) c[r] = 0;
            if (r < nr) S[r * T + j] = c[r];  // zero past the row's own position
            sum[r] = wadd(sum[r], c[r]);
            wide = wide || ((uint64_t)c[r] >> 31) != 0;
        }
    }
    wide = __syncthreads_or(wide);  // also orders the reads of red before its next writes
#pragma unroll
    for (int r = 0; r < R; r++) {
        sum[r] = (int64_t)wave_sum_u64((uint64_t)sum[r]);
        if (lane == 0) red[r][w] = sum[r];
    }
    int64_t acc[R][ND];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int e = 0; e < ND; e++) acc[r][e] = 0;
    auto weigh = [&](auto narrow) {
        int32_t v[8][ND], vn[8][ND];
        auto fetch = [&](int j0, int32_t(&x)[8][ND]) {  // rows past the last read it again, with zero numerators
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int e = 0; e < ND; e++)
                    x[u][e] = a.v[(size_t)(j0 + u < T ? j0 + u : T - 1) * kw + kv * HD + 64 * e + lane];
        };
        fetch(8 * w, vn);
        for (int j0 = 8 * w; j0 < jend; j0 += 32) {
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int e = 0; e < ND; e++) v[u][e] = vn[u][e];
            fetch(j0 + 32, vn);  // under this run's products
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (r >= nr) break;  // uniform
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const int64_t s = j0 + u < jend ? S[r * T + j0 + u] : 0;
#pragma unroll
                    for (int e = 0; e < ND; e++) {
                        if constexpr (decltype(narrow)::value)
                            acc[r][e] = wadd(acc[r][e], (int64_t)(int32_t)s * (int64_t)v[u][e]);
                        else
                            acc[r][e] = wadd(acc[r][e], wmul(s, v[u][e]));
                    }
                }
            }
        }
    };
    if (wide) weigh(std::false_type{});
    else weigh(std::true_type{});
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int e = 0; e < ND; e++) part[w][r][64 * e + lane] = acc[r][e];
    __syncthreads();
    if (w >= nr) return;  // wave r finishes row r (R <= 4)
    const size_t ih = (size_t)(i0 + w) * a.nh + h;
    const int64_t sumc = wadd(wadd(red[w][0], red[w][1]), wadd(red[w][2], red[w][3]));
    int64_t pm = 0;
#pragma unroll
    for (int e = 0; e < ND; e++) {
        const int d = 64 * e + lane;
        int64_t t = wadd(wadd(part[0][w][d], part[1][w][d]), wadd(part[2][w][d], part[3][w][d]));
        if (sumc <= 0) t = 0;
        a.hout[ih * HD + d] = t;
        pm = max64(pm, magnitude(t));
    }
    pm = wave_max_i64(pm);
    const int64_t su = uni64(sumc);
    const Sc sc = su > 0 ? sc_mul(uni(rec_sc(a.vs)), from_ratio(1, (u128)(uint64_t)su)) : Sc{0, 0};
    if (lane == 0) a.hmax[ih] = pm, a.fac[ih] = sc;
}

// Any other head dimension (up to 256): a CTA per (head, row).
__global__ __launch_bounds__(256) void rp_head_any_kernel(RdPrefill a) {
    extern __shared__ int64_t S[];  // T: the dots, then the numerators
    __shared__ int64_t red[4];
    __shared__ int64_t part[256];
    __shared__ int32_t qrow[256];
    const int h = blockIdx.x / a.T, i = blockIdx.x % a.T, hd = a.hd, kv = h / (a.nh / a.nkv);
    const int kw = a.nkv * a.hd, tid = threadIdx.x;
    for (int d = tid; d < hd; d += 256) qrow[d] = a.qd[(size_t)i * a.nh * hd + h * hd + d];
    const Sc lm = rp_index_factor(a);
    __syncthreads();
    int64_t m = INT64_MIN;
    for (int j = tid; j <= i; j += 256) {
        const int32_t* kr = a.kd + (size_t)j * kw + kv * hd;
        int64_t dot = 0;
        for (int d = 0; d < hd; d++) dot = wadd(dot, wmul(qrow[d], kr[d]));
        S[j] = dot;
        m = dot > m ? dot : m;
    }
    const int64_t dmax = block_max_4w(m, red);
    int64_t sum = 0;
    for (int j = tid; j <= i; j += 256) {
        const int64_t idx = lut_index(lm, (int64_t)((uint64_t)S[j] - (uint64_t)dmax), a.exp.lo_index);
        S[j] = idx < 0 ? 0 : lut_code(a.exp_codes, a.exp.n, idx);
        sum += S[j];
    }
    const int64_t sumc = block_sum_4w(sum, red);  // also orders the numerator writes before the reads below
    const int groups = 256 / hd, gq = tid / hd, d = tid - gq * hd;
    int64_t acc = 0;
    if (sumc > 0 && gq < groups)
        for (int j = gq; j <= i; j += groups) acc = wadd(acc, wmul(S[j], a.v[(size_t)j * kw + kv * hd + d]));
    part[tid] = acc;
    __syncthreads();
    const size_t ih = (size_t)i * a.nh + h;
    int64_t t = 0;
    if (tid < hd) {
        for (int q = 0; q < groups; q++) t = wadd(t, part[q * hd + tid]);
        t = sumc > 0 ? t : 0;
        a.hout[ih * hd + tid] = t;
    }
    const int64_t pm = block_max_4w(magnitude(t), red);
    if (tid == 0) {
        a.hmax[ih] = pm;
        a.fac[ih] = sumc > 0 ? sc_mul(rec_sc(a.vs), from_ratio(1, (u128)(uint64_t)sumc)) : Sc{0, 0};
    }
}

__global__ __launch_bounds__(RD_THREADS) void rp_fold_kernel(RdPrefill a) {
    __shared__ uint64_t redk[3 * RD_THREADS / 16];
    __shared__ int64_t red[RD_WAVES];
    Sc common;
    int64_t gmax;
    scale_fold<RD_THREADS>(a.fac, a.hmax, a.T * a.nh, redk, red, common, gmax, [&](int r, Sc f) {
        int64_t b = 0;
        for (int d = 0; d < a.hd; d++) b = max64(b, iabs(sc_apply(f, a.hout[(size_t)r * a.hd + d])));
        return b;
    });
    if (threadIdx.x == 0) *a.common = common, *a.gmax = (uint64_t)gmax;
}

__global__ __launch_bounds__(256) void rp_out_kernel(RdPrefill a) {  // a wave per (row, head)
    const int64_t gmax = (int64_t)*a.gmax;
    const RqDen rd_gmax = rq_den(gmax);
    const Sc common = uni(*a.common);
    const bool live = common.mant != 0 && gmax > 0;
    const int ih = (int)blockIdx.x * 4 + wave_id();
    if (ih < a.T * a.nh) {  // the whole wave
        const Sc f = live ? sc_mul(uni(a.fac[ih]), sc_recip(common)) : Sc{0, 0};
        const size_t at = (size_t)ih * a.hd;
        for (int d = threadIdx.x & 63; d < a.hd; d += 64)
            a.o[at + d] = live ? rq_apply(rd_gmax, sc_apply(f, a.hout[at + d])) : 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        put_rec(a.os, live ? sc_mul(from_ratio((u128)(uint64_t)gmax, (u128)ACT_LEVELS), common) : Sc{0, 0});
}

// argmax_codes (generate.rs:48-56): *token = the first index of the largest of n codes. With record non-null the
// codes go to record + step * n and the scale to rscale[step], and *step advances (the per-step logits the
// generation hash covers) -- only while step lies in [0, cap), the rows record and rscale hold; any other step
// records nothing and stays where it is (the token is still chosen).
__global__ __launch_bounds__(RD_THREADS) void rd_argmax_kernel(const int32_t* __restrict__ logits, int n,
                                                               const kt_hip_qscale* __restrict__ ls,
                                                               int32_t* __restrict__ token, int32_t* record,
                                                               kt_hip_sscale* rscale, int32_t* step, int cap) {
    __shared__ int64_t red[RD_WAVES];
    // key: the value in the high word, the inverted index in the low word (the lower index wins a tie)
    auto key = [](int32_t v, int i) { return (int64_t)v * 4294967296LL + (int64_t)(0x7FFFFFFF - i); };
    int64_t best = INT64_MIN;
    const int s = record ? *step : 0;
    const bool keep = record && s >= 0 && s < cap;
    int32_t* rec = keep ? record + (size_t)s * n : nullptr;
    // one pass over the codes, 16-byte loads (and stores into the record) where n and the addresses allow, several in
    // flight per thread
    const bool vec = n % 4 == 0 && ((uintptr_t)logits & 15) == 0 && (!rec || ((uintptr_t)rec & 15) == 0);
    if (vec) {
        const int n4 = n / 4;
        const int4* l4 = reinterpret_cast<const int4*>(logits);
        constexpr int U = 4;
        for (int i0 = threadIdx.x; i0 < n4; i0 += U * RD_THREADS) {
            int4 v[U];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = i0 + u * RD_THREADS < n4 ? l4[i0 + u * RD_THREADS] : int4{0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = i0 + u * RD_THREADS;
                if (i >= n4) break;
                if (rec) reinterpret_cast<int4*>(rec)[i] = v[u];
                const int64_t k0 = key(v[u].x, 4 * i), k1 = key(v[u].y, 4 * i + 1);
                const int64_t k2 = key(v[u].z, 4 * i + 2), k3 = key(v[u].w, 4 * i + 3);
                const int64_t a = k0 > k1 ? k0 : k1, b = k2 > k3 ? k2 : k3, c = a > b ? a : b;
                best = c > best ? c : best;
            }
        }
    } else {
        for (int i = threadIdx.x; i < n; i += RD_THREADS) {
            const int32_t v = logits[i];
            if (rec) rec[i] = v;
            const int64_t k = key(v, i);
            best = k > best ? k : best;
        }
    }
    best = block_max_i64(best, red);  // every thread has read *step past here
    if (threadIdx.x == 0) {
        if (keep) {
            rscale[s] = kt_hip_sscale{ls->mant, ls->shift, 1};
            *step = s + 1;
        }
        *token = 0x7FFFFFFF - (int32_t)(uint32_t)(best & 0xFFFFFFFF);
    }
}

// The attention step's LDS with hb heads' scores held at once: the per-step factors, hb score rows, the head
// outputs and the rotated q. hb = 1 is the least it runs with.
size_t rd_attention_lds(int max_seq, int nh, int hd, int hb) {
    return (size_t)max_seq * (2 * sizeof(Sc) + 8 * (size_t)hb) + (size_t)nh * hd * (8 + 4);
}
// The dynamic LDS the attention step may take on the current device: KT_REF_ATTN_LDS, less what the device's
// per-block limit leaves after the kernel's static LDS.
static size_t rd_attention_budget() {
    int dev = 0, mx = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&mx, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
        return 0;
    hipFuncAttributes fa{};
    if (hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(&rd_attention_step_kernel)) != hipSuccess ||
        fa.sharedSizeBytes >= (size_t)mx)
        return 0;
    const size_t room = (size_t)mx - fa.sharedSizeBytes;
    return room < KT_REF_ATTN_LDS ? room : KT_REF_ATTN_LDS;
}
static int rd_attention_hb(int max_seq, int nh, int hd, size_t budget) {
    const size_t base = rd_attention_lds(max_seq, nh, hd, 0);
    if (base >= budget) return 0;
    const size_t hb = (budget - base) / (8 * (size_t)max_seq);
    return (int)(hb < (size_t)nh ? hb : (size_t)nh);
}

hipError_t launch_rd_embed(const int32_t* emb, int64_t e_mant, int32_t e_shift, const int32_t* token, int vocab,
                           int dim, int32_t* y, kt_hip_qscale* ys, hipStream_t s) {
    rd_embed_kernel<<<1, RD_THREADS, 0, s>>>(emb, e_mant, e_shift, token, vocab, dim, y, ys);
    return hipGetLastError();
}
hipError_t launch_rd_rmsnorm(const int32_t* x, int rows, int dim, const kt_hip_qscale* xs, const int32_t* g,
                             int64_t g_mant, int32_t g_shift, int64_t e_mant, int32_t e_shift, int32_t* y,
                             kt_hip_qscale* ys, hipStream_t s) {
    if (rows < 1 || rows > RD_MAX_ROWS) return hipErrorInvalidValue;
    rd_rmsnorm_kernel<<<1, RD_THREADS, 0, s>>>(x, rows, dim, xs, g, g_mant, g_shift, e_mant, e_shift, y, ys);
    return hipGetLastError();
}
hipError_t launch_rd_add(const int32_t* a, const kt_hip_qscale* as, const int32_t* b, const kt_hip_qscale* bs, int n,
                         int32_t* y, kt_hip_qscale* ys, hipStream_t s) {
    rd_add_kernel<<<1, RD_THREADS, 0, s>>>(a, as, b, bs, n, y, ys);
    return hipGetLastError();
}
hipError_t launch_rd_add_norm(const int32_t* a, const kt_hip_qscale* as, const int32_t* b, const kt_hip_qscale* bs,
                              int n, int32_t* y, kt_hip_qscale* ys, const int32_t* g, int64_t g_mant, int32_t g_shift,
                              int64_t e_mant, int32_t e_shift, int32_t* h, kt_hip_qscale* hs, hipStream_t s) {
    const auto kernel = n <= RD_THREADS ? rd_add_norm_kernel<false, 1> : rd_add_norm_kernel<false, RD_AN>;
    kernel<<<1, RD_THREADS, 0, s>>>(a, as, b, bs, RqSums{}, n, y, ys, g, g_mant, g_shift, e_mant, e_shift, h, hs);
    return hipGetLastError();
}
hipError_t launch_rd_swiglu(const int32_t* g, const kt_hip_qscale* gs, const int32_t* u, const kt_hip_qscale* us,
                            int rows, int n, const int64_t* codes, const kt_hip_codelut* lut, int32_t* h,
                            kt_hip_qscale* hs, hipStream_t s) {
    rd_swiglu_kernel<false><<<(unsigned)rows, RD_THREADS, 0, s>>>(g, gs, u, us, RqSums{}, RqSums{}, n, codes, *lut, h,
                                                                  hs);
    return hipGetLastError();
}
hipError_t launch_rd_gelu(const int32_t* x, const kt_hip_qscale* xs, int64_t n, const int64_t* codes,
                          const kt_hip_codelut* lut, int32_t* y, kt_hip_qscale* ys, hipStream_t s) {
    const int64_t per = (int64_t)RD_THREADS * 4;
    const int64_t g = (n + per - 1) / per;
    rd_gelu_kernel<<<(unsigned)(g < 1 ? 1 : (g > 4096 ? 4096 : g)), RD_THREADS, 0, s>>>(x, xs, n, codes, *lut, y, ys);
    return hipGetLastError();
}
// With a workspace: the heads kernel (L.parts CTAs per q head) and the combine. Without: the one-CTA kernel, its LDS
// holding at least one head's scores at max_seq positions (the entry point checks which applies).
hipError_t launch_rd_attention_step(const RdAttn& a_in, hipStream_t s) {
    RdAttn a = a_in;
    if (a.ws) {
        const RdHeadsLayout L = rd_heads_layout(a.max_seq, a.nh, a.hd);
        const size_t qk = rd_round256((size_t)2 * a.hd * sizeof(int32_t)), lds = qk + L.arr_stride;
        if (lds <= RD_HEADS_LDS)
            a.sums ? rd_attention_heads_kernel<false, true><<<(unsigned)(a.nh * L.parts), RD_THREADS, lds, s>>>(a, L)
                   : rd_attention_heads_kernel<false, false><<<(unsigned)(a.nh * L.parts), RD_THREADS, lds, s>>>(a, L);
        else
            a.sums ? rd_attention_heads_kernel<true, true><<<(unsigned)(a.nh * L.parts), RD_THREADS, qk, s>>>(a, L)
                   : rd_attention_heads_kernel<true, false><<<(unsigned)(a.nh * L.parts), RD_THREADS, qk, s>>>(a, L);
        rd_attention_combine_kernel<<<1, RD_THREADS, 0, s>>>(a, L);
        return hipGetLastError();
    }
    const size_t budget = rd_attention_budget();
    a.hb = rd_attention_hb(a.max_seq, a.nh, a.hd, budget);
    if (a.hb < 1) return hipErrorInvalidValue;
    rd_attention_step_kernel<<<1, RD_THREADS, rd_attention_lds(a.max_seq, a.nh, a.hd, a.hb), s>>>(a);
    return hipGetLastError();
}
size_t rd_seq_workspace(int64_t rows) {
    return (sizeof(RdSeqWs) + (size_t)rows * (sizeof(Sc) + sizeof(int64_t)) + 255) / 256 * 256;
}

hipError_t launch_rd_seq(const RdSeq& q, hipStream_t s) {
    if (q.op == RS_NORM) {
        const unsigned grid = (unsigned)(q.rows < 1024 ? q.rows : 1024);
        rs_rows_kernel<<<(unsigned)((q.rows + 3) / 4), 256, 0, s>>>(q);
        if (q.rows <= RS_FOLD_ROWS) {
            rs_norm_out_kernel<true><<<grid, 256, 0, s>>>(q);
        } else {
            rs_norm_fold_kernel<<<1, RD_THREADS, 0, s>>>(q);
            rs_norm_out_kernel<false><<<grid, 256, 0, s>>>(q);
        }
        return hipGetLastError();
    }
    const int64_t g = (q.n + 255) / 256, g4 = (q.n + 1023) / 1024;
    const unsigned grid = (unsigned)(g > 2048 ? 2048 : g), parts = (unsigned)(g4 > RS_PARTS ? RS_PARTS : g4);  // n >= 1
    if (q.op == RS_ADD) {
        rs_max_kernel<RS_ADD><<<parts, 256, 0, s>>>(q);
        rs_out_kernel<RS_ADD><<<grid, 256, 0, s>>>(q, (int)parts);
    } else {
        rs_max_kernel<RS_SWIGLU><<<parts, 256, 0, s>>>(q);
        rs_out_kernel<RS_SWIGLU><<<grid, 256, 0, s>>>(q, (int)parts);
    }
    return hipGetLastError();
}

hipError_t launch_rd_embed_seq(const int32_t* emb, int64_t e_mant, int32_t e_shift, const int32_t* tokens, int T,
                               int vocab, int dim, int32_t* y, kt_hip_qscale* ys, hipStream_t s) {
    const int64_t g = ((int64_t)T * dim + 255) / 256;
    rd_embed_seq_kernel<<<(unsigned)(g < 1 ? 1 : (g > 4096 ? 4096 : g)), 256, 0, s>>>(emb, e_mant, e_shift, tokens,
                                                                                     T, vocab, dim, y, ys);
    return hipGetLastError();
}

// The prefill attention's workspace: rotated q and k, the head sums, their largest magnitudes, the scales, gmax and
// the common scale, each part 256-byte aligned.
size_t rd_prefill_workspace(int64_t T, int64_t nh, int64_t nkv, int64_t hd, size_t off[7]) {
    const size_t sizes[7] = {(size_t)(T * nh * hd * 4), (size_t)(T * nkv * hd * 4), (size_t)(nh * T * hd * 8),
                             (size_t)(nh * T * 8), (size_t)(T * nh) * sizeof(Sc), 8, sizeof(Sc)};
    size_t at = 0;
    for (int i = 0; i < 7; i++) {
        off[i] = at;
        at += (sizes[i] + 255) / 256 * 256;
    }
    return at;
}

hipError_t launch_rd_attention_prefill(RdPrefill a, void* ws, hipStream_t s) {
    size_t off[7];
    rd_prefill_workspace(a.T, a.nh, a.nkv, a.hd, off);
    char* b = (char*)ws;
    a.qd = (int32_t*)(b + off[0]), a.kd = (int32_t*)(b + off[1]), a.hout = (int64_t*)(b + off[2]);
    a.hmax = (int64_t*)(b + off[3]), a.fac = (Sc*)(b + off[4]), a.gmax = (uint64_t*)(b + off[5]);
    a.common = (Sc*)(b + off[6]);
    rp_rope_kernel<<<(unsigned)a.T, 256, 0, s>>>(a);
    // R rows of dots in 64 KB of LDS: 4 rows up to 2048 positions, one beyond
    const unsigned ctas4 = (unsigned)((a.T + 3) / 4 * a.nh), ctas1 = (unsigned)(a.T * a.nh);
    const size_t lds = (size_t)a.T * 8;
    const bool four = a.T <= 2048;
    if (a.hd == 64) {
        if (four) rp_head_kernel<64, 4><<<ctas4, 256, 4 * lds, s>>>(a);
        else rp_head_kernel<64, 1><<<ctas1, 256, lds, s>>>(a);
    } else if (a.hd == 128) {
        if (four) rp_head_kernel<128, 4><<<ctas4, 256, 4 * lds, s>>>(a);
        else rp_head_kernel<128, 1><<<ctas1, 256, lds, s>>>(a);
    } else {
        rp_head_any_kernel<<<ctas1, 256, lds, s>>>(a);
    }
    rp_fold_kernel<<<1, RD_THREADS, 0, s>>>(a);
    rp_out_kernel<<<(unsigned)((a.T * a.nh + 3) / 4), 256, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_rd_argmax(const int32_t* logits, int n, const kt_hip_qscale* ls, int32_t* token, int32_t* record,
                            kt_hip_sscale* rscale, int32_t* step, int cap, hipStream_t s) {
    rd_argmax_kernel<<<1, RD_THREADS, 0, s>>>(logits, n, ls, token, record, rscale, step, cap);
    return hipGetLastError();
}

}  // namespace kt


// ---------------------------------------------------------------------------------------------------------------
// C ABI (include/kt_hip.h): argument checks on the host, then one launch on `stream`.
// ---------------------------------------------------------------------------------------------------------------
#define RD_TRY(x)                               \
    do {                                        \
        const hipError_t e_ = (x);              \
        if (e_ != hipSuccess) return (int)e_;   \
    } while (0)

static const int64_t RD_MAX_N = (int64_t)1 << 30;

extern "C" int kt_hip_ref_embed(int dev, const int32_t* emb_dev, int64_t e_mant, int32_t e_shift,
                                const int32_t* token_dev, int64_t vocab, int64_t dim, int32_t* y_dev,
                                kt_hip_qscale* ys_dev, void* stream) {
    if (!emb_dev || !token_dev || !y_dev || !ys_dev || vocab < 1 || dim < 1 || vocab > INT32_MAX ||
        vocab * dim > ((int64_t)1 << 40) || dim > RD_MAX_N || e_mant < 0)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_embed(emb_dev, e_mant, e_shift, token_dev, (int)vocab, (int)dim, y_dev, ys_dev,
                                    (hipStream_t)stream);
}

extern "C" int kt_hip_ref_embed_seq(int dev, const int32_t* emb_dev, int64_t e_mant, int32_t e_shift,
                                    const int32_t* tokens_dev, int64_t T, int64_t vocab, int64_t dim, int32_t* y_dev,
                                    kt_hip_qscale* ys_dev, void* stream) {
    if (!emb_dev || !tokens_dev || !y_dev || !ys_dev || T < 1 || vocab < 1 || dim < 1 || vocab > INT32_MAX ||
        T > INT32_MAX || dim > INT32_MAX || T * dim > RD_MAX_N || e_mant < 0)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_embed_seq(emb_dev, e_mant, e_shift, tokens_dev, (int)T, (int)vocab, (int)dim, y_dev,
                                        ys_dev, (hipStream_t)stream);
}

extern "C" size_t kt_hip_ref_seq_workspace(int64_t rows) {
    return rows < 1 || rows > INT32_MAX ? 0 : kt::rd_seq_workspace(rows);
}

static int rd_seq_call(int dev, const kt::RdSeq& q, size_t ws_bytes, void* stream) {
    if (!q.a || !q.b || !q.as || !q.y || !q.ys || !q.ws || q.n < 1 || q.n > RD_MAX_N ||
        ws_bytes < kt::rd_seq_workspace(q.rows))
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_seq(q, (hipStream_t)stream);
}

extern "C" int kt_hip_ref_add_seq(int dev, const int32_t* a_dev, const kt_hip_qscale* as_dev, const int32_t* b_dev,
                                  const kt_hip_qscale* bs_dev, int64_t n, void* ws_dev, size_t ws_bytes,
                                  int32_t* y_dev, kt_hip_qscale* ys_dev, void* stream) {
    kt::RdSeq q{};
    q.op = kt::RS_ADD, q.a = a_dev, q.b = b_dev, q.as = as_dev, q.bs = bs_dev, q.n = n, q.rows = 1, q.dim = 1;
    q.ws = (kt::RdSeqWs*)ws_dev, q.y = y_dev, q.ys = ys_dev;
    if (!bs_dev) return (int)hipErrorInvalidValue;
    return rd_seq_call(dev, q, ws_bytes, stream);
}

extern "C" int kt_hip_ref_swiglu_seq(int dev, const int32_t* g_dev, const kt_hip_qscale* gs_dev, const int32_t* u_dev,
                                     const kt_hip_qscale* us_dev, int64_t n, const int64_t* silu_codes_dev,
                                     const kt_hip_codelut* silu, void* ws_dev, size_t ws_bytes, int32_t* h_dev,
                                     kt_hip_qscale* hs_dev, void* stream) {
    if (!silu || !silu_codes_dev || !us_dev || silu->n < 1 || !silu->right_identity) return (int)hipErrorInvalidValue;
    kt::RdSeq q{};
    q.op = kt::RS_SWIGLU, q.a = g_dev, q.b = u_dev, q.as = gs_dev, q.bs = us_dev, q.n = n, q.rows = 1, q.dim = 1;
    q.codes = silu_codes_dev, q.lut = *silu, q.ws = (kt::RdSeqWs*)ws_dev, q.y = h_dev, q.ys = hs_dev;
    return rd_seq_call(dev, q, ws_bytes, stream);
}

extern "C" int kt_hip_ref_rmsnorm_seq(int dev, const int32_t* x_dev, const kt_hip_qscale* xs_dev, int64_t rows,
                                      int64_t dim, const int32_t* g_dev, int64_t g_mant, int32_t g_shift,
                                      int64_t eps_mant, int32_t eps_shift, void* ws_dev, size_t ws_bytes,
                                      int32_t* y_dev, kt_hip_qscale* ys_dev, void* stream) {
    if (rows < 1 || dim < 1 || rows > INT32_MAX || dim > INT32_MAX || rows * dim > RD_MAX_N || g_mant < 0 ||
        eps_mant < 0)
        return (int)hipErrorInvalidValue;
    kt::RdSeq q{};
    q.op = kt::RS_NORM, q.a = x_dev, q.b = g_dev, q.as = xs_dev, q.n = rows * dim, q.rows = (int)rows;
    q.dim = (int)dim, q.g_mant = g_mant, q.g_shift = g_shift, q.e_mant = eps_mant, q.e_shift = eps_shift;
    q.ws = (kt::RdSeqWs*)ws_dev, q.y = y_dev, q.ys = ys_dev;
    return rd_seq_call(dev, q, ws_bytes, stream);
}

extern "C" size_t kt_hip_ref_attention_prefill_workspace(int64_t T, int64_t nh, int64_t nkv, int64_t hd) {
    if (T < 1 || nh < 1 || nkv < 1 || hd < 2 || T > 8192 || nh > KT_REF_MAX_HEADS || hd > 256) return 0;
    size_t off[7];
    return kt::rd_prefill_workspace(T, nh, nkv, hd, off);
}

extern "C" int kt_hip_ref_attention_prefill(int dev, const int32_t* q_dev, const kt_hip_qscale* qs_dev,
                                            const int32_t* k_dev, const kt_hip_qscale* ks_dev, const int32_t* v_dev,
                                            const kt_hip_qscale* vs_dev, int64_t T, int64_t nh, int64_t nkv,
                                            int64_t hd, int64_t max_seq, const kt_hip_sscale* cos_dev,
                                            const kt_hip_sscale* sin_dev, int64_t isq_mant, int32_t isq_shift,
                                            const int64_t* exp_codes_dev, const kt_hip_codelut* exp_lut,
                                            void* ws_dev, size_t ws_bytes, int32_t* o_dev, kt_hip_qscale* os_dev,
                                            void* stream) {
    const size_t need = kt_hip_ref_attention_prefill_workspace(T, nh, nkv, hd);
    if (!q_dev || !qs_dev || !k_dev || !ks_dev || !v_dev || !vs_dev || !cos_dev || !sin_dev || !exp_codes_dev ||
        !exp_lut || !ws_dev || !o_dev || !os_dev || need == 0 || ws_bytes < need || T > max_seq || nh % nkv ||
        (hd & 1) || exp_lut->n < 1 || isq_mant < 0)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    kt::RdPrefill a{};
    a.q = q_dev, a.k = k_dev, a.v = v_dev, a.qs = qs_dev, a.ks = ks_dev, a.vs = vs_dev;
    a.T = (int)T, a.nh = (int)nh, a.nkv = (int)nkv, a.hd = (int)hd, a.cos = cos_dev, a.sin = sin_dev;
    a.isq_mant = isq_mant, a.isq_shift = isq_shift, a.exp_codes = exp_codes_dev, a.exp = *exp_lut;
    a.o = o_dev, a.os = os_dev;
    return (int)kt::launch_rd_attention_prefill(a, ws_dev, (hipStream_t)stream);
}

extern "C" int kt_hip_ref_rmsnorm(int dev, const int32_t* x_dev, const kt_hip_qscale* xs_dev, int64_t rows,
                                  int64_t dim, const int32_t* g_dev, int64_t g_mant, int32_t g_shift,
                                  int64_t eps_mant, int32_t eps_shift, int32_t* y_dev, kt_hip_qscale* ys_dev,
                                  void* stream) {
    if (!x_dev || !xs_dev || !g_dev || !y_dev || !ys_dev || rows < 1 || dim < 1 || rows * dim > RD_MAX_N ||
        g_mant < 0 || eps_mant < 0)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_rmsnorm(x_dev, (int)rows, (int)dim, xs_dev, g_dev, g_mant, g_shift, eps_mant, eps_shift,
                                      y_dev, ys_dev, (hipStream_t)stream);
}

extern "C" int kt_hip_ref_add(int dev, const int32_t* a_dev, const kt_hip_qscale* as_dev, const int32_t* b_dev,
                              const kt_hip_qscale* bs_dev, int64_t n, int32_t* y_dev, kt_hip_qscale* ys_dev,
                              void* stream) {
    if (!a_dev || !as_dev || !b_dev || !bs_dev || !y_dev || !ys_dev || n < 1 || n > RD_MAX_N)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_add(a_dev, as_dev, b_dev, bs_dev, (int)n, y_dev, ys_dev, (hipStream_t)stream);
}

extern "C" int kt_hip_ref_add_rmsnorm(int dev, const int32_t* a_dev, const kt_hip_qscale* as_dev,
                                      const int32_t* b_dev, const kt_hip_qscale* bs_dev, int64_t n, int32_t* y_dev,
                                      kt_hip_qscale* ys_dev, const int32_t* g_dev, int64_t g_mant, int32_t g_shift,
                                      int64_t eps_mant, int32_t eps_shift, int32_t* h_dev, kt_hip_qscale* hs_dev,
                                      void* stream) {
    if (!a_dev || !as_dev || !b_dev || !bs_dev || !y_dev || !ys_dev || !g_dev || !h_dev || !hs_dev || n < 1 ||
        n > (int64_t)kt::RD_THREADS * kt::RD_AN || g_mant < 0 || eps_mant < 0 || h_dev == y_dev || h_dev == a_dev ||
        h_dev == b_dev || (void*)hs_dev == (void*)ys_dev)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_add_norm(a_dev, as_dev, b_dev, bs_dev, (int)n, y_dev, ys_dev, g_dev, g_mant, g_shift,
                                       eps_mant, eps_shift, h_dev, hs_dev, (hipStream_t)stream);
}

// The device view of one call's output of kt_hip_quant_linear_multi_sums (its workspace parts as ql_workspace_bytes
// lays them out at one row); false for a malformed description or one of other than n values.
static bool rq_sums_of(const kt_hip_ql_sums* d, int64_t n, kt::RqSums* r) {
    if (!d || !d->ws || d->seg < 0 || d->seg >= KT_QL_MAX_SEGMENTS || d->in_f < 1 || d->out_f < 1 || d->col0 < 0 ||
        d->n != n || d->col0 + d->n > d->out_f || (reinterpret_cast<uintptr_t>(d->ws) & 15))
        return false;
    size_t off[KT_QL_WS_PARTS];
    kt::ql_workspace_bytes(1, d->in_f, d->out_f, off);
    const char* base = static_cast<const char*>(d->ws);
    r->acc = reinterpret_cast<const int64_t*>(base + off[1]) + d->col0;
    r->st = reinterpret_cast<const kt::QlState*>(base + off[4]) + d->seg;
    r->rec = d->rec;
    return true;
}

extern "C" int kt_hip_ref_add_rmsnorm_sums(int dev, const int32_t* a_dev, const kt_hip_qscale* as_dev,
                                           const kt_hip_ql_sums* b, int64_t n, int32_t* y_dev, kt_hip_qscale* ys_dev,
                                           const int32_t* g_dev, int64_t g_mant, int32_t g_shift, int64_t eps_mant,
                                           int32_t eps_shift, int32_t* h_dev, kt_hip_qscale* hs_dev, void* stream) {
    kt::RqSums bs{};
    if (!a_dev || !as_dev || !y_dev || !ys_dev || !g_dev || !h_dev || !hs_dev || n < 1 ||
        n > (int64_t)kt::RD_THREADS * kt::RD_AN || g_mant < 0 || eps_mant < 0 || h_dev == y_dev || h_dev == a_dev ||
        (void*)hs_dev == (void*)ys_dev || !rq_sums_of(b, n, &bs) || bs.rec == as_dev || bs.rec == ys_dev ||
        bs.rec == hs_dev)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    const auto kernel = n <= kt::RD_THREADS ? kt::rd_add_norm_kernel<true, 1> : kt::rd_add_norm_kernel<true, kt::RD_AN>;
    kernel<<<1, kt::RD_THREADS, 0, (hipStream_t)stream>>>(
        a_dev, as_dev, nullptr, nullptr, bs, (int)n, y_dev, ys_dev, g_dev, g_mant, g_shift, eps_mant, eps_shift, h_dev,
        hs_dev);
    return (int)hipGetLastError();
}

extern "C" int kt_hip_ref_swiglu_sums(int dev, const kt_hip_ql_sums* g, const kt_hip_ql_sums* u, int64_t n,
                                      const int64_t* silu_codes_dev, const kt_hip_codelut* silu, int32_t* h_dev,
                                      kt_hip_qscale* hs_dev, void* stream) {
    kt::RqSums gs{}, us{};
    if (!silu_codes_dev || !silu || !h_dev || !hs_dev || n < 1 || n > (int64_t)kt::RD_THREADS * 8 || silu->n < 1 ||
        !silu->right_identity || !rq_sums_of(g, n, &gs) || !rq_sums_of(u, n, &us) || gs.rec == hs_dev ||
        us.rec == hs_dev || (gs.rec && gs.rec == us.rec))
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    kt::rd_swiglu_kernel<true><<<1, kt::RD_THREADS, 0, (hipStream_t)stream>>>(
        nullptr, nullptr, nullptr, nullptr, gs, us, (int)n, silu_codes_dev, *silu, h_dev, hs_dev);
    return (int)hipGetLastError();
}

// The workspace: the down product's (kt_hip_quant_linear_workspace of one row), then the products, their partial maxima
// and their Scale.
static size_t rd_swiglu_ws(int64_t n, int64_t out, size_t off[3]) {
    size_t ql[KT_QL_WS_PARTS];
    const size_t parts = (size_t)(n + kt::RD_SPLIT - 1) / kt::RD_SPLIT;
    size_t at = kt::ql_workspace_bytes(1, n, out, ql);
    const size_t sizes[3] = {(size_t)n * 8, parts * 8, sizeof(kt_hip_qscale)};
    for (int i = 0; i < 3; i++) {
        off[i] = at;
        at += kt::rd_round256(sizes[i]);
    }
    return at;
}

extern "C" size_t kt_hip_quant_linear_swiglu_workspace(int64_t n, int64_t out_f, int pw) {
    size_t off[3];
    return kt_hip_quant_linear_sums_ok(n, out_f, pw) ? rd_swiglu_ws(n, out_f, off) : 0;
}

extern "C" int kt_hip_quant_linear_swiglu_sums(int dev, const kt_hip_ql_sums* g, const kt_hip_ql_sums* u, int64_t n,
                                               const int64_t* silu_codes_dev, const kt_hip_codelut* silu,
                                               const int8_t* w_planes_dev, int pw, int64_t out_f, int64_t w_mant,
                                               int32_t w_shift, void* ws_dev, size_t ws_bytes, void* stream) {
    kt::RqSums gs{}, us{};
    if (!silu_codes_dev || !silu || !w_planes_dev || !ws_dev || n < 1 || w_mant < 0 || silu->n < 1 ||
        !silu->right_identity || !rq_sums_of(g, n, &gs) || !rq_sums_of(u, n, &us) || (gs.rec && gs.rec == us.rec) ||
        ws_dev == g->ws || ws_dev == u->ws || (reinterpret_cast<uintptr_t>(ws_dev) & 15))
        return (int)hipErrorInvalidValue;
    const size_t need = kt_hip_quant_linear_swiglu_workspace(n, out_f, pw);
    if (need == 0 || ws_bytes < need) return (int)hipErrorInvalidValue;
    // the maxima come from the slots of g's and u's product, one per 8 columns: the outputs are whole slots (as the
    // product's boundaries are), of a row whose CTAs have 8 columns
    const int64_t cols = kt::ql_skinny_cols(g->in_f, g->out_f);
    const kt_hip_ql_sums* d[2] = {g, u};
    const int64_t* part[2];
    for (int i = 0; i < 2; i++) {
        if (d[i]->col0 % 8 || (d[i]->n % 8 && d[i]->col0 + d[i]->n != d[i]->out_f) ||
            kt::ql_skinny_cols(d[i]->in_f, d[i]->out_f) != cols)
            return (int)hipErrorInvalidValue;
        size_t off[KT_QL_WS_PARTS];
        kt::ql_workspace_bytes(1, d[i]->in_f, d[i]->out_f, off);
        part[i] = reinterpret_cast<const int64_t*>(static_cast<const char*>(d[i]->ws) + off[2]) + d[i]->col0 / cols;
    }
    RD_TRY(hipSetDevice(dev));
    size_t off[3];
    rd_swiglu_ws(n, out_f, off);
    char* base = static_cast<char*>(ws_dev);
    int64_t *hv = reinterpret_cast<int64_t*>(base + off[0]), *hp = reinterpret_cast<int64_t*>(base + off[1]);
    kt_hip_qscale* scale = reinterpret_cast<kt_hip_qscale*>(base + off[2]);
    const int ctas = (int)((n + kt::RD_SPLIT - 1) / kt::RD_SPLIT);
    kt::rd_swiglu_split_kernel<<<ctas, kt::RD_SPLIT, 0, (hipStream_t)stream>>>(
        gs, us, part[0], part[1], (int)((n + cols - 1) / cols), (int)n, silu_codes_dev, *silu, hv, hp, scale);
    RD_TRY(hipGetLastError());
    return (int)kt::launch_quant_linear_hv(kt::QlHv{hv, hp, ctas, scale}, n, w_planes_dev, pw, out_f, w_mant, w_shift,
                                           kt_hip_flush_k(3, pw), ws_dev, (hipStream_t)stream);
}

extern "C" int kt_hip_ref_swiglu(int dev, const int32_t* g_dev, const kt_hip_qscale* gs_dev, const int32_t* u_dev,
                                 const kt_hip_qscale* us_dev, int64_t rows, int64_t n, const int64_t* silu_codes_dev,
                                 const kt_hip_codelut* silu, int32_t* h_dev, kt_hip_qscale* hs_dev, void* stream) {
    if (!g_dev || !gs_dev || !u_dev || !us_dev || !silu_codes_dev || !silu || !h_dev || !hs_dev || rows < 1 ||
        rows > INT32_MAX || n < 1 || n > RD_MAX_N || silu->n < 1 || !silu->right_identity)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_swiglu(g_dev, gs_dev, u_dev, us_dev, (int)rows, (int)n, silu_codes_dev, silu, h_dev,
                                     hs_dev, (hipStream_t)stream);
}

extern "C" int kt_hip_ref_gelu(int dev, const int32_t* x_dev, const kt_hip_qscale* xs_dev, int64_t n,
                               const int64_t* gelu_codes_dev, const kt_hip_codelut* gelu, int32_t* y_dev,
                               kt_hip_qscale* ys_dev, void* stream) {
    if (!x_dev || !xs_dev || !gelu_codes_dev || !gelu || !y_dev || !ys_dev || n < 1 || gelu->n < 1 ||
        !gelu->right_identity || (const void*)ys_dev == (const void*)xs_dev)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_gelu(x_dev, xs_dev, n, gelu_codes_dev, gelu, y_dev, ys_dev, (hipStream_t)stream);
}

extern "C" size_t kt_hip_ref_conv2d_workspace(int64_t ci, int64_t h, int64_t w, int64_t co, int64_t kh, int64_t kw,
                                              int64_t stride, int64_t pad) {
    if (ci < 1 || h < 1 || w < 1 || co < 1 || kh < 1 || kw < 1 || stride < 1 || pad < 0 || h + 2 * pad < kh ||
        w + 2 * pad < kw)
        return 0;
    const int64_t oh = (h + 2 * pad - kh) / stride + 1, ow = (w + 2 * pad - kw) / stride + 1;
    size_t off[KT_QL_WS_PARTS];
    return kt::ql_workspace_bytes(oh * ow, ci * kh * kw, co, off);
}

extern "C" int kt_hip_ref_conv2d(int dev, const int32_t* x_dev, const kt_hip_qscale* xs_dev, int64_t ci, int64_t h,
                                 int64_t w, const int8_t* w_planes_dev, int pw, int64_t co, int64_t kh, int64_t kw,
                                 int64_t stride, int64_t pad, int64_t w_mant, int32_t w_shift,
                                 const int64_t* bias_dev, int64_t b_mant, int32_t b_shift, void* ws_dev,
                                 size_t ws_bytes, int32_t* y_dev, kt_hip_qscale* os_dev, void* stream) {
    if (!x_dev || !xs_dev || !w_planes_dev || !ws_dev || !y_dev || !os_dev || (pw != 1 && pw != 3 && pw != 5) ||
        w_mant < 0 || b_mant < 0)
        return (int)hipErrorInvalidValue;
    const size_t need = kt_hip_ref_conv2d_workspace(ci, h, w, co, kh, kw, stride, pad);
    if (need == 0 || ws_bytes < need || ci * h * w >= ((int64_t)1 << 31) || kh >= 65536 || kw >= 65536 ||
        stride >= 65536 || pad >= 65536)  // the gather's pixel arithmetic stays within int32
        return (int)hipErrorInvalidValue;
    const int64_t oh = (h + 2 * pad - kh) / stride + 1, ow = (w + 2 * pad - kw) / stride + 1;
    const int64_t rows = oh * ow, kp = (ci * kh * kw + 63) / 64 * 64;
    if (rows * kp >= ((int64_t)1 << 31) || rows * co >= ((int64_t)1 << 31)) return (int)hipErrorInvalidValue;
    const kt::ConvGeom g{(int32_t)ci, (int32_t)h, (int32_t)w, (int32_t)kh, (int32_t)kw, (int32_t)stride,
                         (int32_t)pad, (int32_t)oh, (int32_t)ow};
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_ref_conv2d(x_dev, g, xs_dev, w_planes_dev, pw, co, w_mant, w_shift, bias_dev, b_mant,
                                      b_shift, kt_hip_flush_k(3, pw), ws_dev, y_dev, os_dev, (hipStream_t)stream);
}

extern "C" size_t kt_hip_ref_attention_step_workspace(int64_t max_seq, int64_t nh, int64_t hd) {
    if (nh < 1 || nh > KT_REF_MAX_HEADS || hd < 2 || hd > 1024 || max_seq < 1 || max_seq > KT_REF_ATTN_MAX_SEQ)
        return 0;
    const kt::RdHeadsLayout L = kt::rd_heads_layout((int)max_seq, (int)nh, (int)hd);
    return L.arr + (size_t)nh * L.parts * L.arr_stride;
}

extern "C" int kt_hip_ref_attention_step_ws(int dev, const int32_t* q_dev, const kt_hip_qscale* qs_dev,
                                            const int32_t* k_dev, const kt_hip_qscale* ks_dev, const int32_t* v_dev,
                                            const kt_hip_qscale* vs_dev, const int32_t* pos_dev, int64_t nh,
                                            int64_t nkv, int64_t hd, int64_t max_seq, int32_t* kc_dev,
                                            int32_t* vc_dev, kt_hip_sscale* kscale_dev, kt_hip_sscale* vscale_dev,
                                            const kt_hip_sscale* cos_dev, const kt_hip_sscale* sin_dev,
                                            int64_t isq_mant, int32_t isq_shift, const int64_t* exp_codes_dev,
                                            const kt_hip_codelut* exp_lut, int32_t* o_dev, kt_hip_qscale* os_dev,
                                            void* ws_dev, size_t ws_bytes, void* stream) {
    if (!q_dev || !qs_dev || !k_dev || !ks_dev || !v_dev || !vs_dev || !pos_dev || !kc_dev || !vc_dev ||
        !kscale_dev || !vscale_dev || !cos_dev || !sin_dev || !exp_codes_dev || !exp_lut || !o_dev || !os_dev)
        return (int)hipErrorInvalidValue;
    if (nh < 1 || nkv < 1 || nh % nkv || nh > KT_REF_MAX_HEADS || hd < 2 || (hd & 1) || hd > 1024 || max_seq < 1 ||
        max_seq > KT_REF_ATTN_MAX_SEQ || exp_lut->n < 1 || isq_mant < 0)
        return (int)hipErrorInvalidValue;
    if (ws_dev ? ((reinterpret_cast<uintptr_t>(ws_dev) & 15) ||
                  ws_bytes < kt_hip_ref_attention_step_workspace(max_seq, nh, hd))
               : kt::rd_attention_lds((int)max_seq, (int)nh, (int)hd, 1) > KT_REF_ATTN_LDS)
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    kt::RdAttn a{};
    a.q = q_dev, a.k = k_dev, a.v = v_dev, a.qs = qs_dev, a.ks = ks_dev, a.vs = vs_dev, a.pos = pos_dev;
    a.nh = (int)nh, a.nkv = (int)nkv, a.hd = (int)hd, a.max_seq = (int)max_seq;
    a.kc = kc_dev, a.vc = vc_dev, a.kscale = kscale_dev, a.vscale = vscale_dev, a.cos = cos_dev, a.sin = sin_dev;
    a.isq_mant = isq_mant, a.isq_shift = isq_shift, a.exp_codes = exp_codes_dev, a.exp = *exp_lut;
    a.o = o_dev, a.os = os_dev, a.ws = (unsigned char*)ws_dev;
    return (int)kt::launch_rd_attention_step(a, (hipStream_t)stream);
}

extern "C" int kt_hip_ref_attention_step_sums(int dev, const kt_hip_ql_sums* q, const kt_hip_ql_sums* k,
                                              const kt_hip_ql_sums* v, const int32_t* pos_dev, int64_t nh,
                                              int64_t nkv, int64_t hd, int64_t max_seq, int32_t* kc_dev,
                                              int32_t* vc_dev, kt_hip_sscale* kscale_dev, kt_hip_sscale* vscale_dev,
                                              const kt_hip_sscale* cos_dev, const kt_hip_sscale* sin_dev,
                                              int64_t isq_mant, int32_t isq_shift, const int64_t* exp_codes_dev,
                                              const kt_hip_codelut* exp_lut, int32_t* o_dev, kt_hip_qscale* os_dev,
                                              void* ws_dev, size_t ws_bytes, void* stream) {
    if (!pos_dev || !kc_dev || !vc_dev || !kscale_dev || !vscale_dev || !cos_dev || !sin_dev || !exp_codes_dev ||
        !exp_lut || !o_dev || !os_dev || !ws_dev)
        return (int)hipErrorInvalidValue;
    if (nh < 1 || nkv < 1 || nh % nkv || nh > KT_REF_MAX_HEADS || hd < 2 || (hd & 1) || hd > 1024 || max_seq < 1 ||
        max_seq > KT_REF_ATTN_MAX_SEQ || exp_lut->n < 1 || isq_mant < 0 ||
        (reinterpret_cast<uintptr_t>(ws_dev) & 15) || ws_bytes < kt_hip_ref_attention_step_workspace(max_seq, nh, hd))
        return (int)hipErrorInvalidValue;
    kt::RdAttn a{};
    if (!rq_sums_of(q, nh * hd, &a.qsum) || !rq_sums_of(k, nkv * hd, &a.ksum) || !rq_sums_of(v, nkv * hd, &a.vsum))
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    a.sums = 1, a.pos = pos_dev;
    a.nh = (int)nh, a.nkv = (int)nkv, a.hd = (int)hd, a.max_seq = (int)max_seq;
    a.kc = kc_dev, a.vc = vc_dev, a.kscale = kscale_dev, a.vscale = vscale_dev, a.cos = cos_dev, a.sin = sin_dev;
    a.isq_mant = isq_mant, a.isq_shift = isq_shift, a.exp_codes = exp_codes_dev, a.exp = *exp_lut;
    a.o = o_dev, a.os = os_dev, a.ws = (unsigned char*)ws_dev;
    return (int)kt::launch_rd_attention_step(a, (hipStream_t)stream);
}

extern "C" int kt_hip_ref_attention_step(int dev, const int32_t* q_dev, const kt_hip_qscale* qs_dev,
                                         const int32_t* k_dev, const kt_hip_qscale* ks_dev, const int32_t* v_dev,
                                         const kt_hip_qscale* vs_dev, const int32_t* pos_dev, int64_t nh,
                                         int64_t nkv, int64_t hd, int64_t max_seq, int32_t* kc_dev, int32_t* vc_dev,
                                         kt_hip_sscale* kscale_dev, kt_hip_sscale* vscale_dev,
                                         const kt_hip_sscale* cos_dev, const kt_hip_sscale* sin_dev,
                                         int64_t isq_mant, int32_t isq_shift, const int64_t* exp_codes_dev,
                                         const kt_hip_codelut* exp_lut, int32_t* o_dev, kt_hip_qscale* os_dev,
                                         void* stream) {
    return kt_hip_ref_attention_step_ws(dev, q_dev, qs_dev, k_dev, ks_dev, v_dev, vs_dev, pos_dev, nh, nkv, hd,
                                        max_seq, kc_dev, vc_dev, kscale_dev, vscale_dev, cos_dev, sin_dev, isq_mant,
                                        isq_shift, exp_codes_dev, exp_lut, o_dev, os_dev, nullptr, 0, stream);
}

extern "C" int kt_hip_ref_argmax(int dev, const int32_t* logits_dev, int64_t n, const kt_hip_qscale* ls_dev,
                                 int32_t* token_dev, int32_t* record_dev, kt_hip_sscale* rscale_dev,
                                 int32_t* step_dev, int64_t record_rows, void* stream) {
    if (!logits_dev || !ls_dev || !token_dev || n < 1 || n > INT32_MAX ||
        (record_dev && (!rscale_dev || !step_dev || record_rows < 1 || record_rows > INT32_MAX)))
        return (int)hipErrorInvalidValue;
    RD_TRY(hipSetDevice(dev));
    return (int)kt::launch_rd_argmax(logits_dev, (int)n, ls_dev, token_dev, record_dev, rscale_dev, step_dev,
                                     record_dev ? (int)record_rows : 0, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------------------------------------------
// Offline tables (host, f64): Scale::from_f64, CodeLut::build, Attention::new's RoPE Scales. No float expression
// here is contracted into a fused multiply-add, so each value is the one the reference's f64 arithmetic gives.
// ---------------------------------------------------------------------------------------------------------------
#pragma clang fp contract(off)

// frexp (kt-int/src/lib.rs:46-60) by bit surgery; x > 0 finite.
static double rd_frexp(double x, int* e) {
    uint64_t bits;
    memcpy(&bits, &x, 8);
    const int ef = (int)((bits >> 52) & 0x7ff);
    if (ef == 0) {
        int e2;
        const double m = rd_frexp(x * 9007199254740992.0, &e2);
        *e = e2 - 53;
        return m;
    }
    *e = ef - 1022;
    const uint64_t mb = (bits & ~(0x7ffULL << 52)) | (1022ULL << 52);
    double m;
    memcpy(&m, &mb, 8);
    return m;
}

extern "C" void kt_hip_ref_scale_from_f64(double x, int64_t* mant, int32_t* shift) {
    *mant = 0, *shift = 0;
    if (!(x > 0.0 && isfinite(x))) return;
    int e;
    const double m = rd_frexp(x, &e);
    *mant = (int64_t)round(m * 2147483648.0);
    *shift = 31 - e;
}

extern "C" int kt_hip_ref_from_reals(const double* real, int64_t n, int64_t levels, int32_t* codes, int64_t* mant,
                                     int32_t* shift) {
    if (!real || !codes || !mant || !shift || n < 0 || levels < 1 || levels > ((int64_t)1 << 30))
        return (int)hipErrorInvalidValue;
    double mx = 0.0;
    for (int64_t i = 0; i < n; i++) {
        if (!isfinite(real[i])) return (int)hipErrorInvalidValue;
        const double a = fabs(real[i]);
        mx = a > mx ? a : mx;
    }
    *mant = 0, *shift = 0;
    if (mx == 0.0) {
        memset(codes, 0, (size_t)n * sizeof(int32_t));
        return 0;
    }
    const double step = mx / (double)levels, inv = (double)levels / mx;
    for (int64_t i = 0; i < n; i++) codes[i] = (int32_t)round(real[i] * inv);  // |value| <= levels
    kt_hip_ref_scale_from_f64(step, mant, shift);
    return 0;
}

// erf by Abramowitz & Stegun 7.1.26 (|error| <= 1.5e-7) and the exact GELU 0.5 x (1 + erf(x / sqrt 2)), in the
// reference's operation order (kt-model-vision/src/nonlin.rs:7-21).
static double rd_erf_as(double x) {
    const double sign = x < 0.0 ? -1.0 : 1.0;
    x = fabs(x);
    const double t = 1.0 / (1.0 + 0.3275911 * x);
    const double p = (((((1.061405429 * t - 1.453152027) * t) + 1.421413741) * t - 0.284496736) * t + 0.254829592);
    return sign * (1.0 - p * t * exp(-x * x));
}
static double rd_gelu_f64(double x) { return 0.5 * x * (1.0 + rd_erf_as(x / 1.4142135623730951)); }

static double rd_lut_fn(int kind, double x) {
    switch (kind) {
        case KT_LUT_EXP:
            return exp(x);
        case KT_LUT_SILU:
            return x / (1.0 + exp(-x));
        case KT_LUT_SIGMOID:
            return 1.0 / (1.0 + exp(-x));
        case KT_LUT_GELU:
            return rd_gelu_f64(x);
        default:
            return 0.0;
    }
}

extern "C" int kt_hip_ref_codelut(int kind, double lo, double hi, int idx_bits, int code_bits, int right_identity,
                                  int64_t* codes, kt_hip_codelut* lut) {
    if (kind < KT_LUT_EXP || kind > KT_LUT_GELU || idx_bits < 1 || idx_bits > 24 || code_bits < 0 ||
        code_bits > 52 || !(hi > lo) || !lut)
        return (int)hipErrorInvalidValue;
    const int64_t n = (int64_t)1 << idx_bits;
    const double k = (double)(1ULL << code_bits);
    if (codes)
        for (int64_t i = 0; i < n; i++) {
            const double x = lo + (hi - lo) * ((double)i / (double)(n - 1));
            codes[i] = (int64_t)round(rd_lut_fn(kind, x) * k);
        }
    const double inv_step = (double)(n - 1) / (hi - lo);
    kt_hip_codelut L{};
    kt_hip_ref_scale_from_f64(inv_step, &L.inv_mant, &L.inv_shift);
    L.n = (int32_t)n;
    L.lo_index = (int64_t)round(lo * inv_step);
    kt_hip_ref_scale_from_f64(1.0 / k, &L.code_mant, &L.code_shift);
    L.right_identity = right_identity;
    *lut = L;
    return 0;
}

extern "C" int kt_hip_ref_rope_tables(int64_t max_seq, int64_t rot_dim, double theta, kt_hip_sscale* cos_tab,
                                      kt_hip_sscale* sin_tab) {
    if (max_seq < 1 || rot_dim < 2 || (rot_dim & 1) || !cos_tab || !sin_tab) return (int)hipErrorInvalidValue;
    const int64_t half = rot_dim / 2;
    for (int64_t p = 0; p < max_seq; p++)
        for (int64_t j = 0; j < half; j++) {
            const double inv_freq = pow(theta, -(2.0 * (double)j) / (double)rot_dim);
            const double ang = (double)p * inv_freq;
            const double c = cos(ang), s = sin(ang);
            kt_hip_sscale& C = cos_tab[p * half + j];
            kt_hip_sscale& S = sin_tab[p * half + j];
            kt_hip_ref_scale_from_f64(fabs(c), &C.mant, &C.shift);
            kt_hip_ref_scale_from_f64(fabs(s), &S.mant, &S.shift);
            C.sign = c < 0.0 ? -1 : 1;
            S.sign = s < 0.0 ? -1 : 1;
        }
    return 0;
}
#pragma clang fp contract(on)
