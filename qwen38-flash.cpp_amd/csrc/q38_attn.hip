// q38_attn.hip — the full-attention verify step on its dense path: the attention half of a
// decoder layer for S verify rows (1..64) of one slot over the slot's KV cache, the cache
// extended by the rows (SelfAttention::forward_verify, src/self_attention.cpp:1450-1720; the
// QSA mask, built only once a context exceeds the indexer budget, :764-766, and the Q8 KV
// cache are not part of this path). A row's checkpoint is the cache prefix up to it, so the
// call writes no state copies.
//
// Seven launches:
//   k_affine_rows    q (each head's D query rows, then its D gate rows), k and v of the S
//                    rows in one launch (q38_affine.hip), rounded to bf16;
//   k_attn_prework   per (row, head): the q / k RMS norms T(w * T(x * inv)), RoPE on the first
//                    R dims with the bf16 cos / sin of position * theta^(-2i / R) formed in
//                    double (:641-679), T(sigmoid(gate)), and the new keys and values written
//                    into the cache at the row's token;
//   k_attn_scores    per (1 or 4 64-token tiles, kv head, up to 64 queries): s = T(T(q . k) *
//                    T(1 / sqrt D)) for every token a query sees (t <= T0 + r) on bf16 MFMA
//                    (exact products, float sums), and per query and 64-token tile the max and
//                    the float sum of exp(s - max);
//   k_attn_stats     per query: the max over its tiles and the sum of the tiles' sums scaled
//                    to it;
//   k_attn_pv        per (token tile, kv head, up to 64 queries, dim slice): p = T(exp(s - max)
//                    / sum) on bf16 MFMA against the tile's values (staged transposed in LDS, 64
//                    tokens at a time), one float partial row per (tile, query);
//   k_attn_combine   per query: the tiles' partials added in a fixed order, rounded, times the
//                    gate, rounded;
//   k_affine_rows    the output projection.
// Tiles start at multiples of their size from token 0, and the P.V tile's size depends on a
// query's token count alone (attn_pv_tokens), so a query's sums do not depend on how many rows
// the call carries: S rows give the bits of S one-row calls.
// Cache layout (q38_attn_cache_bytes): keys [HKV][capacity][D] bf16, then values alike.
#include "q38_device.hpp"
#include "q38_internal.hpp"

namespace q38 {

namespace {

constexpr int kTok = 64;  // tokens per score tile and per P.V sub-tile (16 per wave)
constexpr int kMtMax = 4;  // 16-query M-tiles per workgroup
// Tokens per P.V tile: 128 for queries of up to kPvMid tokens (256 halves the workgroups that
// 4-row calls need at 4K tokens), 256 up to kPvLong and 512 beyond, where a partial row per 128
// tokens costs more traffic than the keys and values. Measured, whole step: 23 rows at 16,500
// tokens 103 us with 256, 114 with 512; at 32,704 tokens 130 and 124.
constexpr int64_t kPvMid = 16384, kPvLong = 24576;
constexpr int attn_pv_tokens(int64_t tokens) {
    return tokens <= kPvMid ? 2 * kTok : tokens <= kPvLong ? 4 * kTok : 8 * kTok;
}
// P.V workgroups below which the dims are split over D / 64 of them (512: 16 rows at 16,000 tokens
// 80 -> 90 us, 64 dims too little work for the p that every slice forms again).
constexpr int64_t kSliceWgs = 256;

__device__ __forceinline__ float tbf(float v) { return bf2f(f2bf(v)); }
__device__ __forceinline__ float sigmoid_bf(float x) { return tbf(1.0f / (1.0f + expf(-x))); }

// Two floats rounded to bf16 (nearest even, as rbf_cvt), packed lo first, in one instruction.
__device__ __forceinline__ uint32_t pack_bf(float lo, float hi) {
    typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
    const bf2_t v = {static_cast<__bf16>(own(lo)), static_cast<__bf16>(own(hi))};
    return __builtin_bit_cast(uint32_t, v);
}
// exp(x) for x <= 0 within one unit in the last place, subnormal results included: 2^(k + f) for
// x log2(e) = k + f with k whole, |f| <= 1/2, and f formed from the two-part log2(e), so that
// only the hardware's 2^f and the last scaling round (the range checks of a general expf are not
// needed; below -150 the result is 0, and a NaN stays one). Checked against double over every
// float in [-160, 0]: 0.97 units (expf 0.86 for normal results, 1.00 for subnormal ones).
__device__ __forceinline__ float exp_neg(float x) {
    constexpr float kHi = 1.44269504088896341f, kLo = static_cast<float>(1.44269504088896340736 - static_cast<double>(kHi));
    const float c = x < -150.0f ? -150.0f : x;  // (keeps -inf out of the products)
    const float k = rintf(c * kHi);
    const float f = fmaf(c, kLo, fmaf(c, kHi, -k));
    return ldexpf(__builtin_amdgcn_exp2f(f), static_cast<int>(k));
}

// q / k: norm + RoPE into B.q or the cache; gate: T(sigmoid); v: into the cache.
template <int CPL>
__global__ __launch_bounds__(64) void k_attn_prework(AttnDev A, AttnBufs B, uint16_t* __restrict__ keys,
                                                     uint16_t* __restrict__ values, int64_t cap, int64_t T0,
                                                     int64_t position) {
    __shared__ float nv[64 * CPL];
    __shared__ float csk[32 * CPL], snk[32 * CPL];  // the rotary table of this row: pair k's T(cos), T(sin)
    const int head = blockIdx.x, r = blockIdx.y, lane = threadIdx.x;
    const int HQ = A.hq, HKV = A.hkv, D = A.d, R = A.rot, half = R / 2;
    const int QW = HQ * D, KW = HKV * D;
    const int role = head < HQ ? 0 : head < HQ + HKV ? 1 : 2;  // query, key, value head
    const int h = role == 0 ? head : role == 1 ? head - HQ : head - HQ - HKV;
    const int64_t tok = T0 + r;
    if (role == 2) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int i = lane * CPL + c;
            values[(static_cast<int64_t>(h) * cap + tok) * D + i] = B.vr[static_cast<size_t>(r) * KW + h * D + i];
        }
        return;
    }
    const uint16_t* src = role == 0 ? B.qg + static_cast<size_t>(r) * 2 * QW + static_cast<size_t>(h) * 2 * D
                                    : B.kr + static_cast<size_t>(r) * KW + h * D;
    const uint16_t* wn = role == 0 ? A.qn : A.kn;
    float x[CPL];
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        x[c] = bf2f(src[lane * CPL + c]);
        ss = fmaf(x[c], x[c], ss);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(D) + A.eps);
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int i = lane * CPL + c;
        nv[i] = tbf(bf2f(wn[i]) * tbf(x[c] * inv));
    }
    // one rotary pair per lane (the two elements of a pair share its angle), in double as
    // before: pos * theta^(-2k / R)
    const double pos = static_cast<double>(position + r);
    for (int k = lane; k < half; k += 64) {
        const double ang = pos * pow(A.theta, -2.0 * static_cast<double>(k) / static_cast<double>(R));
        csk[k] = tbf(static_cast<float>(cos(ang)));
        snk[k] = tbf(static_cast<float>(sin(ang)));
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int i = lane * CPL + c;
        float y = nv[i];
        if (i < R) {
            const int k = i < half ? i : i - half;
            const float cs = csk[k], sn = snk[k];
            const float rot = i < half ? -nv[i + half] : nv[i - half];
            y = tbf(tbf(nv[i] * cs) + tbf(rot * sn));
        }
        if (role == 0) {
            const size_t at = (static_cast<size_t>(r) * HQ + h) * D + i;
            B.q[at] = f2bf(y);
            B.gs[at] = f2bf(sigmoid_bf(bf2f(src[D + i])));
        } else {
            keys[(static_cast<int64_t>(h) * cap + tok) * D + i] = f2bf(y);
        }
    }
}

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f4_t mfma_bf16(uint4 a, uint4 b, f4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, a), __builtin_bit_cast(bf8_t, b), c, 0,
                                                   0, 0);
}

// The workgroup's (unit, query chunk) of a grid of `units` (token tile, kv head) pairs times nmc
// query chunks: the chunks of a pair run on one XCD, so that its L2 serves their shared tokens.
// False past the last unit.
__device__ __forceinline__ bool attn_unit(int units, int nmc, int* unit, int* mc) {
    const int idx = static_cast<int>(blockIdx.x >> 3);
    *mc = idx % nmc;
    *unit = (idx / nmc) * 8 + static_cast<int>(blockIdx.x & 7);
    return *unit < units;
}

// Scores and tile statistics of NS 64-token tiles of kv head g for MT 16-query M-tiles of the
// head's group (query j: row j / G, head g G + j % G), transposed: A = the keys (wave w: tokens
// 16 w .. 16 w + 15 of each tile; lane (c, q): token c, dims 8 q .. 8 q + 7 of each 32-dim step),
// B = the queries (lane (c, q): query c, the same dims), both read as 16-byte runs straight into
// registers; the lane then holds tokens 4 q .. 4 q + 3 of query c, one 8-byte store. Per query
// and tile the max and the float sum of exp(s - max) over the tokens it sees go to B.stats.
// Latency-bound: every key of the workgroup is in flight before the first product, and the
// maxima and sums of all M-tiles meet in LDS together (two barriers a workgroup; one 16-query
// M-tile at a time with three barriers each took 84 us at 23 rows over 30,001 tokens, now 37 us).
template <int D, int MT, int NS>
__global__ __launch_bounds__(256, 2) void k_attn_scores(AttnDev A, AttnBufs B, int S, const uint16_t* __restrict__ keys,
                                                        int64_t cap, int64_t T0, int64_t tpad, int nmc) {
    constexpr int KS = D / 32, QB = MT * 16;
    __shared__ float red_m[4][NS][QB], red_s[4][NS][QB];
    const int HQ = A.hq, HKV = A.hkv, G = HQ / HKV, NQ = S * G;
    const int64_t Ttot = T0 + S;
    const int ntile = static_cast<int>((Ttot + kTok - 1) / kTok);
    int unit, mc;
    if (!attn_unit((ntile + NS - 1) / NS * HKV, nmc, &unit, &mc)) return;
    const int tile0 = unit / HKV * NS, g = unit % HKV, j0 = mc * QB;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, q = lane >> 4;
    const int64_t tw = static_cast<int64_t>(tile0) * kTok + 16 * w;  // the wave's first token
    // several M-tiles of several tiles: the queries go through LDS (rows padded by 16 bytes), requested with the
    // keys, instead of one load latency per M-tile
    constexpr bool kStage = MT > 1 && NS > 1;
    constexpr int QS = D + 8, QR = kStage ? QB * D / 8 / 256 : 1;
    __shared__ __align__(16) uint16_t qs[kStage ? QB * QS : 8];
    auto query = [&](int row) {  // (past the end: the last one repeated, unused)
        const int j = j0 + row < NQ ? j0 + row : NQ - 1;
        return static_cast<size_t>(j / G) * HQ + g * G + j % G;
    };
    uint4 qv[QR];
    if constexpr (kStage)
#pragma unroll
        for (int k = 0; k < QR; ++k) {
            const int i = threadIdx.x + 256 * k;
            qv[k] = *reinterpret_cast<const uint4*>(B.q + query(i / (D / 8)) * D + i % (D / 8) * 8);
        }
    uint4 kb[NS][KS];  // (a token past the end repeats the last one, unused)
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int64_t tk = tw + kTok * s + c;
        const uint16_t* krow = keys + (static_cast<int64_t>(g) * cap + (tk < Ttot ? tk : Ttot - 1)) * D + 8 * q;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kb[s][ks] = *reinterpret_cast<const uint4*>(krow + 32 * ks);
    }
    if constexpr (kStage) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < QR; ++k) {
            const int i = threadIdx.x + 256 * k;
            *reinterpret_cast<uint4*>(qs + i / (D / 8) * QS + i % (D / 8) * 8) = qv[k];
        }
        lds_barrier();
    }
    const float scale = tbf(static_cast<float>(1.0 / sqrt(static_cast<double>(D))));
    float sv[MT][NS][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int j = j0 + mt * 16 + c, r = (j < NQ ? j : NQ - 1) / G;
        const size_t qi = query(mt * 16 + c);
        const uint16_t* qrow = kStage ? qs + (mt * 16 + c) * QS + 8 * q : B.q + qi * D + 8 * q;
        uint4 qb[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qb[ks] = *reinterpret_cast<const uint4*>(qrow + 32 * ks);
        const int64_t last = T0 + r;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            f4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) acc = mfma_bf16(kb[s][ks], qb[ks], acc);
            const int64_t t = tw + kTok * s + 4 * q;
            uint32_t b[2];
            float m = -INFINITY;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t d = pack_bf(acc[2 * i], acc[2 * i + 1]);
                b[i] = pack_bf(bflo(d) * scale, bfhi(d) * scale);
                sv[mt][s][2 * i] = t + 2 * i <= last ? bflo(b[i]) : -INFINITY;
                sv[mt][s][2 * i + 1] = t + 2 * i + 1 <= last ? bfhi(b[i]) : -INFINITY;
                m = fmaxf(m, fmaxf(sv[mt][s][2 * i], sv[mt][s][2 * i + 1]));
            }
            // (scores past the query's last token, inside its padded row, are never read as such)
            if (j < NQ && t < tpad) *reinterpret_cast<uint2*>(B.sc + qi * tpad + t) = make_uint2(b[0], b[1]);
            m = fmaxf(m, xor_lane_f<16>(m));
            m = fmaxf(m, xor_lane_f<32>(m));
            if (q == 0) red_m[w][s][mt * 16 + c] = m;
        }
    }
    lds_barrier();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int row = mt * 16 + c;
            const float m = fmaxf(fmaxf(red_m[0][s][row], red_m[1][s][row]), fmaxf(red_m[2][s][row], red_m[3][s][row]));
            float e = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) e += sv[mt][s][i] == -INFINITY ? 0.0f : exp_neg(sv[mt][s][i] - m);
            e += xor_lane_f<16>(e);
            e += xor_lane_f<32>(e);
            if (q == 0) red_s[w][s][row] = e;
        }
    lds_barrier();
    const size_t NQall = static_cast<size_t>(S) * HQ;
    for (int i = threadIdx.x; i < NS * QB; i += 256) {
        const int s = i / QB, row = i % QB, j = j0 + row;
        if (j >= NQ || tile0 + s >= ntile) continue;
        const size_t qi = static_cast<size_t>(j / G) * HQ + g * G + j % G;
        B.stats[static_cast<size_t>(tile0 + s) * NQall + qi] =
            make_float2(fmaxf(fmaxf(red_m[0][s][row], red_m[1][s][row]), fmaxf(red_m[2][s][row], red_m[3][s][row])),
                        (red_s[0][s][row] + red_s[1][s][row]) + (red_s[2][s][row] + red_s[3][s][row]));
    }
}

// Per query: max and sum over its tiles' statistics (m = max m_t, sum = sum s_t exp(m_t - m)).
__global__ __launch_bounds__(256) void k_attn_stats(AttnDev A, AttnBufs B, int S, int64_t T0) {
    __shared__ float red[4];
    const int qi = blockIdx.x, r = qi / A.hq, tid = threadIdx.x;
    const size_t NQall = static_cast<size_t>(S) * A.hq;
    const int64_t nt = (T0 + r + 1 + kTok - 1) / kTok;
    float m = -INFINITY;
    for (int64_t k = tid; k < nt; k += 256) m = fmaxf(m, B.stats[static_cast<size_t>(k) * NQall + qi].x);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    float s = 0.0f;
    for (int64_t k = tid; k < nt; k += 256) {
        const float2 st = B.stats[static_cast<size_t>(k) * NQall + qi];
        s += st.y * expf(st.x - m);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
        B.mx[qi] = m;
        B.sm[qi] = (red[0] + red[1]) + (red[2] + red[3]);
    }
}

// P.V of one token tile (NS 64-token sub-tiles) of kv head g for a DW-dim slice and MT 16-query
// M-tiles of the queries of rows [row0, row0 + rows), on v_mfma_f32_16x16x32_bf16, transposed: A
// = the sub-tile's values of the slice, staged transposed in LDS ([dim][token], rows padded by 16
// bytes), B = p = T(exp(s - m) / sum) of 8 tokens of one query (0 for tokens it does not see);
// wave w forms p for tokens 16 w .. 16 w + 15 of the sub-tile (each p once per workgroup, shared
// through LDS) and owns dims 16 NTW w .. of the slice; the lane ends with 4 dims of query c, one
// 16-byte store per (tile, query). The next sub-tile's values and scores are in flight while the
// current one computes.
// Bound by the serial chain of a sub-tile (loads, p, two barriers, products) and, at long
// contexts, by the bytes of values, scores and partials. With every wave forming every p (an
// expf and a division each) and 128-token tiles throughout, 23 rows over 30,001 tokens took 127
// us, now 33 us; 4 rows over 4,096 tokens 15.7 -> 5.7 us.
template <int D, int DW, int MT, int NS>
__global__ __launch_bounds__(256) void k_attn_pv(AttnDev A, AttnBufs B, int S, int row0, int rows,
                                                 const uint16_t* __restrict__ values, int64_t cap, int64_t T0,
                                                 int64_t tpad, int nmc) {
    constexpr int VS = kTok + 8, PS = kTok + 8;  // LDS row strides (bf16)
    constexpr int NSL = D / DW;                  // dim slices (DW dims per workgroup)
    constexpr int NTW = DW / 64;                 // 16-dim tiles per wave
    constexpr int CPT = DW / 64;                 // 8-dim chunks a thread stages per sub-tile (two tokens each)
    constexpr int QB = MT * 16;
    __shared__ __align__(16) uint16_t vt[DW * VS];
    __shared__ __align__(16) uint16_t pt[QB * PS];
    const int HQ = A.hq, HKV = A.hkv, G = HQ / HKV, NQ = rows * G;
    const int64_t Ttot = T0 + row0 + rows;
    int unit, mc;
    if (!attn_unit(static_cast<int>((Ttot + NS * kTok - 1) / (NS * kTok)) * HKV, nmc * NSL, &unit, &mc)) return;
    const int tile = unit / HKV, g = unit % HKV, j0 = mc / NSL * QB, d0 = mc % NSL * DW;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, q = lane >> 4;
    const int64_t tb = static_cast<int64_t>(tile) * NS * kTok, left = Ttot - tb;
    const int nsub = static_cast<int>(left >= NS * kTok ? NS : (left + kTok - 1) / kTok);
    // staging: thread (token pair tp, 8-dim chunks dc0 + 8 k) of the slice
    const int tp = tid & 31, dc0 = tid >> 5;
    uint4 va[CPT], vb[CPT];
    auto load = [&](int64_t ts) {
        const int64_t t = ts + 2 * tp;
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const uint16_t* src = values + (static_cast<int64_t>(g) * cap + t) * D + d0 + 8 * (dc0 + 8 * k);
            va[k] = t < Ttot ? *reinterpret_cast<const uint4*>(src) : make_uint4(0u, 0u, 0u, 0u);
            vb[k] = t + 1 < Ttot ? *reinterpret_cast<const uint4*>(src + D) : make_uint4(0u, 0u, 0u, 0u);
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const uint32_t a[4] = {va[k].x, va[k].y, va[k].z, va[k].w}, b[4] = {vb[k].x, vb[k].y, vb[k].z, vb[k].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = 8 * (dc0 + 8 * k) + 2 * e;
                *reinterpret_cast<uint32_t*>(vt + d * VS + 2 * tp) = (a[e] & 0xFFFFu) | (b[e] << 16);
                *reinterpret_cast<uint32_t*>(vt + (d + 1) * VS + 2 * tp) = (a[e] >> 16) | (b[e] & 0xFFFF0000u);
            }
        }
    };
    // per M-tile: the lane's query, its softmax max and sum (a query past the end repeats the last
    // one, unused), and its scores of tokens 16 w + 4 q .. + 3 of a sub-tile
    size_t qi[MT];
    int64_t last[MT];
    float mrow[MT], srow[MT], irow[MT];
    uint2 scv[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int j = j0 + mt * 16 + c, jc = j < NQ ? j : NQ - 1, r = row0 + jc / G;
        qi[mt] = static_cast<size_t>(r) * HQ + g * G + jc % G;
        last[mt] = T0 + r;
        mrow[mt] = B.mx[qi[mt]];
        srow[mt] = B.sm[qi[mt]];
        irow[mt] = 1.0f / srow[mt];
    }
    // T(exp(s - max) / sum) of a pair: the quotient from the reciprocal, corrected once
    auto prob = [&](int mt, float s) {
        const float e = exp_neg(s - mrow[mt]), d = e * irow[mt];
        return fmaf(fmaf(-d, srow[mt], e), irow[mt], d);
    };
    auto load_sc = [&](int64_t ts) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            scv[mt] = *reinterpret_cast<const uint2*>(B.sc + qi[mt] * tpad + ts + 16 * w + 4 * q);
    };
    f4_t acc[MT][NTW];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) acc[mt][nt] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    load_sc(tb);
    load(tb);
    for (int s = 0; s < nsub; ++s) {
        const int64_t ts = tb + static_cast<int64_t>(kTok) * s, t = ts + 16 * w + 4 * q;
        uint2 pk[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const uint32_t u[2] = {scv[mt].x, scv[mt].y};
            uint32_t o[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                o[e] = pack_bf(t + 2 * e <= last[mt] ? prob(mt, bflo(u[e])) : 0.0f,
                               t + 2 * e + 1 <= last[mt] ? prob(mt, bfhi(u[e])) : 0.0f);
            }
            pk[mt] = make_uint2(o[0], o[1]);
        }
        if (s > 0) lds_barrier();  // the previous sub-tile's reads are done
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            *reinterpret_cast<uint2*>(pt + (mt * 16 + c) * PS + 16 * w + 4 * q) = pk[mt];
        store();
        if (s + 1 < nsub) {
            load_sc(ts + kTok);
            load(ts + kTok);
        }
        lds_barrier();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            uint4 p[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                p[mt] = *reinterpret_cast<const uint4*>(pt + (mt * 16 + c) * PS + 32 * ks + 8 * q);
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) {
                const uint4 v = *reinterpret_cast<const uint4*>(vt + ((w * NTW + nt) * 16 + c) * VS + 32 * ks + 8 * q);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt][nt] = mfma_bf16(v, p[mt], acc[mt][nt]);
            }
        }
    }
    const size_t NQall = static_cast<size_t>(S) * HQ;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        if (j0 + mt * 16 + c >= NQ) continue;
        float* dst = B.part + (static_cast<size_t>(tile) * NQall + qi[mt]) * D + d0;
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) *reinterpret_cast<f4_t*>(dst + (w * NTW + nt) * 16 + 4 * q) = acc[mt][nt];
    }
}

// attended = T(sum of the tiles' partials), gated = T(attended * gate): TG groups of D
// threads, group k adds tiles k, k + TG, .. (8 loads in flight), the groups added in order.
template <int D>
__global__ __launch_bounds__(1024) void k_attn_combine(AttnDev A, AttnBufs B, int S, int row0, int64_t T0,
                                                       int pv_tokens) {
    constexpr int TG = 1024 / D;
    __shared__ float red[1024];
    const int qi = row0 * A.hq + static_cast<int>(blockIdx.x), d = threadIdx.x % D, k = threadIdx.x / D;
    const int r = qi / A.hq, h = qi % A.hq;
    const int64_t ntile = (T0 + r + pv_tokens) / pv_tokens;
    const size_t NQall = static_cast<size_t>(S) * A.hq;
    const float* src = B.part + static_cast<size_t>(qi) * D + d;
    const size_t step = NQall * D;
    float a = 0.0f;
    int64_t t = k;
    for (; t + 7 * TG < ntile; t += 8 * TG) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = src[static_cast<size_t>(t + u * TG) * step];
#pragma unroll
        for (int u = 0; u < 8; ++u) a += v[u];
    }
    for (; t < ntile; t += TG) a += src[static_cast<size_t>(t) * step];
    red[threadIdx.x] = a;
    __syncthreads();
    if (k != 0) return;
    float s = red[d];
#pragma unroll
    for (int kk = 1; kk < TG; ++kk) s += red[kk * D + d];
    B.gated[static_cast<size_t>(r) * A.hq * D + static_cast<size_t>(h) * D + d] =
        f2bf(tbf(s) * bf2f(B.gs[static_cast<size_t>(qi) * D + d]));
}

unsigned attn_grid(int64_t units, int chunks) { return static_cast<unsigned>((units + 7) / 8 * 8 * chunks); }
int attn_mtiles(int queries) { return queries <= 16 ? 1 : queries <= 32 ? 2 : kMtMax; }

template <int D, int MT, int NS>
hipError_t launch_scores_t(const AttnDev& A, const AttnBufs& B, int S, const uint16_t* keys, int64_t cap, int64_t T0,
                           int64_t tpad, hipStream_t st) {
    const int nmc = (S * (A.hq / A.hkv) + MT * 16 - 1) / (MT * 16);
    const int64_t ntile = (T0 + S + kTok - 1) / kTok;
    return launch(k_attn_scores<D, MT, NS>, dim3(attn_grid((ntile + NS - 1) / NS * A.hkv, nmc)), dim3(256), 0, st, A, B, S,
                  keys, cap, T0, tpad, nmc);
}
template <int D>
hipError_t launch_scores(const AttnDev& A, const AttnBufs& B, int S, const uint16_t* keys, int64_t cap, int64_t T0,
                         int64_t tpad, hipStream_t st) {
    const int mt = attn_mtiles(S * (A.hq / A.hkv));
    // four tiles a workgroup (the queries read once for them) where that still leaves two
    // workgroups per CU
    const bool wide = (T0 + S) / kTok * A.hkv * ((S * (A.hq / A.hkv) + 63) / 64) >= 4 * 512;
    switch (mt) {
        case 1: return wide ? launch_scores_t<D, 1, 4>(A, B, S, keys, cap, T0, tpad, st)
                            : launch_scores_t<D, 1, 1>(A, B, S, keys, cap, T0, tpad, st);
        case 2: return wide ? launch_scores_t<D, 2, 4>(A, B, S, keys, cap, T0, tpad, st)
                            : launch_scores_t<D, 2, 1>(A, B, S, keys, cap, T0, tpad, st);
        default: return wide ? launch_scores_t<D, 4, 4>(A, B, S, keys, cap, T0, tpad, st)
                             : launch_scores_t<D, 4, 1>(A, B, S, keys, cap, T0, tpad, st);
    }
}

template <int D, int DW, int MT, int NS>
hipError_t launch_pv_t(const AttnDev& A, const AttnBufs& B, int S, int row0, int rows, const uint16_t* values, int64_t cap,
                       int64_t T0, int64_t tpad, hipStream_t st) {
    const int nmc = (rows * (A.hq / A.hkv) + MT * 16 - 1) / (MT * 16);
    const int64_t tiles = (T0 + row0 + rows + NS * kTok - 1) / (NS * kTok);
    return launch(k_attn_pv<D, DW, MT, NS>, dim3(attn_grid(tiles * A.hkv, nmc * (D / DW))), dim3(256), 0, st, A, B, S, row0,
                  rows, values, cap, T0, tpad, nmc);
}
template <int D, int NS>
hipError_t launch_pv(const AttnDev& A, const AttnBufs& B, int S, int row0, int rows, const uint16_t* values, int64_t cap,
                     int64_t T0, int64_t tpad, hipStream_t st) {
    const int nq = rows * (A.hq / A.hkv), mt = attn_mtiles(nq);
    const int64_t wgs = (T0 + row0 + rows + NS * kTok - 1) / (NS * kTok) * A.hkv * ((nq + 63) / 64);
    // few tiles: 64-dim slices per workgroup for parallelism (p formed again by each)
    const bool slice = D > 64 && wgs < kSliceWgs;
    switch (mt) {
        case 1: return slice ? launch_pv_t<D, 64, 1, NS>(A, B, S, row0, rows, values, cap, T0, tpad, st)
                             : launch_pv_t<D, D, 1, NS>(A, B, S, row0, rows, values, cap, T0, tpad, st);
        case 2: return slice ? launch_pv_t<D, 64, 2, NS>(A, B, S, row0, rows, values, cap, T0, tpad, st)
                             : launch_pv_t<D, D, 2, NS>(A, B, S, row0, rows, values, cap, T0, tpad, st);
        default: return slice ? launch_pv_t<D, 64, 4, NS>(A, B, S, row0, rows, values, cap, T0, tpad, st)
                              : launch_pv_t<D, D, 4, NS>(A, B, S, row0, rows, values, cap, T0, tpad, st);
    }
}

template <int D>
hipError_t launch_attn_core(const AttnDev& A, const AttnBufs& B, int S, uint16_t* keys, uint16_t* values, int64_t cap,
                            int64_t T0, int64_t position, int64_t tpad, hipStream_t st) {
    hipError_t e = launch(k_attn_prework<D / 64>, dim3(A.hq + 2 * A.hkv, S), dim3(64), 0, st, A, B, keys, values, cap, T0,
                          position);
    if (e == hipSuccess) e = launch_scores<D>(A, B, S, keys, cap, T0, tpad, st);
    if (e == hipSuccess) e = launch(k_attn_stats, dim3(S * A.hq), dim3(256), 0, st, A, B, S, T0);
    // rows of one P.V tile size together (a call whose rows cross a limit of attn_pv_tokens: one
    // launch for the rows up to it and one for the rest)
    for (int r0 = 0, n; r0 < S && e == hipSuccess; r0 += n) {
        const int pt = attn_pv_tokens(T0 + r0 + 1);
        for (n = 1; r0 + n < S && attn_pv_tokens(T0 + r0 + n + 1) == pt; ++n) {}
        e = pt == 2 * kTok   ? launch_pv<D, 2>(A, B, S, r0, n, values, cap, T0, tpad, st)
            : pt == 4 * kTok ? launch_pv<D, 4>(A, B, S, r0, n, values, cap, T0, tpad, st)
                             : launch_pv<D, 8>(A, B, S, r0, n, values, cap, T0, tpad, st);
        if (e == hipSuccess)
            e = launch(k_attn_combine<D>, dim3(n * A.hq), dim3(1024), 0, st, A, B, S, r0, T0, pt);
    }
    return e;
}

} // namespace

bool attn_geometry_ok(int hidden, int hq, int hkv, int d, int rot) {
    return hidden > 0 && hq > 0 && hkv > 0 && hq % hkv == 0 && (d == 64 || d == 128 || d == 256) && rot > 0 &&
           rot % 2 == 0 && rot <= d;
}

int64_t attn_score_stride(int64_t tokens) { return (tokens + kTok - 1) / kTok * kTok; }
// The most P.V tiles of any query of up to `tokens` tokens.
int64_t attn_pv_tiles(int64_t tokens) {
    int64_t n = 0;
    for (const int64_t t : {tokens, tokens < kPvLong ? tokens : kPvLong, tokens < kPvMid ? tokens : kPvMid}) {
        const int64_t v = (t + attn_pv_tokens(t) - 1) / attn_pv_tokens(t);
        n = v > n ? v : n;
    }
    return n;
}
int64_t attn_score_tiles(int64_t tokens) { return (tokens + kTok - 1) / kTok; }

hipError_t launch_attn_verify(const AttnDev& A, const AttnBufs& B, int S, const uint16_t* x, uint16_t* keys,
                              uint16_t* values, int64_t cap, int64_t T0, int64_t position, uint16_t* out,
                              hipStream_t st) {
    const int QW = A.hq * A.d, KW = A.hkv * A.d;
    AffineRowSet in{};
    in.n = 3;
    in.p[0] = AffineRows{A.w[0], A.s[0], A.b[0], B.qg, 2 * QW, 2 * QW, 0};
    in.p[1] = AffineRows{A.w[1], A.s[1], A.b[1], B.kr, KW, KW, 0};
    in.p[2] = AffineRows{A.w[2], A.s[2], A.b[2], B.vr, KW, KW, 0};
    hipError_t e = launch_affine_rows(in, x, S, A.hidden, A.group, A.bits, A.f16, st);
    if (e != hipSuccess) return e;
    const int64_t tpad = attn_score_stride(T0 + S);
    switch (A.d) {
        case 64: e = launch_attn_core<64>(A, B, S, keys, values, cap, T0, position, tpad, st); break;
        case 128: e = launch_attn_core<128>(A, B, S, keys, values, cap, T0, position, tpad, st); break;
        case 256: e = launch_attn_core<256>(A, B, S, keys, values, cap, T0, position, tpad, st); break;
        default: return hipErrorInvalidValue;
    }
    if (e != hipSuccess) return e;
    AffineRowSet o{};
    o.n = 1;
    o.p[0] = AffineRows{A.w[3], A.s[3], A.b[3], out, A.hidden, A.hidden, 0};
    return launch_affine_rows(o, B.gated, S, QW, A.group, A.bits, A.f16, st);
}

} // namespace q38
