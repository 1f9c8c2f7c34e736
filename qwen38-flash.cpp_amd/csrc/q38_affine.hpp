// q38_affine.hpp — products of bf16 rows with MLX affine-quantized weight rows on the matrix
// cores, shared by the affine shared expert, the GatedDeltaNet and the attention projections
// (q38_affine.hip): quantized_matmul's arithmetic as this build computes it.
//
// Row o of a [OUT, IN] projection holds IN values q in [0, 2^BITS) packed LSB-first in 32-bit
// words (32 / BITS per word); w[o, c] = scale[o, c / G] * q[o, c] + bias[o, c / G], scales and
// biases bf16 or fp16. A workgroup takes 16 weight rows (the columns of the MFMA tile) and
// 16 * MT request rows (its rows); its waves take 512-input slabs of the K axis in turn, and
// their sums meet in LDS in wave order. Per scale group the wave forms sum(q x) and sum(x) on
// v_mfma_f32_16x16x32_bf16 (q <= 255 and x are exact in bf16, the products exact, the sums
// float; sum(x) is the product with a tile of ones, whose result lands in the same lanes) and
// accumulates scale * sum(q x) + bias * sum(x) in float. A lane owns one weight row (column
// lane & 15), so it reads that row's own scales; lane quarter q takes inputs 16 q .. 16 q + 15
// of each 64-input block (8 q .. 8 q + 7 of 32 for G = 32) of both operands. A request row's
// sums do not depend on the other rows of the call.
//
// Bound by the latency and the bytes of the weights at verify widths: every load of a slab
// (8 KiB of 8-bit weights per wave, the scales, half of the inputs) is issued before the first
// product, so that a whole projection is in flight at once; the products themselves are a few
// hundred matrix cycles per wave. Beyond 16 rows four M-tiles share the expanded weights, so
// they are read once per 64 rows instead of once per 16. Measured (kernel traces), 8-bit g64,
// against dot products on the vector units with the rows staged in LDS: 4 rows by 12,352 x 2048
// 16.0 -> 10.9 us (2.5 TB/s), by 2048 x 4096 12.0 -> 7.8 us; 23 rows by 9216 x 2048 55 -> 16 us,
// by 2048 x 4096 58 -> 12 us; the shared expert of 2048 rows, gate and up 601 -> 54 us, down
// 173 -> 43 us, of 13 rows 23.4 -> 8.2 and 8.5 -> 4.3 us.
#pragma once

#include "q38_moe_dev.hpp"

namespace q38 {
namespace {

constexpr int kAffSlab = 512;  // K inputs of a wave's slab
constexpr int kAffTile = 16;   // weight rows per workgroup

typedef __bf16 aff_bf8_t __attribute__((ext_vector_type(8)));
typedef float aff_f4_t __attribute__((ext_vector_type(4)));
// (caller tensors: words on 4-byte, scales on 2-byte addresses)
typedef uint32_t aff_u4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t aff_u2_t __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ aff_f4_t aff_mfma(uint4 a, uint4 b, aff_f4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(aff_bf8_t, a), __builtin_bit_cast(aff_bf8_t, b),
                                                   c, 0, 0, 0);
}

// This lane's weight row: its packed words and group parameters.
struct AffCol {
    const char* w;
    const uint16_t* s;
    const uint16_t* b;
};
__device__ __forceinline__ AffCol aff_col(const uint32_t* w, const uint16_t* s, const uint16_t* b, int row, int IN,
                                          int bits, int G) {
    const size_t r = static_cast<size_t>(row);
    const size_t ng = static_cast<size_t>(IN / G);
    return {reinterpret_cast<const char*>(w) + r * (IN / 32) * bits * 4, s + r * ng, b + r * ng};
}

// Two floats with integer values 0..255 (exact in bf16) packed as bf16, lo first.
__device__ __forceinline__ uint32_t aff_pack(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
template <int K>
__device__ __forceinline__ float aff_byte(uint32_t w) {
    return static_cast<float>((w >> (8 * K)) & 0xFFu);
}

// The packed values of a lane's quarter of one block (KB / 4 inputs), as loaded.
template <int BITS, int KB>
struct AffRaw {
    static constexpr int kBytes = KB / 4 * BITS / 8;  // 16, 8, 4 or 2
    static constexpr int kWords = kBytes < 4 ? 1 : kBytes / 4;
    uint32_t v[kWords];
    __device__ __forceinline__ void load(const char* p) {
        if constexpr (kBytes == 16) {
            const aff_u4_t u = *reinterpret_cast<const aff_u4_t*>(p);
            v[0] = u[0]; v[1] = u[1]; v[2] = u[2]; v[3] = u[3];
        } else if constexpr (kBytes == 8) {
            const aff_u2_t u = *reinterpret_cast<const aff_u2_t*>(p);
            v[0] = u[0]; v[1] = u[1];
        } else if constexpr (kBytes == 4) {
            v[0] = *reinterpret_cast<const uint32_t*>(p);
        } else {
            v[0] = *reinterpret_cast<const uint16_t*>(p);
        }
    }
    // values 8 st .. 8 st + 7 as bf16
    __device__ __forceinline__ uint4 frag(int st) const {
        if constexpr (BITS == 8) {
            const uint32_t a = v[2 * st], b = v[2 * st + 1];
            return make_uint4(aff_pack(aff_byte<0>(a), aff_byte<1>(a)), aff_pack(aff_byte<2>(a), aff_byte<3>(a)),
                              aff_pack(aff_byte<0>(b), aff_byte<1>(b)), aff_pack(aff_byte<2>(b), aff_byte<3>(b)));
        } else if constexpr (BITS == 4) {
            const uint32_t e = v[st] & 0x0F0F0F0Fu, o = (v[st] >> 4) & 0x0F0F0F0Fu;  // even, odd values
            return make_uint4(aff_pack(aff_byte<0>(e), aff_byte<0>(o)), aff_pack(aff_byte<1>(e), aff_byte<1>(o)),
                              aff_pack(aff_byte<2>(e), aff_byte<2>(o)), aff_pack(aff_byte<3>(e), aff_byte<3>(o)));
        } else {
            const uint32_t w = v[0] >> (16 * st);
            float f[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) f[j] = static_cast<float>((w >> (2 * j)) & 3u);
            return make_uint4(aff_pack(f[0], f[1]), aff_pack(f[2], f[3]), aff_pack(f[4], f[5]), aff_pack(f[6], f[7]));
        }
    }
};

// One slab of nb blocks at input k0 (FULL: 512 inputs), added to acc. The 16 * MT request rows
// start at row r0 of x; a tile row at `rows` or beyond repeats the last row (its sums are unused).
template <int BITS, int G, int MT, int NT, bool FULL>
__device__ __forceinline__ void aff_slab(const AffCol (&col)[NT], const uint16_t* __restrict__ x, int r0, int rows,
                                         int IN, int f16, int k0, int nb, aff_f4_t (&acc)[MT][NT]) {
    constexpr int KB = G == 32 ? 32 : 64, ST = KB / 32, NB = kAffSlab / KB;
    constexpr int GB = G == 128 ? 2 : 1;  // blocks per group
    // RAW blocks of weights and group parameters are loaded together, SUB blocks of inputs: the
    // whole slab's weights and half of its inputs for one M-tile (within 128 VGPRs, four waves
    // per SIMD); where several M-tiles share the weights, RAW = SUB blocks are expanded once
    // for all of them.
    constexpr int W2 = KB == 32 && NT == 2 ? 2 : 1;  // (two columns of 32-input groups: half as much)
    constexpr int SUB = MT == 1 ? NB / (2 * W2) : NB * KB / 128 / NT, RAW = MT == 1 ? NB / W2 : SUB, NG = RAW / GB;
    const int lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
    const uint4 ones = make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u);
    auto param = [&](uint32_t w, int g) {
        return f16 ? h2f(static_cast<uint16_t>(g & 1 ? w >> 16 : w)) : g & 1 ? bfhi(w) : bflo(w);
    };
#pragma unroll 1
    for (int h = 0; h < (FULL ? NB : nb); h += RAW) {
        AffRaw<BITS, KB> raw[NT][RAW];
        uint32_t sv[NT][(NG + 1) / 2], bv[NT][(NG + 1) / 2];  // two groups' scales (biases) per word
        const int g0 = k0 / G + h / GB;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const char* wp = col[t].w + (static_cast<size_t>(k0) + h * KB) * BITS / 8 + q * AffRaw<BITS, KB>::kBytes;
#pragma unroll
            for (int j = 0; j < RAW; ++j)
                raw[t][j].load(wp + static_cast<size_t>(FULL ? j : min(j, nb - 1 - h)) * KB * BITS / 8);
            if constexpr (FULL) {
                __builtin_memcpy(sv[t], col[t].s + g0, NG * 2);
                __builtin_memcpy(bv[t], col[t].b + g0, NG * 2);
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // (the scheduler would sink the loads to their uses)
#pragma unroll
        for (int hs = 0; hs < RAW; hs += SUB) {
            if (!FULL && h + hs >= nb) break;
            uint4 wf[NT][SUB][ST];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if (MT > 1 && r0 + 16 * mt >= rows) break;
                const uint16_t* xp = x + static_cast<size_t>(min(r0 + 16 * mt + c, rows - 1)) * IN + k0 + h * KB + KB / 4 * q;
                uint4 a[SUB][ST];
#pragma unroll
                for (int j = 0; j < SUB; ++j)
#pragma unroll
                    for (int s = 0; s < ST; ++s)
                        a[j][s] = *reinterpret_cast<const uint4*>(xp + (FULL ? hs + j : min(hs + j, nb - 1 - h)) * KB + 8 * s);
                __builtin_amdgcn_sched_barrier(0);
                if (mt == 0)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int j = 0; j < SUB; ++j)
#pragma unroll
                            for (int s = 0; s < ST; ++s) wf[t][j][s] = raw[t][hs + j].frag(s);
                aff_f4_t sx = {0.0f, 0.0f, 0.0f, 0.0f}, qx[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) qx[t] = aff_f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < SUB; ++j) {
                    if (!FULL && h + hs + j >= nb) break;
#pragma unroll
                    for (int s = 0; s < ST; ++s) {
                        sx = aff_mfma(a[j][s], ones, sx);
#pragma unroll
                        for (int t = 0; t < NT; ++t) qx[t] = aff_mfma(a[j][s], wf[t][j][s], qx[t]);
                    }
                    if ((j + 1) % GB) continue;
                    const int g = (hs + j) / GB;
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        // (a partial slab reads its group's parameters here: a row has one at most)
                        const float sc = FULL ? param(sv[t][g / 2], g) : param(col[t].s[g0 + g], 0);
                        const float bi = FULL ? param(bv[t][g / 2], g) : param(col[t].b[g0 + g], 0);
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[mt][t][i] = fmaf(sc, qx[t][i], fmaf(bi, sx[i], acc[mt][t][i]));
                        qx[t] = aff_f4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    }
                    sx = aff_f4_t{0.0f, 0.0f, 0.0f, 0.0f};
                }
            }
        }
    }
}

// The workgroup's tile: acc summed over its waves' slabs. emit(mt, v) receives, in one wave
// per M-tile, v[t][i] = the product of request row r0 + 16 mt + 4 (lane >> 4) + i with column
// lane & 15 of col t. red: blockDim.x * MT * NT float4 of LDS.
template <int BITS, int G, int MT, int NT, typename F>
__device__ __forceinline__ void aff_tile(const AffCol (&col)[NT], const uint16_t* __restrict__ x, int r0, int rows,
                                         int IN, int f16, aff_f4_t* red, F emit) {
    constexpr int KB = G == 32 ? 32 : 64;
    const int lane = threadIdx.x & 63, W = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    aff_f4_t acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[mt][t] = aff_f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int k0 = wave * kAffSlab; k0 < IN; k0 += W * kAffSlab) {
        const int nb = min(kAffSlab, IN - k0) / KB;
        if (nb == kAffSlab / KB)
            aff_slab<BITS, G, MT, NT, true>(col, x, r0, rows, IN, f16, k0, nb, acc);
        else
            aff_slab<BITS, G, MT, NT, false>(col, x, r0, rows, IN, f16, k0, nb, acc);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) red[((mt * NT + t) * W + wave) * 64 + lane] = acc[mt][t];
    lds_barrier();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        if (mt % W != wave || r0 + 16 * mt >= rows) continue;
        aff_f4_t v[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            v[t] = red[(mt * NT + t) * W * 64 + lane];
            for (int w = 1; w < W; ++w) v[t] += red[((mt * NT + t) * W + w) * 64 + lane];
        }
        emit(mt, v);
    }
}

} // namespace
} // namespace q38
