// q38_affine.hip — the shared expert in MLX affine form (R10 in the layout of the reference's
// checkpoints: the affine branch of SparseMoe::load_projection, src/sparse_moe.cpp:474-480,
// 662-700, applied by SparseMoe::forward_shared, :1306-1313, through quantized_matmul).
//
// Two launches per layer call, before the routed experts' kernels (the tiles of
// q38_affine.hpp):
//   k_sa_gu  gate and up rows of the shared expert for the call's rows, SwiGLU with the
//            reference's rounding points, into the workspace's SwiGLU rows (bf16-exact values);
//   k_sa_dn  the down projection of those rows into the shared expert's down-output rows of
//            the partial-sum planes (value in plane 0, 0 in plane 1 where the combine adds a
//            second plane), which the combine reads as it reads a VQ shared expert's.
// k_affine_rows runs several projections of the same rows in one launch.
#include "q38_affine.hpp"

namespace q38 {
namespace {

// Gate and up rows o of the shared expert, SwiGLU: hs[r][o] (bf16) for the workgroup's rows.
template <int BITS, int G, int MT>
__global__ __launch_bounds__(512) void k_sa_gu(LayerDev L, MoeBufs B, int M) {
    extern __shared__ __align__(16) aff_f4_t red[];
    const int H = L.H, Is = L.sa_inter, r0 = blockIdx.y * 16 * MT, lane = threadIdx.x & 63;
    const int o = blockIdx.x * kAffTile + (lane & 15), oc = min(o, Is - 1);
    const AffCol col[2] = {aff_col(L.sa[0].w, L.sa[0].s, L.sa[0].b, oc, H, BITS, G),
                           aff_col(L.sa[1].w, L.sa[1].s, L.sa[1].b, oc, H, BITS, G)};
    aff_tile<BITS, G, MT, 2>(col, B.x, r0, M, H, L.sa_f16, red, [&](int mt, const aff_f4_t (&v)[2]) {
        if (o >= Is) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + 16 * mt + 4 * (lane >> 4) + i;
            if (r < M) B.h16[static_cast<size_t>(r) * Is + o] = f2bf(swiglu(v[0][i], v[1][i]));
        }
    });
}

// Down rows o of the shared expert over the SwiGLU rows: the shared expert's rows of the down
// partial-sum planes, d[M*K + r][o] (plane 0; plane 1, where the call has one, gets 0).
template <int BITS, int G, int MT>
__global__ __launch_bounds__(512) void k_sa_dn(LayerDev L, MoeBufs B, int M) {
    extern __shared__ __align__(16) aff_f4_t red[];
    const int H = L.H, Is = L.sa_inter, r0 = blockIdx.y * 16 * MT, lane = threadIdx.x & 63;
    const int o = blockIdx.x * kAffTile + (lane & 15);  // (H is a multiple of 16)
    const AffCol col[1] = {aff_col(L.sa[2].w, L.sa[2].s, L.sa[2].b, o, Is, BITS, G)};
    aff_tile<BITS, G, MT, 1>(col, B.h16, r0, M, Is, L.sa_f16, red, [&](int mt, const aff_f4_t (&v)[1]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + 16 * mt + 4 * (lane >> 4) + i;
            if (r >= M) continue;
            const size_t at = static_cast<size_t>(M * L.K + r) * H + o;
            B.d[at] = v[0][i];
            if (L.d_parts == 2) B.d[B.d_plane + at] = 0.0f;
        }
    });
}

// Rows of several affine projections of the same S input rows in one launch: workgroups
// [p.first_block, next first_block) take projection p's weight rows, 16 each.
template <int BITS, int G, int MT>
__global__ __launch_bounds__(512) void k_affine_rows(AffineRowSet set, const uint16_t* __restrict__ x, int S, int IN,
                                                     int f16) {
    extern __shared__ __align__(16) aff_f4_t red[];
    // the projection of this block (uniform selects over the argument block)
    const int bx = static_cast<int>(blockIdx.x);
    const int pi = set.n > 3 && bx >= set.p[3].first_block ? 3
                   : set.n > 2 && bx >= set.p[2].first_block ? 2
                   : set.n > 1 && bx >= set.p[1].first_block ? 1
                                                             : 0;
    const AffineRows P = pi == 3 ? set.p[3] : pi == 2 ? set.p[2] : pi == 1 ? set.p[1] : set.p[0];
    const int r0 = blockIdx.y * 16 * MT, lane = threadIdx.x & 63;
    const int o = (bx - P.first_block) * kAffTile + (lane & 15);
    const AffCol col[1] = {aff_col(P.w, P.s, P.b, min(o, P.out - 1), IN, BITS, G)};
    aff_tile<BITS, G, MT, 1>(col, x, r0, S, IN, f16, red, [&](int mt, const aff_f4_t (&v)[1]) {
        if (o >= P.out) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + 16 * mt + 4 * (lane >> 4) + i;
            if (r < S) P.dst[static_cast<size_t>(r) * P.dst_stride + o] = f2bf(v[0][i]);
        }
    });
}

// Waves of a tile: one per 512-input slab, at most 8 (a function of the input width alone, so
// that a row's sums keep their order whatever the call's row count).
int aff_waves(int IN) {
    const int n = (IN + kAffSlab - 1) / kAffSlab;
    return n > 8 ? 8 : n;
}
size_t aff_lds(int waves, int mt, int nt) { return static_cast<size_t>(waves) * 64 * mt * nt * sizeof(aff_f4_t); }

// Calls KERN<BITS, G, MT> by the layout and the row count: one 16-row M-tile per workgroup up
// to 16 rows, four (the weights read once per 64 rows) beyond.
#define Q38_AFF_MT(K, BITS, G, grid_x, IN, nt, rows, ...)                                                            \
    (rows <= 16 ? launch(K<BITS, G, 1>, dim3(grid_x, 1), dim3(64 * aff_waves(IN)), aff_lds(aff_waves(IN), 1, nt),    \
                         __VA_ARGS__)                                                                                \
                : launch(K<BITS, G, 4>, dim3(grid_x, (rows + 63) / 64), dim3(64 * aff_waves(IN)),                    \
                         aff_lds(aff_waves(IN), 4, nt), __VA_ARGS__))
#define Q38_AFF_G(K, BITS, G, ...) \
    (G == 32 ? Q38_AFF_MT(K, BITS, 32, __VA_ARGS__) : G == 64 ? Q38_AFF_MT(K, BITS, 64, __VA_ARGS__) \
     : G == 128 ? Q38_AFF_MT(K, BITS, 128, __VA_ARGS__) : hipErrorInvalidValue)
#define Q38_AFF(K, bits, G, ...) \
    (bits == 2 ? Q38_AFF_G(K, 2, G, __VA_ARGS__) : bits == 4 ? Q38_AFF_G(K, 4, G, __VA_ARGS__) \
     : bits == 8 ? Q38_AFF_G(K, 8, G, __VA_ARGS__) : hipErrorInvalidValue)
} // namespace

hipError_t launch_shared_affine(const LayerDev& L, const MoeBufs& B, int M, hipStream_t st) {
    if (!L.shared_affine) return hipSuccess;
    const int G = L.sa_group;
    const hipError_t e =
        Q38_AFF(k_sa_gu, L.sa_bits, G, (L.sa_inter + kAffTile - 1) / kAffTile, L.H, 2, M, st, L, B, M);
    if (e != hipSuccess) return e;
    return Q38_AFF(k_sa_dn, L.sa_bits, G, L.H / kAffTile, L.sa_inter, 1, M, st, L, B, M);
}

hipError_t launch_affine_rows(const AffineRowSet& in, const uint16_t* x, int S, int IN, int G, int bits, int f16,
                              hipStream_t st) {
    AffineRowSet set = in;
    int blocks = 0;
    for (int i = 0; i < set.n; ++i) {
        set.p[i].first_block = blocks;
        blocks += (set.p[i].out + kAffTile - 1) / kAffTile;
    }
    return Q38_AFF(k_affine_rows, bits, G, blocks, IN, 1, S, st, set, x, S, IN, f16);
}

} // namespace q38
