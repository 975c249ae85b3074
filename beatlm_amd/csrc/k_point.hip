// Short products over many rows, one launch for what took two or for what the
// vector ALUs did: a transposed convolution whose kernel is its stride (each
// input pixel times f f cout columns of weights, MainOp::ConvTranspose2d), and
// a bilinear resampling followed by a 1x1 convolution (the fusion stages'
// resample and projection), its corners blended as A is loaded.
//
// What bounds them is memory and the launch itself: k is at most 96, so a wave
// keeps its 64 columns of weights in registers (from the fragment-major pack,
// 1 KB a load) and walks 16-row tiles: A straight into fragments (8 consecutive k a
// lane), the products, then bias and epilogue through a tile of LDS of its own
// so that every store is 8 consecutive columns of a row. No barrier.
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"

namespace bl {
namespace {

constexpr int PT_WAVES = 4, PT_COLS = 64, PT_ROW = PT_COLS + 4;

template <Math M> struct PointOp;
template <> struct PointOp<Math::F32> {
    struct Frag {
        float v[8];
    };
    static __device__ __forceinline__ void take(Frag &f, const float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 8; e++) f.v[e] = v[e];
    }
    // Eight packed elements from element i on (planes: the lo plane's distance).
    static __device__ __forceinline__ void load(Frag &f, const void *b, uint64_t i, uint64_t) {
        const f32x4 x = *(const f32x4 *)((const float *)b + i), y = *(const f32x4 *)((const float *)b + i + 4);
#pragma unroll
        for (int e = 0; e < 8; e++) f.v[e] = e < 4 ? x[e] : y[e - 4];
    }
    static __device__ __forceinline__ f32x4 mma(const Frag &a, const Frag &b, f32x4 c) {
#pragma unroll
        for (int s = 0; s < 8; s++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[s], b.v[s], c, 0, 0, 0);
        return c;
    }
};
template <> struct PointOp<Math::SPLIT> {
    struct Frag {
        bf16x8 h, l;
    };
    static __device__ __forceinline__ void take(Frag &f, const float (&v)[8]) { split8_bf16(v, f.h, f.l); }
    static __device__ __forceinline__ void load(Frag &f, const void *b, uint64_t i, uint64_t planes) {
        f.h = *(const bf16x8 *)((const __bf16 *)b + i);
        f.l = *(const bf16x8 *)((const __bf16 *)b + planes + i);
    }
    static __device__ __forceinline__ f32x4 mma(const Frag &a, const Frag &b, f32x4 c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l, b.h, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.l, c, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.h, c, 0, 0, 0);
    }
};
template <> struct PointOp<Math::F16> {
    struct Frag {
        f16x8 v;
    };
    static __device__ __forceinline__ void take(Frag &f, const float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 8; e++) f.v[e] = (_Float16)v[e];
    }
    static __device__ __forceinline__ void load(Frag &f, const void *b, uint64_t i, uint64_t) {
        f.v = *(const f16x8 *)((const _Float16 *)b + i);
    }
    static __device__ __forceinline__ f32x4 mma(const Frag &a, const Frag &b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a.v, b.v, c, 0, 0, 0);
    }
};

__device__ __forceinline__ void load8(const float *p, float (&v)[8]) {
    const f32x4 a = *(const f32x4 *)p, b = *(const f32x4 *)(p + 4);
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = e < 4 ? a[e] : b[e - 4];
}
__device__ __forceinline__ void load8(const _Float16 *p, float (&v)[8]) {
    const f16x8 a = *(const f16x8 *)p;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (float)a[e];
}

// KS: 32-wide slices of k. UP: A is a bilinear resampling of the image x.
template <Math M, int KS, bool UP>
__global__ __launch_bounds__(64 * PT_WAVES) void point_kernel(PointArgs a) {
    using T = typename std::conditional<M == Math::F16, _Float16, float>::type;
    using Op = PointOp<M>;
    using Frag = typename Op::Frag;
    constexpr int TN = PT_COLS / 16;
    __shared__ __attribute__((aligned(16))) float tiles[PT_WAVES][16 * PT_ROW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l16 = lane & 15, g = lane >> 4;
    const uint32_t N = a.n, K = a.k, nb = (N + PT_COLS - 1) / PT_COLS;
    const uint32_t n0 = blockIdx.x % nb * PT_COLS, per_block = gridDim.x / nb;
    const T *X = (const T *)a.x;
    float *tile = tiles[wave];

    // The wave's weights: its 4 blocks of 16 columns.
    Frag b[KS][TN];
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
            Op::load(b[ks][j], a.b, ((uint64_t)(n0 / 16 + j) * (a.k_pad / 32) + min((uint32_t)ks, a.k_pad / 32 - 1)) * 512 + lane * 8,
                     (uint64_t)a.n_pad * a.k_pad);
    // The lane's columns of the epilogue: 8 consecutive ones, rows lane / 8 and 8 on.
    const uint32_t col = n0 + 8 * (lane & 7), tap = a.f ? col / a.cout : 0, co = a.f ? col - tap * a.cout : col;
    const bool col_ok = col < N;
    float bias[8];
#pragma unroll
    for (int e = 0; e < 8; e++) bias[e] = 0.0f;
    if (a.bias && col_ok) load8((const T *)a.bias + co, bias);

    const uint32_t row_tiles = (a.rows + 15) / 16;
    for (uint32_t rt = (blockIdx.x / nb) * PT_WAVES + wave; rt < row_tiles; rt += per_block * PT_WAVES) {
        const uint32_t row = min(16 * rt + l16, a.rows - 1);  // rows past the last re-read it; never stored
        f32x4 acc[TN];
#pragma unroll
        for (int j = 0; j < TN; j++) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        Frag f[KS];
        if constexpr (UP) {
            // Aligned corners, as the resampling kernel computes them.
            const uint32_t oy = row / a.ow, ox = row - oy * a.ow;
            const float py = a.ry * (float)oy, px = a.rx * (float)ox;
            const uint32_t y0 = min((uint32_t)py, a.ih - 1), x0 = min((uint32_t)px, a.iw - 1);
            const uint32_t y1 = min(y0 + 1, a.ih - 1), x1 = min(x0 + 1, a.iw - 1);
            const float ly = py - (float)y0, lx = px - (float)x0;
            const T *p00 = X + ((uint64_t)y0 * a.iw + x0) * K, *p01 = X + ((uint64_t)y0 * a.iw + x1) * K;
            const T *p10 = X + ((uint64_t)y1 * a.iw + x0) * K, *p11 = X + ((uint64_t)y1 * a.iw + x1) * K;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const uint32_t k = 32 * ks + 8 * g;
                float v[8], c00[8], c01[8], c10[8], c11[8];
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = 0.0f;
                if (k < K) {
                    load8(p00 + k, c00);
                    load8(p01 + k, c01);
                    load8(p10 + k, c10);
                    load8(p11 + k, c11);
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const float top = (1.0f - lx) * c00[e] + lx * c01[e];
                        const float bottom = (1.0f - lx) * c10[e] + lx * c11[e];
                        v[e] = (1.0f - ly) * top + ly * bottom;
                    }
                }
                Op::take(f[ks], v);
            }
        } else {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const uint32_t k = 32 * ks + 8 * g;
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = 0.0f;
                if (k < K) load8(X + (uint64_t)row * K + k, v);
                Op::take(f[ks], v);
            }
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[j] = Op::mma(f[ks], b[ks][j], acc[j]);
        // Accumulator j holds rows 4 g + r of column 16 j + l16.
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) tile[(4 * g + r) * PT_ROW + 16 * j + l16] = acc[j][r];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint32_t tr = (lane >> 3) + 8 * q, m = 16 * rt + tr;
            const float *t = tile + tr * PT_ROW + 8 * (lane & 7);
            const f32x4 t0 = *(const f32x4 *)t, t1 = *(const f32x4 *)(t + 4);
            if (!col_ok || m >= a.rows) continue;
            uint64_t idx = (uint64_t)m * N + col;
            if (a.f) {
                // Input pixel (y, x) and tap (ky, kx): output pixel (y f + ky, x f + kx).
                const uint32_t y = m / a.width, x = m - y * a.width, ky = tap / a.f, kx = tap - ky * a.f;
                idx = ((uint64_t)(y * a.f + ky) * (a.width * a.f) + x * a.f + kx) * a.cout + co;
            }
            f32x4 o0, o1;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o0[e] = apply_epilogue<T>(a.epi, t0[e] + bias[e], idx + e);
                o1[e] = apply_epilogue<T>(a.epi, t1[e] + bias[4 + e], idx + 4 + e);
            }
            if constexpr (M == Math::F16) {
                f16x8 h;
#pragma unroll
                for (int e = 0; e < 8; e++) h[e] = (_Float16)(e < 4 ? o0[e] : o1[e - 4]);
                *(f16x8 *)((_Float16 *)a.y + idx) = h;
            } else {
                store_f32x4((float *)a.y, idx, o0, a.y_planes);
                store_f32x4((float *)a.y, idx + 4, o1, a.y_planes);
            }
        }
    }
}

template <Math M, bool UP>
hipError_t point_slices(const PointArgs &a, hipStream_t s) {
    const uint32_t nb = (a.n + PT_COLS - 1) / PT_COLS, row_tiles = (a.rows + 15) / 16;
    // Four workgroups of 4 waves per CU at most, each keeping its columns.
    const uint32_t per_block = std::min((row_tiles + PT_WAVES - 1) / PT_WAVES, std::max(1u, POINT_GROUPS / nb));
    const dim3 grid(per_block * nb), block(64 * PT_WAVES);
    if (a.k <= 32) hipLaunchKernelGGL((point_kernel<M, 1, UP>), grid, block, 0, s, a);
    else if (a.k <= 64) hipLaunchKernelGGL((point_kernel<M, 2, UP>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((point_kernel<M, 3, UP>), grid, block, 0, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_point(const PointArgs &a, Math m, hipStream_t s) {
    if (!point_fits(a)) return hipErrorInvalidValue;
    if (a.ih)
        return m == Math::F16 ? point_slices<Math::F16, true>(a, s) : m == Math::SPLIT ? point_slices<Math::SPLIT, true>(a, s)
                                                                                       : point_slices<Math::F32, true>(a, s);
    // A transposed convolution was and stays a sum of f32 products.
    return m == Math::F16 ? point_slices<Math::F16, false>(a, s) : point_slices<Math::F32, false>(a, s);
}

}  // namespace bl
