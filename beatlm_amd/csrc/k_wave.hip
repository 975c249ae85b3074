// The wave-split product: C = A B + bias and the spec's epilogue for shapes
// whose tiles are too few for the ring kernel (gemm_pipe_kernel) to hide its
// serial k-loop: the MLP's second product and the out-projection at small
// token counts, the patch embedding, the decoder's 3x3 convolutions on images
// of up to a few thousand pixels.
//
// What bounds such a launch is latency: a ring of k-steps behind barriers is
// a chain of L2 round trips (fc2 at 257 tokens: 24 steps on 54 workgroups),
// and splitting k over workgroups costs a second launch (about 4.7 us each,
// back to back) to add the parts. Here the 8 waves of a workgroup split the
// k-steps of one small tile (wave w: steps w, w + 8, ...). Each wave issues
// all loads of up to NS of its steps at once, A by direct loads into LDS of
// its own (whole lines, no barrier), B straight into registers from the
// fragment-major pack (packed_at: 1 KB a load), waits once, multiplies, and
// leaves its partial tile in LDS; after the kernel's one barrier the first
// waves add the 8 partial tiles in wave order (deterministic) and run the
// epilogue, 8 consecutive columns an invocation, its operands loaded before
// the k-loop.
#include "k_gemm.inc"

namespace bl {
namespace {

constexpr int WV_WAVES = 8, WV_THREADS = 64 * WV_WAVES;

// One 32-wide k-slice's A fragments (rows 16 i + l16, k = 8 g .. 8 g + 7).
template <Math M, int TM> struct WaveA;
template <int TM> struct WaveA<Math::F16, TM> {
    f16x8 v[TM];
};
template <int TM> struct WaveA<Math::SPLIT, TM> {
    bf16x8 h[TM], l[TM];
};
template <int TM> struct WaveA<Math::F32, TM> {
    float v[TM][8];
};
// B's fragments of one slice: [plane][column block], 8 elements a lane.
template <Math M, int TN> struct WaveB {
    using V = typename std::conditional<M == Math::F16, f16x8, bf16x8>::type;
    V v[M == Math::SPLIT ? 2 : 1][TN];
};
template <int TN> struct WaveB<Math::F32, TN> {
    f32x4 v[2][TN];
};

template <Math M, int TN>
__device__ __forceinline__ void wave_load_b(const char *base, uint64_t plane_bytes, uint32_t blocks, uint32_t slice, int lane,
                                            WaveB<M, TN> &b) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const uint64_t at = ((uint64_t)j * blocks + slice) * 512 + lane * 8;  // elements
        if constexpr (M == Math::F32) {
            b.v[0][j] = *(const f32x4 *)(base + at * 4);
            b.v[1][j] = *(const f32x4 *)(base + at * 4 + 16);
        } else {
            using V = typename WaveB<M, TN>::V;
            b.v[0][j] = *(const V *)(base + at * 2);
            if constexpr (M == Math::SPLIT) b.v[1][j] = *(const V *)(base + plane_bytes + at * 2);
        }
    }
}

template <Math M, int TM, int TN>
__device__ __forceinline__ void wave_mma(f32x4 (&acc)[TM][TN], const WaveA<M, TM> &a, const WaveB<M, TN> &b) {
    if constexpr (M == Math::F16) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.v[i], b.v[0][j], acc[i][j], 0, 0, 0);
    } else if constexpr (M == Math::SPLIT) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l[i], b.v[0][j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h[i], b.v[1][j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h[i], b.v[0][j], acc[i][j], 0, 0, 0);
    } else {
        // Four k a product: lane group g gives k = 8 g + s of step s.
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[i][s], b.v[s / 4][j][s % 4], acc[i][j], 0, 0, 0);
    }
}

// Eight values of the lane's A fragment row as the math's operand; relu: the
// convolution's ReLU prologue.
template <Math M, int TM>
__device__ __forceinline__ void wave_take(WaveA<M, TM> &a, int i, const float (&v)[8]) {
    if constexpr (M == Math::SPLIT) {
        split8_bf16(v, a.h[i], a.l[i]);
    } else if constexpr (M == Math::F32) {
#pragma unroll
        for (int e = 0; e < 8; e++) a.v[i][e] = v[e];
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) a.v[i][e] = (_Float16)v[e];
    }
}

// LOAD: 0 plain rows, 2 the patch gather, 3 the 3x3 convolution's windows.
// AP: A kept as hi and lo bf16 planes (bf16x3). KS: 32-wide slices per k-step.
// NS: steps of a wave in flight at once.
// FOLD: the consumer of a folded LayerNorm (plain rows; it has no bias, and its
// epilogue's operands are loaded where they are used).
template <Math M, int BM, int BN, int LOAD, bool AP, int KS, int NS, bool FOLD = false>
__global__ __launch_bounds__(WV_THREADS, NS == 1 && BN == 32 ? 4 : 2) void gemm_wave_kernel(GemmArgs args) {
    using T = typename GemmTraits<M>::T;
    static_assert(!AP || (M == Math::SPLIT && LOAD != 2), "split A planes feed the bf16x3 math");
    static_assert(LOAD != 2 || KS == 1, "the patch gather takes one slice a step");
    constexpr int A_CPR = PipeTraits<M>::A_CPR * KS;
    constexpr int TM = BM / 16, TN = BN / 16;
    constexpr int STAGE = LOAD == 2 ? 0 : BM * A_CPR * 16;
    constexpr int TROW = BN + 4;
    constexpr int RED = BM * TROW * 4;
    constexpr int REGION = NS * STAGE > RED ? NS * STAGE : RED;  // one wave's LDS
    __shared__ __attribute__((aligned(16))) char smem[WV_WAVES * REGION];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    TileCoord tc;
    if (!xcd_tile(BM, BN, args, tc)) return;
    const uint32_t m0 = tc.m0, n0 = tc.n0, N = args.n, K = args.k, KP = args.k_pad, row_end = args.row1;
    const uint32_t a_limit = row_end - 1 - m0;  // rows past the part re-read its last row; never stored
    constexpr int AESZ = AP ? 2 : (int)sizeof(T), BESZ = M == Math::F32 ? 4 : 2;
    char *mine = smem + wave * REGION;

    // The epilogue's operands (chunk c = tid: 8 columns of one row).
    constexpr int CPR = BN / 8, CHUNKS = BM * CPR;
    static_assert(CHUNKS % 64 == 0 && CHUNKS <= WV_THREADS && CPR % 4 == 0, "whole waves of chunks, whole quads");
    const bool chunk = tid < CHUNKS;
    const int tr = tid / CPR, cc = tid % CPR;
    const uint32_t row = m0 + tr, col = n0 + 8 * cc;
    const bool live = chunk && row < row_end && col < N;
    const uint64_t idx = (uint64_t)row * N + col;
    // Of the epilogue's tensors the first two are loaded here (LayerScale, the
    // adds: a residual unit's sums take two); a step past them loads its own.
    Raw8<T> bias, op0, op1;
    bias.zero();
    op0.zero();
    op1.zero();
    // A folded LayerNorm's consumer (plain rows): the row's block statistics (a
    // quad's lane every fourth pair of blocks, as fold_load takes them), d and c.
    f32x4 stats[FOLD ? FOLD_PER : 1];
    Raw8<float> fd, fc;
    if constexpr (FOLD) {
        fd.zero();
        fc.zero();
        if (chunk) {
            const f32x4 *st = (const f32x4 *)(args.ln_stats + 2 * (uint64_t)min(row, row_end - 1) * args.ln_blocks);
#pragma unroll
            for (int q = 0; q < FOLD_PER; q++) {
                const uint32_t b = cc % 4 + 4 * q;
                stats[q] = b < args.ln_blocks / 2 ? st[b] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            if (col < N) {
                fd.load(args.ln_d + col);
                if (M == Math::F16) fc.load(args.ln_c + col);
            }
        }
    }
    const EpilogueArgs &epi = args.epi;
    auto operand8 = [&](int s, Raw8<T> &r) {
        if (epi.kind[s] == BL_EPI_ADD) r.load((const T *)epi.operand[s] + idx);
        else if (epi.kind[s] == BL_EPI_CHANNEL_SCALE && epi.channels[s] == N) r.load((const T *)epi.operand[s] + col);
    };
    if (!FOLD && live) {
        if (args.bias) bias.load((const T *)args.bias + col);
        if (epi.n > 0) operand8(0, op0);
        if (epi.n > 1) operand8(1, op1);
    }

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const uint32_t blocks = KP / 32, steps = blocks / KS;
    const char *Bb = (const char *)args.b + (uint64_t)(n0 / 16) * blocks * 512 * BESZ;
    const uint64_t b_plane = (uint64_t)args.n_pad * KP * 2;

    if constexpr (LOAD == 2) {
        // The lane's patches (rows l16 of each 16-row block): a patch's k runs
        // over P image rows of seg = P cin contiguous values each.
        const T *A = (const T *)args.a;
        const uint32_t gw = args.p0, P = args.p1, cin = args.p2, seg = P * cin, stride = args.p3 * cin;
        uint64_t pbase[TM];
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const uint32_t gr = m0 + min((uint32_t)(16 * i + l16), a_limit);
            pbase[i] = ((uint64_t)(gr / gw) * P * args.p3 + (uint64_t)(gr % gw) * P) * cin;
        }
        // Pairs of elements lie in one patch row when runs and offsets are even.
        const bool even = seg % 2 == 0 && stride % 2 == 0;
        typedef T T2 __attribute__((ext_vector_type(2)));
        for (uint32_t j0 = wave; j0 < steps; j0 += WV_WAVES * NS) {
            T av[NS][TM][8];
            WaveB<M, TN> bq[NS];
#pragma unroll
            for (int u = 0; u < NS; u++) {
                const uint32_t s = j0 + WV_WAVES * u;
                if (s < steps) {
                    const uint32_t k = 32 * s + 8 * g;
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        const uint32_t ke = k + e, y0 = ke / seg, x0 = ke - y0 * seg;
                        const uint32_t y1 = x0 + 1 == seg ? y0 + 1 : y0, x1 = x0 + 1 == seg ? 0 : x0 + 1;
#pragma unroll
                        for (int i = 0; i < TM; i++) {
                            T v0 = (T)0, v1 = (T)0;
                            if (even) {
                                if (ke < K) {
                                    const T2 w = *(const T2 *)(A + pbase[i] + (uint64_t)y0 * stride + x0);
                                    v0 = w[0];
                                    v1 = w[1];
                                }
                            } else {
                                if (ke < K) v0 = A[pbase[i] + (uint64_t)y0 * stride + x0];
                                if (ke + 1 < K) v1 = A[pbase[i] + (uint64_t)y1 * stride + x1];
                            }
                            av[u][i][e] = v0;
                            av[u][i][e + 1] = v1;
                        }
                    }
                    wave_load_b<M, TN>(Bb, b_plane, blocks, s, lane, bq[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < NS; u++) {
                if (j0 + WV_WAVES * u < steps) {
                    WaveA<M, TM> a;
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        float v[8];
#pragma unroll
                        for (int e = 0; e < 8; e++) v[e] = to_f32(av[u][i][e]);
                        wave_take<M, TM>(a, i, v);
                    }
                    wave_mma<M, TM, TN>(acc, a, bq[u]);
                }
            }
        }
    } else {
        using RLoader = RowLoader<BM, A_CPR, 1>;
        constexpr int EPC = AP ? 8 : 16 / (int)sizeof(T);  // A elements per 16-byte chunk
        using Loader = typename std::conditional<LOAD == 3, ConvLoader<BM, A_CPR, EPC, AP, 1>, RLoader>::type;
        auto make = [&]() {
            if constexpr (LOAD == 3) return Loader(args, m0, a_limit, 0, lane);
            else return Loader(K * AESZ, a_limit, 0, lane, AP ? (uint32_t)(args.a_planes * 2) : 0u);
        };
        const Loader load = make();
        if constexpr (FOLD && M != Math::F16) {
            // A centred fold's correction (fold_correct) from the last wave,
            // which has the fewest steps: delta[row][block] = the block's mean
            // less the row's, times cb, one more 32-deep slice. Lane group g
            // holds blocks 8 g .. 8 g + 7 of both.
            if (wave == WV_WAVES - 1) {
                WaveA<M, TM> da;
                WaveB<M, TN> cb;
                const uint32_t nb = args.ln_blocks;
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const uint32_t r = m0 + min((uint32_t)(16 * i + l16), a_limit);
                    const f32x4 *st = (const f32x4 *)(args.ln_stats + 2 * ((uint64_t)r * nb + 8 * g));
                    float d[8], sum = 0.0f;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const f32x4 x = 8 * g + 2 * q < nb ? st[q] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                        d[2 * q] = x[0];
                        d[2 * q + 1] = x[2];
                        sum += x[0] + x[2];
                    }
                    sum += __shfl_xor(sum, 16, WAVE);
                    sum += __shfl_xor(sum, 32, WAVE);
                    const float mean = sum / (float)nb;
#pragma unroll
                    for (int e = 0; e < 8; e++) d[e] = 8 * g + e < nb ? d[e] - mean : 0.0f;
                    wave_take<M, TM>(da, i, d);
                }
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const f32x4 *p = (const f32x4 *)(args.ln_cb + (uint64_t)(n0 + 16 * j + l16) * 32 + 8 * g);
                    const f32x4 c0 = p[0], c1 = p[1];
                    if constexpr (M == Math::F32) {
                        cb.v[0][j] = c0;
                        cb.v[1][j] = c1;
                    } else {
                        float c[8];
#pragma unroll
                        for (int e = 0; e < 8; e++) c[e] = e < 4 ? c0[e] : c1[e - 4];
                        split8_bf16(c, cb.v[0][j], cb.v[1][j]);
                    }
                }
                wave_mma<M, TM, TN>(acc, da, cb);
            }
        }
        const char *Ab = (const char *)args.a + (uint64_t)m0 * K * AESZ;
        constexpr int AROWB = A_CPR * 16;
        const int xa = swz<A_CPR>(l16, 0);
        for (uint32_t j0 = wave; j0 < steps; j0 += WV_WAVES * NS) {
            WaveB<M, TN> bq[NS][KS];
            // The round before is done with this wave's LDS.
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            asm volatile("" ::: "memory");
#pragma unroll
            for (int u = 0; u < NS; u++) {
                const uint32_t s = j0 + WV_WAVES * u;
                if (s < steps) {
                    if constexpr (LOAD == 3) load.template issue<T>(args, s * 32 * KS, mine + u * STAGE);
                    else load.issue(Ab + (uint64_t)s * 32 * KS * AESZ, mine + u * STAGE);
#pragma unroll
                    for (int ks = 0; ks < KS; ks++) wave_load_b<M, TN>(Bb, b_plane, blocks, s * KS + ks, lane, bq[u][ks]);
                }
            }
            wait_vmcnt<0>();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int u = 0; u < NS; u++) {
                if (j0 + WV_WAVES * u < steps) {
#pragma unroll
                    for (int ks = 0; ks < KS; ks++) {
                        WaveA<M, TM> a;
#pragma unroll
                        for (int i = 0; i < TM; i++) {
                            const char *as = mine + u * STAGE + (16 * i + l16) * AROWB;
                            if constexpr (AP) {
                                a.h[i] = *(const bf16x8 *)(as + (((4 * ks + g) ^ xa) << 4));
                                a.l[i] = *(const bf16x8 *)(as + (((A_CPR / 2 + 4 * ks + g) ^ xa) << 4));
                                if (LOAD == 3 && args.p5) {
                                    // x = hi + lo has hi's sign; a zero hi leaves x below the smallest bf16.
#pragma unroll
                                    for (int e = 0; e < 8; e++) {
                                        const bool keep = (float)a.h[i][e] > 0.0f;
                                        a.h[i][e] = keep ? a.h[i][e] : (__bf16)0.0f;
                                        a.l[i][e] = keep ? a.l[i][e] : (__bf16)0.0f;
                                    }
                                }
                            } else if constexpr (M == Math::F16) {
                                a.v[i] = *(const f16x8 *)(as + (((4 * ks + g) ^ xa) << 4));
                                if (LOAD == 3 && args.p5) {
#pragma unroll
                                    for (int e = 0; e < 8; e++) a.v[i][e] = a.v[i][e] > (_Float16)0 ? a.v[i][e] : (_Float16)0;
                                }
                            } else {
                                const f32x4 x0 = *(const f32x4 *)(as + (((8 * ks + 2 * g) ^ xa) << 4));
                                const f32x4 x1 = *(const f32x4 *)(as + (((8 * ks + 2 * g + 1) ^ xa) << 4));
                                float v[8];
#pragma unroll
                                for (int e = 0; e < 8; e++) {
                                    v[e] = e < 4 ? x0[e] : x1[e - 4];
                                    if (LOAD == 3 && args.p5) v[e] = fmaxf(v[e], 0.0f);
                                }
                                wave_take<M, TM>(a, i, v);
                            }
                        }
                        wave_mma<M, TM, TN>(acc, a, bq[u][ks]);
                    }
                }
            }
        }
    }

    // This wave's partial tile, in its own LDS (its fragment reads are done:
    // the products above took them).
    float *part = (float *)mine;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) part[(16 * i + 4 * g + r) * TROW + 16 * j + l16] = acc[i][j][r];
    __syncthreads();
    if (LOAD == 2 && args.cls_out && m0 == args.row0 && wave == WV_WAVES - 1) cls_row<M, T>(args, n0, BN, lane);  // x's first row
    // The attention's operands: K and V columns of a QKV projection.
    constexpr bool FLASH = LOAD == 0 && M != Math::F32;
    const uint32_t D = N / 3;
    const bool k_region = FLASH && args.flash_ops && n0 >= D && n0 < 2 * D, v_region = FLASH && args.flash_ops && n0 >= 2 * D;
    if (chunk) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = 0.0f;
#pragma unroll
    for (int w = 0; w < WV_WAVES; w++) {
        const float *p = (const float *)(smem + w * REGION) + tr * TROW + 8 * cc;
        const f32x4 x0 = *(const f32x4 *)p, x1 = *(const f32x4 *)(p + 4);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] += e < 4 ? x0[e] : x1[e - 4];
    }
    if constexpr (FOLD) {
        // The row's mean and variance from its blocks', as fold_finish.
        float s = 0.0f, m2 = 0.0f;
#pragma unroll
        for (int q = 0; q < FOLD_PER; q++) s += stats[q][0] + stats[q][2];
        const float mean = quad_sum(s) * (1.0f / (float)args.ln_blocks);
#pragma unroll
        for (int q = 0; q < FOLD_PER; q++) {
            const float d0 = stats[q][0] - mean, d1 = stats[q][2] - mean;
            if (cc % 4 + 4 * q < args.ln_blocks / 2) m2 += stats[q][1] + stats[q][3] + 32.0f * (d0 * d0 + d1 * d1);
        }
        m2 = quad_sum(m2);
        const float rstd = 1.0f / sqrtf(m2 / (float)(32 * args.ln_blocks) + args.ln_eps), shift = M == Math::F16 ? mean : 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = rstd * (v[e] - (M == Math::F16 ? shift * fc.at(e) : 0.0f)) + fd.at(e);
    }
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] += bias.at(e);
    if (live) {
        // The steps in order, each over the chunk.
        for (int st = 0; st < epi.n; st++) {
            const int kind = epi.kind[st];
            if (kind == BL_EPI_ADD) {
                Raw8<T> o = st == 0 ? op0 : op1;
                if (FOLD || st > 1) o.load((const T *)epi.operand[st] + idx);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] += o.at(e);
            } else if (kind == BL_EPI_CHANNEL_SCALE && epi.channels[st] == N) {
                Raw8<T> o = st == 0 ? op0 : op1;
                if (FOLD || st > 1) o.load((const T *)epi.operand[st] + col);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] *= o.at(e);
            } else if (kind == BL_EPI_CHANNEL_SCALE) {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] *= to_f32(((const T *)epi.operand[st])[(idx + e) % epi.channels[st]]);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    if (kind == BL_EPI_RELU) v[e] = fmaxf(v[e], 0.0f);
                    else if (kind == BL_EPI_GELU) v[e] = gelu_tanh(v[e]);
                    else if (kind == BL_EPI_GELU_ERF) v[e] = gelu_erf(v[e]);
                    else if (kind == BL_EPI_SCALE) v[e] *= epi.factor[st];
                }
            }
        }
    }
    if (live && !(args.flash_ops == 2 && (k_region || v_region))) store8<T>((T *)args.c, idx, v, args.c_planes);
    if constexpr (FLASH) {
        if (k_region && live) {
            const uint32_t kc = col - D;
            store8_operand<M>(args.fl_kp, ((uint64_t)(kc / 64) * args.fl_tpad + row) * 64 + kc % 64, v,
                              (uint64_t)(D / 64) * args.fl_tpad * 64);
        }
        if (v_region) {
            // Into wave 0's partial tile (this invocation's own chunk) for the pass by columns.
            float *t = (float *)smem + tr * TROW + 8 * cc;
            *(f32x4 *)t = f32x4{v[0], v[1], v[2], v[3]};
            *(f32x4 *)(t + 4) = f32x4{v[4], v[5], v[6], v[7]};
        }
    }
    if (args.ln_out) {
        // A fold's producer: the 32-column block of the values as stored is
        // the 4 chunks of one quad.
        float k[8], s = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            k[e] = to_f32(from_f32<T>(v[e]));
            s += k[e];
        }
        const float mean = quad_sum(s) * (1.0f / 32.0f);
        float m2 = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) m2 += (k[e] - mean) * (k[e] - mean);
        m2 = quad_sum(m2);
        if (live && cc % 4 == 0) *(f32x2 *)(args.ln_out + 2 * ((uint64_t)row * (N / 32) + col / 32)) = f32x2{mean, m2};
        if constexpr (sizeof(T) == 4)
            if (args.ln_shadow && live) {
                // The consumer's A: the values less their block's mean.
                float dv[8];
#pragma unroll
                for (int e = 0; e < 8; e++) dv[e] = k[e] - mean;
                store8<T>((T *)args.ln_shadow, idx, dv, M == Math::SPLIT ? (args.ln_plane ? args.ln_plane : (uint64_t)args.m * N) : 0);
            }
    }
    }
    if constexpr (FLASH) {
        if (v_region) {
            // Column cl, 16 tokens, as chunk_epilogue writes them: m0 is a
            // multiple of 16, position s of the run holds token vt_pos(s).
            __syncthreads();
            const float *tile = (const float *)smem;
            const uint64_t plane = (uint64_t)(D / 64) * args.fl_tpad * 64;
            if (tid < BN * (BM / 16)) {
                const int cl = tid % BN, tr0 = tid / BN * 16;
                const uint32_t row0 = m0 + tr0, vc = n0 + cl - 2 * D;
                const uint64_t base = (uint64_t)vc * args.fl_tpad;
                if (row0 < row_end) {
                    float y0[8], y1[8];
#pragma unroll
                    for (int s = 0; s < 8; s++) {
                        y0[s] = tile[(tr0 + vt_pos(s)) * TROW + cl];
                        y1[s] = tile[(tr0 + vt_pos(s + 8)) * TROW + cl];
                    }
                    if (row0 + 16 <= row_end) {
                        store8_operand<M>(args.fl_vt, base + row0, y0, plane);
                        store8_operand<M>(args.fl_vt, base + row0 + 8, y1, plane);
                    } else {
#pragma unroll
                        for (int s = 0; s < 16; s++) {
                            if (row0 + vt_pos(s) >= row_end) continue;
                            const float x = s < 8 ? y0[s] : y1[s - 8];
                            const uint64_t i = base + row0 + s;
                            if constexpr (M == Math::SPLIT) {
                                __bf16 h, l;
                                split_bf16(x, h, l);
                                ((__bf16 *)args.fl_vt)[i] = h;
                                ((__bf16 *)args.fl_vt)[plane + i] = l;
                            } else {
                                ((_Float16 *)args.fl_vt)[i] = (_Float16)x;
                            }
                        }
                    }
                }
            }
        }
    }
}

template <Math M, int BM, int BN, int LOAD, bool AP, int KS>
hipError_t wave_ns(const GemmArgs &a, hipStream_t s) {
    const dim3 grid(xcd_grid(BM, BN, a)), block(WV_THREADS);
    if constexpr (LOAD == 0) {
        // x of at most 1024 columns: one or two steps a wave.
        if (a.ln_stats) {
            if (a.k <= 64 * WV_WAVES) hipLaunchKernelGGL((gemm_wave_kernel<M, BM, BN, LOAD, AP, KS, 1, true>), grid, block, 0, s, a);
            else hipLaunchKernelGGL((gemm_wave_kernel<M, BM, BN, LOAD, AP, KS, 2, true>), grid, block, 0, s, a);
            return hipGetLastError();
        }
    }
    if constexpr (LOAD == 2) {
        hipLaunchKernelGGL((gemm_wave_kernel<M, BM, BN, LOAD, AP, KS, 3>), grid, block, 0, s, a);
    } else {
        // As many steps a wave in flight as it has, where LDS holds them: 1 or
        // 2 (so that two workgroups fit a CU), 4, or 8.
        constexpr int STAGE = WV_WAVES * BM * PipeTraits<M>::A_CPR * KS * 16;
        const uint32_t n = (a.k_pad / (32 * KS) + WV_WAVES - 1) / WV_WAVES;
        if constexpr (M == Math::F16 && 8 * STAGE <= 160 * 1024 && LOAD == 0) {
            if (n > 4) {
                hipLaunchKernelGGL((gemm_wave_kernel<M, BM, BN, LOAD, AP, KS, 8>), grid, block, 0, s, a);
                return hipGetLastError();
            }
        }
        if constexpr (M == Math::F16 && BM == 32 && BN == 32 && LOAD == 0) {
            if (n == 1) {
                hipLaunchKernelGGL((gemm_wave_kernel<M, BM, BN, LOAD, AP, KS, 1>), grid, block, 0, s, a);
                return hipGetLastError();
            }
        }
        if constexpr (4 * STAGE <= 160 * 1024) {
            if (n > 2) {
                hipLaunchKernelGGL((gemm_wave_kernel<M, BM, BN, LOAD, AP, KS, 4>), grid, block, 0, s, a);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL((gemm_wave_kernel<M, BM, BN, LOAD, AP, KS, 2>), grid, block, 0, s, a);
    }
    return hipGetLastError();
}

template <Math M, int BM, int BN>
hipError_t wave_load(const GemmArgs &a, hipStream_t s) {
    if (a.load == 2) return a.a_planes ? hipErrorInvalidValue : wave_ns<M, BM, BN, 2, false, 1>(a, s);
    // A k-step stays inside one tap where it can.
    const bool two = a.load == 3 ? a.p2 % 64 == 0 : a.k % 64 == 0;
    if (a.load == 3) {
        if constexpr (M == Math::SPLIT) {
            if (a.a_planes) return two ? wave_ns<M, BM, BN, 3, true, 2>(a, s) : wave_ns<M, BM, BN, 3, true, 1>(a, s);
        }
        return two ? wave_ns<M, BM, BN, 3, false, 2>(a, s) : wave_ns<M, BM, BN, 3, false, 1>(a, s);
    }
    if (!two) return hipErrorInvalidValue;
    if constexpr (M == Math::SPLIT) {
        if (a.a_planes) return wave_ns<M, BM, BN, 0, true, 2>(a, s);
    }
    return wave_ns<M, BM, BN, 0, false, 2>(a, s);
}

template <Math M>
hipError_t wave_tile(const GemmArgs &a, int tile, hipStream_t s) {
    return tile == TILE_W32x32 ? wave_load<M, 32, 32>(a, s)
         : tile == TILE_W32x64 ? wave_load<M, 32, 64>(a, s) : wave_load<M, 16, 32>(a, s);
}

}  // namespace

hipError_t launch_gemm_wave(const GemmArgs &a, Math m, int tile, hipStream_t s) {
    if (!gemm_wave_fits(a, m)) return hipErrorInvalidValue;
    if (a.a_planes && m != Math::SPLIT) return hipErrorInvalidValue;
    return m == Math::F32 ? wave_tile<Math::F32>(a, tile, s)
         : m == Math::SPLIT ? wave_tile<Math::SPLIT>(a, tile, s) : wave_tile<Math::F16>(a, tile, s);
}

}  // namespace bl
