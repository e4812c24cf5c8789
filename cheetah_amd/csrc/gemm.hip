// Prefill GEMM Y[n, rows] = X[n, cols] · Wᵀ on the gfx950 matrix cores
// (the batched projections of forward_layer_chunk, qwen2.rs:240-426; gemm,
// ops.rs:308, and the per-row quantized linear_batch loop, ops.rs:1244-1326).
//
// Operands: W stays in the reference layout and is converted to BF16 while
// it is staged into LDS — BF16 as stored, Q8/Q4 codes exactly (|code| <= 127
// fits BF16's 8-bit significand) with the row scale applied to the f32 sum in
// the epilogue. X is f32; it is split into hi = bf16(x) and lo = bf16(x - hi)
// so two v_mfma_f32_32x32x16_bf16 per k-step carry x to ~2^-17 relative
// error (f32 accumulation), instead of bf16's 2^-9.
//
// Tiling: blocks of 64 x 128, 128 x 128 or 128 x 256 (tokens x weight rows),
// chosen with the K split by ring_plan; K advances 32 per LDS stage, the next
// stages' copies in flight during the MFMAs.
//
// Accumulation order: K is cut into chunks of a depth fixed by K alone; each
// chunk is accumulated from zero. A single matrix's n chunk sums are folded
// as two halves, t = (c0 + ... + c(h-1)) + (ch + ... + c(n-1)) with
// h = ceil(n / 2), each half left to right (for n <= 3 this is the plain left
// fold); the dual gate/up GEMM folds its chunks left to right. With many tiles
// a block folds its chunks in registers; with fewer tiles the chunks go to
// split-K blocks (every chunk its own block, or a single matrix's two halves
// one block each) and the stored sums are folded by a reduce kernel or by the
// kernel that reads the output, in the same association. Every path gives
// the same bits, so a token's outputs never depend on how many tokens share
// the call (chunked prefill stays bit-exact however the prompt is cut).
#include <algorithm>
#include <cstdlib>

#include "kernels.hpp"

namespace chip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;
constexpr int BN = 128, BK = 32;
constexpr int LDK = BK + 8;  // 80-byte LDS rows: 16 consecutive rows start on distinct bank groups

struct GArgs {
    const uint8_t *w, *w2;
    const float *sc, *sc2;
    size_t stride;
    int N, K, M;  // N = weight rows, K = cols, M = tokens
    const float *x;
    const uint16_t *xh, *xl;  // x pre-split into hi / lo BF16 halves, [M][xs] (or null)
    int xs;                   // elements between rows of xh / xl (K, or K padded with zeros)
    const float *bias;
    float *y, *residual;
    uint16_t *yh, *yl;  // SwiGLU: the output also as BF16 halves (or null)
    int defer;          // split-K: leave the chunk sums for the caller
    int epi;
    int chunk, nchunks;  // accumulation chunk depth (multiple of BK) and count
    int nstored;         // split-K: sums stored per output (nchunks, or 2 halves of a single matrix)
    int n_first, n_tiles;  // ring: first weight row and row tiles of the launch (0 tiles: to the end)
    float *ws;           // split-K: [nstored][M][N] sums (a second set for the dual matrix)
    int vec_x, vec_w;    // 16-byte global loads allowed
};

__device__ __forceinline__ uint32_t pack2(uint16_t lo, uint16_t hi) { return (uint32_t)lo | ((uint32_t)hi << 16); }

// BF16 bits of a small integer code (exact).
__device__ __forceinline__ uint16_t code_bf16(int code) { return (uint16_t)(__float_as_uint((float)code) >> 16); }

__device__ __forceinline__ bf16x8 frag(const uint16_t *base, int row, int k) {
    return __builtin_bit_cast(bf16x8, *(const u32x4 *)(base + row * LDK + k));
}

// One stage's operands in flight: X as f32, W as raw reference bytes.
template <int MT>
struct Regs {
    static constexpr int XV = 64 * MT * BK / 4 / kThreads;  // float4 per thread
    static constexpr int XB = 64 * MT * BK / 8 / kThreads;  // 8-element BF16 chunks per thread
    f32x4 x[XV];
    u32x4 xh[XB], xl[XB];
    u32x4 w[2];   // BF16: 2 x 8 elements; Q8: w[0] = 16 codes; Q4: w[0].xy = 16 codes
    u32x4 w2[2];  // dual matrix
};

template <int MT>
__device__ __forceinline__ void load_x(const GArgs &a, int m0, int k0, Regs<MT> &r) {
#pragma unroll
    for (int i = 0; i < Regs<MT>::XV; ++i) {
        const int c = threadIdx.x + kThreads * i;
        const int row = c >> 3, kc = (c & 7) * 4;
        const int m = m0 + row, k = k0 + kc;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (m < a.M && k < a.K) {
            const float *src = a.x + (size_t)m * a.K + k;
            if (a.vec_x) {
                v = *(const f32x4 *)src;
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = k + q < a.K ? src[q] : 0.f;
            }
        }
        r.x[i] = v;
    }
}

// Pre-split x: BM x BK BF16 per half, 16-byte chunks (K % 8 == 0).
template <int MT>
__device__ __forceinline__ void load_xs(const GArgs &a, int m0, int k0, Regs<MT> &r) {
#pragma unroll
    for (int i = 0; i < Regs<MT>::XB; ++i) {
        const int c = threadIdx.x + kThreads * i;
        const int row = c >> 2, kc = (c & 3) * 8;
        const int m = m0 + row, k = k0 + kc;
        if (m < a.M && k < a.K) {
            r.xh[i] = *(const u32x4 *)(a.xh + (size_t)m * a.K + k);
            r.xl[i] = *(const u32x4 *)(a.xl + (size_t)m * a.K + k);
        } else {
            r.xh[i] = u32x4{0u, 0u, 0u, 0u};
            r.xl[i] = u32x4{0u, 0u, 0u, 0u};
        }
    }
}

template <int MT>
__device__ __forceinline__ void store_xs(const Regs<MT> &r, uint16_t *xh, uint16_t *xl) {
#pragma unroll
    for (int i = 0; i < Regs<MT>::XB; ++i) {
        const int c = threadIdx.x + kThreads * i;
        *(u32x4 *)(xh + (c >> 2) * LDK + (c & 3) * 8) = r.xh[i];
        *(u32x4 *)(xl + (c >> 2) * LDK + (c & 3) * 8) = r.xl[i];
    }
}

template <int MT>
__device__ __forceinline__ void store_x(const Regs<MT> &r, uint16_t *xh, uint16_t *xl) {
#pragma unroll
    for (int i = 0; i < Regs<MT>::XV; ++i) {
        const int c = threadIdx.x + kThreads * i;
        const int row = c >> 3, kc = (c & 7) * 4;
        uint16_t h[4], l[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const __bf16 hb = (__bf16)r.x[i][q];
            h[q] = __builtin_bit_cast(uint16_t, hb);
            l[q] = __builtin_bit_cast(uint16_t, (__bf16)(r.x[i][q] - (float)hb));
        }
        *(uint2 *)(xh + row * LDK + kc) = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
        *(uint2 *)(xl + row * LDK + kc) = make_uint2(pack2(l[0], l[1]), pack2(l[2], l[3]));
    }
}

// W stage: BN rows x BK columns of the reference layout.
template <int FMT>
__device__ __forceinline__ void load_w(const GArgs &a, const uint8_t *w, int n0, int k0, u32x4 (&out)[2]) {
    const int tid = threadIdx.x;
    if constexpr (FMT == FMT_BF16) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = tid + kThreads * j;
            const int row = c >> 2, kc = (c & 3) * 8;
            const int n = n0 + row, k = k0 + kc;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (n < a.N && k < a.K) {
                const uint16_t *src = (const uint16_t *)(w + (size_t)n * a.stride) + k;
                if (a.vec_w) {
                    v = *(const u32x4 *)src;
                } else {
                    uint16_t e[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) e[q] = k + q < a.K ? src[q] : 0;
                    v = u32x4{pack2(e[0], e[1]), pack2(e[2], e[3]), pack2(e[4], e[5]), pack2(e[6], e[7])};
                }
            }
            out[j] = v;
        }
    } else {
        // Q8 / Q4: 16 codes per thread, rows tid / 2, codes 16 (tid % 2) ..
        const int row = tid >> 1, kc = (tid & 1) * 16;
        const int n = n0 + row, k = k0 + kc;
        u32x4 v = {0u, 0u, 0u, 0u};
        if (n < a.N && k < a.K) {
            const uint8_t *rp = w + (size_t)n * a.stride;
            if constexpr (FMT == FMT_Q8) {
                if (a.vec_w) {
                    v = *(const u32x4 *)(rp + k);
                } else {
                    uint32_t d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                    for (int q = 0; q < 16; ++q)
                        if (k + q < a.K) d[q >> 2] |= (uint32_t)rp[k + q] << (8 * (q & 3));
                    v = u32x4{d[0], d[1], d[2], d[3]};
                }
            } else {
                // Rows are 4-byte aligned; k is a multiple of 16, so the 8 code
                // bytes are 8-byte aligned within the row.
                if (k + 16 <= a.K) {
                    const uint32_t *p = (const uint32_t *)(rp + (k >> 1));
                    v = u32x4{p[0], p[1], 0u, 0u};
                } else {
                    uint32_t d[2] = {0u, 0u};
                    for (int q = 0; q < 16 && k + q < a.K; ++q) {
                        const uint8_t byte = rp[(k + q) >> 1];
                        const uint32_t nib = ((k + q) & 1) ? (byte >> 4) : (byte & 0xF);
                        d[q >> 3] |= nib << (4 * (q & 7));
                    }
                    v = u32x4{d[0], d[1], 0u, 0u};
                }
            }
        }
        out[0] = v;
    }
}

template <int FMT>
__device__ __forceinline__ void store_w(const u32x4 (&in)[2], uint16_t *ws) {
    const int tid = threadIdx.x;
    if constexpr (FMT == FMT_BF16) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = tid + kThreads * j;
            *(u32x4 *)(ws + (c >> 2) * LDK + (c & 3) * 8) = in[j];
        }
    } else {
        const int row = tid >> 1, kc = (tid & 1) * 16;
        uint16_t e[16];
        if constexpr (FMT == FMT_Q8) {
#pragma unroll
            for (int q = 0; q < 16; ++q) e[q] = code_bf16((int)(int8_t)(in[0][q >> 2] >> (8 * (q & 3))));
        } else {
#pragma unroll
            for (int q = 0; q < 16; ++q) e[q] = code_bf16(((int)(in[0][q >> 3] << (28 - 4 * (q & 7)))) >> 28);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
            *(u32x4 *)(ws + row * LDK + kc + 8 * h) =
                u32x4{pack2(e[8 * h], e[8 * h + 1]), pack2(e[8 * h + 2], e[8 * h + 3]),
                      pack2(e[8 * h + 4], e[8 * h + 5]), pack2(e[8 * h + 6], e[8 * h + 7])};
    }
}

// out = f(v * row scale (+ bias)); dual: SwiGLU of gate v and up u.
template <bool DUAL>
__device__ __forceinline__ void epilogue(const GArgs &a, int m, int n, float v, float u) {
    if (a.sc) v = v * a.sc[n];
    const size_t o = (size_t)m * a.N + n;
    if constexpr (DUAL) {
        if (a.sc2) u = u * a.sc2[n];
        // silu_multiply, ops.rs:743-747: g * (u / (1 + exp(-g))).
        const float g = v * (u / (1.0f + expf(-v)));
        if (a.y) a.y[o] = g;
        if (a.yh) {
            const __bf16 hb = (__bf16)g;
            a.yh[o] = __builtin_bit_cast(uint16_t, hb);
            a.yl[o] = __builtin_bit_cast(uint16_t, (__bf16)(g - (float)hb));
        }
    } else {
        if (a.bias) v = v + a.bias[n];
        if (a.epi == EPI_RESIDUAL) a.residual[o] = a.residual[o] + v;
        else a.y[o] = v;
    }
}

// The epilogue for one lane's outputs of a finished tile: column n per j,
// rows m = mbase + 32 i + 8 (q / 4) + 4 (lane / 32) + q % 4. The column's scale
// and bias, then a 32-row block's residuals, are loaded before any store (one
// wait instead of one per output); each output's arithmetic is epilogue's.
template <bool DUAL, int MT, int NJ = 2>
__device__ __forceinline__ void epilogue_tile(const GArgs &a, const f32x16 (&tot)[MT][NJ],
                                              const f32x16 (&tot2)[DUAL ? MT : 1][NJ], int mbase, int nbase, int lane) {
    const bool resid = !DUAL && a.epi == EPI_RESIDUAL;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int n = nbase + 32 * j + (lane & 31);
        if (n >= a.N) continue;
        const float scn = a.sc ? a.sc[n] : 1.0f;
        const float sc2n = DUAL && a.sc2 ? a.sc2[n] : 1.0f;
        const float bn = !DUAL && a.bias ? a.bias[n] : 0.0f;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            float res[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int m = mbase + 32 * i + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
                res[q] = resid && m < a.M ? a.residual[(size_t)m * a.N + n] : 0.0f;
            }
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int m = mbase + 32 * i + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
                if (m >= a.M) continue;
                const size_t o = (size_t)m * a.N + n;
                float v = tot[i][j][q];
                if (a.sc) v = v * scn;
                if constexpr (DUAL) {
                    float u = tot2[i][j][q];
                    if (a.sc2) u = u * sc2n;
                    // silu_multiply, ops.rs:743-747: g * (u / (1 + exp(-g))).
                    const float g = v * (u / (1.0f + expf(-v)));
                    if (a.y) a.y[o] = g;
                    if (a.yh) {
                        const __bf16 hb = (__bf16)g;
                        a.yh[o] = __builtin_bit_cast(uint16_t, hb);
                        a.yl[o] = __builtin_bit_cast(uint16_t, (__bf16)(g - (float)hb));
                    }
                } else {
                    if (a.bias) v = v + bn;
                    if (resid) a.residual[o] = res[q] + v;
                    else a.y[o] = v;
                }
            }
        }
    }
}

// Output tile of this block. Blocks are numbered so that the token tiles of
// one weight-row tile are consecutive, and (with the 8 XCDs taking block ids
// round-robin) run on one XCD: each weight tile streams from HBM about once
// and the block's neighbours find it in that XCD's L2, instead of every token
// tile re-reading the whole matrix.
__device__ __forceinline__ void tile_of(int nN, int nM, int &n0, int &m0, int BMt, int BNt = BN) {
    const int total = nN * nM, bid = blockIdx.x;
    const int lid = total % 8 == 0 ? (bid % 8) * (total / 8) + bid / 8 : bid;
    m0 = (lid % nM) * BMt;
    n0 = (lid / nM) * BNt;
}

// blockIdx: x = output tile (tile_of), z = chunk (split-K) or 0.
template <int FMT, bool DUAL, int MT, bool PRE>
__global__ __launch_bounds__(kThreads) void gemm_kernel(GArgs a, int split) {
    constexpr int BM = 64 * MT;
    __shared__ __attribute__((aligned(16))) uint16_t xh[2][BM * LDK];
    __shared__ __attribute__((aligned(16))) uint16_t xl[2][BM * LDK];
    __shared__ __attribute__((aligned(16))) uint16_t wsm[2][BN * LDK];
    __shared__ __attribute__((aligned(16))) uint16_t wsm2[DUAL ? 2 : 1][DUAL ? BN * LDK : 8];

    int n0, m0;
    tile_of((a.N + BN - 1) / BN, (a.M + BM - 1) / BM, n0, m0, BM);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * 32 * MT, wn = (wave & 1) * 64;
    const int kbeg = split ? blockIdx.z * a.chunk : 0;
    const int kend = split ? min(a.K, kbeg + a.chunk) : a.K;
    // Single matrix, folding in registers: the first half's total moves to
    // th when the second half begins (two-half association).
    const int khalf = (a.nchunks + 1) / 2 * a.chunk;

    f32x16 acc[MT][2], acc2[DUAL ? MT : 1][2], tot[MT][2], tot2[DUAL ? MT : 1][2], th[DUAL ? 1 : MT][2];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            acc[i][j] = f32x16{};
            tot[i][j] = f32x16{};
            if constexpr (DUAL) {
                acc2[i][j] = f32x16{};
                tot2[i][j] = f32x16{};
            } else {
                th[i][j] = f32x16{};
            }
        }

    Regs<MT> r;
    if constexpr (PRE) load_xs<MT>(a, m0, kbeg, r);
    else load_x<MT>(a, m0, kbeg, r);
    load_w<FMT>(a, a.w, n0, kbeg, r.w);
    if constexpr (DUAL) load_w<FMT>(a, a.w2, n0, kbeg, r.w2);
    if constexpr (PRE) store_xs<MT>(r, xh[0], xl[0]);
    else store_x<MT>(r, xh[0], xl[0]);
    store_w<FMT>(r.w, wsm[0]);
    if constexpr (DUAL) store_w<FMT>(r.w2, wsm2[0]);
    __syncthreads();
    int b = 0;
    for (int k0 = kbeg; k0 < kend; k0 += BK) {
        const bool more = k0 + BK < kend;
        if (more) {
            if constexpr (PRE) load_xs<MT>(a, m0, k0 + BK, r);
            else load_x<MT>(a, m0, k0 + BK, r);
            load_w<FMT>(a, a.w, n0, k0 + BK, r.w);
            if constexpr (DUAL) load_w<FMT>(a, a.w2, n0, k0 + BK, r.w2);
        }
#pragma unroll
        for (int ks = 0; ks < BK; ks += 16) {
            const int kf = ks + 8 * (lane >> 5);
            bf16x8 ah[MT], al[MT], bw[2], bw2[DUAL ? 2 : 1];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                ah[i] = frag(xh[b], wm + 32 * i + (lane & 31), kf);
                al[i] = frag(xl[b], wm + 32 * i + (lane & 31), kf);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                bw[j] = frag(wsm[b], wn + 32 * j + (lane & 31), kf);
                if constexpr (DUAL) bw2[j] = frag(wsm2[b], wn + 32 * j + (lane & 31), kf);
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bw[j], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], bw[j], acc[i][j], 0, 0, 0);
                    if constexpr (DUAL) {
                        acc2[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bw2[j], acc2[i][j], 0, 0, 0);
                        acc2[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], bw2[j], acc2[i][j], 0, 0, 0);
                    }
                }
        }
        // Chunk end: fold the chunk sum into the running total (t += c); a
        // single matrix's first half ends here: th = t, t = 0.
        if (k0 + BK >= kend || ((k0 + BK) % a.chunk) == 0) {
            const bool half_end = !DUAL && !split && k0 + BK == khalf && khalf < kend;
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    tot[i][j] += acc[i][j];
                    acc[i][j] = f32x16{};
                    if constexpr (DUAL) {
                        tot2[i][j] += acc2[i][j];
                        acc2[i][j] = f32x16{};
                    } else if (half_end) {
                        th[i][j] = tot[i][j];
                        tot[i][j] = f32x16{};
                    }
                }
        }
        if (more) {
            if constexpr (PRE) store_xs<MT>(r, xh[b ^ 1], xl[b ^ 1]);
            else store_x<MT>(r, xh[b ^ 1], xl[b ^ 1]);
            store_w<FMT>(r.w, wsm[b ^ 1]);
            if constexpr (DUAL) store_w<FMT>(r.w2, wsm2[b ^ 1]);
        }
        __syncthreads();
        b ^= 1;
    }
    // D layout of the 32x32 MFMA: column = lane % 32, row = 8*(r/4) + 4*(lane/32) + r%4.
    if (!split) {
        if constexpr (!DUAL) {
            if (khalf < kend) {
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) tot[i][j] = th[i][j] + tot[i][j];
            }
        }
        epilogue_tile<DUAL, MT>(a, tot, tot2, m0 + wm, n0 + wn, lane);
        return;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn + 32 * j + (lane & 31);
        if (n >= a.N) continue;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int m = m0 + wm + 32 * i + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
                if (m >= a.M) continue;
                const size_t o = ((size_t)blockIdx.z * a.M + m) * a.N + n;
                a.ws[o] = tot[i][j][q];
                if constexpr (DUAL) a.ws[(size_t)a.nstored * a.M * a.N + o] = tot2[i][j][q];
            }
    }
}

// LDS tiles are unpadded 32-element (64-byte) rows; 16-byte chunk c of row r
// sits at slot c ^ ((r / 4) % 4), which keeps the fragment reads of 16
// consecutive rows on distinct LDS banks.
__device__ __forceinline__ int swz(int r, int c) { return c ^ ((r >> 2) & 3); }

template <bool DUAL>
__global__ __launch_bounds__(kThreads) void gemm_reduce_kernel(GArgs a);

// s_waitcnt immediate waiting until at most n vector-memory ops are pending.
constexpr int vm_wait_imm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8); }

// Stages of the deeper BF16 ring of 4-wave blocks (launch_ring_plan).
constexpr int kDeepStages = 5;

// Raw weight bytes per row and 32-column stage.
template <int FMT>
constexpr int w_row_bytes() { return FMT == FMT_BF16 ? 64 : FMT == FMT_Q8 ? 32 : 16; }

// ---------------------------------------------------------------------------
// Ring GEMM, every weight format (x pre-split; BF16 K % 32 == 0, Q8/Q4 any K on
// halves padded with zeros): WM x WN waves of 32 MT tokens x 64 weight rows
// (DUAL: 32 gate and the matching 32 up rows).
// Per 32-wide K stage the block's x halves and its raw weight bytes (BF16
// rows, Q8 codes, Q4 nibbles) go global -> LDS by buffer loads that write LDS
// directly: a lane's source offset is fixed for the whole launch and the
// stage's K offset is a scalar, so a copy costs no vector instructions. The
// ring holds NS stages. Q8/Q4 codes are converted to BF16 (exactly) once per
// block, two stages ahead, into one of two converted tiles; BF16 weights are
// read straight from the ring. One barrier per stage.
//
// Fragments run one k-step (16 columns) ahead: the LDS reads of k-step s + 1
// and the copies of a later stage sit between the MFMAs of k-step s, so
// neither a read's latency nor a burst of copies holds the matrix cores, and
// the barrier falls inside a stage's MFMAs. Iteration st (fragments F0 read):
//   MFMAs of F0, reading F1(st); wait for this wave's copies of the next
//   stage(s); barrier; MFMAs of F1, reading F0(st + 1) and issuing stage
//   st + NS - 1 (its slot held stage st - 1, whose reads every wave finished
//   before the barrier); Q8/Q4: convert stage st + 2 (its tile held stage st).
// The MFMA sequence per output and the chunk folds are those of gemm_kernel,
// so the results are the same bits whatever the tile.
//
// Bound: the matrix cores, at the clock they leave (39 to 49 % busy over a
// dispatch of 512 tokens; a large BF16 product of the BLAS library reaches 1.2
// PFLOP/s on this card, this kernel up to 1.08 executed). Tiles, per
// block: 128 tokens x 256 rows on 8 waves of 64 x 64 (an LDS byte feeds 1.5
// times the MFMAs of 32 x 64, and the block's L2 traffic per MFMA is 2/3 of
// 128 x 128); 128 x 128 on 8 waves of 32 x 64; 64 x 128 on 4 waves, two blocks
// per CU. Before, 8-wave 128 x 128 blocks read a whole stage's fragments after
// its barrier. TFLOP/s (x split included), before -> now: 14336 x 4096 at 512
// tokens BF16 359 -> 504, Q8 315 -> 457, Q4 310 -> 450; 4096 x 4096 at 2,048
// tokens 366 -> 509 / 338 -> 467 / 347 -> 475; 3584 x 18944 at 1,024 407 ->
// 509 / 366 -> 441 / 354 -> 438. Measured and not kept: 128 x 128 on 4 waves
// of 64 x 64, two blocks per CU (393 TFLOP/s at 2,048 tokens); rings one or
// two stages deeper (even); the first half's total in memory instead of
// registers (471 against 509); the copies in one burst after the barrier (423).
// ---------------------------------------------------------------------------
template <int FMT, int MT, int WM, int WN, int NS>
constexpr size_t ring_lds_bytes() {
    constexpr size_t bn = 64 * WN, slot = 2 * (32 * MT * WM) * 64 + bn * w_row_bytes<FMT>();
    return NS * slot + (FMT == FMT_BF16 ? 0 : 2 * bn * 64);
}

template <int FMT, bool DUAL, int MT, int WM, int WN, int NS, int QG>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_ring_kernel(GArgs a, int split) {
    constexpr int WV = WM * WN, NT = 64 * WV;
    constexpr int BM = 32 * MT * WM, BNR = 64 * WN;  // tokens, weight rows of the block (DUAL: half of each matrix)
    constexpr int BNO = DUAL ? BNR / 2 : BNR;        // output columns of the block
    constexpr int XB = BM * 64;
    constexpr int WRB = w_row_bytes<FMT>();
    constexpr int WB = BNR * WRB;
    constexpr int SLOT = 2 * XB + WB;
    constexpr bool CONV = FMT != FMT_BF16;
    constexpr int WCB = BNR * 64;
    // Weight copy granule (bytes per lane): Q4 rows are only 4-byte aligned, Q8
    // ones where the row count is odd (QG = 4); Q8 also 4 where 16 would leave
    // some waves without a copy.
    constexpr int GW = FMT == FMT_Q4 || (FMT == FMT_Q8 && (QG == 4 || WB / 1024 % WV)) ? 4 : 16;
    constexpr int NIX = XB / 1024, NIW = WB / (64 * GW);
    constexpr int D = 2 * NIX / WV + NIW / WV;       // copies per wave and stage
    constexpr int CPT = BNR * 32 / NT;               // codes each thread converts per stage
    static_assert(NIX % WV == 0 && NIW % WV == 0, "copies must split evenly over the waves");
    static_assert(CPT == 8 || CPT == 16, "8 or 16 codes per converting thread");
    static_assert(NS >= (CONV ? 4 : 3), "stages in flight behind the one computed");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t *ring = smem;
    uint8_t *wcv = smem + NS * SLOT;  // CONV: [2] converted tiles

    int n0, m0;
    tile_of(a.n_tiles, (a.M + BM - 1) / BM, n0, m0, BM, BNO);
    n0 += a.n_first;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wm = (wave / WN) * 32 * MT, wj = wave % WN;
    // Weight-tile row of the wave's column group j.
    auto wrow = [&](int j) { return DUAL ? j * (BNR / 2) + 32 * wj : 64 * wj + 32 * j; };
    // split 0: all of K; 1: chunk blockIdx.z; 2: half blockIdx.z of a single
    // matrix's chunks (the first hc chunks, then the rest).
    const int hc = (a.nchunks + 1) / 2;
    const int kbeg = split == 1 ? blockIdx.z * a.chunk : split == 2 && blockIdx.z ? hc * a.chunk : 0;
    const int kend = split == 1 ? min(a.K, kbeg + a.chunk) : split == 2 && !blockIdx.z ? min(a.K, hc * a.chunk) : a.K;
    const int nst = (kend - kbeg + BK - 1) / BK;  // a part stage only against zero-padded x (Q8/Q4)

    const __amdgpu_buffer_rsrc_t rxh = __builtin_amdgcn_make_buffer_rsrc((void *)a.xh, (short)0, a.M * a.xs * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t rxl = __builtin_amdgcn_make_buffer_rsrc((void *)a.xl, (short)0, a.M * a.xs * 2, 0x00020000);
    const int wbytes = (int)((size_t)a.N * a.stride);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)a.w, (short)0, wbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw2 =
        __builtin_amdgcn_make_buffer_rsrc((void *)(DUAL ? a.w2 : a.w), (short)0, wbytes, 0x00020000);

    int xoff[NIX / WV], woff[NIW / WV];
#pragma unroll
    for (int i = 0; i < NIX / WV; ++i) {
        const int q = wave + WV * i, r = 16 * q + (lane >> 2);
        const int m = min(m0 + r, a.M - 1);  // rows past M feed only unstored outputs
        xoff[i] = (m * a.xs + 8 * swz(r, lane & 3)) * 2;
    }
    // Weight copy q covers rows RPC q .. RPC q + RPC - 1 of the tile; with
    // DUAL the first half of the copies reads the gate matrix, the rest up.
    constexpr int RPC = 64 * GW / WRB;
    auto w_up = [&](int i) { return DUAL && (wave + WV * i) * RPC >= BNR / 2; };
#pragma unroll
    for (int i = 0; i < NIW / WV; ++i) {
        const int q = wave + WV * i;
        int r, byte;
        if constexpr (FMT == FMT_BF16) { r = 16 * q + (lane >> 2); byte = 16 * swz(r, lane & 3); }
        else if constexpr (FMT == FMT_Q8 && GW == 16) { r = 32 * q + (lane >> 1); byte = 16 * (lane & 1); }
        else if constexpr (FMT == FMT_Q8) { r = 8 * q + (lane >> 3); byte = 4 * (lane & 7); }
        else { r = 16 * q + (lane >> 2); byte = 4 * (lane & 3); }
        const int n = min(n0 + (w_up(i) ? r - BNR / 2 : r), a.N - 1);
        woff[i] = n * (int)a.stride + byte;
    }
    // Stage st sits in ring slot st % NS; the loop keeps the byte offsets of
    // the slots it uses and advances them (no division on the scalar unit).
    auto next_slot = [&](int off) { return off == (NS - 1) * SLOT ? 0 : off + SLOT; };
    // Copy d (0 .. D - 1) of this wave's copies of stage st into the slot at
    // `off` (stages past the range re-read the last one into a free slot, so
    // every wave issues the same count).
    auto issue1 = [&](int st, int off, int d) {
        const int k0 = kbeg + min(st, nst - 1) * BK;
        uint8_t *slot = ring + off;
        constexpr int XI = NIX / WV;
        if (d < 2 * XI) {
            const int i = d >> 1, q = wave + WV * i;
            if (d & 1) buf_to_lds<16>(rxl, slot + XB + 1024 * q, xoff[i], k0 * 2);
            else buf_to_lds<16>(rxh, slot + 1024 * q, xoff[i], k0 * 2);
        } else {
            const int i = d - 2 * XI;
            const int kw = FMT == FMT_BF16 ? k0 * 2 : FMT == FMT_Q8 ? k0 : k0 / 2;
            uint8_t *dst = slot + 2 * XB + 64 * GW * (wave + WV * i);
            if (w_up(i)) buf_to_lds<GW>(rw2, dst, woff[i], kw);
            else buf_to_lds<GW>(rw, dst, woff[i], kw);
        }
    };
    // Stage st's codes -> BF16 tile wcv[st % 2], thread t: row t / TPR, codes
    // CPT (t % TPR) .. + CPT - 1, written in the swizzled layout the MFMA
    // reads. The raw codes are read by inline assembly: the compiler, which
    // cannot tell these reads from the ring's in-flight copies, would
    // otherwise wait for every copy before them. The copies they need were
    // awaited explicitly, and each read waits for its data inside its own asm
    // statement, so no use of the result can be scheduled ahead of the wait.
    auto convert = [&](int st, int off) {
        constexpr int TPR = 32 / CPT, RB = FMT == FMT_Q8 ? CPT : CPT / 2;
        const uint8_t *slot = ring + off + 2 * XB;
        const int row = threadIdx.x / TPR, h = threadIdx.x % TPR;
        const uint32_t addr = (uint32_t)(uintptr_t)(slot + row * WRB + RB * h);
        u32x4 rv;
        if constexpr (RB == 16) {
            asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(rv) : "v"(addr) : "memory");
        } else if constexpr (RB == 8) {
            uint2 t;
            asm volatile("ds_read_b64 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(t) : "v"(addr) : "memory");
            rv = u32x4{t.x, t.y, 0u, 0u};
        } else {
            uint32_t t;
            asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(t) : "v"(addr) : "memory");
            rv = u32x4{t, 0u, 0u, 0u};
        }
        float f[CPT];
        if constexpr (FMT == FMT_Q8) {
#pragma unroll
            for (int q = 0; q < CPT; ++q) f[q] = (float)(int)(int8_t)(rv[q >> 2] >> (8 * (q & 3)));
        } else {
#pragma unroll
            for (int h2 = 0; h2 < CPT / 8; ++h2) {
                // 16 x code: each nibble moved to the top of a byte, read as
                // int8 in one instruction (exact in BF16; the chunk sums are
                // scaled back by 1/16, exactly).
                const uint32_t wd = rv[h2];
                const uint32_t ev = (wd << 4) & 0xF0F0F0F0u, od = wd & 0xF0F0F0F0u;
                f[8 * h2 + 0] = sbyte_f32<0>(ev);
                f[8 * h2 + 1] = sbyte_f32<0>(od);
                f[8 * h2 + 2] = sbyte_f32<1>(ev);
                f[8 * h2 + 3] = sbyte_f32<1>(od);
                f[8 * h2 + 4] = sbyte_f32<2>(ev);
                f[8 * h2 + 5] = sbyte_f32<2>(od);
                f[8 * h2 + 6] = sbyte_f32<3>(ev);
                f[8 * h2 + 7] = sbyte_f32<3>(od);
            }
        }
        uint8_t *dst = wcv + (st & 1) * WCB + row * 64;
#pragma unroll
        for (int c = 0; c < CPT / 8; ++c) {
            bf16x8 b;
#pragma unroll
            for (int e = 0; e < 8; ++e) b[e] = (__bf16)f[8 * c + e];
            *(bf16x8 *)(dst + 16 * swz(row, (CPT / 8) * h + c)) = b;
        }
    };
    struct Frags {
        bf16x8 ah[MT], al[MT], bw[2];
    };
    // Fragment read d (0 .. NR - 1) of k-step k of stage st in the slot at off.
    constexpr int NR = 2 + 2 * MT;
    auto read1 = [&](int st, int off, int k, int d, Frags &f) {
        const uint8_t *xs = ring + off;
        const uint8_t *wt = CONV ? wcv + (st & 1) * WCB : xs + 2 * XB;
        const int c = 2 * k + (lane >> 5);
        if (d < 2) {
            const int r = wrow(d) + (lane & 31);
            f.bw[d] = *(const bf16x8 *)(wt + r * 64 + 16 * swz(r, c));
        } else {
            const int i = (d - 2) % MT, r = wm + 32 * i + (lane & 31);
            if (d - 2 < MT) f.ah[i] = *(const bf16x8 *)(xs + r * 64 + 16 * swz(r, c));
            else f.al[i] = *(const bf16x8 *)(xs + XB + r * 64 + 16 * swz(r, c));
        }
    };
    f32x16 acc[MT][2], tot[MT][2];
    // MFMA t (0 .. 4 MT - 1) of a k-step: the high halves of x, then the low.
    constexpr int NM = 4 * MT;
    auto mma1 = [&](const Frags &f, int t) {
        const int i = (t / 2) % MT, j = t & 1;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(t < 2 * MT ? f.ah[i] : f.al[i], f.bw[j], acc[i][j], 0, 0, 0);
    };
    // One k-step: the MFMAs of f with the reads of the next k-step into g and
    // copies d0 .. d1 - 1 of stage sti into the slot at wr between them.
    constexpr int RPM = 2;  // fragment reads per MFMA, until all are issued
    auto kstep = [&](const Frags &f, Frags &g, int st, int rd, int k, int sti, int wr, int d0, int d1) {
#pragma unroll
        for (int t = 0; t < NM; ++t) {
            mma1(f, t);
#pragma unroll
            for (int d = RPM * t; d < min(RPM * t + RPM, NR); ++d) read1(st, rd, k, d, g);
#pragma unroll
            for (int d = d0 + t * (d1 - d0) / NM; d < d0 + (t + 1) * (d1 - d0) / NM; ++d) issue1(sti, wr, d);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) tot[i][j] = f32x16{};

    // Copies issued in a stage's second k-step, the rest in the next stage's
    // first: half of them; on the deep BF16 ring, whose time is the weight
    // stream and not the MFMAs, all (18944 x 3584 at 2 tokens 41.7 -> 40.8 us,
    // 10112 x 2304 at 16 23.8 -> 21.7; Q8/Q4 3 % slower at small sizes).
    constexpr int DH = !CONV && NS >= kDeepStages ? D : D / 2 + D % 2;
#pragma unroll
    for (int st = 0; st < NS - 1; ++st)
#pragma unroll
        for (int d = 0; d < (st == NS - 2 ? DH : D); ++d) issue1(st, st * SLOT, d);
    __builtin_amdgcn_s_waitcnt(vm_wait_imm(D * (CONV ? NS - 4 : NS - 3) + DH));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if constexpr (CONV) {
        convert(0, 0);
        convert(1, SLOT);
        __builtin_amdgcn_s_waitcnt(vm_wait_imm(63) & ~(0xF << 8));  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
    }
    Frags f0, f1;
#pragma unroll
    for (int d = 0; d < NR; ++d) read1(0, 0, 0, d, f0);
    // Slots of stage st, of the one before it (the next copies' target) and of
    // the copies begun in the previous iteration.
    int rd = 0, wr = (NS - 1) * SLOT, wr_prev = (NS - 2) * SLOT;
    const int cs = a.chunk / BK;  // stages per accumulation chunk
    // Stages [s0, s1), whole chunks, folded into tot.
    auto run = [&](int s0, int s1) {
        for (int c0 = s0; c0 < s1; c0 += cs) {
            const int c1 = min(c0 + cs, s1);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
            for (int st = c0; st < c1; ++st) {
                kstep(f0, f1, st, rd, 1, st + NS - 2, wr_prev, DH, D);
                __builtin_amdgcn_s_waitcnt(vm_wait_imm(D * (CONV ? NS - 4 : NS - 3)));
                __builtin_amdgcn_s_waitcnt(vm_wait_imm(63) & ~(0xF << 8));  // lgkmcnt(0)
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                const int nx = next_slot(rd);
                kstep(f1, f0, st + 1, nx, 0, st + NS - 1, wr, 0, DH);  // past the last stage: stale bytes, unused
                if constexpr (CONV) convert(st + 2, next_slot(nx));
                wr_prev = wr;
                wr = rd;
                rd = nx;
            }
            constexpr float cs16 = FMT == FMT_Q4 ? 0.0625f : 1.0f;
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) tot[i][j] += FMT == FMT_Q4 ? acc[i][j] * cs16 : acc[i][j];
        }
    };
    const bool halves = !DUAL && !split && hc < a.nchunks;
    run(0, halves ? hc * cs : nst);
    f32x16 th[DUAL ? 1 : MT][2];
    if constexpr (!DUAL) {
        if (halves) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    th[i][j] = tot[i][j];
                    tot[i][j] = f32x16{};
                }
            run(hc * cs, nst);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) tot[i][j] = th[i][j] + tot[i][j];
        }
    }
    // Drain the copies of stages past the range before the block exits.
    __builtin_amdgcn_s_waitcnt(vm_wait_imm(0));
    if (!split) {
        if constexpr (!DUAL) {
            epilogue_tile<false, MT>(a, tot, reinterpret_cast<const f32x16(&)[1][2]>(tot), m0 + wm, n0 + 64 * wj, lane);
        } else {
            f32x16 gt[MT][1], up[MT][1];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                gt[i][0] = tot[i][0];
                up[i][0] = tot[i][1];
            }
            epilogue_tile<true, MT, 1>(a, gt, up, m0 + wm, n0 + 32 * wj, lane);
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + (DUAL ? 32 * wj : 64 * wj + 32 * j) + (lane & 31);
        if (n >= a.N) continue;
        float *ws = a.ws + (DUAL && j ? (size_t)a.nstored * a.M * a.N : 0);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int m = m0 + wm + 32 * i + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
                if (m < a.M) ws[((size_t)blockIdx.z * a.M + m) * a.N + n] = tot[i][j][q];
            }
    }
}

template <int FMT, bool DUAL, int MT, int WM, int WN, int NS, int QG>
int launch_ring(GArgs a, int split, hipStream_t s) {
    constexpr int BM = 32 * MT * WM, BNO = (DUAL ? 32 : 64) * WN;
    if (!a.n_tiles) a.n_tiles = (a.N - a.n_first + BNO - 1) / BNO;
    constexpr size_t lds = ring_lds_bytes<FMT, MT, WM, WN, NS>();
    static std::atomic<uint64_t> lds_set{0};
    CHIP_TRY(allow_dynamic_lds((const void *)gemm_ring_kernel<FMT, DUAL, MT, WM, WN, NS, QG>, lds, lds_set));
    const dim3 grid(a.n_tiles * ((a.M + BM - 1) / BM), 1, split ? a.nstored : 1);
    hipLaunchKernelGGL((gemm_ring_kernel<FMT, DUAL, MT, WM, WN, NS, QG>), grid, dim3(64 * WM * WN), lds, s, a, split);
    CHIP_CHECK(hipGetLastError());
    if (split && !a.defer) {
        const size_t MN = (size_t)a.M * a.N;
        hipLaunchKernelGGL((gemm_reduce_kernel<DUAL>), dim3((unsigned)((MN + kThreads - 1) / kThreads)),
                           dim3(kThreads), 0, s, a);
        CHIP_CHECK(hipGetLastError());
    }
    return 0;
}

// Folds the stored sums (a.nstored per output: every chunk's, or a single
// matrix's two halves) in the GEMM's association and applies the epilogue:
// the same bits as the in-register fold. Dual: left to right (t = 0;
// t += c_z); single matrix: the first ceil(n / 2) left to right, the rest
// left to right, then the two added.
template <bool DUAL>
__global__ __launch_bounds__(kThreads) void gemm_reduce_kernel(GArgs a) {
    const size_t MN = (size_t)a.M * a.N;
    const size_t e = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (e >= MN) return;
    const int n = a.nstored, hs = DUAL ? n : (n + 1) / 2;
    // Eight stored sums (of each matrix) loaded at a time, folded in order.
    float v = 0.f, v2 = 0.f, u = 0.f;
    for (int z0 = 0; z0 < n; z0 += 8) {
        float t[8], t2[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool in = z0 + j < n;
            t[j] = in ? a.ws[(size_t)(z0 + j) * MN + e] : 0.f;
            if constexpr (DUAL) t2[j] = in ? a.ws[((size_t)n + z0 + j) * MN + e] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (z0 + j < hs) v += t[j];
            else if (z0 + j < n) v2 += t[j];
            if constexpr (DUAL)
                if (z0 + j < n) u += t2[j];
        }
    }
    if (!DUAL && hs < n) v = v + v2;
    epilogue<DUAL>(a, (int)(e / a.N), (int)(e % a.N), v, u);
}

template <int FMT, bool DUAL, int MT>
int launch_mt(const GArgs &a, bool split, hipStream_t s) {
    constexpr int BM = 64 * MT;
    const dim3 grid((a.N + BN - 1) / BN * ((a.M + BM - 1) / BM), 1, split ? a.nchunks : 1);
    if (a.xh) hipLaunchKernelGGL((gemm_kernel<FMT, DUAL, MT, true>), grid, dim3(kThreads), 0, s, a, split ? 1 : 0);
    else hipLaunchKernelGGL((gemm_kernel<FMT, DUAL, MT, false>), grid, dim3(kThreads), 0, s, a, split ? 1 : 0);
    CHIP_CHECK(hipGetLastError());
    if (split && !a.defer) {
        const size_t MN = (size_t)a.M * a.N;
        hipLaunchKernelGGL((gemm_reduce_kernel<DUAL>), dim3((unsigned)((MN + kThreads - 1) / kThreads)),
                           dim3(kThreads), 0, s, a);
        CHIP_CHECK(hipGetLastError());
    }
    return 0;
}

// Ring stages by format: the 4-wave tile keeps two blocks per CU (64 to 80 KB
// each), the others one. BF16 blocks of 4 waves have a second, deeper ring
// (launch_ring_plan).
template <int FMT>
constexpr int ring_stages() { return FMT == FMT_BF16 ? 4 : 5; }

enum Tile : int { TILE_64x128, TILE_128x128, TILE_128x256 };
// How a ring GEMM runs: its tile and its K split (0 none, 1 per chunk, 2 a
// single matrix's two halves) with the sums stored per output.
// head_tiles: 128 x 256 row tiles of a launch of their own before the plan's
// (unsplit) takes the remaining rows; 0 = none.
struct RingPlan {
    int tile, split, nstored;
    size_t ws_floats;
    int head_tiles;
};

// The plan with the least estimated time of those whose stored sums fit
// ws_floats. The estimate, in us: rounds of the tile's blocks (one per CU, two
// for the 4-wave tile) times the time of 1,024 columns of a block in a full
// round (with no more blocks than CUs, of a block alone), and a fixed time per
// tile, with and without a split; a split adds its sums' write and read at 3.5
// TB/s, an unsplit wave's epilogue takes 3 us for 32 rows. The figures are
// those with which the choice came closest to the best of every tile and
// split, timed at 1,772 sizes of 64 to 20000 rows, 64 to 18944 columns and 2 to
// 2,048 tokens in the three formats: 0.3 % behind it on average (1.8 % with one
// fixed time for all tiles, unsplit less than split: 2240 x 128 Q8 at 37 tokens
// then ran 64 x 128 unsplit, 11.9 us against 9.5 split).
RingPlan ring_plan(int fmt, bool dual, int N, int K, int M, size_t ws_floats) {
    static constexpr struct {
        int bm, bn, per_cu;
        float us_bf16, us_quant;    // a full round
        float low_bf16, low_quant;  // no more blocks than CUs
        float fixed, fixed_split;   // without and with a split
    } kTiles[] = {{64, 128, 2, 26.f, 29.f, 13.f, 17.5f, 3.f, 2.f},
                  {128, 128, 1, 21.f, 22.f, 17.5f, 19.f, 4.f, 4.f},
                  {128, 256, 1, 30.f, 34.f, 25.5f, 32.5f, 5.5f, 4.5f}};
    const int chunk = gemm_chunk_depth(K), nchunks = (K + chunk - 1) / chunk;
    const long cus = device_cus();
    const float mn = (float)M * (float)N;
    RingPlan best{TILE_128x128, 0, 1, 0, 0};
    float best_us = 0.f;
    for (int t = 0; t < 3; ++t) {
        const int bno = dual ? kTiles[t].bn / 2 : kTiles[t].bn;
        const long tiles = (long)((N + bno - 1) / bno) * ((M + kTiles[t].bm - 1) / kTiles[t].bm);
        const bool bf = fmt == FMT_BF16;
        for (int split = 0; split < 3; ++split) {
            if (split && (nchunks == 1 || (split == 2 && dual))) continue;
            const int parts = split == 1 ? nchunks : split == 2 ? 2 : 1;
            const int depth = split == 1 ? chunk : split == 2 ? (nchunks + 1) / 2 * chunk : K;
            const size_t need = split ? (size_t)parts * M * N * (dual ? 2 : 1) : 0;
            if (need > ws_floats) continue;
            const long slots = cus * kTiles[t].per_cu, rounds = (tiles * parts + slots - 1) / slots;
            const float us = tiles * parts > cus ? bf ? kTiles[t].us_bf16 : kTiles[t].us_quant
                                                 : bf ? kTiles[t].low_bf16 : kTiles[t].low_quant;
            float est = (float)rounds * (float)depth / 1024.f * us + (split ? kTiles[t].fixed_split : kTiles[t].fixed);
            if (split) {
                est += 8.f * (float)parts * (dual ? 2.f : 1.f) * mn / 3.5e6f;
            } else {
                const int rows = t == TILE_128x256 ? 64 : 32;  // of a wave
                est -= 3.f * (float)(rows - std::min(M, rows)) / 32.f;
            }
            if (best_us == 0.f || est < best_us) {
                best_us = est;
                best = RingPlan{t, split, parts, need, 0};
            }
        }
    }
    // Full rounds of 128 x 256 tiles, and the rows left over on 128 x 128 ones
    // instead of a nearly empty last round: 18944 x 3584 at 1,024 tokens (592
    // tiles, 2.3 rounds) BF16 312 -> 295 us, Q8 353 -> 309; 11008 x 4096 at
    // 1,024 222 -> 205; 14336 x 4096 Q8 at 2,048 583 -> 488.
    const auto &big = kTiles[TILE_128x256], &mid = kTiles[TILE_128x128];
    const float us_big = (fmt == FMT_BF16 ? big.us_bf16 : big.us_quant) * (float)K / 1024.f;
    const float us_mid = (fmt == FMT_BF16 ? mid.us_bf16 : mid.us_quant) * (float)K / 1024.f;
    const int bno = dual ? big.bn / 2 : big.bn, bno_mid = dual ? mid.bn / 2 : mid.bn;
    const long m_tiles = (M + big.bm - 1) / big.bm, n_tiles = (N + bno - 1) / bno;
    const long rounds = m_tiles * n_tiles / cus, head = rounds * cus / m_tiles;
    if (head > 0 && head * bno < N) {
        const long rest = (N - head * bno + bno_mid - 1) / bno_mid * m_tiles;
        const float est = (float)rounds * us_big + (float)((rest + cus - 1) / cus) * us_mid + 11.f;
        if (est < best_us) {
            best_us = est;
            best = RingPlan{TILE_128x128, 0, 1, 0, (int)head};
        }
    }
    return best;
}

template <int FMT, bool DUAL, int QG>
int launch_ring_plan(GArgs &a, const RingPlan &p, hipStream_t s) {
    constexpr int NS = ring_stages<FMT>();
    a.nstored = p.nstored;
    if (p.head_tiles) {
        GArgs head = a;
        head.n_tiles = p.head_tiles;
        CHIP_TRY((launch_ring<FMT, DUAL, 2, 2, 4, NS, QG>(head, 0, s)));
        a.n_first = p.head_tiles * (DUAL ? 128 : 256);
    }
    switch (p.tile) {
        case TILE_64x128:
            // BF16 at few tokens is the weight stream: five stages, two of them
            // in flight at every wait (with four one: 4864 x 14336 at 16 tokens
            // 51.0 -> 43.2 us, 896 x 18944 at 4 21.6 -> 18.2). Four where a
            // split leaves nine stages or fewer a block and one to four blocks
            // a CU, or K is six or fewer, so that a deeper fill shows (4096 x
            // 4096 at 16 tokens 15.5 against 16.3, 6144 x 4096 at 37 27.6
            // against 28.4, 640 x 128 at 4 6.9 against 7.2).
            if constexpr (FMT == FMT_BF16) {
                constexpr int BNO = DUAL ? 64 : 128;
                const long blocks = (long)((a.N + BNO - 1) / BNO) * ((a.M + 63) / 64) * p.nstored, cus = device_cus();
                const bool short_blocks = a.K <= 6 * BK || (p.split == 1 && a.chunk <= 9 * BK && blocks > cus &&
                                                            blocks <= 4 * cus);
                if (!short_blocks) return launch_ring<FMT, DUAL, 1, 2, 2, kDeepStages, QG>(a, p.split, s);
            }
            return launch_ring<FMT, DUAL, 1, 2, 2, NS, QG>(a, p.split, s);
        case TILE_128x128: return launch_ring<FMT, DUAL, 1, 4, 2, NS, QG>(a, p.split, s);
        default: return launch_ring<FMT, DUAL, 2, 2, 4, NS, QG>(a, p.split, s);
    }
}

template <int FMT>
int launch_fmt(GArgs a, bool dual, size_t ws_floats, hipStream_t s, bool &split_out, int &stored_out) {
    // Pre-split x with K a multiple of the stage (Q8/Q4: or x padded to one
    // with zeros, which whatever codes follow the row's meet; a BF16 row's
    // neighbour could hold a NaN) and 32-bit buffer offsets: the ring kernel (weights copied 16 bytes at a time, Q4 and unaligned Q8 4).
    const int galign = FMT == FMT_BF16 ? 16 : 4;
    const int kpad = (a.K + BK - 1) / BK * BK;
    const bool ring = a.xh && (FMT == FMT_BF16 ? a.K : a.xs) % BK == 0 && a.xs >= kpad && a.stride % galign == 0 &&
                      ((uintptr_t)a.w % galign) == 0 &&
                      (!dual || (((uintptr_t)a.w | (uintptr_t)a.w2 | a.stride) % (FMT == FMT_Q4 ? 4 : 16)) == 0) &&
                      (size_t)a.M * a.xs * 2 < (1ull << 31) && (size_t)a.N * a.stride < (1ull << 31);
    if (ring) {
        const RingPlan p = ring_plan(FMT, dual, a.N, a.K, a.M, a.ws ? ws_floats : 0);
        split_out = p.split != 0;
        stored_out = p.nstored;
        if constexpr (FMT == FMT_Q8) {  // a single matrix of odd row count
            if (!dual && ((uintptr_t)a.w % 16 || a.stride % 16)) return launch_ring_plan<FMT, false, 4>(a, p, s);
        }
        return dual ? launch_ring_plan<FMT, true, 16>(a, p, s) : launch_ring_plan<FMT, false, 16>(a, p, s);
    }
    // Otherwise (K not a multiple of the stage, x not pre-split, or operands
    // beyond the buffer loads' 32-bit offsets): the register-staged kernel.
    if (a.xs != a.K) a.xh = a.xl = nullptr;
    // Many tiles: fold in registers. Few tiles: split-K over the chunks when
    // the workspace holds them.
    const long n_tiles = (a.N + BN - 1) / BN;
    const long tiles128 = n_tiles * ((a.M + 127) / 128), tiles64 = n_tiles * ((a.M + 63) / 64);
    const long cus = device_cus();
    const bool split = a.nchunks > 1 && tiles64 < cus && a.ws &&
                       ws_floats >= (size_t)a.nchunks * a.M * a.N * (dual ? 2 : 1);
    split_out = split;
    a.nstored = a.nchunks;
    stored_out = a.nstored;
    if (dual) return launch_mt<FMT, true, 1>(a, split, s);
    if (!split && tiles128 >= cus) return launch_mt<FMT, false, 2>(a, false, s);
    return launch_mt<FMT, false, 1>(a, split, s);
}

// x -> hi = bf16(x), lo = bf16(x - hi), 4 elements per thread.
__global__ __launch_bounds__(kThreads) void split_bf16_kernel(const float *x, size_t n, uint16_t *xh, uint16_t *xl) {
    const size_t i = ((size_t)blockIdx.x * kThreads + threadIdx.x) * 4;
    if (i >= n) return;
    if (i + 4 <= n) {
        const f32x4 v = *(const f32x4 *)(x + i);
        uint16_t h[4], l[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const __bf16 hb = (__bf16)v[q];
            h[q] = __builtin_bit_cast(uint16_t, hb);
            l[q] = __builtin_bit_cast(uint16_t, (__bf16)(v[q] - (float)hb));
        }
        *(uint2 *)(xh + i) = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
        *(uint2 *)(xl + i) = make_uint2(pack2(l[0], l[1]), pack2(l[2], l[3]));
    } else {
        for (size_t q = i; q < n; ++q) {
            const __bf16 hb = (__bf16)x[q];
            xh[q] = __builtin_bit_cast(uint16_t, hb);
            xl[q] = __builtin_bit_cast(uint16_t, (__bf16)(x[q] - (float)hb));
        }
    }
}

// The same for rows of K elements into rows of ks (a multiple of 4), zeros
// past K.
__global__ __launch_bounds__(kThreads) void split_bf16_rows_kernel(const float *x, size_t n, int K, int ks,
                                                                   uint16_t *xh, uint16_t *xl) {
    const size_t i = ((size_t)blockIdx.x * kThreads + threadIdx.x) * 4;
    if (i >= n * ks) return;
    const size_t row = i / ks;
    const int c = (int)(i % ks);
    uint16_t h[4], l[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float v = c + q < K ? x[row * K + c + q] : 0.f;
        const __bf16 hb = (__bf16)v;
        h[q] = __builtin_bit_cast(uint16_t, hb);
        l[q] = __builtin_bit_cast(uint16_t, (__bf16)(v - (float)hb));
    }
    *(uint2 *)(xh + i) = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
    *(uint2 *)(xl + i) = make_uint2(pack2(l[0], l[1]), pack2(l[2], l[3]));
}

}  // namespace

size_t gemm_half_stride(int fmt, size_t cols) { return fmt == FMT_BF16 ? cols : (cols + BK - 1) / BK * BK; }

int launch_split_bf16_rows(const float *x, size_t n, size_t cols, size_t stride, uint16_t *xh, uint16_t *xl,
                           hipStream_t s) {
    if (stride == cols) return launch_split_bf16(x, n * cols, xh, xl, s);
    if (n == 0) return 0;
    if (!x || !xh || !xl || stride < cols || stride % 4 || stride > (size_t)INT32_MAX || ((uintptr_t)x % 16) ||
        ((uintptr_t)xh % 8) || ((uintptr_t)xl % 8))
        return fail("HIP backend: split needs 16-byte aligned input, rows padded to a multiple of 4 and 8-byte aligned "
                    "halves.");
    const size_t blocks = (n * stride / 4 + kThreads - 1) / kThreads;
    if (blocks > (size_t)INT32_MAX) return fail("HIP backend: split shape too large.");
    hipLaunchKernelGGL(split_bf16_rows_kernel, dim3((unsigned)blocks), dim3(kThreads), 0, s, x, n, (int)cols,
                       (int)stride, xh, xl);
    CHIP_CHECK(hipGetLastError());
    return 0;
}

int launch_split_bf16(const float *x, size_t n, uint16_t *xh, uint16_t *xl, hipStream_t s) {
    if (n == 0) return 0;
    if (!x || !xh || !xl || ((uintptr_t)x % 16) || ((uintptr_t)xh % 8) || ((uintptr_t)xl % 8))
        return fail("HIP backend: split needs 16-byte aligned input and 8-byte aligned halves.");
    const size_t threads = (n + 3) / 4;
    hipLaunchKernelGGL(split_bf16_kernel, dim3((unsigned)((threads + kThreads - 1) / kThreads)), dim3(kThreads), 0, s,
                       x, n, xh, xl);
    CHIP_CHECK(hipGetLastError());
    return 0;
}

// Accumulation chunk depth, a function of K alone (so a token's bits never
// depend on the call's token count): at least 256 and K / 16; K up to 1024
// in three chunks instead (K = 896: 320 + 320 + 256 rather than 3 x 256 +
// 128; the split-K blocks of a 128-token chunk then fit the chip in one
// round: Qwen2-0.5B prefill 61.0K -> 65.0K tok/s; two chunks 63.0K, four
// equal 61.0K, one 49.9K).
int gemm_chunk_depth(int K) {
    const int want = K <= 1024 ? (K + 2) / 3 : std::max(256, (K + 15) / 16);
    return (want + BK - 1) / BK * BK;
}

size_t gemm_workspace_floats(int fmt, size_t N, size_t K, size_t M, bool dual) {
    if (std::max({N, K, M}) > (size_t)INT32_MAX) return 0;  // launch_gemm refuses it
    // The register-staged kernel (unaligned operands, other K) splits per
    // chunk while 64-token tiles leave CUs idle.
    const int chunk = gemm_chunk_depth((int)K);
    const size_t nchunks = (K + chunk - 1) / chunk, tiles = (N + BN - 1) / BN * ((M + 63) / 64);
    const size_t staged = nchunks > 1 && tiles < (size_t)device_cus() ? nchunks * M * N * (dual ? 2 : 1) : 0;
    return K % BK && fmt == FMT_BF16 ? staged : std::max(staged, ring_plan(fmt, dual, (int)N, (int)K, (int)M, SIZE_MAX).ws_floats);
}

size_t gemm_split_workspace_floats(int fmt, size_t N, size_t K, size_t m_max, bool dual) {
    size_t need = gemm_workspace_floats(fmt, N, K, m_max, dual);
    for (size_t m = 64; m < m_max; m += 64) need = std::max(need, gemm_workspace_floats(fmt, N, K, m, dual));
    return need;
}

bool gemm_takes_halves(size_t K) { return K % 8 == 0; }

int launch_gemm(const GemmJob &job, hipStream_t s) {
    const WMat &w = job.w;
    if (job.n == 0) return 0;
    // Pre-split halves are used when every 8-element chunk is 16-byte aligned;
    // x itself is then not read.
    const size_t xs = job.x_stride ? job.x_stride : w.cols;
    if (xs < w.cols || xs > (size_t)INT32_MAX) return fail("HIP backend: gemm input rows are too short or too long.");
    const bool pre = job.xh && job.xl && xs % 8 == 0 && ((uintptr_t)job.xh % 16) == 0 && ((uintptr_t)job.xl % 16) == 0;
    if (!w.base || (!job.x && !(pre && xs == w.cols)) || w.rows == 0 || w.cols == 0)
        return fail("HIP backend: gemm needs a weight and an input.");
    if (w.rows > (size_t)INT32_MAX || w.cols > (size_t)INT32_MAX || job.n > 65535u * 64u)
        return fail("HIP backend: gemm shape too large.");
    const bool dual = job.epi == EPI_SWIGLU;
    if (dual && (!job.w2.base || job.w2.fmt != w.fmt || job.w2.rows != w.rows || job.w2.cols != w.cols))
        return fail("HIP backend: SwiGLU gemm needs gate and up matrices of one shape and format.");
    if (job.epi == EPI_RESIDUAL ? !job.residual : !job.y && !(dual && job.yh)) return fail("HIP backend: gemm has no output.");
    GArgs a{};
    a.w = w.payload();
    a.sc = w.scales();
    a.w2 = dual ? job.w2.payload() : nullptr;
    a.sc2 = dual ? job.w2.scales() : nullptr;
    a.stride = w.row_stride();
    a.N = (int)w.rows;
    a.K = (int)w.cols;
    a.M = (int)job.n;
    a.x = job.x;
    a.bias = job.bias;
    a.y = job.y;
    a.residual = job.residual;
    if (!job.yh != !job.yl) return fail("HIP backend: gemm output halves need both BF16 buffers or neither.");
    a.yh = dual ? job.yh : nullptr;
    a.yl = dual ? job.yl : nullptr;
    a.defer = job.deferred && !dual ? 1 : 0;
    if (job.deferred) *job.deferred = 0;
    a.epi = job.epi;
    a.chunk = gemm_chunk_depth(a.K);
    a.nchunks = (a.K + a.chunk - 1) / a.chunk;
    a.ws = job.ws;
    a.vec_x = (a.K % 4) == 0 && ((uintptr_t)job.x % 16) == 0;
    a.xs = (int)xs;
    a.xh = pre ? job.xh : nullptr;
    a.xl = pre ? job.xl : nullptr;
    const uintptr_t p1 = (uintptr_t)a.w, p2 = dual ? (uintptr_t)a.w2 : p1;
    if (w.fmt == FMT_BF16) a.vec_w = a.stride % 16 == 0 && p1 % 16 == 0 && p2 % 16 == 0 && a.K % 8 == 0;
    else if (w.fmt == FMT_Q8) a.vec_w = a.stride % 16 == 0 && p1 % 16 == 0 && p2 % 16 == 0 && a.K % 16 == 0;
    else a.vec_w = 0;
    if (w.fmt == FMT_Q4 && (a.stride % 4 != 0 || p1 % 4 != 0 || p2 % 4 != 0))
        return fail("HIP backend: Q4 rows must be 4-byte aligned.");
    bool split = false;
    int stored = 0, rc = -1;
    switch (w.fmt) {
        case FMT_BF16: rc = launch_fmt<FMT_BF16>(a, dual, job.ws_floats, s, split, stored); break;
        case FMT_Q8: rc = launch_fmt<FMT_Q8>(a, dual, job.ws_floats, s, split, stored); break;
        case FMT_Q4: rc = launch_fmt<FMT_Q4>(a, dual, job.ws_floats, s, split, stored); break;
        default: return fail("HIP backend: unknown weight format.");
    }
    if (rc == 0 && a.defer && split) *job.deferred = stored;
    return rc;
}

}  // namespace chip
