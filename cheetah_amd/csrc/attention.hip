// GQA causal attention over the paged KV cache (the math of
// OpsToolbox::attention / attention_head, ops.rs:1357-1467: scores k·q scaled
// by 1/sqrt(head_dim), softmax, weighted value mix), as split-K flash
// decoding:
//
//   attn_kernel (f32 K/V decode, one query row; BF16 K/V decode runs on the
//   matrix cores, attn_dec_mfma_kernel below, and chunked prefill on
//   attn_prefill_kernel or attn_prefill_f32_kernel): grid (splits, kv_heads);
//   block = 256 threads.
//   Each block owns one KV head and one contiguous slice of the row's
//   visible positions [0, pos]; it streams the slice in tiles of
//   64 positions (one page-aligned 64 x head_dim tile of K, then of V),
//   scores all G = q_heads / kv_heads query heads of the group against each K
//   row it loads (K and V are read once per group, not once per head), keeps
//   an online softmax (running max / sum) per head and accumulates p * V.
//   With one split it writes the normalised output; otherwise it writes a
//   partial (unnormalised sum, max, denominator) and
//   attn_combine_kernel merges the splits of each q head in split order, so
//   results are deterministic.
//
// Split boundaries depend only on a row's own context length and the split
// count. The position comes from a device word in the decode graph (pos_dev)
// or from the host. K/V elements are BF16 (default) or f32.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "kernels.hpp"

namespace chip {
namespace {

constexpr int kThreads = 256;
constexpr int TP = 64;  // positions per tile (page_size is a multiple of it)
constexpr int kMaxSplits = 128;

// Block barrier that waits on LDS traffic only (outstanding global loads
// stay in flight across it).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct AttnArgs {
    const float *q;
    long q_stride;
    const void *k, *v;
    const int32_t *page_table;
    int page_size, kv_heads, q_heads;
    long offset;
    const int32_t *pos_dev;
    float *part;
    float *out;
    // Fused decode RoPE (attn_dec_mfma_kernel<.., ROPE>): raw QKV row and
    // the cos/sin table; K/V are then also written (the new row).
    const float *qkv;
    const float *rope_cos, *rope_sin;
    int rotary_dim;
    // Chunked prefill: BF16 halves of out (null: not written).
    uint16_t *out_hi, *out_lo;
};

// hi = bf16(v), lo = bf16(v - hi) (hardware round-to-nearest-even) of four
// consecutive outputs at element i: the split the next GEMM takes as input.
__device__ __forceinline__ void store_halves4(uint16_t *hi, uint16_t *lo, size_t i, f32x4 v) {
    uint16_t h[4], l[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const __bf16 hb = (__bf16)v[q];
        h[q] = __builtin_bit_cast(uint16_t, hb);
        l[q] = __builtin_bit_cast(uint16_t, (__bf16)(v[q] - (float)hb));
    }
    *(uint2 *)(hi + i) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
    *(uint2 *)(lo + i) = make_uint2((uint32_t)l[0] | ((uint32_t)l[1] << 16), (uint32_t)l[2] | ((uint32_t)l[3] << 16));
}

// Eight consecutive K or V elements as loaded (converted to f32 at use), so
// a whole tile can be in flight while the previous one computes.
template <class KT>
struct Raw8;
template <>
struct Raw8<uint16_t> {
    u32x4 w;
    __device__ void load(const uint16_t *p) { w = *(const u32x4 *)p; }
    __device__ void get(float (&f)[8]) const {
        f[0] = bf16_lo(w[0]); f[1] = bf16_hi(w[0]); f[2] = bf16_lo(w[1]); f[3] = bf16_hi(w[1]);
        f[4] = bf16_lo(w[2]); f[5] = bf16_hi(w[2]); f[6] = bf16_lo(w[3]); f[7] = bf16_hi(w[3]);
    }
};
template <>
struct Raw8<float> {
    f32x4 a, b;
    __device__ void load(const float *p) {
        a = *(const f32x4 *)p;
        b = *(const f32x4 *)(p + 4);
    }
    __device__ void get(float (&f)[8]) const {
        f[0] = a[0]; f[1] = a[1]; f[2] = a[2]; f[3] = a[3];
        f[4] = b[0]; f[5] = b[1]; f[6] = b[2]; f[7] = b[3];
    }
};

template <int HD, int G, class KT, bool DIRECT>
__global__ __launch_bounds__(kThreads) void attn_kernel(AttnArgs a) {
    constexpr int T = HD / 8;          // threads per position row (8 dims each)
    constexpr int P = kThreads / T;    // positions per pass
    constexpr int JW = (G + 3) / 4;    // heads per wave in the softmax step
    __shared__ float s_p[G][TP];
    __shared__ float s_alpha[G];
    __shared__ float s_red[kThreads / 64][G][HD];
    __shared__ float s_l[G];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int d8 = tid % T, pg = tid / T;
    const int split = blockIdx.x, S = gridDim.x;
    const int g = blockIdx.y;
    const long pos = a.pos_dev ? (long)*a.pos_dev : a.offset;
    const long ctx = pos + 1;
    long chunk = (ctx + S - 1) / S;
    chunk = (chunk + TP - 1) / TP * TP;
    const long start = (long)split * chunk;
    const long end = min(start + chunk, ctx);
    const size_t part_head = (size_t)S * (HD + 2);
    float *part = a.part + (size_t)g * G * part_head + (size_t)split * (HD + 2);

    if (start >= ctx) {  // empty split: contributes nothing to the merge
        if (tid < G) part[tid * part_head + HD] = -INFINITY;
        return;
    }

    const float scale = 1.0f / sqrtf((float)HD);
    float qr[G][8];
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const float *qp = a.q + (size_t)(g * G + j) * HD + d8 * 8;
        const f32x4 q0 = *(const f32x4 *)qp, q1 = *(const f32x4 *)(qp + 4);
        qr[j][0] = q0[0]; qr[j][1] = q0[1]; qr[j][2] = q0[2]; qr[j][3] = q0[3];
        qr[j][4] = q1[0]; qr[j][5] = q1[1]; qr[j][6] = q1[2]; qr[j][7] = q1[3];
    }
    float acc[G][8];
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[j][e] = 0.f;
    float m_run[JW], l_run[JW];
#pragma unroll
    for (int i = 0; i < JW; ++i) {
        m_run[i] = -INFINITY;
        l_run[i] = 0.f;
    }

    // K/V tiles ping-pong between two register sets: tile t0 + TP loads while
    // tile t0 computes. A position past `end` reads the row at end - 1 (the
    // compute masks it), and the tile barriers wait on LDS only, so the loads
    // of the next tile stay in flight across the current tile's barriers.
    // (Four sets, three tiles in flight, measured slower: 254 registers.)
    constexpr int NB = 2;
    Raw8<KT> bk[NB][TP / P], bv[NB][TP / P];
    const long last_tile = start + (end - 1 - start) / TP * TP;
    auto issue = [&](long t, Raw8<KT> (&kr)[TP / P], Raw8<KT> (&vr)[TP / P]) {
        t = min(t, last_tile);
        const int page = a.page_table[t / a.page_size];
        const size_t tile_off = (((size_t)page * a.kv_heads + g) * a.page_size + t % a.page_size) * HD;
        const KT *kt = (const KT *)a.k + tile_off;
        const KT *vt = (const KT *)a.v + tile_off;
        const int rmax = (int)(end - 1 - t);
#pragma unroll
        for (int p = 0; p < TP / P; ++p) {
            const int r = min(p * P + pg, rmax);
            kr[p].load(kt + (size_t)r * HD + d8 * 8);
            vr[p].load(vt + (size_t)r * HD + d8 * 8);
        }
    };
    auto tile = [&](long t0, const Raw8<KT> (&kc)[TP / P], const Raw8<KT> (&vc)[TP / P]) {
        // Scores of every head of the group for the tile's rows (each K row
        // widened to f32 where it is used).
#pragma unroll
        for (int p = 0; p < TP / P; ++p) {
            const int pi = p * P + pg;
            const bool valid = t0 + pi < end;
            float kf[8];
            kc[p].get(kf);
            float dot[G];
#pragma unroll
            for (int j = 0; j < G; ++j) dot[j] = 0.f;
            if (valid) {
#pragma unroll
                for (int j = 0; j < G; ++j)
#pragma unroll
                    for (int e = 0; e < 8; ++e) dot[j] = fmaf(kf[e], qr[j][e], dot[j]);
            }
#pragma unroll
            for (int j = 0; j < G; ++j) {
                const float sum = group_sum<T>(dot[j]);
                if (d8 == 0) s_p[j][pi] = valid ? sum * scale : -INFINITY;
            }
        }
        lds_barrier();
        // Online softmax per head: one wave per head, one lane per position.
#pragma unroll
        for (int i = 0; i < JW; ++i) {
            const int j = wave + 4 * i;
            if (j < G) {
                const float sc = s_p[j][lane];
                const float m_new = fmaxf(m_run[i], wave_max(sc));
                const float pv = sc == -INFINITY ? 0.f : expf(sc - m_new);
                s_p[j][lane] = pv;
                const float l_tile = wave_sum(pv);
                const float alpha = m_run[i] == -INFINITY ? 0.f : expf(m_run[i] - m_new);
                l_run[i] = l_run[i] * alpha + l_tile;
                m_run[i] = m_new;
                if (lane == 0) s_alpha[j] = alpha;
            }
        }
        lds_barrier();
        // acc = acc * alpha + sum_p p * V[p].
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const float al = s_alpha[j];
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[j][e] *= al;
        }
#pragma unroll
        for (int p = 0; p < TP / P; ++p) {
            const int pi = p * P + pg;
            if (t0 + pi < end) {
                float vf[8];
                vc[p].get(vf);
#pragma unroll
                for (int j = 0; j < G; ++j) {
                    const float pj = s_p[j][pi];
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[j][e] = fmaf(pj, vf[e], acc[j][e]);
                }
            }
        }
        lds_barrier();
    };
    issue(start, bk[0], bv[0]);
    if (end - start <= TP) {
        tile(start, bk[0], bv[0]);
    } else {
#pragma unroll
        for (int b = 1; b < NB; ++b) issue(start + b * TP, bk[b], bv[b]);
        for (long t0 = start; t0 < end; t0 += NB * TP) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const long tb = t0 + b * TP;
                if (b == 0 || tb < end) tile(tb, bk[b], bv[b]);
                issue(tb + NB * TP, bk[b], bv[b]);
            }
        }
    }
    // Reduce acc over the position groups: lanes d8, d8+T, ... of a wave,
    // then across the 4 waves through LDS.
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float v = acc[j][e];
#pragma unroll
            for (int off = T; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
            acc[j][e] = v;
        }
    if (lane < T) {
#pragma unroll
        for (int j = 0; j < G; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) s_red[wave][j][d8 * 8 + e] = acc[j][e];
    }
#pragma unroll
    for (int i = 0; i < JW; ++i) {
        const int j = wave + 4 * i;
        if (j < G && lane == 0) {
            if constexpr (DIRECT) {
                s_l[j] = l_run[i];
            } else {
                part[j * part_head + HD] = m_run[i];
                part[j * part_head + HD + 1] = l_run[i];
            }
        }
    }
    __syncthreads();
    for (int t = tid; t < G * HD; t += kThreads) {
        const int j = t / HD, d = t % HD;
        const float o = s_red[0][j][d] + s_red[1][j][d] + s_red[2][j][d] + s_red[3][j][d];
        if constexpr (DIRECT) a.out[(size_t)(g * G + j) * HD + d] = o / s_l[j];
        else part[j * part_head + d] = o;
    }
}

// ---------------------------------------------------------------------------
// Decode attention on the matrix cores (BF16 KV, head_dim 64 or 128, up to 8
// query heads per KV head): grid (splits, kv_heads) as attn_kernel, the
// same split boundaries and partial layout. The block's positions are cut
// into 32-position tiles dealt round-robin to its 4 waves; each wave runs its
// own online softmax over its tiles with no block barrier, and the 4 wave
// partials are merged in wave order at the end.
//
// Per tile, with v_mfma_f32_16x16x32_bf16 (lane L: n = L % 16, kg = L / 16):
//   S^T = K Q^T  A = K rows straight from global memory: M-block mb's row m
//                is position t + 8(m/4) + 4mb + m%4; B = the group's queries
//                as hi/lo BF16 halves of the f32 values (heads >= G zero).
//                Lane L then holds the scores of head n at positions
//                t + 8kg + 4mb + j, j = 0..3.
//   O^T += V^T P^T  B = those 8 probabilities (hi/lo halves) exactly as they
//                sit in the lane; A = V^T read from a per-wave LDS copy of the
//                V tile with ds_read_b64_tr_b16 (lane L gets V[t + 8kg + e]
//                [16db + n], e = 0..7, in two reads of four).
// The V tile is stored row-major with the 16-byte chunks of row r permuted
// (chunk c at slot c ^ vswz(r)) so the transposing reads of a half wave hit
// distinct banks. Every K/V load is issued unconditionally (positions past
// the end re-read the last one and are masked), so tile i + 1 streams in
// while tile i computes.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

template <int HD>
__device__ __forceinline__ int vswz(int r) {
    if constexpr (HD == 128) return 2 * ((r & 3) | ((r >> 1) & 4));
    else return 2 * (((r >> 1) & 1) | ((r >> 2) & 2));
}

__device__ __forceinline__ void split_hilo(const float (&v)[8], bf16x8_t &hi, bf16x8_t &lo) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        hi[q] = (__bf16)v[q];
        lo[q] = (__bf16)(v[q] - (float)hi[q]);
    }
}

template <int HD, int G, bool DIRECT, bool ROPE>
__global__ __launch_bounds__(kThreads) void attn_dec_mfma_kernel(AttnArgs a) {
    constexpr int TW = 32;             // positions per wave tile
    constexpr int NS = HD / 32;        // K steps of the score product
    constexpr int NDB = HD / 16;       // 16-dim blocks of the value product
    constexpr int CH = HD / 8;         // 16-byte chunks per K/V row
    constexpr int VI = TW * CH / 64;   // V loads per lane per tile
    constexpr int ROWB = HD * 2;       // bytes per K/V row
    __shared__ __attribute__((aligned(16))) uint8_t s_v[4][TW * ROWB];
    __shared__ float s_o[4][G][HD];
    __shared__ float s_m[4][G], s_l[4][G];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int n = lane & 15, kg = lane >> 4;
    const int split = blockIdx.x, S = gridDim.x;
    const int g = blockIdx.y;
    const long pos = a.pos_dev ? (long)*a.pos_dev : a.offset;
    const long ctx = pos + 1;
    long chunk = (ctx + S - 1) / S;
    chunk = (chunk + TP - 1) / TP * TP;
    const long start = (long)split * chunk;
    const long end = min(start + chunk, ctx);
    const size_t part_head = (size_t)S * (HD + 2);
    float *part = a.part + (size_t)g * G * part_head + (size_t)split * (HD + 2);
    if (start >= ctx) {  // empty split: contributes nothing to the merge
        if (threadIdx.x < G) part[threadIdx.x * part_head + HD] = -INFINITY;
        return;
    }

    // ROPE: the block whose range ends at the context holds position pos,
    // whose K/V row is not in the cache yet. The wave whose tile holds it
    // rotates k (rope_elem, as launch_rope_append), rounds K and V to BF16,
    // appends them to the cache and keeps them in LDS to patch into its
    // tile registers (bits equal to what the cache will hold).
    __shared__ __attribute__((aligned(16))) uint16_t s_new[2][HD];
    const int q_dim = a.q_heads * HD, kv_dim = a.kv_heads * HD, half = a.rotary_dim / 2;
    const float *qkv_row = ROPE ? a.qkv : nullptr;
    const float *cr = ROPE ? a.rope_cos + (size_t)pos * half : nullptr;
    const float *sr = ROPE ? a.rope_sin + (size_t)pos * half : nullptr;
    const int pos_tile = (int)((pos - start) / TW);  // tile index of pos in this block's range
    const bool has_new = ROPE && end == ctx;
    if constexpr (ROPE) {
        if (has_new && wave == pos_tile % 4) {
            const float *kr = qkv_row + q_dim + g * HD, *vr = qkv_row + q_dim + kv_dim + g * HD;
            const int page = a.page_table[pos / a.page_size];
            const size_t off = (((size_t)page * a.kv_heads + g) * a.page_size + pos % a.page_size) * HD;
#pragma unroll
            for (int d = lane; d < HD; d += 64) {
                const uint16_t kb = f32_bf16_rne(rope_elem(kr, d, half, a.rotary_dim, cr, sr));
                const uint16_t vb = f32_bf16_rne(vr[d]);
                s_new[0][d] = kb;
                s_new[1][d] = vb;
                ((uint16_t *)a.k)[off + d] = kb;
                ((uint16_t *)a.v)[off + d] = vb;
            }
        }
    }

    const float scale = 1.0f / sqrtf((float)HD);
    bf16x8_t qh[NS], ql[NS];
    f32x4 o[NDB];
#pragma unroll
    for (int d = 0; d < NDB; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;

    const int ntile = (int)((end - start + TW - 1) / TW);
    const int nt = ntile > wave ? (ntile - 1 - wave) / 4 + 1 : 0;  // this wave's tiles
    struct Regs {
        u32x4 k[2][NS];
        u32x4 v[VI];
    };
    // Buffer loads over the tile's valid rows: a row past `end` reads as
    // zeros and moves no memory (its score is masked, its probability 0).
    // Page of tile i (a scalar load), fetched one tile ahead of its use so
    // the lookup does not add a memory round trip before each tile's loads.
    auto page_of = [&](int i) {
        const long t = start + (long)TW * (wave + 4 * min(i, nt - 1));
        return ((const __attribute__((address_space(4))) int32_t *)a.page_table)[t / a.page_size];
    };
    auto load_tile = [&](int i, int page, Regs &R) {
        i = min(i, nt - 1);
        const long t = start + (long)TW * (wave + 4 * i);
        const size_t base = (((size_t)page * a.kv_heads + g) * a.page_size + t % a.page_size) * HD;
        const int valid = (int)min((long)TW, end - t) * ROWB;
        const __amdgpu_buffer_rsrc_t rk =
            __builtin_amdgcn_make_buffer_rsrc((void *)((const uint16_t *)a.k + base), (short)0, valid, 0x00020000);
        const __amdgpu_buffer_rsrc_t rv =
            __builtin_amdgcn_make_buffer_rsrc((void *)((const uint16_t *)a.v + base), (short)0, valid, 0x00020000);
        const int koff = (8 * (n >> 2) + (n & 3)) * ROWB + 16 * kg;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int s = 0; s < NS; ++s)
                R.k[mb][s] = __builtin_bit_cast(
                    u32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, koff + 4 * mb * ROWB + 64 * s, 0, 0));
        const int voff = (lane / CH) * ROWB + 16 * (lane % CH);
#pragma unroll
        for (int i2 = 0; i2 < VI; ++i2)
            R.v[i2] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, voff, 1024 * i2, 0));
    };
    uint8_t *sv = s_v[wave];
    // First half of a tile: the V tile into this wave's LDS copy and the
    // scores; after it the registers are free for the next tile's loads.
    auto scores = [&](int i, Regs &R, f32x4 (&sc)[2]) {
        if constexpr (ROPE) {
            // The tile holding pos gets the new K/V row (the cache row may
            // not be written yet when the tile was loaded).
            if (has_new && i * 4 + wave == pos_tile) {
                const int rp = (int)(pos - (start + (long)TW * pos_tile));
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const bool mine = 8 * (n >> 2) + 4 * mb + (n & 3) == rp;
#pragma unroll
                    for (int s = 0; s < NS; ++s) {
                        const u32x4 nk = *(const u32x4 *)&s_new[0][32 * s + 8 * kg];
                        R.k[mb][s] = mine ? nk : R.k[mb][s];
                    }
                }
#pragma unroll
                for (int i2 = 0; i2 < VI; ++i2) {
                    const int f = 64 * i2 + lane;
                    const u32x4 nv = *(const u32x4 *)&s_new[1][8 * (f % CH)];
                    R.v[i2] = f / CH == rp ? nv : R.v[i2];
                }
            }
        }
        // V tile into this wave's LDS copy (row f / CH, chunk f % CH).
#pragma unroll
        for (int i2 = 0; i2 < VI; ++i2) {
            const int f = 64 * i2 + lane, r = f / CH, c = f % CH;
            *(u32x4 *)(sv + r * ROWB + 16 * (c ^ vswz<HD>(r))) = R.v[i2];
        }
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const bf16x8_t kA = __builtin_bit_cast(bf16x8_t, R.k[mb][s]);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kA, qh[s], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kA, ql[s], acc, 0, 0, 0);
            }
            sc[mb] = acc;
        }
    };
    // Second half: online softmax and the value product.
    auto mix = [&](int i, const f32x4 (&sc)[2]) {
        const long t = start + (long)TW * (wave + 4 * i);
        // Online softmax of head n over the tile (positions t + 8kg + 4mb + j).
        float p[8];
        float tmax = -INFINITY;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool ok = t + 8 * kg + 4 * mb + j < end;
                const float v = ok ? sc[mb][j] * scale : -INFINITY;
                p[4 * mb + j] = v;
                tmax = fmaxf(tmax, v);
            }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
        const float m_new = fmaxf(m_run, tmax);
        const float alpha = m_run == -INFINITY ? 0.f : expf(m_run - m_new);
        float lsum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            p[e] = p[e] == -INFINITY ? 0.f : expf(p[e] - m_new);
            lsum += p[e];
        }
        lsum += __shfl_xor(lsum, 16, 64);
        lsum += __shfl_xor(lsum, 32, 64);
        l_run = l_run * alpha + lsum;
        m_run = m_new;
        bf16x8_t ph, pl;
        split_hilo(p, ph, pl);
        // O^T += V^T P^T.
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
            s16x4_t h0, h1;
            {
                const int r0 = 8 * kg + (n >> 2), c = 2 * db + ((n & 3) >> 1), b8 = (n & 1) * 8;
                const int r1 = r0 + 4;
                h0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s16x4_t *)(sv + r0 * ROWB + 16 * (c ^ vswz<HD>(r0)) + b8));
                h1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s16x4_t *)(sv + r1 * ROWB + 16 * (c ^ vswz<HD>(r1)) + b8));
            }
            const bf16x8_t vA = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7));
            f32x4 acc = o[db] * alpha;
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vA, ph, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vA, pl, acc, 0, 0, 0);
            o[db] = acc;
        }
    };
    // One register set: tile i + 1's loads are issued as soon as tile i's
    // registers have been consumed, and stream in during its softmax and
    // value product (and the other waves' work).
    if (nt > 0) {
        // The group's queries (raw f32 now, converted after the first tile's
        // loads are issued, so the two round trips overlap).
        f32x4 qraw[NS][2];
        // ROPE (rotary width = head_dim): the raw pairs and cos/sin of the
        // lane's 8 dims (all below or all at/above half: multiples of 8).
        f32x4 qpair[ROPE ? NS : 1][4], qcs[ROPE ? NS : 1][4];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            // Every lane loads (lanes past the group re-read head 0 and are
            // zeroed at conversion): no divergent load for the waits to trip on.
            if constexpr (ROPE) {
                const int d0 = 32 * s + 8 * kg;
                const float *src = qkv_row + (size_t)(g * G + (n < G ? n : 0)) * HD;
                const int i0 = d0 < half ? d0 : d0 - half;
#pragma unroll
                for (int k = 0; k < 4; ++k) qpair[s][k] = *(const f32x4 *)(src + 2 * i0 + 4 * k);
                qcs[s][0] = *(const f32x4 *)(cr + i0);
                qcs[s][1] = *(const f32x4 *)(cr + i0 + 4);
                qcs[s][2] = *(const f32x4 *)(sr + i0);
                qcs[s][3] = *(const f32x4 *)(sr + i0 + 4);
            } else {
                const float *qp = a.q + (size_t)(g * G + (n < G ? n : 0)) * HD + 32 * s + 8 * kg;
                qraw[s][0] = *(const f32x4 *)qp;
                qraw[s][1] = *(const f32x4 *)(qp + 4);
            }
        }
        const int pg0 = page_of(0);
        int pg_next = page_of(1);
        Regs R;
        load_tile(0, pg0, R);
        __builtin_amdgcn_sched_barrier(0);
        // The queries as the score product's B operand, hi/lo BF16 halves.
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            float qv[8];
            const int d0 = 32 * s + 8 * kg;
            if constexpr (ROPE) {
                // rope_elem's arithmetic: a*c - b*s below half, b*c + a*s above.
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float pa = qpair[ROPE ? s : 0][(2 * e) >> 2][(2 * e) & 3];
                    const float pb = qpair[ROPE ? s : 0][(2 * e + 1) >> 2][(2 * e + 1) & 3];
                    const float c = qcs[ROPE ? s : 0][e >> 2][e & 3], sn = qcs[ROPE ? s : 0][2 + (e >> 2)][e & 3];
                    const float r = d0 < half ? pa * c - pb * sn : pb * c + pa * sn;
                    qv[e] = n < G ? r : 0.f;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    qv[e] = n < G ? qraw[s][0][e] : 0.f;
                    qv[4 + e] = n < G ? qraw[s][1][e] : 0.f;
                }
            }
            split_hilo(qv, qh[s], ql[s]);
        }
        for (int i = 0; i < nt; ++i) {
            f32x4 sc[2];
            scores(i, R, sc);
            const int pg_after = page_of(i + 2);
            load_tile(i + 1, pg_next, R);
            pg_next = pg_after;
            __builtin_amdgcn_sched_barrier(0);
            mix(i, sc);
        }
    }
    // Merge the wave partials in wave order.
    if (n < G) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j) s_o[wave][n][16 * db + 4 * kg + j] = o[db][j];
        if (kg == 0) {
            s_m[wave][n] = m_run;
            s_l[wave][n] = l_run;
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * HD; idx += kThreads) {
        const int j = idx / HD, d = idx % HD;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) M = fmaxf(M, s_m[w][j]);
        float acc = 0.f, L = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float mw = s_m[w][j];
            if (mw != -INFINITY) {
                const float sw = expf(mw - M);
                acc = fmaf(sw, s_o[w][j][d], acc);
                L = fmaf(sw, s_l[w][j], L);
            }
        }
        if constexpr (DIRECT) {
            a.out[(size_t)(g * G + j) * HD + d] = acc / L;
        } else {
            part[j * part_head + d] = acc;
            if (d == 0) {
                part[j * part_head + HD] = M;
                part[j * part_head + HD + 1] = L;
            }
        }
    }
}

// Merge the splits of one q head in split order: one wave turns the
// split maxima into weights w_s = exp(m_s - M) and 1 / sum_s w_s l_s, then
// all threads sum w_s * o_s[d] over the non-empty splits.
template <int HD>
__global__ __launch_bounds__(kThreads) void attn_combine_kernel(const float *part, int S, float *out) {
    constexpr int GR = kThreads / HD;  // split groups
    __shared__ float s_w[kMaxSplits];
    __shared__ float s_inv;
    __shared__ float s_o[GR][HD];
    const int h = blockIdx.x, tid = threadIdx.x;
    const float *p = part + (size_t)h * (size_t)S * (HD + 2);
    static_assert(kMaxSplits <= 128, "one wave holds two splits per lane");
    if (tid < 64) {
        const int s1 = tid + 64;
        const float m0 = tid < S ? p[(size_t)tid * (HD + 2) + HD] : -INFINITY;
        const float m1 = s1 < S ? p[(size_t)s1 * (HD + 2) + HD] : -INFINITY;
        const float M = wave_max(fmaxf(m0, m1));
        const float w0 = m0 == -INFINITY ? 0.f : expf(m0 - M);
        const float w1 = m1 == -INFINITY ? 0.f : expf(m1 - M);
        const float l0 = w0 != 0.f ? p[(size_t)tid * (HD + 2) + HD + 1] : 0.f;
        const float l1 = w1 != 0.f ? p[(size_t)s1 * (HD + 2) + HD + 1] : 0.f;
        const float L = wave_sum(w0 * l0) + wave_sum(w1 * l1);
        if (tid < S) s_w[tid] = w0;
        if (s1 < S) s_w[s1] = w1;
        if (tid == 0) s_inv = 1.0f / L;
    }
    __syncthreads();
    const int d = tid % HD, grp = tid / HD;
    // The split values this thread folds are loaded 16 at a time (one memory
    // round trip per batch), then folded in split order.
    constexpr int PER = kMaxSplits / GR, BATCH = PER < 16 ? PER : 16;
    float o = 0.f;
    for (int i0 = 0; i0 < PER && grp + GR * i0 < S; i0 += BATCH) {
        float v[BATCH];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int s = grp + GR * (i0 + i);
            v[i] = s < S ? p[(size_t)s * (HD + 2) + d] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int s = grp + GR * (i0 + i);
            const float w = s < S ? s_w[s] : 0.f;
            if (w != 0.f) o = fmaf(w, v[i], o);
        }
    }
    s_o[grp][d] = o;
    __syncthreads();
    if (tid < HD) {
        float sum = s_o[0][tid];
#pragma unroll
        for (int k = 1; k < GR; ++k) sum += s_o[k][tid];
        out[(size_t)h * HD + tid] = sum * s_inv;
    }
}

// ---------------------------------------------------------------------------
// Chunked prefill on the matrix cores (BF16 KV): flash attention with the
// score and value products as v_mfma_f32_32x32x16_bf16.
//
// A block is 4 waves and one KV head; each wave owns 32 "M rows" = RW query
// rows x G heads of the group (RW = 32 / G). Per 64-position tile:
//   S^T = K Q^T  (A = K rows from LDS, B = Q^T kept in registers as hi/lo
//                BF16 halves of the f32 query, so scores carry ~2^-17
//                relative error); every lane ends up holding one M row's
//                scores (column = lane % 32), so the online softmax (running
//                max / sum, rescale) is lane-local plus one exchange with
//                lane ^ 32.
//   O^T += V^T P^T (A = V^T from LDS, B = P^T straight from the S^T
//                registers, again as hi/lo BF16 halves).
// K rows are staged in LDS with bits 2 and 3 of the position swapped, which
// makes the S^T output registers exactly the B operand layout of the second
// product (8 consecutive positions per lane), so P never moves between lanes.
// V rows are staged as they come and read transposed (ds_read_b64_tr_b16).
//
// Bound: the matrix cores at two waves per SIMD (236 registers at head_dim
// 128). Both tiles' copies go global -> LDS by buffer loads and the LDS reads
// are such that the compiler waits for no copy in flight: with global loads to
// LDS, builtin transposing reads or a vector load of the page table it waited
// for the next tile's copies (or the table) inside every tile. V through
// registers and 16-bit transposing stores cost the rest. 512 rows on a 4K
// prefix, 32 q / 8 KV heads of 128: 113 -> 89.8 us (316 -> 398 TFLOP/s, twice
// that executed), with the same bits; rows direct to LDS and transposing reads
// alone 97.5 us. At head_dim 64 (the small decoder's 16-block grids, where a
// wave's chain of tiles is the time) both halves of a tile share one softmax
// round: Qwen2-0.5B prefill of 512 tokens 7.47 -> 7.42 ms.
//
// Splits are absolute position ranges of `span` keys (fixed per model), so
// every row's result depends only on its own position (the same bits however
// the prompt is chunked); the splits of a row are merged in order by
// attn_merge2_kernel.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// LDS row of a position within a 64-position tile (an involution).
__device__ __forceinline__ int krow_of(int p) { return (p & ~12) | ((p & 4) << 1) | ((p & 8) >> 1); }

// hi = bf16(v) and lo = bf16(v - hi) (hardware round-to-nearest-even
// conversions), so hi + lo carries v to ~2^-17 relative error.
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8 &hi, bf16x8 &lo) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        hi[q] = (__bf16)v[q];
        lo[q] = (__bf16)(v[q] - (float)hi[q]);
    }
}

// Column of position p (0..63) in row d of the transposed V tile: groups of 8
// positions are XOR-swizzled by the row's dim group, so the transposing
// stores of one wave spread over the LDS banks while every 8-position group
// stays one aligned 16-byte read.
__device__ __forceinline__ int vcol(int d, int p) { return (((p >> 3) ^ ((d >> 3) & 7)) << 3) | (p & 7); }

// A prefill lane's results, O^T registers of its M row: dims
// 32 u + 8 (r / 4) + 4 half + r % 4. One split: the normalised output at
// element ob (with its BF16 halves where asked for); more: the partial.
template <int HD>
__device__ __forceinline__ void store_prefill_rows(const AttnArgs &a, const f32x16 (&oacc)[HD / 32], float m2, float l,
                                                   float *part, size_t ob, int S, int half) {
    constexpr int UT = HD / 32;
    if (S == 1) {
        const float inv = 1.0f / l;
#pragma unroll
        for (int u = 0; u < UT; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 v = f32x4{oacc[u][4 * q] * inv, oacc[u][4 * q + 1] * inv, oacc[u][4 * q + 2] * inv,
                                      oacc[u][4 * q + 3] * inv};
                if (a.out) *(f32x4 *)(a.out + ob + 32 * u + 8 * q + 4 * half) = v;
                if (a.out_hi) store_halves4(a.out_hi, a.out_lo, ob + 32 * u + 8 * q + 4 * half, v);
            }
    } else {
#pragma unroll
        for (int u = 0; u < UT; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *(f32x4 *)(part + 32 * u + 8 * q + 4 * half) =
                    f32x4{oacc[u][4 * q], oacc[u][4 * q + 1], oacc[u][4 * q + 2], oacc[u][4 * q + 3]};
        if (half == 0) {
            part[HD] = m2;
            part[HD + 1] = l;
        }
    }
}

// Chunk swizzle of V row r: the rows a transposing read takes together (four
// consecutive ones, 64 bytes each) fall on distinct banks, and rows r and
// r + 4 share it.
template <int HD>
__device__ __forceinline__ int vseg(int r) {
    return HD == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1);
}

// The V^T fragments of 16 positions, all HD dims, by transposing LDS reads at
// the UT lane addresses + OFF (rows 0..3) and + OFF + 4 rows. Inline assembly:
// for the builtin the compiler waits for every copy in flight (the next tile's)
// first; each block waits for its own data.
template <int HD, int OFF>
__device__ __forceinline__ void read_vt(const uint32_t (&addr)[HD / 32], bf16x8 (&va)[HD / 32]) {
    constexpr int OFF4 = OFF + 4 * HD * 2;
    s16x4_t r[HD / 32][2];
    if constexpr (HD == 128) {
        asm volatile(
            "ds_read_b64_tr_b16 %0, %8 offset:%12\n\tds_read_b64_tr_b16 %1, %8 offset:%13\n\t"
            "ds_read_b64_tr_b16 %2, %9 offset:%12\n\tds_read_b64_tr_b16 %3, %9 offset:%13\n\t"
            "ds_read_b64_tr_b16 %4, %10 offset:%12\n\tds_read_b64_tr_b16 %5, %10 offset:%13\n\t"
            "ds_read_b64_tr_b16 %6, %11 offset:%12\n\tds_read_b64_tr_b16 %7, %11 offset:%13\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(r[0][0]), "=&v"(r[0][1]), "=&v"(r[1][0]), "=&v"(r[1][1]), "=&v"(r[2][0]), "=&v"(r[2][1]),
              "=&v"(r[3][0]), "=&v"(r[3][1])
            : "v"(addr[0]), "v"(addr[1]), "v"(addr[2]), "v"(addr[3]), "i"(OFF), "i"(OFF4)
            : "memory");
    } else {
        asm volatile(
            "ds_read_b64_tr_b16 %0, %4 offset:%6\n\tds_read_b64_tr_b16 %1, %4 offset:%7\n\t"
            "ds_read_b64_tr_b16 %2, %5 offset:%6\n\tds_read_b64_tr_b16 %3, %5 offset:%7\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(r[0][0]), "=&v"(r[0][1]), "=&v"(r[1][0]), "=&v"(r[1][1])
            : "v"(addr[0]), "v"(addr[1]), "i"(OFF), "i"(OFF4)
            : "memory");
    }
#pragma unroll
    for (int u = 0; u < HD / 32; ++u)
        va[u] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(r[u][0], r[u][1], 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int HD, int G>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void attn_prefill_kernel(AttnArgs a, int rows, int S, int span) {
    constexpr int RW = 32 / G, MV = RW * G;
    constexpr int KSTEPS = HD / 16, UT = HD / 32, KC = HD / 32;
    constexpr int CPR = HD / 8;  // 16-byte chunks per K row
    constexpr int NH = HD == 64 ? 2 : 1;  // 32-position halves per softmax step
    // Two tiles each. K rows unpadded, chunk c of LDS row r stored at chunk
    // c ^ (r % CPR); V rows as they come, 64-byte segments swizzled by vseg.
    extern __shared__ __attribute__((aligned(16))) uint8_t smem_kv[];
    uint8_t *ks = smem_kv, *vs = smem_kv + 2 * 64 * HD * 2;
    constexpr int TB = 64 * HD * 2;  // bytes of one tile
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int n = lane & 31, half = lane >> 5;
    const int rb = blockIdx.x, g = blockIdx.y, split = blockIdx.z;
    const int row = rb * 4 * RW + wave * RW + n / G;
    const int head = g * G + n % G;
    const bool rvalid = n < MV && row < rows;
    // Positions fit in 32 bits (the KV capacity is checked on the host).
    const int off = (int)a.offset;
    const int my_pos = off + row;
    const int first_pos = off + rb * 4 * RW;
    const int ctx = off + min(rows, (rb + 1) * 4 * RW);
    const int start = split * span;
    const int end = min(start + span, ctx);
    float *part = a.part + (((size_t)row * a.q_heads + head) * S + split) * (HD + 2);
    if (start >= ctx) {  // block-uniform: no row of this block reaches the split
        if (rvalid && half == 0) part[HD] = -INFINITY;
        return;
    }

    // Q^T operands (B of S^T = K Q^T): lane holds Q[m = lane % 32][16 s + 8 half .. +8],
    // pre-scaled by log2(e) / sqrt(HD) so scores come out in the exp2 domain.
    bf16x8 qh[KSTEPS], ql[KSTEPS];
    {
        const float sl2 = (1.0f / sqrtf((float)HD)) * 1.44269504088896340736f;
        const float *qp = a.q + (size_t)(rvalid ? row : 0) * a.q_stride + (size_t)(rvalid ? head : 0) * HD + 8 * half;
        const float sq = rvalid ? sl2 : 0.f;  // rows without a query: their scores are not used
        f32x4 raw[KSTEPS][2];  // every load before the first use: one round trip
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
            raw[s][0] = *(const f32x4 *)(qp + 16 * s);
            raw[s][1] = *(const f32x4 *)(qp + 16 * s + 4);
        }
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
            const float v[8] = {raw[s][0][0] * sq, raw[s][0][1] * sq, raw[s][0][2] * sq, raw[s][0][3] * sq,
                                raw[s][1][0] * sq, raw[s][1][1] * sq, raw[s][1][2] * sq, raw[s][1][3] * sq};
            split8(v, qh[s], ql[s]);
        }
    }

    // K and V: direct global->LDS copies (buffer loads: the compiler waits for
    // no copy in flight when it reads LDS). Copy c of a wave fills 1 KB =
    // 64 / CPR LDS rows from row r0 = (wave + 4 c) 64 / CPR on; lane i lands at
    // byte 16 i, so it fetches the global chunk that the swizzle places there.
    // c moves r0 by a multiple of 16: the lane's offset is the same plus 4 KB.
    // K rows past the split end may hold stale bytes: their scores are masked
    // before use.
    constexpr int RPI = 64 / CPR;
    const int lr = wave * RPI + lane / CPR;  // LDS row of copy 0
    const int koff = krow_of(lr) * HD * 2 + 16 * ((lane % CPR) ^ (lr % CPR));
    const int voff = lr * HD * 2 + 16 * ((lane % CPR) ^ vseg<HD>(lr));
    // Page of the tile at t0: a scalar load, one tile ahead of its use.
    auto page_of = [&](int t0) {
        return ((const __attribute__((address_space(4))) int32_t *)a.page_table)[t0 / a.page_size];
    };
    auto fetch = [&](int t0, int page, int b) {
        const size_t tile = (((size_t)page * a.kv_heads + g) * a.page_size + (t0 % a.page_size)) * HD;
        const __amdgpu_buffer_rsrc_t rk =
            __builtin_amdgcn_make_buffer_rsrc((void *)((const uint16_t *)a.k + tile), (short)0, TB, 0x00020000);
        const __amdgpu_buffer_rsrc_t rv =
            __builtin_amdgcn_make_buffer_rsrc((void *)((const uint16_t *)a.v + tile), (short)0, TB, 0x00020000);
#pragma unroll
        for (int c = 0; c < KC; ++c) buf_to_lds<16>(rk, ks + b * TB + wave * 1024 + 4096 * c, koff, 4096 * c);
#pragma unroll
        for (int c = 0; c < KC; ++c) buf_to_lds<16>(rv, vs + b * TB + wave * 1024 + 4096 * c, voff, 4096 * c);
    };
    // This wave's V rows past the split end, once they have landed: they may
    // be unwritten memory, and a probability of 0 does not clear a NaN. (An
    // infinite or NaN V that was written does reach the tile's earlier rows so.)
    auto clear_v = [&](int t0, int b) {
#pragma unroll
        for (int c = 0; c < KC; ++c)
            if (t0 + lr + 4 * RPI * c >= end)
                *(u32x4 *)(vs + b * TB + wave * 1024 + 4096 * c + 16 * lane) = u32x4{0u, 0u, 0u, 0u};
    };
    // This lane's transposing V reads in a 16-position block: rows
    // 8 half + i / 4 (and + 4), dims 32 u + 16 ((lane / 16) % 2) + 4 (i % 4).
    const int vi = lane & 15, vrow = 8 * half + (vi >> 2);
    uint32_t vaddr[UT];
#pragma unroll
    for (int u = 0; u < UT; ++u) {
        const int chunk = (4 * u + 2 * ((lane >> 4) & 1) + ((vi & 3) >> 1)) ^ vseg<HD>(vrow);
        vaddr[u] = (uint32_t)(uintptr_t)(vs + vrow * HD * 2 + 16 * chunk + 8 * (vi & 1));
    }

    f32x16 oacc[UT];
#pragma unroll
    for (int u = 0; u < UT; ++u) oacc[u] = f32x16{};
    float m2 = -INFINITY, l = 0.f;
    fetch(start, page_of(start), 0);
    const int last_tile = start + (end - 1 - start) / 64 * 64;
    int page_next = page_of(min(start + 64, last_tile));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (start + 64 > end) clear_v(start, 0);
    __syncthreads();
    int b = 0;
    for (int t0 = start; t0 < end; t0 += 64) {
        const bool more = t0 + 64 < end;
        if (more) {
            fetch(t0 + 64, page_next, b ^ 1);
            page_next = page_of(min(t0 + 128, last_tile));
        }
        // Steps of 32 NH positions, each: S^T, online softmax, O^T update. At
        // head_dim 64 the registers hold both halves of the tile at once: two
        // independent score chains and one softmax round for 64 keys.
        uint32_t vad[UT];
#pragma unroll
        for (int u = 0; u < UT; ++u) vad[u] = vaddr[u] + b * TB;
        auto step = [&](auto step_index) {
            constexpr int p0 = 32 * NH * decltype(step_index)::value;
            f32x16 sacc[NH];
#pragma unroll
            for (int x = 0; x < NH; ++x) sacc[x] = f32x16{};
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) {
                bf16x8 ka[NH];
#pragma unroll
                for (int x = 0; x < NH; ++x) {
                    const int r = p0 + 32 * x + n;
                    ka[x] = __builtin_bit_cast(
                        bf16x8, *(const u32x4 *)(ks + b * TB + r * HD * 2 + 16 * ((2 * s + half) ^ (r % CPR))));
                }
#pragma unroll
                for (int x = 0; x < NH; ++x)
                    sacc[x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[x], qh[s], sacc[x], 0, 0, 0);
#pragma unroll
                for (int x = 0; x < NH; ++x)
                    sacc[x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[x], ql[s], sacc[x], 0, 0, 0);
            }
            // The step's V^T fragments, while the score products drain.
            bf16x8 va[2 * NH][UT];
            read_vt<HD, p0 * HD * 2>(vad, va[0]);
            read_vt<HD, (p0 + 16) * HD * 2>(vad, va[1]);
            if constexpr (NH == 2) {
                read_vt<HD, (p0 + 32) * HD * 2>(vad, va[2]);
                read_vt<HD, (p0 + 48) * HD * 2>(vad, va[3]);
            }
            // Causal / split-end mask, only where the step reaches past a
            // row's position or past the split (block-uniform test).
            const int h0 = t0 + p0;
            if (h0 + 32 * NH - 1 > first_pos || h0 + 32 * NH > end) {
#pragma unroll
                for (int x = 0; x < NH; ++x)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int p = h0 + 32 * x + krow_of(8 * (r >> 2) + 4 * half + (r & 3));
                        if (p > my_pos || p >= end) sacc[x][r] = -INFINITY;
                    }
            }
            float tmax = -INFINITY;
#pragma unroll
            for (int x = 0; x < NH; ++x)
#pragma unroll
                for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, sacc[x][r]);
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
            // Delayed rescaling: exponentials are taken against a reference
            // max m2 that is raised only when a score exceeds it by more than
            // 8 (log2 units), so p <= 256 and the O / l rescale is rare. Each
            // row's steps depend only on its own scores.
            const bool raise = tmax > m2 + 8.0f;
            if (__any(raise)) {
                const float mnew = raise ? tmax : m2;
                const float alpha = __builtin_amdgcn_exp2f(m2 - mnew);  // 1 where not raised, 0 from -inf
                l *= alpha;
#pragma unroll
                for (int u = 0; u < UT; ++u)
#pragma unroll
                    for (int r = 0; r < 16; ++r) oacc[u][r] *= alpha;
                m2 = mnew;
            }
            // A row with every score so far masked keeps m2 = -inf; its terms are 0.
            const float mref = m2 == -INFINITY ? 0.f : m2;
            float tsum = 0.f;
#pragma unroll
            for (int x = 0; x < NH; ++x)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float pv = __builtin_amdgcn_exp2f(sacc[x][r] - mref);
                    sacc[x][r] = pv;
                    tsum += pv;
                }
            tsum += __shfl_xor(tsum, 32, 64);
            l += tsum;
            // O^T += V^T P^T over steps of 16 positions.
#pragma unroll
            for (int s2 = 0; s2 < 2 * NH; ++s2) {
                float pv[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) pv[j] = sacc[s2 >> 1][8 * (s2 & 1) + j];
                bf16x8 bh, bl;
                split8(pv, bh, bl);
#pragma unroll
                for (int u = 0; u < UT; ++u) {
                    oacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[s2][u], bh, oacc[u], 0, 0, 0);
                    oacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[s2][u], bl, oacc[u], 0, 0, 0);
                }
            }
        };
        step(std::integral_constant<int, 0>{});
        if constexpr (NH == 1) step(std::integral_constant<int, 1>{});
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (more && t0 + 128 > end) clear_v(t0 + 64, b ^ 1);
        __syncthreads();
        b ^= 1;
    }
    if (!rvalid) return;
    store_prefill_rows<HD>(a, oacc, m2, l, part, (size_t)row * a.q_heads * HD + (size_t)head * HD, S, half);
}

// ---------------------------------------------------------------------------
// Chunked prefill over an f32 K/V cache on the matrix cores: the flash
// attention of attn_prefill_kernel (same blocks, rows per wave, LDS row
// permutation, transposed V, delayed rescaling and split partials) with every
// f32 operand as three BF16 parts (hi = the top 16 bits, mid = bf16 of the
// rest, lo = what is left: all 24 bits exactly). mid is below 2^-7 of the value
// (hi is cut, not rounded) and lo below 2^-16, so of the nine part products the
// three left out (mid x lo twice, lo x lo) are together below 2^-22 of the
// product; the other six are taken, smallest first, and the score's small ones
// add up in an accumulator of their own. Their signs vary: over 128 dims the
// scores are 6e-8 (RMS) off, f32 products summed in order 2e-7.
//
// Bound: the matrix cores (six BF16 products per f32 one, i.e. at most 1/6 of
// the BF16 rate; the f32 MFMA's rate is 1/16 of it). K/V are split once per
// block and tile while they are staged (64 keys x head_dim, three planes of K
// rows and of V columns in LDS: 102 KB at head_dim 128, so one block of four
// waves per CU with 512 registers each; the next tile's rows wait in
// registers during the products).
// Measured on 512-row chunks of a 1,500-token prompt, 32 q / 8 KV heads of
// 128: 40 / 80 / 128 us a chunk against 1,025 to 1,781 us on the vector ALUs
// (attn_kernel, which decodes only now); that prompt through two Q4 layers of
// the shape 11.94 -> 4.36 ms, its logits no further from 64-bit ones.
//
// Infinities and NaN as f32 products give them (plain_row): the parts do not
// carry them. Staging clamps V, the scores' NaN shows in the weight sum; 0.4 %
// of that prompt's time, 2 to 3 % of a 512-row chunk's deep in a long cache.
// ---------------------------------------------------------------------------
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

struct Parts2 {  // two values' parts, packed
    uint32_t h, m, l;
};
__device__ __forceinline__ Parts2 split3(float a, float b) {
    const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
    const float ra = a - __uint_as_float(ua & 0xFFFF0000u), rb = b - __uint_as_float(ub & 0xFFFF0000u);
    const __bf16 ma = (__bf16)ra, mb = (__bf16)rb;
    const __bf16 la = (__bf16)(ra - (float)ma), lb = (__bf16)(rb - (float)mb);
    Parts2 p;
    p.h = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
    p.m = (uint32_t)__builtin_bit_cast(uint16_t, ma) | ((uint32_t)__builtin_bit_cast(uint16_t, mb) << 16);
    p.l = (uint32_t)__builtin_bit_cast(uint16_t, la) | ((uint32_t)__builtin_bit_cast(uint16_t, lb) << 16);
    return p;
}
// Eight values' parts as three matrix operands.
__device__ __forceinline__ void split3x8(const float (&v)[8], bf16x8 (&out)[3]) {
    u32x4 w[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const Parts2 p = split3(v[2 * i], v[2 * i + 1]);
        w[0][i] = p.h;
        w[1][i] = p.m;
        w[2][i] = p.l;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) out[k] = __builtin_bit_cast(bf16x8, w[k]);
}

constexpr int kF32LdV = 64 + 8;  // transposed V row: 64 positions + 16 bytes
template <int HD>
constexpr size_t prefill_f32_lds_bytes() { return (size_t)3 * 2 * (64 * HD + HD * kF32LdV) + 16; }

// One more part of a row's softmax (maximum m, weight sum l, values o) folded
// into the running one (M, L, O), parts in order; a part without a key (m =
// -inf) changes nothing. The factors of a part, for every value of the row.
__device__ __forceinline__ void fold_factors(float m, float &M, float &alpha, float &beta) {
    const float mn = fmaxf(M, m);
    const bool any = m != -INFINITY;
    alpha = any ? __builtin_amdgcn_exp2f(M - mn) : 1.f;
    beta = any ? __builtin_amdgcn_exp2f(m - mn) : 0.f;
    M = mn;
}
__device__ __forceinline__ float fold_value(float O, float o, float alpha, float beta) {
    return fmaf(beta, o, O * alpha);
}

// 2^119: weights of up to 2^8 take the product with a larger V past the largest
// number.
constexpr float kBigV = 0x1p119f;

// One row's attention over positions [p0, p1) in plain f32 products, parts of
// `sub` positions folded in order, a lane's HD / 2 dims of it stored as
// store_prefill_rows does: the rare rows whose operands the BF16 parts do not
// carry. A call, so that it takes no registers of the loop's. A NaN weight sum
// is the row's result: it ends there, with a maximum that no split outweighs.
template <int HD>
__device__ __attribute__((noinline)) void plain_row(AttnArgs a, int row, int head, int g, int half, int p0, int p1, int sub,
                                              float *part, int S) {
    constexpr int UT = HD / 32;
    const float *qp = a.q + (size_t)row * a.q_stride + (size_t)head * HD;
    const float sl2 = (1.0f / sqrtf((float)HD)) * 1.44269504088896340736f;
    f32x16 o[UT];
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int u = 0; u < UT; ++u) o[u] = f32x16{};
#pragma unroll 1
    for (; p0 < p1 && L == L; p0 += sub) {
        f32x16 t[UT];
        float m = -INFINITY, l = 0.f;
#pragma unroll
        for (int u = 0; u < UT; ++u) t[u] = f32x16{};
#pragma unroll 1
        for (int p = p0; p < min(p0 + sub, p1) && l == l; ++p) {
            const size_t at = (((size_t)a.page_table[p / a.page_size] * a.kv_heads + g) * a.page_size + p % a.page_size) * HD;
            const float *kp = (const float *)a.k + at, *vp = (const float *)a.v + at + 4 * half;
            float dot = 0.f;
#pragma unroll 1
            for (int d = 0; d < HD; d += 16) {
                f32x4 q[4], k[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) q[i] = *(const f32x4 *)(qp + d + 4 * i), k[i] = *(const f32x4 *)(kp + d + 4 * i);
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) dot = fmaf(k[i][e], q[i][e], dot);
            }
            const float s = dot * sl2, mn = fmaxf(m, s);
            const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
            const float w = s == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s - mn);
            m = mn;
            l = l * alpha + w;
#pragma unroll
            for (int u = 0; u < UT; ++u)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 v = *(const f32x4 *)(vp + 32 * u + 8 * q);
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[u][4 * q + e] = fmaf(w, v[e], t[u][4 * q + e] * alpha);
                }
        }
        float alpha, beta;
        if (l != l) m = INFINITY;
        const bool any = m != -INFINITY;
        fold_factors(m, M, alpha, beta);
        L = any ? fold_value(L, l, alpha, beta) : L;
#pragma unroll
        for (int u = 0; u < UT; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[u][r] = any ? fold_value(o[u][r], t[u][r], alpha, beta) : o[u][r];
    }
    store_prefill_rows<HD>(a, o, M, L, part, (size_t)row * a.q_heads * HD + (size_t)head * HD, S, half);
}

// FOLD: the block's split is longer than `sub` keys; its parts of `sub` keys
// are folded in registers, in order (launch_prefill_f32).
template <int HD, int G, bool FOLD>
__global__ __launch_bounds__(kThreads, HD == 64 ? 2 : 1) void attn_prefill_f32_kernel(AttnArgs a, int rows, int S,
                                                                                     int span, int sub) {
    constexpr int RW = 32 / G, MV = RW * G;
    constexpr int LDV = kF32LdV;
    constexpr int KSTEPS = HD / 16, UT = HD / 32;
    constexpr int CPR = HD / 8;    // 16-byte chunks per K row and plane
    constexpr int KU = HD / 32;    // K staging units (8 dims of a row) per thread
    constexpr int VU = HD / 64;    // V staging units (4 positions x 4 dims) per thread
    extern __shared__ __attribute__((aligned(16))) uint16_t smem_f32[];
    uint16_t *ks = smem_f32;               // [3][64][HD], chunks swizzled as in attn_prefill_kernel
    uint16_t *vt = smem_f32 + 3 * 64 * HD;  // [3][HD][LDV]
    int *big_pos = (int *)(vt + 3 * HD * LDV);  // first position with a V value of kBigV or more
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 31, half = lane >> 5;
    const int rb = blockIdx.x, g = blockIdx.y, split = blockIdx.z;
    const int row = rb * 4 * RW + wave * RW + n / G;
    const int head = g * G + n % G;
    const bool rvalid = n < MV && row < rows;
    const int off = (int)a.offset;
    const int my_pos = off + row;
    const int first_pos = off + rb * 4 * RW;
    const int ctx = off + min(rows, (rb + 1) * 4 * RW);
    const int start = split * span;
    const int end = min(start + span, ctx);
    float *part = a.part + (((size_t)row * a.q_heads + head) * S + split) * (HD + 2);
    if (start >= ctx) {  // block-uniform: no row of this block reaches the split
        if (rvalid && half == 0) part[HD] = -INFINITY;
        return;
    }

    // The next tile's rows in registers. K unit: 8 dims of position idx / CPR;
    // V unit: 4 dims of positions 4 (idx / (HD / 4)) .. + 3.
    const float *kbase = (const float *)a.k, *vbase = (const float *)a.v;
    f32x4 kr[KU][2], vr[VU][4];
    auto page_of = [&](int t0) {  // a scalar load, one tile ahead of its use
        return ((const __attribute__((address_space(4))) int32_t *)a.page_table)[t0 / a.page_size];
    };
    auto fetch = [&](int t0, int page) {
        const size_t tile = (((size_t)page * a.kv_heads + g) * a.page_size + (t0 % a.page_size)) * HD;
#pragma unroll
        for (int c = 0; c < KU; ++c) {
            const int idx = tid + kThreads * c;
            const float *src = kbase + tile + (size_t)(idx / CPR) * HD + (idx % CPR) * 8;
            kr[c][0] = *(const f32x4 *)src;
            kr[c][1] = *(const f32x4 *)(src + 4);
        }
#pragma unroll
        for (int c = 0; c < VU; ++c) {
            const int idx = tid + kThreads * c, p0 = 4 * (idx / (HD / 4)), d0 = 4 * (idx % (HD / 4));
#pragma unroll
            for (int i = 0; i < 4; ++i)  // positions past the split end may be unwritten: zeros (p = 0 there)
                vr[c][i] = t0 + p0 + i < end ? *(const f32x4 *)(vbase + tile + (size_t)(p0 + i) * HD + d0)
                                             : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // V values of kBigV or more (infinities; NaN comes out as -kBigV) are staged
    // as +-kBigV: as 0 x V they reach no row that does not see them.
    float top = 0.f;
    auto stage = [&]() {
#pragma unroll
        for (int c = 0; c < VU; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    vr[c][i][e] = __builtin_amdgcn_fmed3f(vr[c][i][e], -kBigV, kBigV);
                    top = fmaxf(top, fabsf(vr[c][i][e]));
                }
#pragma unroll
        for (int c = 0; c < KU; ++c) {
            const int idx = tid + kThreads * c, r = krow_of(idx / CPR);
            const float v[8] = {kr[c][0][0], kr[c][0][1], kr[c][0][2], kr[c][0][3],
                                kr[c][1][0], kr[c][1][1], kr[c][1][2], kr[c][1][3]};
            bf16x8 w[3];
            split3x8(v, w);
            uint16_t *dst = ks + r * HD + (((idx % CPR) ^ (r % CPR)) << 3);
#pragma unroll
            for (int k = 0; k < 3; ++k) *(bf16x8 *)(dst + k * 64 * HD) = w[k];
        }
#pragma unroll
        for (int c = 0; c < VU; ++c) {
            const int idx = tid + kThreads * c, p0 = 4 * (idx / (HD / 4)), d0 = 4 * (idx % (HD / 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const Parts2 x = split3(vr[c][0][e], vr[c][1][e]), y = split3(vr[c][2][e], vr[c][3][e]);
                uint16_t *dst = vt + (d0 + e) * LDV + vcol(d0 + e, p0);
                *(u32x2_t *)dst = u32x2_t{x.h, y.h};
                *(u32x2_t *)(dst + HD * LDV) = u32x2_t{x.m, y.m};
                *(u32x2_t *)(dst + 2 * HD * LDV) = u32x2_t{x.l, y.l};
            }
        }
    };
    const int last_tile = start + (end - 1 - start) / 64 * 64;
    fetch(start, page_of(start));
    if (tid == 0) *big_pos = INT32_MAX;

    // Q^T operands, pre-scaled by log2(e) / sqrt(HD) (scores in the exp2 domain).
    bf16x8 q3[KSTEPS][3];
    {
        const float sl2 = (1.0f / sqrtf((float)HD)) * 1.44269504088896340736f;
        const float *qp = a.q + (size_t)(rvalid ? row : 0) * a.q_stride + (size_t)(rvalid ? head : 0) * HD + 8 * half;
        const float sq = rvalid ? sl2 : 0.f;  // rows without a query: their scores are not used
        f32x4 raw[KSTEPS][2];  // every load before the first use: one round trip
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
            raw[s][0] = *(const f32x4 *)(qp + 16 * s);
            raw[s][1] = *(const f32x4 *)(qp + 16 * s + 4);
        }
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
            const float v[8] = {raw[s][0][0] * sq, raw[s][0][1] * sq, raw[s][0][2] * sq, raw[s][0][3] * sq,
                                raw[s][1][0] * sq, raw[s][1][1] * sq, raw[s][1][2] * sq, raw[s][1][3] * sq};
            split3x8(v, q3[s]);
        }
    }

    f32x16 oacc[UT], osum[FOLD ? UT : 1];
    float m2, l, msum = -INFINITY, lsum = 0.f;
    bool odd = false;  // a score of the row's is NaN
#pragma unroll
    for (int u = 0; u < UT; ++u) oacc[u] = f32x16{};
#pragma unroll
    for (int u = 0; u < (FOLD ? UT : 1); ++u) osum[u] = f32x16{};
    m2 = msum = -INFINITY;
    l = lsum = 0.f;
    int page_next = page_of(min(start + 64, last_tile));
    for (int t0 = start; t0 < end; t0 += 64) {
        __syncthreads();  // the previous tile's reads are done
        stage();
        __syncthreads();
        if (t0 + 64 < end) {
            fetch(t0 + 64, page_next);
            page_next = page_of(min(t0 + 128, last_tile));
        }
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            f32x16 sacc = f32x16{}, slow = f32x16{};
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) {
                const int r = 32 * tt + n;
                const uint16_t *kp = ks + r * HD + (((2 * s + half) ^ (r % CPR)) << 3);
                const bf16x8 k0 = *(const bf16x8 *)kp, k1 = *(const bf16x8 *)(kp + 64 * HD),
                             k2 = *(const bf16x8 *)(kp + 2 * 64 * HD);
                slow = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k2, q3[s][0], slow, 0, 0, 0);
                sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k0, q3[s][0], sacc, 0, 0, 0);
                slow = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k1, q3[s][1], slow, 0, 0, 0);
                slow = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k0, q3[s][2], slow, 0, 0, 0);
                slow = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k1, q3[s][0], slow, 0, 0, 0);
                slow = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k0, q3[s][1], slow, 0, 0, 0);
            }
            sacc += slow;
            // Masks, online softmax and delayed rescaling: attn_prefill_kernel's.
            const int h0 = t0 + 32 * tt;
            if (h0 + 31 > first_pos || h0 + 32 > end) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int p = h0 + krow_of(8 * (r >> 2) + 4 * half + (r & 3));
                    if (p > my_pos || p >= end) sacc[r] = -INFINITY;
                }
            }
            float tmax = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, sacc[r]);
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
            const bool raise = tmax > m2 + 8.0f;
            if (__any(raise)) {
                const float mnew = raise ? tmax : m2;
                const float alpha = raise ? __builtin_amdgcn_exp2f(m2 - mnew) : 1.f;  // 0 from -inf
                l *= alpha;
#pragma unroll
                for (int u = 0; u < UT; ++u)
#pragma unroll
                    for (int r = 0; r < 16; ++r) oacc[u][r] *= alpha;
                m2 = mnew;
            }
            const float mref = m2 == -INFINITY ? 0.f : m2;
            float tsum = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float pv = __builtin_amdgcn_exp2f(sacc[r] - mref);
                sacc[r] = pv;
                tsum += pv;
            }
            tsum += __shfl_xor(tsum, 32, 64);
            l += tsum;
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                float pv[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) pv[j] = sacc[8 * s2 + j];
                bf16x8 p3[3];
                split3x8(pv, p3);
#pragma unroll
                for (int u = 0; u < UT; ++u) {
                    const int d = 32 * u + n;
                    const uint16_t *vp = vt + d * LDV + vcol(d, 32 * tt + 16 * s2 + 8 * half);
                    const bf16x8 v0 = *(const bf16x8 *)vp, v1 = *(const bf16x8 *)(vp + HD * LDV),
                                 v2 = *(const bf16x8 *)(vp + 2 * HD * LDV);
                    oacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v2, p3[0], oacc[u], 0, 0, 0);
                    oacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v1, p3[1], oacc[u], 0, 0, 0);
                    oacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v0, p3[2], oacc[u], 0, 0, 0);
                    oacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v1, p3[0], oacc[u], 0, 0, 0);
                    oacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v0, p3[1], oacc[u], 0, 0, 0);
                    oacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v0, p3[0], oacc[u], 0, 0, 0);
                }
            }
        }
        if constexpr (FOLD) {
            if ((t0 + 64) % sub == 0 || t0 + 64 >= end) {
                // A part without a key of the row may hold NaN (its -inf maximum
                // rescaled with its neighbours'): left out, as the merge does.
                const bool any = m2 != -INFINITY;
                odd |= l != l && my_pos >= t0 / sub * sub;
                float alpha, beta;
                fold_factors(m2, msum, alpha, beta);
                lsum = any ? fold_value(lsum, l, alpha, beta) : lsum;
#pragma unroll
                for (int u = 0; u < UT; ++u) {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        osum[u][r] = any ? fold_value(osum[u][r], oacc[u][r], alpha, beta) : osum[u][r];
                    oacc[u] = f32x16{};
                }
                m2 = -INFINITY;
                l = 0.f;
            }
        }
    }
    // The parts of an infinite operand, or of a product past the largest
    // number, add up to NaN where the f32 product is an infinity (a score of
    // -inf weighs nothing). The rows with a NaN score, or with a V value of kBigV
    // or more in sight, are computed again in plain f32, over their own keys.
    if constexpr (!FOLD) odd = l != l;
    odd = odd && my_pos >= start;
    if (__syncthreads_or(top >= kBigV)) {
        for (int e = tid; e < (end - start) * HD; e += kThreads) {
            const int p = start + e / HD;
            const float v = vbase[(((size_t)page_of(p) * a.kv_heads + g) * a.page_size + p % a.page_size) * HD + e % HD];
            if (!(fabsf(v) < kBigV)) atomicMin(big_pos, p);
        }
        __syncthreads();
        odd = odd || *big_pos <= my_pos;
    }
    if (rvalid && odd) {
        plain_row<HD>(a, row, head, g, half, start, min(end, my_pos + 1), FOLD ? sub : span, part, S);
        return;
    }
    if (!rvalid) return;
    const size_t ob = (size_t)row * a.q_heads * HD + (size_t)head * HD;
    if constexpr (FOLD) store_prefill_rows<HD>(a, osum, msum, lsum, part, ob, S, half);
    else store_prefill_rows<HD>(a, oacc, m2, l, part, ob, S, half);
}

// Merges the splits of one (row, q head) of attn_prefill_kernel in split
// order, one wave per (row, head): maxima in the log2 domain, weights
// 2^(m_s - M), output (sum_s w_s o_s) * (1 / sum_s w_s l_s). A row whose only
// non-empty split gives w = 1 gets o * (1 / l), the bits the one-split
// kernel writes.
template <int HD>
__global__ __launch_bounds__(kThreads) void attn_merge2_kernel(const float *part, int S, int q_heads, int items,
                                                              float *out, uint16_t *out_hi, uint16_t *out_lo) {
    const int lane = threadIdx.x & 63;
    const int item = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    if (item >= items) return;
    const float *p = part + (size_t)item * (size_t)S * (HD + 2);
    static_assert(kMaxSplits <= 128, "a lane holds two splits");
    const int s1 = lane + 64;
    const float m0 = lane < S ? p[(size_t)lane * (HD + 2) + HD] : -INFINITY;
    float m1 = -INFINITY, w1 = 0.f;
    if (S > 64 && s1 < S) m1 = p[(size_t)s1 * (HD + 2) + HD];
    const float M = wave_max(fmaxf(m0, m1));
    const float w0 = m0 == -INFINITY ? 0.f : exp2f(m0 - M);
    float L = wave_sum(w0 != 0.f ? w0 * p[(size_t)lane * (HD + 2) + HD + 1] : 0.f);
    if (S > 64) {
        w1 = m1 == -INFINITY ? 0.f : exp2f(m1 - M);
        L += wave_sum(w1 != 0.f ? w1 * p[(size_t)s1 * (HD + 2) + HD + 1] : 0.f);
    }
    const float inv = 1.0f / L;
    constexpr int DPL = HD / 64;  // dims per lane
    float o[DPL];
#pragma unroll
    for (int k = 0; k < DPL; ++k) o[k] = 0.f;
    auto fold = [&](float ws, int s) {
        if (ws != 0.f) {
#pragma unroll
            for (int k = 0; k < DPL; ++k) o[k] = fmaf(ws, p[(size_t)s * (HD + 2) + lane + 64 * k], o[k]);
        }
    };
    for (int s = 0; s < min(S, 64); ++s) fold(__shfl(w0, s, 64), s);
    for (int s = 64; s < S; ++s) fold(__shfl(w1, s - 64, 64), s);
#pragma unroll
    for (int k = 0; k < DPL; ++k) {
        const size_t i = (size_t)item * HD + lane + 64 * k;
        const float v = o[k] * inv;
        if (out) out[i] = v;
        if (out_hi) {
            const __bf16 hb = (__bf16)v;
            out_hi[i] = __builtin_bit_cast(uint16_t, hb);
            out_lo[i] = __builtin_bit_cast(uint16_t, (__bf16)(v - (float)hb));
        }
    }
}

template <int HD>
int launch_merge2(const AttnJob &j, const AttnArgs &a, int S, hipStream_t s) {
    if (S <= 1) return 0;
    const int items = (int)j.rows * j.q_heads;
    hipLaunchKernelGGL((attn_merge2_kernel<HD>), dim3((items + 3) / 4), dim3(kThreads), 0, s, a.part, S, j.q_heads,
                       items, a.out, a.out_hi, a.out_lo);
    CHIP_CHECK(hipGetLastError());
    return 0;
}

// Most parts of attn_merge_parts_kernel (their factors sit in LDS).
constexpr int kMaxParts = 256;

// Merges the parts of one (row, q head) of an f32 prefill, one wave per (row,
// head): the `per` parts of each split folded in order, as the FOLD kernel
// does, then the splits as attn_merge2_kernel does (one lane per split): the
// bits of the FOLD kernel and attn_merge2_kernel.
template <int HD>
__global__ __launch_bounds__(kThreads) void attn_merge_parts_kernel(const float *part, int parts, int per, int q_heads,
                                                                   int items, float *out, uint16_t *out_hi,
                                                                   uint16_t *out_lo) {
    __shared__ float2 s_f[kThreads / 64][kMaxParts];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int item = blockIdx.x * (kThreads / 64) + wave;
    if (item >= items) return;
    const float *p = part + (size_t)item * (size_t)parts * (HD + 2);
    const int S = (parts + per - 1) / per;
    // Lane g: the maximum and the weight sum of split g, its parts' factors.
    float m = -INFINITY, l = 0.f;
    if (lane < S) {
        for (int i = lane * per; i < min(lane * per + per, parts); ++i) {
            const float mi = p[(size_t)i * (HD + 2) + HD];
            const float li = mi == -INFINITY ? 0.f : p[(size_t)i * (HD + 2) + HD + 1];
            float alpha, beta;
            fold_factors(mi, m, alpha, beta);
            l = fold_value(l, li, alpha, beta);
            s_f[wave][i] = make_float2(alpha, mi == -INFINITY ? -1.f : beta);  // -1: the part holds no values
        }
    }
    // The factors are read by the whole wave: its LDS operations run in order.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const float M = wave_max(m);
    const float w = m == -INFINITY ? 0.f : exp2f(m - M);
    const float L = wave_sum(w != 0.f ? w * l : 0.f);
    const float inv = 1.0f / L;
    constexpr int DPL = HD / 64, BATCH = 16;  // dims per lane; parts loaded per round trip
    float o[DPL], t[DPL];
#pragma unroll
    for (int k = 0; k < DPL; ++k) o[k] = t[k] = 0.f;
    for (int i0 = 0; i0 < parts; i0 += BATCH) {
        float v[BATCH][DPL];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int q = min(i0 + i, parts - 1);
#pragma unroll
            for (int k = 0; k < DPL; ++k) v[i][k] = p[(size_t)q * (HD + 2) + lane + 64 * k];
        }
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int q = i0 + i;
            if (q < parts) {
                const float2 f = s_f[wave][q];
#pragma unroll
                for (int k = 0; k < DPL; ++k)
                    t[k] = f.y < 0.f ? t[k] : fold_value(t[k], v[i][k], f.x, f.y);
                if ((q + 1) % per == 0 || q + 1 == parts) {
                    const float ws = __shfl(w, q / per, 64);
#pragma unroll
                    for (int k = 0; k < DPL; ++k) {
                        if (ws != 0.f) o[k] = fmaf(ws, t[k], o[k]);
                        t[k] = 0.f;
                    }
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < DPL; ++k) {
        const size_t i = (size_t)item * HD + lane + 64 * k;
        const float r = o[k] * inv;
        if (out) out[i] = r;
        if (out_hi) {
            const __bf16 hb = (__bf16)r;
            out_hi[i] = __builtin_bit_cast(uint16_t, hb);
            out_lo[i] = __builtin_bit_cast(uint16_t, (__bf16)(r - (float)hb));
        }
    }
}

template <int HD, int G, bool FOLD>
int launch_prefill_f32_blocks(const AttnArgs &a, int kv_heads, size_t rows, int S, int span, hipStream_t s) {
    constexpr size_t lds = prefill_f32_lds_bytes<HD>();
    constexpr int RB = 4 * (32 / G);  // rows of a block
    static std::atomic<uint64_t> lds_set{0};
    CHIP_TRY(allow_dynamic_lds((const void *)attn_prefill_f32_kernel<HD, G, FOLD>, lds, lds_set));
    hipLaunchKernelGGL((attn_prefill_f32_kernel<HD, G, FOLD>), dim3((unsigned)((rows + RB - 1) / RB), kv_heads, S),
                       dim3(kThreads), lds, s, a, (int)rows, S, span, kF32PrefillSpan);
    CHIP_CHECK(hipGetLastError());
    return 0;
}

// Prefill over an f32 cache: a row's keys are cut into parts of
// kF32PrefillSpan keys, and into splits of j.span keys (a multiple); a split's
// parts are folded in order, then the splits merged. Which blocks do it does
// not change the bits: one block a split (its parts folded in registers), or
// one a part (attn_merge_parts_kernel folds them), as many rows at a time as
// the scratch holds the parts of. The second is for calls whose splits would
// leave most of the chip idle while each block walks a long one: with splits
// of 8,192 keys (a 64K cache), position 16,000, two Q4 layers with 32 q / 8 KV
// heads of 128, 2 rows take 2,150 us a forward by split and 630 by part, 512
// rows 3,120 and 4,090. The estimate: 7.5 us (3.2 at head_dim 64) for 64 keys
// of a block and for a part's start; by split the longest block or all of them
// over the CUs, by part rounds of blocks, a merge and its values' write and
// read at 4.5 TB/s.
template <int HD, int G>
int launch_prefill_f32(const AttnJob &j, const AttnArgs &a, int S, hipStream_t s) {
    constexpr size_t RB = 4 * (32 / G), sub = kF32PrefillSpan;
    const int kvh = j.g.kv_heads;
    const size_t ctx = j.offset + j.rows, cus = (size_t)std::max(device_cus(), 1);
    const size_t parts = (size_t)attention_prefill_splits(ctx, (int)sub);
    if (j.span % sub || j.span <= (int)sub || parts == 1) {  // nothing to fold
        CHIP_TRY((launch_prefill_f32_blocks<HD, G, false>(a, kvh, j.rows, S, j.span, s)));
        return launch_merge2<HD>(j, a, S, s);
    }
    const size_t row_floats = attention_part_floats(1, j.q_heads, (int)parts, HD);
    const size_t fit = j.part ? std::min(j.part_floats / row_floats / RB * RB, (j.rows + RB - 1) / RB * RB) : 0;
    if (parts <= (size_t)kMaxParts && S <= 64 && fit > 0) {  // a wave of the merge holds a split per lane
        constexpr float tile = HD == 64 ? 3.2f : 7.5f;
        auto blocks = [&](size_t rows) { return (rows + RB - 1) / RB * (size_t)kvh; };  // of a split or part
        const size_t launches = (j.rows + fit - 1) / fit, tiles = (ctx + 63) / 64;
        const float by_split =
            tile * (float)std::max(std::min(tiles, (size_t)j.span / 64), (blocks(j.rows) * tiles + cus - 1) / cus);
        const float by_part =
            (float)launches * (tile * (float)((blocks(fit) * parts + cus - 1) / cus * (sub / 64 + 1)) + 6.f) +
            8.f * (float)(j.rows * row_floats) / 4.5e6f;
        if (by_part < by_split) {
            for (size_t r = 0; r < j.rows; r += fit) {
                const size_t n = std::min(fit, j.rows - r), o = r * (size_t)j.q_heads * HD;
                const int np = attention_prefill_splits(j.offset + r + n, (int)sub);
                AttnArgs b = a;
                b.q = a.q + r * j.q_stride;
                b.offset = a.offset + (long)r;
                if (b.out) b.out += o;
                if (b.out_hi) b.out_hi += o, b.out_lo += o;
                CHIP_TRY((launch_prefill_f32_blocks<HD, G, false>(b, kvh, n, np, (int)sub, s)));
                if (np == 1) continue;  // one part: written as the output
                const int items = (int)n * j.q_heads;
                hipLaunchKernelGGL((attn_merge_parts_kernel<HD>), dim3((items + 3) / 4), dim3(kThreads), 0, s, b.part,
                                   np, j.span / (int)sub, j.q_heads, items, b.out, b.out_hi, b.out_lo);
                CHIP_CHECK(hipGetLastError());
            }
            return 0;
        }
    }
    CHIP_TRY((launch_prefill_f32_blocks<HD, G, true>(a, kvh, j.rows, S, j.span, s)));
    return launch_merge2<HD>(j, a, S, s);
}

template <int HD, int G>
int launch_prefill_hg(const AttnJob &j, const AttnArgs &a, int S, hipStream_t s) {
    if (j.g.kv_f32) return launch_prefill_f32<HD, G>(j, a, S, s);
    constexpr int RW = 32 / G;
    constexpr size_t lds = (size_t)4 * 64 * HD * 2;
    const int rb = (int)((j.rows + 4 * RW - 1) / (4 * RW));
    static std::atomic<uint64_t> lds_set{0};
    CHIP_TRY(allow_dynamic_lds((const void *)attn_prefill_kernel<HD, G>, lds, lds_set));
    hipLaunchKernelGGL((attn_prefill_kernel<HD, G>), dim3(rb, j.g.kv_heads, S), dim3(kThreads), lds, s, a, (int)j.rows,
                       S, j.span);
    CHIP_CHECK(hipGetLastError());
    return launch_merge2<HD>(j, a, S, s);
}

template <int HD>
int launch_prefill_h(const AttnJob &j, const AttnArgs &a, int G, int S, hipStream_t s) {
    switch (G) {
        case 1: return launch_prefill_hg<HD, 1>(j, a, S, s);
        case 2: return launch_prefill_hg<HD, 2>(j, a, S, s);
        case 3: return launch_prefill_hg<HD, 3>(j, a, S, s);
        case 4: return launch_prefill_hg<HD, 4>(j, a, S, s);
        case 5: return launch_prefill_hg<HD, 5>(j, a, S, s);
        case 6: return launch_prefill_hg<HD, 6>(j, a, S, s);
        case 7: return launch_prefill_hg<HD, 7>(j, a, S, s);
        case 8: return launch_prefill_hg<HD, 8>(j, a, S, s);
    }
    return fail("HIP backend: attention supports 1..8 query heads per KV head.");
}

// Decode attention: BF16 K/V on the matrix cores, f32 K/V on the vector
// ALUs.
template <int HD, int G, class KT>
int launch_hgk(const AttnJob &j, const AttnArgs &a, hipStream_t s) {
    const dim3 grid(j.splits, j.g.kv_heads);
    constexpr bool mfma = std::is_same<KT, uint16_t>::value;
    const bool rope = a.qkv != nullptr;
    if (rope && !mfma) return fail("HIP backend: fused RoPE needs the matrix-core attention kernel.");
    if (j.splits == 1) {
        if constexpr (mfma) {
            if (rope) hipLaunchKernelGGL((attn_dec_mfma_kernel<HD, G, true, true>), grid, dim3(kThreads), 0, s, a);
            else hipLaunchKernelGGL((attn_dec_mfma_kernel<HD, G, true, false>), grid, dim3(kThreads), 0, s, a);
        } else {
            hipLaunchKernelGGL((attn_kernel<HD, G, KT, true>), grid, dim3(kThreads), 0, s, a);
        }
        CHIP_CHECK(hipGetLastError());
        return 0;
    }
    if constexpr (mfma) {
        if (rope) hipLaunchKernelGGL((attn_dec_mfma_kernel<HD, G, false, true>), grid, dim3(kThreads), 0, s, a);
        else hipLaunchKernelGGL((attn_dec_mfma_kernel<HD, G, false, false>), grid, dim3(kThreads), 0, s, a);
    } else {
        hipLaunchKernelGGL((attn_kernel<HD, G, KT, false>), grid, dim3(kThreads), 0, s, a);
    }
    CHIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL((attn_combine_kernel<HD>), dim3(j.q_heads), dim3(kThreads), 0, s, a.part, j.splits, a.out);
    CHIP_CHECK(hipGetLastError());
    return 0;
}

template <int HD, int G>
int launch_hg(const AttnJob &j, const AttnArgs &a, hipStream_t s) {
    if (j.g.kv_f32) return launch_hgk<HD, G, float>(j, a, s);
    return launch_hgk<HD, G, uint16_t>(j, a, s);
}

template <int HD>
int launch_h(const AttnJob &j, const AttnArgs &a, int G, hipStream_t s) {
    switch (G) {
        case 1: return launch_hg<HD, 1>(j, a, s);
        case 2: return launch_hg<HD, 2>(j, a, s);
        case 3: return launch_hg<HD, 3>(j, a, s);
        case 4: return launch_hg<HD, 4>(j, a, s);
        case 5: return launch_hg<HD, 5>(j, a, s);
        case 6: return launch_hg<HD, 6>(j, a, s);
        case 7: return launch_hg<HD, 7>(j, a, s);
        case 8: return launch_hg<HD, 8>(j, a, s);
    }
    return fail("HIP backend: attention supports 1..8 query heads per KV head.");
}

}  // namespace

size_t attention_part_floats(size_t rows, int q_heads, int splits, int head_dim) {
    return rows * (size_t)q_heads * (size_t)splits * (size_t)(head_dim + 2);
}

int attention_max_splits() { return kMaxSplits; }

// Split-K of a decode-style launch: across the KV heads and rows about one
// block per CU for the matrix-core kernel (BF16 K/V; measured 13 % faster
// than two at 16K keys, where the K/V stream, not the block count, sets the
// time) and two for the VALU kernel (f32 K/V), at most one split per
// 64-position tile and kMaxSplits. A short BF16 context takes one block per
// KV head, which needs no merge launch: up to 256 positions at head_dim 128
// (32 q / 8 KV heads, split -> one block: 128 keys 7.9 -> 6.2 us, 256 7.9 ->
// 6.8, 320 7.9 -> 8.0) and 384 at 64 (14 / 2 heads: 128 6.9 -> 5.2, 384 7.1 ->
// 6.8, 512 7.2 -> 7.5). One block of 8 or 16 waves was slower from 200 keys on
// (512 keys, 14 / 2 heads of 64: 9.4 us).
int attention_decode_splits(size_t ctx, int kv_heads, size_t rows, bool kv_f32, int head_dim) {
    if (!kv_f32 && rows == 1 && ctx <= (head_dim == 64 ? 384u : 256u)) return 1;
    const size_t per_cu = kv_f32 ? 2 : 1;
    const size_t target = per_cu * (size_t)std::max(device_cus(), 1);
    const size_t per = (size_t)std::max(kv_heads, 1) * std::max<size_t>(rows, 1);
    size_t s = (target + per - 1) / per;
    s = std::min({s, (ctx + TP - 1) / TP, (size_t)kMaxSplits});
    return (int)std::max<size_t>(s, 1);
}

int attention_prefill_splits(size_t ctx, int span) {
    return (int)std::max<size_t>(1, (ctx + (size_t)span - 1) / (size_t)span);
}

// Longer spans mean fewer splits to merge per row and fewer, larger blocks:
// measured on 1,024-row chunks at up to 32K keys (Qwen2-7B turn 1 / turn 2
// prefill) 19,130 / 14,155 tok/s with 1,024, 20,418 / 15,737 with 4,096;
// on 512-row chunks at up to 8K keys (Llama-3-8B) 20,766 tok/s with 1,024,
// 19,178 with 4,096. Capacity / 8 picks 4,096 for the 33K cache and 1,024
// for the 8K one. The f32 kernel runs one block per CU and a tile takes it
// about three times as long, so short caches take spans from 256 on (longer
// ones run part by part where that is faster, launch_prefill_f32).
int attention_prefill_span(size_t kv_capacity, bool kv_f32) {
    int span = kv_f32 ? kF32PrefillSpan : kDefaultPrefillSpan;
    while ((size_t)span * 2 <= kv_capacity / 8 && span < (1 << 20)) span *= 2;
    return span;
}

bool attention_decode_fuses_rope(const KvGeom &g, int q_heads, int rotary_dim) {
    return !g.kv_f32 && (g.head_dim == 64 || g.head_dim == 128) && g.kv_heads > 0 &&
           q_heads % g.kv_heads == 0 && q_heads / g.kv_heads <= 8 && rotary_dim == g.head_dim;
}

int launch_attention(const AttnJob &j, hipStream_t s) {
    if (j.rows == 0) return 0;
    const bool halves_only = j.prefill && j.out_hi;
    if ((!j.q && !j.qkv) || (!j.out && !halves_only) || !j.k || !j.v || !j.g.page_table || (!j.prefill && j.splits > 1 && !j.part))
        return fail("HIP backend: attention is missing a buffer.");
    if (j.g.kv_heads <= 0 || j.q_heads <= 0 || j.q_heads % j.g.kv_heads)
        return fail("HIP backend: q_heads must be a multiple of kv_heads.");
    if (j.g.page_size <= 0 || j.g.page_size % TP)
        return fail("HIP backend: the KV page size must be a multiple of 64 positions.");
    if (j.splits <= 0 || j.splits > kMaxSplits || j.rows > 65535 || j.q_heads > 65535)
        return fail("HIP backend: attention grid out of range.");
    AttnArgs a{};
    a.q = j.q;
    a.q_stride = (long)j.q_stride;
    a.k = j.k;
    a.v = j.v;
    a.page_table = j.g.page_table;
    a.page_size = j.g.page_size;
    a.kv_heads = j.g.kv_heads;
    a.q_heads = j.q_heads;
    a.offset = (long)j.offset;
    a.pos_dev = j.pos_dev;
    a.part = j.part;
    a.out = j.out;
    if (j.qkv) {
        if (j.prefill || j.rows != 1 || !attention_decode_fuses_rope(j.g, j.q_heads, j.rotary_dim) || !j.rope_cos ||
            !j.rope_sin)
            return fail("HIP backend: fused RoPE attention takes one BF16 decode row with full-width rotary.");
        a.qkv = j.qkv;
        a.rope_cos = j.rope_cos;
        a.rope_sin = j.rope_sin;
        a.rotary_dim = j.rotary_dim;
    }
    const int G = j.q_heads / j.g.kv_heads;
    if (j.g.head_dim != 64 && j.g.head_dim != 128) return fail("HIP backend: attention supports head_dim 64 and 128.");
    if (G > 8) return fail("HIP backend: attention supports 1..8 query heads per KV head.");
    if (!j.prefill && j.rows != 1) return fail("HIP backend: decode attention takes one row.");
    if (j.prefill) {
        if (j.pos_dev) return fail("HIP backend: prefill attention takes a host position.");
        if (j.offset + j.rows > (size_t)INT32_MAX) return fail("HIP backend: prefill position out of range.");
        if (j.span < 64 || j.span % 64) return fail("HIP backend: prefill span must be a positive multiple of 64.");
        const int S = attention_prefill_splits(j.offset + j.rows, j.span);
        if (S > kMaxSplits) return fail("HIP backend: prefill context exceeds the attention split limit.");
        if (S > 1 && (!j.part || j.part_floats < attention_part_floats(j.rows, j.q_heads, S, j.g.head_dim)))
            return fail("HIP backend: prefill attention partial buffer too small.");
        if (!j.out_hi != !j.out_lo || ((uintptr_t)j.out_hi % 8) || ((uintptr_t)j.out_lo % 8))
            return fail("HIP backend: prefill attention halves need both 8-byte aligned buffers.");
        a.out_hi = j.out_hi;
        a.out_lo = j.out_lo;
        if (j.g.head_dim == 64) return launch_prefill_h<64>(j, a, G, S, s);
        return launch_prefill_h<128>(j, a, G, S, s);
    }
    if (j.g.head_dim == 64) return launch_h<64>(j, a, G, s);
    return launch_h<128>(j, a, G, s);
}

}  // namespace chip
