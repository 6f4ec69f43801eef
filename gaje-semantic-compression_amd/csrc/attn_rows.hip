// Causal GQA attention of several consecutive tokens of one sequence (a prompt's
// rows), bit for bit the decode attention of each token
// (GenomicAttention::forward_attention_core, src/nn/attention.rs:87-127):
//   s_t = dot_product(q, k_t) * (1/sqrt(hd))   eight FMA chains (dot.rs:43-67),
//         ((a0+a4)+(a1+a5)) + ((a2+a6)+(a3+a7)), one rounded multiply;
//   e_t = expf(s_t - max), sum = e_0 + e_1 + ... serially, inv = 1 / (sum + 1e-12);
//   out_i = sum over t of (e_t * inv) * v_t[i] in t order, every operation rounded.
//
// One workgroup per (query head, tile of at most 16 tokens).  Against one
// workgroup per (head, token) it reads the keys and values once for 16 queries and
// runs the dots and the products on the f32 matrix cores:
// - Scores: v_mfma_f32_16x16x1_4b, one k step, rounds like fmaf, so block b of two
//   instructions runs chains b and 4 + b of 16 positions x 16 queries, hd / 8 steps.
// - Products: the same instruction with C = 0 is round(w * v) (the sums never see
//   the sign of a zero product: they start at +0), four positions per instruction;
//   the serial sums then take one v_add_f32 per product, in t order.
// The exponentials sit in LDS, a row of positions per query, rows 4 banks apart;
// each query's serial sum runs in its own lane (chain_lds).  Positions past a
// query's own are dropped where they appear (score masked, exponential +0, product
// +0), and adding +0 to a sum that started at +0 changes no bit.
//
// Bound by the serial parts: about 6 cycles per position for the softmax sum and 26
// per position and wave for the products and sums.  201 tokens x 14 heads of 64:
// 13.9 us per layer, 64.8 with one workgroup per (head, token).
#include <hip/hip_runtime.h>

#include "common.h"
#include "device_util.h"
#include "kernels.h"

namespace gaje {
namespace {

typedef float vf16 __attribute__((ext_vector_type(16)));

constexpr int AR_TQ = 16;  // queries per tile (ATTN_ROWS_TILE)
// LDS floats of a query's row for positions 0..ctx-1 (whole 64-value chunks for
// chain_lds, rows 4 banks apart), and of the workgroup (chain_lds reads 32 past).
__host__ __device__ constexpr int64_t ar_len(int64_t ctx) { return (ctx + 63) / 64 * 64; }
__host__ __device__ constexpr int64_t ar_floats(int64_t ctx) { return AR_TQ * (ar_len(ctx) + 4) + 32; }

template <int HD>
__global__ __launch_bounds__(HD * 4) void attn_rows_kernel(AttnParams p) {
    constexpr int NW = HD / 16, NC = HD / 8;  // waves (one per 16 output dimensions), steps of a chain
    extern __shared__ __align__(16) float sc[];  // [AR_TQ][LD]: scores, then exponentials
    __shared__ float red[NW][AR_TQ];
    __shared__ float inv_q[AR_TQ];
    __shared__ uint64_t tab[32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = blockIdx.x % p.n_head, tile = p.n_tiles - 1 - blockIdx.x / p.n_head;  // the longest contexts first
    const int row0 = p.tiles[2 * tile], nq = p.tiles[2 * tile + 1];
    const int pos0 = p.seq_pos[row0], ctx = pos0 + nq;  // query i: positions 0..pos0 + i
    const int64_t kvz = p.row_seq ? p.row_seq[row0] : 0;  // (row_seq null: one cache)
    const int g = h / (p.n_head / p.n_head_kv);
    const float *Kh = p.k_cache + kvz * p.seq_kv_stride + (size_t)g * p.kv_head_stride;
    const float *Vh = p.v_cache + kvz * p.seq_kv_stride + (size_t)g * p.kv_head_stride;
    const int64_t cap = p.kv_cap;
    const int n = (int)ar_len(ctx), LD = n + 4, nkt = (ctx + 15) >> 4;
    const int c16 = lane & 15, g4 = lane >> 4;
    const float scale = 1.0f / sqrtf((float)HD);
    if (tid < 32) tab[tid] = kExp2Tab[tid];

    // ---- scores: tiles of 16 positions, wave w takes tiles w, w + NW, .. ----
    {
        const float *q = p.q + (size_t)(row0 + min(c16, nq - 1)) * p.seq_q_stride + (size_t)h * HD;
        float qb[2][NC];  // B: query c16, chain 4 hh + g4, step c
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) qb[hh][c] = q[8 * c + 4 * hh + g4];
        // A: position 16 kt + c16 (the caches hold whole tiles of 16), the same chain and step
        auto keys = [&](float (&k)[2][NC], int kt) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) k[hh][c] = Kh[(size_t)(8 * c + 4 * hh + g4) * cap + 16 * kt + c16];
        };
        float ka[2][NC], kb[2][NC], mx = -INFINITY;
        auto score = [&](const float (&k)[2][NC], int kt) {
            vf16 a0 = {}, a1 = {};
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                a0 = __builtin_amdgcn_mfma_f32_16x16x1f32(k[0][c], qb[0][c], a0, 0, 0, 0);
                a1 = __builtin_amdgcn_mfma_f32_16x16x1f32(k[1][c], qb[1][c], a1, 0, 0, 0);
            }
            // register 4 b + r: chain b (a1: 4 + b), position 4 g4 + r, query c16
            float s[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float u0 = a0[r] + a1[r], u1 = a0[4 + r] + a1[4 + r];
                const float u2 = a0[8 + r] + a1[8 + r], u3 = a0[12 + r] + a1[12 + r];
                s[r] = ((u0 + u1) + (u2 + u3)) * scale;
                if (16 * kt + 4 * g4 + r <= pos0 + c16) mx = fmaxf(mx, s[r]);
            }
            *(float4 *)(sc + c16 * LD + 16 * kt + 4 * g4) = make_float4(s[0], s[1], s[2], s[3]);
        };
        if (wave < nkt) keys(ka, wave);
        for (int kt = wave; kt < nkt; kt += 2 * NW) {
            if (kt + NW < nkt) keys(kb, kt + NW);
            score(ka, kt);
            if (kt + NW >= nkt) break;
            if (kt + 2 * NW < nkt) keys(ka, kt + 2 * NW);
            score(kb, kt + NW);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
        if (lane < AR_TQ) red[wave][lane] = mx;
    }
    __syncthreads();
    // ---- exponentials, +0 past each query's positions ----
    for (int i = wave; i < AR_TQ; i += NW) {
        float mq = red[0][i];
#pragma unroll
        for (int w = 1; w < NW; ++w) mq = fmaxf(mq, red[w][i]);
        const int end = i < nq ? pos0 + i + 1 : 0;  // rows past the tile's last stay +0
        for (int t = 4 * lane; t < n; t += 4 * WAVE) {
            float4 e = *(const float4 *)(sc + i * LD + t);
            e.x = t < end ? expf_ref_t(e.x - mq, tab) : 0.0f;
            e.y = t + 1 < end ? expf_ref_t(e.y - mq, tab) : 0.0f;
            e.z = t + 2 < end ? expf_ref_t(e.z - mq, tab) : 0.0f;
            e.w = t + 3 < end ? expf_ref_t(e.w - mq, tab) : 0.0f;
            *(float4 *)(sc + i * LD + t) = e;
        }
    }
    // ---- output: wave w's 16 dimensions; AH tiles of values in flight ----
    const float *vr = Vh + (size_t)(16 * wave + c16) * cap + 4 * g4;
    constexpr int AH = HD == 64 ? 4 : 2;  // (four spill at 128)
    vf4 v[AH];
#pragma unroll
    for (int u = 0; u < AH; ++u) v[u] = *(const vf4 *)(vr + 16 * min(u, nkt - 1));
    __syncthreads();
    if (wave == 0 && lane < AR_TQ) inv_q[lane] = 1.0f / (chain_lds(0.0f, sc + lane * LD, n) + 1e-12f);
    __syncthreads();
    const float inv = inv_q[c16];
    float acc[4] = {0.f, 0.f, 0.f, 0.f};  // query 4 g4 + r, dimension 16 wave + c16
    auto tile16 = [&](int kt, const vf4 &vv, auto masked) {
        const vf4 e = *(const vf4 *)(sc + c16 * LD + 16 * kt + 4 * g4);
        vf16 d[4];
        const vf16 zero = {};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // A: w of query c16, B: v of dimension c16, both at position 16 kt + 4 g4 + j;
            // register 4 b + r: position 16 kt + 4 b + j, query 4 g4 + r, dimension c16
            const float w = e[j] * inv;
            d[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(w, vv[j], zero, 0, 0, 0);
        }
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool in = !decltype(masked)::value || 16 * kt + 4 * b + j <= pos0 + 4 * g4 + r;
                    acc[r] = acc[r] + (in ? d[j][4 * b + r] : 0.0f);
                }
    };
    const int full = (pos0 + 1) >> 4;  // tiles that every query attends to
    int kt = 0;
    for (; kt + AH <= full; kt += AH)
#pragma unroll
        for (int u = 0; u < AH; ++u) {
            const vf4 vv = v[u];
            v[u] = *(const vf4 *)(vr + 16 * min(kt + u + AH, nkt - 1));
            tile16(kt + u, vv, std::false_type{});
        }
    for (; kt < nkt; kt += AH)
#pragma unroll
        for (int u = 0; u < AH; ++u) {
            if (kt + u >= nkt) continue;
            const vf4 vv = v[u];
            v[u] = *(const vf4 *)(vr + 16 * min(kt + u + AH, nkt - 1));
            if (kt + u < full) tile16(kt + u, vv, std::false_type{});
            else tile16(kt + u, vv, std::true_type{});
        }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (4 * g4 + r < nq) p.out[(size_t)(row0 + 4 * g4 + r) * p.seq_q_stride + (size_t)h * HD + 16 * wave + c16] = acc[r];
}

}  // namespace

static bool attn_rows_fits(int head_dim, int64_t kv_cap, int64_t ctx) {
    return (head_dim == 64 || head_dim == 128) && kv_cap % 16 == 0 && (size_t)ar_floats(ctx) * 4 + 2048 <= max_lds_per_block();
}

// Against one workgroup per (head, row), which costs by the round of workgroups, a
// tile costs a longer serial pass whatever its rows: it takes about two rounds, three
// at 64 dimensions over a long context, to pay.  Prompts of n tokens over a cache, us
// (8 layers), tiles against rows: 12 heads of 128: 32 tokens at 1024 1358 / 1264, 48
// 1552 / 1623; 14 of 64: 32 at 1024 1001 / 830, 48 1087 / 1041, 64 1127 / 1209, 48 at 0
// 723 / 767; 9 of 64: 2 at 2200 1124 / 649, 64 1336 / 1186, 96 1380 / 1453.
bool attn_rows_serves(int head_dim, int n_head, int64_t kv_cap, int64_t ctx, int64_t rows) {
    const int64_t rounds = ctx <= 64 ? 1 : head_dim == 128 || ctx <= 256 ? 2 : 3;
    return rows * n_head >= rounds * device_cu_count() && attn_rows_fits(head_dim, kv_cap, ctx);
}

int launch_attn_rows(const AttnParams &p, hipStream_t s) {
    if (!p.q || !p.k_cache || !p.v_cache || !p.out || !p.seq_pos || !p.tiles || p.n_tiles <= 0 || p.n_head <= 0 ||
        p.n_head_kv <= 0 || p.n_head % p.n_head_kv || p.kv_cap <= 0 || p.kv_head_stride != p.kv_cap * p.head_dim ||
        p.ctx <= 0 || p.ctx > p.kv_cap || !attn_rows_fits(p.head_dim, p.kv_cap, p.ctx) ||
        (((uintptr_t)p.k_cache | (uintptr_t)p.v_cache) & 15) || p.seq_kv_stride % 4 ||
        (int64_t)p.n_tiles * p.n_head > INT32_MAX)
        return set_error(GAJE_ERR_INVALID_ARG, "attention rows: bad arguments");
    const dim3 grid((unsigned)(p.n_tiles * p.n_head));
    const size_t lds = (size_t)ar_floats(p.ctx) * 4;
    if (p.head_dim == 64) hipLaunchKernelGGL(attn_rows_kernel<64>, grid, dim3(256), lds, s, p);
    else hipLaunchKernelGGL(attn_rows_kernel<128>, grid, dim3(512), lds, s, p);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

}  // namespace gaje
