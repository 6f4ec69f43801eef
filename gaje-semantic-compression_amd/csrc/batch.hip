// Rows of several sequences or of a prompt, as if as many GenomicLLM instances
// (llm/forward.rs:7-64) stepped over shared weights: the passes per row (norms, SwiGLU,
// the steps' begin and end, argmax) and the batch's f32 lm_head.  Every product and
// reduction follows the batch-1 decode kernels' order, so each row's values are
// bit-identical to its own forward_core.  (The Q4_0 products are launch_q4_rows, where
// the 4, 16 or 32 activation rows of a tile share each dequantised weight.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "device_util.h"
#include "kernels.h"

namespace gaje {
namespace {

__device__ __forceinline__ void seq_flag(uint32_t *codes, int s, int layer, int stage) {
    if (codes && stage >= 0) atomicMin(&codes[s], (uint32_t)(layer * 8 + stage));
}

// F32 rows in the tiled layout x NV vectors (dot_product, dot.rs:23-94, per
// vector): lanes 2r, 2r+1 of a wave own row r of the wave's 32-row tile,
// chains 0..3 and 4..7; each chunk of the tile is one coalesced KiB.  All NV
// vectors sit in LDS in plain layout.
template <int NV>
__global__ __launch_bounds__(256) void gemv_batch_f32_kernel(BatchGemvParams p) {
    extern __shared__ __align__(16) float xs[];  // [NV][K]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t K = p.K, K4 = K / 4;
    for (int64_t i = tid; i < NV * K4; i += 256) {
        const int64_t v = i / K4, q = i - v * K4;
        *(float4 *)(xs + v * K + 4 * q) = *(const float4 *)(p.x + (size_t)v * p.ldx + 4 * q);
    }
    __syncthreads();
    const int s = lane & 1;
    const int64_t row = (int64_t)blockIdx.x * 128 + wave * 32 + (lane >> 1);
    const bool row_ok = row < p.N;
    const int64_t lrow = row_ok ? row : p.N - 1;
    const float *wl = (const float *)p.w + (size_t)(lrow >> 5) * (size_t)K * 32 + (lrow & 31) * 8 + 4 * s;
    const int64_t chunks = K / 8;
    float acc[NV][4];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v][0] = acc[v][1] = acc[v][2] = acc[v][3] = 0.0f;
    constexpr int AHEAD = 8;
    float4 ring[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) ring[u] = ld_f4<true>(wl + 256 * (u < chunks ? u : chunks - 1));
    for (int64_t c0 = 0; c0 < chunks; c0 += AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int64_t c = c0 + u;
            if (c >= chunks) break;
            const float4 w = ring[u];
            const int64_t cn = c + AHEAD < chunks ? c + AHEAD : chunks - 1;
            ring[u] = ld_f4<true>(wl + 256 * cn);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const float4 x = *(const float4 *)(xs + v * K + 8 * c + 4 * s);
                acc[v][0] = fmaf(x.x, w.x, acc[v][0]);
                acc[v][1] = fmaf(x.y, w.y, acc[v][1]);
                acc[v][2] = fmaf(x.z, w.z, acc[v][2]);
                acc[v][3] = fmaf(x.w, w.w, acc[v][3]);
            }
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        // lane 2r: chains 0..3, lane 2r+1: 4..7 -> ((a0+a4)+(a1+a5)) + ((a2+a6)+(a3+a7))
        const float u0 = acc[v][0] + __shfl_xor(acc[v][0], 1, WAVE);
        const float u1 = acc[v][1] + __shfl_xor(acc[v][1], 1, WAVE);
        const float u2 = acc[v][2] + __shfl_xor(acc[v][2], 1, WAVE);
        const float u3 = acc[v][3] + __shfl_xor(acc[v][3], 1, WAVE);
        if (s != 0 || !row_ok || v >= p.nv) continue;
        float y = (u0 + u1) + (u2 + u3);
        if (row < p.bias_len) y = y + p.bias[row];
        p.y[(size_t)v * p.ldy + row] = y;
    }
}

// The same products on the f32 matrix cores, up to 16 vectors in LDS.  A matrix
// instruction with one k step is one fma per output (see rows.hip): block b of
// v_mfma_f32_16x16x1 runs chain 2b (and, in a second one, 2b + 1) of 16 rows x
// 16 vectors, so a lane's operand is two neighbouring floats of its row's
// chunk, a wave's load of 16 rows one contiguous 512 bytes, and every output's
// eight chains end in one lane.  No VALU work per weight, so the weights' bytes
// bind it: 16 vectors, 151936 x 1536 322 us with one chain per VALU lane -> 159 (5.9
// TB/s; 32768 rows 106 -> 37), 8 vectors 173 -> 150, 4 vectors 148 -> 146 (32768 rows
// 45 -> 35); reading 16 chunks ahead instead of 8 the same or 1-2 us more.
// One workgroup of eight waves per compute unit walks 128-row blocks, each wave
// 16 rows of them, F32M_AHEAD chunks ahead across the end of a block; rows of x
// sit K + 4 floats apart (K a multiple of 8: the 16 rows' reads hit all banks).
constexpr int F32M_AHEAD = 8, F32M_NT = 512, F32M_ROWS = 128;
typedef float vf2 __attribute__((ext_vector_type(2)));
typedef float vf16 __attribute__((ext_vector_type(16)));

__global__ __launch_bounds__(F32M_NT) void gemv_batch_f32_mfma_kernel(BatchGemvParams p, int nv, int64_t nblk) {
    extern __shared__ __align__(16) float xs[];  // [16][K + 4], rows past nv zero
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, fr = lane & 15, b = lane >> 4;
    const int64_t K = p.K;
    const int chunks = (int)(K / 8), K4 = (int)(K / 4);
    // this wave's 16 rows of block blk (past the padded last tile: the last tile's)
    const int64_t tiles = (p.N + 31) / 32;
    auto rows_at = [&](int64_t blk) {
        const int64_t r = blk * F32M_ROWS + 16 * wave, tile = min(r >> 5, tiles - 1);
        return (const float *)p.w + tile * K * 32 + (r & 16) * 8 + fr * 8 + 2 * b;
    };
    const float *w = rows_at(blockIdx.x);
    vf2 ring[F32M_AHEAD];
#pragma unroll
    for (int u = 0; u < F32M_AHEAD; ++u) ring[u] = __builtin_nontemporal_load((const vf2 *)(w + 256 * min(u, chunks - 1)));
    for (int i = tid; i < 16 * K4; i += F32M_NT) {
        const int v = i / K4, q = i - v * K4;
        const float4 t = v < nv ? *(const float4 *)(p.x + (size_t)v * p.ldx + 4 * q) : make_float4(0.f, 0.f, 0.f, 0.f);
        *(float4 *)(xs + v * (K + 4) + 4 * q) = t;
    }
    __syncthreads();
    const float *xl = xs + fr * (K + 4) + 2 * b;
    for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        const float *wn = rows_at(blk + gridDim.x < nblk ? blk + gridDim.x : blk);
        vf16 a0 = {}, a1 = {};
        auto group = [&](int c0, auto full) {
            const bool last = c0 + F32M_AHEAD >= chunks;
            const float *src = last ? wn : w;
#pragma unroll
            for (int u = 0; u < F32M_AHEAD; ++u) {
                const vf2 wv = ring[u];
                ring[u] = __builtin_nontemporal_load((const vf2 *)(src + 256 * min(last ? u : c0 + F32M_AHEAD + u, chunks - 1)));
                if (decltype(full)::value || c0 + u < chunks) {
                    const vf2 x = *(const vf2 *)(xl + 8 * (c0 + u));
                    a0 = __builtin_amdgcn_mfma_f32_16x16x1f32(wv.x, x.x, a0, 0, 0, 0);
                    a1 = __builtin_amdgcn_mfma_f32_16x16x1f32(wv.y, x.y, a1, 0, 0, 0);
                }
            }
        };
        int c0 = 0;
        for (; c0 + F32M_AHEAD <= chunks; c0 += F32M_AHEAD) group(c0, std::true_type{});
        if (c0 < chunks) group(c0, std::false_type{});
        w = wn;
        // lane (fr, b): vector fr, rows 4b + r; ((s0+s4)+(s1+s5)) + ((s2+s6)+(s3+s7))
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = blk * F32M_ROWS + 16 * wave + 4 * b + r;
            if (row >= p.N || fr >= p.nv) continue;
            float y = ((a0[r] + a0[8 + r]) + (a1[r] + a1[8 + r])) + ((a0[4 + r] + a0[12 + r]) + (a1[4 + r] + a1[12 + r]));
            if (row < p.bias_len) y = y + p.bias[row];
            p.y[(size_t)fr * p.ldy + row] = y;
        }
    }
}

// The same products for a batch of 16 whose activations exceed LDS, register-
// blocked over rows: lanes 2r, 2r+1 of a wave own rows r + 32j (j < RB; one 32-row
// tile each) of the wave's 32*RB rows, chains 0..3 and 4..7 as above, and a
// workgroup takes VG of the vectors, so each activation quad read from LDS feeds
// RB rows.  The batch splits over the grid, workgroups b, b+8, b+16, b+24 taking
// one row block's four vector groups; consecutive workgroups go to the eight XCDs
// in turn, so the four land on one XCD and its L2 serves the block's rows three
// times of four.
constexpr int F32B_AHEAD = 4, F32B_RB = 4, F32B_VG = 4, F32B_NT = 256;
constexpr int64_t F32B_ROWS = F32B_NT / 2 * F32B_RB;  // rows per workgroup

__global__ __launch_bounds__(F32B_NT) void gemv_batch_f32_rb_kernel(BatchGemvParams p, int64_t nblk) {
    constexpr int AHEAD = F32B_AHEAD, RB = F32B_RB, VG = F32B_VG, NT = F32B_NT;
    extern __shared__ __align__(16) float xs[];  // [VG][K]
    const int b = blockIdx.x;
    const int64_t blk = ((int64_t)(b >> 5) << 3) | (b & 7);
    if (blk >= nblk) return;  // whole workgroup: the grid is rounded up to 32
    const int vz = ((b >> 3) & 3) * VG;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t K = p.K, K4 = K / 4;
    for (int64_t i = tid; i < VG * K4; i += NT) {
        const int64_t v = i / K4, q = i - v * K4;
        *(float4 *)(xs + v * K + 4 * q) = *(const float4 *)(p.x + (size_t)(vz + v) * p.ldx + 4 * q);
    }
    __syncthreads();
    const int s = lane & 1;
    const int64_t r0 = blk * F32B_ROWS + wave * (32 * RB) + (lane >> 1);
    const float *wl[RB];
#pragma unroll
    for (int j = 0; j < RB; ++j) {
        const int64_t row = r0 + 32 * j;
        const int64_t lrow = row < p.N ? row : p.N - 1;
        wl[j] = (const float *)p.w + (size_t)(lrow >> 5) * (size_t)K * 32 + (lrow & 31) * 8 + 4 * s;
    }
    const int64_t chunks = K / 8;
    float acc[RB][VG][4];
#pragma unroll
    for (int j = 0; j < RB; ++j)
#pragma unroll
        for (int v = 0; v < VG; ++v) acc[j][v][0] = acc[j][v][1] = acc[j][v][2] = acc[j][v][3] = 0.0f;
    float4 ring[AHEAD][RB];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
#pragma unroll
        for (int j = 0; j < RB; ++j) ring[u][j] = ld_f4<true>(wl[j] + 256 * (u < chunks ? u : chunks - 1));
    for (int64_t c0 = 0; c0 < chunks; c0 += AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int64_t c = c0 + u;
            if (c >= chunks) break;
            float4 w[RB];
#pragma unroll
            for (int j = 0; j < RB; ++j) w[j] = ring[u][j];
            const int64_t cn = c + AHEAD < chunks ? c + AHEAD : chunks - 1;
#pragma unroll
            for (int j = 0; j < RB; ++j) ring[u][j] = ld_f4<true>(wl[j] + 256 * cn);
#pragma unroll
            for (int v = 0; v < VG; ++v) {
                const float4 x = *(const float4 *)(xs + v * K + 8 * c + 4 * s);
#pragma unroll
                for (int j = 0; j < RB; ++j) {
                    acc[j][v][0] = fmaf(x.x, w[j].x, acc[j][v][0]);
                    acc[j][v][1] = fmaf(x.y, w[j].y, acc[j][v][1]);
                    acc[j][v][2] = fmaf(x.z, w[j].z, acc[j][v][2]);
                    acc[j][v][3] = fmaf(x.w, w[j].w, acc[j][v][3]);
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < RB; ++j) {
        const int64_t row = r0 + 32 * j;
#pragma unroll
        for (int v = 0; v < VG; ++v) {
            // lane 2r: chains 0..3, lane 2r+1: 4..7 -> ((a0+a4)+(a1+a5)) + ((a2+a6)+(a3+a7))
            const float u0 = acc[j][v][0] + __shfl_xor(acc[j][v][0], 1, WAVE);
            const float u1 = acc[j][v][1] + __shfl_xor(acc[j][v][1], 1, WAVE);
            const float u2 = acc[j][v][2] + __shfl_xor(acc[j][v][2], 1, WAVE);
            const float u3 = acc[j][v][3] + __shfl_xor(acc[j][v][3], 1, WAVE);
            const int sv = vz + v;
            if (s != 0 || row >= p.N || sv >= p.nv) continue;
            float y = (u0 + u1) + (u2 + u3);
            if (row < p.bias_len) y = y + p.bias[row];
            p.y[(size_t)sv * p.ldy + row] = y;
        }
    }
}

// rms_norm per sequence row (norm.rs:52-88): threads 0..7 run the chains,
// out = (x * inv) * w.  Guards: st_a on the input, st_b on the output.
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(BatchRowParams p) {
    extern __shared__ __align__(16) float xs[];
    __shared__ float inv_slot;
    const int s = blockIdx.x;
    const int tid = threadIdx.x;
    const float *x = p.x + (size_t)s * p.ldx;
    int bad = 0;
    for (int64_t k = tid; k < p.K; k += 256) {
        const float v = x[k];
        bad |= isnan(v);
        xs[k] = v;
    }
    if (__syncthreads_or(bad) && tid == 0) seq_flag(p.nan_codes, s, p.layer, p.st_a);
    float inv = 1.0f;
    if (p.w) {
        rms_inv_plain(xs, p.K, p.eps, &inv_slot);
        __syncthreads();
        inv = inv_slot;
    }
    bad = 0;
    for (int64_t k = tid; k < p.K; k += 256) {
        float o = xs[k];  // no weight: the plain rows (an empty norm tensor is skipped, block/forward.rs:18-28)
        if (p.w) {
            const float t = o * inv;
            o = t * p.w[k];
        }
        bad |= isnan(o);
        p.y[(size_t)s * p.ldy + k] = o;
    }
    if (__syncthreads_or(bad) && tid == 0) seq_flag(p.nan_codes, s, p.layer, p.st_b);
}

// The same norm for K % 32 == 0 and K <= 16 * 256: each thread loads its
// float4s of x and of the weights in one batch, the eight sum-of-squares
// chains (thread l: elements 8i + l, fma(v, v, acc) in i order) read a
// chain-major LDS copy whose rows are zero past K/8 (fma(0, 0, acc) = acc, acc
// >= +0), and the outputs are formed from the registers.  The reduction
// ((a0+a4)+(a1+a5)) + ((a2+a6)+(a3+a7)) and the rounding of every step are
// those of rmsnorm_rows_kernel.
constexpr int RN_XB4 = 4;
__host__ __device__ constexpr int rn_chain_row(int64_t K) { return (int)((K / 8 + 63) / 64 * 64 + 36); }

__global__ __launch_bounds__(256) void rmsnorm_rows_cm_kernel(BatchRowParams p) {
    extern __shared__ __align__(16) float xs[];  // [8][rn_chain_row(K)]
    __shared__ float inv_slot;
    const int s = blockIdx.x, tid = threadIdx.x;
    const int64_t K = p.K, K4 = K / 4, K8 = K / 8;
    const int row = rn_chain_row(K), n = (int)((K8 + 63) / 64 * 64), tail = row - (int)K8;
    const float *x = p.x + (size_t)s * p.ldx;
    float4 xr[RN_XB4], wr[RN_XB4];
#pragma unroll
    for (int u = 0; u < RN_XB4; ++u) {
        const int64_t m = u * 256 + tid;
        xr[u] = m < K4 ? *(const float4 *)(x + 4 * m) : make_float4(0.f, 0.f, 0.f, 0.f);
        wr[u] = (p.w && m < K4) ? *(const float4 *)(p.w + 4 * m) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // the rows' zero tails [K8, row) (the chains read up to n + 32)
    for (int t = tid; t < 8 * tail; t += 256) xs[(t / tail) * row + K8 + t % tail] = 0.0f;
    int bad = 0;
#pragma unroll
    for (int u = 0; u < RN_XB4; ++u) {
        const int64_t m = u * 256 + tid;
        if (m >= K4) continue;
        const float v[4] = {xr[u].x, xr[u].y, xr[u].z, xr[u].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t k = 4 * m + j;
            xs[(k & 7) * row + (k >> 3)] = v[j];
            bad |= isnan(v[j]);
        }
    }
    if (__syncthreads_or(bad) && tid == 0) seq_flag(p.nan_codes, s, p.layer, p.st_a);
    float inv = 1.0f;
    if (p.w) {
        if (tid < 8) {
            const float acc = chain_lds_sq(0.0f, xs + tid * row, n);
            const float a = acc + __shfl(acc, (tid + 4) & 7, 8);  // lane l<4: a_l + a_{l+4}
            const float b = a + __shfl(a, (tid + 1) & 7, 8);      // lane 0: u0+u1, lane 2: u2+u3
            const float tot = b + __shfl(b, (tid + 2) & 7, 8);    // lane 0: (u0+u1) + (u2+u3)
            if (tid == 0) {
                const float mean = tot / (float)K;
                inv_slot = 1.0f / sqrtf(mean + p.eps);
            }
        }
        __syncthreads();
        inv = inv_slot;
    }
    bad = 0;
    float *y = p.y + (size_t)s * p.ldy;
    const bool wide = !((uintptr_t)y & 15);
#pragma unroll
    for (int u = 0; u < RN_XB4; ++u) {
        const int64_t m = u * 256 + tid;
        if (m >= K4) continue;
        const float v[4] = {xr[u].x, xr[u].y, xr[u].z, xr[u].w}, w[4] = {wr[u].x, wr[u].y, wr[u].z, wr[u].w};
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            o[j] = v[j];  // no weight: the plain rows
            if (p.w) {
                const float t = v[j] * inv;
                o[j] = t * w[j];
            }
            bad |= isnan(o[j]);
            if (!wide) y[4 * m + j] = o[j];
        }
        if (wide) *(float4 *)(y + 4 * m) = make_float4(o[0], o[1], o[2], o[3]);
    }
    if (__syncthreads_or(bad) && tid == 0) seq_flag(p.nan_codes, s, p.layer, p.st_b);
}

// swiglu_balanced per element (block/forward.rs:87-113) without the genomic
// norm: a grid over (sequence, 256-element slices).
__global__ __launch_bounds__(256) void swiglu_elems_kernel(BatchRowParams p) {
    const int s = blockIdx.y;
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const float *g = p.x + (size_t)s * p.ldx, *u = g + p.K;
    int bad_u = 0, bad_o = 0;
    if (k < p.K) {
        const float uv = u[k];
        bad_u = isnan(uv);
        const float o = swiglu1(g[k], uv);
        bad_o = isnan(o);
        p.y[(size_t)s * p.ldy + k] = o;
    }
    if (__any(bad_u) && (threadIdx.x & 63) == 0) seq_flag(p.nan_codes, s, p.layer, p.st_a);
    if (__any(bad_o) && (threadIdx.x & 63) == 0) seq_flag(p.nan_codes, s, p.layer, p.st_b);
}

// swiglu_balanced per element of each sequence's gate/up row pair
// (block/forward.rs:87-113), with use_genomic_norm (:115-123) when set.
__global__ __launch_bounds__(256) void swiglu_rows_kernel(BatchRowParams p) {
    extern __shared__ __align__(16) float xs[];
    __shared__ float rms_slot;
    const int s = blockIdx.x;
    const int tid = threadIdx.x;
    const float *g = p.x + (size_t)s * p.ldx, *u = g + p.K;
    int bad_u = 0, bad_o = 0;
    for (int64_t k = tid; k < p.K; k += 256) {
        const float uv = u[k];
        bad_u |= isnan(uv);
        const float o = swiglu1(g[k], uv);
        bad_o |= isnan(o);
        xs[k] = o;
    }
    const bool any_u = __syncthreads_or(bad_u);
    const bool any_o = __syncthreads_or(bad_o);
    if (tid == 0) {
        if (any_u) seq_flag(p.nan_codes, s, p.layer, p.st_a);
        if (any_o) seq_flag(p.nan_codes, s, p.layer, p.st_b);
    }
    float sc = 1.0f;
    if (p.gnorm) {
        if (tid == 0) {
            float ss = 0.0f;
            for (int64_t k = 0; k < p.K; ++k) {
                const float sq = xs[k] * xs[k];
                ss = ss + sq;
            }
            rms_slot = sqrtf(ss / (float)p.K + p.eps);
        }
        __syncthreads();
        const float rms = rms_slot;
        if (rms > p.h_scale) sc = p.h_scale / rms;
    }
    for (int64_t k = tid; k < p.K; k += 256)
        p.y[(size_t)s * p.ldy + k] = p.gnorm ? xs[k] * sc : xs[k];
}

// Greedy argmax per sequence (llm/forward.rs:262-271: strict '>', so the first
// maximum; NaN never wins; all-NaN gives 0).
__global__ __launch_bounds__(1024) void argmax_rows_kernel(const float *x, int64_t n, int64_t ld, uint32_t *out) {
    __shared__ unsigned long long best[16];
    const int s = blockIdx.x;
    const int tid = threadIdx.x;
    unsigned long long key = 0ull;
    for (int64_t i = tid; i < n; i += 1024) {
        const float v = x[(size_t)s * ld + i];
        if (isnan(v)) continue;
        const unsigned long long k = ((unsigned long long)max_key(v) << 32) | (0xFFFFFFFFu - (uint32_t)i);
        key = k > key ? k : key;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = __shfl_xor(key, o, WAVE);
        key = other > key ? other : key;
    }
    if ((tid & 63) == 0) best[tid >> 6] = key;
    __syncthreads();
    if (tid == 0) {
        unsigned long long k = best[0];
        for (int w = 1; w < 16; ++w) k = best[w] > k ? best[w] : k;
        out[s] = k ? 0xFFFFFFFFu - (uint32_t)(k & 0xFFFFFFFFull) : 0u;
    }
}

// Start of a step: sequence s takes token ids[s * n + i] (forced tokens) or
// keeps tok[s] (its previous greedy output); it runs at its cached length
// unless it is past nseq, halted, or fed the inactive id.
__global__ void batch_begin_kernel(BatchState b, const uint32_t *ids, int64_t n, int64_t i) {
    const int s = threadIdx.x;
    if (s >= b.lanes) return;
    uint32_t t = b.tok[s];
    if (ids && s < b.nseq) t = ids[(size_t)s * n + i];
    b.tok[s] = t;
    const bool run = s < b.nseq && !b.halted[s] && t != BATCH_INACTIVE;
    b.cur_pos[s] = run ? b.pos[s] : -1;
    b.nan_codes[s] = NAN_NONE;
    b.embed_ids[s] = run ? t : 0u;
}

// End of a step: a sequence whose guards held advances and (greedy) feeds its
// argmax back; one whose guard fired halts with the stage code.
__global__ void batch_end_kernel(BatchState b, uint32_t *out, int64_t n, int64_t i, int greedy) {
    const int s = threadIdx.x;
    if (s >= b.nseq || b.cur_pos[s] < 0) return;
    if (b.nan_codes[s] != NAN_NONE) {
        b.halted[s] = 1;
        b.err[s] = b.nan_codes[s];
        return;
    }
    b.pos[s] += 1;
    const uint32_t nx = b.next[s];
    if (greedy) b.tok[s] = nx;
    if (out) out[(size_t)s * n + i] = nx;
}

template <int NV>
int launch_f32(const BatchGemvParams &p, hipStream_t s) {
    const size_t lds = (size_t)NV * p.K * 4;
    if (lds + 1024 > max_lds_per_block())
        return set_error(GAJE_ERR_UNSUPPORTED, "batched f32 matvec: %d x %lld activations exceed LDS", NV, (long long)p.K);
    hipLaunchKernelGGL((gemv_batch_f32_kernel<NV>), dim3((unsigned)((p.N + 127) / 128)), dim3(256), lds, s, p);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

}  // namespace

int batch_lanes(int64_t n) { return n <= 4 ? 4 : n <= 8 ? 8 : 16; }

int launch_gemv_batch(const BatchGemvParams &p, hipStream_t s) {
    if (p.fmt == FMT_Q4_0) return launch_q4_rows(p, s);
    if (!p.w || !p.x || !p.y || p.N <= 0 || p.nv <= 0 || p.nv > 16 || p.ldx < p.K || p.ldy < p.N)
        return set_error(GAJE_ERR_INVALID_ARG, "batched matvec: bad arguments");
    const int nv = batch_lanes(p.nv);
    if (p.fmt == FMT_F32) {
        if (!p.f32_tiled || p.K % 8) return set_error(GAJE_ERR_UNSUPPORTED, "batched matvec: f32 rows must be tiled");
        if (p.mode != MODE_STORE) return set_error(GAJE_ERR_UNSUPPORTED, "batched matvec: f32 rows store only");
        // 16 vectors in LDS (K to 2540 or so): the matrix cores.  For up to four vectors, whose
        // VALU form is bound by the weights too and spreads over the compute units evenly,
        // not where the last round of blocks is mostly empty (2 vectors, 40000 x 1536 55.7 us
        // against 50.4, 49152 x 576 24.5 against 22.1; 32768 x 1536 34.9 against 46.0, 65536 x
        // 1536 64.9 against 67.1).
        const int64_t nblk = (p.N + F32M_ROWS - 1) / F32M_ROWS, cu = device_cu_count(), rounds = (nblk + cu - 1) / cu;
        if ((size_t)16 * p.K * 4 + 1024 <= max_lds_per_block() && (nv > 4 || rounds == 1 || 10 * nblk >= 9 * rounds * cu)) {
            hipLaunchKernelGGL(gemv_batch_f32_mfma_kernel, dim3((unsigned)std::min<int64_t>(nblk, cu)),
                               dim3(F32M_NT), (size_t)16 * (p.K + 4) * 4, s, p, nv, nblk);
            GAJE_HIP_CHECK(hipGetLastError());
            return GAJE_OK;
        }
        if (nv == 4) return launch_f32<4>(p, s);
        if (nv == 8) return launch_f32<8>(p, s);
        if ((size_t)4 * p.K * 4 + 1024 <= max_lds_per_block()) {
            const int64_t blocks = (p.N + F32B_ROWS - 1) / F32B_ROWS;
            const int64_t grid = (blocks + 7) / 8 * 32;  // 4 vector groups per block
            hipLaunchKernelGGL(gemv_batch_f32_rb_kernel, dim3((unsigned)grid), dim3(F32B_NT), (size_t)4 * p.K * 4, s, p, blocks);
            GAJE_HIP_CHECK(hipGetLastError());
            return GAJE_OK;
        }
        return set_error(GAJE_ERR_UNSUPPORTED, "batched f32 matvec: 4 x %lld activations exceed LDS", (long long)p.K);
    }
    return set_error(GAJE_ERR_UNSUPPORTED, "batched matvec: weight format %d", p.fmt);
}

int launch_rmsnorm_rows(const BatchRowParams &p, hipStream_t s) {
    if (!p.x || !p.y || p.K <= 0 || p.nv <= 0 || p.nv > INT32_MAX)
        return set_error(GAJE_ERR_INVALID_ARG, "rmsnorm rows: bad arguments");
    if (p.K % 32 == 0 && p.K <= RN_XB4 * 4 * 256 && p.ldx % 4 == 0 && !(((uintptr_t)p.x | (uintptr_t)p.w) & 15)) {
        hipLaunchKernelGGL(rmsnorm_rows_cm_kernel, dim3((unsigned)p.nv), dim3(256), (size_t)8 * rn_chain_row(p.K) * 4, s, p);
        GAJE_HIP_CHECK(hipGetLastError());
        return GAJE_OK;
    }
    if ((size_t)p.K * 4 + 1024 > max_lds_per_block()) return set_error(GAJE_ERR_UNSUPPORTED, "rmsnorm rows: K too large");
    hipLaunchKernelGGL(rmsnorm_rows_kernel, dim3((unsigned)p.nv), dim3(256), (size_t)p.K * 4, s, p);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_swiglu_rows(const BatchRowParams &p, hipStream_t s) {
    if (!p.x || !p.y || p.K <= 0 || p.nv <= 0 || p.nv > 65535) return set_error(GAJE_ERR_INVALID_ARG, "swiglu rows: bad arguments");
    if (!p.gnorm) {
        hipLaunchKernelGGL(swiglu_elems_kernel, dim3((unsigned)((p.K + 255) / 256), (unsigned)p.nv), dim3(256), 0, s, p);
        GAJE_HIP_CHECK(hipGetLastError());
        return GAJE_OK;
    }
    if ((size_t)p.K * 4 + 1024 > max_lds_per_block()) return set_error(GAJE_ERR_UNSUPPORTED, "swiglu rows: K too large");
    hipLaunchKernelGGL(swiglu_rows_kernel, dim3((unsigned)p.nv), dim3(256), (size_t)p.K * 4, s, p);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_batch_begin(const BatchState &b, const uint32_t *ids, int64_t n, int64_t i, hipStream_t s) {
    hipLaunchKernelGGL(batch_begin_kernel, dim3(1), dim3(64), 0, s, b, ids, n, i);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_batch_end(const BatchState &b, uint32_t *out, int64_t n, int64_t i, int greedy, hipStream_t s) {
    hipLaunchKernelGGL(batch_end_kernel, dim3(1), dim3(64), 0, s, b, out, n, i, greedy);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_argmax_rows(const float *x, int64_t n, int64_t ld, int64_t rows, uint32_t *out, hipStream_t s) {
    if (!x || !out || n <= 0 || rows <= 0 || n > 0xFFFFFFFFll) return set_error(GAJE_ERR_INVALID_ARG, "argmax rows: bad arguments");
    hipLaunchKernelGGL(argmax_rows_kernel, dim3((unsigned)rows), dim3(1024), 0, s, x, n, ld, out);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

}  // namespace gaje
