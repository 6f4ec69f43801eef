// Small kernels of the decode step and the operator API (gfx950).
#include "common.h"
#include "device_util.h"

namespace gaje {

namespace {

// Embedding row of the current token: GenomicLinear::get_row_core with
// safe_idx = token % out_features (src/nn/linear/forward.rs:195-285).  The
// first workgroup also resets the per-token reductions.
__global__ __launch_bounds__(256) void embed_kernel(EmbedParams p) {
    DevState *st = p.st;
    if (st->halted) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->argmax_key = 0ull;
        st->nan_code = NAN_NONE;
    }
    const int64_t row = (int64_t)(st->token % (uint32_t)p.vocab);
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < p.K; k += (int64_t)gridDim.x * blockDim.x)
        p.h[k] = embed_value(p, row, k);
}

// get_row_core for a batch of token ids: rows [n][K] of h (prompt prefill).
__global__ __launch_bounds__(256) void embed_rows_kernel(EmbedParams p, const uint32_t *ids, int64_t n) {
    const int64_t t = blockIdx.y;
    const int64_t row = (int64_t)(ids[t] % (uint32_t)p.vocab);
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < p.K; k += (int64_t)gridDim.x * blockDim.x)
        p.h[t * p.K + k] = embed_value(p, row, k);
}

// End of a token: NaN guard -> halt, else argmax -> next token, advance.
__global__ void finalize_kernel(DevState *st, uint32_t *out_tokens) {
    if (st->halted) return;
    if (st->nan_code != NAN_NONE) {
        st->halted = 1;
        return;
    }
    const unsigned long long key = st->argmax_key;
    const uint32_t idx = key ? 0xFFFFFFFFu - (uint32_t)(key & 0xFFFFFFFFull) : 0u;
    st->token = idx;
    if (out_tokens && st->step < st->out_cap) out_tokens[st->step] = idx;
    st->step += 1;
    st->pos += 1;
}

// Host-driven state changes (kept as a kernel so they order with the stream).
__global__ void state_set_kernel(DevState *st, int32_t pos, uint32_t token, int32_t out_cap, int32_t step,
                                 int reset_guards) {
    if (pos >= 0) st->pos = pos;
    st->token = token;
    if (out_cap >= 0) st->out_cap = out_cap;
    if (step >= 0) st->step = step;
    if (reset_guards) {
        st->halted = 0;
        st->nan_code = NAN_NONE;
        st->argmax_key = 0ull;
    }
}

// lateral_inhibition_kwta (src/compute/kernels/lut.rs:45-61): the k-th largest
// value by a 4-pass radix select over orderable keys (8 bits a pass, the top
// byte first), then x < thr -> -1e9.  One workgroup of T threads.
//  - Each wave counts into its own 256-bin LDS histogram (at most 8 copies:
//    waves w and w + 8 share one), so waves barely contend.  (Merging a
//    wave's equal bins with ballots before the atomics measured slower on
//    the blocks' hidden states, whose keys spread over many top bytes.)
//  - The bin holding the rank-th largest key comes from a parallel scan of
//    the bins in descending order (256 threads, wave scans plus wave totals).
//  - Rows of at most 4 values per thread keep their keys in registers;
//    longer ones (the logits) are re-read per pass with 16-byte loads where
//    aligned.
//  - Each pass has its own histograms, zeroed once at the start.
constexpr int KW_REG = 4;  // keys per thread held in registers

// Counts key into the wave's histogram h when `in` (the key matches the
// prefix selected so far).
__device__ __forceinline__ void kw_count(uint32_t *h, uint32_t key, bool in, int shift) {
    if (in) atomicAdd(&h[(key >> shift) & 255u], 1u);
}

template <int T>
__global__ __launch_bounds__(T) void kwta_kernel(float *x, int64_t n, int64_t k, DevState *st, int64_t ld) {
    x += (size_t)blockIdx.x * ld;
    constexpr int W = T / 64, HW = W < 8 ? W : 8;  // waves, histogram copies (waves w and w + 8 share one)
    if (st && st->halted) return;
    if (n <= k || k <= 0) return;
    __shared__ uint32_t hist[4][HW][256];  // per pass and copy, zeroed once
    __shared__ uint32_t wsum[4];
    __shared__ uint32_t sel_prefix;
    __shared__ int64_t sel_rank;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    {
        uint32_t *hw = &hist[0][0][0];
        for (int i = tid; i < 4 * HW * 256; i += T) hw[i] = 0u;
    }
    const bool inreg = n <= (int64_t)T * KW_REG;
    uint32_t rk[KW_REG];
    if (inreg) {
#pragma unroll
        for (int j = 0; j < KW_REG; ++j) {
            const int64_t i = tid + (int64_t)j * T;
            rk[j] = i < n ? order_key(x[i]) : 0u;
        }
    }
    __syncthreads();
    const bool vec = ((uintptr_t)x & 15) == 0;
    uint32_t prefix = 0, mask = 0;
    int64_t rank = k;
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        uint32_t *h = hist[pass][wave % HW];
        auto match = [&](uint32_t key) { return (key & mask) == prefix; };
        if (inreg) {
#pragma unroll
            for (int j = 0; j < KW_REG; ++j) {
                const bool ok = tid + (int64_t)j * T < n;
                kw_count(h, rk[j], ok && match(rk[j]), shift);
            }
        } else if (vec) {
            const int64_t n4 = n >> 2;
            for (int64_t q = tid; q < ((n4 + T - 1) / T) * T; q += T) {
                const bool ok = q < n4;
                const float4 v = ok ? ((const float4 *)x)[q] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                const uint32_t k0 = order_key(v.x), k1 = order_key(v.y), k2 = order_key(v.z), k3 = order_key(v.w);
                kw_count(h, k0, ok && match(k0), shift);
                kw_count(h, k1, ok && match(k1), shift);
                kw_count(h, k2, ok && match(k2), shift);
                kw_count(h, k3, ok && match(k3), shift);
            }
            for (int64_t i = 4 * n4 + tid; i < n; i += T) {
                const uint32_t kk = order_key(x[i]);
                kw_count(h, kk, match(kk), shift);
            }
        } else {
            for (int64_t i = tid; i < ((n + T - 1) / T) * T; i += T) {
                const bool ok = i < n;
                const uint32_t kk = ok ? order_key(x[i]) : 0u;
                kw_count(h, kk, ok && match(kk), shift);
            }
        }
        __syncthreads();
        // bins in descending order: thread t < 256 holds bin 255 - t
        uint32_t v = 0, incl = 0;
        if (tid < 256) {
#pragma unroll
            for (int w = 0; w < HW; ++w) v += hist[pass][w][255 - tid];
            incl = v;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t u = (uint32_t)__shfl_up((int)incl, o, 64);
                if (lane >= o) incl += u;
            }
            if (lane == 63) wsum[wave] = incl;
        }
        __syncthreads();
        if (tid < 256) {
            for (int w = 0; w < wave; ++w) incl += wsum[w];
            const int64_t ex = (int64_t)incl - v;
            if (ex < rank && (int64_t)incl >= rank) {
                sel_prefix = prefix | ((uint32_t)(255 - tid) << shift);
                sel_rank = rank - ex;
            }
        }
        __syncthreads();
        prefix = sel_prefix;
        rank = sel_rank;
        mask |= 255u << shift;
    }
    const float thr = order_key_inv(prefix);
    if (inreg) {
#pragma unroll
        for (int j = 0; j < KW_REG; ++j) {
            const int64_t i = tid + (int64_t)j * T;
            if (i < n && order_key_inv(rk[j]) < thr) x[i] = -1e9f;
        }
    } else {
        for (int64_t i = tid; i < n; i += T)
            if (x[i] < thr) x[i] = -1e9f;
    }
}

// The same K-WTA for rows of at most 64 * 4 * KW_WQ values with n % 4 == 0
// (the blocks' hidden states): one wave, the row copied into LDS, wave_kwta
// (the fused form the QKV matvec runs), the row written back.
constexpr int KWW_MAX = WAVE * 4 * KW_WQ;
__global__ __launch_bounds__(WAVE) void kwta_wave_kernel(float *x, int n, int64_t k, DevState *st, int64_t ld) {
    x += (size_t)blockIdx.x * ld;
    __shared__ __align__(16) float xs[KWW_MAX];
    __shared__ __align__(16) uint32_t hist[4 * 320];
    if (st && st->halted) return;
    const int lane = threadIdx.x;
    for (int i = lane; i < n; i += WAVE) xs[i] = x[i];
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    wave_kwta(xs, n, k, hist, lane);
    for (int i = lane; i < n; i += WAVE) x[i] = xs[i];
}

// First maximum with a strict '>' (llm/forward.rs:262-271).
__global__ __launch_bounds__(1024) void argmax_kernel(const float *x, int64_t n, uint32_t *idx) {
    __shared__ unsigned long long best;
    if (threadIdx.x == 0) best = 0ull;
    __syncthreads();
    float bv = -INFINITY;
    int64_t bi = 0;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const float v = x[i];
        if (v > bv) { bv = v; bi = i; }
    }
    if (bv > -INFINITY)
        atomicMax(&best, ((unsigned long long)max_key(bv) << 32) | (0xFFFFFFFFull - (uint64_t)bi));
    __syncthreads();
    if (threadIdx.x == 0) *idx = best ? 0xFFFFFFFFu - (uint32_t)(best & 0xFFFFFFFFull) : 0u;
}

// generate_native_core's penalty and greedy choice (llm/forward.rs:243-271):
// v = logits[t], and for a generated (seen) t with penalty > 1, v * penalty if
// v < 0 else v / penalty; the first maximum with a strict '>' (NaN never wins,
// all -inf/NaN -> 0), folded into gs->key as (orderable v, ~t).  The K-WTA
// filter (forward_core's) has already been applied to the logits in place.
__global__ __launch_bounds__(256) void gen_select_kernel(const float *x, int64_t n, const uint32_t *seen,
                                                        const DevState *st, GenState *gs) {
    if (st->halted) return;
    const float pen = gs->penalty;
    float bv = -INFINITY;
    int64_t bi = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        float v = x[i];
        if ((seen[i >> 5] >> (i & 31)) & 1u) v = v < 0.0f ? v * pen : v / pen;
        if (v > bv) { bv = v; bi = i; }
    }
    unsigned long long key = bv > -INFINITY ? ((unsigned long long)max_key(bv) << 32) | (0xFFFFFFFFull - (uint64_t)bi) : 0ull;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = __shfl_xor(key, o, WAVE);
        key = other > key ? other : key;
    }
    if ((threadIdx.x & 63) == 0 && key) atomicMax(&gs->key, key);
}

// The loop's bookkeeping after a token's choice (llm/forward.rs:296-318): the
// penalised choice (if any) becomes st->token; the token is appended and
// marked seen (EOS ids are not: an EOS ends the loop, :300-302); then the
// repetition-loop detector: for w = 2..=48 with n >= 3w, the last three
// w-long chunks equal -> stop.  A stop halts the state, so later token steps
// and these kernels do nothing.  One wave; lane w - 2 checks window w.
__global__ __launch_bounds__(64) void gen_control_kernel(DevState *st, GenState *gs, uint32_t *seen, int64_t n_seen,
                                                        uint32_t *tokens, int select) {
    if (st->halted) return;
    const int lane = threadIdx.x;
    uint32_t tok = st->token;
    if (select) {
        const unsigned long long key = gs->key;
        tok = key ? 0xFFFFFFFFu - (uint32_t)(key & 0xFFFFFFFFull) : 0u;
    }
    const int n = gs->n_gen + 1;  // tokens generated including this one
    bool eos = false;
    for (int i = 0; i < gs->n_eos; ++i) eos |= gs->eos[i] == tok;
    int rep = 0;
    const int w = lane + 2;
    if (!eos && w <= 48 && n >= 3 * w) {
        // chunk [n-w, n) against [n-2w, n-w) and [n-3w, n-2w); token n-1 is tok
        bool same = true;
        for (int i = 0; i < w && same; ++i) {
            const uint32_t a = (n - w + i == n - 1) ? tok : tokens[n - w + i];
            same = a == tokens[n - 2 * w + i] && a == tokens[n - 3 * w + i];
        }
        rep = same;
    }
    rep = __any(rep);
    __syncthreads();
    if (lane == 0) {
        tokens[n - 1] = tok;
        gs->n_gen = n;
        gs->key = 0ull;
        st->token = tok;
        if (!eos && (int64_t)tok < n_seen) atomicOr(&seen[tok >> 5], 1u << (tok & 31));
        if (eos || rep) {
            gs->stop = eos ? GEN_EOS : GEN_LOOP;
            st->halted = 1;
        }
    }
}

// Q4_0Block::dequantize_weight (io/header/blocks.rs:18-30): q*scale then +min,
// rounded separately (no FMA contraction).
__global__ void dequant_q4_0_kernel(const uint8_t *blocks, float *out, int64_t nblocks) {
    const int64_t total = nblocks * 32;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = e >> 5;
        const int i = (int)(e & 31);
        const uint8_t *blk = blocks + b * 20;
        const uint8_t byte = blk[4 + i / 2];
        const float q = (float)((i % 2 == 0) ? (byte & 0x0F) : (byte >> 4));
        const uint32_t sm = (uint32_t)blk[0] | ((uint32_t)blk[1] << 8) | ((uint32_t)blk[2] << 16) |
                            ((uint32_t)blk[3] << 24);
        out[e] = __fadd_rn(__fmul_rn(q, half_lo(sm)), half_hi(sm));
    }
}

// Q8_0Block::dequantize_weight (blocks.rs:43-49): f32(q) * scale, file layout.
__global__ void dequant_q8_0_kernel(const uint8_t *blocks, float *out, int64_t nblocks) {
    const int64_t total = nblocks * 32;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const uint8_t *blk = blocks + (e >> 5) * 34;
        const float q = (float)(int32_t)(int8_t)blk[2 + (e & 31)];
        out[e] = __fmul_rn(q, half_bits((uint16_t)blk[0] | ((uint16_t)blk[1] << 8)));
    }
}

__global__ __launch_bounds__(1024) void rmsnorm_kernel(const float *x, const float *w, float eps, float *y, int64_t n) {
    extern __shared__ __align__(16) float xs[];
    __shared__ float inv_slot;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) xs[i] = x[i];
    __syncthreads();
    rmsnorm_inplace(xs, n, w, eps, &inv_slot);
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) y[i] = xs[i];
}

__global__ void expf_kernel(const float *x, float *y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = expf_ref(x[i]);
}

__global__ void swiglu_kernel(const float *g, const float *u, float *out, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = swiglu1(g[i], u[i]);
}

__global__ void fill_u32_kernel(uint32_t *p, uint32_t v, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Floor probes for the benchmarks: a kernel that does nothing, and one that
// reads n16 16-byte words (four loads in flight per thread, grid-strided) and
// folds them, writing only when the fold hits one fixed value so the loads
// stay.  Launch boundary and plain-read time of a launch of the same grid.
__global__ void empty_kernel() {}

__global__ __launch_bounds__(256) void read_kernel(const uint8_t *buf, int64_t n16, uint32_t *sink) {
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    uint32_t acc = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += 4 * step) {
        vu4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t j = i + u * step;
            v[u] = j < n16 ? ld_u4<true>(buf + 16 * j) : vu4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    }
    if (acc == 0x9E3779B9u) sink[blockIdx.x & 63] = acc;
}

unsigned grid_for(int64_t n, int threads, unsigned cap = 4096) {
    int64_t g = (n + threads - 1) / threads;
    if (g < 1) g = 1;
    return (unsigned)(g > cap ? cap : g);
}

}  // namespace

int launch_embed(const EmbedParams &p, hipStream_t s) {
    if (!p.st || !p.h || p.vocab <= 0 || p.K <= 0) return set_error(GAJE_ERR_INVALID_ARG, "embed: bad arguments");
    hipLaunchKernelGGL(embed_kernel, dim3(grid_for(p.K, 256, 64)), dim3(256), 0, s, p);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_embed_rows(const EmbedParams &p, const uint32_t *ids, int64_t n, hipStream_t s) {
    if (!p.h || !ids || p.vocab <= 0 || p.K <= 0 || n <= 0 || n > 65535)
        return set_error(GAJE_ERR_INVALID_ARG, "embed rows: bad arguments");
    hipLaunchKernelGGL(embed_rows_kernel, dim3(grid_for(p.K, 256, 16), (unsigned)n), dim3(256), 0, s, p, ids, n);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_finalize(DevState *st, uint32_t *out_tokens, hipStream_t s) {
    hipLaunchKernelGGL(finalize_kernel, dim3(1), dim3(1), 0, s, st, out_tokens);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_state_set(DevState *st, int32_t pos, uint32_t token, int32_t out_cap, int32_t step, int reset_guards,
                     hipStream_t s) {
    hipLaunchKernelGGL(state_set_kernel, dim3(1), dim3(1), 0, s, st, pos, token, out_cap, step, reset_guards);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

namespace {
int kwta_grid(float *x, int64_t n, int64_t ld, int64_t rows, int64_t k, DevState *st, hipStream_t s) {
    if (!x || n < 0 || rows < 1 || rows > INT32_MAX || (rows > 1 && ld < n)) return set_error(GAJE_ERR_INVALID_ARG, "kwta: bad arguments");
    if (n <= k || k <= 0) return GAJE_OK;
    if (n % 4 == 0 && n <= KWW_MAX)
        hipLaunchKernelGGL(kwta_wave_kernel, dim3((unsigned)rows), dim3(WAVE), 0, s, x, (int)n, k, st, ld);
    else
        hipLaunchKernelGGL(kwta_kernel<1024>, dim3((unsigned)rows), dim3(1024), 0, s, x, n, k, st, ld);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}
}  // namespace

int launch_kwta(float *x, int64_t n, int64_t k, DevState *st, hipStream_t s) { return kwta_grid(x, n, n, 1, k, st, s); }

int launch_kwta_rows(float *x, int64_t n, int64_t ld, int64_t rows, int64_t k, hipStream_t s) {
    return kwta_grid(x, n, ld, rows, k, nullptr, s);
}

int launch_argmax(const float *x, int64_t n, uint32_t *idx, hipStream_t s) {
    if (!x || !idx || n < 0) return set_error(GAJE_ERR_INVALID_ARG, "argmax: bad arguments");
    hipLaunchKernelGGL(argmax_kernel, dim3(1), dim3(1024), 0, s, x, n, idx);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_dequant_q4_0(const uint8_t *blocks, float *out, int64_t nblocks, hipStream_t s) {
    if (nblocks < 0 || (nblocks > 0 && (!blocks || !out))) return set_error(GAJE_ERR_INVALID_ARG, "dequant: bad arguments");
    if (nblocks == 0) return GAJE_OK;
    hipLaunchKernelGGL(dequant_q4_0_kernel, dim3(grid_for(nblocks * 32, 256)), dim3(256), 0, s, blocks, out, nblocks);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_dequant_q8_0(const uint8_t *blocks, float *out, int64_t nblocks, hipStream_t s) {
    if (nblocks < 0 || (nblocks > 0 && (!blocks || !out))) return set_error(GAJE_ERR_INVALID_ARG, "dequant: bad arguments");
    if (nblocks == 0) return GAJE_OK;
    hipLaunchKernelGGL(dequant_q8_0_kernel, dim3(grid_for(nblocks * 32, 256)), dim3(256), 0, s, blocks, out, nblocks);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_rmsnorm(const float *x, const float *w, float eps, float *y, int64_t n, hipStream_t s) {
    if (!x || !w || !y || n <= 0) return set_error(GAJE_ERR_INVALID_ARG, "rmsnorm: bad arguments");
    if (n * 4 + 1024 > 64 * 1024) return set_error(GAJE_ERR_UNSUPPORTED, "rmsnorm: n = %lld too large", (long long)n);
    hipLaunchKernelGGL(rmsnorm_kernel, dim3(1), dim3(1024), (size_t)n * 4, s, x, w, eps, y, n);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_expf(const float *x, float *y, int64_t n, hipStream_t s) {
    if (n < 0 || (n > 0 && (!x || !y))) return set_error(GAJE_ERR_INVALID_ARG, "expf: bad arguments");
    if (n == 0) return GAJE_OK;
    hipLaunchKernelGGL(expf_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, x, y, n);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_swiglu(const float *g, const float *u, float *out, int64_t n, hipStream_t s) {
    if (n < 0 || (n > 0 && (!g || !u || !out))) return set_error(GAJE_ERR_INVALID_ARG, "swiglu: bad arguments");
    if (n == 0) return GAJE_OK;
    hipLaunchKernelGGL(swiglu_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, g, u, out, n);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_gen_select(const float *logits, int64_t n, const uint32_t *seen, DevState *st, GenState *gs, hipStream_t s) {
    if (!logits || !seen || !st || !gs || n <= 0) return set_error(GAJE_ERR_INVALID_ARG, "gen_select: bad arguments");
    hipLaunchKernelGGL(gen_select_kernel, dim3(grid_for(n, 256, 256)), dim3(256), 0, s, logits, n, seen, st, gs);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_gen_control(DevState *st, GenState *gs, uint32_t *seen, int64_t n_seen, uint32_t *tokens, int select,
                       hipStream_t s) {
    if (!st || !gs || !seen || !tokens) return set_error(GAJE_ERR_INVALID_ARG, "gen_control: bad arguments");
    hipLaunchKernelGGL(gen_control_kernel, dim3(1), dim3(64), 0, s, st, gs, seen, n_seen, tokens, select);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_floor_probe(const void *buf, int64_t bytes, unsigned grid, unsigned block, hipStream_t s) {
    if (grid == 0 || block == 0 || block > 1024 || (bytes > 0 && (!buf || bytes < 256 || block > 256)))
        return set_error(GAJE_ERR_INVALID_ARG, "floor probe: bad arguments");
    if (bytes == 0) hipLaunchKernelGGL(empty_kernel, dim3(grid), dim3(block), 0, s);
    else
        hipLaunchKernelGGL(read_kernel, dim3(grid), dim3(block), 0, s, (const uint8_t *)buf, bytes / 16,
                           (uint32_t *)const_cast<void *>(buf));
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

int launch_fill_u32(uint32_t *p, uint32_t v, int64_t n, hipStream_t s) {
    if (n <= 0) return GAJE_OK;
    hipLaunchKernelGGL(fill_u32_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, p, v, n);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

}  // namespace gaje
