// Q4_0 weight rows x several activation rows, bit for bit
// genomic_dot_product_q4_0_avx2 (genomic.rs:263-336) per (weight row,
// activation row), on the f32 matrix cores.
//
// The reference's dot is eight independent FMA chains (chain l takes element
// 8c + l of each block's chunk c, in order) and one fixed reduction.  A matrix
// instruction with a single k step, v_mfma_f32_{16x16x1_4b,32x32x1_2b}, is one
// fma per output, rounded once: checked against fmaf over normal, subnormal,
// infinite, NaN and zero operands, no difference.  (Here a row's flush of |t| < 1e-6
// hides what a subnormal could change; the f32 head and the attention of a prompt's
// rows, which rest on the same property, have tests where it shows.)  So one MFMA block runs one
// chain: block b of the instruction holds chain l(b) of a 16 x 16 or 32 x 32
// tile of (weight row, activation row) pairs, each step feeds it one
// dequantised weight and one activation per row, and the accumulators of the
// eight chains are reduced in the reference's order at the end.  Against one
// chain per VALU lane this shares each dequantised weight between 16 or 32
// activation rows (about 1.9 VALU instructions per weight, once per tile) and
// runs the FMAs at the f32 matrix rate (122-130 TFLOP/s measured for
// independent MFMAs, against 67 for v_fma_f32).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.h"
#include "device_util.h"
#include "kernels.h"

namespace gaje {
namespace {

typedef float vf16 __attribute__((ext_vector_type(16)));
typedef float vf32 __attribute__((ext_vector_type(32)));

// Bytes of a stage (TM activation rows and TN packed weight rows of one group)
// and of the workgroup's LDS: the ring, reused for the reduction.
constexpr int rq_stage(int TM, int TN) { return TM * 512 + TN * 80; }
constexpr int rq_lds(int TM, int TN, int S) {
    const int ring = S * rq_stage(TM, TN), red = TM == 32 ? TN / 32 * 16384 : TN / 16 * 4096;
    return ring > red ? ring : red;
}

__device__ __forceinline__ void row_flag(uint32_t *codes, int64_t row, int layer, int stage) {
    if (codes && stage >= 0) atomicMin(&codes[row], (uint32_t)(layer * 8 + stage));
}

// The row epilogue for outputs n .. n+3 of activation row m, from the reduced
// dots t: flush, sparse anchors, bias (linear/forward.rs:84-115), residual.
__device__ __forceinline__ void rows_finish(const BatchGemvParams &p, int64_t m, int64_t n, const float (&t)[4]) {
    if (m >= p.nv || n >= p.N) return;
    const int cnt = (int)min((int64_t)4, p.N - n);
    float v[4];
    float *dst = p.y + (size_t)m * p.ldy + n;
    const bool wide = cnt == 4 && !((uintptr_t)dst & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        v[r] = flush_small(t[r]);
        if (r >= cnt) continue;
        if (p.a_ptr)
            for (int64_t k = p.a_ptr[n + r]; k < p.a_ptr[n + r + 1]; ++k) {
                const float prod = p.x[(size_t)m * p.ldx + p.a_col[k]] * half_bits(p.a_val[k]);
                v[r] = v[r] + prod;
            }
        if (n + r < p.bias_len) v[r] = v[r] + p.bias[n + r];
    }
    if (p.mode == MODE_RESIDUAL) {
        bool bad_a = false, bad_b = false;
        float old[4] = {0.f, 0.f, 0.f, 0.f};
        if (wide) {
            const float4 o = *(const float4 *)dst;
            old[0] = o.x, old[1] = o.y, old[2] = o.z, old[3] = o.w;
        } else {
            for (int r = 0; r < cnt; ++r) old[r] = dst[r];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (r >= cnt) continue;
            bad_a |= isnan(v[r]);
            v[r] = old[r] + v[r];
            bad_b |= isnan(v[r]);
        }
        if (bad_a) row_flag(p.nan_codes, m, p.layer, p.st_a);
        if (bad_b) row_flag(p.nan_codes, m, p.layer, p.st_b);
    }
    if (wide) {
        *(float4 *)dst = make_float4(v[0], v[1], v[2], v[3]);
    } else {
        for (int r = 0; r < cnt; ++r) dst[r] = v[r];
    }
}

// One workgroup of TN / 8 waves: TN weight rows x TM activation rows.
//
// TM = 32: wave 4t + j runs chains 2j and 2j + 1 of weight rows 32t .. 32t + 31
// (32x32x1_2b, two blocks).  TM = 16: waves 2t and 2t + 1 run chains 0..3 and
// 4..7 of weight rows 16t .. 16t + 15 (16x16x1_4b, four blocks).  Splitting a tile by chain
// keeps a wave's serial length at K / 8 MFMAs, so that a few hundred tiles fill
// the chip.  Lane i of a wave feeds row i % TMF of chain i / TMF as both
// operands (weight row for A, activation row for B).
//
// Per packed group (128 elements) a ring of S stages in LDS holds the TM
// activation rows (512 bytes each, 16-byte pieces XORed by row & 7 so that a
// chain's strided reads spread over the banks) and the 32 rows' packed groups
// as they are; all of it is copied by LDS-direct loads S - 1 groups ahead, one
// barrier per group.  The copies are the loop's only vector memory accesses,
// and every wave issues the same number, so the waits are exact counts.
template <int TM, int TN, int S>
__global__ __launch_bounds__(TN * 8) void rows_q4_kernel(BatchGemvParams p, int64_t ntiles, int64_t mtiles) {
    constexpr int XR = TM / (TN / 8);       // activation rows a wave copies per stage
    constexpr int XI = XR / 2;              // copies they take (two rows each)
    constexpr int CP = XI + 1;              // + one of eight packed rows
    static_assert(XI >= 1, "every wave copies activations");
    constexpr int STAGE = rq_stage(TM, TN);
    extern __shared__ __align__(16) uint8_t lds[];
    // An XCD takes every activation tile of the weight tiles congruent to it
    // (workgroups go to the eight XCDs in turn), so each weight row is read
    // into one L2 once.
    const int64_t j = blockIdx.x >> 3;
    const int64_t nt = (j / mtiles) * 8 + (blockIdx.x & 7);
    if (nt >= ntiles) return;  // whole workgroup
    const int64_t n0 = nt * TN, m0 = (j % mtiles) * TM;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = p.nb, G = (nb + 3) >> 2;

    // ---- copies: sources of this lane ----
    const float *xb = p.x + (size_t)m0 * p.ldx;
    const uint8_t *wb = p.w + (size_t)n0 * G * 80;
    const int mlast = (int)min((int64_t)TM, p.nv - m0) - 1, nlast = (int)min((int64_t)TN, p.N - n0) - 1;
    uint32_t xrow[XI];
    int xpiece[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int r = wave * XR + 2 * i + (lane >> 5);
        xrow[i] = (uint32_t)min(r, mlast) * (uint32_t)p.ldx * 4;
        xpiece[i] = 4 * ((lane & 31) ^ (r & 7));
    }
    const int wl = min(lane, 39), wr = wave * 8 + wl / 5;
    const uint32_t woff = (uint32_t)min(wr, nlast) * (uint32_t)G * 80 + (uint32_t)(wl % 5) * 16;
    const uint32_t lds0 = lds_addr(lds);
    const int K = nb * 32;
    auto issue = [&](int g, int slot) {
        const uint32_t base = lds0 + (uint32_t)slot * STAGE;
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            // pieces past the row's end (its last group may be partial) read the row's start; unused
            const int k = g * 128 + xpiece[i];
            lds_dma16_so(xb, xrow[i] + (uint32_t)(k < K ? k : 0) * 4, base + (wave * XR + 2 * i) * 512);
        }
        if (lane < 40) lds_dma16_so(wb, woff + (uint32_t)g * 80, base + TM * 512 + wave * 640);
    };

    // ---- operands of this lane ----
    const int m = lane & (TM - 1);
    const int row = (TM == 32 ? 32 * (wave >> 2) : 16 * (wave >> 1)) + m;
    const int l = TM == 32 ? 2 * (wave & 3) + (lane >> 5) : 4 * (wave & 1) + (lane >> 4);  // chain
    uint32_t xo[4];  // of step 4b + c in block b: + 128 b
#pragma unroll
    for (int c = 0; c < 4; ++c) xo[c] = m * 512 + (((2 * c + (l >> 2)) ^ (m & 7)) << 4) + 4 * (l & 3);
    const uint32_t wo = TM * 512 + row * 80;

    typename std::conditional<TM == 32, vf32, vf16>::type acc = {};
    auto step = [&](float w, float x) {
        if constexpr (TM == 32) acc = __builtin_amdgcn_mfma_f32_32x32x1f32(w, x, acc, 0, 0, 0);
        else acc = __builtin_amdgcn_mfma_f32_16x16x1f32(w, x, acc, 0, 0, 0);
    };

    // operands of a group: read from its stage a group ahead of its MFMAs, so
    // that the LDS reads and the dequantisation run under the previous group's
    // (two operand sets, used in turn)
    vu2 n;
    vu4 sc;
    float x[2][16], d[4][4];
    auto read = [&](float (&xr)[16], int slot) {
        const uint8_t *st = lds + slot * STAGE;
        n = *(const vu2 *)(st + wo + 8 * l);
        sc = *(const vu4 *)(st + wo + 64);
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int c = 0; c < 4; ++c) xr[4 * b + c] = *(const float *)(st + xo[c] + 128 * b);
    };
    auto dequant = [&]() {
        q4_dequant_dw<0>(d[0], n.x, sc.x);
        q4_dequant_dw<1>(d[1], n.x, sc.y);
        q4_dequant_dw<0>(d[2], n.y, sc.z);
        q4_dequant_dw<1>(d[3], n.y, sc.w);
    };

#pragma unroll
    for (int s = 0; s < S; ++s) issue(min(s, G - 1), s);
    wait_vmcnt<(S - 1) * CP>();
    lds_barrier();
    read(x[0], 0);
    dequant();
    int slot = 0;
    // group g (whole: not the last) from set cur
    auto group = [&](int g, float (&xc)[16], float (&xr)[16]) {
        const int next = slot + 1 == S ? 0 : slot + 1;
        wait_vmcnt<(S - 2) * CP>();
        lds_barrier();  // stage g + 1 has landed for every wave, and stage g has been read
        issue(min(g + S, G - 1), slot);
        read(xr, next);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) step(d[i >> 2][i & 3], xc[i]);
        dequant();
        slot = next;
    };
    auto last = [&](float (&xc)[16]) {
        const int left = nb - 4 * (G - 1);  // blocks of the last group (uniform)
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (b == 0 || b < left) {
#pragma unroll
                for (int c = 0; c < 4; ++c) step(d[b][c], xc[4 * b + c]);
            }
    };
    int g = 0;
    for (; g + 2 < G; g += 2) {
        group(g, x[0], x[1]);
        group(g + 1, x[1], x[0]);
    }
    if (g + 1 < G) {
        group(g, x[0], x[1]);
        last(x[1]);
    } else {
        last(x[0]);
    }
    wait_vmcnt<0>();
    lds_barrier();

    // ---- ((a0+a4)+(a2+a6)) + ((a1+a5)+(a3+a7)), then the row epilogue ----
    float t[4];
    if constexpr (TM == 32) {
        // registers 16 bk + 4 q + r: chain 2 (wave & 3) + bk, weight row 8 q + 4 (lane >> 5) + r;
        // wave j of the four sums q = j, two q in LDS at a time
        uint8_t *red = lds + (wave >> 2) * 16384;
        const int jw = wave & 3;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int bk = 0; bk < 2; ++bk)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int i = 16 * bk + 8 * h + 4 * q;
                    *(float4 *)(red + (((2 * jw + bk) * 2 + q) * 64 + lane) * 16) = make_float4(acc[i], acc[i + 1], acc[i + 2], acc[i + 3]);
                }
            lds_barrier();
            if ((jw >> 1) == h) {
                vf4 a[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) a[c] = *(const vf4 *)(red + ((c * 2 + (jw & 1)) * 64 + lane) * 16);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    t[r] = ((a[0][r] + a[4][r]) + (a[2][r] + a[6][r])) + ((a[1][r] + a[5][r]) + (a[3][r] + a[7][r]));
            }
            if (h == 0) lds_barrier();
        }
        rows_finish(p, m0 + m, n0 + 32 * (wave >> 2) + 8 * jw + 4 * (lane >> 5), t);
    } else {
        // registers 4 b + r: chain 4 (wave & 1) + b, weight row 4 (lane >> 4) + r
        uint8_t *red = lds + (wave >> 1) * 4096;
        if (wave & 1) {
#pragma unroll
            for (int b = 0; b < 4; ++b)
                *(float4 *)(red + (b * 64 + lane) * 16) = make_float4(acc[4 * b], acc[4 * b + 1], acc[4 * b + 2], acc[4 * b + 3]);
        }
        lds_barrier();
        if (wave & 1) return;
        vf4 a[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) a[b] = *(const vf4 *)(red + (b * 64 + lane) * 16);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            t[r] = ((acc[r] + a[0][r]) + (acc[8 + r] + a[2][r])) + ((acc[4 + r] + a[1][r]) + (acc[12 + r] + a[3][r]));
        rows_finish(p, m0 + m, n0 + 16 * (wave >> 1) + 4 * (lane >> 4), t);
    }
}

// A launch holds at most 2^32 - 1 threads in a dimension, so a product of more tiles
// goes in several (33.5M activation rows x 64).
template <int TM, int TN, int S>
int launch_rows(const BatchGemvParams &p, hipStream_t s) {
    const int64_t ntiles = (p.N + TN - 1) / TN, mtiles = (p.nv + TM - 1) / TM;
    const int64_t ngrid = (ntiles + 7) / 8 * 8, most = (int64_t)UINT32_MAX / (TN * 8) / ngrid;  // row tiles a launch takes
    if (most < 1) return set_error(GAJE_ERR_UNSUPPORTED, "q4_0 rows: %lld weight rows", (long long)p.N);
    for (int64_t t = 0; t < mtiles; t += most) {
        BatchGemvParams q = p;
        const int64_t n = std::min(most, mtiles - t), m0 = t * TM;
        q.x += m0 * p.ldx;
        q.y += m0 * p.ldy;
        if (q.nan_codes) q.nan_codes += m0;
        q.nv = std::min(p.nv - m0, n * TM);
        hipLaunchKernelGGL((rows_q4_kernel<TM, TN, S>), dim3((unsigned)(ngrid * n)), dim3(TN * 8), rq_lds(TM, TN, S), s, q,
                           ntiles, n);
        GAJE_HIP_CHECK(hipGetLastError());
    }
    return GAJE_OK;
}

// Few tiles: v_mfma_f32_4x4x1_16b, whose step is 8 weight rows x 4 activation
// rows x 8 chains in a wave (8 cycles, 13 when it waits for the step before it): a
// product of few rows spreads over four times as many waves as with the
// 16x16 form, and its serial length of K / 8 steps costs less.
//
// One workgroup of four waves: 32 weight rows (an octet each) x 4 activation
// rows.  Lane i is (row quad i >> 5, chain (i >> 2) & 7, i & 3): A is weight row
// 4 (i >> 5) + (i & 3) of the octet and B activation row i & 3, both of that chain;
// register r is weight row r of the quad against activation row i & 3.
//
// A wave pays for everything beside its MFMAs in issue slots between them (an f32
// MFMA and its own wave's VALU do not overlap): about two VALU instructions of
// dequantisation a step, the loads, and the activations' way into LDS.  Measured
// on 16 x 1536 x 8960 by leaving parts out: 21.0 us in all, 11.8 without
// dequantisation, loads and staging; the rest splits evenly between the three.
// So the weights go straight into a register ring of R4_D groups, loads are a
// uniform offset that advances and a lane's constant one, and the activations are
// transposed into one row of steps per (chain, activation row), so that a lane
// reads four steps with one conflict-free 16-byte read.  Their ring holds three
// chunks of R4_CG groups: written two chunks ahead of their use, loaded two before
// that, and read a group ahead of the MFMAs across the chunk's barrier.
// (Operands dequantised and transposed into LDS by other waves: 22.9 us, bound by
// the LDS port.)
constexpr int R4_CG = 4, R4_D = 2 * R4_CG;
constexpr int R4_ROW = 16 * R4_CG + 4;   // floats of a (chain, row): rows 4 banks apart
constexpr int R4_CHAIN = 4 * R4_ROW, R4_BUF = 8 * R4_CHAIN;
constexpr int R4_XT = R4_CG / 2;         // activation quads of a thread and chunk

__device__ __forceinline__ auto tile_buffer(const void *p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, 0x7FFFFFFF, 0x00027000);
}

__global__ __launch_bounds__(256) void rows4_q4_kernel(BatchGemvParams p, int64_t ntiles, int64_t mtiles) {
    __shared__ __align__(16) float lds[3 * R4_BUF];
    const int64_t j = blockIdx.x >> 3;  // (XCD order as above)
    const int64_t nt = (j / mtiles) * 8 + (blockIdx.x & 7);
    if (nt >= ntiles) return;  // whole workgroup
    const int64_t n0 = nt * 32, m0 = (j % mtiles) * 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = p.nb, G = (nb + 3) >> 2, K = nb * 32;
    const int m = lane & 3, l = (lane >> 2) & 7, row = 8 * wave + 4 * (lane >> 5) + m;

    // ---- weights: 8 code bytes of this lane's chain and the 16 scale bytes, per group ----
    const auto wbuf = tile_buffer(p.w + (size_t)n0 * G * 80);
    const uint32_t wscale = (uint32_t)min((int64_t)row, p.N - 1 - n0) * (uint32_t)G * 80 + 64, wcode = wscale - 64 + 8 * l;
    vu2 wn[R4_D];
    vu4 ws[R4_D];
    auto load_w = [&](int i, int g) {  // past the row's end its last group is read again
        const int at = min(g, G - 1) * 80;
        wn[i] = __builtin_bit_cast(vu2, __builtin_amdgcn_raw_buffer_load_b64(wbuf, wcode, at, 0));
        ws[i] = __builtin_bit_cast(vu4, __builtin_amdgcn_raw_buffer_load_b128(wbuf, wscale, at, 0));
    };
    // ---- activations ----
    const auto xbuf = tile_buffer(p.x + (size_t)m0 * p.ldx);
    uint32_t xsrc[R4_XT];
    float *xdst[R4_XT];
#pragma unroll
    for (int i = 0; i < R4_XT; ++i) {
        // elements k .. k+3 of a row's chunk: chains 4 (k / 4 % 2) .. + 3, step k / 8
        const int u = tid + 256 * i, r = u / (32 * R4_CG), q = u % (32 * R4_CG);
        xsrc[i] = ((uint32_t)min((int64_t)r, p.nv - 1 - m0) * (uint32_t)p.ldx + 4 * q) * 4;
        xdst[i] = lds + 4 * (q & 1) * R4_CHAIN + r * R4_ROW + (q >> 1);
    }
    auto xk = [&](int i, int c) { return c * 128 * R4_CG + 4 * ((tid + 256 * i) % (32 * R4_CG)); };
    const int whole = K / (128 * R4_CG);  // chunks that lie inside the row
    vf4 xq[2][R4_XT];
    auto load_x = [&](vf4 (&x)[R4_XT], int c) {  // past the row's end its start is read, and stored as zeros
        const int at = c * 512 * R4_CG;
#pragma unroll
        for (int i = 0; i < R4_XT; ++i)
            x[i] = c < whole ? __builtin_bit_cast(vf4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, xsrc[i], at, 0))
                             : __builtin_bit_cast(vf4, __builtin_amdgcn_raw_buffer_load_b128(
                                                           xbuf, xk(i, c) < K ? xsrc[i] + at : xsrc[i] - xk(i, 0) * 4, 0, 0));
    };
    auto store_x = [&](const vf4 (&x)[R4_XT], int c, int buf) {
        if (c < whole) {
#pragma unroll
            for (int i = 0; i < R4_XT; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) xdst[i][buf * R4_BUF + e * R4_CHAIN] = x[i][e];
        } else {
#pragma unroll
            for (int i = 0; i < R4_XT; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) xdst[i][buf * R4_BUF + e * R4_CHAIN] = xk(i, c) < K ? x[i][e] : 0.0f;
        }
    };
    const float *xl = lds + l * R4_CHAIN + m * R4_ROW;
    vf4 x[2][4];
    auto read_x = [&](vf4 (&xr)[4], int buf, int g) {
#pragma unroll
        for (int b = 0; b < 4; ++b) xr[b] = *(const vf4 *)(xl + buf * R4_BUF + 16 * g + 4 * b);
    };

    load_x(xq[0], 0);
    load_x(xq[1], 1);
#pragma unroll
    for (int i = 0; i < R4_D; ++i) load_w(i, i);
    store_x(xq[0], 0, 0);
    store_x(xq[1], 1, 1);
    load_x(xq[0], 2);
    load_x(xq[1], 3);
    lds_barrier();
    read_x(x[0], 0, 0);
    vf4 acc = {0.f, 0.f, 0.f, 0.f};
    int buf = 0;
    // R4_D groups (`all`: every one exists, else the row ends among them).  The
    // blocks that the row's last group lacks are zero weights against zero
    // activations, and fma(0, 0, acc) = acc (never -0).
    auto round = [&](int g0, auto all) {
#pragma unroll
        for (int u = 0; u < R4_D; ++u) {
            if (!decltype(all)::value && g0 + u >= G) continue;  // (uniform)
            const int next = buf == 2 ? 0 : buf + 1;
            if (u % R4_CG == 0) {
                const int c = (g0 + u) / R4_CG, nn = next == 2 ? 0 : next + 1;
                store_x(xq[u / R4_CG], c + 2, nn);
                load_x(xq[u / R4_CG], c + 4);
            }
            vf4(&xc)[4] = x[u & 1];
            if (u % R4_CG != R4_CG - 1) read_x(x[(u + 1) & 1], buf, u % R4_CG + 1);
            else read_x(x[(u + 1) & 1], next, 0);
            __builtin_amdgcn_sched_barrier(0);
            float d[4][4];
            q4_dequant_dw<0>(d[0], wn[u].x, ws[u].x);
            q4_dequant_dw<1>(d[1], wn[u].x, ws[u].y);
            q4_dequant_dw<0>(d[2], wn[u].y, ws[u].z);
            q4_dequant_dw<1>(d[3], wn[u].y, ws[u].w);
            if (decltype(all)::value) load_w(u, g0 + u + R4_D);
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc = __builtin_amdgcn_mfma_f32_4x4x1f32(d[e >> 2][e & 3], xc[e >> 2][e & 3], acc, 0, 0, 0);
            if (u % R4_CG == R4_CG - 1) {
                buf = next;
                lds_barrier();
            }
        }
    };
    int g0 = 0;
    for (; g0 + R4_D <= G; g0 += R4_D) round(g0, std::true_type{});
    if (g0 < G) round(g0, std::false_type{});

    // ((a0+a4)+(a2+a6)) + ((a1+a5)+(a3+a7)): the chains are lane bits 2..4
    float t[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float v = acc[r];
        v = v + __shfl_xor(v, 16, WAVE);
        v = v + __shfl_xor(v, 8, WAVE);
        t[r] = v + __shfl_xor(v, 4, WAVE);
    }
    if (l == 0) rows_finish(p, m0 + m, n0 + 8 * wave + 4 * (lane >> 5), t);
}

int launch_rows4(const BatchGemvParams &p, hipStream_t s) {
    const int64_t ntiles = (p.N + 31) / 32, mtiles = (p.nv + 3) / 4;
    hipLaunchKernelGGL(rows4_q4_kernel, dim3((unsigned)((ntiles + 7) / 8 * 8 * mtiles)), dim3(256), 0, s, p, ntiles, mtiles);
    GAJE_HIP_CHECK(hipGetLastError());
    return GAJE_OK;
}

}  // namespace

bool q4_rows_serve(int64_t m, int64_t n, int64_t k) {
    const int64_t cu = device_cu_count();
    if (m != 2 || n <= 80 * cu) return m >= 2;
    if (k > 2816) return false;
    if (k <= 640) return n <= 192 * cu;
    if (k <= 1024) return n <= 224 * cu && !(k < 1024 && n > 96 * cu && n <= 128 * cu);
    return true;
}

int launch_q4_rows(const BatchGemvParams &p, hipStream_t s) {
    if (!p.w || !p.x || !p.y || p.N <= 0 || p.nv <= 0 || p.ldx < p.K || p.ldx % 4 || p.ldy < p.N || p.nb <= 0 ||
        (int64_t)p.nb * 32 != p.K || p.K > (1 << 20) || (((uintptr_t)p.x | (uintptr_t)p.w) & 15) ||
        (p.mode != MODE_STORE && p.mode != MODE_RESIDUAL))
        return set_error(GAJE_ERR_INVALID_ARG, "q4_0 rows: bad arguments");
    // 4-row tiles while they are few enough to run at once, about two and a half
    // workgroups per CU: 8.6 -> 6.9 us for 16 x 2048 x 1536, 35.4 -> 21.0 for 16 x 1536
    // x 8960, 17.7 -> 12.8 for 4 x 17920 x 1536 (560 workgroups); past that the
    // larger tiles' reuse wins (768 workgroups, 64 x 1536 x 8960: 47 against 37 us;
    // 1216, 16 x 9728 x 896: 12.8 against 8.9).
    if (((p.nv + 3) / 4) * ((p.N + 31) / 32) <= 5 * (int64_t)device_cu_count() / 2) return launch_rows4(p, s);
    // 32 x 64 tiles read an activation row's group once for 64 weight rows and
    // a weight row's once for 32 activations (1536 x 17920 x 1536: 834 us
    // against 999 with 16 x 32 tiles; 1536 x 1536 x 8960: 405 against 476), but
    // need enough tiles to fill the chip: at 1064 of them (201 x 9728 x 896)
    // 53 us against 48, at 560 (64 x 17920 x 1536) 51 against 47.  Up to 16 rows
    // would leave half of each unused (5 x 151936 x 896: 89 us against 51, x 1536:
    // 145 against 82).
    if (p.nv > 16 && ((p.nv + 31) / 32) * ((p.N + 63) / 64) >= 9 * (int64_t)device_cu_count() / 2)
        return launch_rows<32, 64, 2>(p, s);
    return launch_rows<16, 32, 2>(p, s);
}

}  // namespace gaje
