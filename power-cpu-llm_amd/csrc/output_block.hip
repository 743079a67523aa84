// The attention output block on gfx950: projected = W_o . attended, then
// result = residual + rms_norm(projected, post_scale) (src/engine/
// attention.rs:866-884; project_streamed / project_streamed_batch_with over
// p9_ref_matvec, src/kernels/portable/reference.rs:36-78).
//
// The engine's exact projection sums f64 products of f32 weights and inputs
// (each product is exact in f64) per output row. Every projection kernel here
// accumulates in f64 as well, in its own order, so a projected value is the
// f32 rounding of nearly the same f64 sum: it equals the engine's except when
// the two f64 sums straddle an f32 rounding boundary, and a sum like
// 2^24 + 1 - 2^24 stays exact. The order depends on the token count only: one
// for up to 32 tokens (the first three kernels give the same bits), one for
// more (the chains and the tiles of every shape).
//
//   project_rows_kernel: up to five tokens. HBM-bound on the
//     weights: one wave per output row streams the row once with 16-byte
//     loads, 4096 columns in flight at a time, and keeps one f64 accumulator
//     per token per lane; the tokens' inputs come from L2.
//   project_row_lds_kernel: one token (decode), input rows up to 16384
//     wide: as project_rows_kernel<1>, with the input row staged once per
//     workgroup in LDS (requested ahead of the weights) instead of read from
//     L2 by every wave.
//   project_few_kernel: up to 32 tokens (verification, short prompts): the
//     waves of a workgroup split the columns of 16 output rows, f64 MFMAs on
//     operands loaded straight from memory.
//   project_chain_kernel: more tokens, while 16 x 16 blocks are one per SIMD:
//     f64 MFMAs on operands loaded straight from memory, one chain a wave.
//   project_tiles_kernel: more tokens (prompt). MFMA-bound: output
//     tiles of 128 x 128 down to 32 x 32, K steps double-buffered in LDS as
//     f32, the products on v_mfma_f64_16x16x4f64 after converting the
//     operands to f64.
//   post_norm_kernel: one workgroup per token: the row's f64 sum of squares
//     (per-thread partial sums, then a fixed tree of lane shuffles and the
//     four waves), inv = 1/sqrt(ms + eps) in f64, y = f32(x * inv) * scale,
//     result = residual + y (f32).
#include "attention_device.hpp"
#include "context.hpp"
#include "launch.hpp"
#include "pcl_attention.h"

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <iterator>
#include <type_traits>

namespace pcl {

constexpr int kErrBlock = 8; // non-finite value in the output block

struct BlockParams {
    const float *x;     // attended rows [n][in]
    const float *w;     // weights [out][in]
    float *proj;        // projected rows [n][out]
    const float *scale; // post-norm scale [out]
    const float *res;   // residual rows [n][out]
    float *result;      // [n][out]
    int n, in, out;
    float eps;
    int *err;
};

// One wave per output row, NT = n tokens (a kernel for each count: tests for
// absent tokens in the inner loop cost 1 to 5 us at 2 to 4 tokens). Every
// token's f64 sum runs in the same order in every instantiation.
template <int NT>
__global__ __launch_bounds__(256) void project_rows_kernel(BlockParams p)
{
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= p.out)
        return;
    const float *wr = p.w + (int64_t)r * p.in;
    double acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        acc[t] = 0.0;
    // 16-byte steps of the row: 4096 columns (16 per lane) in flight at once,
    // so a wave's row costs one memory round trip
    const int vecs = p.in / 4;
    int v = lane;
    for (; v + 960 < vecs; v += 1024) {
        f4 wv[16];
#pragma unroll
        for (int k = 0; k < 16; ++k)
            wv[k] = ldg4_stream(wr + 4 * (v + 64 * k));
#pragma unroll
        for (int k = 0; k < 16; ++k) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const f4 xv = ldg4(p.x + (int64_t)t * p.in + 4 * (v + 64 * k));
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[t] = __builtin_fma((double)wv[k][e], (double)xv[e], acc[t]);
            }
        }
    }
    for (; v < vecs; v += 64) {
        const f4 wv = ldg4_stream(wr + 4 * v);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const f4 xv = ldg4(p.x + (int64_t)t * p.in + 4 * v);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[t] = __builtin_fma((double)wv[e], (double)xv[e], acc[t]);
        }
    }
    // columns past the last whole 16-byte step
    for (int c = 4 * vecs + lane; c < p.in; c += 64) {
        const double wc = (double)ldg(wr + c);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            acc[t] = __builtin_fma(wc, (double)ldg(p.x + (int64_t)t * p.in + c), acc[t]);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        double s = acc[t];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1)
            s += __shfl_xor(s, o);
        acc[t] = s;
    }
    if (lane < NT) {
        double mine = 0.0;
#pragma unroll
        for (int t = 0; t < NT; ++t)
            mine = lane == t ? acc[t] : mine;
        stg(p.proj + (int64_t)lane * p.out + r, (float)mine);
    }
}

// TM x TN output tile per 256-thread workgroup (2 x 2 waves of TM/2 x TN/2),
// K in steps of TK columns, LDS rows padded by 4 floats (16-byte aligned, and
// the 16 rows an MFMA operand read touches fall in distinct banks). Every
// output sums its columns in the same order in every instantiation.
typedef double d4 __attribute__((ext_vector_type(4)));

template <int TM, int TN, int TK>
constexpr size_t tile_lds_bytes()
{
    return 2 * sizeof(float) * (TM + TN) * (TK + 4);
}

// Two workgroups per CU (at most 2 x 72 KiB of LDS; registers held to 256
// per lane, which also keeps the f64 accumulators out of AGPRs): 16 % faster
// than one on a 4K-token projection, where the other workgroup hides a
// wave's LDS and conversion latency between MFMAs.
template <int TM, int TN, int TK>
__global__ __launch_bounds__(256, 2) void project_tiles_kernel(BlockParams p)
{
    constexpr int kRow = TK + 4;
    constexpr int kQuads = TK / 4;              // float4 per row and K step
    constexpr int kLoadA = TM * kQuads / 256;   // float4 per thread and K step
    constexpr int kLoadB = TN * kQuads / 256;
    constexpr int kI = TM / 32, kJ = TN / 32;   // 16 x 16 blocks of a wave
    extern __shared__ __attribute__((aligned(16))) float tiles[];
    // two buffers of A rows, then two of B rows
    float *const sa = tiles, *const sb = tiles + 2 * TM * kRow;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TN / 2);
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;

    // global -> registers -> LDS; the next step's loads are in flight during
    // this step's MFMAs. Rows past the last repeat it (not written), columns
    // past the last are zero: a branch around each load of a whole step cost
    // 6 to 16 % (256 tokens of 4096 columns 159 -> 142 us, 2000 tokens 866 -> 791).
    f4 ra[kLoadA], rb[kLoadB];
    auto load = [&](int k0) {
        if (k0 + TK <= p.in) { // all loads go out together
#pragma unroll
            for (int i = 0; i < kLoadA; ++i) {
                const int idx = tid + 256 * i;
                ra[i] = ldg4(p.x + (int64_t)min(m0 + idx / kQuads, p.n - 1) * p.in + k0 +
                             4 * (idx % kQuads));
            }
#pragma unroll
            for (int i = 0; i < kLoadB; ++i) {
                const int idx = tid + 256 * i;
                rb[i] = ldg4_stream(p.w + (int64_t)min(n0 + idx / kQuads, p.out - 1) * p.in + k0 +
                                    4 * (idx % kQuads));
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < kLoadA; ++i) {
            const int idx = tid + 256 * i;
            const int k = k0 + 4 * (idx % kQuads);
            const float *src = p.x + (int64_t)min(m0 + idx / kQuads, p.n - 1) * p.in + k;
            for (int e = 0; e < 4; ++e)
                ra[i][e] = k + e < p.in ? ldg(src + e) : 0.f;
        }
#pragma unroll
        for (int i = 0; i < kLoadB; ++i) {
            const int idx = tid + 256 * i;
            const int k = k0 + 4 * (idx % kQuads);
            const float *src = p.w + (int64_t)min(n0 + idx / kQuads, p.out - 1) * p.in + k;
            for (int e = 0; e < 4; ++e)
                rb[i][e] = k + e < p.in ? ldg(src + e) : 0.f;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kLoadA; ++i) {
            const int idx = tid + 256 * i;
            *(f4 *)(sa + buf * TM * kRow + idx / kQuads * kRow + 4 * (idx % kQuads)) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < kLoadB; ++i) {
            const int idx = tid + 256 * i;
            *(f4 *)(sb + buf * TN * kRow + idx / kQuads * kRow + 4 * (idx % kQuads)) = rb[i];
        }
    };

    d4 acc[kI][kJ];
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int j = 0; j < kJ; ++j)
            acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};

    const int steps = (p.in + TK - 1) / TK;
    load(0);
    store(0);
    __syncthreads();
    const int r16 = lane & 15, kq = lane >> 4;
    for (int s = 0; s < steps; ++s) {
        const int buf = s & 1;
        if (s + 1 < steps)
            load((s + 1) * TK);
        if constexpr (kI * kJ == 1) {
            // A single chain of MFMAs: each would wait for its operands'
            // conversions, and these for the MFMA before it that still reads
            // their registers. Operands are read 32 and converted 16 columns
            // ahead into registers of their own (256 tokens of 4096 columns, 2816
            // rows: 135.7 -> 125.7 us; 64 tokens 57.8 -> 52.5 us).
            const float *ar = sa + (buf * TM + wm + r16) * kRow + 4 * kq;
            const float *br = sb + (buf * TN + wn + r16) * kRow + 4 * kq;
            f4 a[2], b[2];
            double ca[2][4], cb[2][4];
            auto read = [&](int kc, int set) {
                a[set] = *(const f4 *)(ar + kc);
                b[set] = *(const f4 *)(br + kc);
            };
            auto convert = [&](int set) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    ca[set][j] = (double)a[set][j];
                    cb[set][j] = (double)b[set][j];
                }
            };
            read(0, 0);
            read(16, 1);
            convert(0);
#pragma unroll
            for (int kc = 0; kc < TK; kc += 16) {
                const int set = (kc / 16) & 1;
                if (kc + 32 < TK)
                    read(kc + 32, set);
                if (kc + 16 < TK)
                    convert(set ^ 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ca[set][j], cb[set][j],
                                                                     acc[0][0], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int kc = 0; kc < TK; kc += 16) {
                // MFMA k slot kq of step j holds column kc + 4 kq + j
                f4 a[kI], b[kJ];
#pragma unroll
                for (int i = 0; i < kI; ++i)
                    a[i] = *(const f4 *)(sa + (buf * TM + wm + 16 * i + r16) * kRow + kc + 4 * kq);
#pragma unroll
                for (int i = 0; i < kJ; ++i)
                    b[i] = *(const f4 *)(sb + (buf * TN + wn + 16 * i + r16) * kRow + kc + 4 * kq);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < kI; ++i)
#pragma unroll
                        for (int jj = 0; jj < kJ; ++jj)
                            acc[i][jj] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                (double)a[i][j], (double)b[jj][j], acc[i][jj], 0, 0, 0);
            }
        }
        if (s + 1 < steps)
            store(buf ^ 1); // read last in step s - 1, before that step's barrier
        __syncthreads();
    }
    // acc[i][jj][e]: row wm + 16i + kq + 4e, column wn + 16 jj + r16 (the f64
    // MFMA's output rows interleave by lane group, unlike the f32 one's)
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = m0 + wm + 16 * i + kq + 4 * e;
            if (row >= p.n)
                continue;
#pragma unroll
            for (int jj = 0; jj < kJ; ++jj) {
                const int col = n0 + wn + 16 * jj + r16;
                if (col < p.out)
                    stg(p.proj + (int64_t)row * p.out + col, (float)acc[i][jj][e]);
            }
        }
}

// One 256-thread workgroup per token row; rows up to 4096 wide stay in
// registers between the sum of squares and the output.
constexpr int kNormPer = 16;

__global__ __launch_bounds__(256) void post_norm_kernel(BlockParams p)
{
    __shared__ double part[4];
    const int t = blockIdx.x;
    const int tid = threadIdx.x;
    const float *x = p.proj + (int64_t)t * p.out;
    const float *res = p.res + (int64_t)t * p.out;
    float *y = p.result + (int64_t)t * p.out;
    const bool cached = p.out <= 256 * kNormPer;
    float xv[kNormPer], rv[kNormPer], sv[kNormPer];
    double sum = 0.0;
    bool bad = false;
    if (cached) {
#pragma unroll
        for (int k = 0; k < kNormPer; ++k) {
            const int c = tid + 256 * k;
            xv[k] = c < p.out ? ldg(x + c) : 0.f;
            rv[k] = c < p.out ? ldg(res + c) : 0.f;
            sv[k] = c < p.out ? ldg(p.scale + c) : 0.f;
        }
#pragma unroll
        for (int k = 0; k < kNormPer; ++k) {
            bad |= !is_finite(xv[k]);
            sum = __builtin_fma((double)xv[k], (double)xv[k], sum);
        }
    } else {
        for (int c = tid; c < p.out; c += 256) {
            const float v = ldg(x + c);
            bad |= !is_finite(v);
            sum = __builtin_fma((double)v, (double)v, sum);
        }
    }
    // the block's sum: a fixed tree over lanes, then over the four waves
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1)
        sum += __shfl_xor(sum, o);
    if ((tid & 63) == 0)
        part[tid >> 6] = sum;
    __syncthreads();
    const double total = (part[0] + part[1]) + (part[2] + part[3]);
    const double inv = 1.0 / __builtin_sqrt(total / (double)p.out + (double)p.eps);
    if (cached) {
#pragma unroll
        for (int k = 0; k < kNormPer; ++k) {
            const int c = tid + 256 * k;
            if (c < p.out) {
                const float r = rv[k] + (float)((double)xv[k] * inv) * sv[k];
                bad |= !is_finite(r);
                stg(y + c, r);
            }
        }
    } else {
        for (int c = tid; c < p.out; c += 256) {
            const float normed = (float)((double)ldg(x + c) * inv) * ldg(p.scale + c);
            const float r = ldg(res + c) + normed;
            bad |= !is_finite(r);
            stg(y + c, r);
        }
    }
    if (bad)
        atomicOr(p.err, kErrBlock);
}

// The largest input row project_row_lds_kernel stages (64 KiB of LDS).
constexpr int kLdsRowFloats = 16384;

// One token, t0 (p.in % 4 == 0, p.in <= kLdsRowFloats), one wave per output
// row as in project_rows_kernel<1> (the same f64 sums in the same order):
// the workgroup stages the input row in LDS once, its first 4096 columns
// requested before the rows' first weights so that the LDS stores wait only
// for them.
__global__ __launch_bounds__(256) void project_row_lds_kernel(BlockParams p, int t0)
{
    extern __shared__ f4 xs[];
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int vecs = p.in / 4;
    const bool live = r < p.out;
    // a wave past the last row streams row 0 (in bounds; unused)
    const float *wr = p.w + (int64_t)(live ? r : 0) * p.in;
    const float *xr = p.x + (int64_t)t0 * p.in;
    f4 wv[16];
    int v = lane;
    if (vecs >= 1024) {
        f4 t[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            t[j] = ldg4(xr + 4 * (threadIdx.x + 256 * j));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 16; ++k)
            wv[k] = ldg4_stream(wr + 4 * (v + 64 * k));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            xs[threadIdx.x + 256 * j] = t[j];
        if (vecs > 1024)
            for (int i = 1024 + threadIdx.x; i < vecs; i += 256)
                xs[i] = ldg4(xr + 4 * i);
    } else {
        for (int i = threadIdx.x; i < vecs; i += 256)
            xs[i] = ldg4(xr + 4 * i);
    }
    __syncthreads();
    if (!live)
        return;
    double acc = 0.0;
    for (; v + 960 < vecs; v += 1024) {
        // the first step's weights are in flight already when every lane
        // takes it (vecs >= 1024); below that only lanes lane + 960 < vecs
        // take it, and request them here
        if (v != lane || vecs < 1024) {
#pragma unroll
            for (int k = 0; k < 16; ++k)
                wv[k] = ldg4_stream(wr + 4 * (v + 64 * k));
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const f4 xv = xs[v + 64 * k];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc = __builtin_fma((double)wv[k][e], (double)xv[e], acc);
        }
    }
    for (; v < vecs; v += 64) {
        const f4 w1 = ldg4_stream(wr + 4 * v);
        const f4 xv = xs[v];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc = __builtin_fma((double)w1[e], (double)xv[e], acc);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1)
        acc += __shfl_xor(acc, o);
    if (lane == 0)
        stg(p.proj + (int64_t)t0 * p.out + r, (float)acc);
}

// The 4 x 4 transpose of four registers over a wave's four 16-lane groups:
// lane group g's element i becomes lane group i's element g.
__device__ __forceinline__ f4 transpose_groups(f4 v)
{
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[2]),
                                                    false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[1]), __float_as_uint(v[3]),
                                                    false, false);
    const auto lo = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    return f4{__uint_as_float(lo[0]), __uint_as_float(lo[1]), __uint_as_float(hi[0]),
              __uint_as_float(hi[1])};
}

// 16 output rows x 16 NB tokens per workgroup, its eight waves splitting the
// columns. A wave loads MFMA operands straight from memory (every weight is
// used by one wave only, so LDS would add a pass), the next 256 columns'
// requested ahead of the ones being multiplied. Two waves share a 128-byte
// line of the weights, so these are plain loads: streaming ones took 37.9
// against 35.6 us at 8 tokens of 8192 columns, 2816 rows from HBM (25.2 against
// 21.9 us at 16 tokens of 4096 columns from the last-level cache).
//
// Every output is the sum that project_rows_kernel forms, bit for bit, so a
// token's row does not depend on how many tokens come with it: that kernel's
// lane l sums the 16-byte quads l, l + 64, ... of a row, and here each l has
// an accumulator of its own, wave w those of lanes 4w to 4w + 3 and 32 + 4w to
// 35 + 4w. The f64 MFMA adds its four k slots as an ascending chain of fmas;
// transposing the quads over the lane groups makes the slots the quad's
// columns. The lane sums meet as in the shuffles there: over lanes 32 in the
// wave, 16, 8 and 4 with other waves through LDS, 2 and 1 in the wave.
//
// Bound by the weights' stream and its round trips, at 32 tokens also by the
// MFMAs of the CUs that have a group of rows (13.7 us of the 31 at 4096
// columns, at the fp64 peak). 2816 x 4096 with its post-norm, one wave per row
// against this: 8 tokens 33.2 -> 19.5 us, 16 tokens 52 -> 21.9 us, 32 tokens
// 117 -> 31.4 us (from HBM 21.3, 25.1 and 34.8 us).
constexpr int kFewWaves = 8;
constexpr int kFewStep = 256; // columns per step: one quad of every lane sum

template <int NB>
__global__ __launch_bounds__(64 * kFewWaves, 2) void project_few_kernel(BlockParams p)
{
    static_assert(NB == 1 || NB == 2, "half of the waves gather a token block's sums");
    // partner sums of the waves that gather: [wave][accumulator][element][lane]
    __shared__ double sums[4 * NB][4][4][64];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int r0 = blockIdx.x * 16, t0 = blockIdx.y * 16 * NB;
    const int c0 = 16 * wave + 4 * kq; // this lane's first column
    const int whole = p.in & ~3;       // columns in whole quads
    // rows and tokens past the last repeat it (not written)
    const float *wr = p.w + (int64_t)min(r0 + r16, p.out - 1) * p.in;
    const float *xr[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
        xr[b] = p.x + (int64_t)min(t0 + 16 * b + r16, p.n - 1) * p.in;

    struct Piece {
        f4 w[2], x[NB][2];
    };
    // a quad past the last whole one reads the row's first and is zeroed below
    auto load = [&](int k, Piece &v) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int c = k + c0 + 128 * h;
            const int at = c < whole ? c : 0;
            v.w[h] = ldg4(wr + at);
#pragma unroll
            for (int b = 0; b < NB; ++b)
                v.x[b][h] = ldg4(xr[b] + at);
        }
    };
    // acc[b][h][i]: the sums of lane 32 h + 4 wave + i of project_rows_kernel
    d4 acc[NB][2][4];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[b][h][i] = d4{0.0, 0.0, 0.0, 0.0};
    // masked: the step may hold quads past the last whole one
    auto multiply = [&](int k, const Piece &v, auto masked) {
        const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool in = !masked || k + c0 + 128 * h < whole;
            const f4 w = transpose_groups(in ? v.w[h] : zero);
            f4 x[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b)
                x[b] = transpose_groups(in ? v.x[b][h] : zero);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[b][h][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        (double)x[b][i], (double)w[i], acc[b][h][i], 0, 0, 0);
        }
    };
    if (whole > 0) {
        Piece even, odd;
        load(0, even);
        int k = 0;
        for (; k + 2 * kFewStep <= whole; k += 2 * kFewStep) {
            load(k + kFewStep, odd);
            __builtin_amdgcn_sched_barrier(0);
            multiply(k, even, std::false_type{});
            load(k + 2 * kFewStep, even);
            __builtin_amdgcn_sched_barrier(0);
            multiply(k + kFewStep, odd, std::false_type{});
        }
        if (k < whole) {
            load(k + kFewStep, odd);
            multiply(k, even, std::true_type{});
            multiply(k + kFewStep, odd, std::true_type{});
        }
    }
    // columns past the last whole quad belong to lanes 0, 1 and 2
    if (wave == 0) {
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            const int c = whole + l;
            if (c < p.in) {
                const double w = kq == 0 ? (double)ldg(wr + c) : 0.0;
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[b][0][l] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        kq == 0 ? (double)ldg(xr[b] + c) : 0.0, w, acc[b][0][l], 0, 0, 0);
            }
        }
    }

    // Waves 0-3 gather token block 0, waves 4-7 block 1.
    auto put = [&](int slot, const d4 (&v)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                sums[slot][i][e][lane] = v[i][e];
    };
    d4 s[4];
    auto add = [&](int slot) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s[i][e] += sums[slot][i][e][lane];
    };
    auto halves = [&](int b) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            s[i] = acc[b][0][i] + acc[b][1][i];
    };
    const bool upper = wave >= 4;
    const bool gathers = NB == 2 || !upper;
    const int mine = upper ? NB - 1 : 0;
    if (upper) {
        halves(0);
        put(wave ^ 4, s);
        if (NB == 2)
            halves(NB - 1);
    } else {
        if (NB == 2) {
            halves(NB - 1);
            put(wave ^ 4, s);
        }
        halves(0);
    }
    __syncthreads();
    if (gathers) {
        add(wave);
        if (wave & 2)
            put(wave, s); // only this wave's own lanes have read the slot
    }
    __syncthreads();
    if (gathers && !(wave & 2)) {
        add(wave ^ 2);
        if (wave & 1)
            put(wave, s);
    }
    __syncthreads();
    if (!gathers || (wave & 3))
        return;
    add(wave ^ 1);
    // element e: token 16 mine + kq + 4e, row r16
    const d4 sum = (s[0] + s[2]) + (s[1] + s[3]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int t = t0 + 16 * mine + kq + 4 * e, r = r0 + r16;
        if (t < p.n && r < p.out)
            stg(p.proj + (int64_t)t * p.out + r, (float)sum[e]);
    }
}

// 16 output rows x 16 tokens per wave, a workgroup of its own: one f64 MFMA
// chain over the columns in the order of the tiles (the same bits), operands
// loaded straight from memory kChainAhead groups of 16 columns ahead and
// converted one group ahead (a conversion into registers that an MFMA still
// reads waits for it). No LDS and no barriers, and up to 1024 blocks run one
// chain per SIMD.
constexpr int kChainAhead = 16;

__global__ __launch_bounds__(64) void project_chain_kernel(BlockParams p, int blocks)
{
    const int lane = threadIdx.x;
    const int r16 = lane & 15, kq = lane >> 4;
    // consecutive workgroups go to the 8 XCDs in turn: a row group's token
    // blocks take one XCD, whose L2 then serves its weights
    const int slot = blockIdx.x / 8;
    const int r0 = (slot / blocks * 8 + blockIdx.x % 8) * 16, t0 = slot % blocks * 16;
    if (r0 >= p.out)
        return;
    // rows and tokens past the last repeat it (not written)
    const float *wr = p.w + (int64_t)min(r0 + r16, p.out - 1) * p.in + 4 * kq;
    const float *xr = p.x + (int64_t)min(t0 + r16, p.n - 1) * p.in + 4 * kq;
    const int groups = p.in / 16;

    d4 acc = {0.0, 0.0, 0.0, 0.0};
    double cx[2][4], cw[2][4];
    auto convert = [&](const f4 &x, const f4 &w, int set) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            cx[set][j] = (double)x[j];
            cw[set][j] = (double)w[j];
        }
    };
    // MFMA k slot kq of step j holds column 16 g + 4 kq + j
    auto multiply = [&](int set) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(cx[set][j], cw[set][j], acc, 0, 0, 0);
    };
    if (groups > 0) {
        f4 x[kChainAhead], w[kChainAhead];
        // a group past the last whole one repeats it (not multiplied)
        auto load = [&](int g, int d) {
            const int at = 16 * min(g, groups - 1);
            x[d] = ldg4(xr + at);
            w[d] = ldg4(wr + at);
        };
#pragma unroll
        for (int d = 0; d < kChainAhead; ++d)
            load(d, d);
        convert(x[0], w[0], 0);
        static_assert(kChainAhead % 2 == 0, "a group's operand set by its place in the loop");
        for (int g = 0; g < groups; g += kChainAhead) {
#pragma unroll
            for (int d = 0; d < kChainAhead; ++d) {
                if (g + d < groups) {
                    load(g + d + kChainAhead, d);
                    __builtin_amdgcn_sched_barrier(0);
                    convert(x[(d + 1) % kChainAhead], w[(d + 1) % kChainAhead], (d + 1) & 1);
                    __builtin_amdgcn_sched_barrier(0);
                    multiply(d & 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    }
    if (p.in % 16) {
        f4 x, w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool in = 16 * groups + 4 * kq + e < p.in;
            x[e] = in ? ldg(xr + 16 * groups + e) : 0.f;
            w[e] = in ? ldg(wr + 16 * groups + e) : 0.f;
        }
        convert(x, w, 0);
        multiply(0);
    }
    // element e: token kq + 4e, row r16
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int t = t0 + kq + 4 * e, r = r0 + r16;
        if (t < p.n && r < p.out)
            stg(p.proj + (int64_t)t * p.out + r, (float)acc[e]);
    }
}

template <int TM, int TN, int TK>
static hipError_t launch_tile(const BlockParams &p, hipStream_t stream)
{
    constexpr size_t lds = tile_lds_bytes<TM, TN, TK>();
    static std::atomic<bool> configured[kMaxDevices];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return e;
    if (dev < 0 || dev >= kMaxDevices)
        return hipErrorInvalidDevice;
    if (!configured[dev].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute((const void *)project_tiles_kernel<TM, TN, TK>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess)
            return e;
        configured[dev].store(true, std::memory_order_release);
    }
    const dim3 grid((p.out + TN - 1) / TN, (p.n + TM - 1) / TM);
    project_tiles_kernel<TM, TN, TK><<<grid, 256, lds, stream>>>(p);
    return hipGetLastError();
}

// The tile shapes and their time by the busiest CU's rounds of tiles: every
// K step of a shape costs `fill` once and `round` for each tile the CU works
// (10 ns units, fitted over 33 to 4096 tokens, 64 to 16384 columns and 16 to
// 11264 output rows on one MI355X; columns are whole K steps, so a row of 96
// pays for 128 in the smallest tile).
struct Tile {
    int m, n, k;
    int fill, round;
    hipError_t (*launch)(const BlockParams &, hipStream_t);
};
constexpr Tile kTiles[] = {
    {128, 128, 32, 52, 366, launch_tile<128, 128, 32>},
    {128, 64, 32, 30, 196, launch_tile<128, 64, 32>},
    {64, 64, 64, 38, 201, launch_tile<64, 64, 64>},
    {64, 32, 64, 43, 102, launch_tile<64, 32, 64>},
    {32, 32, 128, 19, 122, launch_tile<32, 32, 128>},
};

// The tile with the least time: 352 tiles of 128 x 128 (2000 tokens, 2816
// rows) cost two rounds for 1.4 rounds of work, and a few tokens leave most
// CUs idle under large tiles, while small ones reach a lower MFMA rate. Of 224
// sizes timed in every shape the choice is 0.6 % from the best on average.
// Projection of 2816 rows of 4096 columns, 128 x 128 alone (its loads
// branching over rows and columns) against the chosen tile: 100 tokens 577 ->
// 85 us, 256 tokens 581 -> 126 us, 1000 tokens 589 -> 421 us, 2000 tokens 1076
// -> 783 us, 4096 tokens 1.62 -> 1.49 ms (0.81 of the fp64 MFMA peak); 2000
// tokens of 96 columns 44 -> 38 us (49 us by a rule without the column count).
static const Tile &choose_tile(int64_t n, int64_t in, int64_t out, int64_t cus)
{
    auto count = [&](int tm, int tn) { return ((out + tn - 1) / tn) * ((n + tm - 1) / tm); };
    // past 8192 tiles of 128 x 128 (32 rounds) a last round is a few percent,
    // and the grids of smaller tiles could leave the launch limits (65535
    // blocks of rows)
    if (count(128, 128) > 8192)
        return kTiles[0];
    auto cost = [&](const Tile &t) {
        const int64_t rounds = (count(t.m, t.n) + cus - 1) / cus;
        return (in + t.k - 1) / t.k * (t.fill + rounds * t.round);
    };
    return *std::min_element(std::begin(kTiles), std::end(kTiles),
                             [&](const Tile &a, const Tile &b) { return cost(a) < cost(b); });
}

// Tokens project_few_kernel takes: from 6 (one wave per row spreads over more
// CUs; 3 tokens 8192 -> 5376 rows of weights 59.7 us there and 71.6 us here,
// 16384 -> 1024 34.0 and 55.8 us, 4096 -> 2816 17.7 and 19.5 us; 5 tokens 4096
// -> 2816 19.8 and 20.0 us; 6 tokens 25.8 and 19.3 us) up to the 32 that two
// 16-token blocks of a workgroup hold. Past 16 tokens each workgroup takes
// both (the weights are read once) unless single blocks fit one round of the
// CUs (2048 x 2048, 32 tokens: 15.5 us in single blocks, 19.0 us in pairs;
// 2816 x 4096: 42.7 us against 35.2 us).
constexpr int kFewFrom = 6, kFewTo = 32;

// Token blocks of a project_few_kernel workgroup.
static int few_blocks(int64_t n, int64_t out, int64_t cus)
{
    const int64_t blocks = (n + 15) / 16;
    return blocks == 1 || blocks * ((out + 15) / 16) <= cus ? 1 : 2;
}

// Whether project_chain_kernel takes n tokens: up to 128 of them while every
// 16 x 16 block is the only chain of its SIMD. Its time is then the chain's,
// where the tiles' K steps add theirs and a half-empty tile of 32 tokens its
// own: 2816 x 4096, weights from HBM, 33 tokens 48.8 us against 52.4 us in tiles
// of 32 x 32, 80 tokens 72 against 85 us; 96 tokens, where some SIMDs take two
// chains, 88 against 84 us (from the last-level cache). Full tiles on more
// than half of the CUs read the weights once for two chains: 64 tokens 55.9
// against 52.1 us. More tokens of few rows crowd the few XCDs that have a row
// group (1024 -> 300, 800 tokens: 29.4 against 22.8 us).
constexpr int kChainTo = 128;

static bool chain_fits(int64_t n, int64_t out, int64_t cus)
{
    const int64_t blocks = (n + 15) / 16;
    const bool full_tiles = blocks % 2 == 0 && 2 * (blocks / 2 * ((out + 31) / 32)) > cus;
    return n <= kChainTo && blocks * ((out + 15) / 16) <= 4 * cus && !full_tiles;
}

hipError_t launch_output_block(const BlockParams &p, hipStream_t stream)
{
    const int cus = std::max(device_cus(), 1);
    if (p.n < kFewFrom) {
        const dim3 grid((p.out + 3) / 4);
        if (p.n == 1 && p.in % 4 == 0 && p.in <= kLdsRowFloats)
            project_row_lds_kernel<<<grid, 256, p.in * 4, stream>>>(p, 0);
        else if (p.n == 1)
            project_rows_kernel<1><<<grid, 256, 0, stream>>>(p);
        else if (p.n == 2)
            project_rows_kernel<2><<<grid, 256, 0, stream>>>(p);
        else if (p.n == 3)
            project_rows_kernel<3><<<grid, 256, 0, stream>>>(p);
        else if (p.n == 4)
            project_rows_kernel<4><<<grid, 256, 0, stream>>>(p);
        else
            project_rows_kernel<5><<<grid, 256, 0, stream>>>(p);
    } else if (p.n <= kFewTo) {
        const int rows = (p.out + 15) / 16;
        if (few_blocks(p.n, p.out, cus) == 1)
            project_few_kernel<1><<<dim3(rows, (p.n + 15) / 16), 64 * kFewWaves, 0, stream>>>(p);
        else
            project_few_kernel<2><<<rows, 64 * kFewWaves, 0, stream>>>(p);
    } else if (chain_fits(p.n, p.out, cus)) {
        const int rows = (p.out + 15) / 16, blocks = (p.n + 15) / 16;
        project_chain_kernel<<<(rows + 7) / 8 * 8 * blocks, 64, 0, stream>>>(p, blocks);
    } else {
        const hipError_t e = choose_tile(p.n, p.in, p.out, cus).launch(p, stream);
        if (e != hipSuccess)
            return e;
    }
    hipLaunchKernelGGL(post_norm_kernel, dim3(p.n), dim3(256), 0, stream, p);
    return hipGetLastError();
}

} // namespace pcl

extern "C" int pcl_attention_output(pcl_context *ctx, const float *attended, int64_t n,
                                    int64_t in, const float *weights, int64_t out,
                                    const float *post_scale, float epsilon,
                                    const float *residual, float *projected, float *result)
{
    if (!ctx || !attended || !weights || !post_scale || !residual || !projected || !result)
        return PCL_INVALID_SHAPE;
    // sizes keep every grid below 2^31 work-items (post-norm: 256 per token)
    if (n <= 0 || in <= 0 || out <= 0 || n > (1 << 22) || in > (1 << 20) || out > (1 << 20))
        return PCL_INVALID_SHAPE;
    if (!(epsilon > 0.0f) || !__builtin_isfinite(epsilon))
        return PCL_INVALID_PARAMETER;
    (void)hipSetDevice(ctx->device);
    pcl::BlockParams p{};
    p.x = attended;
    p.w = weights;
    p.proj = projected;
    p.scale = post_scale;
    p.res = residual;
    p.result = result;
    p.n = (int)n;
    p.in = (int)in;
    p.out = (int)out;
    p.eps = epsilon;
    p.err = ctx->err;
    const hipError_t e = pcl::launch_output_block(p, ctx->stream);
    if (e != hipSuccess) {
        std::fprintf(stderr, "pcl_attention_output: launch: %s\n", hipGetErrorString(e));
        return PCL_NON_FINITE_VALUE;
    }
    return PCL_OK;
}

extern "C" int pcl_debug_projection_form(int64_t n, int64_t in, int64_t out, int cus)
{
    if (n < pcl::kFewFrom)
        return 1;
    if (n <= pcl::kFewTo)
        return 16 * pcl::few_blocks(n, out, cus);
    if (pcl::chain_fits(n, out, std::max(cus, 1)))
        return 16016;
    const pcl::Tile &t = pcl::choose_tile(n, in, out, std::max(cus, 1));
    return 1000 * t.m + t.n;
}
