// HQQ's quantiser (hqq Quantizer.quantize / optimize_weights, called at src/custom_layers.py:35-39 and
// src/build_model.py:108-120) for the grouping this path uses: the tensor seen as a row-major (rows, cols) matrix
// whose COLUMNS are the groups (axis 0: rows = group size, cols = N*K / group size), and the one-group form used for
// the zero table's 8-bit meta (min and max over the whole tensor).
//
//   scale = min((2^b - 1) / (max - min), 2e4),  zero = -min * scale  (rounded when asked),
//   optionally refined by the half-quadratic solver (shrinkage of the residual in the l_p norm, p < 1, and the
//   closed-form zero update, beta growing by kappa per iteration, stopped by the mean absolute error of the whole
//   tensor),  q = clamp(round(w * scale + zero), 0, 2^b - 1),  outputs q, 1 / scale, zero.
//
// One thread owns CP neighbouring groups (4, 2 or 1, by what the registers hold) and keeps their values in registers,
// so every iteration of the solver is register arithmetic; consecutive threads read consecutive pieces of a row, so
// every row is a coalesced streaming read of 4 to 16 bytes per thread.  The solver
// stops for the WHOLE tensor at once: passes of kQChunk iterations add up the error of every iteration (fp64 atomics,
// on several sums side by side) and leave the zero points they reached in one of the two output vectors (the next pass reads it and writes the
// other, so both ends of a pass are at hand); every block of a later pass finds from the errors so far whether the
// host loop would have stopped, and returns if so; the last pass repeats the iterations of the one pass the stop fell
// into and writes the result.  All arithmetic is fp32 with separate multiplies and adds, as the tensor ops it replaces;
// only the quotients in the errors that decide the stop are made another way (divide_by).
//
// An iteration is a dozen operations a value.  It was over a hundred: the shrinkage's power took most of them and a full
// division the next, and all iterations ran before the stop was looked for.  The power is evaluated only where its term
// can be other than zero (shrink_skip), the division is a product by the reciprocal in two floats (divide_by; sixteen
// operations a value with a correction by the residual, 614 -> 576 us), and the blocks' error sums do not queue for one
// line of memory (kQSums; 576 -> 510 us).  Registers set how many waves share a unit: sums that the compiler moved past a
// branch kept two values of every weight alive with it (16 x 4 values a thread: 156 -> 113 registers, four waves for
// three, 510 -> 462 us; 64 x 2: 496 -> 215, two waves for one, 3-bit 1876 -> 1057 us and 4-bit 1863 -> 1047 us by all
// three steps).  Times are of a 14336 x 4096 layer, taken to 2 bits in groups of 16 where nothing else is said and then
// stopped within the third of five passes; that one began at 2238 us, with the same bits.
//
// What bounds it, by counters: in groups of 16 the vector units, whose instructions (50.6 M, four cycles each, on 1024
// units) are 87 to 98 % of a pass of 86 to 98 us.  In groups of 64, with two waves to a unit, they are 49 % of 157 us, and
// a wave waits for 54 % of its time: its 128 values arrive before it begins, and one other wave is there to cover that
// (the same reads and no iteration: 67 us).
#include "hqq_common.hpp"

#include <cmath>

namespace hqq {
namespace {

constexpr int kQThreads = 256;
constexpr int kQMaxIters = 64;
constexpr int kQChunk = 4; // iterations between two looks at the stop: a pass more costs one read of the tensor
// Sums of an iteration's error, blocks taking them in turn: atomics on one line follow each other at some 10 ns, so that
// on a single sum the four of each of 3584 blocks (58.7 M values) take longer than the pass's arithmetic.  But every block
// of every pass reads all sums, so a tensor of few blocks takes one for 32 of its blocks (groups of 8, 20 iterations, us
// with one sum / 32 blocks a sum / 32 sums: 16 blocks 33.5 / 33.5 / 40.0, 256 blocks 56.0 / 38.4 / 41.0, 1024 blocks
// 138.6 / 58.6 / 58.6; groups of 16 and 64 alike).
constexpr int kQSums = 32;
constexpr int kQBlocksPerSum = 32;

struct QuantParams {
    const void *w;
    int fp32_in;
    int64_t rows, cols;
    float max_v;
    int round_zero;
    int iters;
    float lp;
    uint8_t *codes;   // (rows, cols)
    float *inv_scale; // (cols)
    float *zero;      // (cols)
    double *err;      // [sums][kQMaxIters]: |w - w_r| added up per iteration, each block in one of the sums
    int sums;         // as many as the workspace has room for; launched with no more than the blocks are worth
    int first;        // solver pass: its first iteration
    float skip;       // shrink_skip(): residuals up to this one shrink to zero
    float inv_beta[kQMaxIters]; // 1 / beta of every iteration
};

// CP consecutive values starting at element `at` (a multiple of CP)
template <int CP> __device__ __forceinline__ void load_w(const QuantParams &p, int64_t at, float (&out)[CP])
{
    if (p.fp32_in) {
        typedef float vec __attribute__((ext_vector_type(CP)));
        const vec v = *reinterpret_cast<const vec *>(static_cast<const float *>(p.w) + at);
#pragma unroll
        for (int j = 0; j < CP; ++j)
            out[j] = CP == 1 ? reinterpret_cast<const float *>(&v)[0] : v[j];
    } else {
        typedef _Float16 vec __attribute__((ext_vector_type(CP)));
        const vec v = *reinterpret_cast<const vec *>(static_cast<const f16 *>(p.w) + at);
#pragma unroll
        for (int j = 0; j < CP; ++j)
            out[j] = (float)(CP == 1 ? reinterpret_cast<const f16 *>(&v)[0] : v[j]);
    }
}

// sign(x) * relu(|x| - (1 / beta) * (|x| + 1e-8)^(p - 1))
__device__ __forceinline__ float shrink_lp(float x, float inv_beta, float pm1)
{
    const float a = __builtin_fabsf(x);
    const float t = a - inv_beta * __builtin_powf(a + 1e-8f, pm1);
    const float r = t > 0.f ? t : 0.f;
    return x > 0.f ? r : (x < 0.f ? -r : 0.f);
}

// x / s from 1 / s as the sum hi + lo of two floats.  The sum is within 2^-46 of 1 / s, so before its one rounding the
// quotient is within 2^-45 of its size: it is rounded as a division rounds it unless it lies that near the middle
// between two floats, and then to the other of two neighbours that are as good as equally far (25 of 8 * 10^9 quotients
// of this kind, off by 0.50000004 of an ulp at most; the mean error is a division's, 0.25 ulp).  Two operations, where
// correcting x * hi by the exact residual takes five.  Only the errors that decide the stop are made with it; neither
// zero points nor codes are.  For |s| and |x| where nothing leaves the normal range: see divide_safe.
__device__ __forceinline__ float divide_by(float x, float hi, float lo) { return __builtin_fmaf(x, hi, x * lo); }
// x = q - zero with q whole: zero itself, or not below the distance of neighbouring floats around a whole number
// (2^-24, or 2^-40 where zero is that small); hi above 2^-40 and lo, if not 0, above 2^-48 of it leave x * lo above
// 2^-128, 2^-48 of the quotient, where a denormal result still has all the bits that count
__device__ __forceinline__ bool divide_safe(float scale, float zero)
{
    const float a = __builtin_fabsf(zero);
    return scale > 0x1p-40f && scale < 0x1p40f && (a == 0.f || (a > 0x1p-40f && a < 0x1p40f));
}

// One iteration of the solver on a column: its zero point moves, its error is returned.  The plain sums are made again
// with divisions and the shrinkage in them where a lane of the wave may need either.
template <int GS, int CP>
__device__ __forceinline__ float solver_step(const QuantParams &p, const float (&w)[GS][CP], int j, float scale, float hi,
                                             float lo, float inv_beta, float &zero)
{
    float e = 0.f, acc = 0.f, top = 0.f;
#pragma unroll
    for (int r = 0; r < GS; ++r) {
        const float ws = w[r][j] * scale;
        // the middle of the three is the clamped value in one operation (0 for a NaN, as of the two)
        const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(ws + zero), 0.f, p.max_v);
        const float a = __builtin_fabsf(w[r][j] - divide_by(q - zero, hi, lo));
        e += a;
        top = __builtin_fmaxf(top, a);
        acc += q - ws;
        if (r % 16 == 15 || r == GS - 1) {
            // the sums are made here, not past the branch below, where every q and ws would have to be kept until then
            asm volatile("" : "+v"(e), "+v"(acc), "+v"(top));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (__any(top > p.skip || !divide_safe(scale, zero))) {
        const float pm1 = p.lp - 1.0f;
        e = 0.f, acc = 0.f;
#pragma unroll
        for (int r = 0; r < GS; ++r) {
            float q = __builtin_rintf(w[r][j] * scale + zero);
            q = __builtin_fminf(__builtin_fmaxf(q, 0.f), p.max_v);
            const float d = w[r][j] - (q - zero) / scale;
            e += __builtin_fabsf(d);
            const float we = shrink_lp(d, inv_beta, pm1);
            acc += q - (w[r][j] - we) * scale;
            __builtin_amdgcn_sched_barrier(0); // one power at a time: interleaved, their registers spill
        }
    }
    zero = acc / (float)GS;
    return e;
}

// The iteration count of the host loop, from the errors of its first `known` iterations: it updates zero, then stops at
// the first iteration whose error (taken before the update) is not below the best so far.  0: not stopped yet.  All
// threads of the block call it.
__device__ __forceinline__ int solver_stop(const QuantParams &p, int known)
{
    static_assert(kQMaxIters == 64, "a wave's lanes are the iterations");
    __shared__ double part[kQThreads / 64][kQMaxIters];
    __shared__ float mean[kQMaxIters];
    __shared__ int stop;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane < known) {
        double t = 0.0;
        for (int i = wave; i < p.sums; i += kQThreads / 64)
            t += p.err[i * kQMaxIters + lane];
        part[wave][lane] = t;
    }
    __syncthreads();
    if ((int)threadIdx.x < known) {
        double t = 0.0;
#pragma unroll
        for (int i = 0; i < kQThreads / 64; ++i)
            t += part[i][threadIdx.x];
        mean[threadIdx.x] = (float)(t / ((double)p.rows * (double)p.cols));
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float best = 1e4f;
        int n = 0;
        for (int it = 0; it < known && n == 0; ++it) {
            if (mean[it] < best)
                best = mean[it];
            else
                n = it + 1;
        }
        stop = n;
    }
    __syncthreads();
    return stop;
}

// PASS 0: no refinement, write the result.  PASS 1: kQChunk iterations of the solver from p.first on, their errors added
// up, unless an earlier one was the last.  PASS 2: the iterations that count of the pass the stop fell into, the result.
template <int GS, int CP, int PASS> __global__ __launch_bounds__(kQThreads) void quantize_groups_kernel(QuantParams p)
{
    const int64_t c = ((int64_t)blockIdx.x * kQThreads + threadIdx.x) * CP; // first group of the thread
    const bool on = c < p.cols;
    const int64_t cc = on ? c : p.cols - CP;
    int first = 0, last = 0;
    if constexpr (PASS == 1) {
        if (p.first > 0 && solver_stop(p, p.first) != 0)
            return;
        first = p.first;
        last = first + kQChunk < p.iters ? first + kQChunk : p.iters;
    } else if constexpr (PASS == 2) {
        last = solver_stop(p, p.iters);
        last = last ? last : p.iters;
        first = (last - 1) / kQChunk * kQChunk;
    }
    float w[GS][CP];
#pragma unroll
    for (int r = 0; r < GS; ++r)
        load_w<CP>(p, (int64_t)r * p.cols + cc, w[r]);
    float scale[CP], zero[CP];
#pragma unroll
    for (int j = 0; j < CP; ++j) {
        float mn = w[0][j], mx = w[0][j];
#pragma unroll
        for (int r = 1; r < GS; ++r) {
            mn = __builtin_fminf(mn, w[r][j]);
            mx = __builtin_fmaxf(mx, w[r][j]);
        }
        float sc = p.max_v / (mx - mn);
        scale[j] = sc < 2e4f ? sc : 2e4f; // (a constant group gives inf, clamped like any other large value)
        zero[j] = -mn * scale[j];
        if (p.round_zero)
            zero[j] = __builtin_rintf(zero[j]);
    }
    if constexpr (PASS != 0) {
        // the pass at iteration f finds its zero points in p.zero if f / kQChunk is odd, in p.inv_scale if it is even
        // (and not 0), and leaves them in the other one
        const bool odd = (first / kQChunk) & 1;
        if (first > 0) {
            const float *from = odd ? p.zero : p.inv_scale;
#pragma unroll
            for (int j = 0; j < CP; ++j)
                zero[j] = from[cc + j];
        }
        __shared__ float err_lds[kQChunk][kQThreads];
        float hi[CP], lo[CP]; // 1 / scale
#pragma unroll
        for (int j = 0; j < CP; ++j) {
            hi[j] = 1.0f / scale[j];
            lo[j] = __builtin_fmaf(-scale[j], hi[j], 1.0f) * hi[j];
        }
#pragma unroll 1
        for (int it = first; it < last; ++it) {
            const float inv_beta = p.inv_beta[it];
            float e = 0.f;
#pragma unroll
            for (int j = 0; j < CP; ++j) {
                float sc = scale[j];
                asm volatile("" : "+v"(sc)); // keeps w * scale out of registers of its own across iterations
                e += solver_step<GS, CP>(p, w, j, sc, hi[j], lo[j], inv_beta, zero[j]);
            }
            if constexpr (PASS == 1)
                err_lds[it - first][threadIdx.x] = on ? e : 0.f;
        }
        if constexpr (PASS == 1) {
            // the block's errors, one wave an iteration, once all iterations are through: none waits for lane exchanges
            __syncthreads();
            const int lane = threadIdx.x & 63;
            for (int it = threadIdx.x >> 6; it < last - first; it += kQThreads / 64) {
                double t = 0.0;
#pragma unroll
                for (int i = 0; i < kQThreads / 64; ++i)
                    t += (double)err_lds[it][64 * i + lane];
#pragma unroll
                for (int off = 32; off > 0; off >>= 1)
                    t += __shfl_xor(t, off, 64);
                if (lane == 0)
                    atomicAdd(&p.err[(int)(blockIdx.x % (unsigned)p.sums) * kQMaxIters + first + it], t);
            }
            if (on) {
                float *to = odd ? p.inv_scale : p.zero;
#pragma unroll
                for (int j = 0; j < CP; ++j)
                    to[c + j] = zero[j];
            }
        }
    }
    if constexpr (PASS != 1) {
        if (on) {
            typedef uint8_t bvec __attribute__((ext_vector_type(CP)));
#pragma unroll
            for (int r = 0; r < GS; ++r) {
                uint8_t qb[CP];
#pragma unroll
                for (int j = 0; j < CP; ++j) {
                    float q = __builtin_rintf(w[r][j] * scale[j] + zero[j]);
                    q = __builtin_fminf(__builtin_fmaxf(q, 0.f), p.max_v);
                    qb[j] = (uint8_t)q;
                }
                if constexpr (CP == 1) {
                    p.codes[(int64_t)r * p.cols + c] = qb[0];
                } else {
                    bvec v;
#pragma unroll
                    for (int j = 0; j < CP; ++j)
                        v[j] = qb[j];
                    *reinterpret_cast<bvec *>(p.codes + (int64_t)r * p.cols + c) = v;
                }
            }
#pragma unroll
            for (int j = 0; j < CP; ++j) {
                p.inv_scale[c + j] = 1.0f / scale[j];
                p.zero[c + j] = zero[j];
            }
        }
    }
}

__global__ __launch_bounds__(kQThreads) void quantize_clear_kernel(double *err, int n)
{
    for (int i = threadIdx.x; i < n; i += kQThreads)
        err[i] = 0.0;
}

// The largest residual a of which it is certain that a - (1 / beta) (a + 1e-8)^(p - 1) is not positive, in whatever
// iteration: the difference grows with a and is zero at a = (1 / beta)^(1 / (2 - p)) but for the 1e-8; two per cent below
// that it is negative by more than two per cent of a, a thousand times what the 1e-8 and the roundings can add.
// (p = 0.7, 1 / beta = 0.1: 0.14.)  The kernel compares the residuals themselves, and a wave with a larger one takes the
// power.  Weights of a spread of 0.02 stay far below, although clamped codes, a moved zero point and, at 4 bits, its
// rounding leave residuals of up to 0.6 (3-bit) or 0.9 (4-bit) of a step there; a group that an outlier gives steps of
// some 0.15 to 0.3 need not.
static float shrink_skip(double beta, double kappa, int iters, float lp)
{
    const double last = beta * std::pow(kappa, (double)iters), most = last > beta ? last : beta;
    if (!(lp >= 0.0f && lp <= 1.0f) || !(beta > 0) || !(last > 0) || !(most < 1e30))
        return -1.0f; // never skipped
    const double at = 0.98 * std::pow(1.0 / most, 1.0 / (2.0 - (double)lp));
    return at > 1e-4 ? (float)at : -1.0f;
}

// One group for the whole tensor (channel_wise = False).  Three launches: the extremes are cleared, every block
// folds its share of the tensor into them (floats ordered as integers, so that integer atomics find min and max),
// then every element is coded.
__device__ __forceinline__ int ordered(float v) // monotonic map of fp32 onto int32
{
    const int b = __builtin_bit_cast(int, v);
    return b >= 0 ? b : b ^ 0x7fffffff;
}
__device__ __forceinline__ float unordered(int o) { return __builtin_bit_cast(float, o >= 0 ? o : o ^ 0x7fffffff); }

__global__ void whole_clear_kernel(int *extremes)
{
    extremes[0] = 0x7fffffff; // min
    extremes[1] = (int)0x80000000; // max
}

// Four 16-byte loads a thread and trip where the pointer allows, and few blocks: with one 4-byte load a trip and a block
// per 2048 values the blocks' atomics on the two words, not the reading, took the time (3.7 M values: 44.5 -> 9.4 us).
__global__ __launch_bounds__(256) void whole_extremes_kernel(const float *x, int64_t n, int *extremes)
{
    typedef float vec4 __attribute__((ext_vector_type(4)));
    __shared__ float mn_s[4], mx_s[4];
    const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
    float mn = x[first < n ? first : 0], mx = mn;
    const int64_t quads = (reinterpret_cast<uintptr_t>(x) & 15u) == 0 ? n / 4 : 0;
    const vec4 *xv = reinterpret_cast<const vec4 *>(x);
    for (int64_t i = first; i < quads; i += 4 * stride) {
        vec4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            v[u] = xv[i + u * stride < quads ? i + u * stride : i];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                mn = __builtin_fminf(mn, v[u][e]);
                mx = __builtin_fmaxf(mx, v[u][e]);
            }
    }
    for (int64_t i = 4 * quads + first; i < n; i += stride) {
        mn = __builtin_fminf(mn, x[i]);
        mx = __builtin_fmaxf(mx, x[i]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        mn = __builtin_fminf(mn, __shfl_xor(mn, off, 64));
        mx = __builtin_fmaxf(mx, __shfl_xor(mx, off, 64));
    }
    if ((threadIdx.x & 63) == 0)
        mn_s[threadIdx.x >> 6] = mn, mx_s[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 4; ++i) {
            mn = __builtin_fminf(mn, mn_s[i]);
            mx = __builtin_fmaxf(mx, mx_s[i]);
        }
        atomicMin(&extremes[0], ordered(mn));
        atomicMax(&extremes[1], ordered(mx));
    }
}

__global__ __launch_bounds__(256) void whole_codes_kernel(const float *x, int64_t n, float max_v, const int *extremes,
                                                          uint8_t *codes, float *inv_scale, float *zero_out)
{
    const float mn = unordered(extremes[0]), mx = unordered(extremes[1]);
    float scale = max_v / (mx - mn);
    scale = scale < 2e4f ? scale : 2e4f;
    const float zero = -mn * scale;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        float q = __builtin_rintf(x[i] * scale + zero);
        q = __builtin_fminf(__builtin_fmaxf(q, 0.f), max_v);
        codes[i] = (uint8_t)q;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *inv_scale = 1.0f / scale;
        *zero_out = zero;
    }
}

template <int GS, int CP> int run_groups_cp(const QuantParams &p, hipStream_t s)
{
    const int64_t per_block = (int64_t)kQThreads * CP;
    const unsigned blocks = (unsigned)((p.cols + per_block - 1) / per_block);
    if (p.iters == 0) {
        quantize_groups_kernel<GS, CP, 0><<<blocks, kQThreads, 0, s>>>(p);
        return launch_status();
    }
    QuantParams q = p;
    const int worth = blocks / kQBlocksPerSum > 0 ? (int)(blocks / kQBlocksPerSum) : 1;
    q.sums = worth < p.sums ? worth : p.sums;
    quantize_clear_kernel<<<1, kQThreads, 0, s>>>(q.err, q.sums * kQMaxIters);
    for (q.first = 0; q.first < p.iters; q.first += kQChunk)
        quantize_groups_kernel<GS, CP, 1><<<blocks, kQThreads, 0, s>>>(q);
    quantize_groups_kernel<GS, CP, 2><<<blocks, kQThreads, 0, s>>>(q);
    return launch_status();
}

// groups per thread: as many as GS * CP values fit the registers, the column count and the pointers' alignment allow
template <int GS> int run_groups(const QuantParams &p, hipStream_t s)
{
    const int elem = p.fp32_in ? 4 : 2;
    auto fits = [&](int cp) {
        return p.cols % cp == 0 && (reinterpret_cast<uintptr_t>(p.w) % (size_t)(cp * elem)) == 0 &&
               (reinterpret_cast<uintptr_t>(p.codes) % (size_t)cp) == 0;
    };
    if constexpr (GS <= 32) {
        if (fits(4))
            return run_groups_cp<GS, 4>(p, s);
    }
    if constexpr (GS <= 64) {
        if (fits(2))
            return run_groups_cp<GS, 2>(p, s);
    }
    return run_groups_cp<GS, 1>(p, s);
}

} // namespace

constexpr size_t kQSumBytes = kQMaxIters * sizeof(double); // an iteration's words in the sums lie four lines of memory apart
size_t quantize_workspace_bytes() { return kQSums * kQSumBytes + 64; }

int launch_quantize_groups(const void *w, int fp32_in, int64_t rows, int64_t cols, int nbits, int round_zero, int iters,
                           float lp, double beta, double kappa, uint8_t *codes, float *inv_scale, float *zero, void *ws,
                           size_t ws_bytes, hipStream_t s)
{
    if (rows < 1 || cols < 1 || nbits < 1 || nbits > 8 || iters < 0 || iters > kQMaxIters)
        return HQQ_E_SHAPE;
    if (cols >= (1ll << 31) * (int64_t)kQThreads)
        return HQQ_E_UNSUPPORTED;
    // (one sum is enough to go on with)
    if (iters > 0 && (!ws || ws_bytes < kQSumBytes + 64 || (reinterpret_cast<uintptr_t>(ws) & 7u)))
        return HQQ_E_WORKSPACE;
    QuantParams p = {};
    p.w = w, p.fp32_in = fp32_in, p.rows = rows, p.cols = cols;
    p.max_v = (float)((1 << nbits) - 1), p.round_zero = round_zero, p.iters = iters;
    p.lp = lp;
    double b = beta; // the host loop keeps beta as a double and hands 1 / beta to fp32 tensor ops
    for (int it = 0; it < iters; ++it, b *= kappa)
        p.inv_beta[it] = (float)(1.0 / b);
    p.codes = codes, p.inv_scale = inv_scale, p.zero = zero;
    p.err = static_cast<double *>(ws);
    const size_t room = (ws_bytes - (iters > 0 ? 64 : 0)) / kQSumBytes;
    p.sums = room < (size_t)kQSums ? (int)room : kQSums;
    p.skip = shrink_skip(beta, kappa, iters, lp);
    switch (rows) {
    case 8: return run_groups<8>(p, s);
    case 16: return run_groups<16>(p, s);
    case 32: return run_groups<32>(p, s);
    case 64: return run_groups<64>(p, s);
    case 128: return run_groups<128>(p, s);
    default: return HQQ_E_UNSUPPORTED; // group sizes of the reference's configurations and of the 8-bit meta tables
    }
}

int launch_quantize_whole(const float *x, int64_t n, int nbits, uint8_t *codes, float *inv_scale, float *zero, void *ws,
                          size_t ws_bytes, hipStream_t s)
{
    if (n < 1 || nbits < 1 || nbits > 8)
        return HQQ_E_SHAPE;
    if (!ws || ws_bytes < kQSumBytes + 64 || (reinterpret_cast<uintptr_t>(ws) & 7u))
        return HQQ_E_WORKSPACE;
    int *extremes = static_cast<int *>(ws);
    int64_t blocks = (n + 256 * 8 - 1) / (256 * 8);
    blocks = blocks < 1 ? 1 : (blocks > 2048 ? 2048 : blocks);
    whole_clear_kernel<<<1, 1, 0, s>>>(extremes);
    const int64_t few = blocks < 256 ? blocks : 256;
    whole_extremes_kernel<<<(unsigned)few, 256, 0, s>>>(x, n, extremes);
    whole_codes_kernel<<<(unsigned)blocks, 256, 0, s>>>(x, n, (float)((1 << nbits) - 1), extremes, codes, inv_scale, zero);
    return launch_status();
}

} // namespace hqq
