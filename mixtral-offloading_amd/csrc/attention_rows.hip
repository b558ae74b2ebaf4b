// Causal attention of the new tokens of one sequence over its KV cache (the prompt pass; HF transformers' Mixtral
// attention in the reference).  Grouped-query heads, keys already rotated, one launch: scores, softmax and the weighted
// sum of the values stay in registers, so nothing of size tokens x positions goes through memory.
//
// The rows of one key/value head are (token, query head of its group) pairs, row = token * group + head: a block of four
// waves takes 64 * NQ consecutive ones and walks the positions in steps of 64, keys and values of a step double-buffered
// in LDS and shared by all heads of the group.  Scores are computed transposed, S^T = K Q^T (rows = positions, columns =
// query rows), because the result layout of v_mfma_f32_16x16x32_f16 (four consecutive rows per lane) of two 16-position
// tiles then IS the B operand layout of O^T = V^T P^T: the 32 positions of a product are taken in the order (lane group,
// tile, element), which only asks for V^T to be read from LDS in that order (two 8-byte pieces), and a probability never
// leaves its lane.  A lane's columns are one query row each, so the running maximum and sum are two shuffles a step and
// the rescaling of O is a multiplication by a number of the lane's own.
//
// Scores, maximum, sum and O are fp32; the un-normalised probabilities (0..1) enter the product in fp16, as the
// normalised ones did before.  Bound by the vector units (about fourteen operations a score beside 2 x 16 matrix cycles
// a 16 x 16 tile).  Two query tiles a wave (NQ = 2) halve the LDS reads a product; the shorter blocks (NQ = 1) spread the
// rows further and are the faster form until the longer ones make two blocks a compute unit (32 heads on 8 key/value
// heads, head size 128, NQ = 1 and 2: 1024 tokens 35 and 44 us, 1999: 78 and 86, 2400: 116 and 104, 4000: 269 and 204).
// The library products and the elementwise passes that this replaces took 970 us a layer at 1999 tokens.
#include "hqq_common.hpp"

namespace hqq {
namespace {

constexpr int kRowsThreads = 256;
constexpr int kStep = 64; // positions per step
constexpr int64_t kWideBlocks = 512; // from here on two query tiles a wave: two such blocks a compute unit

struct AttRowsParams {
    const f16 *q;
    const f16 *ck, *cv;
    f16 *out;
    int64_t start, max_len;
    int64_t rows; // tokens * group
    int group, n_heads, n_kv;
    float scale_log2; // log2(e) / sqrt(head size)
};

template <int HD, int NQ> __global__ __launch_bounds__(kRowsThreads, 2) void attention_rows_kernel(AttRowsParams p)
{
    constexpr int KT = HD / 32;           // k steps of a score tile
    constexpr int HT = HD / 16;           // 16-row tiles of O^T
    constexpr int KP = HD + 8;            // pitches that keep 16 rows on different banks
    constexpr int VP = kStep + 4;
    constexpr int CH = HD / 8;            // 16-byte pieces of a row
    constexpr int KR = kRowsThreads / CH; // key rows per load instruction of the block
    constexpr int KL = kStep / KR;
    __shared__ __attribute__((aligned(16))) f16 k_lds[2][kStep][KP];
    __shared__ __attribute__((aligned(16))) f16 v_lds[2][HD][VP]; // transposed
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, grp = lane >> 4;
    const int kv = blockIdx.x % p.n_kv;
    // the last rows see the most positions: they go first
    const int64_t tiles = gridDim.x / p.n_kv, tile = tiles - 1 - blockIdx.x / p.n_kv;
    const int64_t row0 = tile * (64 * NQ), wrow = row0 + wave * (16 * NQ);
    const int64_t last_row = (row0 + 64 * NQ < p.rows ? row0 + 64 * NQ : p.rows) - 1;
    const int64_t len = p.start + last_row / p.group + 1; // positions any row of the block sees
    const int steps = (int)((len + kStep - 1) / kStep);
    // this wave's rows: the positions all of them see, and the last one any of them sees
    const int64_t wlast = wrow + 16 * NQ - 1 < p.rows ? wrow + 16 * NQ - 1 : p.rows - 1;
    const int64_t wfirst = wrow < p.rows ? wrow : p.rows - 1;
    const int64_t full = p.start + wfirst / p.group + 1, seen = p.start + wlast / p.group + 1;

    const f16 *kb = p.ck + (int64_t)kv * p.max_len * HD, *vb = p.cv + (int64_t)kv * p.max_len * HD;
    const int kc = tid % CH, kr = tid / CH;  // key loads: piece, row
    const int vq = tid & 15, vh = tid >> 4;  // value loads: four positions, eight columns
    const bool von = vh < CH;
    f16x8 kreg[KL], vreg[4];
    auto request = [&](int step) {
        const int64_t at = (int64_t)step * kStep;
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            const int64_t r = at + kr + i * KR;
            kreg[i] = *reinterpret_cast<const f16x8 *>(kb + (r < len ? r : len - 1) * HD + kc * 8);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t r = at + vq * 4 + i;
            vreg[i] = *reinterpret_cast<const f16x8 *>(vb + (r < len ? r : len - 1) * HD + (von ? vh : 0) * 8);
        }
    };
    auto deposit = [&](int buf) {
#pragma unroll
        for (int i = 0; i < KL; ++i)
            *reinterpret_cast<f16x8 *>(&k_lds[buf][kr + i * KR][kc * 8]) = kreg[i];
        if (von) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                *reinterpret_cast<f16x4 *>(&v_lds[buf][vh * 8 + e][vq * 4]) =
                    f16x4{vreg[0][e], vreg[1][e], vreg[2][e], vreg[3][e]};
        }
    };

    request(0);
    f16x8 qf[NQ][KT];
    int64_t limit[NQ]; // last position the lane's row sees
#pragma unroll
    for (int t = 0; t < NQ; ++t) {
        const int64_t r0 = wrow + t * 16 + col, r = r0 < p.rows ? r0 : p.rows - 1;
        const int64_t tok = r / p.group;
        limit[t] = p.start + tok;
        const f16 *src = p.q + (tok * p.n_heads + kv * p.group + (r - tok * p.group)) * HD + grp * 8;
#pragma unroll
        for (int k = 0; k < KT; ++k)
            qf[t][k] = *reinterpret_cast<const f16x8 *>(src + k * 32);
    }
    f32x4 acc[NQ][HT];
    float top[NQ], sum[NQ];
#pragma unroll
    for (int t = 0; t < NQ; ++t) {
        top[t] = -__builtin_inff();
        sum[t] = 0.f;
#pragma unroll
        for (int h = 0; h < HT; ++h)
            acc[t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    deposit(0);
    __syncthreads();
    for (int step = 0; step < steps; ++step) {
        const int buf = step & 1;
        const bool more = step + 1 < steps;
        if (more)
            request(step + 1);
        const int64_t at = (int64_t)step * kStep;
        if (at < seen) {
            f32x4 s[NQ][4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
#pragma unroll
                for (int t = 0; t < NQ; ++t)
                    s[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < KT; ++k) {
                    const f16x8 kf = *reinterpret_cast<const f16x8 *>(&k_lds[buf][c * 16 + col][k * 32 + grp * 8]);
#pragma unroll
                    for (int t = 0; t < NQ; ++t)
                        s[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[t][k], s[t][c], 0, 0, 0);
                }
            }
            if (at + kStep > full) { // some row of the wave does not see all of the step
#pragma unroll
                for (int t = 0; t < NQ; ++t) {
                    const int upto = limit[t] - at < kStep ? (int)(limit[t] - at) : kStep;
#pragma unroll
                    for (int c = 0; c < 4; ++c)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            s[t][c][i] = c * 16 + grp * 4 + i <= upto ? s[t][c][i] : -__builtin_inff();
                }
            }
            f16x8 pf[NQ][2];
#pragma unroll
            for (int t = 0; t < NQ; ++t) {
                float m = s[t][0][0];
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        m = __builtin_fmaxf(m, s[t][c][i]);
                m = __builtin_fmaxf(m, __shfl_xor(m, 16, 64));
                m = __builtin_fmaxf(m, __shfl_xor(m, 32, 64));
                m = __builtin_fmaxf(m, top[t]);
                if (__any(m != top[t])) {
                    // (nothing but -inf so far: the exponents below stay -inf, and the weights zero)
                    const float from = top[t] == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((top[t] - m) * p.scale_log2);
                    sum[t] *= from;
#pragma unroll
                    for (int h = 0; h < HT; ++h)
                        acc[t][h] *= from;
                    top[t] = m;
                }
                const float off = m == -__builtin_inff() ? 0.f : m * p.scale_log2;
                float part = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][c][i], p.scale_log2, -off));
                        part += e;
                        pf[t][c >> 1][(c & 1) * 4 + i] = (f16)e;
                    }
                sum[t] += part;
            }
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int h = 0; h < HT; ++h) {
                    const f16 *src = &v_lds[buf][h * 16 + col][c * 32 + grp * 4];
                    const f16x4 lo = *reinterpret_cast<const f16x4 *>(src), hi = *reinterpret_cast<const f16x4 *>(src + 16);
                    const f16x8 vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                    for (int t = 0; t < NQ; ++t)
                        acc[t][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf[t][c], acc[t][h], 0, 0, 0);
                }
        }
        if (more)
            deposit(buf ^ 1); // last read before the barrier that ended the step before this one
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < NQ; ++t) {
        float l = sum[t];
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        const float inv = 1.0f / l;
        const int64_t r = wrow + t * 16 + col;
        if (r < p.rows) {
            const int64_t tok = r / p.group;
            f16 *dst = p.out + (tok * p.n_heads + kv * p.group + (r - tok * p.group)) * HD + grp * 4;
#pragma unroll
            for (int h = 0; h < HT; ++h)
                *reinterpret_cast<f16x4 *>(dst + h * 16) = f16x4{(f16)(acc[t][h][0] * inv), (f16)(acc[t][h][1] * inv),
                                                                (f16)(acc[t][h][2] * inv), (f16)(acc[t][h][3] * inv)};
        }
    }
}

template <int HD> int run_rows(const AttRowsParams &p, hipStream_t s)
{
    const int64_t wide = (p.rows + 127) / 128 * p.n_kv, narrow = (p.rows + 63) / 64 * p.n_kv;
    if (narrow > 0x7fffffff)
        return HQQ_E_SHAPE;
    if (wide >= kWideBlocks)
        attention_rows_kernel<HD, 2><<<(unsigned)wide, kRowsThreads, 0, s>>>(p);
    else
        attention_rows_kernel<HD, 1><<<(unsigned)narrow, kRowsThreads, 0, s>>>(p);
    return launch_status();
}

} // namespace

int launch_attention_rows(const f16 *q, const f16 *cache_k, const f16 *cache_v, int64_t start, int64_t tokens, int64_t max_len,
                          int n_heads, int n_kv, int head_dim, f16 *out, hipStream_t s)
{
    if ((head_dim != 64 && head_dim != 128) || n_kv < 1 || n_heads < n_kv || n_heads % n_kv != 0 || tokens < 1 || start < 0 ||
        start + tokens > max_len || max_len > 0x7fffffff)
        return HQQ_E_SHAPE;
    if (!aligned16(q) || !aligned16(cache_k) || !aligned16(cache_v) || !aligned16(out))
        return HQQ_E_ALIGN;
    AttRowsParams p = {};
    p.q = q, p.ck = cache_k, p.cv = cache_v, p.out = out;
    p.start = start, p.max_len = max_len;
    p.group = n_heads / n_kv, p.n_heads = n_heads, p.n_kv = n_kv;
    p.rows = tokens * p.group;
    p.scale_log2 = (float)(1.4426950408889634 / __builtin_sqrt((double)head_dim));
    return head_dim == 128 ? run_rows<128>(p, s) : run_rows<64>(p, s);
}

} // namespace hqq
