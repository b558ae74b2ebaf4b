// Causal attention of the new tokens of one sequence over its KV cache (the prompt pass; HF transformers' Mixtral
// attention in the reference).  Grouped-query heads, keys already rotated, one launch: scores, softmax and the weighted
// sum of the values stay in registers, so nothing of size tokens x positions goes through memory.  Few tokens behind a
// long cache take a second launch, which adds up the shares of blocks that each walked a part of the positions (rows_split).
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
// normalised ones did before.  Products that round the scores to fp16 first are off from 64 bits by more in every case
// measured (2 to 2100 tokens behind 0 to 4000 positions, scores of a spread of 0.3 to 4): this form's error is 0.97 to
// 0.11 of theirs, the less the larger the scores.
// Bound by the chain of a step with two blocks a compute unit (70 KB of LDS each): by the counters at 1999 tokens the
// matrix cores are busy for 17 % of the launch, the vector units issue in 36 %, the LDS works in 44 % (a fifth of that
// bank conflicts), and a wave waits on a load, the LDS or the barrier for half of its time.
// Two query tiles a wave (NQ = 2) halve the LDS reads a product; the shorter blocks (NQ = 1) spread the
// rows further and are the faster form until the longer ones make two blocks a compute unit (32 heads on 8 key/value
// heads, head size 128, NQ = 1 and 2: 1024 tokens 35 and 44 us, 1999: 78 and 86, 2400: 116 and 104, 4000: 269 and 204).
// The library products and the elementwise passes that this replaces took 970 us a layer at 1999 tokens.
#include "hqq_common.hpp"

namespace hqq {
namespace {

constexpr int kRowsThreads = 256;
constexpr int kStep = 64; // positions per step
constexpr int64_t kWideBlocks = 512; // from here on two query tiles a wave: two such blocks a compute unit
constexpr int64_t kMaxParts = 256; // of the positions (rows_split)

using f32x2 = float __attribute__((ext_vector_type(2)));

struct AttRowsParams {
    const f16 *q;
    const f16 *ck, *cv;
    f16 *out;
    int64_t start, max_len;
    int64_t rows; // tokens * group
    int group, n_heads, n_kv;
    float scale_log2; // log2(e) / sqrt(head size)
    // positions over several blocks (SPLIT): part s takes the steps s * chunk .. (s + 1) * chunk - 1
    int64_t tiles;
    int chunk;
    float *part; // [parts][n_kv * rows][HD] un-normalised outputs, then [parts][n_kv * rows] (maximum, sum)
    f32x2 *part_ml;
};

template <int HD, int NQ, bool SPLIT> __global__ __launch_bounds__(kRowsThreads, 2) void attention_rows_kernel(AttRowsParams p)
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
    const int64_t tiles = SPLIT ? p.tiles : gridDim.x / p.n_kv;
    const int64_t nth = blockIdx.x / p.n_kv, part_no = SPLIT ? nth / tiles : 0, tile = tiles - 1 - (nth - part_no * tiles);
    const int64_t row0 = tile * (64 * NQ), wrow = row0 + wave * (16 * NQ);
    const int64_t last_row = (row0 + 64 * NQ < p.rows ? row0 + 64 * NQ : p.rows) - 1;
    const int64_t len = p.start + last_row / p.group + 1; // positions any row of the block sees
    int first = 0, steps = (int)((len + kStep - 1) / kStep);
    if constexpr (SPLIT) {
        first = (int)part_no * p.chunk;
        if (first >= steps) // the whole block: none of its rows sees a position of this part
            return;
        steps = steps < first + p.chunk ? steps : first + p.chunk;
    }
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

    request(first);
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
    for (int step = first; step < steps; ++step) {
        const int buf = (step - first) & 1;
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
        const int64_t r = wrow + t * 16 + col;
        if constexpr (SPLIT) {
            if (r < p.rows) {
                const int64_t at = (part_no * p.n_kv + kv) * p.rows + r;
                if (grp == 0)
                    p.part_ml[at] = f32x2{top[t], l};
#pragma unroll
                for (int h = 0; h < HT; ++h)
                    *reinterpret_cast<f32x4 *>(p.part + at * HD + h * 16 + grp * 4) = acc[t][h];
            }
            continue;
        }
        const float inv = 1.0f / l;
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

// The parts of a row put together in the order of the positions: the weight of a part is exp2 of the distance of its
// maximum to the row's.  HD / 4 threads a row; what a part has not seen (it starts behind the row's block) is not read.
template <int HD> __global__ __launch_bounds__(kRowsThreads) void attention_rows_combine_kernel(AttRowsParams p)
{
    constexpr int LPR = HD / 4, RPB = kRowsThreads / LPR;
    __shared__ float w_lds[RPB][kMaxParts];
    const int64_t all = (int64_t)p.n_kv * p.rows;
    const int sub = threadIdx.x / LPR, lane = threadIdx.x % LPR;
    const int64_t row = (int64_t)blockIdx.x * RPB + sub, rr = row < all ? row : all - 1;
    const int64_t kv = rr / p.rows, r = rr - kv * p.rows, tok = r / p.group;
    const int64_t block_end = (r / 64 + 1) * 64 < p.rows ? (r / 64 + 1) * 64 : p.rows;
    const int64_t len = p.start + (block_end - 1) / p.group + 1; // positions the row's block walked
    const int parts = (int)(((len + kStep - 1) / kStep + p.chunk - 1) / p.chunk);
    float m = -__builtin_inff();
    for (int s = lane; s < parts; s += LPR)
        m = __builtin_fmaxf(m, p.part_ml[s * all + rr][0]);
#pragma unroll
    for (int d = LPR / 2; d; d >>= 1)
        m = __builtin_fmaxf(m, __shfl_xor(m, d, LPR));
    float l = 0.f;
    for (int s = lane; s < parts; s += LPR) {
        const f32x2 ml = p.part_ml[s * all + rr];
        // (nothing above -inf in the part: its sum and outputs are zero, or NaN, which the product keeps)
        const float w = ml[0] == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((ml[0] - m) * p.scale_log2);
        w_lds[sub][s] = w;
        l += w * ml[1];
    }
#pragma unroll
    for (int d = LPR / 2; d; d >>= 1)
        l += __shfl_xor(l, d, LPR);
    __syncthreads();
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < parts; ++s)
        o += *reinterpret_cast<const f32x4 *>(p.part + (s * all + rr) * HD + lane * 4) * w_lds[sub][s];
    const float inv = 1.0f / l;
    if (row < all)
        *reinterpret_cast<f16x4 *>(p.out + (tok * p.n_heads + kv * p.group + (r - tok * p.group)) * HD + lane * 4) =
            f16x4{(f16)(o[0] * inv), (f16)(o[1] * inv), (f16)(o[2] * inv), (f16)(o[3] * inv)};
}

// How the positions of a call are split: parts of `chunk` steps each, one part: not at all.
// A block walks its positions in series at 1.8 us a step, so few tokens behind a long cache, whose rows make few blocks,
// take as many parts as give every compute unit a block; a part has four steps at least, or six from a quarter of the chip
// on, so that the combining launch (3 us) and the parts' outputs cost less than what they save.  A second block a unit
// slows the first one down, which pays from ten steps a part.  32 heads on 8 key/value heads, head size 128, one part
// and this rule, 500 / 2000 / 4000 / 16000 cached positions: 1 token 16 -> 12, 58 -> 15, 113 -> 19, 449 -> 32 us;
// 64 tokens 18 -> 16, 62 -> 21, 117 -> 28, 467 -> 50; 256 tokens 24 -> 23, 68 -> 38, 124 -> 49, 483 -> 149.
// 500 tokens behind 100 lose with two parts (21 -> 27 us) and stay whole.
struct RowsSplit {
    int parts, chunk;
};
RowsSplit rows_split(int64_t start, int64_t tokens, int64_t rows, int64_t n_kv)
{
    const int64_t steps = (start + tokens + kStep - 1) / kStep, blocks = (rows + 63) / 64 * n_kv;
    auto at_most = [](int64_t a, int64_t b) { return a < b ? a : b; };
    const int64_t one = at_most(256 / blocks, steps / (blocks <= 64 ? 4 : 6)), two = at_most(512 / blocks, steps / 10);
    const int64_t parts = tuning_int("HQQ_ROWS_PARTS", (int)at_most(one > two ? one : two, kMaxParts));
    if (parts < 2)
        return {1, (int)steps};
    const int64_t chunk = (steps + parts - 1) / parts;
    return {(int)((steps + chunk - 1) / chunk), (int)chunk};
}

template <int HD> int run_rows(AttRowsParams p, int64_t tokens, void *ws, hipStream_t s)
{
    const int64_t wide = (p.rows + 127) / 128 * p.n_kv, narrow = (p.rows + 63) / 64 * p.n_kv;
    if (narrow > 0x7fffffff)
        return HQQ_E_SHAPE;
    const RowsSplit sp = ws ? rows_split(p.start, tokens, p.rows, p.n_kv) : RowsSplit{1, 0};
    if (sp.parts > 1) {
        const int64_t all = p.n_kv * p.rows;
        p.tiles = narrow / p.n_kv, p.chunk = sp.chunk;
        p.part = static_cast<float *>(ws);
        p.part_ml = reinterpret_cast<f32x2 *>(p.part + sp.parts * all * HD);
        attention_rows_kernel<HD, 1, true><<<(unsigned)(narrow * sp.parts), kRowsThreads, 0, s>>>(p);
        const int rc = launch_status();
        if (rc != HQQ_OK)
            return rc;
        constexpr int RPB = kRowsThreads / (HD / 4);
        attention_rows_combine_kernel<HD><<<(unsigned)((all + RPB - 1) / RPB), kRowsThreads, 0, s>>>(p);
    } else if (wide >= kWideBlocks) {
        attention_rows_kernel<HD, 2, false><<<(unsigned)wide, kRowsThreads, 0, s>>>(p);
    } else {
        attention_rows_kernel<HD, 1, false><<<(unsigned)narrow, kRowsThreads, 0, s>>>(p);
    }
    return launch_status();
}

} // namespace

static bool rows_shape_ok(int64_t start, int64_t tokens, int64_t max_len, int n_heads, int n_kv, int head_dim)
{
    return (head_dim == 64 || head_dim == 128) && n_kv >= 1 && n_heads >= n_kv && n_heads % n_kv == 0 && tokens >= 1 && start >= 0 &&
           tokens <= max_len && start <= max_len - tokens && max_len <= 0x7fffffff;
}

size_t attention_rows_workspace_bytes(int64_t start, int64_t tokens, int n_heads, int n_kv, int head_dim)
{
    if (!rows_shape_ok(start, tokens, 0x7fffffff, n_heads, n_kv, head_dim))
        return 0;
    const int64_t rows = tokens * (n_heads / n_kv);
    const RowsSplit sp = rows_split(start, tokens, rows, n_kv);
    return sp.parts > 1 ? (size_t)sp.parts * (size_t)(n_kv * rows) * (size_t)(head_dim + 2) * sizeof(float) : 0;
}

int launch_attention_rows(const f16 *q, const f16 *cache_k, const f16 *cache_v, int64_t start, int64_t tokens, int64_t max_len,
                          int n_heads, int n_kv, int head_dim, f16 *out, hipStream_t s, void *ws)
{
    if (!rows_shape_ok(start, tokens, max_len, n_heads, n_kv, head_dim))
        return HQQ_E_SHAPE;
    if (!aligned16(q) || !aligned16(cache_k) || !aligned16(cache_v) || !aligned16(out) || !aligned16(ws))
        return HQQ_E_ALIGN;
    AttRowsParams p = {};
    p.q = q, p.ck = cache_k, p.cv = cache_v, p.out = out;
    p.start = start, p.max_len = max_len;
    p.group = n_heads / n_kv, p.n_heads = n_heads, p.n_kv = n_kv;
    p.rows = tokens * p.group;
    p.scale_log2 = (float)(1.4426950408889634 / __builtin_sqrt((double)head_dim));
    return head_dim == 128 ? run_rows<128>(p, tokens, ws, s) : run_rows<64>(p, tokens, ws, s);
}

} // namespace hqq
