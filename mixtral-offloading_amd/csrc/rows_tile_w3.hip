// The 3-bit form of the rows kernel (rows_tile_kernel.hpp): ten codes to a 32-bit word, word row w holding output rows 10 w .. 10 w
// + 9.  Word rows P = G / gcd(10, G) apart use the same ten table rows, (10 w + i) mod G: the sixteen A rows of an MFMA are word
// rows w0 + P t (13 of them at Mixtral's shapes), and a wave makes ten A operands, one per field, of every eight words it holds.
// Windows w0 are taken in the order of their first table row, so those of a block's waves overlap in all but gcd(10, G) rows: the
// block de-quantises 10 + gcd (JW - 1) table rows for all of its waves, one chunk of eight columns a lane (each wave for itself:
// two and a half).  A lane reads the words of columns 16 j + 4 g .. + 3, 64 consecutive bytes of a word row a load; the x tile is
// kept in natural order and read as two halves.
// Vector instructions bound it (640 a step of 128 columns for 40 to 120 MFMAs, with half of the fields 375 for 80 to 120).  Eight
// experts of Mixtral's shapes with 16 rows each 204 us (2.98 TB/s), 64 rows 357, 300 rows 1353 (625 TFLOP/s), 700 rows 2926; one
// after the other, the codes rewritten in 4 bits from 17 rows on, 663, 827, 2782 and 3215 us.
#include "rows_tile_parts.hpp"

#include <type_traits>

namespace hqq {
namespace rows {
namespace {

constexpr int F = 10;
// where field i of a pair of words is masked in place: of the low halves, these shifted by six, the halves that begin at bit 8
// (field 4 lies across bit 16), the high halves, these shifted by six
constexpr int field_pos(int i) { return i == 9 ? 0 : i == 8 ? 3 : i == 7 ? 6 : i == 6 ? 3 : i == 5 ? 6 : i == 4 ? 7 : i == 3 ? 2 : i == 2 ? 5 : i == 1 ? 2 : 5; }

// fn(0) ... fn(E - 1) with constants: more groups than a loop is unrolled for
template <int B, int E, typename Fn> __device__ __forceinline__ void each(Fn &&fn)
{
    if constexpr (B < E) {
        fn(std::integral_constant<int, B>{});
        each<B + 1, E>(fn);
    }
}

// a word row's outputs from row n on, as far as the layer has them
template <int FW> __device__ __forceinline__ void store_fields(f16 *row, uint32_t n, int N, const f16 (&o)[FW])
{
#pragma unroll
    for (int i = 0; i < FW; i += FW % 2 ? 1 : 2)
        if (n + i < (uint32_t)N) { // N is even, and so is n with all fields
            if constexpr (FW % 2)
                row[n + i] = o[i];
            else
                *reinterpret_cast<f16x2 *>(row + n + i) = (f16x2){o[i], o[i + 1]};
        }
}

// FH: waves that share a window, each with half of its fields: from four row tiles on, for which a wave has no room with all ten
// fields, so that a weight is still rebuilt once in a block of 96 rows.
template <int CT, int FH, bool GATE, bool F16T>
__device__ __forceinline__ void tile(const Params HQQ_KERNARG &p, const Member HQQ_KERNARG &g, int unit, int kp, int col, char *lds)
{
    constexpr int JW = kBlockWaves / (GATE ? 2 : 1) / FH;      // windows per block
    constexpr int FW = F / FH;                                 // fields of a wave
    constexpr int XTILE = CT * 16 * 16 * 16;                   // bytes of an x tile: [row tile][8 columns][row]
    constexpr int NR = F + kMaxStep3 * (JW - 1);               // table rows of a block, at most
    constexpr int TTILE = NR * 4 * 4 * 32;                     // bytes: [row][q][k group] 8 scales, 8 zeros
    constexpr int XCH = (4 * CT + kBlockWaves - 1) / kBlockWaves; // kilobytes of the x tile a wave stages per step
    char *const x_lds = lds, *const t_lds = lds + 2 * XTILE;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int proj = GATE ? wave & 1 : 0, wk = GATE ? wave >> 1 : wave, jl = wk / FH;
    const int low = FH == 2 ? 5 * ((wk & 1) ^ 1) : 0; // the lowest of this wave's fields
    const int idx0 = unit * JW;
    const bool live = idx0 + jl < p.GP;
    const uint32_t idx = live ? idx0 + jl : p.GP - 1;
    const uint32_t w0 = idx * (uint32_t)p.inv % (uint32_t)p.GP;
    const uint8_t *const l_codes = g.l[proj].codes, *const l_sq = g.l[proj].sq, *const l_zq = g.l[proj].zq;
    const f16 *const l_sms = g.l[proj].s_ms, *const l_smz = g.l[proj].s_mz;
    const int rr = lane & 15, kg = lane >> 4;
    const int K = p.K, M = g.M;
    const int m0 = col * (CT * 16);
    const int s0 = kp * g.spp, n_it = (s0 + g.spp < p.steps ? s0 + g.spp : p.steps) - s0, last = n_it - 1;

    const uint32_t w = w0 + (uint32_t)rr * (uint32_t)p.GP;
    const uint32_t co = (w < (uint32_t)p.words ? w : w0) * (uint32_t)K * 4u + 16u * kg;
    // the chunk of eight columns that this lane de-quantises: row tl of the block's, columns 8 * tc .. + 7 of the step
    const int nr = F + p.dstep * (JW - 1);
    const int chunk = wk * 64 + lane;
    const int tl = (chunk >> 4) < nr ? chunk >> 4 : nr - 1, tc = chunk & 15;
    uint32_t trow = (uint32_t)(p.dstep * idx0 + tl);
    trow -= trow >= (uint32_t)p.G ? p.G : 0; // idx0 < G / dstep and nr <= G: once round at most
    trow = trow * (uint32_t)K + 8u * tc;
    uint32_t cm0 = 0;
    float zneg = 0.f, zoff = 0.f;
    if constexpr (!F16T) {
        zneg = uniform(-(float)gemv::gload<f16>(g.l[proj].z_ms));
        zoff = uniform(-(float)gemv::gload<f16>(g.l[proj].z_mz) * zneg);
        cm0 = mod_cols(trow + (uint32_t)s0 * kStep, p.s_cols, p.s_inv);
    }
    const f16 *xb = g.x + (size_t)m0 * K + (size_t)s0 * kStep;
    uint32_t xo[XCH], xd[XCH];
#pragma unroll
    for (int c = 0; c < XCH; ++c) {
        int pi = wave + kBlockWaves * c;
        pi = pi < 4 * CT ? pi : 4 * CT - 1;
        const int q = pi & 3, b = pi >> 2; // 32 columns of a row tile
        const int m = m0 + 16 * b + rr < M ? 16 * b + rr : M - 1 - m0;
        xo[c] = 2 * ((uint32_t)m * (uint32_t)K + 32 * q + 8 * kg);
        xd[c] = (uint32_t)(uintptr_t)(HQQ_LDS char *)x_lds + (b * 4 + q) * 1024;
    }

    struct Next {
        u32x4 a, b;
        u32x2 sq, zq;
    };
    auto issue = [&](Next &r, int it, int buf) __attribute__((always_inline)) {
        const int st = it < last ? it : last;
        const uint32_t k0 = (uint32_t)(s0 + st) * kStep;
        const f16 *const xs = xb + (size_t)st * kStep;
#pragma unroll
        for (int c = 0; c < XCH; ++c)
            load_to_lds(xo[c], xs, xd[c] + buf * XTILE);
        if constexpr (F16T) {
            r.a = load_at<u32x4>(l_sq + 2 * (size_t)k0, 2 * trow);
            r.b = load_at<u32x4>(l_zq + 2 * (size_t)k0, 2 * trow);
        } else {
            r.sq = load_at<u32x2>(l_sq + k0, trow);
            r.zq = load_at<u32x2>(l_zq + k0, trow);
            const uint32_t cm = mod_cols(cm0 + (uint32_t)st * kStep, p.s_cols, p.s_inv);
            r.a = load_at<u32x4>(l_sms, 2 * cm);
            r.b = load_at<u32x4>(l_smz, 2 * cm);
        }
    };
    // columns 8 tc .. + 3 and + 4 .. + 7: q = tc / 4, half (tc / 2) % 2, k groups 2 (tc % 2) and the next
    char *const t_w = t_lds + proj * TTILE + ((tl * 4 + (tc >> 2)) * 4 + 2 * (tc & 1)) * 32 + 8 * ((tc >> 1) & 1);
    auto stage = [&](const Next &r, int buf) __attribute__((always_inline)) {
        u32x4 S, Z;
        decode_tables<F16T, 8, 0>(r.a, r.b, r.sq, r.zq, zneg, zoff, S, Z);
        char *const d = t_w + buf * ((GATE ? 2 : 1) * TTILE);
        *reinterpret_cast<u32x2 *>(d) = (u32x2){S.x, S.y};
        *reinterpret_cast<u32x2 *>(d + 16) = (u32x2){Z.x, Z.y};
        *reinterpret_cast<u32x2 *>(d + 32) = (u32x2){S.z, S.w};
        *reinterpret_cast<u32x2 *>(d + 48) = (u32x2){Z.z, Z.w};
    };
    auto codes_at = [&](int st, int slab, int j) __attribute__((always_inline)) {
        return load_at<u32x4>(l_codes + ((size_t)(s0 + st) * kStep + 64 * slab + 16 * j) * 4, co);
    };

    f32x4 acc[FW][CT]; // [field low + FW - 1 - k]
#pragma unroll
    for (int i = 0; i < FW; ++i)
#pragma unroll
        for (int b = 0; b < CT; ++b)
            acc[i][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // Groups take a wave's fields from the highest down.  With half of the fields which half decides, for each, whence it comes
    // and where it stands: scalars instead of constants.
    const auto pos_of = [&](int k) __attribute__((always_inline)) { return FH == 1 ? field_pos(F - 1 - k) : low ? field_pos(9 - k) : field_pos(4 - k); };
    // the insertion's exponents in vector registers: with a second scalar operand it would be two instructions
    constexpr int NE = FH == 1 ? 8 : FW;
    uint32_t expo[NE], mask[FW];
    uint32_t off[FW];
#pragma unroll
    for (int k = 0; k < NE; ++k) {
        expo[k] = (uint32_t)((10 - (FH == 1 ? k : pos_of(k)) + 15) << 10) * 0x00010001u;
        asm volatile("" : "+v"(expo[k]));
    }
#pragma unroll
    for (int k = 0; k < FW; ++k) {
        const f16 o = (f16)(float)(1 << (10 - pos_of(k)));
        mask[k] = (7u * 0x00010001u) << pos_of(k), off[k] = u2((f16x2){o, o});
    }
    const uint32_t sel0 = low || FH == 1 ? 0x05040100u : 0x06050201u, sel1 = low ? 0x05040100u : 0x07060302u;
    Next nx;
    u32x4 cw[4][2]; // the words of the step's four sets of 32 columns
    issue(nx, 0, 0);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int o = 0; o < 2; ++o)
            cw[q][o] = codes_at(0, q >> 1, 2 * (q & 1) + o);
    stage(nx, 0);
    __builtin_amdgcn_s_waitcnt(kWaitLoads);
    __syncthreads();
    for (int it = 0; it < n_it; ++it) {
        const int buf = it & 1;
        issue(nx, it + 1, buf ^ 1);
        const char *xr = x_lds + buf * XTILE + ((kg >> 1) * 16 + rr) * 16 + 8 * (kg & 1);
        const char *tr = t_lds + buf * ((GATE ? 2 : 1) * TTILE) + proj * TTILE + (p.dstep * jl + low) * 512 + kg * 32;
        constexpr int NG = 4 * FW;
        u32x4 S[2], Z[2], A[2], P;
        f16x8 B[CT];
        auto tables = [&](int gi) __attribute__((always_inline)) { // group gi = q * FW + k
            const char *at = tr + (FW - 1 - gi % FW) * 512 + gi / FW * 128;
            S[gi & 1] = *reinterpret_cast<const u32x4 *>(at);
            Z[gi & 1] = *reinterpret_cast<const u32x4 *>(at + 16);
        };
        auto operand = [&](int q, int b) __attribute__((always_inline)) {
            const char *at = xr + (b * 4 + q) * 1024;
            const u32x2 lo = *reinterpret_cast<const u32x2 *>(at), hi = *reinterpret_cast<const u32x2 *>(at + 512);
            return __builtin_bit_cast(f16x8, (u32x4){lo.x, lo.y, hi.x, hi.y});
        };
        auto build = [&](int gi) __attribute__((always_inline)) {
            const int q = gi / FW, k = gi % FW, i = F - 1 - k;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t a = cw[q][t >> 1][2 * (t & 1)], b = cw[q][t >> 1][2 * (t & 1) + 1];
                if constexpr (FH == 1) {
                    if (i == 9)
                        P[t] = __builtin_amdgcn_perm(b, a, 0x05040100u);
                    else if (i == 4)
                        P[t] = __builtin_amdgcn_perm(b, a, 0x06050201u);
                    else if (i == 3)
                        P[t] = __builtin_amdgcn_perm(b, a, 0x07060302u);
                    else if (i == 6 || i == 1)
                        P[t] >>= 6;
                } else if (k < 2) {
                    P[t] = __builtin_amdgcn_perm(b, a, k == 0 ? sel0 : sel1);
                } else if (k == 3) {
                    P[t] >>= 6;
                }
            }
            f16x2 v[4]; // stage by stage: a packed instruction's result can be read by the next but one
#pragma unroll
            for (int t = 0; t < 4; ++t)
                v[t] = h2((P[t] & mask[k]) | expo[FH == 1 ? field_pos(i) : k]);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                v[t] = v[t] - h2(off[k]); // the exact code
#pragma unroll
            for (int t = 0; t < 4; ++t)
                A[gi & 1][t] = u2(__builtin_elementwise_fma(v[t], h2(S[gi & 1][t]), h2(Z[gi & 1][t])));
        };
        tables(0);
#pragma unroll
        for (int b = 0; b < CT; ++b)
            B[b] = operand(0, b);
        tables(1);
        build(0);
        each<0, NG>([&](auto index) __attribute__((always_inline)) {
            constexpr int gi = decltype(index)::value, q = gi / FW, k = gi % FW;
            __builtin_amdgcn_sched_barrier(0);
            if (gi + 1 < NG)
                build(gi + 1);
            if (gi + 2 < NG)
                tables(gi + 2);
            if (k == (FH == 1 ? 7 : 2)) { // the words of these columns have been taken apart: their registers wait for the next step's
                const int st = it < last ? it + 1 : last;
                cw[q][0] = codes_at(st, q >> 1, 2 * (q & 1));
                cw[q][1] = codes_at(st, q >> 1, 2 * (q & 1) + 1);
            }
            constexpr bool turn = k == FW - 1 && q + 1 < 4;
#pragma unroll
            for (int b = 0; b < CT; ++b) {
                acc[k][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, A[gi & 1]), B[b], acc[k][b], 0, 0, 0);
                if (turn)
                    B[b] = operand(q + 1, b);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (12 + CT - 1) / CT, 0);
#pragma unroll
            for (int b = 1; b < CT; ++b) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (12 + CT - 1) / CT, 0);
            }
        });
        __builtin_amdgcn_sched_barrier(0);
        if (it + 1 < n_it)
            stage(nx, buf ^ 1);
        __builtin_amdgcn_s_waitcnt(kWaitLoads); // the x tile has arrived
        __syncthreads();
    }

    // acc[k][b][v]: batch row 16 b + er of the block's, field low + FW - 1 - k of word row w0 + P (4 eg + v).  (The lane's place is
    // worked out again: kept over the loop it would cost the loop registers.)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int er = tid & 15, eg = (tid >> 4) & 3;
    const auto word_row = [&](int v) __attribute__((always_inline)) { return w0 + (uint32_t)(4 * eg + v) * (uint32_t)p.GP; };
    if constexpr (GATE) {
        // both projections' waves hold the same outputs: the first finishes two of a lane's four word rows, the second two
        uint32_t *const gx = reinterpret_cast<uint32_t *>(lds) + (tid & 63); // [wave][tile][field][lane] pairs
#pragma unroll
        for (int b = 0; b < CT; ++b)
#pragma unroll
            for (int k = 0; k < FW; ++k) {
                const f32x4 a = acc[k][b];
                gx[((wave * CT + b) * FW + k) * 64] = u2((f16x2){(f16)(proj ? a[0] : a[2]), (f16)(proj ? a[1] : a[3])});
            }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < CT; ++b) {
            const int m = m0 + 16 * b + er;
            f16 o[2][FW];
#pragma unroll
            for (int k = 0; k < FW; ++k) {
                const f16x2 other = h2(gx[(((wave ^ 1) * CT + b) * FW + k) * 64]);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const f16 own = (f16)(proj ? acc[k][b][2 + e] : acc[k][b][e]);
                    const float u = (float)(proj ? other[e] : own);
                    const f16 up = proj ? own : other[e];
                    o[e][FW - 1 - k] = (f16)(u / (1.0f + __expf(-u))) * up; // rounded thrice, as the reference's three operations
                }
            }
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const uint32_t wr = word_row(2 * proj + e);
                if (m < M && live && wr < (uint32_t)p.words)
                    store_fields<FW>(g.y + (size_t)m * p.N, F * wr + low, p.N, o[e]);
            }
        }
    } else {
#pragma unroll
        for (int b = 0; b < CT; ++b) {
            const int m = m0 + 16 * b + er;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const uint32_t wr = word_row(v), n0 = F * wr + low;
                if (m >= M || !live || wr >= (uint32_t)p.words)
                    continue;
                if (g.part) {
                    float *dst = g.part + (((size_t)kp * p.words + wr) * M + m) * F + low;
                    if constexpr (FW % 2 == 0) {
#pragma unroll
                        for (int i = 0; i < FW; i += 2)
                            *reinterpret_cast<float2 *>(dst + i) = make_float2(acc[FW - 1 - i][b][v], acc[FW - 2 - i][b][v]);
                    } else {
#pragma unroll
                        for (int i = 0; i < FW; ++i)
                            dst[i] = acc[FW - 1 - i][b][v];
                    }
                    continue;
                }
                f16 o[FW];
                f16 *dst = g.y + (size_t)m * p.N;
#pragma unroll
                for (int i = 0; i < FW; ++i) {
                    const bool in = n0 + i < (uint32_t)p.N;
                    o[i] = (f16)acc[FW - 1 - i][b][v];
                    if (g.bias && in)
                        o[i] = o[i] + g.bias[n0 + i];
                    if (g.row_scale)
                        o[i] = o[i] * g.row_scale[m];
                    if (g.accumulate && in)
                        o[i] = dst[n0 + i] + o[i];
                }
                store_fields<FW>(dst, n0, p.N, o);
            }
        }
    }
}

constexpr size_t lds_bytes(bool gate, int ct, int fh)
{
    const size_t jw = kBlockWaves / (gate ? 2 : 1) / fh;
    const size_t work = 2 * (size_t)ct * 4096 + 2 * (gate ? 2 : 1) * (F + kMaxStep3 * (jw - 1)) * 512;
    const size_t exchange = gate ? (size_t)kBlockWaves * ct * (F / fh) * 256 : 0;
    return work > exchange ? work : exchange;
}
constexpr size_t lds_most(bool gate)
{
    const size_t a = lds_bytes(gate, kHalfFields3, 1), b = lds_bytes(gate, max_tiles(3), 2);
    return a > b ? a : b;
}

template <bool GATE, bool F16T> __global__ __launch_bounds__(kBlockWaves * 64, 2) void rows_tile3_kernel(Params)
{
    const Params HQQ_KERNARG &p = *(const Params HQQ_KERNARG *)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ __attribute__((aligned(16))) char lds[lds_most(GATE)];
    int unit, kp, col;
    const Member HQQ_KERNARG *g = work_of(p, unit, kp, col);
    if (!g)
        return;
    static_assert(kHalfFields3 == 3 && max_tiles(3) == 6, "the tiles below");
    switch (g->ct) {
    case 1: return tile<1, 1, GATE, F16T>(p, *g, unit, kp, col, lds);
    case 2: return tile<2, 1, GATE, F16T>(p, *g, unit, kp, col, lds);
    case 3: return tile<3, 1, GATE, F16T>(p, *g, unit, kp, col, lds);
    case 4: return tile<4, 2, GATE, F16T>(p, *g, unit, kp, col, lds);
    case 5: return tile<5, 2, GATE, F16T>(p, *g, unit, kp, col, lds);
    default: return tile<6, 2, GATE, F16T>(p, *g, unit, kp, col, lds);
    }
}

} // namespace

void launch_w3(const Params &p, bool gate, bool, bool f16_tables, unsigned blocks, hipStream_t s)
{
    const dim3 block(kBlockWaves * 64);
    if (gate)
        f16_tables ? rows_tile3_kernel<true, true><<<blocks, block, 0, s>>>(p) : rows_tile3_kernel<true, false><<<blocks, block, 0, s>>>(p);
    else
        f16_tables ? rows_tile3_kernel<false, true><<<blocks, block, 0, s>>>(p) : rows_tile3_kernel<false, false><<<blocks, block, 0, s>>>(p);
}

} // namespace rows
} // namespace hqq
