// Batch rows through the quantised layers of several experts in one launch, on the matrix cores (2- and 4-bit codes; included by
// one translation unit per code width).
//
// A block is eight wavefronts on one tile of at most 128 (4-bit: 96) batch rows.  A wave owns the 64 output rows of one packed
// row that share table rows (2-bit: 16 rows r of four fields; 4-bit: 32 rows of two), so its lanes hold 16 code bytes of a row
// and every weight is rebuilt in registers, once per block: mask-and-insert, subtract, fma with the scale and minus scale * zero.
// Per 128 columns the block reads its x tile straight into LDS (operand order, one barrier), each wave de-quantises its own
// table entries into LDS, and a wave issues 16 groups of ct MFMAs; see the loop for how they overlap.
//   * 2-bit: a weight is rounded once after its scale: against 64 bits the FFN of an expert on 48 rows is off by 0.74e-3, with the
//     reference's five roundings of a weight by 1.17e-3, a 4096x14336 layer on 333 rows by 0.38e-3 and 0.78e-3.  4-bit: the
//     reference's roundings (1.20e-3, as before).
//   * Up to 64 rows there are few MFMAs to hide behind: the block's waves split its columns in two halves and meet in LDS, and up
//     to 32 rows 128 registers let two blocks share a unit.  There the loads of a step (codes, tables, their meta, x) bound the
//     launch: eight 2-bit Mixtral experts with 1 to 16 rows each take 170 us (3.1 TB/s), with 32 rows 208 us; the launches of one
//     expert after the other 172 to 256 and 411 us.
//   * From 65 rows on the matrix cores' issue does: 3.1 vector instructions an MFMA, two waves to a SIMD.  Eight experts with
//     128 rows 402 us (897 TFLOP/s), with 500 rows 1332 us (1058 TFLOP/s); one after the other 788 and 1929 us.  What that took,
//     at 500 rows: the tables read two groups ahead 1522 -> 1437 us, x straight to LDS and the vector instructions spread between
//     the MFMAs (their own registers are then free for the operands of the next step) 1437 -> 1376, loads from a uniform base
//     1376 -> 1332.
#pragma once

#include "rows_tile_parts.hpp"

namespace hqq {
namespace rows {
namespace {

using gemv::gload;

template <int BITS> struct Codes {
    static constexpr int F = 8 / BITS;       // output rows per packed row
    static constexpr int RBW = 4 / F;        // row blocks of sixteen a wave takes (they share its table rows)
    static constexpr int RT = F * RBW;       // 16-row tiles per wave
    // 2-bit: a weight is scale * (code - 2) + scale * (2 - zero): a zero lies near the middle of the codes, and the second product,
    // which is rounded, is small there.  4-bit, the codes of attention layers: (code - zero) * scale, rounded as hqq_dequantize rounds
    // (a layer's keys are then no further from those of its de-quantised weights than the order of the sums makes them).
    static constexpr int CENTRE = BITS == 2 ? 2 : kStored, OFF = BITS == 2 ? 2 : 0, VALU = BITS == 2 ? 12 : 16;
    static constexpr int pos(int f) { return BITS * (F - 1 - f); }
    static constexpr uint32_t mask(int f) { return (((1u << BITS) - 1u) * 0x00010001u) << pos(f); }
    // a field masked in place and OR-ed into the mantissa of 2^(10 - pos) reads as 2^(10 - pos) + code
    static constexpr uint32_t expo(int f) { return (uint32_t)((10 - pos(f) + 15) << 10) * 0x00010001u; }
};

template <int BITS, int CT, bool GATE, int KW, bool F16T>
__device__ __forceinline__ void tile(const Params HQQ_KERNARG &p, const Member HQQ_KERNARG &g, int unit, int kp, int col, char *lds)
{
    typedef Codes<BITS> C;
    constexpr int F = C::F, RBW = C::RBW, RT = C::RT;
    constexpr int NWK = kBlockWaves / KW;           // waves per K half
    constexpr int JW = NWK / (GATE ? 2 : 1);        // packed rows per block
    constexpr int XTILE = 2 * CT * 2048;            // bytes of one x tile: [64 columns][row tile][row] 128 bytes, see below
    constexpr int CTILE = RBW * 2048;               // bytes of one wave's codes: [row block][row] 128 bytes
    constexpr int TTILE = 4 * F * 4 * 32;           // bytes of one wave's tables: [q][field][k group] 8 scales, 8 zeros
    constexpr int XCH = (4 * CT + NWK - 1) / NWK;   // kilobytes of the x tile a wave brings in per step
    char *const x_lds = lds, *const c_lds = lds + 2 * KW * XTILE + (threadIdx.x >> 6) * (2 * CTILE);
    char *const t_lds = lds + 2 * KW * XTILE + kBlockWaves * 2 * CTILE + (threadIdx.x >> 6) * TTILE;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kh = KW == 1 ? 0 : wave / NWK, wk = KW == 1 ? wave : wave % NWK;
    const int proj = GATE ? wk & 1 : 0, jl = GATE ? wk >> 1 : wk;
    const int jblk = unit / p.RBU, rbu = unit - jblk * p.RBU;
    const int jw = jblk * JW + jl;
    const bool live = jw < p.GP;
    const int jp = live ? jw : p.GP - 1;
    const uint8_t *const l_codes = g.l[proj].codes, *const l_sq = g.l[proj].sq, *const l_zq = g.l[proj].zq;
    const f16 *const l_sms = g.l[proj].s_ms, *const l_smz = g.l[proj].s_mz;
    const int rr = lane & 15, kg = lane >> 4;
    const int K = p.K, M = g.M;
    const int m0 = col * (CT * 16);

    const int b0 = kp * g.spp, b1 = b0 + g.spp < p.steps ? b0 + g.spp : p.steps;
    const int nh = (b1 - b0 + KW - 1) / KW;                   // iterations of every wave of the block
    const int from = b0 + kh * nh, s0 = from < b1 ? from : b1 - 1;
    const int mine = from >= b1 ? 0 : (b1 - from < nh ? b1 - from : nh); // steps of this wave's K half
    const int last = mine > 0 ? mine - 1 : 0;

    // Codes and x come in by eight lanes a row, 128 consecutive bytes (with a lane a row, as the matrix cores want them, the address
    // unit took four times as long, and the waves waited to be let in), and lie in LDS as they come: sixteen-byte chunk c of row r at
    // chunk c ^ (r / 2) % 8 of its row, so that the sixteen lanes of a read, a row each, fall into different banks.
    const int r8 = lane >> 3, c8 = (lane & 7) ^ (r8 >> 1); // of the first eight rows of sixteen; of the other eight chunk c8 ^ 4
    const uint32_t co = (uint32_t)(jp + (16 * rbu * RBW + r8) * p.GP) * (uint32_t)K + 16u * c8; // K is a multiple of 128
    const uint32_t c_half = 8u * (uint32_t)p.GP * (uint32_t)K;                                  // from the first eight rows to the others
    // a lane de-quantises TE entries of one of the wave's table rows per step: columns tk .. tk + TE - 1 of row ti
    constexpr int TE = 2 * F;
    const int ti = lane / (kStep / TE), tk = TE * (lane % (kStep / TE));
    const uint32_t trow = (uint32_t)(F * jp + ti) * (uint32_t)K + (uint32_t)tk;
    uint32_t cm0 = 0;
    float zneg = 0.f, zoff = 0.f; // of the zero table: decode_tables
    if constexpr (!F16T) {
        zneg = uniform(-(float)gload<f16>(g.l[proj].z_ms));
        const float zmz = (float)gload<f16>(g.l[proj].z_mz);
        zoff = uniform(C::CENTRE == kStored ? zmz : (float)C::CENTRE - zmz * zneg);
        const uint32_t c = trow + (uint32_t)s0 * kStep;
        cm0 = mod_cols(c, p.s_cols, p.s_inv);
    }
    // this wave's kilobytes of the x tile: 64 columns wk % 2, rows 8 * (wk / 2 % 2) .. + 7 of row tiles wk / 4, wk / 4 + NWK / 4 ...
    const f16 *xb = g.x + (size_t)m0 * K + (size_t)s0 * kStep + 64 * (wk & 1);
    const int xhr = wk >> 1 & 1;
    const uint32_t xc8 = 16u * (xhr ? c8 ^ 4 : c8), x_last = 2u * (uint32_t)(M - 1 - m0) * (uint32_t)K + xc8;
    uint32_t x_from = 2u * (uint32_t)(16 * (wk >> 2) + 8 * xhr + r8) * (uint32_t)K + xc8; // byte offset of the lane's part of the first
    const uint32_t cd = (uint32_t)(uintptr_t)(HQQ_LDS char *)c_lds;

    typedef uint32_t Halves __attribute__((ext_vector_type(TE / 2)));
    typedef uint32_t Bytes __attribute__((ext_vector_type(TE / 4)));
    struct Next {
        Halves a, b; // meta of the scale / fp16 scales, fp16 zeros
        Bytes sq, zq;
    };
    // What a wave requests for a step, a piece at a time: all at once, it would wait to be let in by the address unit.
    auto issue = [&](Next &r, int it, int buf, int order) __attribute__((always_inline)) {
        const int piece = (order + XCH + 2 * RBW) % (XCH + 2 * RBW + 2); // the tables first: they have a way to go after they arrive
        const int st = it < last ? it : last;
        const uint32_t k0 = (uint32_t)(s0 + st) * kStep;
        if (piece < XCH) {
            int b = (wk >> 2) + NWK / 4 * piece;
            b = b < CT ? b : CT - 1; // (past the end: the last one once more, the same bytes to the same place)
            asm volatile("" : "+v"(x_from)); // the sum is made here, not kept in a register over the loop
            const uint32_t o = x_from + 32u * (uint32_t)(b - (wk >> 2)) * (uint32_t)K; // past the last row: that row once more
            load_to_lds(o < x_last ? o : x_last, xb + (size_t)st * kStep,
                        (uint32_t)(uintptr_t)(HQQ_LDS char *)x_lds + (buf * KW + kh) * XTILE + (((wk & 1) * CT + b) * 2 + xhr) * 1024);
        } else if (piece < XCH + 2 * RBW) {
            const int i = piece - XCH;
            load_to_lds(i & 1 ? co ^ 64u : co, l_codes + k0 + (size_t)i * c_half, cd + buf * CTILE + i * 1024);
        } else if constexpr (F16T) {
            if (piece == XCH + 2 * RBW)
                r.a = load_at<Halves>(l_sq + 2 * (size_t)k0, 2 * trow);
            else
                r.b = load_at<Halves>(l_zq + 2 * (size_t)k0, 2 * trow);
        } else if (piece == XCH + 2 * RBW) {
            r.sq = load_at<Bytes>(l_sq + k0, trow);
            r.zq = load_at<Bytes>(l_zq + k0, trow);
        } else {
            const uint32_t cm = mod_cols(cm0 + (uint32_t)st * kStep, p.s_cols, p.s_inv); // less than K + columns before
            r.a = load_at<Halves>(l_sms, 2 * cm);
            r.b = load_at<Halves>(l_smz, 2 * cm);
        }
    };
    constexpr int PIECES = XCH + 2 * RBW + 2;
    // where they go: slab tk / 64, k group (tk / 16) % 4, half (tk / 8) % 2
    char *const t_w = t_lds + (((((tk >> 6) * 2 + ((tk >> 3) & 1)) * F + ti) * 4 + ((tk >> 4) & 3)) * 32) + 2 * (tk & 7);
    auto stage = [&](const Next &r) __attribute__((always_inline)) { // (a wave's own: in place of those it has read)
        Halves S, Z;
        decode_tables<F16T, TE, C::CENTRE>(r.a, r.b, r.sq, r.zq, zneg, zoff, S, Z);
        *reinterpret_cast<Halves *>(t_w) = S;
        *reinterpret_cast<Halves *>(t_w + 16) = Z;
    };

    f32x4 acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int b = 0; b < CT; ++b)
            acc[i][b] = (f32x4){0.f, 0.f, 0.f, 0.f};

    uint32_t expo[F]; // in vector registers: with a second scalar operand the insertion would be two instructions
#pragma unroll
    for (int f = 0; f < F; ++f) {
        expo[f] = C::expo(f);
        asm volatile("" : "+v"(expo[f]));
    }
    Next nx;
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
        issue(nx, 0, 0, i);
    stage(nx);
    __builtin_amdgcn_s_waitcnt(kWaitLoads);
    __syncthreads();
    const char *const tr = t_lds + kg * 32;
    for (int it = 0; it < nh; ++it) {
        const int buf = it & 1;
        if (KW == 1 || it < mine) {
            // chunks 2 * kg + q % 2 of the lane's batch row, kg and kg + 4 of its code rows
            const char *const xr = x_lds + (buf * KW + kh) * XTILE + rr * 128, *const cr = c_lds + buf * CTILE + rr * 128;
            const int xc = 16 * ((2 * kg) ^ (rr >> 1)), cc = 16 * (kg ^ (rr >> 1));
            // Groups of CT MFMAs: while those of group g run, the weights of group g + 1 are built and the tables of
            // group g + 2 are read (the compiler's own order reads them where they are used, and waits).
            constexpr int NG = 4 * RT;
            u32x4 S[2], Z[2], A[2];
            f16x8 B[CT];
            uint32_t P[4];
            u32x4 cw[RBW]; // codes of 64 columns
            auto codes = [&](int w, int slab) __attribute__((always_inline)) {
                cw[w] = *reinterpret_cast<const u32x4 *>(cr + w * 2048 + (slab ? cc ^ 64 : cc));
            };
            auto tables = [&](int h) __attribute__((always_inline)) { // h = q * F + field
                S[h & 1] = *reinterpret_cast<const u32x4 *>(tr + h * 128);
                Z[h & 1] = *reinterpret_cast<const u32x4 *>(tr + h * 128 + 16);
            };
            auto operand = [&](int q, int b) __attribute__((always_inline)) {
                return *reinterpret_cast<const f16x8 *>(xr + ((q >> 1) * CT + b) * 2048 + (q & 1 ? xc ^ 16 : xc));
            };
            auto build = [&](int gi) __attribute__((always_inline)) { // group gi = (q * RBW + row block) * F + field
                const int f = gi % F, w = gi / F % RBW, q = gi / RT, h = q * F + f;
                if (f == 0)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        P[t] = __builtin_amdgcn_perm(0u, cw[w][2 * (q & 1) + (t >> 1)], t & 1 ? 0x0c030c02u : 0x0c010c00u);
                const f16 offv = (f16)(float)((1 << (10 - C::pos(f))) + C::OFF);
                const f16x2 off = {offv, offv};
                f16x2 v[4]; // stage by stage: a packed instruction's result can be read by the next but one
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    v[t] = h2((P[t] & C::mask(f)) | expo[f]);
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    v[t] = v[t] - off; // the code (2-bit: less 2), exact
                if constexpr (C::CENTRE == kStored) {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        v[t] = v[t] + h2(Z[h & 1][t]);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        A[gi & 1][t] = u2(v[t] * h2(S[h & 1][t]));
                } else {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        A[gi & 1][t] = u2(__builtin_elementwise_fma(v[t], h2(S[h & 1][t]), h2(Z[h & 1][t])));
                }
            };
            tables(0);
#pragma unroll
            for (int w = 0; w < RBW; ++w)
                codes(w, 0);
#pragma unroll
            for (int b = 0; b < CT; ++b)
                B[b] = operand(0, b);
            tables(1);
            build(0);
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                const int f = gi % F, w = gi / F % RBW, q = gi / RT;
                __builtin_amdgcn_sched_barrier(0);
                if (gi + 1 < NG)
                    build(gi + 1);
                // the tables two fields on, once the last row block that uses those in their place has been built
                constexpr int LAST = (RBW - 1) * F;
                if (gi > 0 && (gi + 1) % RT >= LAST && (gi + 1) / RT * F + (gi + 1) % F + 2 < 4 * F && RBW > 1)
                    tables((gi + 1) / RT * F + (gi + 1) % F + 2);
                else if (RBW == 1 && gi + 2 < NG && gi + 2 >= 2)
                    tables(gi + 2);
                if (gi < PIECES)
                    issue(nx, it + 1, buf ^ 1, gi);
                if (q == 1 && f == 0) // the first 64 columns' codes have been taken apart
                    codes(w, 1);
                const bool turn = f == F - 1 && w == RBW - 1 && q + 1 < 4; // the last MFMAs on these operands
#pragma unroll
                for (int b = 0; b < CT; ++b) {
                    acc[w * F + f][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, A[gi & 1]), B[b],
                                                                               acc[w * F + f][b], 0, 0, 0);
                    if (turn)
                        B[b] = operand(q + 1, b);
                }
                // an MFMA, what its operand's register is read into next, and the vector instructions that it hides
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (C::VALU + CT - 1) / CT, 0);
#pragma unroll
                for (int b = 1; b < CT; ++b) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, (C::VALU + CT - 1) / CT, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (it + 1 < nh)
            stage(nx);
        __builtin_amdgcn_s_waitcnt(kWaitLoads); // x and the codes have arrived
        __syncthreads();
    }

    // The K halves' sums meet in LDS; the first half finishes the tiles below CB, the second one the others.  (Which
    // values a wave keeps is selected value by value: with one branch per half the accumulators would be addressed.)
    constexpr int CB = KW == 1 ? CT : (CT + 1) / 2;
    int tid = threadIdx.x; // (the lane's place is worked out again: kept over the loop it would cost the loop registers)
    asm volatile("" : "+v"(tid));
    const int el = tid & 63, er = tid & 15, eg = (tid >> 4) & 3;
    f32x4 sum[RT][CB];
    if constexpr (KW == 2) {
        f32x4 *const kx = reinterpret_cast<f32x4 *>(lds) + el; // [wk][K half][tile][row tile][lane]
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const f32x4 hi = acc[i][CB + j < CT ? CB + j : j];
                sum[i][j] = kh ? hi : acc[i][j];
                kx[(((wk * 2 + kh) * CB + j) * RT + i) * 64] = kh ? acc[i][j] : hi;
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int i = 0; i < RT; ++i)
                sum[i][j] += kx[(((wk * 2 + 1 - kh) * CB + j) * RT + i) * 64];
        if constexpr (GATE)
            __syncthreads();
    } else {
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int i = 0; i < RT; ++i)
                sum[i][j] = acc[i][j];
    }
    // sum[i][j][v]: batch row 16 * (kh * CB + j) + er of the block's, field i % F, row 4 * eg + v of row block i / F
    auto row_group = [&](int w, int v) __attribute__((always_inline)) {
        return (uint32_t)jp + (uint32_t)(16 * (rbu * RBW + w) + 4 * eg + v) * (uint32_t)p.GP;
    };
    if constexpr (GATE) {
        // both projections' waves hold the same outputs: each sends the other the tiles that it finishes
        constexpr int M0 = (CB + 1) / 2; // the first projection's waves finish the tiles below M0
        uint32_t *const gx = reinterpret_cast<uint32_t *>(lds) + el; // [wave][tile][8 pairs][lane]
        f32x4 own[RT][M0];
#pragma unroll
        for (int j = 0; j < M0; ++j)
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const f32x4 hi = sum[i][M0 + j < CB ? M0 + j : j], lo = sum[i][j], out = proj ? lo : hi;
                own[i][j] = proj ? hi : lo;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    gx[((wave * M0 + j) * (2 * RT) + 2 * i + h) * 64] = u2((f16x2){(f16)out[2 * h], (f16)out[2 * h + 1]});
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < M0; ++j) {
            const int jb = proj * M0 + j, tb = kh * CB + jb, m = m0 + 16 * tb + er;
            if (jb >= CB || tb >= CT || m >= M || !live)
                continue;
            f16 o[RT][4];
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const f16x2 other = h2(gx[(((wave ^ 1) * M0 + j) * (2 * RT) + 2 * i + h) * 64]);
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const f16 mine16 = (f16)own[i][j][2 * h + e];
                        const float u = (float)(proj ? other[e] : mine16);
                        const f16 up = proj ? mine16 : other[e];
                        o[i][2 * h + e] = (f16)(u / (1.0f + __expf(-u))) * up; // rounded thrice, as the reference's three operations
                    }
                }
#pragma unroll
            for (int w = 0; w < RBW; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    f16 *dst = g.y + (size_t)m * p.N + (size_t)F * row_group(w, v);
                    if constexpr (F == 4)
                        *reinterpret_cast<f16x4 *>(dst) = (f16x4){o[0][v], o[1][v], o[2][v], o[3][v]};
                    else
                        *reinterpret_cast<f16x2 *>(dst) = (f16x2){o[w * F][v], o[w * F + 1][v]};
                }
        }
    } else {
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int tb = kh * CB + j, m = m0 + 16 * tb + er;
            if (tb >= CT || m >= M || !live)
                continue;
#pragma unroll
            for (int w = 0; w < RBW; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const uint32_t rg = row_group(w, v);
                    if (g.part) {
                        float *dst = g.part + (((size_t)kp * (p.N / F) + rg) * M + m) * F;
                        if constexpr (F == 4)
                            *reinterpret_cast<f32x4 *>(dst) = (f32x4){sum[0][j][v], sum[1][j][v], sum[2][j][v], sum[3][j][v]};
                        else
                            *reinterpret_cast<float2 *>(dst) = make_float2(sum[w * F][j][v], sum[w * F + 1][j][v]);
                        continue;
                    }
                    f16 o[F];
                    f16 *dst = g.y + (size_t)m * p.N + (size_t)F * rg;
#pragma unroll
                    for (int f = 0; f < F; ++f) {
                        o[f] = (f16)sum[w * F + f][j][v];
                        if (g.bias)
                            o[f] = o[f] + g.bias[F * rg + f];
                        if (g.row_scale)
                            o[f] = o[f] * g.row_scale[m];
                        if (g.accumulate)
                            o[f] = dst[f] + o[f];
                    }
                    if constexpr (F == 4)
                        *reinterpret_cast<f16x4 *>(dst) = (f16x4){o[0], o[1], o[2], o[3]};
                    else
                        *reinterpret_cast<f16x2 *>(dst) = (f16x2){o[0], o[1]};
                }
        }
    }
}

template <int BITS> constexpr size_t lds_bytes(int tiles) // tiles: row tiles times K halves
{
    typedef Codes<BITS> C;
    return (size_t)tiles * 8192 + (size_t)kBlockWaves * (2 * C::RBW * 2048 + 4 * C::F * 128);
}

// WIDE: members of any number of rows; else of at most 32, whose few accumulators let two blocks share a compute unit
template <int BITS, bool GATE, bool WIDE, bool F16T>
__global__ __launch_bounds__(kBlockWaves * 64, WIDE ? 2 : 4) void rows_tile_kernel(Params)
{
    const Params HQQ_KERNARG &p = *(const Params HQQ_KERNARG *)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ __attribute__((aligned(16))) char lds[lds_bytes<BITS>(WIDE ? 8 : 4)];
    int unit, kp, col;
    const Member HQQ_KERNARG *at = work_of(p, unit, kp, col);
    if (!at)
        return;
    const Member HQQ_KERNARG &g = *at;
    if constexpr (WIDE) {
        switch (g.ct) {
        case 1: return tile<BITS, 1, GATE, 2, F16T>(p, g, unit, kp, col, lds);
        case 2: return tile<BITS, 2, GATE, 2, F16T>(p, g, unit, kp, col, lds);
        case 3: return tile<BITS, 3, GATE, 2, F16T>(p, g, unit, kp, col, lds);
        case 4: return tile<BITS, 4, GATE, 2, F16T>(p, g, unit, kp, col, lds);
        case 5: return tile<BITS, 5, GATE, 1, F16T>(p, g, unit, kp, col, lds);
        case 6: return tile<BITS, 6, GATE, 1, F16T>(p, g, unit, kp, col, lds);
        default: break;
        }
        if constexpr (max_tiles(BITS) == 8) {
            if (g.ct == 7)
                tile<BITS, 7, GATE, 1, F16T>(p, g, unit, kp, col, lds);
            else
                tile<BITS, 8, GATE, 1, F16T>(p, g, unit, kp, col, lds);
        }
    } else {
        if (g.ct == 1)
            tile<BITS, 1, GATE, 2, F16T>(p, g, unit, kp, col, lds);
        else
            tile<BITS, 2, GATE, 2, F16T>(p, g, unit, kp, col, lds);
    }
}

template <int BITS>
void launch(const Params &p, bool gate, bool wide, bool f16_tables, unsigned blocks, hipStream_t s)
{
    const dim3 block(kBlockWaves * 64);
#define HQQ_ROWS(G, W, T) rows_tile_kernel<BITS, G, W, T><<<blocks, block, 0, s>>>(p)
    if constexpr (BITS == 2) // (4-bit: the codes' place in LDS leaves room for one block a unit in any case)
        if (!wide) {
            if (gate)
                f16_tables ? HQQ_ROWS(true, false, true) : HQQ_ROWS(true, false, false);
            else
                f16_tables ? HQQ_ROWS(false, false, true) : HQQ_ROWS(false, false, false);
            return;
        }
    if (gate)
        f16_tables ? HQQ_ROWS(true, true, true) : HQQ_ROWS(true, true, false);
    else
        f16_tables ? HQQ_ROWS(false, true, true) : HQQ_ROWS(false, true, false);
#undef HQQ_ROWS
}

} // namespace
} // namespace rows
} // namespace hqq
