// Batches of 17 rows and more, the layers of several experts in one launch: shapes, splits and launches.  The kernel is in
// rows_tile_kernel.hpp.
#include "rows_tile.hpp"
#include "gemv_parts.hpp"

#include <algorithm>
#include <numeric>

namespace hqq {
using namespace rows;

namespace {

struct Shape {
    int F, GP, RBU, steps;
    int words, G, dstep, inv; // 3-bit codes
    bool f16_tables;
};

bool ptr_aligned(const void *p, unsigned n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

bool shape_of(const hqq_linear *l, Shape &sh)
{
    const int64_t G = l->N / l->group_size;
    sh = Shape{};
    if (l->K % kStep != 0 || G * l->K >= (1ll << 31) || l->K >= (1 << 24) || l->N >= (1ll << 30) || !ptr_aligned(l->codes, 16))
        return false;
    sh.steps = (int)(l->K / kStep);
    if (l->nbits == 3) {
        const int64_t d = std::gcd((int64_t)10, G), P = G / d, words = (l->N + 9) / 10;
        // table rows of a block: at most 24, once round G at most; a window: at most sixteen word rows
        if (d > kMaxStep3 || G < 10 + kMaxStep3 * (kBlockWaves - 1) || (words + P - 1) / P > 16 || l->N % 2 != 0 ||
            words * l->K * 4 >= (1ll << 32) || P >= (1 << 15))
            return false;
        sh.F = 10, sh.GP = (int)P, sh.RBU = 1, sh.words = (int)words, sh.G = (int)G, sh.dstep = (int)d;
        while (sh.inv < P && 10 / d * sh.inv % P != 1 % P)
            ++sh.inv;
    } else {
        sh.F = 8 / l->nbits;
        const int64_t rbw = 4 / sh.F;
        if (l->group_size % (16 * rbw) != 0 || G % sh.F != 0 || l->N / sh.F * l->K >= (1ll << 32)) // 32-bit offsets within a layer
            return false;
        sh.GP = (int)(G / sh.F), sh.RBU = (int)(l->group_size / (16 * rbw));
    }
    const int sk = gemv::table_kind(l->scale), zk = gemv::table_kind(l->zero);
    sh.f16_tables = sk == gemv::TK_F16 && zk == gemv::TK_F16;
    if (sh.f16_tables)
        return ptr_aligned(l->scale.data, 16) && ptr_aligned(l->zero.data, 16);
    return sk == gemv::TK_U8_COLS && zk == gemv::TK_U8_SCALAR && l->scale.meta_cols % 8 == 0 && l->scale.meta_cols < (1ll << 31) &&
           ptr_aligned(l->scale.data, 8) && ptr_aligned(l->zero.data, 8) && ptr_aligned(l->scale.meta_scale, 16) &&
           ptr_aligned(l->scale.meta_zero, 16);
}

// How M rows are cut: ncol blocks of ct tiles of sixteen rows, as even as they come
struct Cut {
    int ct, ncol;
    int share; // waves of a block that work on the same output rows (of one projection)
};
Cut cut_rows(int nbits, int64_t M, int ct)
{
    const int tiles = (int)((M + 15) / 16), most = max_tiles(nbits), n = (tiles + most - 1) / most;
    Cut c;
    c.ct = ct ? ct : (tiles + n - 1) / n, c.ncol = (tiles + c.ct - 1) / c.ct, c.share = (nbits == 3 ? c.ct > kHalfFields3 : c.ct <= kHalvesTiles) ? 2 : 1;
    return c;
}
int units(const Shape &sh, const Cut &c, bool gate)
{
    const int jw = kBlockWaves / c.share / (gate ? 2 : 1);
    return (sh.GP + jw - 1) / jw * sh.RBU;
}

} // namespace

bool rows_supported(const hqq_linear *l, int64_t M)
{
    Shape sh;
    return M > 0 && M < (1 << 24) && M * l->K < (1ll << 31) && shape_of(l, sh); // 32-bit byte offsets within x
}

bool rows_alike(const hqq_linear *a, const hqq_linear *b)
{
    return a->nbits == b->nbits && a->group_size == b->group_size && a->N == b->N && a->K == b->K && a->scale.kind == b->scale.kind &&
           a->zero.kind == b->zero.kind && a->scale.meta_cols == b->scale.meta_cols && a->zero.meta_cols == b->zero.meta_cols;
}

int64_t rows_blocks(const hqq_linear *l, int64_t M, bool gate)
{
    Shape sh;
    if (!shape_of(l, sh))
        return 0;
    const Cut c = cut_rows(l->nbits, M, 0);
    return (int64_t)units(sh, c, gate) * c.ncol;
}

int rows_outputs_together(const hqq_linear *l) { return l->nbits == 3 ? 10 : 8 / l->nbits; }

int rows_k_blocks(const hqq_linear *l, int64_t blocks, bool wide)
{
    Shape sh;
    if (!shape_of(l, sh))
        return 1;
    const int64_t slots = wide || l->nbits != 2 ? 256 : 512; // blocks that run at a time
    int best = 1;
    int64_t cost = -1;
    for (int k = 1; k <= 8 && sh.steps / k >= 4; ++k) { // in steps of a block; 4: its first loads and its end
        const int64_t c = (blocks * k + slots - 1) / slots * ((sh.steps + k - 1) / k + 4) + (k > 1 ? 4 + k : 0);
        if (cost < 0 || c < cost)
            best = k, cost = c;
    }
    const int spp = (sh.steps + best - 1) / best; // parts of equal length, none of them empty
    return (sh.steps + spp - 1) / spp;
}

// What a step of 128 columns (of a K half: of both) and a tile of it take in a block when all units are at work, in ns: the fit of
// 5800 launches of single layers (2- to 4-bit, 1024x1024 to 14336x4096, 17 to 1270 rows, every cut and 1 to 16 blocks along K),
// which it meets to 10 % (rms).  What it chooses is on average 3 % slower than the fastest of them.  At 2-bit 4096x14336 with 128
// rows that is 4 tiles and 8 blocks along K, 30 us; as wide as a block can be (8 tiles) 49; 4-bit 4096x4096 with 256 rows 23, 31.
struct StepCost {
    int start, step, tile;
};
static StepCost step_cost(int nbits, int ct)
{
    if (nbits == 3)
        return ct <= kHalfFields3 ? StepCost{10200, 2030, 1060} : StepCost{9600, 1400, 330};
    if (nbits == 2)
        return ct <= 2 ? StepCost{6300, 2270, 160} : ct <= kHalvesTiles ? StepCost{6000, 1380, 180} : StepCost{5200, 1050, 240};
    return ct <= kHalvesTiles ? StepCost{5200, 1320, 180} : StepCost{7400, 1240, 190};
}

RowsPlan rows_plan(const hqq_linear *l, int64_t M, bool gate)
{
    RowsPlan best = {0, 1};
    Shape sh;
    if (!shape_of(l, sh))
        return best;
    const int64_t tiles = (M + 15) / 16;
    double least = 0;
    for (int ct = 1; ct <= max_tiles(l->nbits) && ct <= tiles; ++ct) {
        const Cut c = cut_rows(l->nbits, M, ct);
        const StepCost t = step_cost(l->nbits, ct);
        const bool narrow = l->nbits == 2 && ct <= 2; // two blocks share a unit, and a step takes half as long where one has it alone
        const int halves = l->nbits != 3 && c.share == 2 ? 2 : 1, slots = narrow ? 512 : 256;
        for (int k = 1; k <= (gate ? 1 : 16) && sh.steps / k >= (k > 1 ? 4 : 1); ++k) {
            const int spp = (sh.steps + k - 1) / k, kpb = (sh.steps + spp - 1) / spp;
            if (kpb != k)
                continue;
            const int64_t blocks = ((int64_t)units(sh, c, gate) * k + 7) / 8 * 8 * c.ncol; // of a die: an eighth, rounded up
            const int64_t rounds = (blocks + slots - 1) / slots;
            const double load = narrow && blocks < slots ? 0.5 + 0.5 * (double)blocks / slots : 1.0;
            double ns = t.start + (double)rounds * ((spp + halves - 1) / halves) * (t.step + t.tile * ct) * load;
            if (k > 1) // the partial sums' way to memory and back, and a launch
                ns += 2500.0 + 200.0 * k + 1.5e-3 * k * (double)M * (double)l->N;
            if (best.ct == 0 || ns < least)
                best = RowsPlan{ct, k}, least = ns;
        }
    }
    return best;
}

// One layer, the tile kernel against this one, in us: 2-bit 14336x4096 with 32 rows 20.0 / 17.5, 128 rows 38.2 / 29.4, 290 rows 79 / 53,
// 630 rows 162 / 92; 4096x14336 333 rows 66 / 54, 1000 rows 140 / 117; 4-bit 4096x4096 32 rows 12.6 / 13.4, 64 rows 18.0 / 17.0, 630 rows
// 75 / 45; 14336x4096 17 rows 24.3 / 16.7, 290 rows 138 / 58.  3-bit codes have few blocks where there are few windows, and the tile kernel's rewrite is
// cheap there: 112 windows (14336x4096) 17 rows 34.5 / 27.6, 64 rows 37.6 / 35.5, 290 rows 149 / 81; 32 windows, 4096x14336 64 rows
// 38.7 / 40.2, 96 rows 49.0 / 44.5, 4096x4096 256 rows 35.2 / 38.0, 290 rows 48.3 / 43.5.
bool rows_preferred(const hqq_linear *l, int64_t M)
{
    Shape sh;
    if (M <= 16 || !rows_supported(l, M) || !shape_of(l, sh))
        return false;
    if (l->nbits == 3)
        return M > (sh.GP >= 64 ? 16 : l->K >= 8192 ? 64 : 256);
    return M > 32 || l->nbits == 2 || l->N * l->K > (1ll << 24);
}

size_t rows_partial_bytes(const hqq_linear *l, int64_t M, int kpb)
{
    const int64_t F = rows_outputs_together(l), N = (l->N + F - 1) / F * F;
    return kpb > 1 ? ((size_t)kpb * (size_t)M * (size_t)N * sizeof(float) + 255) & ~(size_t)255 : 0;
}

int launch_rows(const RowsItem *item, const int *kpb, int n, bool gate, hipStream_t s)
{
    int order[64];
    if (n < 1 || n > 64)
        return HQQ_E_UNSUPPORTED;
    for (int i = 0; i < n; ++i)
        order[i] = i;
    std::stable_sort(order, order + n, [&](int a, int b) { return item[a].M > item[b].M; });
    for (int at = 0; at < n; at += kMembers) {
        const hqq_linear *l = item[order[at]].l0;
        Shape sh;
        if (!shape_of(l, sh))
            return HQQ_E_UNSUPPORTED;
        Params p = {};
        p.N = (int)l->N, p.K = (int)l->K, p.GP = sh.GP, p.RBU = sh.RBU, p.steps = sh.steps;
        p.words = sh.words, p.G = sh.G, p.dstep = sh.dstep, p.inv = sh.inv;
        p.s_cols = (uint32_t)l->scale.meta_cols;
        p.s_inv = p.s_cols ? (uint32_t)(0xFFFFFFFFull / p.s_cols) : 0;
        int64_t slots = 0;
        bool wide = false;
        for (int i = at; i < n && i < at + kMembers; ++i) {
            const RowsItem &it = item[order[i]];
            Member &m = p.m[p.n++];
            for (int q = 0; q < (gate ? 2 : 1); ++q) {
                const hqq_linear *ll = q ? it.l1 : it.l0;
                m.l[q] = Layer{static_cast<const uint8_t *>(ll->codes), static_cast<const uint8_t *>(ll->scale.data),
                               static_cast<const uint8_t *>(ll->zero.data), static_cast<const f16 *>(ll->scale.meta_scale),
                               static_cast<const f16 *>(ll->scale.meta_zero), static_cast<const f16 *>(ll->zero.meta_scale),
                               static_cast<const f16 *>(ll->zero.meta_zero)};
            }
            m.x = it.x, m.y = it.y, m.part = it.part, m.row_scale = it.row_scale, m.accumulate = it.accumulate;
            m.bias = gate ? nullptr : static_cast<const f16 *>(it.l0->bias);
            if (it.ct < 0 || it.ct > max_tiles(l->nbits))
                return HQQ_E_UNSUPPORTED;
            const Cut c = cut_rows(l->nbits, it.M, it.ct);
            m.M = (int)it.M, m.ct = c.ct, m.ncol = c.ncol;
            const int kb = gate ? 1 : kpb[order[i]];
            m.spp = (sh.steps + kb - 1) / kb, m.kpb = (sh.steps + m.spp - 1) / m.spp;
            if (m.kpb != kb || (kb > 1) != (it.part != nullptr))
                return HQQ_E_UNSUPPORTED;
            m.units = units(sh, c, gate);
            m.first = (int)slots;
            slots += ((int64_t)m.units * m.kpb + 7) / 8 * m.ncol;
            wide = wide || c.ct > 2;
        }
        if (slots * 8 > 0x7fffffff)
            return HQQ_E_UNSUPPORTED;
        if (l->nbits == 2)
            launch_w2(p, gate, wide, sh.f16_tables, (unsigned)(slots * 8), s);
        else if (l->nbits == 3)
            launch_w3(p, gate, wide, sh.f16_tables, (unsigned)(slots * 8), s);
        else
            launch_w4(p, gate, wide, sh.f16_tables, (unsigned)(slots * 8), s);
        const int rc = launch_status();
        if (rc != HQQ_OK)
            return rc;
    }
    return HQQ_OK;
}

} // namespace hqq
