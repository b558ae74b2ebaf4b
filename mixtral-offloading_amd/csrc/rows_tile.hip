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
Cut cut_rows(int nbits, int64_t M)
{
    const int tiles = (int)((M + 15) / 16), most = max_tiles(nbits), n = (tiles + most - 1) / most;
    Cut c;
    c.ct = (tiles + n - 1) / n, c.ncol = (tiles + c.ct - 1) / c.ct, c.share = (nbits == 3 ? c.ct > kHalfFields3 : c.ct <= kHalvesTiles) ? 2 : 1;
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
    return M > 0 && M < (1 << 24) && shape_of(l, sh);
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
    const Cut c = cut_rows(l->nbits, M);
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
            const Cut c = cut_rows(l->nbits, it.M);
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
