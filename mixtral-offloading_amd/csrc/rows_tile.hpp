// Matrix-core tile over batch rows, the layers of several experts in one launch: what a launch is given.
#pragma once

#include "hqq_common.hpp"

namespace hqq {
namespace rows {

constexpr int kStep = 128;     // columns a block works on between two barriers
constexpr int kBlockWaves = 8;
constexpr int kMembers = 12;   // layers (gates: pairs of layers) of a launch: their records travel in the kernel arguments
// 16-row tiles of a block: what the accumulators leave registers for (4-bit codes: two row blocks' codes in flight)
constexpr int max_tiles(int nbits) { return nbits == 2 ? 8 : 6; }
constexpr int kHalfFields3 = 3; // 3-bit codes: with more tiles two waves share a window's ten fields
constexpr int kMaxStep3 = 2; // 3-bit codes: table rows from one window to the next, at most
// up to so many tiles the waves of a block split its columns in two halves
constexpr int kHalvesTiles = 4;

// One projection as the kernel reads it: codes, the 8-bit (or fp16) tables and their meta
struct Layer {
    const uint8_t *codes;
    const uint8_t *sq, *zq;
    const f16 *s_ms, *s_mz, *z_ms, *z_mz;
};

struct Member {
    Layer l[2]; // the second one: the gate's other projection
    const f16 *x;
    f16 *y;
    float *part; // [K part][N / F][M][F] partial sums, or null: the output goes to y
    const f16 *row_scale, *bias;
    int M, ct, ncol; // rows, 16-row tiles per block, blocks along the rows
    int kpb, spp;    // blocks along K, steps per block
    int first;       // of the launch's list entries (each stands for eight blocks), this member's first
    int units;       // blocks along N
    int accumulate;
};

struct Params {
    int n;
    int N, K, GP, RBU; // GP: packed rows that share no table rows (3-bit: windows), RBU: row blocks of one packed row
    int words, G, dstep, inv; // 3-bit: word rows, table rows, table rows from window to window, window (idx * inv) mod GP is idx-th
    int steps;
    uint32_t s_cols, s_inv; // meta columns of the scale tables, floor(2^32 / columns)
    Member m[kMembers];
};

// kernels of one code width (a translation unit each); wide: some member has more than 32 rows
void launch_w2(const Params &p, bool gate, bool wide, bool f16_tables, unsigned blocks, hipStream_t s);
void launch_w3(const Params &p, bool gate, bool wide, bool f16_tables, unsigned blocks, hipStream_t s);
void launch_w4(const Params &p, bool gate, bool wide, bool f16_tables, unsigned blocks, hipStream_t s);

} // namespace rows
} // namespace hqq
