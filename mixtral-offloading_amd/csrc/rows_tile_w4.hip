#include "rows_tile_kernel.hpp"

namespace hqq {
namespace rows {
void launch_w4(const Params &p, bool gate, bool wide, bool f16_tables, unsigned blocks, hipStream_t s)
{
    launch<4>(p, gate, wide, f16_tables, blocks, s);
}
} // namespace rows
} // namespace hqq
