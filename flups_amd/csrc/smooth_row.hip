#include "smooth_pen.hpp"

namespace flups {

namespace {
template <bool WIDE, typename TI, typename TO>
using smooth_row = smooth_pen<WIDE, false, TI, TO>;
}  // namespace

void launch_smooth_row(const PassDesc& P, dim3 grid, dim3 block, size_t lds, hipStream_t s) { launch_io<smooth_row>(P, grid, block, lds, s); }

}  // namespace flups
