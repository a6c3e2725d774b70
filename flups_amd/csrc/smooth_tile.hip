#include "smooth_pen.hpp"

namespace flups {

namespace {
template <bool WIDE, typename TI, typename TO>
using smooth_tile = smooth_pen<WIDE, true, TI, TO>;
}  // namespace

void launch_smooth_tile(const PassDesc& P, dim3 grid, dim3 block, size_t lds, hipStream_t s) { launch_io<smooth_tile>(P, grid, block, lds, s); }

}  // namespace flups
