// Argument blocks of the column kernels of the fused pipeline (fast.hip, zrot.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace flups {

// column passes along y or z of the stage arrays
struct ColArgs {
    const void* src;
    void* dst;
    const void* green;   // z_fused only: normfact * G, [kz'][ky'][kx], kx padded to ldx
    const void* tw;
    int nx;              // valid x columns
    int ldx;             // x row length in complex elements (multiple of 8/16)
    long long s_col;     // element stride between rows of a column (src and dst share it for z; y differs below)
    long long s_col_dst;
    long long s_other_src, s_other_dst;   // stride of the other (batch) dimension
    int nother;
    int nin, nout;       // valid input rows, rows to store
    int gy, gmy;         // z_fused: ky' extent, M1 (for ky' = min(y, M1-y))
    long long comp_src, comp_dst;   // component strides in complex elements
    int rev;             // 1: blocks walk the batch from its last entry
    int xcd;             // z_fused: 1 = XCD-grouped block numbering
    int nopair;          // z_fused: 1 = the other dim has no mirror rows (one row per block, G stored per row); 2 = the two
                         // rows of a pair in neighbouring blocks
    int x0;              // z_fused / z_rot: spectral x index of column 0 (slab offset, a multiple of TX)
    int gntx;            // z_fused / z_rot: x tiles of one ky' row of the compressed G
    int gtx;             // z_rot: tile width of the compressed G
    int nt;              // col_fft forward: 1 = non-temporal stores
};

// derivative symbols of the rotational z pass by mode index: x (nx), y (M1), z (M2), type R, from off[d] on
struct RotSym {
    const void* sym;
    int off[3];
};

}  // namespace flups
