// Rotational (Biot-Savart) z pass of the fused pipeline, in place on the three components of S1:
// forward FFT of omega_x, omega_y, omega_z along z, psi = normfact G omega, then u = curl psi =
// i K x psi with the derivative symbol K of each direction (the wave number itself, or the symbol of
// the 2nd/4th/6th-order centred difference), inverse FFTs, keep the first nin rows.
// src/dothemagic_rot.ipp:102-349.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fast_args.hpp"
#include "fft_core.hpp"
#include "group.hpp"

namespace flups {

namespace {

struct ZRotArgs {
    ColArgs a;
    RotSym rk;
};

// A block transforms one row of TX columns (64-byte rows of HBM) of the three components at a time:
// M/8 threads per column, 8 values of each component per thread, so that the curl sits in registers
// between the last forward and the first inverse stage. Three sets of values need all 256 registers
// of two waves per SIMD (FP64; 128 of four, FP32): eight waves of a CU hold 196 KB of it, and
// nothing but the block itself can overlap its loads, its LDS exchanges and its arithmetic:
//  * the blocks are persistent, and a component's next row is loaded as soon as its stores are issued
//    (its registers are free then), two inverse transforms before it is used;
//  * the exchanges take two LDS buffers in turn (one barrier each instead of two), the twiddle table
//    is a copy in LDS;
//  * HALF (unbounded: nin = M/2, or M/2 + 1 node-centred): four rows (and one thread's fifth) are
//    loaded and stored, the zero half is pruned from the first forward stage.
// Three-component solves on MI355X, one row pair per block before -> now: 513^3 node-centred 27.2 ->
// 23.9 ms, this pass 14.2 -> 11.2 (26 GB in and out: 2.4 TB/s) (FP32 17.1 -> 16.2), 256^3 2.63 -> 2.49, 128^3 0.346 -> 0.301 ms.
template <typename R, int M, int TX, bool HALF>
struct z_rot {
    using Args = ZRotArgs;
    static constexpr int NT = TX * M / 8;
    static constexpr int kWaves = sizeof(R) == 8 ? 2 : 4;
    static __device__ __forceinline__ void run(const ZRotArgs& z, Blk bk) {
        constexpr int T = M / 8, E = column_exchanges(M), NL = HALF ? 5 : 8;
        constexpr bool LTW = sizeof(R) == 4;   // seven LDS reads per stage instead of three and four products
        __shared__ C2<R> lds[2 * M * TX];
        __shared__ C2<R> ltw[M];
        const ColArgs& a = z.a;
        int c = threadIdx.x % TX, j = threadIdx.x / TX;
        for (int i = threadIdx.x; i < M; i += NT) ltw[i] = reinterpret_cast<const C2<R>*>(a.tw)[i];
        __syncthreads();
        // items: rows y0 and M1 - y0 of a tile side by side (they share G's slice), then the tiles of
        // y0; each XCD walks its own eighth of them
        const int ntx = (a.nx + TX - 1) / TX;
        const int items = 2 * ntx * (a.gmy / 2 + 1);
        int it = bk.x, step = bk.nx, end = items;
        if (a.xcd && bk.nx % 8 == 0) {
            const int x = bk.x % 8;
            step = bk.nx / 8;
            it = (int)((long long)items * x / 8) + bk.x / 8;
            end = (int)((long long)items * (x + 1) / 8);
        }
        auto absent = [&](int i) {   // rows 0 and M1/2 have no mirror
            const int y0 = (i >> 1) / ntx;
            return (i & 1) && (y0 == 0 || 2 * y0 == a.gmy);
        };
        auto next = [&](int i) {
            do i += step;
            while (i < end && absent(i));
            return i;
        };
        if (it < end && absent(it)) it = next(it);
        if (it >= end) return;
        const size_t cstride = (size_t)sizeof(C2<R>) * a.comp_src;
        const size_t rstride = (size_t)sizeof(C2<R>) * T * a.s_col;
        const R* sym = reinterpret_cast<const R*>(z.rk.sym);
        C2<R> v[3][8];
        // component cc of item i: lanes past nx load the last valid column and store nothing
        auto load = [&](int cc, int i) {
            const int tile = (i >> 1) % ntx, y0 = (i >> 1) / ntx, y = (i & 1) ? a.gmy - y0 : y0;
            const char* b = reinterpret_cast<const char*>(a.src) +
                            (size_t)sizeof(C2<R>) * ((long long)tile * TX + (long long)y * a.s_other_src) + cc * cstride;
            const unsigned off = (unsigned)(sizeof(C2<R>) * ((size_t)j * a.s_col + min(c, a.nx - 1 - tile * TX)));
#pragma unroll
            for (int r = 0; r < NL; ++r)
                v[cc][r] = (HALF && r < 4) || j + r * T < a.nin ? *reinterpret_cast<const C2<R>*>(b + r * rstride + off) : C2<R>{0, 0};
        };
        load(0, it);
        load(1, it);
        load(2, it);
        while (true) {
            asm volatile("" : "+v"(c), "+v"(j));   // the stages' addresses are formed again for each row, not kept in registers
            const int tile = (it >> 1) % ntx, y0 = (it >> 1) / ntx, y = (it & 1) ? a.gmy - y0 : y0;
            const int x = tile * TX + c;
            const bool live = x < a.nx;
            column_fft<R, M, true, TX, HALF ? 2 : 0, LTW, 0>(v[0], lds + c, j, ltw);
            column_fft<R, M, true, TX, HALF ? 2 : 0, LTW, E & 1>(v[1], lds + c, j, ltw);
            // G and the symbols, in flight during the last forward transform
            const int xg = a.x0 + min(x, a.nx - 1);
            const R* g = reinterpret_cast<const R*>(a.green) + ((long long)y0 * a.gntx + xg / a.gtx) * (M / 2 + 1) * a.gtx + xg % a.gtx;
            R gv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int kz = j + i * T;
                gv[i] = g[min(kz, M - kz) * a.gtx];
            }
            const R kx = sym[z.rk.off[0] + xg], ky = sym[z.rk.off[1] + y];
            column_fft<R, M, true, TX, HALF ? 2 : 0, LTW, 0>(v[2], lds + c, j, ltw);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const R kz = sym[z.rk.off[2] + j + i * T];
                const C2<R> wx = {v[0][i].x * gv[i], v[0][i].y * gv[i]};
                const C2<R> wy = {v[1][i].x * gv[i], v[1][i].y * gv[i]};
                const C2<R> wz = {v[2][i].x * gv[i], v[2][i].y * gv[i]};
                // u = i K x w: (K x w) then multiply by i: (p + i q) i = -q + i p
                const C2<R> cx = {ky * wz.x - kz * wy.x, ky * wz.y - kz * wy.y};
                const C2<R> cy = {kz * wx.x - kx * wz.x, kz * wx.y - kx * wz.y};
                const C2<R> cz = {kx * wy.x - ky * wx.x, kx * wy.y - ky * wx.y};
                v[0][i] = {-cx.y, cx.x};
                v[1][i] = {-cy.y, cy.x};
                v[2][i] = {-cz.y, cz.x};
            }
            const int nit = next(it);
            char* b = reinterpret_cast<char*>(a.dst) + (size_t)sizeof(C2<R>) * ((long long)tile * TX + (long long)y * a.s_other_src);
            const unsigned voff = (unsigned)(sizeof(C2<R>) * ((size_t)j * a.s_col + c));
            auto back = [&](int cc) {   // the component's stores, then its next row's loads
                if (live) {
#pragma unroll
                    for (int r = 0; r < NL; ++r)
                        if ((HALF && r < 4) || j + r * T < a.nout)
                            *reinterpret_cast<C2<R>*>(b + cc * cstride + r * rstride + voff) = v[cc][r];
                }
                if (nit < end) load(cc, nit);
            };
            column_fft<R, M, false, TX, 0, LTW, E & 1>(v[0], lds + c, j, ltw);
            back(0);
            column_fft<R, M, false, TX, 0, LTW, 0>(v[1], lds + c, j, ltw);
            back(1);
            column_fft<R, M, false, TX, 0, LTW, E & 1>(v[2], lds + c, j, ltw);
            back(2);
            if (nit >= end) return;   // uniform over the block
            it = nit;
        }
    }
};

// Blocks that fill the chip: 256 CUs, kWaves waves on each of their four SIMDs. TX: 64-byte rows, but
// at least a whole wave a block, and at most 512 threads.
template <typename R, int M>
void launch(const ColArgs& a, const RotSym& rk, hipStream_t st) {
    constexpr int W = 64 / (int)sizeof(C2<R>);
    constexpr int TX = M <= 64 ? std::max(W, 512 / M) : M == 1024 ? 4 : W;
    constexpr int full = 256 * (sizeof(R) == 8 ? 8 : 16) * 64 / (TX * M / 8);
    const int items = 2 * ((a.nx + TX - 1) / TX) * (a.gmy / 2 + 1);
    const dim3 grid(std::min(full, (items + 7) / 8 * 8));
    const bool half = a.nin == a.nout && (a.nin == M / 2 || a.nin == M / 2 + 1);
    if (half) launch_k<z_rot<R, M, TX, true>>(grid, dim3(TX * M / 8), 0, st, {a, rk});
    else launch_k<z_rot<R, M, TX, false>>(grid, dim3(TX * M / 8), 0, st, {a, rk});
    HIP_CHECK(hipGetLastError());
}

}  // namespace

template <typename R>
void launch_z_rot(int M, const ColArgs& a, const RotSym& rk, hipStream_t st) {
    switch (M) {
        case 32: launch<R, 32>(a, rk, st); break;
        case 64: launch<R, 64>(a, rk, st); break;
        case 128: launch<R, 128>(a, rk, st); break;
        case 256: launch<R, 256>(a, rk, st); break;
        case 512: launch<R, 512>(a, rk, st); break;
        case 1024: launch<R, 1024>(a, rk, st); break;
        default: fail("unsupported column length %d", M);
    }
}
template void launch_z_rot<double>(int, const ColArgs&, const RotSym&, hipStream_t);
template void launch_z_rot<float>(int, const ColArgs&, const RotSym&, hipStream_t);

}  // namespace flups
