// Last direction of the general path fused with the curl (Biot-Savart): forward c2c of the three
// components along z, u = i K x (normfact G omega), inverse c2c, in place, for every length of
// smooth_fft.hpp. src/dothemagic_rot.ipp:102-349.
//
// It takes the place of three forward passes, a multiply sweep and three inverse passes over the
// spectral array (twice the field where z is zero-padded). A block holds the three components of
// one tile of columns in LDS, and one thread runs the same butterflies of each of them: between a
// component's LDS reads and its writes lies one barrier, which also orders the component before it, so a
// stage costs three barriers for three transforms. The last forward stage, the curl and the
// first inverse stage (the same radix) touch a thread's own LDS slots only. 160^3 layer, FP32
// storage, MI355X: 3 x 30 + 70 + 3 x 30 us -> 145 us. 50 MB in, 50 MB out and 4 MB of G, 0.7 TB/s: bound inside the
// block (counters: 2.3 waves per SIMD resident, VALU busy 40 %, LDS bank conflicts 38 % of a CU's cycles).
#include <hip/hip_runtime.h>

#include "core.hpp"
#include "fft_core.hpp"
#include "group.hpp"
#include "smooth_fft.hpp"

namespace flups {

bool smooth_plan_upto(int M, int maxrad, SmoothPlan& p, int minst);   // smooth.hip

namespace {

// Registers for three waves per SIMD: the LDS of three components holds a CU to about 52 / (smallest radix)
// waves anyway
template <typename ST>
struct smooth_rot {
    using Args = SmoothRotArgs;
    static constexpr int NT = 512, kWaves = 3;
    static constexpr bool WIDE = false;   // radices up to 10 (rot_plan)
    static __device__ __forceinline__ void run(const SmoothRotArgs& A, Blk blk) {
        extern __shared__ double smem[];
        const SmoothPlan& S = A.sm;
        const int M = S.M, tx = A.tx;
        const int c = threadIdx.x & (tx - 1), t = threadIdx.x / tx;
        const int ntile = (A.nx + tx - 1) / tx;
        const int b = xcd_group(blk.x, blk.nx);
        const int tile = b % ntile, o = b / ntile;
        // rows that share a G slice in neighbouring blocks: 0, 1, n - 1, 2, n - 2, ...
        const int h = (o + 1) >> 1;
        const int y = !A.mirror ? o : (o & 1) || o == 0 ? h : A.nother - h;
        const int yg = !A.mirror ? o : h;
        const bool live = tile * tx + c < A.nx;
        const int x = min(tile * tx + c, A.nx - 1);   // lanes past nx load the last valid column and store nothing
        C2<ST>* col = reinterpret_cast<C2<ST>*>(A.d) + (long long)y * A.s_other + x;
        C2<double>* lds = reinterpret_cast<C2<double>*>(smem) + c;
        // the thread's number anew for each component: addresses and twiddles of a butterfly are formed
        // where they are used, not kept in registers across the loops (200 spilled ones)
        auto fresh = [&]() {
            int a = t;
            asm volatile("" : "+v"(a));
            return a;
        };
        const int bank = M * tx;   // one component
        const C2<double>* tw = reinterpret_cast<const C2<double>*>(A.tw);
        const int last = S.nst - 1;

        // first forward stage: from HBM, zero rows past nin
        auto first = [&](auto r) {
            constexpr int R = decltype(r)::value;
            const int mp = S.mp[0];
            if (t < mp) {
#pragma unroll 1
                for (int cc = 0; cc < 3; ++cc) {
                    const int t = fresh();
                    const C2<ST>* p = col + cc * A.comp + t * A.s_col;
                    C2<double> v[R];
#pragma unroll
                    for (int q = 0; q < R; ++q) {
                        v[q] = {0.0, 0.0};
                        if (t + q * mp < A.nin) v[q] = c2d(p[(long long)q * mp * A.s_col]);
                    }
                    dft_r<R>(v);
#pragma unroll
                    for (int u = 0; u < R; ++u) lds[cc * bank + (t * R + u) * tx] = v[u];
                }
            }
            __syncthreads();
        };
        // a stage of the three components in LDS (write: false where the values go to HBM)
        auto stage = [&](auto r, int mp, int span, int inv, int stride, bool write) {
            constexpr int R = decltype(r)::value;
            const bool on = t < mp;
#pragma unroll 1
            for (int cc = 0; cc < 3; ++cc) {
                const int t = fresh();
                const int bb = (int)(((unsigned)t * (unsigned)inv) >> 20), k = t - bb * span, w = (bb * span * R + k) * tx;
                C2<double>* l = lds + cc * bank;
                C2<double> v[R];
                if (on) {
#pragma unroll
                    for (int q = 0; q < R; ++q) v[q] = l[(t + q * mp) * tx];
                    if (span > 1) twiddle_r<R>(v, tw, k * stride);
                    dft_r<R>(v);
                }
                if (write) {
                    __syncthreads();   // this component is read, the one before it is written
                    if (on) {
#pragma unroll
                        for (int u = 0; u < R; ++u) l[w + u * span * tx] = v[u];
                    }
                } else if (on && live) {
                    C2<ST>* p = col + cc * A.comp + t * A.s_col;
#pragma unroll
                    for (int u = 0; u < R; ++u)
                        if (t + u * mp < A.nin) p[(long long)u * mp * A.s_col] = c2t<ST>({v[u].y, v[u].x});
                }
            }
        };
        // last forward stage, curl: the thread's own slots
        auto middle = [&](auto r) {
            constexpr int R = decltype(r)::value;
            const int mp = S.mp[last];
            if (t >= mp) return;
            const ST* g = reinterpret_cast<const ST*>(A.g) + ((long long)yg * A.gntx + x / A.gtx) * (M / 2 + 1) * A.gtx + x % A.gtx;
            double gv[R];
#pragma unroll
            for (int u = 0; u < R; ++u) gv[u] = (double)g[min(t + u * mp, M - t - u * mp) * A.gtx];
#pragma unroll 1
            for (int cc = 0; cc < 3; ++cc) {
                const int t = fresh();
                C2<double>* l = lds + cc * bank + t * tx;
                C2<double> v[R];
#pragma unroll
                for (int q = 0; q < R; ++q) v[q] = l[q * mp * tx];
                twiddle_r<R>(v, tw, t);
                dft_r<R>(v);
#pragma unroll
                for (int u = 0; u < R; ++u) l[u * mp * tx] = {v[u].x * gv[u], v[u].y * gv[u]};
            }
            const double kx = A.sym[A.off[0] + x], ky = A.sym[A.off[1] + y];
#pragma unroll 1
            for (int u = 0; u < R; ++u) {
                C2<double>* l = lds + (t + u * mp) * tx;
                const double kz = A.sym[A.off[2] + t + u * mp];
                const C2<double> wx = l[0], wy = l[bank], wz = l[2 * bank];
                // u = i K x w, real and imaginary parts swapped: the inverse transform is a forward one
                l[0] = {ky * wz.x - kz * wy.x, kz * wy.y - ky * wz.y};
                l[bank] = {kz * wx.x - kx * wz.x, kx * wz.y - kz * wx.y};
                l[2 * bank] = {kx * wy.x - ky * wx.x, ky * wx.y - kx * wy.y};
            }
        };
#define FLUPS_CALL(R) first(std::integral_constant<int, R>{})
        FLUPS_SMOOTH_RADIX(S.rad[0], FLUPS_CALL)
#undef FLUPS_CALL
        for (int s = 1; s < last; ++s) {
#define FLUPS_CALL(R) stage(std::integral_constant<int, R>{}, S.mp[s], S.span[s], S.inv[s], S.stride[s], true)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
        }
        if (last > 1) __syncthreads();   // the third component's writes
#define FLUPS_CALL(R) middle(std::integral_constant<int, R>{})
        FLUPS_SMOOTH_RADIX(S.rad[last], FLUPS_CALL)
#undef FLUPS_CALL
        for (int s = last; s >= 0; --s) {
#define FLUPS_CALL(R) stage(std::integral_constant<int, R>{}, S.mp[s], S.rspan[s], S.rinv[s], S.rstride[s], s > 0)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
            if (s == 1) __syncthreads();   // the third component's writes, before the reads that end in HBM
        }
    }
};

// bytes of one block: three blocks share a CU's 160 KB. Narrower tiles rather than two larger blocks: 80^3 open FP32 175 ->
// 161 us (8 -> 4 columns), 160^3 open 1103 -> 1093 (4 -> 2), 160^3 layer 365 -> 361; 32 KB: batch 1548 -> 1635.
// Two columns from 288 points on and one from 567 on (16-byte rows, 8 in FP32) still beat three passes, the multiply
// and three passes by the same kernels, up to the longest column that fits (solves, us, separate -> fused, FP64 / FP32):
// 96 x 96 periodic with 512 points 416 -> 343 / 344 -> 310, 576: 480 -> 437 / 368 -> 361, 640: 550 -> 505 / 417 -> 382, 1024: 958 ->
// 821 / 755 -> 619, 1120: 1256 -> 1017 / 970 -> 743; 48 x 48 open with 450 points 224 -> 165, 640: 284 -> 219, 1120: 723 -> 549
constexpr size_t kRotLds = 54272;

// Radices up to 10 where the tile's LDS limits the waves: 112^3 open 389 -> 367 us, layer 157 -> 143, 96^3 layer 107 ->
// 95, 32 mixed problems 1555 -> 1525 against up to 16 (two stages, but three blocks of 64 threads a
// CU); up to 8 the same within 1 %, up to 6 slower (80^3 open 153 -> 254). Every length that fits has such a plan.
bool rot_plan(int M, SmoothPlan& p) { return smooth_plan_upto(M, 10, p, 2); }

}  // namespace

// columns per block (0: no kernel for this length)
int smooth_rot_tile(int M, bool f32) {
    SmoothPlan p;
    if (!rot_plan(M, p)) return 0;
    int tx = f32 ? 8 : 4;
    while (tx * p.T < 64) tx *= 2;
    while (tx > 1 && (tx * p.T > 512 || (size_t)3 * M * tx * sizeof(C2<double>) > kRotLds)) tx /= 2;
    return tx * p.T <= 512 && (size_t)3 * M * tx * sizeof(C2<double>) <= kRotLds ? tx : 0;
}
void launch_smooth_rot(SmoothRotArgs A, hipStream_t s) {
    FLUPS_REQUIRE(rot_plan(A.sm.M, A.sm), "no stages for columns of %d points", A.sm.M);
    const dim3 grid((A.nx + A.tx - 1) / A.tx * A.nother), block(A.tx * A.sm.T);
    const size_t lds = (size_t)3 * A.tx * A.sm.M * sizeof(C2<double>);
    if (A.f32) launch_k<smooth_rot<float>>(grid, block, lds, s, A);
    else launch_k<smooth_rot<double>>(grid, block, lds, s, A);
    HIP_CHECK(hipGetLastError());
}

}  // namespace flups
