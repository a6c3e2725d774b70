// Pass kernels of the general path for lengths with factors 2, 3, 5, 7 on the run-time mixed-radix FFT of
// smooth_fft.hpp: every length that the register kernels of rowpass.hip do not have (9, 15, 25, ... times a
// power of two: 100, 120, 144, 180, 200, 240, 300, ...), and of the others the passes that they run faster
// (contiguous r2c / c2r of every length; the rules stand at the fit tests in rowpass.hip):
//   smooth_col   c2c along a strided direction, values straight between HBM and the first / last
//                stage's registers;
//   smooth_z     the last direction fused with the multiply: forward c2c, normfact G, inverse c2c;
//   smooth_rz    the same for an r2c last direction, pairs of real columns;
//   smooth_pen   every other pass (r2c, c2r, r2r, c2c of a contiguous pencil; r2c, c2r, r2r of a
//                strided one), pre- and post-maps from tables (smooth_pen.hpp).
// Before, these lengths ran on the generic kernel (up to five radix 2-7 stages over LDS, sines and
// cosines computed in its pre- and post-maps, 2n-point extensions for r2r) with a separate multiply
// sweep: 200 x 144 x 100 open 6 x 262 + 80 us, now 28 (x) + 33 (y) + 85 (fused z) + 33 + 28 us, the
// solve 1589 -> 215 us; 240 x 100 x 180 channel 1009 -> 152 us (MI355X, FP64). The passes move their
// minimum bytes at 2.1-4.2 TB/s. Counters of those two problems: 2.2 to 5.5 waves per SIMD resident, 39-63 % of
// their cycles waiting on memory or a barrier, VALU busy 32-62 %, LDS bank conflicts 9-35 % of a CU's cycles:
// the latency of a block's load - stages - store chain, but for the fused z of three stages (200 points: VALU
// 62 %, conflicts 35 %).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <map>
#include <mutex>
#include <type_traits>
#include <vector>

#include "smooth_pen.hpp"

namespace flups {

void launch_smooth_row(const PassDesc& P, dim3 grid, dim3 block, size_t lds, hipStream_t s);    // smooth_row.hip
void launch_smooth_tile(const PassDesc& P, dim3 grid, dim3 block, size_t lds, hipStream_t s);   // smooth_tile.hip

namespace {

// WIDE: radices up to 16 (two stages for most lengths up to 256) in 168 registers, three waves per SIMD: at
// 128 they spilled 20 to 40 (120^3 open 140 -> 126 us, 240^3 periodic 349 -> 316), and a block of
// 64 threads and 12 KB of LDS reaches no fourth wave. Otherwise up to 10 in 80 registers, six waves: with three
// stages the barriers between them want the waves (200 x 144 x 100 open: fused z 131 us with every
// radix in one kernel, 84 us so; five waves 193 -> 199, seven 196, eight 225 us the solve), although the
// narrow ones of smooth_col and smooth_z spill 20 to 36 bytes at six
template <bool WIDE, typename TI, typename TO>
struct smooth_col {
    using Args = PassDesc;
    static constexpr int NT = 512, kWaves = WIDE ? 3 : 6;
    static __device__ __forceinline__ void run(const PassDesc& P, Blk blk) {
        extern __shared__ double smem[];
        C2<double>* lds = reinterpret_cast<C2<double>*>(smem);
        const SmoothPlan& S = P.sm;
        const int tx = P.ppb;   // a power of two
        const int c = threadIdx.x & (tx - 1), t = threadIdx.x / tx;
        const int ntile = (P.na + tx - 1) / tx;
        const int b = xcd_group(blk.x, blk.nx);
        const int tile = b % ntile, jb = b / ntile;
        int ja = tile * tx + c;
        const bool live = ja < P.na;
        if (!live) ja = P.na - 1;   // dead columns read the last one and store nothing
        const C2<TI>* src = reinterpret_cast<const C2<TI>*>(P.from<TI>(blk.y)) + (long long)ja * P.src_s[P.fa] + (long long)jb * P.src_s[P.fb];
        C2<TO>* dst = reinterpret_cast<C2<TO>*>(P.to<TO>(blk.y)) + (long long)ja * P.dst_s[P.fa] + (long long)jb * P.dst_s[P.fb];
        const long long sd = P.src_s[P.d], dd = P.dst_s[P.d];
        const bool inv = P.sign > 0;
        const C2<double>* tw = reinterpret_cast<const C2<double>*>(P.tw);
        auto slot = [&](int e) { return e * tx + c; };
        auto ext = [&](C2<double>* v, int mp, auto r) {
            constexpr int R = decltype(r)::value;
            const int k0 = t - P.gshift;
            const C2<TI>* p = src + k0 * sd;
            const long long step = mp * sd;
#pragma unroll
            for (int q = 0; q < R; ++q) {   // rows outside the source are zero padding
                v[q] = {0.0, 0.0};
                const int ks = k0 + q * mp;
                if (ks >= 0 && ks < P.src_nd) v[q] = swapped(c2d(p[q * step]), inv);
            }
        };
        auto out = [&](C2<double>* v, int mp, auto r) {
            constexpr int R = decltype(r)::value;
            if (!live) return;
            const int k0 = t - P.sshift;
            C2<TO>* p = dst + k0 * dd;
            const long long step = mp * dd;
#pragma unroll
            for (int u = 0; u < R; ++u) {
                const int k = k0 + u * mp;
                if (k >= 0 && k < P.dst_nd) p[u * step] = c2t<TO>(swapped(v[u], inv));
            }
            if ((P.post & POST_PERIOD) && t == 0) {   // node-centred periodic: X[0] again at position n
                const int k = S.M - P.sshift;
                if (k >= 0 && k < P.dst_nd) dst[k * dd] = c2t<TO>(swapped(v[0], inv));
            }
        };
        auto none = [](C2<double>*, int, auto) {};
        const int last = S.nst - 1;
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[0], 1, S.inv[0], S.stride[0], true, false, lds, slot, tw, ext, none)
        FLUPS_SMOOTH_RADIX(S.rad[0], FLUPS_CALL)
#undef FLUPS_CALL
        for (int s = 1; s < last; ++s) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[s], S.span[s], S.inv[s], S.stride[s], false, false, lds, slot, tw, none, none)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
        }
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[last], S.span[last], S.inv[last], S.stride[last], false, true, lds, slot, tw, none, out)
        FLUPS_SMOOTH_RADIX(S.rad[last], FLUPS_CALL)
#undef FLUPS_CALL
    }
};

template <bool WIDE, typename ST>
struct smooth_z {
    using Args = SmoothZArgs;
    static constexpr int NT = 512, kWaves = WIDE ? 3 : 6;
    static __device__ __forceinline__ void run(const SmoothZArgs& A, Blk blk) {
        extern __shared__ double smem[];
        C2<double>* lds = reinterpret_cast<C2<double>*>(smem);
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
        const int cl = min(c, A.nx - 1 - tile * tx);   // lanes past nx load the last valid column and store nothing
        C2<ST>* col = reinterpret_cast<C2<ST>*>(A.d) + (long long)blk.y * A.comp + (long long)y * A.s_other + (long long)tile * tx;
        const ST* g = reinterpret_cast<const ST*>(A.g) + ((long long)yg * ntile + tile) * (M / 2 + 1) * tx + c;
        const C2<double>* tw = reinterpret_cast<const C2<double>*>(A.tw);
        auto slot = [&](int e) { return e * tx + c; };
        auto ext = [&](C2<double>* v, int mp, auto r) {
            constexpr int R = decltype(r)::value;
            const C2<ST>* p = col + cl + t * A.s_col;
            const long long step = mp * A.s_col;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                v[q] = {0.0, 0.0};
                if (t + q * mp < A.nin) v[q] = c2d(p[q * step]);
            }
        };
        auto out = [&](C2<double>* v, int mp, auto r) {
            constexpr int R = decltype(r)::value;
            if (!live) return;
            C2<ST>* p = col + c + t * A.s_col;
            const long long step = mp * A.s_col;
#pragma unroll
            for (int u = 0; u < R; ++u)
                if (t + u * mp < A.nin) p[u * step] = c2t<ST>({v[u].y, v[u].x});
        };
        auto none = [](C2<double>*, int, auto) {};
        const int last = S.nst - 1;
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[0], 1, S.inv[0], S.stride[0], true, false, lds, slot, tw, ext, none)
        FLUPS_SMOOTH_RADIX(S.rad[0], FLUPS_CALL)
#undef FLUPS_CALL
        for (int s = 1; s < last; ++s) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[s], S.span[s], S.inv[s], S.stride[s], false, false, lds, slot, tw, none, none)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
        }
        // the last forward stage leaves X[t + u mp] in registers, the values that the first stage of the
        // inverse (the same radix) starts from: the multiply sits between them
        auto middle = [&](auto r) {
            constexpr int R = decltype(r)::value;
            const int mp = S.mp[last];
            const bool on = t < mp;
            C2<double> v[R];
            if (on) {
                double gv[R];
#pragma unroll
                for (int u = 0; u < R; ++u) {
                    const int kz = t + u * mp;
                    gv[u] = (double)g[min(kz, M - kz) * tx];
                }
#pragma unroll
                for (int q = 0; q < R; ++q) v[q] = lds[slot(t + q * mp)];
                twiddle_r<R>(v, tw, t);
                dft_r<R>(v);
#pragma unroll
                for (int u = 0; u < R; ++u) v[u] = {v[u].y * gv[u], v[u].x * gv[u]};   // swapped: inverse
                dft_r<R>(v);
            }
            __syncthreads();   // the stage's inputs are read
            if (on) {
#pragma unroll
                for (int u = 0; u < R; ++u) lds[slot(t * R + u)] = v[u];
            }
            __syncthreads();
        };
#define FLUPS_CALL(R) middle(std::integral_constant<int, R>{})
        FLUPS_SMOOTH_RADIX(S.rad[last], FLUPS_CALL)
#undef FLUPS_CALL
        for (int s = last - 1; s > 0; --s) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[s], S.rspan[s], S.rinv[s], S.rstride[s], false, false, lds, slot, tw, none, none)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
        }
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[0], S.rspan[0], S.rinv[0], S.rstride[0], false, true, lds, slot, tw, none, out)
        FLUPS_SMOOTH_RADIX(S.rad[0], FLUPS_CALL)
#undef FLUPS_CALL
    }
};

// An r2c last direction: two neighbouring real columns a, b as one complex column a + i b, whose product
// spectrum is Z'[k] = Ga/2 (Z[k] + conj Z[M-k]) + Gb/2 (Z[k] - conj Z[M-k]) (G real and even in kz). The mirrored value
// lies with another thread: the forward spectrum passes through LDS between the transforms.
// 129 x 161 x 97 node-centred walls, MI355X: r2c 22, multiply 15 and c2r 23 us before, 27 us now. Two sets of G beside the
// values: four waves (128 registers, nothing spilled), three for the wide radices (168, 40 bytes spilled).
template <bool WIDE, typename ST>
struct smooth_rz {
    using Args = SmoothRzArgs;
    static constexpr int NT = 512, kWaves = WIDE ? 3 : 4;
    static __device__ __forceinline__ void run(const SmoothRzArgs& A, Blk blk) {
        extern __shared__ double smem[];
        C2<double>* lds = reinterpret_cast<C2<double>*>(smem);
        const SmoothPlan& S = A.sm;
        const int M = S.M, tx = A.tx;
        const int c = threadIdx.x & (tx - 1), t = threadIdx.x / tx;
        const int npair = (A.nx + 1) / 2, ntile = (npair + tx - 1) / tx;
        const int b = xcd_group(blk.x, blk.nx);
        const int tile = b % ntile, y = b / ntile;
        const int pr = tile * tx + c;
        const bool la = pr < npair;
        const int xa = 2 * min(pr, npair - 1);   // dead pairs read the last pair and store nothing
        const bool hb = xa + 1 < A.nx;           // the partner column exists
        ST* base = reinterpret_cast<ST*>(A.d) + (long long)blk.y * A.comp + (long long)y * A.nx + xa;
        const ST* g = reinterpret_cast<const ST*>(A.g) + 2 * ((long long)y * A.nx + xa);
        const long long gs = 2LL * A.nx * A.ny;   // reals between kz rows of G
        const C2<double>* tw = reinterpret_cast<const C2<double>*>(A.tw);
        auto slot = [&](int e) { return e * tx + c; };
        auto ext = [&](C2<double>* v, int mp, auto r) {
            constexpr int R = decltype(r)::value;
            const ST* p = base + t * A.s_col;
            const long long step = mp * A.s_col;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                v[q] = {0.0, 0.0};
                if (t + q * mp < A.nin) v[q] = {(double)p[q * step], hb ? (double)p[q * step + 1] : 0.0};
            }
        };
        auto out = [&](C2<double>* v, int mp, auto r) {
            constexpr int R = decltype(r)::value;
            if (!la) return;
            ST* p = base + t * A.s_col;
            const long long step = mp * A.s_col;
#pragma unroll
            for (int u = 0; u < R; ++u)
                if (t + u * mp < A.nin) {
                    p[u * step] = (ST)v[u].y;
                    if (hb) p[u * step + 1] = (ST)v[u].x;
                }
        };
        auto none = [](C2<double>*, int, auto) {};
        const int last = S.nst - 1;
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[0], 1, S.inv[0], S.stride[0], true, false, lds, slot, tw, ext, none)
        FLUPS_SMOOTH_RADIX(S.rad[0], FLUPS_CALL)
#undef FLUPS_CALL
        for (int s = 1; s < last; ++s) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[s], S.span[s], S.inv[s], S.stride[s], false, false, lds, slot, tw, none, none)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
        }
        auto middle = [&](auto r) {
            constexpr int R = decltype(r)::value;
            const int mp = S.mp[last];
            const bool on = t < mp;
            C2<double> v[R];
            double ga[R], gb[R];
            if (on) {
#pragma unroll
                for (int u = 0; u < R; ++u) {
                    const int k = t + u * mp, kz = min(k, M - k);
                    ga[u] = (double)g[kz * gs];
                    gb[u] = hb ? (double)g[kz * gs + 2] : ga[u];
                }
#pragma unroll
                for (int q = 0; q < R; ++q) v[q] = lds[slot(t + q * mp)];
                twiddle_r<R>(v, tw, t);
                dft_r<R>(v);
#pragma unroll
                for (int u = 0; u < R; ++u) lds[slot(t + u * mp)] = v[u];   // X[t + u mp], the thread's own slots
            }
            __syncthreads();
            if (on) {
#pragma unroll
                for (int u = 0; u < R; ++u) {
                    const int k = t + u * mp;
                    const C2<double> zc = cconj(lds[slot(k == 0 ? 0 : M - k)]);
                    const C2<double> s = cadd(v[u], zc), d = csub(v[u], zc);
                    const double p = 0.5 * A.normfact * ga[u], q = 0.5 * A.normfact * gb[u];
                    v[u] = {p * s.y + q * d.y, p * s.x + q * d.x};   // swapped: inverse
                }
                dft_r<R>(v);
            }
            __syncthreads();   // the mirrored values are read
            if (on) {
#pragma unroll
                for (int u = 0; u < R; ++u) lds[slot(t * R + u)] = v[u];
            }
            __syncthreads();
        };
#define FLUPS_CALL(R) middle(std::integral_constant<int, R>{})
        FLUPS_SMOOTH_RADIX(S.rad[last], FLUPS_CALL)
#undef FLUPS_CALL
        for (int s = last - 1; s > 0; --s) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[s], S.rspan[s], S.rinv[s], S.rstride[s], false, false, lds, slot, tw, none, none)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
        }
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[0], S.rspan[0], S.rinv[0], S.rstride[0], false, true, lds, slot, tw, none, out)
        FLUPS_SMOOTH_RADIX(S.rad[0], FLUPS_CALL)
#undef FLUPS_CALL
    }
};

constexpr size_t kSmoothLds = 65536;   // bytes of one block
constexpr int kSmoothThreads = 512;

size_t pen_lds(const PassDesc& P, bool col, int np) {
    const size_t H = P.sm.M;
    return np * (col ? H : H + H / 8 + 1) * 2 * sizeof(double);
}
// pencils of a strided tile: `want`, more until the block has a whole wave, fewer until its threads and
// its LDS fit (0: none)
template <typename Lds>
int fit_tile(int want, int T, Lds&& lds) {
    while (want * T < 64 && want < 32) want *= 2;
    for (int np = want; np >= 1; np /= 2)
        if (np * T <= kSmoothThreads && lds(np) <= kSmoothLds) return np;
    return 0;
}
// columns of complex values: rows of 64 bytes. Wider rows need fewer cache-line requests, but the blocks
// get larger and fewer: 200 x 144 x 100 open, fused z (three stages) 84 us with 4 columns, 91 with 8,
// 104 with 2; 240 x 100 x 180 channel (two stages) 21.5 us with 4 or 8
int col_tile(int M, int T, bool f32) {
    return fit_tile(f32 ? 8 : 4, T, [&](int np) { return (size_t)np * M * 2 * sizeof(double); });
}

}  // namespace

// fewest stages, then radices up to 10 (the kernels with fewer registers), then fewest threads (the
// largest smallest radix); radices ascending, so that every thread takes part in the first stage and in
// the last one of a fused inverse, the ones that meet HBM
static bool search_plan(int M, int maxrad, int minst, SmoothPlan& p) {
    static const int rads[13] = {2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16};
    std::vector<int> cur, best;
    auto search = [&](auto&& self, int m, int lo) -> void {
        if (m == 1) {
            if ((int)cur.size() < minst) return;
            const bool low = cur.back() <= 10, blow = !best.empty() && best.back() <= 10;
            if (best.empty() || cur.size() < best.size() ||
                (cur.size() == best.size() && (low != blow ? low : cur[0] > best[0])))
                best = cur;
            return;
        }
        if ((int)cur.size() == kSmoothStages) return;
        for (int i = lo; i < 13; ++i)
            if (m % rads[i] == 0 && rads[i] <= maxrad) {
                cur.push_back(rads[i]);
                self(self, m / rads[i], i);
                cur.pop_back();
            }
    };
    search(search, M, 0);
    if (best.empty()) return false;
    p = SmoothPlan();
    p.M = M;
    p.nst = (int)best.size();
    p.T = M / best[0];
    p.wide = best.back() > 10;
    int span = 1;
    for (int s = 0; s < p.nst; ++s) {
        p.rad[s] = best[s];
        p.mp[s] = M / best[s];
        p.span[s] = span;
        p.inv[s] = ((1 << 20) + span - 1) / span;
        p.stride[s] = M / (span * best[s]);
        span *= best[s];
    }
    span = 1;
    for (int s = p.nst - 1; s >= 0; --s) {
        p.rspan[s] = span;
        p.rinv[s] = ((1 << 20) + span - 1) / span;
        p.rstride[s] = M / (span * best[s]);
        span *= best[s];
    }
    return p.T <= kSmoothThreads;
}
// every pass of every solve asks: the answers (a function of M, of the largest radix and of the fewest stages
// alone, a few thousand at most) are kept
bool smooth_plan_upto(int M, int maxrad, SmoothPlan& p, int minst) {
    if (M < 16 || M > 2048) return false;
    static std::mutex mu;
    static std::map<std::array<int, 3>, SmoothPlan> known;   // M = 0: no plan
    std::lock_guard<std::mutex> lk(mu);
    const std::array<int, 3> key = {M, maxrad, minst};
    auto it = known.find(key);
    if (it == known.end()) {
        SmoothPlan q;
        if (!search_plan(M, maxrad, minst, q)) q = SmoothPlan();
        it = known.emplace(key, q).first;
    }
    p = it->second;
    return p.M == M;
}
bool smooth_plan(int M, SmoothPlan& p) { return smooth_plan_upto(M, 16, p, 2); }

// Pencils: fewest stages, but three of radix 10 at most in the place of two where the two leave the chip short of waves: a stage
// of radix R has M / R threads, so three stages have twice to four times the waves for one more trip through LDS. The
// line lies at 1344 waves (five a CU), at 512 where the three begin with radix 2 (twice the threads of any other
// stage). Measured on whole solves (FP64, two stages -> three) at 40 lengths from 20 to 256: up to 1024 waves
// 0-30 % faster (32 x 320 x 32 walls in x and y, h = 160: 17-20 %), at 1152 to 1300 from 5 % slower (h = 63) to 10 % faster
// (h = 80), from 1500 up to 20 % slower (h = 100); beginning with 2, up to 640 waves 1-20 % faster, at 1024 from 4 %
// slower to 7 % faster. Powers of two keep two: their stages form some twiddles as products, and with one stage more
// 256 x 128 x 96 open is 16-25 % further from the exact solution (all of its rows: Green's function of 512 points; the other
// lengths: within 3 %, as often closer).
static bool pen_plan(const PassDesc& P, int h, SmoothPlan& p) {
    if (!smooth_plan(h, p)) return false;
    SmoothPlan q;
    if (p.nst != 2 || (h & (h - 1)) == 0 || !smooth_plan_upto(h, 10, q, 3)) return true;
    const long long waves = (long long)P.n1 * P.n2 * P.comps * p.T / 64;
    if (waves <= (q.rad[0] == 2 ? 512 : 1344)) p = q;
    return true;
}
// strided pencils for which the plan has a radix above 10
bool smooth_pen_wide(const PassDesc& P, int h) {
    SmoothPlan p;
    return pen_plan(P, h, p) && p.wide;
}

bool smooth_col_tile(PassDesc& P, int n) {
    if (!smooth_plan(n, P.sm)) return false;
    P.ppb = col_tile(n, P.sm.T, P.src_f32 && P.dst_f32);
    return P.ppb > 0;
}
void launch_smooth_col(const PassDesc& P, hipStream_t s) {
    const int ntile = (P.na + P.ppb - 1) / P.ppb;
    launch_io<smooth_col>(P, dim3(ntile * (P.n1 * P.n2 / P.na), P.lda), dim3(P.ppb * P.sm.T), (size_t)P.ppb * P.sm.M * 2 * sizeof(double), s);
}

// about 128 threads a block of contiguous pencils (64: 48, 128: 36, 256: 37, 512: 45 us a pass of 200 reals),
// 16 neighbours of strided ones (128-byte rows; 4: 67, 8: 56, 16: 48, 32: 67 us a pass of 100 reals)
bool smooth_pen_tile(PassDesc& P, int h, bool col) {
    if (!pen_plan(P, h, P.sm)) return false;
    if (col) {
        P.ppb = fit_tile(16, P.sm.T, [&](int np) { return pen_lds(P, true, np); });
        return P.ppb > 0;
    }
    int np = std::max(1, 128 / P.sm.T);
    while (np > 1 && pen_lds(P, false, np) > kSmoothLds) --np;
    P.ppb = std::min(np, P.n1 * P.n2);
    return pen_lds(P, false, P.ppb) <= kSmoothLds;
}
void launch_smooth_pen(const PassDesc& P, bool col, hipStream_t s) {
    const int npen = P.n1 * P.n2;
    const size_t lds = pen_lds(P, col, P.ppb);
    const dim3 block(P.ppb * P.sm.T);
    if (col) launch_smooth_tile(P, dim3((P.na + P.ppb - 1) / P.ppb * (npen / P.na), P.lda), block, lds, s);
    else launch_smooth_row(P, dim3((npen + P.ppb - 1) / P.ppb, P.lda), block, lds, s);
}

// the fused last direction: columns per block (0: no smooth kernel for this length)
int smooth_z_tile(int M, bool f32) {
    SmoothPlan p;
    return smooth_plan(M, p) ? col_tile(M, p.T, f32) : 0;
}
void launch_smooth_z(const SmoothZArgs& A, hipStream_t s) {
    const dim3 grid((A.nx + A.tx - 1) / A.tx * A.nother, A.lda), block(A.tx * A.sm.T);
    const size_t lds = (size_t)A.tx * A.sm.M * 2 * sizeof(double);
    if (A.f32) A.sm.wide ? launch_k<smooth_z<true, float>>(grid, block, lds, s, A) : launch_k<smooth_z<false, float>>(grid, block, lds, s, A);
    else A.sm.wide ? launch_k<smooth_z<true, double>>(grid, block, lds, s, A) : launch_k<smooth_z<false, double>>(grid, block, lds, s, A);
    HIP_CHECK(hipGetLastError());
}

void launch_smooth_rz(const SmoothRzArgs& A, hipStream_t s) {
    const dim3 grid(((A.nx + 1) / 2 + A.tx - 1) / A.tx * A.ny, A.lda), block(A.tx * A.sm.T);
    const size_t lds = (size_t)A.tx * A.sm.M * 2 * sizeof(double);
    if (A.f32) A.sm.wide ? launch_k<smooth_rz<true, float>>(grid, block, lds, s, A) : launch_k<smooth_rz<false, float>>(grid, block, lds, s, A);
    else A.sm.wide ? launch_k<smooth_rz<true, double>>(grid, block, lds, s, A) : launch_k<smooth_rz<false, double>>(grid, block, lds, s, A);
    HIP_CHECK(hipGetLastError());
}

}  // namespace flups
