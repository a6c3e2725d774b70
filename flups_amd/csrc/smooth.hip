// Pass kernels of the general path for the lengths with factors 2, 3, 5, 7 that the register
// kernels of rowpass.hip do not have (9, 15, 25, ... times a power of two: 100, 120, 144, 180, 200,
// 240, 300, ...), on the run-time mixed-radix FFT of smooth_fft.hpp:
//   smooth_col   c2c along a strided direction, values straight between HBM and the first / last
//                stage's registers;
//   smooth_z     the last direction fused with the multiply: forward c2c, normfact G, inverse c2c;
//   smooth_pen   every other pass (r2c, c2r, r2r, c2c of a contiguous pencil; r2c, c2r, r2r of a
//                strided one), pencils staged in LDS, pre- and post-maps from tables.
// Before, these lengths ran on the generic kernel (up to five radix 2-7 stages over LDS, sines and
// cosines computed in its pre- and post-maps, 2n-point extensions for r2r) with a separate multiply
// sweep: 200 x 144 x 100 open 6 x 262 + 80 us, now 48 (x) + 51 (y) + 131 (fused z) + 51 + 48 us, the
// solve 1589 -> 331 us; 240 x 100 x 180 channel 1009 -> 211 us (MI355X, FP64). The passes move their
// minimum bytes at 1.4-2.2 TB/s: bound by the latency of a block's load - stages - store chain.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <vector>

#include "core.hpp"
#include "fft_core.hpp"
#include "group.hpp"
#include "smooth_fft.hpp"

namespace flups {

int r2r_h(int kind, int n);

namespace {

__device__ __forceinline__ C2<double> swapped(C2<double> a, bool s) { return s ? C2<double>{a.y, a.x} : a; }

template <typename TI, typename TO>
struct smooth_col {
    using Args = PassDesc;
    static constexpr int NT = 512, kWaves = 4;
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
        const C2<TI>* src = reinterpret_cast<const C2<TI>*>(P.src) + (long long)ja * P.src_s[P.fa] + (long long)jb * P.src_s[P.fb];
        C2<TO>* dst = reinterpret_cast<C2<TO>*>(P.dst) + (long long)ja * P.dst_s[P.fa] + (long long)jb * P.dst_s[P.fb];
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

template <typename ST>
struct smooth_z {
    using Args = SmoothZArgs;
    static constexpr int NT = 512, kWaves = 4;
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

// Pencils staged in LDS (pb: the pencil's reals; zb: the complex sequence of the FFT). The plan
// semantics are those of the generic kernel; the transforms are the ones of rowpass_kernels.hpp
// (packed half-length FFTs, pre / post tables), without its compile-time lengths.
// COL = false: ppb contiguous pencils, sm.T threads each; COL = true: ppb (a power of two) pencils that
// are neighbours along the unit-stride dimension, interleaved in LDS.
template <bool COL, typename TI, typename TO>
struct smooth_pen {
    using Args = PassDesc;
    static constexpr int NT = 512, kWaves = 4;
    static __device__ __forceinline__ void run(const PassDesc& P, Blk blk) {
        extern __shared__ double smem[];
        const SmoothPlan& S = P.sm;
        const int H = S.M, np = P.ppb, TT = S.T;
        const int nfi = P.nf_in, nfo = P.nf_out, len = P.pen_in * nfi, pin = P.pen_in;
        const int pen = COL ? threadIdx.x & (np - 1) : threadIdx.x / TT;
        const int t = COL ? threadIdx.x / np : threadIdx.x - pen * TT;
        int ja, jb;
        bool live;
        if (COL) {
            const int ntile = (P.na + np - 1) / np;
            const int tile = blk.x % ntile;
            jb = blk.x / ntile;
            ja = tile * np + pen;
            live = ja < P.na;
            if (!live) ja = P.na - 1;   // dead pencils read the last one and store nothing
        } else {
            const int g = blk.x * np + pen;
            live = g < P.n1 * P.n2;
            const int gg = live ? g : 0;
            ja = gg % P.na;
            jb = gg / P.na;
        }
        const TI* src = reinterpret_cast<const TI*>(P.src) + ((long long)ja * P.src_s[P.fa] + (long long)jb * P.src_s[P.fb]) * P.src_nf;
        TO* dst = reinterpret_cast<TO*>(P.dst) + ((long long)ja * P.dst_s[P.fa] + (long long)jb * P.dst_s[P.fb]) * P.dst_nf;
        const long long sd = P.src_s[P.d] * P.src_nf, dd = P.dst_s[P.d] * P.dst_nf;
        double* pb = COL ? smem + pen : smem + pen * len;
        const int es = COL ? np : 1;
        C2<double>* zb = reinterpret_cast<C2<double>*>(smem + ((np * len + 1) & ~1)) + (COL ? pen : pen * (H + H / 8 + 1));
        auto RD = [&](int q) -> double& { return pb[q * es]; };
        auto slot = [&](int e) { return COL ? e * np : e + (e >> 3); };
        const C2<double>* tw = reinterpret_cast<const C2<double>*>(P.tw);     // H-point table
        const C2<double>* A = reinterpret_cast<const C2<double>*>(P.aux);     // r2r: A, B of row_r2r_table; r2c / c2r: n-point table
        const C2<double>* B = A + (H + 1);

        // 1. gather (field shift, zero padding)
        const int lastk = max(P.src_nd - 1, 0);
        if (nfi == 2) {
            staged_gather<4>(t, TT, pin, [&](int k) {
                const int ks = k - P.gshift;
                const TI* p = src + min(max(ks, 0), lastk) * sd;
                const C2<double> x = c2d(*reinterpret_cast<const C2<TI>*>(p));
                return (ks >= 0 && ks < P.src_nd) ? x : C2<double>{0.0, 0.0};
            }, [&](int k, C2<double> x) {
                RD(2 * k) = x.x;
                RD(2 * k + 1) = x.y;
            });
        } else {
            staged_gather<8>(t, TT, pin, [&](int k) {
                const int ks = k - P.gshift;
                const double x = (double)src[min(max(ks, 0), lastk) * sd];
                return (ks >= 0 && ks < P.src_nd) ? x : 0.0;
            }, [&](int k, double x) { RD(k) = x; });
        }
        __syncthreads();

        // 2. pre-map to the complex sequence of length H
        const int kind = P.kind, n = P.n, si = P.si;
        const int dct = kind >= RODFT10 ? kind - 4 : kind;
        const bool r2r = P.op == OP_R2R;
        const bool alt = r2r && kind == RODFT10;                            // input (-1)^q x, output reversed
        const bool rev = r2r && (kind == RODFT01 || kind == RODFT11);       // input reversed, output (-1)^k
        const bool inv = r2r ? dct == REDFT01 : P.op == OP_C2R || (P.op == OP_C2C && P.sign > 0);
        auto xin = [&](int q) -> double {
            const double v = RD(si + (rev ? n - 1 - q : q));
            return (alt && (q & 1)) ? -v : v;
        };
        auto fill = [&](auto z) {
            for (int m = t; m < H; m += TT) zb[slot(m)] = swapped(z(m), inv);
        };
        if (P.op == OP_R2C || P.op == OP_C2C) {
            fill([&](int m) -> C2<double> { return {RD(2 * m), RD(2 * m + 1)}; });
        } else if (P.op == OP_C2R) {
            fill([&](int m) -> C2<double> {
                C2<double> a = {RD(2 * m), RD(2 * m + 1)}, b = {RD(2 * (H - m)), RD(2 * (H - m) + 1)};
                if (m == 0) a.y = b.y = 0.0;   // DC and Nyquist are real
                const C2<double> bc = cconj(b), e = cadd(a, bc), f = csub(a, bc);
                const C2<double> w = cmul(cconj(A[m]), f);   // e^{+2 pi i m / n} (a - conj b)
                return {e.x - w.y, e.y + w.x};
            });
        } else if (kind == REDFT00) {   // e[q] = x[q] (q <= H), x[2H - q] (q > H)
            auto e = [&](int q) { return xin(q <= H ? q : 2 * H - q); };
            fill([&](int m) -> C2<double> { return {e(2 * m), e(2 * m + 1)}; });
        } else if (kind == RODFT00) {   // o[0] = o[H] = 0, o[q] = x[q-1] (q < H), -x[2H-q-1] (q > H)
            auto od = [&](int q) { return (q == 0 || q == H) ? 0.0 : q < H ? xin(q - 1) : -xin(2 * H - q - 1); };
            fill([&](int m) -> C2<double> { return {od(2 * m), od(2 * m + 1)}; });
        } else if (dct == REDFT11) {
            fill([&](int m) -> C2<double> { return cmul(C2<double>{xin(2 * m), xin(n - 1 - 2 * m)}, A[m]); });
        } else if (dct == REDFT10) {
            auto u = [&](int q) { return q < H ? xin(2 * q) : xin(2 * (n - 1 - q) + 1); };
            fill([&](int m) -> C2<double> { return {u(2 * m), u(2 * m + 1)}; });
        } else {   // REDFT01
            auto U = [&](int k) {
                const double a = k < n ? xin(k) : 0.0, b = n - k < n ? xin(n - k) : 0.0;
                return cmul(A[k], C2<double>{a, -b});
            };
            fill([&](int m) -> C2<double> {
                const C2<double> uk = U(m), uc = cconj(U(H - m));
                const C2<double> e = cadd(uk, uc), f = csub(uk, uc), w = cmul(B[m], f);
                return {e.x - w.y, e.y + w.x};
            });
        }
        __syncthreads();

        // 3. FFT of length H
        auto none = [](C2<double>*, int, auto) {};
        for (int s = 0; s < S.nst; ++s) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[s], S.span[s], S.inv[s], S.stride[s], false, false, zb, slot, tw, none, none)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
        }
        auto Z = [&](int k) { return swapped(zb[slot(k)], inv); };
        // real DFT of 2H points from the packed one: (Z[k] + conj Z[H-k])/2 + w[k] (Z[k] - conj Z[H-k])/(2i)
        auto packed = [&](int k, const C2<double>* w) -> C2<double> {
            const C2<double> zk = Z(k), zc = cconj(Z(k == 0 ? 0 : H - k));
            const C2<double> e = {0.5 * (zk.x + zc.x), 0.5 * (zk.y + zc.y)};
            const C2<double> df = {0.5 * (zk.x - zc.x), 0.5 * (zk.y - zc.y)};
            return cadd(e, cmul(w[k], C2<double>{df.y, -df.x}));
        };
        auto nyquist = [&]() { const C2<double> z0 = Z(0); return z0.x - z0.y; };

        // 4. post-map into the pencil
        if (P.op == OP_C2C || P.op == OP_C2R) {
            for (int k = t; k < H; k += TT) {
                const C2<double> z = Z(k);
                RD(2 * k) = z.x;
                RD(2 * k + 1) = z.y;
            }
            if (P.op == OP_C2C) {
                if ((P.post & POST_PERIOD) && t == 0) {   // node-centred periodic copy
                    const C2<double> z = Z(0);
                    RD(2 * H) = z.x;
                    RD(2 * H + 1) = z.y;
                }
            } else {
                for (int q = 2 * H + t; q < P.pen_out; q += TT) RD(q) = (P.post & POST_PERIOD) && q == 2 * H ? Z(0).x : 0.0;
            }
        } else if (P.op == OP_R2C) {
            const int per = (P.post & POST_PERIOD) ? P.n_out_plan - 1 : -1;   // the first value again
            for (int k = t; k < P.pen_out; k += TT) {
                const C2<double> x = k < H ? packed(k, A) : k == H ? C2<double>{nyquist(), 0.0} : k == per ? packed(0, A) : C2<double>{0.0, 0.0};
                RD(2 * k) = x.x;
                RD(2 * k + 1) = x.y;
            }
        } else if (kind == REDFT00) {
            for (int k = t; k <= H; k += TT) RD(k) = k < H ? packed(k, A).x : nyquist();
        } else if (kind == RODFT00) {
            for (int k = 1 + t; k < H; k += TT) RD(k - 1) = -packed(k, A).y;
        } else if (dct == REDFT11) {
            for (int k = t; k < H; k += TT) {
                const C2<double> w = cmul(Z(k), B[k]);
                RD(2 * k) = 2.0 * w.x;
                RD(n - 1 - 2 * k) = -2.0 * w.y;
            }
        } else if (dct == REDFT10) {
            for (int k = t; k < H; k += TT) {
                const C2<double> w = cmul(B[k], packed(k, A));
                RD(k) = 2.0 * w.x;
                if (k > 0) RD(n - k) = -2.0 * w.y;
            }
            if (t == 0) RD(H) = 2.0 * cmul(B[H], C2<double>{nyquist(), 0.0}).x;
        } else {   // REDFT01: u[2m] = Re z[m], u[2m+1] = Im z[m]
            for (int m = t; m < H; m += TT) {
                const C2<double> z = Z(m);
                const int q0 = 2 * m, q1 = 2 * m + 1;
                RD(q0 < H ? 2 * q0 : 2 * (n - 1 - q0) + 1) = z.x;
                RD(q1 < H ? 2 * q1 : 2 * (n - 1 - q1) + 1) = z.y;
            }
        }
        __syncthreads();

        // 5. scatter (truncation)
        if (!live) return;
        if (r2r) {
            const int so = P.so, post = P.post;
            const int nt = kind == REDFT00 ? H + 1 : kind == RODFT00 ? H - 1 : n;
            for (int k = t; k < P.dst_nd; k += TT) {
                const int p = k + P.sshift, q = p - so;
                if (p >= pin) continue;
                double y = 0.0;
                if (!(((post & POST_FIRST) && p == 0) || ((post & POST_LAST) && p == pin - 1)) && q >= 0 && q < nt) {
                    y = RD(alt ? n - 1 - q : q);
                    if (rev && (q & 1)) y = -y;
                }
                dst[k * dd] = (TO)y;
            }
        } else if (nfo == 2) {
            for (int k = t; k < P.dst_nd; k += TT) {
                const int p = k + P.sshift;
                if (p < P.pen_out) *reinterpret_cast<C2<TO>*>(dst + k * dd) = c2t<TO>({RD(2 * p), RD(2 * p + 1)});
            }
        } else {
            for (int k = t; k < P.dst_nd; k += TT) {
                const int p = k + P.sshift;
                if (p < P.pen_out) dst[k * dd] = (TO)RD(p);
            }
        }
    }
};

template <template <typename, typename> class K>
void launch_io(const PassDesc& P, dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    if (!P.src_f32 && !P.dst_f32) launch_k<K<double, double>>(grid, block, lds, s, P);
    else if (!P.src_f32) launch_k<K<double, float>>(grid, block, lds, s, P);
    else if (P.dst_f32) launch_k<K<float, float>>(grid, block, lds, s, P);
    else launch_k<K<float, double>>(grid, block, lds, s, P);
    HIP_CHECK(hipGetLastError());
}
template <typename TI, typename TO>
using smooth_row = smooth_pen<false, TI, TO>;
template <typename TI, typename TO>
using smooth_tile = smooth_pen<true, TI, TO>;

constexpr size_t kSmoothLds = 65536;   // bytes of one block
constexpr int kSmoothThreads = 512;

size_t pen_lds(const PassDesc& P, bool col, int np) {
    const size_t len = (size_t)P.pen_in * P.nf_in, H = P.sm.M;
    return ((np * len + 1) & ~(size_t)1) * sizeof(double) + np * (col ? H : H + H / 8 + 1) * 2 * sizeof(double);
}
// largest power of two <= lim with np T threads and its LDS within one block (0: none)
template <typename Lds>
int fit_tile(int lim, int T, Lds&& lds) {
    for (int np = lim; np >= 1; np /= 2)
        if (np * T <= kSmoothThreads && lds(np) <= kSmoothLds) return np;
    return 0;
}

}  // namespace

// fewest stages, then fewest threads (the largest smallest radix), radices ascending: every thread
// takes part in the first and the last stage, the ones that meet HBM
static bool search_plan(int M, SmoothPlan& p) {
    static const int rads[13] = {2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16};
    std::vector<int> cur, best;
    auto search = [&](auto&& self, int m, int lo) -> void {
        if (m == 1) {
            if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && cur[0] > best[0])) best = cur;
            return;
        }
        if ((int)cur.size() == kSmoothStages) return;
        for (int i = lo; i < 13; ++i)
            if (m % rads[i] == 0) {
                cur.push_back(rads[i]);
                self(self, m / rads[i], i);
                cur.pop_back();
            }
    };
    search(search, M, 0);
    if (best.size() < 2) return false;
    p = SmoothPlan();
    p.M = M;
    p.nst = (int)best.size();
    p.T = M / best[0];
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
// every pass of every solve asks: the answers (a function of M alone, at most 2031 of them) are kept
bool smooth_plan(int M, SmoothPlan& p) {
    if (M < 18 || M > 2048) return false;
    static std::mutex mu;
    static std::map<int, SmoothPlan> known;   // M = 0: no plan
    std::lock_guard<std::mutex> lk(mu);
    auto it = known.find(M);
    if (it == known.end()) {
        SmoothPlan q;
        if (!search_plan(M, q)) q = SmoothPlan();
        it = known.emplace(M, q).first;
    }
    p = it->second;
    return p.M == M;
}

// strided c2c: columns per block, 8 (128-byte rows) where the LDS allows
bool smooth_col_tile(PassDesc& P, int n) {
    if (!smooth_plan(n, P.sm)) return false;
    P.ppb = fit_tile(8, P.sm.T, [&](int np) { return (size_t)np * n * 2 * sizeof(double); });
    return P.ppb > 0;
}
void launch_smooth_col(const PassDesc& P, hipStream_t s) {
    const int ntile = (P.na + P.ppb - 1) / P.ppb;
    launch_io<smooth_col>(P, dim3(ntile * (P.n1 * P.n2 / P.na)), dim3(P.ppb * P.sm.T), (size_t)P.ppb * P.sm.M * 2 * sizeof(double), s);
}

// pencils staged in LDS: about 256 threads a block of contiguous pencils, 16 neighbours of strided ones
bool smooth_pen_tile(PassDesc& P, int h, bool col) {
    if (!smooth_plan(h, P.sm)) return false;
    if (col) {
        P.ppb = fit_tile(16, P.sm.T, [&](int np) { return pen_lds(P, true, np); });
        return P.ppb > 0;
    }
    int np = std::max(1, 256 / P.sm.T);
    while (np > 1 && pen_lds(P, false, np) > kSmoothLds) --np;
    P.ppb = std::min(np, P.n1 * P.n2);
    return pen_lds(P, false, P.ppb) <= kSmoothLds;
}
void launch_smooth_pen(const PassDesc& P, bool col, hipStream_t s) {
    const int npen = P.n1 * P.n2;
    const size_t lds = pen_lds(P, col, P.ppb);
    const dim3 block(P.ppb * P.sm.T);
    if (col) launch_io<smooth_tile>(P, dim3((P.na + P.ppb - 1) / P.ppb * (npen / P.na)), block, lds, s);
    else launch_io<smooth_row>(P, dim3((npen + P.ppb - 1) / P.ppb), block, lds, s);
}

// the fused last direction: columns per block (0: no smooth kernel for this length)
int smooth_z_tile(int M) {
    SmoothPlan p;
    if (!smooth_plan(M, p)) return 0;
    return fit_tile(8, p.T, [&](int np) { return (size_t)np * M * 2 * sizeof(double); });
}
void launch_smooth_z(const SmoothZArgs& A, hipStream_t s) {
    const dim3 grid((A.nx + A.tx - 1) / A.tx * A.nother, A.lda), block(A.tx * A.sm.T);
    const size_t lds = (size_t)A.tx * A.sm.M * 2 * sizeof(double);
    if (A.f32) launch_k<smooth_z<float>>(grid, block, lds, s, A);
    else launch_k<smooth_z<double>>(grid, block, lds, s, A);
    HIP_CHECK(hipGetLastError());
}

}  // namespace flups
