// The pencil kernel of smooth.hip (smooth_pen) and the launch over the storage types of a pass; smooth_row.hip
// and smooth_tile.hip compile its two layouts beside each other.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "core.hpp"
#include "fft_core.hpp"
#include "group.hpp"
#include "smooth_fft.hpp"

namespace flups {

namespace {

__device__ __forceinline__ C2<double> swapped(C2<double> a, bool s) { return s ? C2<double>{a.y, a.x} : a; }

// Every other pass. The pre-map reads the pencil from HBM in the order of the complex sequence of the
// FFT and writes that sequence to LDS, the stages run there, and the post-map computes each stored
// value from it: no copy of the pencil itself (with one, 200 x 144 x 100 open: 48 us a pass of x).
// The plan semantics are those of the generic kernel; the transforms are the ones of
// rowpass_kernels.hpp (packed half-length FFTs, pre / post tables), without its compile-time lengths.
// COL = false: ppb contiguous pencils, sm.T threads each; COL = true: ppb (a power of two) pencils that
// are neighbours along the unit-stride dimension, interleaved in LDS.
template <bool WIDE, bool COL, typename TI, typename TO>
struct smooth_pen {
    using Args = PassDesc;
    static constexpr int NT = 512, kWaves = WIDE ? 4 : 5;
    static __device__ __forceinline__ void run(const PassDesc& P, Blk blk) {
        extern __shared__ double smem[];
        const SmoothPlan& S = P.sm;
        const int H = S.M, np = P.ppb, TT = S.T, pin = P.pen_in;
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
        const TI* src = P.from<TI>(blk.y) + ((long long)ja * P.src_s[P.fa] + (long long)jb * P.src_s[P.fb]) * P.src_nf;
        TO* dst = P.to<TO>(blk.y) + ((long long)ja * P.dst_s[P.fa] + (long long)jb * P.dst_s[P.fb]) * P.dst_nf;
        const long long sd = COL ? P.src_s[P.d] * P.src_nf : P.src_nf, dd = COL ? P.dst_s[P.d] * P.dst_nf : P.dst_nf;
        C2<double>* zb = reinterpret_cast<C2<double>*>(smem) + (COL ? pen : pen * (H + H / 8 + 1));
        auto slot = [&](int e) { return COL ? e * np : e + (e >> 3); };
        const C2<double>* tw = reinterpret_cast<const C2<double>*>(P.tw);     // H-point table
        const C2<double>* A = reinterpret_cast<const C2<double>*>(P.aux);     // r2r: A, B of row_r2r_table; r2c / c2r: n-point table
        const C2<double>* B = A + (H + 1);

        // 1. pencil position k (field shift, zero padding: a load at a clamped address, zero selected)
        const int lastk = max(P.src_nd - 1, 0);
        auto xr = [&](int k) -> double {
            const int ks = k - P.gshift;
            const double x = (double)src[min(max(ks, 0), lastk) * sd];
            return (ks >= 0 && ks < P.src_nd) ? x : 0.0;
        };
        auto xc = [&](int k) -> C2<double> {
            const int ks = k - P.gshift;
            const C2<double> x = c2d(*reinterpret_cast<const C2<TI>*>(src + min(max(ks, 0), lastk) * sd));
            return (ks >= 0 && ks < P.src_nd) ? x : C2<double>{0.0, 0.0};
        };
        const int kind = P.kind, n = P.n, si = P.si;
        const int dct = kind >= RODFT10 ? kind - 4 : kind;
        const bool r2r = P.op == OP_R2R;
        const bool alt = r2r && kind == RODFT10;                            // input (-1)^q x, output reversed
        const bool rev = r2r && (kind == RODFT01 || kind == RODFT11);       // input reversed, output (-1)^k
        const bool inv = r2r ? dct == REDFT01 : P.op == OP_C2R || (P.op == OP_C2C && P.sign > 0);
        auto xin = [&](int q) -> double {
            const double v = xr(si + (rev ? n - 1 - q : q));
            return (alt && (q & 1)) ? -v : v;
        };
        // 2. pre-map: element m of the complex sequence of length H into LDS, two items' loads together.
        // Where elements m and H - m come from the same inputs one thread makes both. r2c and c2c
        // sequences need no map: the first stage reads them from HBM.
        const int HH = H / 2 + 1;
        auto put = [&](int m, C2<double> v) { zb[slot(m)] = swapped(v, inv); };
        auto fill = [&](auto z) { staged_gather<2>(t, TT, H, z, put); };
        struct Pair {
            C2<double> a, b;
        };
        auto fill2 = [&](auto z) {   // z(m): elements m and H - m, m <= H / 2
            staged_gather<2>(t, TT, HH, z, [&](int m, Pair p) {
                put(m, p.a);
                if (m > 0 && 2 * m != H) put(H - m, p.b);
            });
        };
        auto ext = [&](C2<double>* v, int mp, auto r) {
            constexpr int R = decltype(r)::value;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int m = t + q * mp;
                v[q] = swapped(P.op == OP_R2C ? C2<double>{xr(2 * m), xr(2 * m + 1)} : xc(m), inv);
            }
        };
        const bool direct_in = P.op == OP_R2C || P.op == OP_C2C;
        if (P.op == OP_C2R) {
            // Z[m] = (X[m] + conj X[H-m]) + i w (X[m] - conj X[H-m]), w = e^{2 pi i m / n}; Z[H-m] the
            // conjugate of the same terms with the other sign
            fill2([&](int m) -> Pair {
                C2<double> a = xc(m), b = xc(H - m);
                if (m == 0) a.y = b.y = 0.0;   // DC and Nyquist are real
                const C2<double> bc = cconj(b), e = cadd(a, bc), f = csub(a, bc);
                const C2<double> w = cmul(cconj(A[m]), f);
                return {{e.x - w.y, e.y + w.x}, {e.x + w.y, w.x - e.y}};
            });
        } else if (direct_in) {
        } else if (kind == REDFT00) {   // e[q] = x[q] (q <= H), x[2H - q] (q > H)
            auto e = [&](int q) { return xin(q <= H ? q : 2 * H - q); };
            fill([&](int m) -> C2<double> { return {e(2 * m), e(2 * m + 1)}; });
        } else if (kind == RODFT00) {   // o[0] = o[H] = 0, o[q] = x[q-1] (q < H), -x[2H-q-1] (q > H)
            auto od = [&](int q) {
                const double x = xin(q == 0 || q == H ? 0 : q < H ? q - 1 : 2 * H - q - 1);
                return q == 0 || q == H ? 0.0 : q < H ? x : -x;
            };
            fill([&](int m) -> C2<double> { return {od(2 * m), od(2 * m + 1)}; });
        } else if (dct == REDFT11) {
            fill([&](int m) -> C2<double> { return cmul(C2<double>{xin(2 * m), xin(n - 1 - 2 * m)}, A[m]); });
        } else if (dct == REDFT10) {
            auto u = [&](int q) { return xin(q < H ? 2 * q : 2 * (n - 1 - q) + 1); };
            fill([&](int m) -> C2<double> { return {u(2 * m), u(2 * m + 1)}; });
        } else {   // REDFT01: Z[m] = (U[m] + conj U[H-m]) + i B[m] (U[m] - conj U[H-m]), U[k] = A[k] (x[k] - i x[n-k])
            auto U = [&](int k) {   // x[n] = 0
                const double a = xin(k), b = xin(min(n - k, n - 1));
                return cmul(A[k], C2<double>{a, k > 0 ? -b : 0.0});
            };
            fill2([&](int m) -> Pair {
                const C2<double> uk = U(m), uc = cconj(U(H - m));
                const C2<double> e = cadd(uk, uc), f = csub(uk, uc), w = cmul(B[m], f);
                return {{e.x - w.y, e.y + w.x}, {e.x + w.y, w.x - e.y}};
            });
        }

        // 3. FFT of length H; c2r and c2c results go to HBM from the last stage
        const bool per = P.post & POST_PERIOD;   // the first value again at the end of the pencil
        auto out = [&](C2<double>* v, int mp, auto r) {
            constexpr int R = decltype(r)::value;
            if (!live) return;
            const int lim = min(P.dst_nd, P.pen_out - P.sshift);
            if (P.op == OP_C2C) {
                C2<TO>* d = reinterpret_cast<C2<TO>*>(dst);
                const long long ds = dd / 2;
#pragma unroll
                for (int u = 0; u < R; ++u) {
                    const int k = t + u * mp - P.sshift;
                    if (k >= 0 && k < lim) d[k * ds] = c2t<TO>(swapped(v[u], inv));
                }
                const int k = H - P.sshift;
                if (per && t == 0 && k >= 0 && k < lim) d[k * ds] = c2t<TO>(swapped(v[0], inv));
                return;
            }
            // x[2m] = Re z[m], x[2m+1] = Im z[m], stored as one where the pair is contiguous and aligned
            const bool vec = !COL && P.sshift == 0 && (reinterpret_cast<uintptr_t>(dst) & (2 * sizeof(TO) - 1)) == 0;
#pragma unroll
            for (int u = 0; u < R; ++u) {
                const C2<double> z = swapped(v[u], inv);
                const int k = 2 * (t + u * mp) - P.sshift;
                if (vec && k + 1 < lim) {
                    *reinterpret_cast<C2<TO>*>(dst + k) = c2t<TO>(z);
                } else {
                    if (k >= 0 && k < lim) dst[k * dd] = (TO)z.x;
                    if (k + 1 >= 0 && k + 1 < lim) dst[(k + 1) * dd] = (TO)z.y;
                }
            }
            if (t == 0)
                for (int k = max(2 * H - P.sshift, 0); k < lim; ++k)   // positions past the transform
                    dst[k * dd] = per && k + P.sshift == 2 * H ? (TO)swapped(v[0], inv).x : (TO)0;
        };
        auto none = [](C2<double>*, int, auto) {};
        const bool direct_out = P.op == OP_C2R || P.op == OP_C2C;
        int s0 = 0, s1 = S.nst;
        if (direct_in) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[0], 1, S.inv[0], S.stride[0], true, false, zb, slot, tw, ext, none)
            FLUPS_SMOOTH_RADIX(S.rad[0], FLUPS_CALL)
#undef FLUPS_CALL
            s0 = 1;
        } else {
            __syncthreads();
        }
        if (direct_out) --s1;
        for (int s = s0; s < s1; ++s) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[s], S.span[s], S.inv[s], S.stride[s], false, false, zb, slot, tw, none, none)
            FLUPS_SMOOTH_RADIX(S.rad[s], FLUPS_CALL)
#undef FLUPS_CALL
        }
        if (direct_out) {
#define FLUPS_CALL(R) smooth_stage<R>(t, S.mp[s1], S.span[s1], S.inv[s1], S.stride[s1], false, true, zb, slot, tw, none, out)
            FLUPS_SMOOTH_RADIX(S.rad[s1], FLUPS_CALL)
#undef FLUPS_CALL
            return;
        }
        if (!live) return;
        auto Z = [&](int k) { return swapped(zb[slot(k)], inv); };
        // real DFT of 2H points from the packed one, outputs m and H - m (m <= H / 2): X[m] = e + w[m] o,
        // X[H-m] = conj(e - w[m] o), e = (Z[m] + conj Z[H-m]) / 2, o = (Z[m] - conj Z[H-m]) / (2i)
        auto packed = [&](int m, const C2<double>* w) -> Pair {
            const C2<double> zk = Z(m), zc = cconj(Z(m == 0 ? 0 : H - m));
            const C2<double> e = {0.5 * (zk.x + zc.x), 0.5 * (zk.y + zc.y)};
            const C2<double> df = {0.5 * (zk.x - zc.x), 0.5 * (zk.y - zc.y)};
            const C2<double> o = cmul(w[m], C2<double>{df.y, -df.x});
            return {cadd(e, o), cconj(csub(e, o))};
        };

        // 4. post-map and scatter (truncation): pencil position p is stored at element p - sshift; two
        // items' LDS and table loads before the first of their stores
        const int lim = min(P.dst_nd, P.pen_out - P.sshift);
        auto post2 = [&](int items, auto get, auto use) { staged_gather<2>(t, TT, items, get, use); };
        if (P.op == OP_R2C) {
            auto st = [&](int p, C2<double> v) {
                const int k = p - P.sshift;
                if (k >= 0 && k < lim) *reinterpret_cast<C2<TO>*>(dst + k * dd) = c2t<TO>(v);
            };
            post2(HH, [&](int m) { return packed(m, A); }, [&](int m, Pair x) {
                st(m, x.a);
                if (2 * m != H) st(H - m, x.b);
            });
            // positions past H: zero, and the first value again at the end of a node-centred periodic pencil
            for (int p = H + 1 + t; p < P.pen_out; p += TT)
                st(p, per && p == P.n_out_plan - 1 ? packed(0, A).a : C2<double>{0.0, 0.0});
            return;
        }
        const int so = P.so, post = P.post;
        const int nt = kind == REDFT00 ? H + 1 : kind == RODFT00 ? H - 1 : n;   // transform outputs
        auto st = [&](int q, double v) {   // transform output q (before the reflections)
            if (alt) q = n - 1 - q;
            const int p = q + so, k = p - P.sshift;
            if (((post & POST_FIRST) && p == 0) || ((post & POST_LAST) && p == pin - 1)) v = 0.0;
            if (k >= 0 && k < lim) dst[k * dd] = (TO)(rev && (q & 1) ? -v : v);
        };
        if (kind == REDFT00) {
            post2(HH, [&](int m) { return packed(m, A); }, [&](int m, Pair x) {
                st(m, x.a.x);
                if (2 * m != H) st(H - m, x.b.x);
            });
        } else if (kind == RODFT00) {
            post2(HH, [&](int m) { return packed(m, A); }, [&](int m, Pair x) {
                if (m == 0) return;
                st(m - 1, -x.a.y);
                if (2 * m != H) st(H - m - 1, -x.b.y);
            });
        } else if (dct == REDFT11) {   // W[m] = Z[m] B[m]: y[2m] = 2 Re W[m], y[n-1-2m] = -2 Im W[m]
            post2(H, [&](int m) { return cmul(Z(m), B[m]); }, [&](int m, C2<double> w) {
                st(2 * m, 2.0 * w.x);
                st(n - 1 - 2 * m, -2.0 * w.y);
            });
        } else if (dct == REDFT10) {   // W[m] = B[m] X[m]: y[m] = 2 Re W[m] (m <= H), y[n-m] = -2 Im W[m] (0 < m < H)
            post2(HH, [&](int m) -> Pair {
                const Pair x = packed(m, A);
                return {cmul(B[m], x.a), cmul(B[H - m], x.b)};
            }, [&](int m, Pair w) {
                st(m, 2.0 * w.a.x);
                if (m > 0) st(n - m, -2.0 * w.a.y);
                if (2 * m != H) {
                    st(H - m, 2.0 * w.b.x);
                    if (m > 0) st(H + m, -2.0 * w.b.y);
                }
            });
        } else {   // REDFT01: u[2m] = Re z[m], u[2m+1] = Im z[m]; y[2q] = u[q], y[2q+1] = u[n-1-q]
            post2(H, Z, [&](int m, C2<double> z) {
                const int q0 = 2 * m, q1 = 2 * m + 1;
                st(q0 < H ? 2 * q0 : 2 * (n - 1 - q0) + 1, z.x);
                st(q1 < H ? 2 * q1 : 2 * (n - 1 - q1) + 1, z.y);
            });
        }
        // positions before and after the transform's outputs are zero (cleared by the plan's post-correction)
        for (int p = t; p < pin; p += TT) {
            const int k = p - P.sshift;
            if ((p < so || p >= so + nt) && k >= 0 && k < lim) dst[k * dd] = (TO)0;
        }
    }
};

template <template <bool, typename, typename> class K>
void launch_io(const PassDesc& P, dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    auto go = [&](auto wide) {
        constexpr bool W = decltype(wide)::value;
        if (!P.src_f32 && !P.dst_f32) launch_k<K<W, double, double>>(grid, block, lds, s, P);
        else if (!P.src_f32) launch_k<K<W, double, float>>(grid, block, lds, s, P);
        else if (P.dst_f32) launch_k<K<W, float, float>>(grid, block, lds, s, P);
        else launch_k<K<W, float, double>>(grid, block, lds, s, P);
    };
    if (P.sm.wide) go(std::true_type());
    else go(std::false_type());
    HIP_CHECK(hipGetLastError());
}
}  // namespace

}  // namespace flups
