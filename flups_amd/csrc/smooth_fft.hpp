// FFT of any length with factors 2, 3, 5, 7 held in LDS, by stages of radix 2 to 16 chosen at run
// time (SmoothPlan): one thread computes one radix-R butterfly of a stage in registers, a pencil
// of M points takes T = max M / R threads. The stages run in place on one LDS buffer (read,
// barrier, write, barrier). Two stages serve most lengths up to 256, three those up to 1024.
//
// The radices are a run-time choice because the lengths are: a compile-time kernel for each of
// the about 90 even lengths of that kind up to 1024 (and each of the pass shapes) would not be
// buildable, while one division by the span and one switch per stage cost little beside a
// butterfly of 5 to 16 values. Sign: forward transforms only; an inverse one swaps the real and
// imaginary parts of its input and of its output.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "core.hpp"
#include "fft_core.hpp"

namespace flups {

// cos / sin (2 pi e / R) of the radices that need inner twiddles (9 = 3 x 3, 16 = 4 x 4)
template <int R>
__device__ __forceinline__ constexpr C2<double> inner_w(int e) {
    if constexpr (R == 9) {
        return e == 1 ? C2<double>{0.76604444311897803520, -0.64278760968653932632}
             : e == 2 ? C2<double>{0.17364817766693034885, -0.98480775301220805937}
             : e == 4 ? C2<double>{-0.93969262078590838405, -0.34202014332566873304}
                      : C2<double>{1.0, 0.0};
    } else {
        return e == 1 ? C2<double>{0.92387953251128675613, -0.38268343236508977173}
             : e == 2 ? C2<double>{0.70710678118654752440, -0.70710678118654752440}
             : e == 3 ? C2<double>{0.38268343236508977173, -0.92387953251128675613}
             : e == 4 ? C2<double>{0.0, -1.0}
             : e == 6 ? C2<double>{-0.70710678118654752440, -0.70710678118654752440}
             : e == 9 ? C2<double>{-0.92387953251128675613, 0.38268343236508977173}
                      : C2<double>{1.0, 0.0};
    }
}

template <int R>
__device__ __forceinline__ void dft_r(C2<double>* v);

// R = P Q, P and Q coprime (no inner twiddles): n = (Q n1 + P n2) mod R, and output k with
// k mod P = k1, k mod Q = k2
template <int P, int Q>
__device__ __forceinline__ void dft_coprime(C2<double>* v) {
    constexpr int R = P * Q;
    C2<double> t[Q][P];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < P; ++n1) t[n2][n1] = v[(Q * n1 + P * n2) % R];
        dft_r<P>(t[n2]);   // sum over n1 of w_P^(Q n1 k / ...): row (Q k1) mod P below
    }
    // with n = Q n1 + P n2: w_R^(n k) = w_P^(n1 k) w_Q^(n2 k), so row k mod P, column k mod Q
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
        C2<double> u[Q];
#pragma unroll
        for (int n2 = 0; n2 < Q; ++n2) u[n2] = t[n2][k1];
        dft_r<Q>(u);
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k % P == k1) v[k] = u[k % Q];
    }
}

// R = P Q with inner twiddles (9 = 3 x 3, 16 = 4 x 4): n = Q n1 + n2, k = k1 + P k2
template <int P, int Q>
__device__ __forceinline__ void dft_twiddled(C2<double>* v) {
    constexpr int R = P * Q;
    C2<double> t[Q][P];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < P; ++n1) t[n2][n1] = v[Q * n1 + n2];
        dft_r<P>(t[n2]);
#pragma unroll
        for (int k1 = 1; k1 < P; ++k1)
            if (n2 > 0) t[n2][k1] = cmul(t[n2][k1], inner_w<R>(n2 * k1));
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
        C2<double> u[Q];
#pragma unroll
        for (int n2 = 0; n2 < Q; ++n2) u[n2] = t[n2][k1];
        dft_r<Q>(u);
#pragma unroll
        for (int k2 = 0; k2 < Q; ++k2) v[k1 + P * k2] = u[k2];
    }
}

// odd prime R by its symmetric halves: X_k, X_(R-k) = a_0 + sum_j cos(2 pi j k / R) (a_j + a_(R-j))
// -+ i sum_j sin(2 pi j k / R) (a_j - a_(R-j))
template <int R>
__device__ __forceinline__ void dft_odd(C2<double>* v) {
    constexpr int H = (R - 1) / 2;
    constexpr double c[3] = {R == 3 ? -0.5 : R == 5 ? 0.30901699437494742410 : 0.62348980185873353053,
                             R == 5 ? -0.80901699437494742410 : -0.22252093395631440429, -0.90096886790241912624};
    constexpr double s[3] = {R == 3 ? 0.86602540378443864676 : R == 5 ? 0.95105651629515357212 : 0.78183148246802980871,
                             R == 5 ? 0.58778525229247312917 : 0.97492791218182360702, 0.43388373911755812048};
    C2<double> p[H], m[H];
#pragma unroll
    for (int j = 0; j < H; ++j) {
        p[j] = cadd(v[j + 1], v[R - 1 - j]);
        m[j] = csub(v[j + 1], v[R - 1 - j]);
    }
    const C2<double> a0 = v[0];
#pragma unroll
    for (int j = 0; j < H; ++j) v[0] = cadd(v[0], p[j]);
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        C2<double> e = a0, o = {0.0, 0.0};
#pragma unroll
        for (int j = 0; j < H; ++j) {
            const int q = ((j + 1) * k) % R;              // cos even, sin odd around R
            const int h = q <= H ? q - 1 : R - q - 1;
            const double sg = q <= H ? s[h] : -s[h];
            e.x += c[h] * p[j].x;
            e.y += c[h] * p[j].y;
            o.x += sg * m[j].x;
            o.y += sg * m[j].y;
        }
        v[k] = {e.x + o.y, e.y - o.x};       // e - i o
        v[R - k] = {e.x - o.y, e.y + o.x};
    }
}

template <int R>
__device__ __forceinline__ void dft_r(C2<double>* v) {
    if constexpr (R == 2) dft2<double, true>(v[0], v[1]);
    else if constexpr (R == 4) dft4<double, true>(v[0], v[1], v[2], v[3]);
    else if constexpr (R == 8) dft8<double, true>(v);
    else if constexpr (R == 3 || R == 5 || R == 7) dft_odd<R>(v);
    else if constexpr (R == 6) dft_coprime<2, 3>(v);
    else if constexpr (R == 10) dft_coprime<2, 5>(v);
    else if constexpr (R == 12) dft_coprime<4, 3>(v);
    else if constexpr (R == 14) dft_coprime<2, 7>(v);
    else if constexpr (R == 15) dft_coprime<3, 5>(v);
    else if constexpr (R == 9) dft_twiddled<3, 3>(v);
    else dft_twiddled<4, 4>(v);
}

// v[q] *= w^q, q < R, w = tw[e]. Powers of two: w, w^2, w^3 and w^4, w^8, w^12 from the table, the others as one
// product w^(4a) w^b of two of them (fewer loads, one rounding more; with table values alone 2-D 1024^2 66 -> 69 us).
// The other radices take every value from the table: as fast, and more exact.
template <int R>
__device__ __forceinline__ void twiddle_r(C2<double>* v, const C2<double>* tw, int e) {
    if constexpr ((R & (R - 1)) != 0) {
#pragma unroll
        for (int q = 1; q < R; ++q) v[q] = cmul(v[q], tw[q * e]);
    } else {
        C2<double> w[4];
#pragma unroll
        for (int q = 1; q < 4 && q < R; ++q) {
            w[q] = tw[q * e];
            v[q] = cmul(v[q], w[q]);
        }
#pragma unroll
        for (int a = 4; a < R; a += 4) {
            const C2<double> wa = tw[a * e];
            v[a] = cmul(v[a], wa);
#pragma unroll
            for (int q = a + 1; q < a + 4 && q < R; ++q) v[q] = cmul(v[q], cmul(wa, w[q - a]));
        }
    }
}

// Stage of radix R = M / mp over one pencil by its T threads (t < T), in place in LDS. span: product of the
// radices before it; inv: ceil(2^20 / span), so that j / span = (j inv) >> 20 for j < 2048;
// stride = mp / span, the table step of w_(span R). All of them come from the plan's arrays by the
// stage's number: computed from M here, they would be hoisted out of a loop over the stages for every
// radix of the switch (hundreds of spilled registers).
// GET: ext(v, mp) fills v[q] = x[t + q mp] instead of the LDS reads (first stage); PUT: out(v, mp)
// takes v[u] = X[t + u mp] instead of the LDS writes (last stage). Every thread of the block calls this.
template <int R, typename Ext, typename Out, typename Slot>
__device__ __forceinline__ void smooth_stage(int t, int mp, int span, int inv, int stride, bool get, bool put, C2<double>* lds, Slot slot,
                                             const C2<double>* tw, Ext ext, Out out) {
    const bool on = t < mp;
    const int b = (int)(((unsigned)t * (unsigned)inv) >> 20), k = t - b * span;
    C2<double> v[R];
    if (on) {
        if (get) {
            ext(v, mp, std::integral_constant<int, R>{});
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) v[q] = lds[slot(t + q * mp)];
            if (span > 1) twiddle_r<R>(v, tw, k * stride);
        }
        dft_r<R>(v);
    }
    if (put) {
        if (on) out(v, mp, std::integral_constant<int, R>{});
        return;
    }
    __syncthreads();   // the stage's inputs are read
    if (on) {
        const int o = b * span * R + k;
#pragma unroll
        for (int u = 0; u < R; ++u) lds[slot(o + u * span)] = v[u];
    }
    __syncthreads();
}

// one case per radix; WIDE kernels have all of them, the others those up to 10
#define FLUPS_SMOOTH_RADIX(R_, CALL)                                  \
    switch (R_) {                                                     \
        case 2: { CALL(2); } break;                                   \
        case 3: { CALL(3); } break;                                   \
        case 4: { CALL(4); } break;                                   \
        case 5: { CALL(5); } break;                                   \
        case 6: { CALL(6); } break;                                   \
        case 7: { CALL(7); } break;                                   \
        case 8: { CALL(8); } break;                                   \
        case 9: { CALL(9); } break;                                   \
        case 10: { CALL(10); } break;                                 \
        case 12: { if constexpr (WIDE) { CALL(12); } } break;         \
        case 14: { if constexpr (WIDE) { CALL(14); } } break;         \
        case 15: { if constexpr (WIDE) { CALL(15); } } break;         \
        default: { if constexpr (WIDE) { CALL(16); } } break;         \
    }

}  // namespace flups
