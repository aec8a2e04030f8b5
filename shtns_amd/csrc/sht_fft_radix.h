// sht_fft_radix.h -- in-register DFTs, twiddles and block numbering shared by the longitude FFT
// kernels (sht_fft.hip, sht_fft_any.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <utility>

namespace shtns_amd {
namespace {

// ---- compile-time helpers ---------------------------------------------------------------
template <class F, int... I>
__device__ __forceinline__ void sfor_(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
// calls f(integral_constant<int, i>) for i = 0 .. N-1
template <int N, class F>
__device__ __forceinline__ void sfor(F &&f) {
    sfor_(f, std::make_integer_sequence<int, N>{});
}

// cos(2 pi j / 96)
constexpr double cos96(int j) {
    constexpr double c[25] = {1.0,
                              0.997858923238603506738,
                              0.991444861373810411145,
                              0.980785280403230449126,
                              0.96592582628906828675,
                              0.946930129495105664256,
                              0.923879532511286756128,
                              0.896872741532688303894,
                              0.866025403784438646764,
                              0.831469612302545237079,
                              0.79335334029123516458,
                              0.751839807478977396408,
                              0.707106781186547524401,
                              0.659345815100068868425,
                              0.608761429008720639416,
                              0.555570233019602224743,
                              0.5,
                              0.442288690219001281995,
                              0.382683432365089771728,
                              0.321439465303161580701,
                              0.258819045102520762349,
                              0.195090322016128267848,
                              0.130526192220051591548,
                              0.0654031292301430668153,
                              0.0};
    j = ((j % 96) + 96) % 96;
    return j <= 24 ? c[j] : j <= 48 ? -c[48 - j] : j <= 72 ? -c[j - 48] : c[96 - j];
}
constexpr double sin96(int j) { return cos96(j - 24); }

// a * exp(SGN * 2 pi i J / 96), quarter turns without multiplies
template <int J, int SGN>
__device__ __forceinline__ double2 rot96(double2 a) {
    constexpr int j = ((J % 96) + 96) % 96;
    if constexpr (j == 0) {
        return a;
    } else if constexpr (j == 48) {
        return make_double2(-a.x, -a.y);
    } else if constexpr ((j == 24 && SGN > 0) || (j == 72 && SGN < 0)) {
        return make_double2(-a.y, a.x);   // * i
    } else if constexpr (j == 24 || j == 72) {
        return make_double2(a.y, -a.x);   // * -i
    } else {
        constexpr double c = cos96(j), s = SGN * sin96(j);
        return make_double2(a.x * c - a.y * s, a.x * s + a.y * c);
    }
}

__device__ __forceinline__ double2 c_add(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 c_sub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 c_mul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 c_conj(double2 a) { return make_double2(a.x, -a.y); }

// In-register DFT of P points: y_k = sum_n x_n exp(SGN 2 pi i n k / P), P | 96 or 5, 7, 9, 10, 15.
// Composite P = p1 * p2 splits as n = p2 n1 + n2, k = k1 + p1 k2.
template <int P, int SGN>
__device__ __forceinline__ void dft(double2 *x) {
    if constexpr (P == 1) {
    } else if constexpr (P == 2) {
        const double2 a = x[0], b = x[1];
        x[0] = c_add(a, b);
        x[1] = c_sub(a, b);
    } else if constexpr (P == 3) {
        constexpr double h = 0.86602540378443864676 * SGN;   // sin(2 pi / 3)
        const double2 s = c_add(x[1], x[2]), d = c_sub(x[1], x[2]);
        const double2 t = make_double2(x[0].x - 0.5 * s.x, x[0].y - 0.5 * s.y);
        const double2 u = make_double2(-h * d.y, h * d.x);
        x[0] = c_add(x[0], s);
        x[1] = c_add(t, u);
        x[2] = c_sub(t, u);
    } else if constexpr (P == 4) {
        const double2 a = c_add(x[0], x[2]), b = c_sub(x[0], x[2]);
        const double2 c = c_add(x[1], x[3]), d = rot96<24, SGN>(c_sub(x[1], x[3]));
        x[0] = c_add(a, c);
        x[2] = c_sub(a, c);
        x[1] = c_add(b, d);
        x[3] = c_sub(b, d);
    } else if constexpr (P == 5) {
        constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
        constexpr double s1 = SGN * 0.95105651629515357212, s2 = SGN * 0.58778525229247312917;
        const double2 t1 = c_add(x[1], x[4]), t2 = c_add(x[2], x[3]), d1 = c_sub(x[1], x[4]), d2 = c_sub(x[2], x[3]);
        const double2 a1 = make_double2(x[0].x + c1 * t1.x + c2 * t2.x, x[0].y + c1 * t1.y + c2 * t2.y);
        const double2 a2 = make_double2(x[0].x + c2 * t1.x + c1 * t2.x, x[0].y + c2 * t1.y + c1 * t2.y);
        const double2 b1 = make_double2(-(s1 * d1.y + s2 * d2.y), s1 * d1.x + s2 * d2.x);   // i (s1 d1 + s2 d2)
        const double2 b2 = make_double2(-(s2 * d1.y - s1 * d2.y), s2 * d1.x - s1 * d2.x);
        x[0] = c_add(x[0], c_add(t1, t2));
        x[1] = c_add(a1, b1);
        x[4] = c_sub(a1, b1);
        x[2] = c_add(a2, b2);
        x[3] = c_sub(a2, b2);
    } else if constexpr (P == 7) {
        constexpr double c[4] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
        constexpr double s[4] = {0.0, SGN * 0.78183148246802980871, SGN * 0.97492791218182360702, SGN * 0.43388373911755812048};
        double2 t[4], d[4], y[7];
        t[0] = x[0];
        sfor<3>([&](auto jc) {
            constexpr int j = decltype(jc)::value + 1;
            t[j] = c_add(x[j], x[7 - j]);
            d[j] = c_sub(x[j], x[7 - j]);
        });
        y[0] = c_add(c_add(t[0], t[1]), c_add(t[2], t[3]));
        sfor<3>([&](auto kc) {
            constexpr int k = decltype(kc)::value + 1;
            double2 a = t[0], b = make_double2(0.0, 0.0);
            sfor<3>([&](auto jc) {
                constexpr int j = decltype(jc)::value + 1, m = j * k % 7, f = m <= 3 ? m : 7 - m;
                constexpr double sj = m <= 3 ? s[f] : -s[f];
                a = make_double2(a.x + c[f] * t[j].x, a.y + c[f] * t[j].y);
                b = make_double2(b.x - sj * d[j].y, b.y + sj * d[j].x);   // i sin d
            });
            y[k] = c_add(a, b);
            y[7 - k] = c_sub(a, b);
        });
        sfor<7>([&](auto kc) { x[decltype(kc)::value] = y[decltype(kc)::value]; });
    } else if constexpr (P == 9) {   // 3 x 3
        constexpr double c[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, 0.0, -0.93969262078590838405};
        constexpr double s[5] = {0.0, SGN * 0.64278760968653932632, SGN * 0.98480775301220805937, 0.0, SGN * 0.34202014332566873304};
        double2 t[9];
        sfor<3>([&](auto n2c) {
            constexpr int n2 = decltype(n2c)::value;
            double2 u[3] = {x[n2], x[3 + n2], x[6 + n2]};
            dft<3, SGN>(u);
            sfor<3>([&](auto k1c) {
                constexpr int k1 = decltype(k1c)::value, e = n2 * k1;   // exp(2 pi i e / 9), e = 0, 1, 2, 4
                t[n2 * 3 + k1] = e == 0 ? u[k1] : make_double2(u[k1].x * c[e] - u[k1].y * s[e], u[k1].x * s[e] + u[k1].y * c[e]);
            });
        });
        sfor<3>([&](auto k1c) {
            constexpr int k1 = decltype(k1c)::value;
            double2 u[3] = {t[k1], t[3 + k1], t[6 + k1]};
            dft<3, SGN>(u);
            sfor<3>([&](auto k2c) { x[k1 + 3 * decltype(k2c)::value] = u[decltype(k2c)::value]; });
        });
    } else if constexpr (P == 10 || P == 15) {
        // coprime factors (Good-Thomas): n = p2 n1 + p1 n2, output k = k1 mod p1 = k2 mod p2; no twiddles
        constexpr int p1 = P / 5, p2 = 5;
        double2 t[P];
        sfor<p2>([&](auto n2c) {
            constexpr int n2 = decltype(n2c)::value;
            double2 u[p1];
            sfor<p1>([&](auto n1c) { u[decltype(n1c)::value] = x[(p2 * decltype(n1c)::value + p1 * n2) % P]; });
            dft<p1, SGN>(u);
            sfor<p1>([&](auto k1c) { t[n2 * p1 + decltype(k1c)::value] = u[decltype(k1c)::value]; });
        });
        sfor<p1>([&](auto k1c) {
            constexpr int k1 = decltype(k1c)::value;
            double2 u[p2];
            sfor<p2>([&](auto n2c) { u[decltype(n2c)::value] = t[decltype(n2c)::value * p1 + k1]; });
            dft<p2, SGN>(u);
            sfor<p2>([&](auto k2c) {
                constexpr int k2 = decltype(k2c)::value;
                constexpr int k = [] { for (int v = 0; v < P; ++v) if (v % p1 == k1 && v % p2 == k2) return v; return 0; }();
                x[k] = u[k2];
            });
        });
    } else {
        static_assert(96 % P == 0, "radix must divide 96");
        constexpr int p1 = (P % 4 == 0) ? 4 : (P % 3 == 0 ? 3 : 2);
        constexpr int p2 = P / p1;
        double2 t[P];
        sfor<p2>([&](auto n2c) {
            constexpr int n2 = decltype(n2c)::value;
            double2 u[p1];
            sfor<p1>([&](auto n1c) { u[decltype(n1c)::value] = x[p2 * decltype(n1c)::value + n2]; });
            dft<p1, SGN>(u);
            sfor<p1>([&](auto k1c) {
                constexpr int k1 = decltype(k1c)::value;
                t[n2 * p1 + k1] = rot96<(96 / P) * n2 * k1, SGN>(u[k1]);
            });
        });
        sfor<p1>([&](auto k1c) {
            constexpr int k1 = decltype(k1c)::value;
            double2 u[p2];
            sfor<p2>([&](auto n2c) { u[decltype(n2c)::value] = t[decltype(n2c)::value * p1 + k1]; });
            dft<p2, SGN>(u);
            sfor<p2>([&](auto k2c) { x[k1 + p1 * decltype(k2c)::value] = u[decltype(k2c)::value]; });
        });
    }
}

// Twiddles w^r = exp(SGN 2 pi i r e / (2M)), 0 < r < P, of a butterfly with base exponent e
// (roots[e] = exp(2 pi i e / (2M))): the power-of-two r are read from the table, the others
// are products of two earlier ones (r = h + (r - h), h the highest power of two in r), at
// most two roundings from the table values.  Fewer loads in flight keeps the passes'
// register peak down.
template <int P, int SGN>
__device__ __forceinline__ void twiddles(double2 (&w)[P], const double2 *__restrict__ roots, int e) {
    sfor<P>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        if constexpr (r > 0) {
            constexpr int h = 1 << (31 - __builtin_clz(r));
            if constexpr (h == r) {
                w[r] = roots[r * e];
                if constexpr (SGN < 0) w[r].y = -w[r].y;
            } else {
                w[r] = c_mul(w[h], w[r - h]);
            }
        }
    });
}

// Blocks are dealt round-robin to the 8 XCDs; give each XCD a contiguous range of latitude
// groups so that the blocks running together on one XCD touch neighbouring latitudes (which
// share cache lines of that XCD's L2 in the theta-contiguous layout).
__device__ __forceinline__ int xcd_group_w(int bid, int G) {
    if (G % 8) return bid;
    return (bid % 8) * (G / 8) + bid / 8;
}

}  // namespace
}  // namespace shtns_amd
