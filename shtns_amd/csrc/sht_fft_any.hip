// sht_fft_any.hip -- longitude FFTs of any length 2 M whose M factors into 2, 3, 5, 7 (the sizes
// shtns_set_grid picks by itself are 2^a 3^b 5^c): runtime plan, in-place decimation in
// frequency in LDS.
//
// A block holds T latitudes (a power of two) of M complex points.  Bound: LDS traffic and the
// latency of its phases, so the plan takes few passes of large radices (up to 16) done in
// registers: three for M = 360, where radices up to 5 take five; twiddles
// are powers of few table values (twiddles<P>); the index arithmetic of a butterfly is one
// multiplication by a reciprocal; global loads are issued in batches of four, with the
// latitude fastest on the Fourier side, and the latitude or the longitude fastest on the
// spatial side as the layout has it; the real-FFT pre- and post-twiddles take the pair k, M - k
// together, so every Fourier coefficient is read and every transform value used once.
#include <algorithm>

#include "sht_fft_radix.h"
#include "sht_internal.h"

namespace shtns_amd {
namespace {

struct AnyPlan {
    int M, n;
    int radix[24];
    unsigned magic[24];   // ceil(2^32 / q) of a pass' butterfly spacing q (0: q = 1)
};

// One pass of radix P over all butterflies: points a[r q], r < P, of group g, offset n1.
template <int P, int SGN>
__device__ __forceinline__ void any_pass(double2 *buf, int total, int lt, int str, int q, int Ns, unsigned magic, int twm,
                                         const double2 *__restrict__ roots) {
    for (int b = threadIdx.x; b < total; b += blockDim.x) {
        const int t = b & ((1 << lt) - 1), bb = b >> lt;
        const int g = magic ? (int)__umulhi((unsigned)bb, magic) : bb, n1 = bb - g * q;
        double2 *a = buf + t * str + g * Ns + n1;
        double2 x[P];
        sfor<P>([&](auto rc) { x[decltype(rc)::value] = a[decltype(rc)::value * q]; });
        dft<P, SGN>(x);
        if (magic) {   // last pass: n1 = 0, no twiddles
            double2 w[P];
            twiddles<P, SGN>(w, roots, n1 * twm);
            sfor<P>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                if constexpr (r > 0) x[r] = c_mul(x[r], w[r]);
            });
        }
        sfor<P>([&](auto rc) { a[decltype(rc)::value * q] = x[decltype(rc)::value]; });
    }
}

template <int SGN>
__device__ __forceinline__ void any_passes(double2 *buf, const AnyPlan &pl, int lt, int str, const double2 *__restrict__ roots) {
    int Ns = pl.M;
    for (int s = 0; s < pl.n; ++s) {
        const int p = pl.radix[s], q = Ns / p, total = (pl.M / p) << lt, twm = 2 * pl.M / Ns;
        const unsigned magic = pl.magic[s];
        switch (p) {
#define ANY_PASS(P) case P: any_pass<P, SGN>(buf, total, lt, str, q, Ns, magic, twm, roots); break;
            ANY_PASS(2) ANY_PASS(3) ANY_PASS(4) ANY_PASS(5) ANY_PASS(6) ANY_PASS(7) ANY_PASS(8) ANY_PASS(9) ANY_PASS(10)
            ANY_PASS(12) ANY_PASS(15) ANY_PASS(16)
#undef ANY_PASS
            default: break;
        }
        __syncthreads();
        Ns = q;
    }
}

constexpr int AB = 4;   // loads in flight per thread and batch

template <class TV>
__global__ __launch_bounds__(256) void fft_synth_any(const double2 *__restrict__ F, long four_dist, TV *__restrict__ V,
                                                     long spat_dist, const double2 *__restrict__ roots,
                                                     const int *__restrict__ pos, AnyPlan pl, int nlat, int imlim, long sp,
                                                     long stt, int lt, int str, int lat_base, int lat_end) {
    extern __shared__ double2 buf[];
    const int M = pl.M, T = 1 << lt, nt = blockDim.x;
    const int lat0 = lat_base + xcd_group_w(blockIdx.x, gridDim.x) * T;
    const double2 *Ff = F + (size_t)blockIdx.y * four_dist;
    TV *Vf = V + (size_t)blockIdx.y * spat_dist;
    const int Tv = min(T, lat_end - lat0);
    // Z_k = A + i w B, Z_{M-k} = conj A + i conj(w B) with A = X_k + conj X_{M-k}, B = X_k - conj X_{M-k},
    // w = e^{i pi k/M}; k = 0 .. M/2, X_M = 0
    const int total = (M / 2 + 1) << lt;
    for (int e0 = threadIdx.x; e0 < total; e0 += AB * nt) {
        double2 xk[AB], xm[AB], wk[AB];
#pragma unroll
        for (int u = 0; u < AB; ++u) {
            const int e = e0 + u * nt, t = e & (T - 1), k = e >> lt, km = M - k;
            const bool in = e < total && t < Tv;
            xk[u] = (in && k <= imlim) ? Ff[(size_t)k * nlat + lat0 + t] : make_double2(0.0, 0.0);
            xm[u] = (in && k > 0 && km <= imlim) ? Ff[(size_t)km * nlat + lat0 + t] : make_double2(0.0, 0.0);
            wk[u] = roots[e < total ? k : 0];
        }
#pragma unroll
        for (int u = 0; u < AB; ++u) {
            const int e = e0 + u * nt, t = e & (T - 1), k = e >> lt, km = M - k;
            if (e >= total) break;
            const double2 A = c_add(xk[u], c_conj(xm[u])), B = c_sub(xk[u], c_conj(xm[u]));
            const double2 wB = c_mul(wk[u], B);
            buf[t * str + k] = make_double2(A.x - wB.y, A.y + wB.x);
            if (k > 0 && km > k) buf[t * str + km] = make_double2(A.x + wB.y, wB.x - A.y);
        }
    }
    __syncthreads();
    any_passes<1>(buf, pl, lt, str, roots);
    if (sp < stt) {   // longitude fastest
        for (int t = 0; t < Tv; ++t) {
            TV *Vt = Vf + (size_t)(lat0 + t) * stt;
            for (int n = threadIdx.x; n < M; n += nt) {
                const double2 z = buf[t * str + pos[n]];
                Vt[(size_t)(2 * n) * sp] = (TV)z.x;
                Vt[(size_t)(2 * n + 1) * sp] = (TV)z.y;
            }
        }
    } else {
        for (int e = threadIdx.x; e < M << lt; e += nt) {
            const int t = e & (T - 1), n = e >> lt;
            if (t >= Tv) continue;
            const double2 z = buf[t * str + pos[n]];
            TV *v = Vf + (size_t)(2 * n) * sp + (size_t)(lat0 + t) * stt;
            v[0] = (TV)z.x;
            v[sp] = (TV)z.y;
        }
    }
}

template <class TV>
__global__ __launch_bounds__(256) void fft_anal_any(const TV *__restrict__ V, long spat_dist, double2 *__restrict__ F,
                                                    long four_dist, const double2 *__restrict__ roots,
                                                    const int *__restrict__ pos, AnyPlan pl, int nlat, int mmax, int imlim,
                                                    long sp, long stt, int lt, int str, int lat_base, int lat_end) {
    extern __shared__ double2 buf[];
    const int M = pl.M, T = 1 << lt, nt = blockDim.x;
    const int lat0 = lat_base + xcd_group_w(blockIdx.x, gridDim.x) * T;
    const TV *Vf = V + (size_t)blockIdx.y * spat_dist;
    double2 *Ff = F + (size_t)blockIdx.y * four_dist;
    const int Tv = min(T, lat_end - lat0);
    if (sp < stt) {   // longitude fastest
        for (int t = 0; t < Tv; ++t) {
            const TV *Vt = Vf + (size_t)(lat0 + t) * stt;
            for (int n0 = threadIdx.x; n0 < M; n0 += AB * nt) {
                double2 z[AB];
#pragma unroll
                for (int u = 0; u < AB; ++u) {
                    const int n = min(n0 + u * nt, M - 1);
                    z[u] = make_double2((double)Vt[(size_t)(2 * n) * sp], (double)Vt[(size_t)(2 * n + 1) * sp]);
                }
#pragma unroll
                for (int u = 0; u < AB; ++u)
                    if (n0 + u * nt < M) buf[t * str + n0 + u * nt] = z[u];
            }
        }
    } else {
        const int total = M << lt;
        for (int e0 = threadIdx.x; e0 < total; e0 += AB * nt) {
            double2 z[AB];
#pragma unroll
            for (int u = 0; u < AB; ++u) {
                const int e = min(e0 + u * nt, total - 1), t = min(e & (T - 1), Tv - 1), n = e >> lt;
                const TV *v = Vf + (size_t)(2 * n) * sp + (size_t)(lat0 + t) * stt;
                z[u] = make_double2((double)v[0], (double)v[sp]);
            }
#pragma unroll
            for (int u = 0; u < AB; ++u) {
                const int e = e0 + u * nt;
                if (e < total) buf[(e & (T - 1)) * str + (e >> lt)] = z[u];
            }
        }
    }
    __syncthreads();
    any_passes<-1>(buf, pl, lt, str, roots);
    // X_k = A + u, X_{M-k} = conj(A - u), u = conj(w) B, A = (Z_k + conj Z_{M-k})/2, B = (Z_k - conj Z_{M-k})/(2i)
    for (int e = threadIdx.x; e < (M / 2 + 1) << lt; e += nt) {
        const int t = e & (T - 1), k = e >> lt, km = M - k;
        if (t >= Tv || (k > mmax && km > mmax)) continue;
        const double2 Zk = buf[t * str + pos[k]], Zm = buf[t * str + pos[k ? km : 0]];
        const double2 A = make_double2(0.5 * (Zk.x + Zm.x), 0.5 * (Zk.y - Zm.y));
        const double2 D = make_double2(Zk.x - Zm.x, Zk.y + Zm.y);
        const double2 u = c_mul(c_conj(roots[k]), make_double2(0.5 * D.y, -0.5 * D.x));
        double2 *f = Ff + lat0 + t;
        if (k <= mmax) {
            double2 X = make_double2(A.x + u.x, k ? A.y + u.y : 0.0);
            if (k > imlim) X = make_double2(0.0, 0.0);
            f[(size_t)k * nlat] = X;
        }
        if (k > 0 && km > k && km <= mmax)
            f[(size_t)km * nlat] = km <= imlim ? make_double2(A.x - u.x, u.y - A.y) : make_double2(0.0, 0.0);
    }
}

struct AnyGeom {
    AnyPlan pl;
    int lt, str, nt;
    size_t lds;
};

// Latitudes per block: as many as fit twice in a CU's LDS (at most 8, where the Fourier rows
// move in whole 128-byte lines), fewer when the grid would leave CUs idle; threads for about
// four butterflies each.  Rows of str points, str = 8 / T mod 8: the T latitudes x 8 / T
// neighbouring points of one LDS cycle fall on distinct banks.
bool any_geom(const FftPlan &plan, int nlat_chunk, int nfields, AnyGeom &g) {
    g.pl.M = plan.M;
    g.pl.n = plan.nstages;
    int Ns = plan.M;
    for (int s = 0; s < plan.nstages; ++s) {
        const int q = Ns / plan.radix[s];
        g.pl.radix[s] = plan.radix[s];
        g.pl.magic[s] = q == 1 ? 0u : (unsigned)((0x100000000ull + q - 1) / q);
        Ns = q;
    }
    const int M = plan.M;
    auto stride = [&](int lt) {
        int str = M;
        while (str % 8 != (8 >> lt) % 8) ++str;
        return str;
    };
    g.lt = 3;
    while (g.lt > 0 && (((size_t)stride(g.lt) * 16) << g.lt) > 80 * 1024) --g.lt;
    while (g.lt > 1 && (long)((nlat_chunk + (1 << g.lt) - 1) >> g.lt) * nfields < 512) --g.lt;
    g.str = stride(g.lt);
    g.lds = ((size_t)g.str * 16) << g.lt;
    if (g.lds > 160 * 1024) return false;
    const long pts = (long)M << g.lt;
    g.nt = pts <= 1024 ? 64 : pts <= 2048 ? 128 : 256;
    return true;
}

template <class TV>
bool synth_any(const DeviceTables *t, int nlat, int imlim, int nfields, const double2 *F, long four_dist, TV *V,
               long spat_dist, long sp, long st, hipStream_t s, int lat_base, int lat_end) {
    AnyGeom g;
    if (!any_geom(t->any_plan, lat_end - lat_base, nfields, g)) return false;
    ensure_lds_limit((const void *)fft_synth_any<TV>, g.lds);
    const int nb = (lat_end - lat_base + (1 << g.lt) - 1) >> g.lt;
    hipLaunchKernelGGL(fft_synth_any<TV>, dim3(nb, nfields), dim3(g.nt), g.lds, s, F, four_dist, V, spat_dist, t->roots,
                       t->any_pos, g.pl, nlat, imlim, sp, st, g.lt, g.str, lat_base, lat_end);
    return true;
}
template <class TV>
bool anal_any(const DeviceTables *t, int nlat, int mmax, int imlim, int nfields, const TV *V, long spat_dist, double2 *F,
              long four_dist, long sp, long st, hipStream_t s, int lat_base, int lat_end) {
    AnyGeom g;
    if (!any_geom(t->any_plan, lat_end - lat_base, nfields, g)) return false;
    ensure_lds_limit((const void *)fft_anal_any<TV>, g.lds);
    const int nb = (lat_end - lat_base + (1 << g.lt) - 1) >> g.lt;
    hipLaunchKernelGGL(fft_anal_any<TV>, dim3(nb, nfields), dim3(g.nt), g.lds, s, V, spat_dist, F, four_dist, t->roots,
                       t->any_pos, g.pl, nlat, mmax, imlim, sp, st, g.lt, g.str, lat_base, lat_end);
    return true;
}

}  // namespace

bool launch_fft_synth_any(const DeviceTables *t, int nlat, int imlim, int nfields, const double2 *F, long four_dist,
                          double *V, long spat_dist, long sp, long st, hipStream_t s, int lat_base, int lat_end) {
    return synth_any(t, nlat, imlim, nfields, F, four_dist, V, spat_dist, sp, st, s, lat_base, lat_end);
}
bool launch_fft_synth_any(const DeviceTables *t, int nlat, int imlim, int nfields, const double2 *F, long four_dist,
                          float *V, long spat_dist, long sp, long st, hipStream_t s, int lat_base, int lat_end) {
    return synth_any(t, nlat, imlim, nfields, F, four_dist, V, spat_dist, sp, st, s, lat_base, lat_end);
}
bool launch_fft_anal_any(const DeviceTables *t, int nlat, int mmax, int imlim, int nfields, const double *V,
                         long spat_dist, double2 *F, long four_dist, long sp, long st, hipStream_t s, int lat_base,
                         int lat_end) {
    return anal_any(t, nlat, mmax, imlim, nfields, V, spat_dist, F, four_dist, sp, st, s, lat_base, lat_end);
}
bool launch_fft_anal_any(const DeviceTables *t, int nlat, int mmax, int imlim, int nfields, const float *V,
                         long spat_dist, double2 *F, long four_dist, long sp, long st, hipStream_t s, int lat_base,
                         int lat_end) {
    return anal_any(t, nlat, mmax, imlim, nfields, V, spat_dist, F, four_dist, sp, st, s, lat_base, lat_end);
}

}  // namespace shtns_amd
