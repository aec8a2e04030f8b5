// sht_legendre.h -- Legendre-step kernels of shtns_amd as templates, instantiated per
// contraction precision in sht_kernels.hip (FP64), sht_legendre_f32.hip (FP32) and
// sht_legendre_split.hip (FP32 hi/lo split).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

#include "sht_internal.h"

namespace shtns_amd {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------------------
// Helpers shared by the Legendre kernels
// ---------------------------------------------------------------------------------------
// Read-only table viewed through the constant address space: loads with wave-uniform
// indices become scalar (SMEM) loads and stay off the vector-memory counters.
struct UniformTable2 {
    const __attribute__((address_space(4))) double *p;
    __device__ explicit UniformTable2(const double2 *q) : p((const __attribute__((address_space(4))) double *)q) {}
    __device__ double2 operator[](int i) const { return make_double2(p[2 * i], p[2 * i + 1]); }
};
struct OrderInfo {
    int slot;       // table slot (im, or mmax+1 for the m=1 functions of vector m=0)
    int mfun;       // order of the generated functions
    int nsteps;     // recurrence steps to evaluate (degrees mfun .. ltr)
    int spec_base;  // index of degree 0 of this order in the spectral layout (may be virtual)
    bool sinv;      // divide the seeds by sin(theta) (unused: vector seeds have their own table)
    bool real_only; // m = 0: imaginary parts ignored / zero
};

__device__ inline OrderInfo order_info(int im, int lmax_spec, int mmax, int mres, int ltr, int vector_mode) {
    OrderInfo o;
    const int m = im * mres;
    o.real_only = (im == 0);
    if (vector_mode && im == 0) {
        o.slot = mmax + 1;
        o.mfun = 1;
        o.sinv = false;
    } else {
        o.slot = im;
        o.mfun = m;
        o.sinv = false;   // vector mode reads seeds of P/sin(theta) (from sin^(m-1), finite at the poles)
    }
    o.nsteps = (ltr >= o.mfun) ? (ltr - o.mfun) / 2 + 1 : 0;
    o.spec_base = (int)(((long)im * (2 * lmax_spec + 2 - (im + 1) * mres)) / 2);
    return o;
}

// Workgroups are dealt round-robin to the 8 XCDs (block b runs on XCD b % 8).  Map physical
// block b to a logical index so that each run of `gsize` consecutive logical blocks lands on
// one XCD, in dispatch order: XCD x takes groups x, x + 8, x + 16, ...  Identity unless nb is
// a multiple of 8 * gsize.
__device__ inline int xcd_cluster(int b, int nb, int gsize) {
    if (gsize <= 1 || nb % (8 * gsize)) return b;
    const int x = b & 7, s = b >> 3;
    return (x + 8 * (s / gsize)) * gsize + s % gsize;
}

// v of quad lane SEL (DPP quad_perm: lane 4q + i reads lane 4q + sel_i, sel_i = (SEL >> 2i) & 3;
// no LDS traffic).  All lanes of the wave must be active.
template <int SEL>
__device__ __forceinline__ double quad_perm(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), SEL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), SEL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// v of lane l - 1 within each row of 16 lanes (DPP row_shr:1); lanes 0, 16, 32, 48 get 0.
// All lanes of the wave must be active.
__device__ __forceinline__ double row_shr1(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x111, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x111, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// ---------------------------------------------------------------------------------------
// Contraction precision PREC (the recurrence, seeds, tables and the final sums stay FP64):
//   0  FP64 matrix cores: v_mfma_f64_16x16x4f64 on z and the coefficients;
//   1  FP32 matrix cores: z and the coefficients rounded to FP32, v_mfma_f32_16x16x4f32,
//      FP32 partial sums over 16 degrees-pairs added into FP64;
//   2  FP32 split: z = z_hi + z_lo and b = b_hi + b_lo (FP32 pairs) with the three products
//      z_hi b_hi + z_lo b_hi + z_hi b_lo on the FP32 matrix cores, same FP32 partial sums.
// A recurrence value sits in one 8-byte LDS slot either as a double or as an FP32 (hi, lo) pair.
// ---------------------------------------------------------------------------------------
template <int PREC>
struct Contract {
    using acc_t = std::conditional_t<PREC == 0, double4_t, float4_t>;
    using a_t = std::conditional_t<PREC == 0, double, float2>;    // A operand (recurrence value)
    using b_t = std::conditional_t<PREC == 0, double, float2>;    // B operand (coefficient or data)
    __device__ static acc_t zero() {
        if constexpr (PREC == 0) return (double4_t){0.0, 0.0, 0.0, 0.0};
        else return (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
    }
    __device__ static void store_z(double *slot, double z) {
        if constexpr (PREC == 0) {
            *slot = z;
        } else {
            const float hi = (float)z;
            *reinterpret_cast<float2 *>(slot) = make_float2(hi, (float)(z - (double)hi));
        }
    }
    __device__ static a_t load_z(const double *slot) {
        if constexpr (PREC == 0) return *slot;
        else return *reinterpret_cast<const float2 *>(slot);
    }
    __device__ static b_t split(double b) {
        if constexpr (PREC == 0) {
            return b;
        } else {
            const float hi = (float)b;
            return make_float2(hi, (float)(b - (double)hi));
        }
    }
    // acc += A * B for one 16x16x4 tile
    __device__ static acc_t mma(a_t a, b_t b, acc_t acc) {
        if constexpr (PREC == 0) {
            return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
        } else if constexpr (PREC == 1) {
            return __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
        } else {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.y, acc, 0, 0, 0);
            return __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
        }
    }
    // D layout on gfx950: register j of lane l holds D[row][l % 16] with
    //   f64 16x16x4: row = 4 j + l / 16;   f32 16x16x4: row = 4 (l / 16) + j.
    __device__ static int d_row(int j, int lane) {
        if constexpr (PREC == 0) return 4 * j + (lane >> 4);
        else return 4 * (lane >> 4) + j;
    }
};

// ---------------------------------------------------------------------------------------
// Synthesis, step 2: F[f][im][k] = sum_l Q_lm P_lm(x_k)   (both hemispheres)
// One wave = one order im, 4*NCG fields, one latitude tile of 64 pairs (lane = pair); waves
// are independent (no block barrier).  Software pipeline per 4-step block:
//   A operands (z of 16 latitudes x 4 steps) read back from the wave's LDS tile,
//   4 x NCG MFMAs D[16 lat][16 col] += A * B,
//   then, while the matrix cores work, the recurrence of the next 4 steps is advanced on
//   the vector ALUs into the other LDS tile and the next B operands are loaded.
// The accumulators go straight to F: lanes holding E and O of one field are lane^2
// partners (north = E + x O, south = E - x O).
// ---------------------------------------------------------------------------------------
constexpr int kSynthTileBytes = 2 * 4 * 64 * sizeof(double);   // LDS per wave
// Waves (latitude tiles) per block.  Blocks of four waves whose last ones have no tile leave
// their SIMDs idle: with six tiles half of the blocks loaded two SIMDs only (matrix cores busy
// 54%; 64 fields at lmax=511: synthesis call 672 -> 617 us in one-wave blocks), so
// other counts than multiples of four take one-wave blocks (lmax=560, 16 fields: call 257 ->
// 243 us; two-wave ones 257).  One to three fields are bound by latency and keep an order's
// tiles together (lmax=340, 3 fields: 41.5 us, one-wave blocks 44.3).
inline int synth_waves(int ntl, int nfields) {
    if (nfields <= 3) return ntl < 4 ? ntl : 4;
    return ntl % 4 == 0 ? 4 : ntl == 2 ? 2 : 1;
}

// NF4 > 0 (FP64, NCG = 1, at most 3 fields): field c of the group is contracted with
// v_mfma_f64_4x4x4f64 (four 4x4x4 blocks: 16 latitudes x 4 steps x the field's 4 columns),
// so no matrix-core columns are spent on absent fields.  gfx950 lane layouts of that
// instruction: A lane l = (block (l>>2)&3, row l&3, k l>>4), B lane l = (block (l>>2)&3,
// k l>>4, col l&3), D lane l = (block (l>>2)&3, row l>>4, col l&3); with block b and row i
// taken as latitude 4b + i of a 16-latitude row tile, the A operand is the 16x16x4 one.
template <int NCG, int PREC, int NF4 = 0>
__global__ __launch_bounds__(256) void legendre_synth_kernel(
    const double *__restrict__ xk, const double *__restrict__ x2k, const double *__restrict__ stk,
    const double *__restrict__ wqk, const int *__restrict__ step_ofs, const double2 *__restrict__ ab,
    const int *__restrict__ i0tab, const double2 *__restrict__ z0tab, const double *__restrict__ qmix,
    int nsteps_total, int lmax_spec, double2 *__restrict__ F, long four_dist, int mmax, int mres, int nlat,
    int nlat_2, int ltr, int imlim, int nfields, int vector_mode, int lat_weight, int tile0, int ntl) {
    constexpr int NCOL = 16 * NCG;
    extern __shared__ double ytile_lds[];   // [waves][2][4][64]
    double(*ytile)[2][4][64] = reinterpret_cast<double(*)[2][4][64]>(ytile_lds);

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    // heavy orders first: block x -> (order, tile group); the tile groups of one order run on
    // one XCD (they read the same coefficient rows, which then hit in that XCD's L2)
    const int nw = blockDim.x >> 6;
    const int ntg = (ntl + nw - 1) / nw;   // tile groups of this launch
    const int bx = xcd_cluster(blockIdx.x, gridDim.x, ntg);
    const int im = bx / ntg;
    const int tile = tile0 + (bx - im * ntg) * nw + wave;
    const int g = blockIdx.y;
    const int fbase = g * 4 * NCG;
    if (tile >= tile0 + ntl || tile * 64 >= nlat_2) return;   // no block-level synchronization in this kernel
    const int k = tile * 64 + lane;
    const bool kvalid = (k < nlat_2);
    const int kk = kvalid ? k : (nlat_2 - 1);

    using C = Contract<PREC>;
    static_assert(NF4 == 0 || (PREC == 0 && NCG == 1 && NF4 <= 3), "4x4x4 path: FP64, one group of <= 3 fields");
    constexpr int NA = NF4 ? NF4 : NCG;   // accumulator sets: fields (4x4x4) or column groups
    using acc64_t = std::conditional_t<NF4 == 0, double4_t, double>;
    acc64_t acc[4][NA];   // FP64 sums
    typename C::acc_t part[4][NCG];   // FP32 partial sums over 16 steps (PREC > 0; unused at PREC 0)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int c = 0; c < NA; ++c) acc[r][c] = acc64_t{};
#pragma unroll
        for (int c = 0; c < NCG; ++c) part[r][c] = C::zero();
    }
    auto flush = [&]() {
        if constexpr (PREC > 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < NCG; ++c) {
                    acc[r][c] += __builtin_convertvector(part[r][c], double4_t);
                    part[r][c] = C::zero();
                }
        }
    };

    const OrderInfo o = order_info(im, lmax_spec, mmax, mres, (im <= imlim) ? ltr : -1, vector_mode);
    const int nsteps = (im <= imlim) ? o.nsteps : 0;
    if (nsteps > 0) {
        const int sofs = step_ofs[o.slot];
        const int slot_rows = step_ofs[o.slot + 1] - sofs;   // > nsteps: the last rows of qmix are zero
        const UniformTable2 abm(ab + sofs);   // uniform indices -> scalar loads
        const double *qb = qmix + ((size_t)g * nsteps_total + sofs) * NCOL;
        const double x2 = x2k[kk];
        int i0 = kvalid ? i0tab[(size_t)o.slot * nlat_2 + kk] : nsteps;
        double2 sd = z0tab[(size_t)o.slot * nlat_2 + kk];
        if (o.sinv) {
            const double inv = 1.0 / stk[kk];
            sd.x *= inv;
            sd.y *= inv;
        }
        if (i0 > nsteps) i0 = nsteps;
        int wmin = i0, wmax = i0;
        for (int off = 32; off >= 1; off >>= 1) {
            wmin = min(wmin, __shfl_xor(wmin, off));
            wmax = max(wmax, __shfl_xor(wmax, off));
        }
        // wave-uniform: keeps loop control and coefficient loads on the scalar unit
        wmin = __builtin_amdgcn_readfirstlane(wmin);
        wmax = __builtin_amdgcn_readfirstlane(wmax);
        const int ibeg = wmin & ~3;
        double za = 0.0, zb = 0.0;
        if (i0 == ibeg) { za = sd.x; zb = sd.y; }

        // advance 4 recurrence steps starting at step i, writing z_i..z_{i+3} to tile buffer
        // coefficients of steps i .. i+3: the table holds at least nsteps + 7 rows per order
        // (continued past the last degree), so no clamp is needed and the four pairs are one
        // 64-byte scalar load
        auto load_cf = [&](int i, double2 *cf) {
#pragma unroll
            for (int s = 0; s < 4; ++s) cf[s] = abm[i + s];
        };
        auto advance = [&](int i, int buf, const double2 *cf) {
            if (i <= wmax) {   // some lane of this wave starts in this block
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    if (i + s == i0) { za = sd.x; zb = sd.y; }
                    C::store_z(&ytile[wave][buf][s][lane], zb);
                    const double zn = fma(fma(cf[s].x, x2, cf[s].y), zb, za);
                    za = zb;
                    zb = zn;
                }
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    C::store_z(&ytile[wave][buf][s][lane], zb);
                    const double zn = fma(fma(cf[s].x, x2, cf[s].y), zb, za);
                    za = zb;
                    zb = zn;
                }
            }
        };
        // B operand of column group (or field) c for the block at step i
        // (a 32-bit byte offset from the wave-uniform base: one address register)
        auto load_b1 = [&](int i, int c) {
            const int ii = min(i + (lane >> 4), slot_rows - 1);   // rows >= nsteps hold zeros
            const unsigned e = NF4 > 0 ? (unsigned)(ii * NCOL + c * 4 + (lane & 3)) : (unsigned)(ii * NCOL + c * 16 + (lane & 15));
            return *(const double *)((const char *)qb + 8u * e);
        };

        double bcur[NA];
        {
            double2 cf0[4];
            load_cf(ibeg, cf0);
            advance(ibeg, 0, cf0);
        }
        // in column-group order, as in the loop (the first MFMAs then wait for the first load only)
#pragma unroll
        for (int c = 0; c < NA; ++c) {
            bcur[c] = load_b1(ibeg, c);
            __builtin_amdgcn_sched_barrier(0);
        }
        // MFMAs of column group (or field) c on this block's A operands
        auto mma_group = [&](int c, const typename C::a_t *a) {
            if constexpr (NF4 > 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[r][c] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[r], bcur[c], acc[r][c], 0, 0, 0);
            } else {
                const typename C::b_t bb = C::split(bcur[c]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if constexpr (PREC == 0) acc[r][c] = C::mma(a[r], bb, acc[r][c]);
                    else part[r][c] = C::mma(a[r], bb, part[r][c]);
                }
            }
        };
        int buf = 0, blk = 0;
        for (int i = ibeg; i < nsteps; i += 4, ++blk) {
            __builtin_amdgcn_s_waitcnt(0xc07f);   // LDS tile of this block written
            __builtin_amdgcn_wave_barrier();
            typename C::a_t a[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) a[r] = C::load_z(&ytile[wave][buf][lane >> 4][r * 16 + (lane & 15)]);
            mma_group(0, a);
            // The next block's coefficients: a scalar load issued behind the first MFMAs (scalar
            // and LDS loads share one counter, so issued before the A reads it would delay
            // them), in flight while the other MFMAs issue.
            __builtin_amdgcn_sched_barrier(0);
            double2 cfn[4];
            load_cf(i + 4, cfn);
            bcur[0] = load_b1(i + 4, 0);   // next block's B operands, each once its MFMAs have issued
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 1; c < NA; ++c) {
                mma_group(c, a);
                bcur[c] = load_b1(i + 4, c);
                __builtin_amdgcn_sched_barrier(0);
            }
            advance(i + 4, buf ^ 1, cfn);   // also after the last block (in bounds, unused)
            buf ^= 1;
            if ((blk & 3) == 3) flush();
        }
        flush();
    }

    // Epilogue.  D[row][col]: the lane of column col = lane & 15 holds rows C::d_row(j, lane) of
    // row tile r (latitudes tile*64 + 16r + row).  Columns are 4 fields x (E.re, E.im, O.re,
    // O.im), so a quad of lanes is one field's (E, O) pairs: every lane reads its pair's O and
    // E values (DPP), E lanes write north = E + x O and O lanes south = E - x O.
    const int col = NF4 ? (lane & 3) : (lane & 15);
    const int reim = col & 1;
    const bool o_lane = (col & 2) != 0;
    const bool zero_im = (im == 0) && reim;   // order 0 has no imaginary part
    if constexpr (NF4 > 0) {
        // D lane l: latitude tile*64 + 16 r + 4 ((l >> 2) & 3) + (l >> 4), column l & 3
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int kr = tile * 64 + r * 16 + 4 * ((lane >> 2) & 3) + (lane >> 4);
            const int kc = min(kr, nlat_2 - 1);
            const double x = xk[kc];
            const double xs = o_lane ? -x : x;
            const double wz = zero_im ? 0.0 : (lat_weight ? wqk[kc] * ((2 * kr + 1 == nlat) ? 2.0 : 1.0) : 1.0);
            const int row = o_lane ? (nlat - 1 - kr) : kr;
#pragma unroll
            for (int c = 0; c < NA; ++c) {
                const int f = fbase + c;
                const double o = quad_perm<0xEE>(acc[r][c]);
                const double e = quad_perm<0x44>(acc[r][c]);
                const double val = fma(xs, o, e) * wz;
                if (kr < nlat_2 && f < nfields)
                    reinterpret_cast<double *>(F + (size_t)f * four_dist + (size_t)im * nlat)[2 * row + reim] = val;
            }
        }
        return;
    } else {
    // every latitude of the tile and every field of the group exist (wave-uniform)
    const bool full = (tile * 64 + 64 <= nlat_2) && (fbase + 4 * NCG <= nfields);
    auto store_tile = [&](auto check) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            int row[4];
            bool ok[4];
            double xs[4], wz[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int kr = tile * 64 + r * 16 + C::d_row(j, lane);
                const int kc = min(kr, nlat_2 - 1);
                const double x = xk[kc];
                xs[j] = o_lane ? -x : x;
                // the middle row of an odd grid is its own mirror: its stored pair weight is halved
                wz[j] = zero_im ? 0.0 : (lat_weight ? wqk[kc] * ((2 * kr + 1 == nlat) ? 2.0 : 1.0) : 1.0);
                row[j] = o_lane ? (nlat - 1 - kr) : kr;
                ok[j] = kr < nlat_2;
            }
#pragma unroll
            for (int c = 0; c < NCG; ++c) {
                const int f = fbase + c * 4 + (col >> 2);
                double *Ff = reinterpret_cast<double *>(F + (size_t)min(f, nfields - 1) * four_dist +
                                                        (size_t)im * nlat) + reim;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const double o = quad_perm<0xEE>(acc[r][c][j]);   // lanes (2, 3, 2, 3)
                    const double e = quad_perm<0x44>(acc[r][c][j]);   // lanes (0, 1, 0, 1)
                    const double val = fma(xs[j], o, e) * wz[j];
                    if (!decltype(check)::value || (ok[j] && f < nfields)) Ff[2 * row[j]] = val;
                }
            }
        }
    };
    if (full) store_tile(std::false_type{});
    else store_tile(std::true_type{});
    }
}

// SHTNS_AMD_SYNTH_16=1: keep the 16x16x4 kernels for 1 to 3 fields (for comparisons)
inline bool synth_force16() {
    static const bool f = getenv("SHTNS_AMD_SYNTH_16") != nullptr;
    return f;
}

inline int synth_ncg(int nfields, int want = 0) {
    if (want == 1 || want == 2 || want == 4) return want;
    return nfields > 8 ? 4 : (nfields > 4 ? 2 : 1);
}

template <int PREC>
void synth_tiles_launch(const LegendreArgs &a, int spec_ltop, double2 *F, long four_dist, const double *qmix,
                        int nsteps_total, int tile0, int ntl, hipStream_t s) {
    const DeviceTables *t = a.t;
    const int nw = synth_waves(ntl, a.nfields);
    const int ntg = (ntl + nw - 1) / nw;
    const int ncg = synth_ncg(a.nfields, a.synth_ncg);
    const int ng = (a.nfields + 4 * ncg - 1) / (4 * ncg);
    dim3 grid((a.mmax + 1) * ntg, ng);
#define SYNTH_LAUNCH(NC, ...)                                                                                    \
    hipLaunchKernelGGL((legendre_synth_kernel<NC, PREC, ##__VA_ARGS__>), grid, dim3(64 * nw), nw * kSynthTileBytes, s, t->x, t->x2, t->st, t->wq, \
                       t->step_ofs, t->ab, a.vector_mode ? t->i0v : t->i0, a.vector_mode ? t->z0v : t->z0, qmix, \
                       nsteps_total, spec_ltop, F, four_dist, a.mmax,                                              \
                       a.mres, a.nlat, a.nlat_2, a.ltr, a.imlim, a.nfields, a.vector_mode, a.lat_weight, tile0, ntl)
    if constexpr (PREC == 0) {   // 1 to 3 fields: 4x4x4 blocks, no idle matrix-core columns
        if (a.nfields <= 3 && ncg == 1 && !synth_force16()) {
            if (a.nfields == 1) SYNTH_LAUNCH(1, 1);
            else if (a.nfields == 2) SYNTH_LAUNCH(1, 2);
            else SYNTH_LAUNCH(1, 3);
            return;
        }
    }
    if (ncg == 4) SYNTH_LAUNCH(4);
    else if (ncg == 2) SYNTH_LAUNCH(2);
    else SYNTH_LAUNCH(1);
#undef SYNTH_LAUNCH
}

// ---------------------------------------------------------------------------------------
// Synthesis of one to three fields in FP64, on the vector ALUs.
//
// The FP64 matrix and vector instructions share one unit (mixed streams add up to the rate of
// either), so for few fields the vector form costs the same multiply-adds, 2 (recurrence) +
// 4 NF (E/O, re/im) per step and latitude pair, without the LDS transposition of every value
// that the matrix operands need (16 KB per 16 steps x 64 latitudes: at one field the LDS was
// busier than the unit).  lane = latitude pair, R tiles of 64 per wave, sums in registers; the
// wave-uniform coefficients of a step (alpha, beta, then E and O of each field) are read from
// LDS by broadcast, 2 + 4 NF doubles shared by the R tiles.
// The pre-mix is done here, chunk of CS steps by chunk, by the block's threads (the next
// chunk's loads in flight during the current one): no separate pass over the coefficients.
// Same order of summation and same roundings as the matrix-core kernel.
// One field, synthesis call: lmax=4095 4756 -> 3795 us, lmax=2047 715 -> 545, lmax=511 49 -> 33;
// three fields at lmax=340 46 -> 38.
// ---------------------------------------------------------------------------------------
template <int NF, int R>
__global__ __launch_bounds__(256) void legendre_synth_few_kernel(
    const double *__restrict__ xk, const double *__restrict__ x2k, const double *__restrict__ wqk,
    const int *__restrict__ step_ofs, const double2 *__restrict__ ab, const double4 *__restrict__ pm,
    const int *__restrict__ i0tab, const double2 *__restrict__ z0tab, const double2 *__restrict__ Q, long spec_dist,
    int lmax_spec, double2 *__restrict__ F, long four_dist, int mmax, int mres, int nlat, int nlat_2, int ltr, int imlim,
    int vector_mode, double mpos_scale, int lat_weight, int tile0, int ntl, int nblk) {
    constexpr int CS = 64, ROW = 2 + 4 * NF;   // steps per chunk, doubles per step
    __shared__ __attribute__((aligned(16))) double cfs[2][CS][ROW];
    __shared__ int s_beg[4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6, nt = blockDim.x;
    const int im = blockIdx.x / nblk, tb = tile0 + (blockIdx.x - im * nblk) * nw * R;   // heavy orders first

    const OrderInfo o = order_info(im, lmax_spec, mmax, mres, (im <= imlim) ? ltr : -1, vector_mode);
    const int nsteps = (im <= imlim) ? o.nsteps : 0;
    const int sofs = step_ofs[o.slot], last_row = step_ofs[o.slot + 1] - sofs - 1;

    double x2[R], za[R], zb[R], acc[R][NF][4];
    double2 sd[R];
    int i0[R], wmin[R], wlast = 0, wbeg = nsteps;
#pragma unroll
    for (int r = 0; r < R; ++r) {   // neighbouring tiles: they start at similar steps
        const int tile = tb + wave * R + r, k = tile * 64 + lane;
        const bool kv = tile < tile0 + ntl && k < nlat_2;
        const int kk = kv ? k : 0;
        x2[r] = x2k[kk];
        i0[r] = kv ? min(i0tab[(size_t)o.slot * nlat_2 + kk], nsteps) : nsteps;
        sd[r] = z0tab[(size_t)o.slot * nlat_2 + kk];
        za[r] = zb[r] = 0.0;
        wmin[r] = i0[r];
        wlast = max(wlast, i0[r] < nsteps ? i0[r] : 0);   // lanes that never start stay zero
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[r][f][c] = 0.0;
    }
    auto step = [&](int r, const double *c) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[r][f][e] = fma(zb[r], c[2 + 4 * f + e], acc[r][f][e]);
        const double zn = fma(fma(c[0], x2[r], c[1]), zb[r], za[r]);
        za[r] = zb[r];
        zb[r] = zn;
    };
    // mixed coefficients of step ii, field f
    const double qscale = (im == 0) ? 1.0 : mpos_scale;
    constexpr int NE = (CS * NF + 63) / 64;   // (step, field) elements per thread of a one-wave block
    double2 q0[NE], q1[NE], q2[NE], cab[NE];
    double4 cpm[NE];
    auto fetch = [&](int ch) {   // loads of chunk ch
#pragma unroll
        for (int j = 0; j < NE; ++j) {
            const int e = threadIdx.x + j * nt;
            if (j > 0 && j * nt >= CS * NF) break;   // block-uniform
            const int f = e / CS, ii = ch + e % CS, le = o.mfun + 2 * ii;
            const bool in = e < CS * NF && ii < nsteps;
            const double2 *Qf = Q + (size_t)(in ? f : 0) * spec_dist + o.spec_base;
            const int lc = in ? le : max(o.mfun, 0);
            const bool any = nsteps > 0;
            cpm[j] = pm[sofs + min(ii, last_row)];
            cab[j] = ab[sofs + min(ii, last_row)];
            q0[j] = (any && in) ? Qf[lc] : make_double2(0.0, 0.0);
            q1[j] = (any && in && le + 1 <= ltr) ? Qf[lc + 1] : make_double2(0.0, 0.0);
            q2[j] = (any && in && le + 2 <= ltr) ? Qf[lc + 2] : make_double2(0.0, 0.0);
        }
    };
    auto put = [&](int b) {
#pragma unroll
        for (int j = 0; j < NE; ++j) {
            const int e = threadIdx.x + j * nt;
            if (j > 0 && j * nt >= CS * NF) break;
            if (e >= CS * NF) break;
            const int f = e / CS, s = e % CS;
            const double4 cf = cpm[j];
            double4 out;
            out.x = (cf.x * q0[j].x + cf.y * q2[j].x) * qscale;
            out.y = (cf.x * q0[j].y + cf.y * q2[j].y) * qscale;
            out.z = (cf.z * q1[j].x) * qscale;
            out.w = (cf.z * q1[j].y) * qscale;
            if (o.real_only) out.y = out.w = 0.0;
            double *d = &cfs[b][s][2 + 4 * f];
            d[0] = out.x; d[1] = out.y; d[2] = out.z; d[3] = out.w;
            if (f == 0) { cfs[b][s][0] = cab[j].x; cfs[b][s][1] = cab[j].y; }
        }
    };
#pragma unroll
    for (int r = 0; r < R; ++r) {
        for (int off = 32; off >= 1; off >>= 1) {
            wmin[r] = min(wmin[r], __shfl_xor(wmin[r], off));
        }
        wmin[r] = __builtin_amdgcn_readfirstlane(wmin[r]) & ~3;
        wbeg = min(wbeg, wmin[r]);
    }
    for (int off = 32; off >= 1; off >>= 1) wlast = max(wlast, __shfl_xor(wlast, off));
    wlast = __builtin_amdgcn_readfirstlane(wlast);
    if (lane == 0) s_beg[wave] = wbeg;
    __syncthreads();
    int beg = nsteps;
    for (int w = 0; w < nw; ++w) beg = min(beg, s_beg[w]);
    beg = __builtin_amdgcn_readfirstlane(beg) & ~(CS - 1);
    if (beg < nsteps) {
        fetch(beg);
        put(0);
    }
    __syncthreads();
    int b = 0;
    for (int ch = beg; ch < nsteps; ch += CS, b ^= 1) {
        const bool more = ch + CS < nsteps;
        if (more) fetch(ch + CS);
        const int send = min(CS, nsteps - ch), sbeg = max(0, wbeg - ch);
        int s4 = sbeg;
        // some latitude of the wave still starts: tile by tile
        for (; s4 < send && ch + s4 <= wlast; s4 += 4) {   // rows past nsteps hold zeros
            const int i = ch + s4;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (i < wmin[r]) continue;   // wave-uniform: not started
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const double *c = cfs[b][s4 + s];
                    if (i + s == i0[r]) { za[r] = sd[r].x; zb[r] = sd[r].y; }
                    step(r, c);
                }
            }
        }
        // all started: the tiles' independent chains side by side, coefficients read once
        for (; s4 < send; s4 += 2) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                double c[ROW];
#pragma unroll
                for (int e = 0; e < ROW; e += 2) {
                    const double2 v = *reinterpret_cast<const double2 *>(&cfs[b][s4 + s][e]);
                    c[e] = v.x;
                    c[e + 1] = v.y;
                }
#pragma unroll
                for (int r = 0; r < R; ++r) step(r, c);
            }
        }
        if (more) put(b ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int tile = tb + wave * R + r, k = tile * 64 + lane;
        if (tile >= tile0 + ntl || k >= nlat_2) continue;
        const double x = xk[k];
        // the middle row of an odd grid is its own mirror: its stored pair weight is halved
        const double w = lat_weight ? wqk[k] * ((2 * k + 1 == nlat) ? 2.0 : 1.0) : 1.0, wi = (im == 0) ? 0.0 : w;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            double2 *Ff = F + (size_t)f * four_dist + (size_t)im * nlat;
            const double *a = acc[r][f];
            Ff[k] = make_double2(fma(x, a[2], a[0]) * w, fma(x, a[3], a[1]) * wi);
            Ff[nlat - 1 - k] = make_double2(fma(-x, a[2], a[0]) * w, fma(-x, a[3], a[1]) * wi);
        }
    }
}

// Tiles per wave: one up to 12 tiles, then two (the coefficient reads of a step are shared and
// two chains run side by side): lmax=2047, 1 / 2 fields, call 545 / 976 us, one tile per wave
// 679 / 1218, three 548 / 991, six 692; lmax=511, one field 33.6, two tiles 35.8.
template <int NF>
void launch_synth_few(const LegendreArgs &a, const double2 *Q, long spec_dist, int spec_ltop, double2 *F, long four_dist,
                      hipStream_t s) {
    const DeviceTables *t = a.t;
    const int ntl = (a.nlat_2 + 63) / 64;
#define SYNTH_FEW(RR)                                                                                              \
    {                                                                                                              \
        const int nw = std::min(4, (ntl + RR - 1) / RR), nblk = (ntl + nw * RR - 1) / (nw * RR);                   \
        hipLaunchKernelGGL((legendre_synth_few_kernel<NF, RR>), dim3((a.mmax + 1) * nblk), dim3(64 * nw), 0, s,    \
                           t->x, t->x2, t->wq, t->step_ofs, t->ab, t->pm, a.vector_mode ? t->i0v : t->i0,          \
                           a.vector_mode ? t->z0v : t->z0, Q, spec_dist, spec_ltop, F, four_dist, a.mmax, a.mres,  \
                           a.nlat, a.nlat_2, a.ltr, a.imlim, a.vector_mode, a.mpos_scale, a.lat_weight, 0, ntl,    \
                           nblk);                                                                                  \
    }
    if (ntl <= 12) SYNTH_FEW(1)
    else SYNTH_FEW(2)
#undef SYNTH_FEW
}

// ---------------------------------------------------------------------------------------
// Analysis: Q_lm = sum_k w_k P_lm(x_k) F_m(x_k)
// Block = NW waves for one order im and 4*NCG fields; wave w owns latitude tiles
// w + NW*r (r < NLR) of 64 pairs, lane = latitude pair.  The weighted E/O values of the
// block's fields for the owned latitudes are held in registers as MFMA B operands.
// Per 16-step block: each lane advances its recurrences into a wave-private LDS tile, the
// tile is read back as the A operand (16 steps x 4 latitudes) and
// D[16 step][16 col] += A * B runs over all owned K-groups; the waves' partial D go to a
// double-buffered LDS area, one barrier, then every thread sums one (step, column) over
// the waves and applies the post-mix (even: ue_i acc_i + ue1_{i-1} acc_{i-1}; odd:
// uo_i acc_i) and stores Q.  Fixed summation order: results are deterministic.
// ---------------------------------------------------------------------------------------
// NF4 > 0 (FP64, NCG = 1, at most 3 fields): field c is contracted with v_mfma_f64_4x4x4f64
// (four 4x4x4 blocks = 16 steps x 4 latitudes x the field's 4 columns; the A operand is the
// 16x16x4 one, B lane l holds column l & 3 of latitude 4 kg + (l >> 4) in every block, and
// D lane l holds step 4 ((l >> 2) & 3) + (l >> 4), column l & 3).
// NG > 1 (one tile per wave): the block holds NG field groups of the same order, waves
// w = tw + NW g (tile tw, group g); each group's NW partial tiles are reduced separately.
// Six-tile grids then run 12-wave blocks (three waves on every SIMD) instead of 6-wave ones.
// GR > 1 (4x4x4 path, one tile per wave): GR 16-step groups share one barrier pair and one
// reduction round (16 GR rows of partial tiles), for batches whose MFMA work per group is
// too small to cover those fixed costs.
template <int NW, int NLR, int NF4, int GR = 1>
__global__ __launch_bounds__(64 * NW) void legendre_anal_kernel(
    const double *__restrict__ xk, const double *__restrict__ x2k, const double *__restrict__ stk,
    const double *__restrict__ wqk, const int *__restrict__ step_ofs, const double2 *__restrict__ ab,
    const double4 *__restrict__ pm, const int *__restrict__ i0tab, const double2 *__restrict__ z0tab,
    const double2 *__restrict__ F, long four_dist, double2 *__restrict__ Q, long spec_dist, int lmax_spec,
    int spec_ltop, int mmax, int mres, int nlat, int nlat_2, int ltr, int imlim, int nfields, int vector_mode,
    double mpos_scale, int lat_weight, int cf_lds, int tile_base) {
    static_assert(NF4 == 1 || NF4 == 2, "one or two fields");
    static_assert(GR == 1 || (GR == 2 && NLR == 1), "two groups per round: one tile per wave");
    constexpr int RR = 16 * GR;                   // steps per reduction round
    constexpr int NCOL = 4 * NF4;
    constexpr int NT = 64 * NW;                   // threads per block
    __shared__ double ytile[NW][16][65];
    // cf_lds: the order's recurrence coefficients (alpha_i, beta_i), i < nsteps, are copied to
    // LDS once per block (dynamic LDS), so each 16-step group reads them at LDS latency instead
    // of waiting on scalar loads that miss to HBM
    extern __shared__ double2 cfl[];
    // single-buffered: two barriers per block.  Rows padded to NCOL + 2 doubles: a post-mix read
    // (32 lanes = steps 0..15 of two adjacent columns) then falls on 32 distinct bank pairs
    __shared__ double red[NW][RR][NCOL + 2];
    __shared__ double carry[2][NCOL];
    __shared__ int s_ibeg[NW];

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int im = blockIdx.x;   // blocks are dispatched in index order: the heavy low orders start first

    const OrderInfo o = order_info(im, lmax_spec, mmax, mres, (im <= imlim) ? ltr : -1, vector_mode);
    const int nsteps = (im <= imlim) ? o.nsteps : 0;
    const int sofs = step_ofs[o.slot];
    const UniformTable2 abm(ab + sofs);   // uniform indices -> scalar loads
    const double4 *pmm = pm + sofs;

    // (multi-tile waves keep their registers for the operands: scalar loads there)
    if constexpr (NLR >= 3) cf_lds = 0;
    // one-tile waves load the coefficient-table copy before the operands below: global loads
    // complete in issue order, so its LDS store (before the first barrier) then waits only for
    // these (multi-tile waves have no registers to spare and load it afterwards)
    constexpr int NCF = (NLR == 1) ? 4 : 0;   // per thread; the rest of the table, if any, below
    double2 cfr[NCF > 0 ? NCF : 1];
    if (NCF > 0 && cf_lds) {
#pragma unroll
        for (int q = 0; q < NCF; ++q) {
            const int e = threadIdx.x + q * NT;
            cfr[q] = (e < nsteps) ? ab[sofs + e] : make_double2(0.0, 0.0);
        }
    }

    double za[NLR], zb[NLR], x2v[NLR], sdx[NLR], sdy[NLR];
    int i0v[NLR];
    double Ereg[NLR][NF4][16];
    int my_ibeg = nsteps, my_imax = 0;
#pragma unroll
    for (int r = 0; r < NLR; ++r) {
        const int k = (tile_base + wave + NW * r) * 64 + lane;
        const bool kv = (k < nlat_2);
        const int kk = kv ? k : 0;
        x2v[r] = x2k[kk];
        int i0 = kv ? i0tab[(size_t)o.slot * nlat_2 + kk] : nsteps;
        if (i0 > nsteps) i0 = nsteps;
        double2 sd = z0tab[(size_t)o.slot * nlat_2 + kk];
        if (o.sinv) {
            const double inv = 1.0 / stk[kk];
            sd.x *= inv;
            sd.y *= inv;
        }
        i0v[r] = i0;
        sdx[r] = sd.x;
        sdy[r] = sd.y;
        my_ibeg = min(my_ibeg, i0);
        my_imax = max(my_imax, kv ? i0 : 0);
        // B operand for K-group kg: latitude tile_base + 4*kg + lane/16, column lane%16 of group c
        // (E.re, E.im, O.re, O.im = weighted N+S, N+S, (N-S) x, (N-S) x).  Branch-free, every
        // load issued before the first use: the block's first MFMA waits for these.
        const int comp = lane & 3;
        const bool keep = nsteps > 0 && !(o.real_only && (comp & 1));
        // latitude of K-group 0; K-slot k of K-group 2 p + j is latitude 8 p + 2 k + j of the tile,
        // as in legendre_anal_shared_kernel (both sum in the same order: equal results)
        const int kl0 = (tile_base + wave + NW * r) * 64 + 2 * (lane >> 4);
        if constexpr (NLR >= 3) {
#pragma unroll
            for (int c = 0; c < NF4; ++c) {
                const int f = c;
                const bool fv = keep && f < nfields;
                const double2 *Ff = F + (size_t)(fv ? f : 0) * four_dist + (size_t)im * nlat;
#pragma unroll
                for (int kg = 0; kg < 16; ++kg) {
                    // several tiles per wave: one K-group at a time (loads hoisted together
                    // would need more registers than the tiles' operands leave)
                    const int kl = kl0 + 8 * (kg >> 1) + (kg & 1);
                    double v = 0.0;
                    if (fv && kl < nlat_2) {
                        const double2 fn = Ff[kl], fs = Ff[nlat - 1 - kl];
                        const double w = lat_weight ? wqk[kl] : ((2 * kl + 1 == nlat) ? 0.5 : 1.0);   // odd grid: equator row once
                        v = (comp == 0 ? fn.x + fs.x : comp == 1 ? fn.y + fs.y
                             : comp == 2 ? (fn.x - fs.x) * xk[kl] : (fn.y - fs.y) * xk[kl]) * w;
                    }
                    Ereg[r][c][kg] = v;
                }
            }
        } else {
            // Batches of KB K-groups: every load of a batch is issued before its first use
            // (clamped indices, no branches; each lane loads only the real or imaginary part
            // its column takes), and the batches are fenced so the scheduler does not hoist
            // later batches' loads above them.  The arithmetic is that of the branchy form
            // above, rounding for rounding: (a + b) w for E, ((a - b) x) w for O, with a - b
            // as one fma by -1.
            constexpr int KB = 4;
            const bool neg = comp & 2;
            const double sgn = neg ? -1.0 : 1.0;
            const double *Fc[NF4];
            bool fvc[NF4];
#pragma unroll
            for (int c = 0; c < NF4; ++c) {
                const int f = c;
                fvc[c] = keep && f < nfields;
                Fc[c] = reinterpret_cast<const double *>(F + (size_t)(fvc[c] ? f : 0) * four_dist + (size_t)im * nlat) +
                        (comp & 1);
            }
#pragma unroll
            for (int kb = 0; kb < 16; kb += KB) {
                double xq[KB], wq[KB], aq[NF4][KB], bq[NF4][KB];
#pragma unroll
                for (int q = 0; q < KB; ++q) {
                    const int kl = kl0 + 8 * ((kb + q) >> 1) + (q & 1);
                    const int klx = (kl < nlat_2) ? kl : 0;
                    xq[q] = xk[klx];
                    const double wl = wqk[klx];
                    wq[q] = lat_weight ? wl : ((2 * klx + 1 == nlat) ? 0.5 : 1.0);   // odd grid: equator row once
#pragma unroll
                    for (int c = 0; c < NF4; ++c) {
                        const int klc = (fvc[c] && kl < nlat_2) ? kl : 0;
                        aq[c][q] = Fc[c][2 * klc];
                        bq[c][q] = Fc[c][2 * (nlat - 1 - klc)];
                    }
                }
#pragma unroll
                for (int q = 0; q < KB; ++q) {
                    const int kl = kl0 + 8 * ((kb + q) >> 1) + (q & 1);
#pragma unroll
                    for (int c = 0; c < NF4; ++c) {
                        const double s = fma(sgn, bq[c][q], aq[c][q]);
                        double v = (fvc[c] && kl < nlat_2) ? (neg ? s * xq[q] : s) * wq[q] : 0.0;
                        // computed here, not sunk towards the MFMAs (which would keep every
                        // batch's loaded values live across the prologue)
                        asm volatile("" : "+v"(v));
                        Ereg[r][c][kb + q] = v;
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    for (int off = 32; off >= 1; off >>= 1) {
        my_ibeg = min(my_ibeg, __shfl_xor(my_ibeg, off));
        my_imax = max(my_imax, __shfl_xor(my_imax, off));
    }
    my_imax = __builtin_amdgcn_readfirstlane(my_imax);
    if (lane == 0) s_ibeg[wave] = my_ibeg;
    if (threadIdx.x < 2 * NCOL) (&carry[0][0])[threadIdx.x] = 0.0;
    if (cf_lds) {
#pragma unroll
        for (int q = 0; q < NCF; ++q) {
            const int e = threadIdx.x + q * NT;
            if (e < nsteps) cfl[e] = cfr[q];
        }
        for (int e = threadIdx.x + NCF * NT; e < nsteps; e += NT) cfl[e] = ab[sofs + e];   // rest, if any
    }
    __syncthreads();
    int ibeg = nsteps;
    for (int w = 0; w < NW; ++w) ibeg = min(ibeg, s_ibeg[w]);
    ibeg = __builtin_amdgcn_readfirstlane(ibeg) & ~15;   // block-uniform, scalar from here on
#pragma unroll
    for (int r = 0; r < NLR; ++r) {
        za[r] = 0.0;
        zb[r] = 0.0;
        if (i0v[r] == ibeg) { za[r] = sdx[r]; zb[r] = sdy[r]; }
    }

    const double qscale = (im == 0) ? 1.0 : mpos_scale;
    const int nsteps_out = (spec_ltop >= o.mfun) ? (spec_ltop - o.mfun) / 2 + 1 : 0;
    double2 *Qbase = Q + o.spec_base;

    // post-mix work split: thread handles elements e = threadIdx.x + j*NT (j < NE) of the
    // 16 x NCOL block, step row e % 16 of column e / 16, each for all NG field groups (the
    // same coefficient row); the coefficient rows are prefetched before the MFMA phase.
    // Each 16-lane DPP row holds the 16 steps of one column, so the sum of step row - 1 (the
    // even degrees' second term) is the neighbouring lane's, and a wave's stores cover the
    // 32 consecutive degrees of one field (16 NCOL is a multiple of 64: whole waves take part
    // or skip an element together).
    constexpr int NE = (RR * NCOL + NT - 1) / NT;
    auto cf_at = [&](auto from_lds, int idx) {
        idx = min(idx, nsteps - 1);
        if constexpr (decltype(from_lds)::value) return cfl[idx];   // uniform: LDS broadcast
        else return abm[idx];                                        // uniform: scalar load
    };
    // recurrence of the 16-step group from ig of tile r into this wave's tile buffer
    auto recur_plain = [&](int r, int ig, const double2 *cfg) {
        if (ig <= my_imax) {   // some lane of this wave starts its recurrence here
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                if (ig + s == i0v[r]) { za[r] = sdx[r]; zb[r] = sdy[r]; }
                ytile[wave][s][lane] = zb[r];
                const double zn = fma(fma(cfg[s].x, x2v[r], cfg[s].y), zb[r], za[r]);
                za[r] = zb[r];
                zb[r] = zn;
            }
        } else {
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                ytile[wave][s][lane] = zb[r];
                const double zn = fma(fma(cfg[s].x, x2v[r], cfg[s].y), zb[r], za[r]);
                za[r] = zb[r];
                zb[r] = zn;
            }
        }
    };
    auto load_cf16 = [&](double2 *cf, int ig) {
        if (cf_lds) {
#pragma unroll
            for (int s = 0; s < 16; ++s) cf[s] = cf_at(std::true_type{}, ig + s);
        } else {
#pragma unroll
            for (int s = 0; s < 16; ++s) cf[s] = cf_at(std::false_type{}, ig + s);
        }
    };
    int b = 0;
    for (int i = ibeg; i < nsteps; i += RR, ++b) {
        double pcx[NE], pcz[NE], pcp[NE];
#pragma unroll
        for (int j = 0; j < NE; ++j) {
            const int e = threadIdx.x + j * NT;
            const int row = e & (RR - 1);
            const int ii = min(i + row, nsteps - 1);
            const double4 cf4 = pmm[ii];
            pcx[j] = cf4.x;
            pcz[j] = cf4.z;
            pcp[j] = (ii > 0) ? pmm[ii - 1].y : 0.0;
        }
        double acc[GR][NF4], acc2[GR][NF4];   // two chains per field (halves of the tile)
#pragma unroll
        for (int q = 0; q < GR; ++q)
#pragma unroll
            for (int c = 0; c < NF4; ++c) acc[q][c] = acc2[q][c] = 0.0;
#pragma unroll
        for (int q = 0; q < GR; ++q) {
            double2 cf[16];
            load_cf16(cf, i + 16 * q);
#pragma unroll
            for (int r = 0; r < NLR; ++r) {
                recur_plain(r, i + 16 * q, cf);
                double a[16];
                __builtin_amdgcn_s_waitcnt(0xc07f);
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int kg = 0; kg < 16; ++kg) a[kg] = ytile[wave][lane & 15][8 * (kg >> 1) + 2 * (lane >> 4) + (kg & 1)];
                __builtin_amdgcn_s_waitcnt(0xc07f);   // all A operands in registers before the tile is rewritten
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int kg = 0; kg < 8; ++kg)
#pragma unroll
                    for (int c = 0; c < NF4; ++c) {
                        acc[q][c] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[kg], Ereg[r][c][kg], acc[q][c], 0, 0, 0);
                        acc2[q][c] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[kg + 8], Ereg[r][c][kg + 8], acc2[q][c], 0, 0, 0);
                    }
            }
        }
#pragma unroll
        for (int q = 0; q < GR; ++q)
#pragma unroll
            for (int c = 0; c < NF4; ++c) acc[q][c] += acc2[q][c];
        const int pb = b & 1;
        __syncthreads();   // previous block's post-mix has finished reading red
        // 4x4x4 D: step 4 ((lane >> 2) & 3) + (lane >> 4), column lane & 3 of field c
#pragma unroll
        for (int q = 0; q < GR; ++q)
#pragma unroll
            for (int c = 0; c < NF4; ++c)
                red[wave][16 * q + 4 * ((lane >> 2) & 3) + (lane >> 4)][4 * c + (lane & 3)] = acc[q][c];
        __syncthreads();
        // sum over the waves + post-mix
#pragma unroll
        for (int j = 0; j < NE; ++j) {
            const int e = threadIdx.x + j * NT;
            if (e >= RR * NCOL) break;   // wave-uniform
            const int row = e & (RR - 1), col = e / RR;
            const int comp = col & 3;
            const int ii = i + row;
            const int f = col >> 2;
            double sum = 0.0;
#pragma unroll
            for (int w = 0; w < NW; ++w) sum += red[w][row][col];
            // step row - 1 of this column: lane - 1 (the whole wave is active here; within
            // a DPP row for 16-row rounds, a wave-wide shift for 32), or the previous
            // round's last row
            double sprev = (GR == 1) ? row_shr1(sum) : __shfl_up(sum, 1);
            if (row == 0) sprev = carry[pb ^ 1][col];
            if (row == RR - 1 && comp < 2) carry[pb][col] = sum;
            if (f >= nfields || ii >= nsteps_out) continue;
            const int le = o.mfun + 2 * ii;
            double v = 0.0;
            if (ii < nsteps) {
                if (comp < 2) {
                    v = pcx[j] * sum + pcp[j] * sprev;
                } else {
                    v = pcz[j] * sum;
                }
            }
            const int ld = (comp < 2) ? le : le + 1;
            if (ld <= spec_ltop) {
                double out = (ld <= ltr) ? v * qscale : 0.0;
                if (o.real_only && (comp & 1)) out = 0.0;
                reinterpret_cast<double *>(&Qbase[(size_t)f * spec_dist + ld])[comp & 1] = out;
            }
        }
    }
    // degrees not reached by the step loop: before ibeg (negligible functions) and after nsteps
    for (int ii = threadIdx.x; ii < nsteps_out; ii += NT) {
        if (ii >= ibeg && ii < ibeg + ((nsteps - ibeg + RR - 1) / RR) * RR) continue;
        const int le = o.mfun + 2 * ii;
        for (int f = 0; f < nfields; ++f) {
            double2 *Qf = Qbase + (size_t)f * spec_dist;
            if (le <= spec_ltop) Qf[le] = make_double2(0.0, 0.0);
            if (le + 1 <= spec_ltop) Qf[le + 1] = make_double2(0.0, 0.0);
        }
    }
    if (vector_mode && im == 0 && threadIdx.x == 0) {   // degree 0 of the vector m=0 spectra
        for (int f = 0; f < nfields; ++f) Qbase[(size_t)f * spec_dist] = make_double2(0.0, 0.0);
    }
}

// static LDS of legendre_anal_kernel, and whether the order's coefficient table (ltr/2 + 2
// pairs) fits beside it in the 160 KB of a CU
constexpr size_t anal_static_lds(int NW, int NF4, int GR) {
    return sizeof(double) * (NW * 16 * 65 + NW * 16 * GR * (4 * NF4 + 2) + 8 * NF4) + sizeof(int) * NW;
}
inline bool anal_cf_fits(size_t static_lds, int ltr) {
    return static_lds + sizeof(double2) * (size_t)(ltr / 2 + 2) + 1024 <= 160 * 1024;
}

template <int NW, int NLR, int NF4, int GR = 1>
void launch_anal_few(const LegendreArgs &a, const double2 *F, long four_dist, double2 *Q, long spec_dist,
                     int spec_ltop, hipStream_t s, int tile_base = 0) {
    const DeviceTables *t = a.t;
    // static LDS of the kernel, and the coefficient table if it fits beside it in 160 KB
    constexpr size_t static_lds = anal_static_lds(NW, NF4, GR);
    const size_t cf_bytes = sizeof(double2) * (size_t)(a.ltr / 2 + 2);
    const int cf_lds = anal_cf_fits(static_lds, a.ltr) ? 1 : 0;
    const size_t dyn = cf_lds ? cf_bytes : 0;
    ensure_lds_limit((const void *)legendre_anal_kernel<NW, NLR, NF4, GR>, dyn);
    hipLaunchKernelGGL((legendre_anal_kernel<NW, NLR, NF4, GR>), dim3(a.mmax + 1), dim3(64 * NW), dyn, s, t->x, t->x2, t->st,
                       t->wq, t->step_ofs, t->ab, t->pm, a.vector_mode ? t->i0v : t->i0,
                       a.vector_mode ? t->z0v : t->z0, F, four_dist, Q, spec_dist,
                       spec_ltop == a.lmax + 1 ? a.lmax + 1 : a.lmax, spec_ltop, a.mmax, a.mres, a.nlat, a.nlat_2,
                       a.ltr, a.imlim, a.nfields, a.vector_mode, a.mpos_scale, a.lat_weight, cf_lds, tile_base);
}

// ---------------------------------------------------------------------------------------
// Analysis with the recurrence values shared by the block (three or more fields).
//
// Block = CT x TT waves for one order and 4 CT fields.  Per group of 16 steps:
//   1. the owners of the NTB latitude tiles (wave w < NTB, lane = latitude pair) advance their
//      recurrences and write the values to LDS (the quadrature weights are folded into the
//      seeds); the previous group's sums are post-mixed;
//   2. wave (c, t) contracts column tile c (4 fields) over the t-th part of the latitudes, its
//      E/O data held in registers as MFMA B operands (KGW K-groups of 4 latitudes); the
//      TT partial 16 x 16 sums go to LDS.
// A pair of K-groups is one 16-byte LDS read: K-slot k of K-group 2 p + j is latitude
// 8 p + 2 k + j, rows of PS doubles with PS = 2 mod 16 (no bank conflicts).
// Tiles whose functions have not started (first step of the tile beyond the group) are
// skipped: no recurrence, no LDS reads, no MFMAs.
//
// The launch covers latitude pairs tile_base * 64 .. pair_end - 1.  accumulate: add to Q instead
// of storing (the launches after the first where the latitudes do not fit one block).
// ---------------------------------------------------------------------------------------
template <int NTB, int CT, int TT, int H>
struct AnalGeom {
    static constexpr int NW = CT * TT, NT = 64 * NW;
    static constexpr int NTH = NTB / H;            // tiles per half
    static constexpr int KGW = 16 * NTH / TT;      // K-groups per wave and half
    static constexpr int PS = 64 * NTH + 2;        // doubles per step row of a recurrence buffer
    static constexpr int NCOL = 16 * CT;
    static constexpr int TPO = (NTB + NW - 1) / NW;   // tiles per owner
    static_assert(NTB % H == 0 && 16 * NTH % TT == 0 && KGW % 2 == 0 && NW <= 16, "analysis block shape");
    static_assert(H == 1 || TPO == H, "halves: each wave owns one tile of each");
};

// K-groups of the batch of operand loads that starts at K-group kb: two loads each, beside the
// kb operands already in registers
constexpr int anal_batch(int kb, int kgw) {
    int n = kgw > 64 ? (2 * kgw - kb) / 2 & ~3 : (64 - kb) / 2 & ~3;
    if (n < 4) n = 4;
    return n < kgw - kb ? n : kgw - kb;
}

template <int NTB, int CT, int TT, int H, int PREC>
__global__ __launch_bounds__(64 * CT * TT) void legendre_anal_shared_kernel(
    const double *__restrict__ xk, const double *__restrict__ x2k, const double *__restrict__ wqk,
    const int *__restrict__ step_ofs, const double2 *__restrict__ ab, const double4 *__restrict__ pm,
    const int *__restrict__ i0tab, const double2 *__restrict__ z0tab, const double2 *__restrict__ F, long four_dist,
    double2 *__restrict__ Q, long spec_dist, int lmax_spec, int spec_ltop, int mmax, int mres, int nlat, int nlat_2,
    int ltr, int imlim, int nfields, int vector_mode, double mpos_scale, int lat_weight, int tile_base,
    int pair_end, int accumulate) {
    using G = AnalGeom<NTB, CT, TT, H>;
    using C = Contract<PREC>;
    constexpr int NT = G::NT, NW = G::NW, NTH = G::NTH, KGW = G::KGW, PS = G::PS, NCOL = G::NCOL, TPO = G::TPO;
    __shared__ __attribute__((aligned(16))) double pt[16 * PS > 128 * NTB ? 16 * PS : 128 * NTB];
    __shared__ double red[TT][16][NCOL + 2];   // partial sums of the parts
    __shared__ double carry[2][NCOL];
    __shared__ double4 pmr[4][16];   // post-mix coefficients of the groups in flight
    __shared__ int s_tbeg[NTB];
    __shared__ double2 s_seed[64 * NTB];   // seeds and first steps of the block's latitudes
    __shared__ int s_i0[64 * NTB];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = wave % CT, t = wave / CT;   // column tile, latitude part
    const int ngr = gridDim.x / (mmax + 1);
    const int im = blockIdx.x / ngr;          // field groups fastest: heavy low orders start first
    const int fbase = (blockIdx.x - im * ngr) * 4 * CT;

    const OrderInfo o = order_info(im, lmax_spec, mmax, mres, (im <= imlim) ? ltr : -1, vector_mode);
    const int nsteps = (im <= imlim) ? o.nsteps : 0;
    const int sofs = step_ofs[o.slot];
    const int last_row = step_ofs[o.slot + 1] - sofs - 1;   // >= nsteps + 6
    const UniformTable2 abm(ab + sofs);

    // Recurrence state of the owned tiles (every NW-th one; with halves, NTH / NW of each
    // half).  The seeds wait in LDS: they would cost registers through the whole loop.
    auto tile_of = [&](int r) { return H == 1 ? wave + NW * r : wave < NTH ? r * NTH + wave : NTB; };
    int my_ibeg[TPO], my_imax[TPO];
    double x2[TPO], za[TPO], zb[TPO];
    double2 sd[TPO];
#pragma unroll
    for (int r = 0; r < TPO; ++r) {
        const int tile = tile_of(r), k = (tile_base + tile) * 64 + lane;
        const bool kv = tile < NTB && k < pair_end;
        const int kk = kv ? k : 0;
        const size_t at = (size_t)o.slot * nlat_2 + kk;
        x2[r] = x2k[kk];
        za[r] = zb[r] = 0.0;
        my_ibeg[r] = kv ? min(i0tab[at], nsteps) : nsteps;
        sd[r] = z0tab[at];
    }
    // cos(theta) and the weights of the block's latitudes, through LDS (the recurrence buffer)
    constexpr int NX = (64 * NTB + NT - 1) / NT;
    double *xs = pt, *ws = pt + 64 * NTB;
    double xv[NX], wv[NX];
#pragma unroll
    for (int q = 0; q < NX; ++q) {
        const int k = tile_base * 64 + threadIdx.x + q * NT, kx = min(k, nlat_2 - 1);
        xv[q] = xk[kx];
        wv[q] = wqk[kx];
        if (!lat_weight) wv[q] = (2 * kx + 1 == nlat) ? 0.5 : 1.0;   // odd grid: the equator row, both rows of its pair, once
        if (k >= pair_end) wv[q] = 0.0;
    }
    auto put_tables = [&]() {
#pragma unroll
        for (int q = 0; q < NX; ++q) {
            const int e = threadIdx.x + q * NT;
            if (e < 64 * NTB) { xs[e] = xv[q]; ws[e] = wv[q]; }
        }
#pragma unroll
        for (int r = 0; r < TPO; ++r) {
            const int tile = tile_of(r);
            if (tile < NTB) {
                s_seed[tile * 64 + lane] = sd[r];
                s_i0[tile * 64 + lane] = my_ibeg[r];
            }
        }
        __syncthreads();
    };

    // B operands.  The Fourier rows are loaded in as few batches as the registers allow (every
    // load of a batch in flight before the first is used, the batches fenced): each batch costs
    // the block a full memory latency.
    typename C::b_t Breg[H * KGW];
    {
        const int col = lane & 15, comp = col & 3, f = fbase + 4 * c + (col >> 2);
        const bool keep = nsteps > 0 && !(o.real_only && (comp & 1)) && f < nfields;
        const bool neg = comp & 2;
        const double sgn = neg ? -1.0 : 1.0;
        const double *Fc = reinterpret_cast<const double *>(F + (size_t)(keep ? f : 0) * four_dist + (size_t)im * nlat) + (comp & 1);
        const int kloc = t * KGW * 4 + 2 * (lane >> 4), kl0 = tile_base * 64 + kloc;
        // latitude offset of K-group n (halves: the part's share of each)
        auto dk_of = [](int n) { return (n / KGW) * 64 * NTH + 8 * ((n % KGW) >> 1) + (n & 1); };
        auto load = [&](auto full, auto kbc, auto KBc) {   // K-groups kb .. kb + KB - 1
            constexpr int kb = decltype(kbc)::value, KB = decltype(KBc)::value;
            double aq[KB], bq[KB];
#pragma unroll
            for (int q = 0; q < KB; ++q) {
                const int dk = dk_of(kb + q);
                const int kl = decltype(full)::value ? kl0 + dk : min(kl0 + dk, nlat_2 - 1);
                aq[q] = Fc[2 * kl];
                bq[q] = Fc[2 * (nlat - 1 - kl)];
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (kb == 0) put_tables();
#pragma unroll
            for (int q = 0; q < KB; ++q) {
                const int e = kloc + dk_of(kb + q);
                const double s = fma(sgn, bq[q], aq[q]);
                double v = keep ? (neg ? s * xs[e] : s) * ws[e] : 0.0;
                asm volatile("" : "+v"(v));
                Breg[kb + q] = C::split(v);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto all = [&](auto self, auto full, auto kbc) -> void {
            constexpr int kb = decltype(kbc)::value, n = anal_batch(kb, H * KGW);
            load(full, kbc, std::integral_constant<int, n>{});
            if constexpr (kb + n < H * KGW) self(self, full, std::integral_constant<int, kb + n>{});
        };
        constexpr std::integral_constant<int, 0> k0{};
        if ((tile_base + NTB) * 64 <= pair_end) all(all, std::true_type{}, k0);
        else all(all, std::false_type{}, k0);
    }
#pragma unroll
    for (int r = 0; r < TPO; ++r) {
        my_imax[r] = my_ibeg[r] < nsteps ? my_ibeg[r] : 0;   // lanes that never start stay zero
        for (int off = 32; off >= 1; off >>= 1) {
            my_ibeg[r] = min(my_ibeg[r], __shfl_xor(my_ibeg[r], off));
            my_imax[r] = max(my_imax[r], __shfl_xor(my_imax[r], off));
        }
        my_ibeg[r] = __builtin_amdgcn_readfirstlane(my_ibeg[r]);
        my_imax[r] = __builtin_amdgcn_readfirstlane(my_imax[r]);
        if (tile_of(r) < NTB && lane == 0) s_tbeg[tile_of(r)] = my_ibeg[r];
    }
    __syncthreads();
    int ibeg = nsteps;
    for (int w = 0; w < NTB; ++w) ibeg = min(ibeg, s_tbeg[w]);
    ibeg = __builtin_amdgcn_readfirstlane(ibeg) & ~15;
    // first steps of the tiles this wave contracts (one per 16 K-groups, or the one its part is
    // in; parts that straddle tiles take the first of any of them, and every tile is then written)
    constexpr bool STRADDLE = !(KGW % 16 == 0 || 16 % KGW == 0);
    constexpr int TPW = !STRADDLE && KGW >= 16 ? KGW / 16 : 1, KGT = KGW / TPW;
    int tb[H * TPW];
#pragma unroll
    for (int q = 0; q < H * TPW; ++q) {
        int b = nsteps;
        const int k0 = t * KGW + (q % TPW) * KGT, h0 = (q / TPW) * NTH;
        for (int w = k0 / 16; w <= (k0 + KGT - 1) / 16; ++w) b = min(b, s_tbeg[h0 + w]);
        tb[q] = __builtin_amdgcn_readfirstlane(b);
    }
    // the 16 steps from ig of the owned tiles into LDS
    auto recur = [&](int ig, const double2 *cf, int half) {
#pragma unroll
        for (int r = 0; r < TPO; ++r) {
            if (H > 1 && r != half) continue;
            if (tile_of(r) >= NTB || (!STRADDLE && ig + 16 <= my_ibeg[r])) continue;   // not started: nobody reads it
            const int tile = tile_of(r), h = tile / NTH;
            double *dst = &pt[(tile - h * NTH) * 64 + lane];
            if (ig <= my_imax[r]) {   // some lane of this wave starts its recurrence here
                const int i0 = s_i0[tile * 64 + lane];
                const double2 sd = s_seed[tile * 64 + lane];
#pragma unroll
                for (int s = 0; s < 16; ++s) {
                    if (ig + s == i0) { za[r] = sd.x; zb[r] = sd.y; }
                    C::store_z(dst + s * PS, zb[r]);
                    const double zn = fma(fma(cf[s].x, x2[r], cf[s].y), zb[r], za[r]);
                    za[r] = zb[r];
                    zb[r] = zn;
                    if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // few factors ahead: registers
                }
            } else {
#pragma unroll
                for (int s = 0; s < 16; ++s) {
                    C::store_z(dst + s * PS, zb[r]);
                    const double zn = fma(fma(cf[s].x, x2[r], cf[s].y), zb[r], za[r]);
                    za[r] = zb[r];
                    zb[r] = zn;
                    if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // few factors ahead: registers
                }
            }
        }
    };
    // coefficients of a group (wave-uniform: scalar loads), clamped to the order's table
    auto load_cf = [&](double2 *cf, int ig) {
#pragma unroll
        for (int s = 0; s < 16; s += 4) {
            const int i4 = min(ig + s, last_row - 3);
#pragma unroll
            for (int q = 0; q < 4; ++q) cf[s + q] = abm[i4 + q];
        }
    };
    constexpr bool TWO = PREC == 0 && KGW > 8 && H * KGW < 64;   // two chains (halves of a tile) where registers allow
    double4_t acc, acc1;
    const bool active = fbase + 4 * c < nfields;   // the last column tiles of a batch may be empty
    auto contract = [&](int ig, auto hc) {
        constexpr int h = decltype(hc)::value;
        const double *src = &pt[(lane & 15) * PS + t * KGW * 4 + 2 * (lane >> 4)];
#pragma unroll
        for (int q = 0; q < TPW; ++q) {
            if (!active || ig + 16 <= tb[h * TPW + q]) continue;   // wave-uniform
            constexpr int NQ = KGT / 2;
            typename C::acc_t part = C::zero();   // FP32 sums over at most 8 K-groups (unused at PREC 0)
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                // the two chains in turn: pairs 0 .. 3 of a tile to acc, 4 .. 7 to acc1
                const int p = (TWO && NQ == 8) ? (n >> 1) + 4 * (n & 1) : n;
                const double2 a2 = *reinterpret_cast<const double2 *>(src + 8 * (q * NQ + p));
                const typename C::b_t b0 = Breg[h * KGW + q * KGT + 2 * p], b1 = Breg[h * KGW + q * KGT + 2 * p + 1];
                if constexpr (PREC == 0) {
                    double4_t &d = (TWO && (p & 4)) ? acc1 : acc;
                    d = C::mma(a2.x, b0, d);
                    d = C::mma(a2.y, b1, d);
                } else {
                    part = C::mma(C::load_z(&a2.y), b1, C::mma(C::load_z(&a2.x), b0, part));
                    if (p % 4 == 3 || p == NQ - 1) {
                        acc += __builtin_convertvector(part, double4_t);
                        part = C::zero();
                    }
                }
            }
        }
    };

    const double qscale = (im == 0) ? 1.0 : mpos_scale;
    const int nsteps_out = (spec_ltop >= o.mfun) ? (spec_ltop - o.mfun) / 2 + 1 : 0;
    double2 *Qbase = Q + o.spec_base;
    // Sum over the parts and post-mix of group i: element e of the 16 x NCOL block is step row
    // e % 16 of column e / 16, so a 16-lane DPP row holds the 16 steps of one column (the even
    // degrees' second term takes the neighbouring lane's sum) and a wave stores the 32
    // consecutive degrees of one field.
    auto post = [&](int i) {
        const int slot = (i >> 4) & 3, pb = (i >> 4) & 1;
        for (int e = threadIdx.x; e < 16 * NCOL; e += NT) {
            const int row = e & 15, col = e >> 4, comp = col & 3;
            const int ii = i + row, f = fbase + (col >> 2);
            double sum = 0.0;
            if constexpr (TT == 2 * NTB) {   // half-tile parts: tile by tile, as the two chains of whole tiles
#pragma unroll
                for (int w = 0; w < TT; w += 2) sum += red[w][row][col] + red[w + 1][row][col];
            } else {
#pragma unroll
                for (int w = 0; w < TT; ++w) sum += red[w][row][col];
            }
            double sprev = row_shr1(sum);
            if (row == 0) sprev = carry[pb ^ 1][col];
            if (row == 15 && comp < 2) carry[pb][col] = sum;
            const int ld = o.mfun + 2 * ii + (comp >> 1);
            if (f >= nfields || ii >= nsteps_out || ld > spec_ltop) continue;
            double v = 0.0;
            if (ii < nsteps) {
                if (comp < 2) v = pmr[slot][row].x * sum + (row ? pmr[slot][row - 1].y : pmr[(slot + 3) & 3][15].y) * sprev;
                else v = pmr[slot][row].z * sum;
            }
            double out = (ld <= ltr) ? v * qscale : 0.0;
            if (o.real_only && (comp & 1)) out = 0.0;
            double *q = &reinterpret_cast<double *>(&Qbase[(size_t)f * spec_dist + ld])[comp & 1];
            *q = accumulate ? *q + out : out;
        }
    };
    auto put_red = [&]() {
        if constexpr (TWO) acc += acc1;
#pragma unroll
        for (int j = 0; j < 4; ++j) red[t][C::d_row(j, lane)][16 * c + (lane & 15)] = acc[j];
    };
    for (int e = threadIdx.x; e < 2 * NCOL; e += NT) (&carry[0][0])[e] = 0.0;
    // (the step before the first group's has zero sums: its coefficient only has to be finite)
    if (threadIdx.x < 4) pmr[threadIdx.x][15] = make_double4(0.0, 0.0, 0.0, 0.0);
    __syncthreads();
    int ng = 0;
    double2 cf[16];
    load_cf(cf, ibeg);
    for (int i = ibeg; i < nsteps; i += 16, ++ng) {
        auto part_of = [&](auto hc) {
            constexpr int h = decltype(hc)::value;
            double4 pmv;
            if (h == 0 && threadIdx.x >= NT - 16) pmv = pm[sofs + min(i + (int)(threadIdx.x & 15), last_row)];
            recur(i, cf, h);
            if (h == 0 && ng > 0) post(i - 16);
            if (h == 0 && threadIdx.x >= NT - 16) pmr[(i >> 4) & 3][threadIdx.x & 15] = pmv;
            __syncthreads();
            if (h == H - 1) load_cf(cf, i + 16);   // in flight during the contraction
            __builtin_amdgcn_sched_barrier(0);
            if (h == 0) {
                acc = double4_t{};
                if constexpr (TWO) acc1 = double4_t{};
            }
            contract(i, hc);
            if (h == H - 1) put_red();
            __syncthreads();
        };
        part_of(std::integral_constant<int, 0>{});
        if constexpr (H > 1) part_of(std::integral_constant<int, 1>{});
        if constexpr (H > 2) part_of(std::integral_constant<int, 2>{});
    }
    if (ng > 0) post(ibeg + 16 * (ng - 1));
    if (accumulate) return;
    // degrees not reached by the step loop: before ibeg (negligible functions) and after nsteps
    for (int ii = threadIdx.x; ii < nsteps_out; ii += NT) {
        if (ii >= ibeg && ii < ibeg + 16 * ng) continue;
        const int le = o.mfun + 2 * ii;
        for (int f = fbase; f < min(nfields, fbase + 4 * CT); ++f) {
            double2 *Qf = Qbase + (size_t)f * spec_dist;
            if (le <= spec_ltop) Qf[le] = make_double2(0.0, 0.0);
            if (le + 1 <= spec_ltop) Qf[le + 1] = make_double2(0.0, 0.0);
        }
    }
    if (vector_mode && im == 0 && threadIdx.x == 0)   // degree 0 of the vector m=0 spectra
        for (int f = fbase; f < min(nfields, fbase + 4 * CT); ++f) Qbase[(size_t)f * spec_dist] = make_double2(0.0, 0.0);
}

template <int NTB, int CT, int TT, int H, int PREC>
void launch_anal_shared(const LegendreArgs &a, const double2 *F, long four_dist, double2 *Q, long spec_dist,
                        int spec_ltop, hipStream_t s, int tile_base, int tiles, int accumulate) {
    const DeviceTables *t = a.t;
    dim3 grid((a.mmax + 1) * ((a.nfields + 4 * CT - 1) / (4 * CT)));
    hipLaunchKernelGGL((legendre_anal_shared_kernel<NTB, CT, TT, H, PREC>), grid, dim3(64 * CT * TT), 0, s, t->x, t->x2,
                       t->wq, t->step_ofs, t->ab, t->pm, a.vector_mode ? t->i0v : t->i0, a.vector_mode ? t->z0v : t->z0,
                       F, four_dist, Q, spec_dist, spec_ltop == a.lmax + 1 ? a.lmax + 1 : a.lmax, spec_ltop, a.mmax,
                       a.mres, a.nlat, a.nlat_2, a.ltr, a.imlim, a.nfields, a.vector_mode, a.mpos_scale, a.lat_weight,
                       tile_base, std::min(a.nlat_2, (tile_base + tiles) * 64), accumulate);
}

// Q[f][i] = sum_s part[s][f][i], i < n (the latitude splits' partial spectra)
void launch_sum_splits(const double2 *part, long part_dist, int nsplit, int nfields, double2 *Q, long spec_dist,
                       long n, hipStream_t s);

// One or two fields in FP64 (4x4x4 blocks, no idle matrix-core columns).
inline void anal_launch_few(const LegendreArgs &a, const double2 *F, long four_dist, double2 *Q, long spec_dist,
                            int spec_ltop, hipStream_t s) {
    const int ntiles = (a.nlat_2 + 63) / 64;
    const int ns = anal_splits(a);
    if (ns > 1 && a.part) {   // 12-wave blocks over a latitude split each, then the sum
        for (int k = 0; k < ns; ++k) {
            double2 *P = a.part + (size_t)k * a.nfields * a.part_dist;
            // one field: two 16-step groups per barrier round where the coefficient table
            // still fits in LDS beside the larger partial-tile buffer
            if (a.nfields == 1 && anal_cf_fits(anal_static_lds(12, 1, 2), a.ltr))
                launch_anal_few<12, 1, 1, 2>(a, F, four_dist, P, a.part_dist, spec_ltop, s, 12 * k);
            else if (a.nfields == 1) launch_anal_few<12, 1, 1>(a, F, four_dist, P, a.part_dist, spec_ltop, s, 12 * k);
            else launch_anal_few<12, 1, 2>(a, F, four_dist, P, a.part_dist, spec_ltop, s, 12 * k);
        }
        launch_sum_splits(a.part, a.part_dist, ns, a.nfields, Q, spec_dist, a.part_dist, s);
        return;
    }
    // waves per block: one latitude tile per wave up to 12 waves (measured fastest: lowest
    // register count, 3 waves per SIMD); beyond, a divisor of the tile count, at most 8
    int nw = 1;
    if (ntiles <= 12) nw = ntiles;
    else
        for (int d = 8; d >= 1; --d)
            if (ntiles % d == 0) { nw = d; break; }
    static const int nw_env = getenv("SHTNS_AMD_ANAL_NW") ? atoi(getenv("SHTNS_AMD_ANAL_NW")) : 0;
    if (nw_env > 0 && nw_env <= 16 && ntiles % nw_env == 0) nw = nw_env;
    if (a.anal_nw > 0 && ntiles % a.anal_nw == 0 && anal_shape_ok(a.anal_nw, ntiles / a.anal_nw)) nw = a.anal_nw;
    int nlr = ntiles / nw;
    if (nlr > 6) { nw = 8; nlr = (ntiles + 7) / 8; }
#define ANAL_CASE(W, R)                                                                              \
    if (nw == W && nlr <= R) {                                                                       \
        if (a.nfields == 1) launch_anal_few<W, R, 1>(a, F, four_dist, Q, spec_dist, spec_ltop, s);   \
        else launch_anal_few<W, R, 2>(a, F, four_dist, Q, spec_dist, spec_ltop, s);                  \
        return;                                                                                      \
    }
    ANAL_CASE(1, 1) ANAL_CASE(1, 2) ANAL_CASE(1, 3) ANAL_CASE(1, 6)
    ANAL_CASE(2, 1) ANAL_CASE(2, 3) ANAL_CASE(2, 6)
    ANAL_CASE(3, 1) ANAL_CASE(3, 2) ANAL_CASE(3, 4) ANAL_CASE(3, 6)
    ANAL_CASE(4, 1) ANAL_CASE(4, 2) ANAL_CASE(4, 3) ANAL_CASE(4, 6)
    ANAL_CASE(5, 1) ANAL_CASE(5, 3) ANAL_CASE(5, 6)
    ANAL_CASE(6, 1) ANAL_CASE(6, 2) ANAL_CASE(6, 3) ANAL_CASE(6, 6)
    ANAL_CASE(7, 1) ANAL_CASE(7, 3) ANAL_CASE(7, 6)
    ANAL_CASE(8, 1) ANAL_CASE(8, 2) ANAL_CASE(8, 3) ANAL_CASE(8, 4) ANAL_CASE(8, 6)
    ANAL_CASE(9, 1) ANAL_CASE(10, 1) ANAL_CASE(11, 1) ANAL_CASE(12, 1)
#undef ANAL_CASE
    fprintf(stderr, "shtns_amd: no analysis kernel for nlat_2=%d\n", a.nlat_2);
}

// Block shape (tiles, column tiles, parts, halves) of the shared kernel for a number of latitude
// tiles (rounded up to a compiled one) and ctn column tiles of 4 fields.  Measured on FP64
// batches (analysis call with its FFT, us; the one-group kernel it replaced, other shapes):
//   lmax  127,  8 / 32 fields: (2,1,4) 22.5 / 30.2   [28.9 / 36.5; (2,2,2) 25.2 / 32.4]
//   lmax  255,  8 / 16 fields: (3,1,4) 36.6 / 46.1   [43.1 / 52.7; (3,2,2) 41.0 / 50.1]
//               32 fields:     (3,2,2) 69.0          [82.6; (3,1,4) 72.6, (3,4,2) 73.0]
//   lmax  340, 32 fields:      (4,2,4) 115           [(4,2,2) 120, (4,1,4) 123]
//   lmax  511,  8 / 16 fields: (6,2,4) 92 / 162      [100 / 170; (6,4,3) 121 / 170, (6,2,2) 104 / 183]
//               64 fields:     (6,2,4) 591           [(6,4,3) 650, (6,2,2) 653, (6,2,3) 945]
//   lmax  680,  8 / 16 fields: (8,2,4) 230, (8,4,2) 435   [- / 451; (8,1,4) 294 / 594]
//   lmax 1023,  4 / 8 / 16:    (12,1,4,3) 303, (12,2,6) 488, (12,4,3) 885   [310 / 504 / 990]
// Two blocks of eight waves per CU overlap one block's recurrence, loads and barriers with the
// other's contraction where their LDS allows ((6,2,4)); at 12 tiles the recurrence buffer
// leaves one block per CU, and more fields per block amortize those phases.  Six-wave blocks
// load two of the four SIMDs twice.  With few columns, four waves share an order (latency).
// Single precision: the recurrence outweighs the contraction, so 12 tiles take one wave each for up
// to four fields (one field, lmax=1023, longitude-contiguous: analysis call 221 -> 208 us); at 6
// tiles that gave nothing (one / four fields at lmax=511: 57.7 / 71.4, four waves 57.8 / 71.3).
// One and two tiles are split by half tiles, which sums in the order of the one- and two-field
// kernel: there a field's result does not depend on its batch.
template <int PREC>
void anal_launch_shared(const LegendreArgs &a, const double2 *F, long four_dist, double2 *Q, long spec_dist,
                        int spec_ltop, hipStream_t s) {
    const int ntiles = (a.nlat_2 + 63) / 64;
    const int ctn = (a.nfields + 3) / 4;
    // the tuner's choice: 1 for four fields per block, otherwise as many as the shapes below take
    static const int ncg_env = getenv("SHTNS_AMD_ANAL_NCG") ? atoi(getenv("SHTNS_AMD_ANAL_NCG")) : 0;
    const bool one = (a.anal_ncg ? a.anal_ncg : ncg_env) == 1;
    if (ntiles > 6 && ctn > 4 && (ctn % 4 == 1 || ctn % 4 == 2) && !one) {
        // shapes of 16 fields: the last one to eight fields in blocks of their own size (in the
        // 16-field blocks their waves would wait for nothing: 24 fields at lmax=850 1462 us)
        const int nf0 = (ctn & ~3) * 4;
        LegendreArgs a0 = a, a1 = a;
        a0.nfields = nf0;
        a1.nfields = a.nfields - nf0;
        anal_launch_shared<PREC>(a0, F, four_dist, Q, spec_dist, spec_ltop, s);
        anal_launch_shared<PREC>(a1, F + (size_t)nf0 * four_dist, four_dist, Q + (size_t)nf0 * spec_dist, spec_dist, spec_ltop, s);
        return;
    }
    // 12 tiles per launch and the rest in one of its own shape (13 tiles as 7 + 7 in 8-tile
    // blocks: lmax=1067, 4 fields 618 us, as 12 + 1 535; 3 fields 552, 480).  In order on the
    // stream: the later launches add to the first one's result.
    for (int tile0 = 0; tile0 < ntiles; tile0 += 12) {
        const int per = std::min(12, ntiles - tile0);
#define ANAL_SHARED(...) launch_anal_shared<__VA_ARGS__, PREC>(a, F, four_dist, Q, spec_dist, spec_ltop, s, tile0, per, tile0 > 0)
        if (per <= 1) { if (ctn >= 2 && !one) ANAL_SHARED(1, 2, 2, 1); else ANAL_SHARED(1, 1, 2, 1); }
        else if (per <= 2) ANAL_SHARED(2, 1, 4, 1);
        else if (per <= 3) { if (ctn > 4 && !one) ANAL_SHARED(3, 2, 2, 1); else ANAL_SHARED(3, 1, 4, 1); }
        else if (per <= 4) { if (ctn >= 4 && !one) ANAL_SHARED(4, 2, 4, 1); else ANAL_SHARED(4, 1, 4, 1); }
        else if (per <= 6) {
            if (ctn >= 2 && !one) ANAL_SHARED(6, 2, 4, 1);
            else if (per == 6) ANAL_SHARED(6, 1, 4, 1);
            else ANAL_SHARED(5, 1, 5, 1);
        } else if (per <= 8) {
            if (ctn >= 3 && !one) ANAL_SHARED(8, 4, 2, 1);
            else if (ctn >= 2 && !one) ANAL_SHARED(8, 2, 4, 1);
            else ANAL_SHARED(8, 1, 8, 1);
        } else {
            if (ctn >= 3 && !one) ANAL_SHARED(12, 4, 3, 1);
            else if (ctn >= 2 && !one) ANAL_SHARED(12, 2, 6, 1);
            else if (PREC > 0) ANAL_SHARED(12, 1, 12, 1);
            else ANAL_SHARED(12, 1, 4, 3);
        }
#undef ANAL_SHARED
    }
}

template <int PREC>
void anal_launch(const LegendreArgs &a, const double2 *F, long four_dist, double2 *Q, long spec_dist,
                 int spec_ltop, hipStream_t s) {
    if constexpr (PREC == 0) {
        if (a.nfields <= 2 && !synth_force16()) {
            anal_launch_few(a, F, four_dist, Q, spec_dist, spec_ltop, s);
            return;
        }
    }
    anal_launch_shared<PREC>(a, F, four_dist, Q, spec_dist, spec_ltop, s);
}

}  // namespace shtns_amd
