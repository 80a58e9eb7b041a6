// oka_fit.hip -- batched FP64 regional-flow fit and multivariate-normal draw.
//
// Per realization r: the weighted least-squares rows of
// Model.construct_fit (oneka/model.py:540-567) with conductivity K[r],
// thickness b[r] and discharges q[r, :]; the fit of compute_fit
// (model.py:598-604) solved through column-equilibrated normal equations, a
// 6x6 Cholesky factorization and one step of iterative refinement; the
// covariance inv(WA^T WA); and the draw coef = ev + L z of
// oneka/stochastic.py:239-241 with L the lower Cholesky factor of the
// covariance.  The realization-invariant part of the wells' potential at the
// observations, log(r^2) per (well, observation), is computed once per call by
// k_fit_logs.
//
// Layout: a workgroup of 8 waves takes 64 realizations, one per lane.  The
// waves share the realizations' observations, then their sums:
//   1. potentials: each wave sums the wells (in index order) at groups of 8
//      observations; the discharges and the logarithms pass through LDS 32
//      wells at a time (a row of q is read once and contiguously, a logarithm
//      once a workgroup, then broadcast);
//   2. normal equations: the waves form the rows of 8 observations in LDS,
//      then each adds them (in index order) to its share of the 27 sums;
//   3. wave 0 factors and solves;
//   4. refinement: rows and residuals of 8 observations, then one wave per
//      component adds them;
//   5. wave 0 refines, inverts, draws and writes.
// Every sum runs over the same terms in the same order whatever the split, so
// the results are those of one lane doing all of it.
//
// Bound: step 1's broadcast LDS reads, 4 of 16 bytes per 24 FP64 instructions
// (16 cycles of the CU's LDS each, so 25 groups of observations take 1,600
// cycles a well where their FP64 issue takes 600); the potentials take 512
// bytes of LDS an observation, so one workgroup fills a CU from about 90
// observations on, and the solve's chains are then hardly overlapped.  10^5
// realizations of 200 wells and 200 observations: 6.48 ms with one lane per
// realization doing everything (each wave's loads of q in 64 rows, the
// potentials summed twice), 1.27 ms so, of which the solve takes about 0.5.
#include <math.h>

#include <algorithm>

#include "oka_fp64_dev.h"
#include "oka_internal.h"
#include "oka_math.h"

#pragma clang fp contract(off)

namespace oka {
namespace {

constexpr double kC4Pi = 0.07957747154594767;  // model.py:264

// log(r^2) of (well w, observation i) at w * fit_obs_stride + i, padded with 0.
__device__ __forceinline__ void fit_log(const FitArgs &a, int64_t t, double *logr2)
{
    const int np = fit_obs_stride(a.nobs);
    const int i = (int)(t % np), w = (int)(t / np);
    double v = 0.0;
    if (i < a.nobs) {
        const double dx = a.obs[4 * i] - a.wells_xy[2 * w];
        const double dy = a.obs[4 * i + 1] - a.wells_xy[2 * w + 1];
        v = log_rn(dx * dx + dy * dy);
    }
    logr2[t] = v;
}

__global__ void __launch_bounds__(256) k_fit_logs(FitArgs a, double *logr2)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < fit_logs_count(a.nobs, a.nwells))
        fit_log(a, t, logr2);
}

constexpr int kLanes = 64;                     // realizations per workgroup
constexpr int kWaves = 8;
constexpr int kFitBlock = kLanes * kWaves;
constexpr int kObsBlock = 8;                   // observations per wave and group
constexpr int kObsChunk = 240;                 // observations in LDS at once (30 groups)
constexpr int kWellTile = 32;                  // wells in LDS at once
constexpr int kTileLd = kLanes + 1;
constexpr int kSums = 27;                      // 21 of the normal matrix, 6 of its right side
constexpr int kRow = 7;                        // a row and its target
// doubles of the second LDS region: a tile of discharges, then rows, then sums
constexpr int kTileDoubles = kRow * kWaves * kLanes;
static_assert(kTileDoubles >= kWellTile * kTileLd && kTileDoubles >= kSums * kLanes, "they fit");
static_assert(kWellTile * kLanes % kFitBlock == 0, "whole discharges per lane and tile");
// the logarithms of a tile go where the potentials will: 32 wells x (the
// observations rounded up to 8) fit in 64 x the observations from 8 on
constexpr int kMinLogObs = 8;

// A workgroup's LDS: observations (x, y, z, its standard deviation) of the
// chunk, the tile, the potentials.
struct FitLds {
    double4 *obs;
    double *tile, *pw;
};

// The wells' potential (model.py:258-264) of the workgroup's realizations at
// observations c0 .. c0 + min(kObsChunk, nobs - c0) - 1, to pw[(i - c0) * 64 +
// lane].  Wave v sums groups v, v + 8, ... of 8 observations (kGroups of them,
// which may differ between waves), each over the wells in index order.  Every
// lane calls it; it ends with a barrier.
template <int kGroups>
__device__ __forceinline__ void well_potentials(const FitArgs &a, int64_t r0, int c0,
                                                const FitLds &S)
{
    const int tid = threadIdx.x, lane = tid & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kLanes);
    const int np = fit_obs_stride(a.nobs);
    const int nc = fit_obs_stride(min(a.nobs - c0, kObsChunk));   // a tile's row of logarithms
    const int64_t last = a.nreal - 1;
    double acc[kGroups > 0 ? kGroups : 1][kObsBlock];
#pragma unroll
    for (int g = 0; g < kGroups; ++g)
#pragma unroll
        for (int j = 0; j < kObsBlock; ++j)
            acc[g][j] = 0.0;
    double *tile = S.tile, *pw = S.pw, *logs = S.pw;
    for (int i = tid; i < min(a.nobs - c0, kObsChunk); i += kFitBlock) {
        const double *o = a.obs + 4 * (int64_t)(c0 + i);
        S.obs[i] = make_double4(o[0], o[1], o[2], o[3]);
    }
    constexpr int kPer = kWellTile * kLanes / kFitBlock;
    double next[kPer];
    // lane tid of the workgroup moves well w0 + tid % 32 of realizations
    // tid / 32 + 16 k
    auto fetch = [&](int w0) {
        const int w = w0 + tid % kWellTile;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int64_t r = r0 + tid / kWellTile + k * (kFitBlock / kWellTile);
            next[k] = w < a.nwells ? a.q[(r < last ? r : last) * a.nwells + w] : 0.0;
        }
    };
    const bool rows = a.q_well_stride == 0;
    const double *qw = a.q + (r0 + lane < last ? r0 + lane : last);   // well-major
    if (rows)
        fetch(0);
    for (int w0 = 0; w0 < a.nwells; w0 += kWellTile) {
        const int n = min(kWellTile, a.nwells - w0);
        __syncthreads();   // the previous tile has been read
        if (rows) {
#pragma unroll
            for (int k = 0; k < kPer; ++k)
                tile[(tid % kWellTile) * kTileLd + tid / kWellTile + k * (kFitBlock / kWellTile)] =
                    next[k];
        }
        const double2 *src = reinterpret_cast<const double2 *>(a.logr2 + (int64_t)w0 * np + c0);
        for (int k = tid; k < n * (nc / 2); k += kFitBlock) {
            const int w = k / (nc / 2), i = k - w * (nc / 2);
            reinterpret_cast<double2 *>(logs)[k] = src[(int64_t)w * (np / 2) + i];
        }
        __syncthreads();
        if (rows && w0 + kWellTile < a.nwells)
            fetch(w0 + kWellTile);
        if constexpr (kGroups > 0) {
#pragma unroll 2
            for (int w = 0; w < n; ++w) {
                const double q = rows ? tile[w * kTileLd + lane] : qw[(w0 + w) * a.q_well_stride];
                const double *L = logs + w * nc + wave * kObsBlock;
#pragma unroll
                for (int g = 0; g < kGroups; ++g)
#pragma unroll
                    for (int j = 0; j < kObsBlock; ++j)
                        acc[g][j] = acc[g][j] + (q * L[g * kWaves * kObsBlock + j]) * kC4Pi;
            }
        }
    }
    __syncthreads();   // the last tile's logarithms have been read
#pragma unroll
    for (int g = 0; g < kGroups; ++g)
#pragma unroll
        for (int j = 0; j < kObsBlock; ++j) {
            const int i = (wave + g * kWaves) * kObsBlock + j;
            if (c0 + i < a.nobs)
                pw[i * kLanes + lane] = acc[g][j];
        }
    __syncthreads();
}

__device__ __forceinline__ void chunk_potentials(const FitArgs &a, int64_t r0, int c0,
                                                 const FitLds &S)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int groups = (min(a.nobs - c0, kObsChunk) + kObsBlock - 1) / kObsBlock;
    switch ((groups - wave + kWaves - 1) / kWaves) {   // this wave's
    case 0: well_potentials<0>(a, r0, c0, S); break;
    case 1: well_potentials<1>(a, r0, c0, S); break;
    case 2: well_potentials<2>(a, r0, c0, S); break;
    case 3: well_potentials<3>(a, r0, c0, S); break;
    default: well_potentials<4>(a, r0, c0, S); break;
    }
}

// The target and its standard deviation at observation o (model.py:545-558).
// False where the reference raises RangeError.
__device__ __forceinline__ bool fit_target(const FitArgs &a, const double4 &o, double K, double b,
                                           double &pot_ev, double &pot_std)
{
    const double z_ev = o.z, z_std = o.w;
    const double head = z_ev - a.base;
    if (head >= b) {
        pot_ev = (K * b) * (head - 0.5 * b);
        pot_std = (K * b) * z_std;
    } else {
        pot_ev = (0.5 * K) * (head * head + z_std * z_std);
        pot_std = (K * head) * z_std;
    }
    return head >= b || head > 0.0;
}

// Whether x / d needs no scaling in quot_plain, for any number of numerators x.
__device__ __forceinline__ bool plain_numerator(double x)
{
    const double v = fabs(x);
    return v == 0.0 || (v >= 0x1p-300 && v <= 0x1p300);
}

__device__ __forceinline__ bool plain_divisor(double d)
{
    const double v = fabs(d);
    return v >= 0x1p-200 && v <= 0x1p200;
}

// One weighted row (model.py:559-565) of observation o, given the wells'
// potential pw there: IEEE quotients, by the short sequence where the whole
// wave's operands need no scaling.
__device__ __forceinline__ void fit_row(const FitArgs &a, const double4 &o, double pot_ev,
                                        double pot_std, double pw, double *row, double &wb)
{
    const double dx = o.x - a.xo, dy = o.y - a.yo;
    const double x[6] = {dx * dx, dy * dy, dx * dy, dx, dy, 1.0};
    const double y = pot_ev - pw;
    bool ok = plain_divisor(pot_std) && plain_numerator(y);
#pragma unroll
    for (int j = 0; j < 5; ++j)
        ok = ok && plain_numerator(x[j]);
    if (__ballot(!ok) == 0ull) {
        const double r = fp64::recip_plain(pot_std);
#pragma unroll
        for (int j = 0; j < 6; ++j)
            row[j] = fp64::quot_plain(x[j], pot_std, r);
        wb = fp64::quot_plain(y, pot_std, r);
    } else {
#pragma unroll
        for (int j = 0; j < 6; ++j)
            row[j] = x[j] / pot_std;
        wb = y / pot_std;
    }
}

// The sums of one wave: the products of columns kA0 .. kA0 + kNA - 1 with
// kB0 .. kB0 + kNB - 1 of a row and its target (column 6), on and below the
// diagonal.  The blocks of 2 x 2 (3 x 1 of the target) need 26 values of each
// row between the waves, whose LDS reads bound this step.
template <int kWave>
struct NormalSums {
    static constexpr int kA0 = kWave == 0 ? 0 : kWave == 1 ? 2 : kWave == 2 ? 4 : kWave == 3 ? 2
                               : kWave < 6 ? 4 : 6;
    static constexpr int kB0 = kWave == 1 || kWave == 5 ? 2 : kWave == 2 ? 4 : kWave == 7 ? 3 : 0;
    static constexpr int kNA = kWave < 6 ? 2 : 1, kNB = kWave < 6 ? 2 : 3;
    double v[kNA][kNB];
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int i = 0; i < kNA; ++i)
#pragma unroll
            for (int k = 0; k < kNB; ++k)
                v[i][k] = 0.0;
    }
    // one row, its values 64 apart
    __device__ __forceinline__ void add(const double *row)
    {
        double x[kNA], y[kNB];
#pragma unroll
        for (int i = 0; i < kNA; ++i)
            x[i] = row[(kA0 + i) * kLanes];
#pragma unroll
        for (int k = 0; k < kNB; ++k)
            y[k] = row[(kB0 + k) * kLanes];
#pragma unroll
        for (int i = 0; i < kNA; ++i)
#pragma unroll
            for (int k = 0; k < kNB; ++k)
                if (kB0 + k <= kA0 + i)
                    v[i][k] = v[i][k] + x[i] * y[k];
    }
    // (j, k) of the normal matrix to row j (j + 1) / 2 + k, its right side after it
    __device__ __forceinline__ void store(double *sums, int lane) const
    {
#pragma unroll
        for (int i = 0; i < kNA; ++i)
#pragma unroll
            for (int k = 0; k < kNB; ++k) {
                const int j = kA0 + i, c = kB0 + k;
                if (c <= j)
                    sums[(j < 6 ? j * (j + 1) / 2 + c : 21 + c) * kLanes + lane] = v[i][k];
            }
    }
};

// The wave's sums over all observations, to S.tile[t * 64 + lane].  S holds the
// first chunk when it is called, and the last when it returns.  Returns whether the wave's observations were in range.
template <int kWave>
__device__ __forceinline__ bool normal_sums(const FitArgs &a, int64_t r0, double K, double b,
                                            const FitLds &S)
{
    double *tile = S.tile;
    const int lane = threadIdx.x & (kLanes - 1);
    NormalSums<kWave> s;
    s.clear();
    bool good = true;
    for (int c0 = 0; c0 < a.nobs; c0 += kObsChunk) {
        if (c0 > 0)
            chunk_potentials(a, r0, c0, S);
        const int n = min(kObsChunk, a.nobs - c0);
        for (int i0 = 0; i0 < n; i0 += kWaves) {
            const int i = i0 + kWave;
            if (i < n) {
                double pot_ev, pot_std, row[6], wb;
                const double4 ob = S.obs[i];
                good = fit_target(a, ob, K, b, pot_ev, pot_std) && good;
                fit_row(a, ob, pot_ev, pot_std, S.pw[i * kLanes + lane], row, wb);
                double *out = tile + kWave * kRow * kLanes + lane;
#pragma unroll
                for (int j = 0; j < 6; ++j)
                    out[j * kLanes] = row[j];
                out[6 * kLanes] = wb;
            }
            __syncthreads();
            const double *in = tile + lane;
            if (i0 + kWaves <= n) {
#pragma unroll
                for (int o = 0; o < kWaves; ++o)
                    s.add(in + o * kRow * kLanes);
            } else {
                for (int o = 0; o < n - i0; ++o)
                    s.add(in + o * kRow * kLanes);
            }
            __syncthreads();
        }
    }
    s.store(tile, lane);
    return good;
}

// Lower Cholesky factor of a symmetric 6x6 (row-major, lower part read).
__device__ __forceinline__ bool chol6(const double *A, double *L)
{
#pragma unroll
    for (int t = 0; t < 36; ++t)
        L[t] = 0.0;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        double d = A[j * 6 + j];
#pragma unroll
        for (int k = 0; k < j; ++k)
            d = d - L[j * 6 + k] * L[j * 6 + k];
        if (!(d > 0.0))
            return false;
        const double ljj = sqrt(d);
        L[j * 6 + j] = ljj;
#pragma unroll
        for (int i = j + 1; i < 6; ++i) {
            double v = A[i * 6 + j];
#pragma unroll
            for (int k = 0; k < j; ++k)
                v = v - L[i * 6 + k] * L[j * 6 + k];
            L[i * 6 + j] = v / ljj;
        }
    }
    return true;
}

// out = S (L L^T)^{-1} S g with S = diag(s).
__device__ __forceinline__ void chol6_solve(const double *L, const double *s, const double *g,
                                            double *out)
{
    double w[6], y[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        double v = s[j] * g[j];
#pragma unroll
        for (int k = 0; k < j; ++k)
            v = v - L[j * 6 + k] * w[k];
        w[j] = v / L[j * 6 + j];
    }
#pragma unroll
    for (int j = 5; j >= 0; --j) {
        double v = w[j];
#pragma unroll
        for (int k = j + 1; k < 6; ++k)
            v = v - L[k * 6 + j] * y[k];
        y[j] = v / L[j * 6 + j];
    }
#pragma unroll
    for (int j = 0; j < 6; ++j)
        out[j] = s[j] * y[j];
}

// Fit and MVN draw of realizations r0 .. r0 + 63 of the site `a`.
__device__ __forceinline__ void fit_block(const FitArgs &a, int64_t r0, double *lds)
{
    __shared__ int s_bad[kLanes];   // lanes with an observation out of range
    const int tid = threadIdx.x, lane = tid & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kLanes);
    const int nc = min(max(a.nobs, kMinLogObs), kObsChunk);
    FitLds S;
    S.obs = reinterpret_cast<double4 *>(lds);
    S.tile = lds + 4 * nc;
    S.pw = S.tile + kTileDoubles;
    double *tile = S.tile;
    const bool have = r0 + lane < a.nreal;
    const int64_t r = have ? r0 + lane : a.nreal - 1;
    const double K = a.K[r], b = a.b[r];
    if (wave == 0)
        s_bad[lane] = 0;
    chunk_potentials(a, r0, 0, S);
    bool good = true;
    switch (wave) {
    case 0: good = normal_sums<0>(a, r0, K, b, S); break;
    case 1: good = normal_sums<1>(a, r0, K, b, S); break;
    case 2: good = normal_sums<2>(a, r0, K, b, S); break;
    case 3: good = normal_sums<3>(a, r0, K, b, S); break;
    case 4: good = normal_sums<4>(a, r0, K, b, S); break;
    case 5: good = normal_sums<5>(a, r0, K, b, S); break;
    case 6: good = normal_sums<6>(a, r0, K, b, S); break;
    default: good = normal_sums<7>(a, r0, K, b, S); break;
    }
    if (!good)
        atomicOr(&s_bad[lane], 1);
    __syncthreads();
    int st = s_bad[lane] ? OKA_ERR_RANGE : 0;
    double ev[6], L[36], s[6];
    if (wave == 0) {
        double N[36], rhs[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
#pragma unroll
            for (int k = 0; k <= j; ++k)
                N[j * 6 + k] = tile[(j * (j + 1) / 2 + k) * kLanes + lane];
            rhs[j] = tile[(21 + j) * kLanes + lane];
        }
        if (st == 0) {
#pragma unroll
            for (int j = 0; j < 6; ++j)
                s[j] = 1.0 / sqrt(N[j * 6 + j]);
            double Ns[36];
#pragma unroll
            for (int j = 0; j < 6; ++j)
#pragma unroll
                for (int k = 0; k < 6; ++k)
                    Ns[j * 6 + k] = k <= j ? (s[j] * N[j * 6 + k]) * s[k] : 0.0;
            if (!chol6(Ns, L))
                st = OKA_ERR_LINALG;
        }
        if (st == 0)
            chol6_solve(L, s, rhs, ev);
        // only this wave reads the sums: the estimate takes their place
#pragma unroll
        for (int j = 0; j < 6; ++j)
            tile[j * kLanes + lane] = st == 0 ? ev[j] : 0.0;
    }
    __syncthreads();
    double e[6], g = 0.0;   // the estimate; component `wave` of row . residual (waves 0 to 5)
#pragma unroll
    for (int j = 0; j < 6; ++j)
        e[j] = tile[j * kLanes + lane];
    __syncthreads();
    for (int c0 = 0; c0 < a.nobs; c0 += kObsChunk) {
        if (a.nobs > kObsChunk)
            chunk_potentials(a, r0, c0, S);
        const int n = min(kObsChunk, a.nobs - c0);
        for (int i0 = 0; i0 < n; i0 += kWaves) {
            const int i = i0 + wave;
            if (i < n) {
                double pot_ev, pot_std, row[6], res;
                const double4 ob = S.obs[i];
                fit_target(a, ob, K, b, pot_ev, pot_std);
                fit_row(a, ob, pot_ev, pot_std, S.pw[i * kLanes + lane], row, res);
#pragma unroll
                for (int j = 0; j < 6; ++j)
                    res = res - row[j] * e[j];
                double *out = tile + wave * kRow * kLanes + lane;
#pragma unroll
                for (int j = 0; j < 6; ++j)
                    out[j * kLanes] = row[j];
                out[6 * kLanes] = res;
            }
            __syncthreads();
            if (wave < 6) {
                const double *in = tile + wave * kLanes + lane, *rs = tile + 6 * kLanes + lane;
                const int m = min(kWaves, n - i0);
                for (int o = 0; o < m; ++o)
                    g = g + in[o * kRow * kLanes] * rs[o * kRow * kLanes];
            }
            __syncthreads();
        }
    }
    if (wave < 6)
        tile[wave * kLanes + lane] = g;
    __syncthreads();
    if (wave != 0 || !have)
        return;
    if (st == 0) {
        double gs[6], d[6];
#pragma unroll
        for (int j = 0; j < 6; ++j)
            gs[j] = tile[j * kLanes + lane];
        chol6_solve(L, s, gs, d);
#pragma unroll
        for (int j = 0; j < 6; ++j)
            ev[j] = ev[j] + d[j];
    }
    double cov[36];
    if (st == 0) {
        double Li[36];
#pragma unroll
        for (int t = 0; t < 36; ++t)
            Li[t] = 0.0;
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            Li[j * 6 + j] = 1.0 / L[j * 6 + j];
#pragma unroll
            for (int i = j + 1; i < 6; ++i) {
                double v = 0.0;
#pragma unroll
                for (int k = j; k < i; ++k)
                    v = v - L[i * 6 + k] * Li[k * 6 + j];
                Li[i * 6 + j] = v / L[i * 6 + i];
            }
        }
#pragma unroll
        for (int j = 0; j < 6; ++j) {
#pragma unroll
            for (int k = 0; k <= j; ++k) {
                double v = 0.0;
#pragma unroll
                for (int i = j; i < 6; ++i)
                    v = v + Li[i * 6 + j] * Li[i * 6 + k];
                const double c = (s[j] * v) * s[k];
                cov[j * 6 + k] = c;
                cov[k * 6 + j] = c;
            }
        }
    }
    double coef[6];
    if (st == 0) {
        if (a.z) {
            double Lc[36];
            if (!chol6(cov, Lc)) {
                st = OKA_ERR_LINALG;
            } else {
                const double *z = a.z + 6 * (int64_t)r;
#pragma unroll
                for (int j = 0; j < 6; ++j) {
                    double acc = 0.0;
#pragma unroll
                    for (int k = 0; k <= j; ++k)
                        acc = acc + Lc[j * 6 + k] * z[k];
                    coef[j] = ev[j] + acc;
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < 6; ++j)
                coef[j] = ev[j];
        }
    }
    if (st != 0) {
#pragma unroll
        for (int j = 0; j < 6; ++j)
            ev[j] = coef[j] = (double)NAN;
#pragma unroll
        for (int t = 0; t < 36; ++t)
            cov[t] = (double)NAN;
    }
    if (a.ev)
#pragma unroll
        for (int j = 0; j < 6; ++j)
            a.ev[6 * (int64_t)r + j] = ev[j];
    if (a.cov)
#pragma unroll
        for (int t = 0; t < 36; ++t)
            a.cov[36 * (int64_t)r + t] = cov[t];
    if (a.coef)
#pragma unroll
        for (int j = 0; j < 6; ++j)
            a.coef[6 * (int64_t)r + j] = coef[j];
    if (a.status)
        a.status[r] = st;
}

// kTwo holds the kernel to 128 VGPRs, so that two workgroups share a CU.
template <bool kTwo>
__global__ void __launch_bounds__(kFitBlock) __attribute__((amdgpu_waves_per_eu(kTwo ? 4 : 2)))
k_fit_draw(FitArgs a)
{
    extern __shared__ double fit_lds[];
    fit_block(a, (int64_t)blockIdx.x * kLanes, fit_lds);
}

// Site of work item t of a table whose item counts have prefix sums `first`.
__device__ __forceinline__ int table_site(const int64_t *first, int nsites, int64_t t)
{
    int lo = 0, hi = nsites - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= t)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// log(r^2) of every (well, observation) pair of every site of a table.
__global__ void __launch_bounds__(256) k_fit_logs_multi(const FitArgs *sites, int nsites,
                                                        const int64_t *first, int64_t total)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total)
        return;
    const int site = table_site(first, nsites, t);
    const FitArgs &a = sites[site];
    fit_log(a, t - first[site], (double *)a.logr2);
}

// Fit and MVN draw of every realization of every site of a table, 64
// realizations of one site per workgroup (first: prefix sums of fit_blocks).
template <bool kTwo>
__global__ void __launch_bounds__(kFitBlock) __attribute__((amdgpu_waves_per_eu(kTwo ? 4 : 2)))
k_fit_draw_multi(const FitArgs *sites, int nsites, const int64_t *first)
{
    extern __shared__ double fit_lds[];
    const int site = table_site(first, nsites, blockIdx.x);
    const FitArgs a = sites[site];
    fit_block(a, (blockIdx.x - first[site]) * kLanes, fit_lds);
}

// LDS of a workgroup whose sites have at most nobs observations.
size_t fit_lds_bytes(int nobs)
{
    return sizeof(double) *
           (kTileDoubles + (size_t)std::min(std::max(nobs, kMinLogObs), kObsChunk) * (kLanes + 4));
}

// Two workgroups per CU where their LDS fits one (up to about 90
// observations) and there are enough of them to share CUs: 10^5 realizations
// of 200 wells and 64 observations 0.40 against 0.49 ms.  Alone on its CU a
// workgroup is faster without the register limit, whose spills lengthen the
// solve: 200 observations 1.27 against 1.56 ms, 100 realizations of 25 wells
// and 40 observations 32 against 37 us.
bool fit_two(int nobs, int64_t blocks)
{
    int dev = 0, num_cu = 0, lds = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&num_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) !=
            hipSuccess)
        return false;
    return blocks > num_cu && 2 * (fit_lds_bytes(nobs) + 1024) <= (size_t)lds;
}

}  // namespace

int64_t fit_blocks(int64_t nreal) { return (nreal + kLanes - 1) / kLanes; }

hipError_t launch_fit_logs(const FitArgs &a, double *logr2, hipStream_t s)
{
    const int64_t n = fit_logs_count(a.nobs, a.nwells);
    if (n == 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_fit_logs, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, logr2);
    return hipGetLastError();
}

hipError_t launch_fit_logs_multi(const FitArgs *sites, int nsites, const int64_t *first,
                                int64_t total, hipStream_t s)
{
    if (total <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_fit_logs_multi, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                       sites, nsites, first, total);
    return hipGetLastError();
}

hipError_t launch_fit_draw_multi(const FitArgs *sites, int nsites, const int64_t *first,
                                int64_t blocks, int max_nobs, hipStream_t s)
{
    if (blocks <= 0)
        return hipSuccess;
    if (fit_two(max_nobs, blocks))
        hipLaunchKernelGGL(k_fit_draw_multi<true>, dim3((unsigned)blocks), dim3(kFitBlock),
                           fit_lds_bytes(max_nobs), s, sites, nsites, first);
    else
        hipLaunchKernelGGL(k_fit_draw_multi<false>, dim3((unsigned)blocks), dim3(kFitBlock),
                           fit_lds_bytes(max_nobs), s, sites, nsites, first);
    return hipGetLastError();
}

hipError_t launch_fit_draw(const FitArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)fit_blocks(a.nreal)), block(kFitBlock);
    if (fit_two(a.nobs, grid.x))
        hipLaunchKernelGGL(k_fit_draw<true>, grid, block, fit_lds_bytes(a.nobs), s, a);
    else
        hipLaunchKernelGGL(k_fit_draw<false>, grid, block, fit_lds_bytes(a.nobs), s, a);
    return hipGetLastError();
}

}  // namespace oka
