// oka_fp32.hip -- FP32 particle tracing for gfx950 (confined or unconfined
// velocity): one workgroup of up to 256 lanes per realization, taken
// from a queue, the last ones shared (next_realization).  The step,
// field and rasterizer are in oka_fp32_dev.h.  Results are not bit-identical
// to the FP64 path; the difference in capture probability is reported against
// the FP64-exact mode.
#include <math.h>

#include <type_traits>

#include "oka_fp32_dev.h"
#include "oka_internal.h"

namespace oka {
namespace {

using namespace fp32;

// At most 128 VGPRs, so that at least 4 waves share a SIMD: the tracer is
// bound by VALU issue, and with 3 waves the SIMDs idled about 12 % of the time
// on LDS and scalar waits.
//
// kPlaces: the wells' places come from a.wells32 (Field32Site).  Without it,
// where nothing outside the launch may hold them, they are records in LDS.
template <int kKind, bool kConfined, bool kPlaces>
__global__ void __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(4)))
k_trace_fp32(TraceArgs a)
{
    extern __shared__ float4 smem4[];
    using Field = typename std::conditional<kPlaces, Field32Site, Field32Lds>::type;
    // a record a well, or strengths, then (unconfined) the potential's, of 4
    // wells a float4
    const int nw4 = (a.nwells + 3) / 4;
    float *s_q = reinterpret_cast<float *>(smem4), *s_p = reinterpret_cast<float *>(smem4 + nw4);
    uint32_t *s_bm = reinterpret_cast<uint32_t *>(
        smem4 + (!kPlaces ? a.nwells : (kConfined ? 1 : 2) * nw4));
    using Bits = typename std::conditional<kKind == kBmTiled, TileBits, FlatBits>::type;
    __shared__ int s_next;
    __shared__ ShareLds s_share;
    __shared__ unsigned long long s_stat[kStatCount];
    __shared__ float s_reg[11];

    const int tid = threadIdx.x;
    const int P = a.npaths;
    Integ32 I;
    I.dur = a.duration;
    I.absdur = fabs(a.duration);
    I.sg = a.duration > 0.0 ? 1.0 : (a.duration < 0.0 ? -1.0 : (a.duration == 0.0 ? 0.0 : (double)NAN));
    I.tol = (float)a.tol;
    I.maxstep = (float)a.maxstep;
    I.cap = a.max_steps;
    const float umbra = (float)a.umbra;
    const float u2 = umbra * umbra;
    const float gdx = (float)a.gdx, gdy = (float)a.gdy;
    const float igdx = (float)(1.0 / a.gdx), igdy = (float)(1.0 / a.gdy);
    const float gx0 = (float)(a.gxmin - a.xo), gx1 = (float)(a.gxmax - a.xo);
    const float gy0 = (float)(a.gymin - a.yo), gy1 = (float)(a.gymax - a.yo);
    Bits bits;
    uint32_t *lds_tail = s_bm;
    if constexpr (kKind == kBmTiled) {
        bits = tile_bits(a, s_bm);
        tile_init(bits);
        lds_tail += tile_lds_words(a.ntiles, a.tile_slots);
    } else if constexpr (kKind == kBmLdsFlat) {
        bits = FlatBits{s_bm, a.gncols};
        lds_tail += a.rasterize ? a.nwords : 0;
    } else {
        bits = FlatBits{a.gbitmap + (int64_t)blockIdx.x * a.nwords, a.gncols};
    }
    unsigned int *s_win = nullptr;
    if (a.rasterize && a.wmarks) {
        s_win = lds_tail;
        for (int c = threadIdx.x; c < a.w_nr * a.w_nc; c += blockDim.x)
            s_win[c] = 0u;
    }

    for (int r = next_realization(a, -1, s_share); r < a.nreal;
         r = next_realization(a, r, s_share)) {
        int32_t *const shared = shared_counter(a, r);
        if (tid < kStatCount)
            s_stat[tid] = 0;
        const double bn = a.b[r] * a.n[r];
        // h = K b^2 / 2, the potential at which the head reaches the top of
        // the aquifer (model.py:344)
        const double h = kConfined ? 1.0 : 0.5 * a.K[r] * (a.b[r] * a.b[r]);
        for (int i = tid; i < a.nwells; i += blockDim.x) {
            const double qw = a.q[(int64_t)r * a.nwells + i];
            const float st = (float)(qw * kInv2Pi / bn);
            const float pt = kConfined ? 0.0f : (float)(qw * (kInv4Pi * kLn2) / h);
            if constexpr (kPlaces) {
                s_q[i] = st;
                if constexpr (!kConfined)
                    s_p[i] = pt;
            } else {
                smem4[i] = make_float4((float)(a.wells_xy[2 * i] - a.xo),
                                       (float)(a.wells_xy[2 * i + 1] - a.yo), st, pt);
            }
        }
        if (tid == 0) {
            const double *c = a.coef + 6 * (int64_t)r;
            s_reg[0] = (float)(2.0 * c[0] / bn);
            s_reg[1] = (float)(2.0 * c[1] / bn);
            s_reg[2] = (float)(c[2] / bn);
            s_reg[3] = (float)(c[3] / bn);
            s_reg[4] = (float)(c[4] / bn);
            for (int j = 0; j < 6; ++j)
                s_reg[5 + j] = (float)(c[j] / h);
            s_next = blockDim.x;
        }
        if constexpr (kKind != kBmTiled) {   // a tiled bitmap is left empty by its flush
            if (a.rasterize)
                for (int w = tid; w < a.nwords; w += blockDim.x)
                    bits.bm[w] = 0u;
        }
        __syncthreads();

        Field f;
        if constexpr (kPlaces) {
            f.xy = (ConstF32)a.wells32;
            f.q4 = smem4;
            f.p4 = smem4 + nw4;
        } else {
            f.w = smem4;
        }
        f.nw = a.nwells;
        f.a2 = s_reg[0];
        f.b2 = s_reg[1];
        f.c = s_reg[2];
        f.d = s_reg[3];
        f.e = s_reg[4];
        if constexpr (!kConfined) {
            f.pa = s_reg[5];
            f.pb = s_reg[6];
            f.pc = s_reg[7];
            f.pd = s_reg[8];
            f.pe = s_reg[9];
            f.pf = s_reg[10];
        }
        // per-trace statistics go to LDS when the trace ends (few registers)
        unsigned long long n_cand = 0;   // candidate nodes of the lane's trace

        Trace32 s;
        Epoch32 ep;
        int p = shared ? claim_one(shared) : tid;
        bool have = p < P;
        bool live = false, fresh = false;
        bool a_done = false;   // the disk around the trace's current point is marked
        bool dry = false;      // an evaluation of the trace raised AquiferError
        for (;;) {
            bool ended = false;
            const int64_t k = (int64_t)r * P + p;
            if (!live) {
                if (!have)
                    break;
                if (a.rasterize)
                    ep = find_epoch32(a, k);
                open32(s, I, (float)(a.start_xy[2 * p] - a.xo),
                       (float)(a.start_xy[2 * p + 1] - a.yo));
                live = fresh = true;
                a_done = false;
                dry = false;
            }
            // one field evaluation for every lane: k1 of a fresh trace, else
            // the first stage of an attempted step
            double dtd;
            float dt, px, py, kx, ky;
            first_point(I, s, fresh, dtd, dt, px, py);
            feval32<kConfined>(f, px, py, kx, ky, dry);
            if (fresh) {
                fresh = false;
                if (dry) {   // k1 raised: the trace is its start vertex (capturezone.py:218, 249)
                    s.status = OKA_TRACE_TRUNCATED;
                    live = false;
                    ended = true;
                } else if (!take_k1(I, s, kx, ky)) {
                    live = false;
                    ended = true;
                }
            } else {
                float ox, oy;
                const int res = finish32(LaneEval<kConfined, Field>{f, dry}, I, s, dtd, dt, kx, ky,
                                         ox, oy);
                // a stage raised: the step is not accepted and the trace ends
                if (!kConfined && dry)
                    s.status = OKA_TRACE_TRUNCATED;
                if ((res & 1) && a.rasterize)
                    n_cand += (unsigned long long)raster32(bits, ep, gdx, gdy, igdx, igdy, umbra,
                                                           u2, ox, oy, s.x, s.y, !a_done, a_done);
                if (res & 2) {
                    live = false;
                    ended = true;
                }
            }
            if (ended) {
                atomicAdd(&s_stat[kStatAttempted], (unsigned long long)s.att);
                atomicAdd(&s_stat[kStatAccepted], (unsigned long long)s.acc);
                atomicAdd(&s_stat[kStatStatus0 + (s.status & 3)], 1ull);
                atomicAdd(&s_stat[kStatCandidates], n_cand);
                n_cand = 0;
                if (!(s.bx0 > gx0 && s.bx1 < gx1 && s.by0 > gy0 && s.by1 < gy1))
                    atomicAdd(&s_stat[kStatEscaped], 1ull);
                if (a.bbox) {
                    a.bbox[4 * k] = a.xo + (double)s.bx0;
                    a.bbox[4 * k + 1] = a.xo + (double)s.bx1;
                    a.bbox[4 * k + 2] = a.yo + (double)s.by0;
                    a.bbox[4 * k + 3] = a.yo + (double)s.by1;
                }
                if (a.trace_status)
                    a.trace_status[k] = s.status;
                if (a.trace_steps)
                    a.trace_steps[k] = s.att;
                p = shared ? claim_one(shared) : atomicAdd(&s_next, 1);
                have = p < P;
            }
        }
        __syncthreads();
        if (a.rasterize) {
            uint32_t *const merged = merged_bits(a, r, traced(s_stat));
            if constexpr (kKind == kBmTiled)
                atomicAdd(&s_stat[kStatVisited], flush_tiles(a, bits, s_win, merged));
            else
                atomicAdd(&s_stat[kStatVisited], flush_bitmap(a, bits.bm, s_win, merged));
        }
        __syncthreads();
        if (s_win) {
            store_window(a, r, s_win);
            __syncthreads();
        }
        if (tid < kStatCount && a.stats)
            atomicAdd(&a.stats[tid], s_stat[tid]);
        __syncthreads();
    }
}

// The wells' places relative to the origin, as the FP32 tracer adds them up.
__global__ void __launch_bounds__(256) k_site_wells32(const double *wells_xy, int nwells, double xo,
                                                      double yo, float2 *out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nwells)
        out[i] = make_float2((float)(wells_xy[2 * i] - xo), (float)(wells_xy[2 * i + 1] - yo));
}

// The FP32 tracers' segment rasterizer over the segments of one polyline (one
// per lane), in coordinates relative to the grid's centre node.
__global__ void __launch_bounds__(256) k_raster_fp32(RasterArgs a)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.nseg)
        return;
    const double ox = a.xmin + (double)(a.ncols / 2) * a.dx;
    const double oy = a.ymin + (double)(a.nrows / 2) * a.dy;
    const Epoch32 e{(float)(a.xmin - ox), (float)(a.ymin - oy), a.nrows, a.ncols, 0, 0};
    FlatBits bits{a.bitmap, a.ncols};
    const float umbra = (float)a.umbra;
    bool covered;
    raster32(bits, e, (float)a.dx, (float)a.dy, (float)(1.0 / a.dx), (float)(1.0 / a.dy), umbra,
             umbra * umbra, (float)(a.xy[2 * i] - ox), (float)(a.xy[2 * i + 1] - oy),
             (float)(a.xy[2 * i + 2] - ox), (float)(a.xy[2 * i + 3] - oy), true, covered);
}

}  // namespace

size_t trace_fp32_wells_lds(int nwells, bool confined, bool places)
{
    return sizeof(float4) *
           (!places ? (size_t)nwells : (size_t)((nwells + 3) / 4) * (confined ? 1 : 2));
}

hipError_t launch_site_wells32(const TraceArgs &a, float2 *out, hipStream_t s)
{
    if (a.nwells <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_site_wells32, dim3((unsigned)((a.nwells + 255) / 256)), dim3(256), 0, s,
                       a.wells_xy, a.nwells, a.xo, a.yo, out);
    return hipGetLastError();
}

namespace {

template <int kKind>
hipError_t launch_kind(const TraceArgs &a, int grid_blocks, size_t lds, hipStream_t s)
{
    const dim3 grid(grid_blocks), block(trace_block(a.npaths));
    if (a.confined && a.wells32)
        hipLaunchKernelGGL((k_trace_fp32<kKind, true, true>), grid, block, lds, s, a);
    else if (a.confined)
        hipLaunchKernelGGL((k_trace_fp32<kKind, true, false>), grid, block, lds, s, a);
    else if (a.wells32)
        hipLaunchKernelGGL((k_trace_fp32<kKind, false, true>), grid, block, lds, s, a);
    else
        hipLaunchKernelGGL((k_trace_fp32<kKind, false, false>), grid, block, lds, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_trace_fp32(const TraceArgs &a, int grid_blocks, int kind, hipStream_t s)
{
    size_t lds = trace_fp32_wells_lds(a.nwells, a.confined, a.wells32 != nullptr) +
                 (a.wmarks ? (size_t)a.w_nr * a.w_nc * 4 : 0);
    if (!a.rasterize || kind == kBmLdsFlat)
        return launch_kind<kBmLdsFlat>(a, grid_blocks,
                                       lds + (a.rasterize ? (size_t)a.nwords * 4 : 0), s);
    if (kind == kBmTiled)
        return launch_kind<kBmTiled>(
            a, grid_blocks, lds + (size_t)tile_lds_words(a.ntiles, a.tile_slots) * 4, s);
    return launch_kind<kBmHbmFlat>(a, grid_blocks, lds, s);
}

hipError_t launch_raster_fp32(const RasterArgs &a, hipStream_t s)
{
    const int64_t blocks = (a.nseg + 255) / 256;
    hipLaunchKernelGGL(k_raster_fp32, dim3((unsigned)blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace oka
