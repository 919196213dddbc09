// Per-curve data preparation and point bucketing.
//
// One workgroup per curve:
//   phase A  reductions: tmin/tmax, and for raw input the weighted mean and
//            variance of LombScargleMemory.setdata (cuvarbase/lombscargle.py:
//            243-257) after the nanmean centring of normalize_light_curves
//            (cuvarbase/utils.py:134-141);
//   phase B  (NFFT method) for each of the two node sets -- x = df (t - tref)
//            for SYW and SW(f), 2x for SW(2f) -- the grid cell U, the in-cell
//            offset and the band-centring modulation exp(2 pi i Fc (t - tref))
//            of every point, in FP64 before the cast to FP32, then a counting
//            sort of the points by pass-1 column block (so every pass-1 tile
//            reads only the points that touch it); for curves of more than
//            16,384 points both phases run over chunks of 1,024 points, as a
//            reduction, a counting and a scatter kernel (LDS counts per chunk,
//            one global atomic per bucket and chunk);
//            (direct method) the FP32 weights and FP64 time offsets.
// With FP32 coordinates (GLS_PRECISION_FP32, for comparison with the
// reference's arithmetic) t is rounded to FP32 after centring on its mean and
// the time offset, cell coordinate and modulation phase of every point are
// FP32 operations; everything else is unchanged.
#include <algorithm>

#include "device_util.hpp"

namespace gls {

namespace {

struct PrepVals {
    double t;
    double yv;   // raw: y; weighted: yw; nfft: y
    double wv;   // raw: dy; weighted: w
};

template <int KIND>  // 0 raw, 1 weighted, 2 nfft
__device__ __forceinline__ PrepVals load_point(const double* t, const void* a, const void* b,
                                               int64_t i, int y_is_f32) {
    PrepVals p;
    p.t = t[i];
    if (KIND == 0) {
        p.yv = ((const double*)a)[i];
        p.wv = ((const double*)b)[i];
    } else if (KIND == 1) {
        p.yv = (double)((const float*)a)[i];
        p.wv = (double)((const float*)b)[i];
    } else {
        p.yv = y_is_f32 ? (double)((const float*)a)[i] : ((const double*)a)[i];
        p.wv = 1.0;
    }
    return p;
}

// time offset of a point from the curve's origin: t - tref in FP64, or with
// F32 the reference's FP32 arithmetic, (float)(t - tmean) - (float)(tref - tmean)
template <bool F32>
__device__ __forceinline__ double point_dt(double t, double tref, double tmean) {
    if (F32) return (double)((float)(t - tmean) - (float)(tref - tmean));
    return t - tref;
}

// grid cell U (first of the 2m+1 it touches) of a point at time offset dt in
// node set g (x = g df dt); yc = its position in cells (FP32 operations with F32)
template <bool F32>
__device__ __forceinline__ int prep_cell(double dt, int g, const CurveGeom& G, int m,
                                         double& yc) {
    if (F32) {
        const float x = (float)dt * (float)((double)g * G.df);
        float ycf = (x - floorf(x)) * (float)G.n;
        if (ycf >= (float)G.n) ycf -= (float)G.n;   // a fraction just below 1 rounded up
        yc = (double)ycf;
        return (int)floorf(ycf) - m;
    }
    const double x = dt * ((double)g * G.df);
    yc = (x - floor(x)) * (double)G.n;
    return (int)floor(yc) - m;
}

// band-centring modulation exp(2 pi i g Fc dt): the phase reduced in FP64
// before the FP32 sine and cosine, or with F32 formed and reduced in FP32
template <int KIND, bool F32>
__device__ __forceinline__ float2 prep_phase(double dt, int g, double Fc) {
    if (F32) {
        float r = (float)g * ((float)Fc * (float)dt);
        r -= rintf(r);
        float sn, cs;
        sincospif(2.0f * r, &sn, &cs);
        return make_float2(cs, sn);
    }
    if (KIND == 2) return expi_rev((double)g * (Fc * dt));
    return expi_turn4(4.0 * ((double)g * (Fc * dt)));
}

// weights of a point as FP64: (w, yw) for lomb, (-, y) for nfft
template <int KIND>
__device__ __forceinline__ void prep_weights(const PrepVals& p, double ymean, double ybar,
                                             double s0inv, double& w, double& yw) {
    if (KIND == 0) {
        w = s0inv / (p.wv * p.wv);
        yw = w * (p.yv - ymean - ybar);
    } else if (KIND == 1) {
        w = p.wv;
        yw = p.yv;
    } else {
        w = 0.0;
        yw = p.yv;
    }
}

// writes a point's entries into both node sets (one for nfft) and, for the
// low-frequency sums, its prepared weights in original order; cursor(g,
// bucket) returns the point's slot in the bucket order
template <int KIND, bool F32, typename Cursor>
__device__ __forceinline__ void prep_emit(const PointArrays& pa, const CurveGeom& G, int j,
                                          double dt, double w, double yw, double Fc, int m,
                                          Cursor&& cursor) {
    constexpr int NG = (KIND == 2) ? 1 : 2;
    const bool lowfix = KIND != 2 && pa.dt != nullptr;
    const bool ok = isfinite(dt);
    if (lowfix) {
        pa.w[G.pts + j] = ok ? (float)w : 0.f;
        pa.yw[G.pts + j] = ok ? (float)yw : 0.f;
        pa.dt[G.pts + j] = ok ? dt : 0.0;
    }
    if (!ok) return;   // non-finite times contribute nothing
    const int n2 = 1 << G.p2;
    const int lc1 = 31 - __clz(G.c1);
#pragma unroll
    for (int g = 1; g <= NG; ++g) {
        double yc;
        const int U = prep_cell<F32>(dt, g, G, m, yc);
        const float fr = (float)(yc - floor(yc));
        const float2 e = prep_phase<KIND, F32>(dt, g, Fc);
        const int pos = cursor(g - 1, (U & (n2 - 1)) >> lc1);
        const int64_t o = G.pts + pos;
        auto rec = [&](double s) {
            return make_int4(U, __float_as_int(fr), __float_as_int((float)s * e.x),
                             __float_as_int((float)s * e.y));
        };
        if (g == 1) {
            pa.nd0[o] = rec(yw);
            if (KIND != 2) pa.nd1[o] = rec(w);
        } else {
            pa.nd2[o] = rec(w);
        }
    }
}

// In-place exclusive scan of h[0 .. n) by the whole block; returns the total.
template <int NTP>
__device__ int block_exclusive_scan(int* h, int n, int* wsum) {
    const int tid = threadIdx.x;
    const int per = (n + NTP - 1) / NTP;
    const int lo = min(n, tid * per), hi = min(n, lo + per);
    int local = 0;
    for (int i = lo; i < hi; ++i) local += h[i];
    // inclusive scan of the chunk sums over the wave, then over the waves
    const int lane = tid & (kWave - 1), wv = tid / kWave;
    int v = local;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int u = __shfl_up(v, o, kWave);
        if (lane >= o) v += u;
    }
    if (lane == kWave - 1) wsum[wv] = v;
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NTP / kWave; ++w) {
        const int x = wsum[w];
        before += w < wv ? x : 0;
        total += x;
    }
    int run = v - local + before;   // exclusive prefix of this chunk
    for (int i = lo; i < hi; ++i) {
        const int x = h[i];
        h[i] = run;
        run += x;
    }
    __syncthreads();
    return total;
}

// The reductions of phase A: value number q of a wave's partials, the first
// two by minimum and the others by sum, over the 8 waves of a block: every wave
// reads one partial per lane, 8 q + wave, and folds the waves by exchange within
// rows.  part[] in LDS, written before a barrier.
template <int NQ>
__device__ __forceinline__ void block_fold(const double* part, int lane, double (&v)[NQ]) {
    static_assert(NQ * 8 <= kWave, "one partial per lane");
    double x = lane < NQ * 8 ? part[lane] : 0.0;
    auto op = [&](double y) { return lane < 16 ? fmin(x, y) : x + y; };
    x = op(row_move<0xB1>(x));
    x = op(row_move<0x4E>(x));
    x = op(row_move<0x141>(x));
#pragma unroll
    for (int q = 0; q < NQ; ++q) v[q] = lane_value(x, 8 * q);
}

// The descriptors of a launch: already in the workspace, or (META) in its own
// arguments, from where the first workgroup also stores them for the kernels
// that follow (one launch less than an upload of its own).
template <bool META>
struct MetaIn {};
template <>
struct MetaIn<true> {
    MetaArg arg;
};
template <bool META>
__device__ __forceinline__ const char* meta_base(char* ws, int words, int nt) {
    if (!META) return ws;
    const int4* const w = meta_arg_words();
    if (blockIdx.x == 0 && blockIdx.y == 0)
        for (int i = threadIdx.x; i < words; i += nt) ((int4*)ws)[i] = w[i];
    return (const char*)w;
}

// One workgroup per curve (number blockIdx.x of the list; in order, curve
// blockIdx.x, whose geometry then loads at once).  A thread keeps kPrepPts points
// in registers, so a curve of up to kPrepNT kPrepPts = 1,024 points is read
// once; longer ones are read again, tile by tile, in each phase.  The sums of
// phase A are folded together: one barrier for the time range and the weighted
// sums, one for the bucket counts and the variance, two for the scan of both
// node sets' buckets as one array.  Bound by the latency of that chain
// and, for thousands of points, by the scattered 16-byte records (one per lane
// and clock of the one CU).  Measured, against 256 threads that read the points
// five times and folded every sum by itself: one curve of 1,000 points 13.6 ->
// 6.3 us, 37 of 400-3,000 24.5 -> 14 us, 29 of up to 16,384 63 -> 41 us, 2,000
// of 20-300 23 -> 20 us; one set of 1,000-4,000 points (plain NFFT) 14.7 -> 9.1
// us.
constexpr int kPrepNT = 512;
constexpr int kPrepPts = 2;
template <int KIND, bool F32, bool META>
__global__ __launch_bounds__(kPrepNT, 6) void prep_kernel(MetaIn<META>, char* ws, int meta_words,
                                                       int off_geom, int off_list, bool in_order,
                                                       CurveState* __restrict__ state,
                                                       const double* __restrict__ t,
                                                       const void* __restrict__ a,
                                                       const void* __restrict__ b,
                                                       PointArrays pa, int32_t* __restrict__ bkt,
                                                       int m, int method, int y_is_f32) {
    constexpr int W = kPrepNT / kWave;
    static_assert(W == 8, "block_fold folds eight waves");
    constexpr int NQ = F32 ? 8 : 6;
    constexpr int TILE = kPrepNT * kPrepPts;
    __shared__ double red[NQ * W];
    __shared__ double redyy[W];
    __shared__ int wsum[W];
    extern __shared__ __align__(16) int hist[];   // the buckets of both node sets
    const char* const desc = meta_base<META>(ws, meta_words, kPrepNT);
    const int c = in_order ? (int)blockIdx.x : ((const int32_t*)(desc + off_list))[blockIdx.x];
    const CurveGeom G = ((const CurveGeom*)(desc + off_geom))[c];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1), wv = tid / kWave;
    const int N = G.n_obs;
    const bool direct = method != GLS_METHOD_NFFT;
    constexpr int NG = (KIND == 2) ? 1 : 2;
    const int n2 = 1 << G.p2;
    const int lc1 = direct ? 0 : 31 - __clz(G.c1);   // (c1 is a power of two)
    const int nb = direct ? 0 : n2 >> lc1;

    PrepVals q[kPrepPts];
    auto load_tile = [&](int base) {
#pragma unroll
        for (int u = 0; u < kPrepPts; ++u) {
            if (base + u * kPrepNT >= N) break;   // (the whole block)
            const int j = base + u * kPrepNT + tid;
            if (j < N) q[u] = load_point<KIND>(t, a, b, G.obs + j, y_is_f32);
        }
    };
    // f(j, point) for this thread's points; a curve of one tile is in registers
    auto each = [&](auto&& f, bool loaded) {
        for (int base = 0; base < N; base += TILE) {
            if (!(loaded && N <= TILE)) load_tile(base);
#pragma unroll
            for (int u = 0; u < kPrepPts; ++u) {
                if (base + u * kPrepNT >= N) break;
                const int j = base + u * kPrepNT + tid;
                if (j < N) f(j, q[u]);
            }
        }
    };

    // ---- phase A: reductions ------------------------------------------------
    if (N <= TILE) load_tile(0);
    for (int i = tid; i < NG * nb; i += kPrepNT) hist[i] = 0;
    // time range (as minima), then raw input: sum and count of the finite y,
    // sums of 1/dy^2 and y/dy^2; FP32 coordinates: sum and count of the finite t
    double v[NQ] = {INFINITY, INFINITY};
    each([&](int, const PrepVals& p) {
        v[0] = fmin(v[0], p.t);
        v[1] = fmin(v[1], -p.t);
        if (KIND == 0) {
            if (isfinite(p.yv)) {
                v[2] += p.yv;
                v[3] += 1.0;
            }
            const double iw = 1.0 / (p.wv * p.wv);
            v[4] += iw;
            v[5] += p.yv * iw;
        }
        if constexpr (F32)
            if (isfinite(p.t)) {
                v[NQ - 2] += p.t;
                v[NQ - 1] += 1.0;
            }
    }, true);
    // (waves past a short curve's points have nothing to fold or to emit; they
    // only clear, scan and meet the barriers)
    const bool busy = wv * kWave < N || wv == 0;
    if (busy) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            if (KIND != 0 && i >= 2 && i < 6) continue;
            v[i] = i < 2 ? wave_min(v[i]) : wave_sum(v[i]);
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) red[i * W + wv] = v[i];
    }
    __syncthreads();
    if (busy) block_fold<NQ>(red, lane, v);
    const double tref = v[0], tmax = -v[1];
    const double tmean = F32 ? v[NQ - 2] / v[NQ - 1] : 0.0;
    double ymean = 0.0, ybar = G.ybar_in, s0inv = 1.0;
    if (KIND == 0) {
        ymean = v[2] / v[3];
        s0inv = 1.0 / v[4];
        ybar = v[5] / v[4] - ymean;
    }

    // ---- phase B: bucket counts of both node sets (x = df (t - tref) for SYW
    // and SW(f), 2x for SW(2f)) and the variance ------------------------------
    double s2 = 0.0;
    if (!direct || KIND == 0)
        each([&](int, const PrepVals& p) {
            if (KIND == 0) {
                const double d = p.yv - ymean - ybar;
                s2 += d * d / (p.wv * p.wv);
            }
            if (direct) return;
            const double dt = point_dt<F32>(p.t, tref, tmean);
            if (!isfinite(dt)) return;   // non-finite times contribute nothing
#pragma unroll
            for (int g = 1; g <= NG; ++g) {
                double yc;
                const int U = prep_cell<F32>(dt, g, G, m, yc);
                atomicAdd(&hist[(g - 1) * nb + ((U & (n2 - 1)) >> lc1)], 1);
            }
        }, true);
    if (KIND == 0) {
        if (busy) s2 = wave_sum(s2);
        if (lane == 0) redyy[wv] = s2;
    }
    __syncthreads();
    if (tid == 0) {
        CurveState st;
        st.tref = tref;
        st.ybar = ybar;
        st.yy = G.yy_in;
        if (KIND == 0) {
            double yy = redyy[0];
            for (int w = 1; w < W; ++w) yy += redyy[w];
            st.yy = yy * s0inv;
        }
        st.tspan = tmax - tref;
        st.tmean = tmean;
        st.klow = N > 0 ? low_count(G, st.tspan) : 0;
        state[c] = st;
    }
    if (direct) {
        each([&](int j, const PrepVals& p) {
            double w, yw;
            prep_weights<KIND>(p, ymean, ybar, s0inv, w, yw);
            pa.w[G.pts + j] = (float)w;
            pa.yw[G.pts + j] = (float)yw;
            pa.dt[G.pts + j] = p.t - tref;
        }, true);
        return;
    }
    // both sets hold the same points: the second's offsets start at half the total
    const int total = block_exclusive_scan<kPrepNT>(hist, NG * nb, wsum) / NG;
    int32_t* const bk = bkt + G.bkt;
    for (int i = tid; i < NG * nb; i += kPrepNT) {
        const int second = i >= nb ? 1 : 0;
        bk[i + second] = hist[i] - second * total;   // (nb + 1 entries per set)
    }
    if (tid < NG) bk[tid * (nb + 1) + nb] = total;
    __syncthreads();
    const double Fc = G.f0 + (double)G.kc * G.df;
    each([&](int j, const PrepVals& p) {
        double w, yw;
        prep_weights<KIND>(p, ymean, ybar, s0inv, w, yw);
        prep_emit<KIND, F32>(pa, G, j, point_dt<F32>(p.t, tref, tmean), w, yw, Fc, m,
                             [&](int gs, int bucket) {
                                 return atomicAdd(&hist[gs * nb + bucket], 1) - gs * total;
                             });
    }, true);
}

// Wide curves (more than kWidePrep points, NFFT method) are prepared by three
// kernels over chunks of their points: blockIdx.y picks the curve (number
// blockIdx.y of the wide ones, record aux[blockIdx.y], chunk partials part[
// blockIdx.y gridDim.x ..]), blockIdx.x its chunk.  A chunk is kWideChunk
// points, or as many times that as leave at most kWideBlocks chunks (the chunks
// of a curve depend on its own points alone, so its results are the same in any
// batch).  The grid has as many chunks as the longest curve may need; those
// past a curve's end do nothing.  A thread holds kWidePts points of a chunk of
// kWideChunk in registers.  Nothing waits for a last block: what a chunk leaves is
// folded by every block of the next kernel.  Bound by latency (a chain of loads,
// folds and atomics, all chunks at a time) and the scatter by its 16-byte
// records.  Measured (200,000 points), against chunks of 2,048, last blocks
// behind fences and a clearing launch: reduction 23 -> 5 us, counting 17 -> 12,
// scatter 34 -> 19.
constexpr int kWideNT = 512;
constexpr int kWidePts = kWideChunk / kWideNT;
static_assert(kWidePts * kWideNT == kWideChunk, "whole points per thread");

struct WideSpan {
    int j0, j1;    // this block's points
    int chunks;    // chunks of the curve
    __device__ __forceinline__ explicit WideSpan(int N) {
        constexpr int kAll = kWideChunk * kWideBlocks;
        const int64_t len = (int64_t)kWideChunk * (((int64_t)N + kAll - 1) / kAll);
        chunks = (int)((N + len - 1) / len);
        j0 = (int)min((int64_t)N, blockIdx.x * len);
        j1 = (int)min((int64_t)N, j0 + len);
    }
    // f(j, u) for this thread's points, u their places in kWidePts registers; load
    // fills the registers of a round (a span of one round is loaded once)
    template <class L, class F>
    __device__ __forceinline__ void each(L&& load, F&& f, bool loaded) const {
        for (int base = j0; base < j1; base += kWideChunk) {
            if (!(loaded && j1 - j0 <= kWideChunk)) load(base);
#pragma unroll
            for (int u = 0; u < kWidePts; ++u) {
                const int j = base + u * kWideNT + (int)threadIdx.x;
                if (j < j1) f(j, u);
            }
        }
    }
};

// wide_reduce_kernel: the reductions of phase A per chunk (time range; for
// raw input the sums of the finite y, of 1/dy^2 and y/dy^2; with FP32
// coordinates the sum of the finite t), each chunk's partials into its slot;
// it also clears the record's counters for the kernels that follow.
template <int KIND, bool F32, bool META>
__global__ __launch_bounds__(kWideNT) void wide_reduce_kernel(MetaIn<META>, char* ws, int meta_words,
                                                              int off_geom, int off_wide,
                                                              const double* __restrict__ t,
                                                              const void* __restrict__ a,
                                                              const void* __restrict__ b,
                                                              WideAux* __restrict__ aux,
                                                              WidePart* __restrict__ part,
                                                              int y_is_f32) {
    constexpr int W = kWideNT / kWave;
    constexpr int NQ = F32 ? 8 : 6;
    __shared__ double red[NQ * W];
    const char* const desc = meta_base<META>(ws, meta_words, kWideNT);
    const int c = ((const int32_t*)(desc + off_wide))[blockIdx.y];
    const CurveGeom& G = ((const CurveGeom*)(desc + off_geom))[c];
    WideAux& X = aux[blockIdx.y];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1), wv = tid / kWave;
    const WideSpan sp(G.n_obs);
    if (sp.j0 >= sp.j1) return;
    const int64_t obs = G.obs;
    PrepVals q[kWidePts];
    auto load = [&](int base) {
#pragma unroll
        for (int u = 0; u < kWidePts; ++u) {
            const int j = base + u * kWideNT + tid;
            if (j < sp.j1) q[u] = load_point<KIND>(t, a, b, obs + j, y_is_f32);
        }
    };
    load(sp.j0);
    const int nb = (1 << G.p2) / G.c1;
    for (int i = (int)blockIdx.x * kWideNT + tid; i < 2 * nb; i += sp.chunks * kWideNT) {
        X.hist[i] = 0;
        X.taken[i] = 0;
    }
    if (blockIdx.x == 0)
        for (int i = tid; i < kLowSlots / 2; i += kWideNT) X.low_done[i] = 0;
    double v[NQ] = {INFINITY, INFINITY};
    sp.each(load, [&](int, int u) {
        const PrepVals& p = q[u];
        v[0] = fmin(v[0], p.t);
        v[1] = fmin(v[1], -p.t);
        if (KIND == 0) {
            if (isfinite(p.yv)) {
                v[2] += p.yv;
                v[3] += 1.0;
            }
            const double iw = 1.0 / (p.wv * p.wv);
            v[4] += iw;
            v[5] += p.yv * iw;
        }
        if constexpr (F32)
            if (isfinite(p.t)) {
                v[NQ - 2] += p.t;
                v[NQ - 1] += 1.0;
            }
    }, true);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        if (KIND != 0 && i >= 2 && i < 6) continue;
        v[i] = i < 2 ? wave_min(v[i]) : wave_sum(v[i]);
    }
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) red[i * W + wv] = v[i];
    }
    __syncthreads();
    if (wv != 0) return;
    block_fold<NQ>(red, lane, v);
    if (lane == 0) {
        WidePart& P = part[(int64_t)blockIdx.y * gridDim.x + blockIdx.x];
#pragma unroll
        for (int i = 0; i < NQ; ++i) P.v[i] = v[i];
    }
}

// this chunk's points per bucket of both node sets, h[0 .. NG nb)
template <int KIND, bool F32, class Load, class Q>
__device__ __forceinline__ void wide_chunk_counts(int* h, const CurveGeom& G, const WideSpan& sp,
                                                  Load&& load, const Q& q, double tref,
                                                  double tmean, int m) {
    constexpr int NG = (KIND == 2) ? 1 : 2;
    const int n2 = 1 << G.p2;
    const int lc1 = 31 - __clz(G.c1);
    const int nb = n2 >> lc1;
    for (int i = threadIdx.x; i < NG * nb; i += kWideNT) h[i] = 0;
    __syncthreads();
    sp.each(load, [&](int, int u) {
        const double dt = point_dt<F32>(q[u].t, tref, tmean);
        if (!isfinite(dt)) return;
#pragma unroll
        for (int g = 1; g <= NG; ++g) {
            double yc;
            const int U = prep_cell<F32>(dt, g, G, m, yc);
            atomicAdd(&h[(g - 1) * nb + ((U & (n2 - 1)) >> lc1)], 1);
        }
    }, true);
    __syncthreads();
}

// wide_count_kernel: every block folds the chunk partials, in chunk order (the
// first writes the curve's state and weight constants), counts its chunk's
// points per bucket in LDS and adds them to the record, two buckets in one 64-bit
// atomic (no count reaches 2^32; per-point global atomics on a few hundred
// counters would serialise on their cache lines).  It also sums its points'
// (y - ymean - ybar)^2 / dy^2 (raw input).
template <int KIND, bool F32>
__global__ __launch_bounds__(kWideNT) void wide_count_kernel(const CurveGeom* __restrict__ geom,
                                                             const int32_t* __restrict__ wide,
                                                             CurveState* __restrict__ state,
                                                             const double* __restrict__ t,
                                                             const void* __restrict__ a,
                                                             const void* __restrict__ b,
                                                             WideAux* __restrict__ aux,
                                                             WidePart* __restrict__ part, int m,
                                                             int y_is_f32) {
    constexpr int W = kWideNT / kWave;
    constexpr int NQ = F32 ? 8 : 6;
    constexpr int NG = (KIND == 2) ? 1 : 2;
    __shared__ double red[NQ * W];
    __shared__ double redyy[W];
    extern __shared__ __align__(16) int h[];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1), wv = tid / kWave;
    const int c = wide[blockIdx.y];
    const CurveGeom G = geom[c];
    const WideSpan sp(G.n_obs);
    if (sp.j0 >= sp.j1) return;
    WideAux& X = aux[blockIdx.y];
    PrepVals q[kWidePts];
    auto load = [&](int base) {
#pragma unroll
        for (int u = 0; u < kWidePts; ++u) {
            const int j = base + u * kWideNT + tid;
            if (j < sp.j1) q[u] = load_point<KIND>(t, a, b, G.obs + j, y_is_f32);
        }
    };
    load(sp.j0);
    WidePart* const P = part + (int64_t)blockIdx.y * gridDim.x;
    double v[NQ] = {INFINITY, INFINITY};
    for (int i = tid; i < sp.chunks; i += kWideNT) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) v[k] = k < 2 ? fmin(v[k], P[i].v[k]) : v[k] + P[i].v[k];
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        if (KIND != 0 && i >= 2 && i < 6) continue;
        v[i] = i < 2 ? wave_min(v[i]) : wave_sum(v[i]);
    }
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) red[i * W + wv] = v[i];
    }
    __syncthreads();
    block_fold<NQ>(red, lane, v);
    const double tref = v[0], tmean = F32 ? v[NQ - 2] / v[NQ - 1] : 0.0;
    double ymean = 0.0, ybar = G.ybar_in, s0inv = 1.0;
    if (KIND == 0) {
        ymean = v[2] / v[3];
        s0inv = 1.0 / v[4];
        ybar = v[5] / v[4] - ymean;
    }
    if (blockIdx.x == 0 && tid == 0) {
        CurveState st;
        st.tref = tref;
        st.tspan = -v[1] - tref;
        st.tmean = tmean;
        st.klow = low_count(G, st.tspan);
        st.ybar = ybar;
        st.yy = G.yy_in;   // (raw input: the scatter's first block writes it)
        X.ymean = ymean;
        X.s0inv = s0inv;
        state[c] = st;
    }
    wide_chunk_counts<KIND, F32>(h, G, sp, load, q, tref, tmean, m);
    const int nb = (1 << G.p2) / G.c1;
    for (int i = tid; i < NG * nb / 2; i += kWideNT) {
        const unsigned long long two = ((const unsigned long long*)h)[i];
        if (two != 0) atomicAdd((unsigned long long*)X.hist + i, two);
    }
    if (KIND != 0) return;
    double s2 = 0.0;
    sp.each(load, [&](int, int u) {
        const PrepVals& p = q[u];
        const double d = p.yv - ymean - ybar;
        s2 += d * d / (p.wv * p.wv);
    }, true);
    s2 = block_sum<kWideNT>(s2, redyy);
    if (tid == 0) P[blockIdx.x].syy = s2;
}

// wide_scatter_kernel: each block scans the buckets' totals into their starts
// (the first writes them to bkt and folds the chunks' variance partials, in
// order, into the curve's yy), counts its chunk again, reserves its slots per
// bucket with one atomic for two buckets, then ranks its points in LDS.
template <int KIND, bool F32>
__global__ __launch_bounds__(kWideNT) void wide_scatter_kernel(const CurveGeom* __restrict__ geom,
                                                               const int32_t* __restrict__ wide,
                                                               CurveState* __restrict__ state,
                                                               const double* __restrict__ t,
                                                               const void* __restrict__ a,
                                                               const void* __restrict__ b,
                                                               PointArrays pa,
                                                               int32_t* __restrict__ bkt,
                                                               WideAux* __restrict__ aux,
                                                               const WidePart* __restrict__ part,
                                                               int m, int y_is_f32) {
    constexpr int W = kWideNT / kWave;
    constexpr int NG = (KIND == 2) ? 1 : 2;
    __shared__ double red[W];
    __shared__ int wsum[W];
    extern __shared__ __align__(16) int h[];   // counts, then the buckets' starts
    const int tid = threadIdx.x;
    const int c = wide[blockIdx.y];
    const CurveGeom G = geom[c];
    const WideSpan sp(G.n_obs);
    if (sp.j0 >= sp.j1) return;
    WideAux& X = aux[blockIdx.y];
    PrepVals q[kWidePts];
    auto load = [&](int base) {
#pragma unroll
        for (int u = 0; u < kWidePts; ++u) {
            const int j = base + u * kWideNT + tid;
            if (j < sp.j1) q[u] = load_point<KIND>(t, a, b, G.obs + j, y_is_f32);
        }
    };
    load(sp.j0);
    const double tref = state[c].tref, tmean = F32 ? state[c].tmean : 0.0, ybar = state[c].ybar;
    const double ymean = X.ymean, s0inv = X.s0inv;
    const int nb = (1 << G.p2) / G.c1;
    int* const start = h + NG * nb;
    for (int i = tid; i < NG * nb; i += kWideNT) start[i] = X.hist[i];
    __syncthreads();
    // (both sets hold the same points: the second's starts begin at half the total)
    const int total = block_exclusive_scan<kWideNT>(start, NG * nb, wsum) / NG;
    if (blockIdx.x == 0) {
        int32_t* const bk = bkt + G.bkt;
        for (int i = tid; i < NG * nb; i += kWideNT) {
            const int second = i >= nb ? 1 : 0;
            bk[i + second] = start[i] - second * total;
        }
        if (tid < NG) bk[tid * (nb + 1) + nb] = total;
        if (KIND == 0) {
            const WidePart* const P = part + (int64_t)blockIdx.y * gridDim.x;
            double s2 = 0.0;
            for (int i = tid; i < sp.chunks; i += kWideNT) s2 += P[i].syy;
            s2 = block_sum<kWideNT>(s2, red);
            if (tid == 0) state[c].yy = s2 * s0inv;
        }
    }
    wide_chunk_counts<KIND, F32>(h, G, sp, load, q, tref, tmean, m);
    // this block's first slot in each bucket
    for (int i = tid; i < NG * nb / 2; i += kWideNT) {
        const unsigned long long two = ((const unsigned long long*)h)[i];
        if (two == 0) continue;
        const unsigned long long was = atomicAdd((unsigned long long*)X.taken + i, two);
        const int off = 2 * i >= nb ? total : 0;   // (nb is even)
        h[2 * i] = start[2 * i] + (int)(uint32_t)was - off;
        h[2 * i + 1] = start[2 * i + 1] + (int)(uint32_t)(was >> 32) - off;
    }
    __syncthreads();
    const double Fc = G.f0 + (double)G.kc * G.df;
    sp.each(load, [&](int j, int u) {
        const PrepVals& p = q[u];
        double w, yw;
        prep_weights<KIND>(p, ymean, ybar, s0inv, w, yw);
        prep_emit<KIND, F32>(pa, G, j, point_dt<F32>(p.t, tref, tmean), w, yw, Fc, m,
                             [&](int gs, int bucket) { return atomicAdd(&h[gs * nb + bucket], 1); });
    }, true);
}

}  // namespace

namespace {
template <bool F32>
hipError_t launch_prep_t(const CurveGeom* d_geom, const int32_t* small, int nsmall,
                         const int32_t* wide, int nwide, CurveState* state, const double* t,
                         const void* a, const void* b, PointArrays pa, int32_t* bkt,
                         const PlanParams& pp, int y_is_f32, WideAux* aux, WidePart* part,
                         int wide_max_obs, int max_buckets, bool in_order,
                         const MetaArg* meta, int meta_words, char* ws, hipStream_t s) {
    const int kind = (pp.kind == 1) ? 2 : (pp.input_kind == GLS_INPUT_RAW ? 0 : 1);
    const int method = (pp.kind == 1) ? GLS_METHOD_NFFT : pp.method;
    const int yf = (pp.kind == 1) ? y_is_f32 : 0;
    const int off_geom = (int)((const char*)d_geom - ws), off_list = (int)((const char*)small - ws);
    MetaIn<true> in;
    if (meta) in.arg = *meta;
#define GLS_PREP_LAUNCH(K, M, IN)                                                             \
    hipLaunchKernelGGL((prep_kernel<K, F32, M>), dim3(nblocks), dim3(kPrepNT), lds, s, IN, ws, \
                       meta_words, off_geom, off_list, in_order, state, t, a, b, pa, bkt,    \
                       pp.m, method, yf)
#define GLS_PREP_KIND(M, IN)                   \
    if (kind == 0) GLS_PREP_LAUNCH(0, M, IN);  \
    else if (kind == 1) GLS_PREP_LAUNCH(1, M, IN); \
    else GLS_PREP_LAUNCH(2, M, IN)
    // wide curves take the chunked kernels on the NFFT path, else the same one
    // workgroup as the others, which they follow in the list
    const bool split = aux != nullptr && part != nullptr && method == GLS_METHOD_NFFT &&
                       wide_max_obs > 0;
    const int nblocks = nsmall + (split ? 0 : nwide);
    const size_t lds = sizeof(int) * (kind == 2 ? 1 : 2) * (size_t)max_buckets;
    if (nblocks > 0) {
        if (meta) {
            GLS_PREP_KIND(true, in);
        } else {
            GLS_PREP_KIND(false, MetaIn<false>{});
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
#undef GLS_PREP_KIND
#undef GLS_PREP_LAUNCH
    if (nwide <= 0 || !split) return hipSuccess;
    const int off_wide = (int)((const char*)wide - ws);
    const dim3 grid((unsigned)std::min(kWideBlocks, (wide_max_obs + kWideChunk - 1) / kWideChunk),
                    (unsigned)nwide);
    const bool ride = meta && nblocks == 0;
#define GLS_WIDE_REDUCE(K, M, IN)                                                             \
    hipLaunchKernelGGL((wide_reduce_kernel<K, F32, M>), grid, dim3(kWideNT), 0, s, IN, ws,     \
                       meta_words, off_geom, off_wide, t, a, b, aux, part, yf)
#define GLS_WIDE_LAUNCH(K)                                                                     \
    if (ride) GLS_WIDE_REDUCE(K, true, in);                                                    \
    else GLS_WIDE_REDUCE(K, false, MetaIn<false>{});                                           \
    hipLaunchKernelGGL((wide_count_kernel<K, F32>), grid, dim3(kWideNT), lds, s, d_geom, wide, \
                       state, t, a, b, aux, part, pp.m, yf);                                   \
    hipLaunchKernelGGL((wide_scatter_kernel<K, F32>), grid, dim3(kWideNT), 2 * lds, s, d_geom, \
                       wide, state, t, a, b, pa, bkt, aux, part, pp.m, yf)
    if (kind == 0) {
        GLS_WIDE_LAUNCH(0);
    } else if (kind == 1) {
        GLS_WIDE_LAUNCH(1);
    } else {
        GLS_WIDE_LAUNCH(2);
    }
#undef GLS_WIDE_LAUNCH
#undef GLS_WIDE_REDUCE
    return hipGetLastError();
}
}  // namespace

hipError_t launch_prep(const CurveGeom* d_geom, const int32_t* small, int nsmall,
                       const int32_t* wide, int nwide, CurveState* state, const double* t,
                       const void* a, const void* b, PointArrays pa, int32_t* bkt,
                       const PlanParams& pp, int y_is_f32, WideAux* aux, WidePart* part,
                       int wide_max_obs, int max_buckets, bool in_order,
                         const MetaArg* meta, int meta_words, char* ws, hipStream_t s) {
    if (pp.fp32_coords && pp.kind == 0)
        return launch_prep_t<true>(d_geom, small, nsmall, wide, nwide, state, t, a, b, pa, bkt,
                                   pp, y_is_f32, aux, part, wide_max_obs, max_buckets, in_order, meta,
                                   meta_words, ws, s);
    return launch_prep_t<false>(d_geom, small, nsmall, wide, nwide, state, t, a, b, pa, bkt, pp,
                                y_is_f32, aux, part, wide_max_obs, max_buckets, in_order, meta,
                                   meta_words, ws, s);
}

}  // namespace gls
