// Direct-summation GLS (use_fft=False).
//
// Replaces lomb_dirsum (cuvarbase/kernels/lomb.cu:144-165): six O(N) sums per
// frequency, then the power.  On a linear grid the sums are small matrix
// products and run on the matrix cores in FP32: write a frequency of a tile as
// f = F_a +- D_b, F_a the centre of its row of 32 frequencies and D_b = (b +
// 1/2) df, b < 16.  With A_c[a, j] = v_j cos(2 pi F_a dt_j), A_s with the sine,
// and B_c[j, b] = cos(2 pi D_b dt_j), B_s likewise, the four products over the
// points CC = A_c B_c, CS, SC, SS give both frequencies of the pair:
//   cosine sums CC -+ SS, sine sums SC +- CS   at F_a +- D_b.
// Six multiply-adds per point and frequency for the three sums (yw and w at f,
// w at 2f), against twelve by a plain complex product.  Each phase is reduced in FP64;
// the products are accumulated in FP32 over kDirChunk points of a wave and in
// FP64 beyond.
#include <algorithm>

#include "device_util.hpp"
#include "lds_fft.hpp"

namespace gls {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// points of one wave between two folds of its FP32 sums into FP64
constexpr int kDirChunk = 128;

// One wave computes a tile of 16 rows x 32 frequencies with 16 x 16 x 4 matrix
// instructions, 4 points at a time: lane l holds row a = l % 16 (and column b
// = l % 16) of point l / 16, so it evaluates two sines and cosines per 4
// points and 12 matrix instructions (the doubled angles follow from them).
// Those two halves cost about the same (75 vector instructions, 300 clocks,
// against 384 of the matrix pipe) and overlap between the two waves of a SIMD.
// WS waves share a tile, every WS-th group of 4 points each, and add their
// FP64 sums in LDS; a workgroup of 8 waves holds 8 / WS tiles.  Measured (10
// curves of 300-2,000 points, 10,007 frequencies, 1.05e8 point-frequencies):
// 43 us against 229 us of one frequency run per thread on the vector ALU; the
// matrix pipe alone would take 8 us, the longest curve's chain sets the rest.
template <int WS, int OUT>
__global__ __launch_bounds__(kDirNT) void dirsum_kernel(const CurveGeom* __restrict__ geom,
                                                        const CurveState* __restrict__ state,
                                                        const int32_t* __restrict__ tile_curve,
                                                        const int32_t* __restrict__ tile_first,
                                                        PointArrays pa, PlanParams pp,
                                                        void* __restrict__ out) {
    constexpr int WAVES = kDirNT / kWave;
    // LDS of the reduction: the upper half of a tile's waves hands 48 sums per
    // lane to the lower half
    __shared__ double red[WS > 1 ? WAVES / 2 : 1][WS > 1 ? 48 : 1][kWave];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int part = wv % WS;      // which of the tile's waves
    const int tl = wv / WS;        // which of the workgroup's tiles
    const int ci = tile_curve[blockIdx.x];
    const CurveGeom& G = geom[ci];
    const int N = G.n_obs;
    const int k0 = tile_first[blockIdx.x] + tl * kDirTile;
    const int col = lane & 15, sub = lane >> 4;
    // quarter turns per unit time of this lane's row centre and column offset
    const double fa = 4.0 * (G.f0 + ((double)(k0 + 32 * col) + 15.5) * G.df);
    const double fb = 4.0 * (((double)col + 0.5) * G.df);
    const double* const dt = pa.dt + G.pts;
    const float* const pw = pa.w + G.pts;
    const float* const py = pa.yw + G.pts;

    v4f acc[12];
    double sum[12][4];
#pragma unroll
    for (int q = 0; q < 12; ++q) {
        acc[q] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[q][r] = 0.0;
    }
    auto fold = [&]() {
#pragma unroll
        for (int q = 0; q < 12; ++q) {
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[q][r] += (double)acc[q][r];
            acc[q] = v4f{0.f, 0.f, 0.f, 0.f};
        }
    };
    if (k0 < G.nf) {
        int j = part * 4 + sub;
        double x = 0.0;
        float w = 0.f, yw = 0.f;
        if (j < N) {
            x = dt[j];
            w = pw[j];
            yw = py[j];
        }
        int left = kDirChunk / 4;
        // the wave's groups of 4 points (the same count in every lane)
        for (int base = part * 4; base < N; base += 4 * WS) {
            const double xc = x;
            const float wc = w, yc = yw;
            j += 4 * WS;
            x = 0.0;
            w = yw = 0.f;
            if (j < N) {   // the next group's points, loaded ahead
                x = dt[j];
                w = pw[j];
                yw = py[j];
            }
            const float2 ea = expi_turn4(fa * xc);
            const float2 eb = expi_turn4(fb * xc);
            const float wca = wc * ea.x, wsa = wc * ea.y;
            const float c2 = ea.x * ea.x - ea.y * ea.y, s2 = 2.f * ea.x * ea.y;
            const float cb2 = eb.x * eb.x - eb.y * eb.y, sb2 = 2.f * eb.x * eb.y;
            const float A[6] = {yc * ea.x, yc * ea.y, wca, wsa, wc * c2, wc * s2};
            const float B[6] = {eb.x, eb.y, eb.x, eb.y, cb2, sb2};
#pragma unroll
            for (int h = 0; h < 3; ++h)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc[4 * h + q] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        A[2 * h + (q >> 1)], B[2 * h + (q & 1)], acc[4 * h + q], 0, 0, 0);
            if (--left == 0) {
                fold();
                left = kDirChunk / 4;
            }
        }
        fold();
    }
    // the tile's waves add up, halving their number
    if constexpr (WS > 1) {
#pragma unroll
        for (int s = WS / 2; s >= 1; s /= 2) {
            const int slot = tl * (WS / 2) + (part % s);
            if (part >= s && part < 2 * s) {
#pragma unroll
                for (int q = 0; q < 48; ++q) red[slot][q][lane] = sum[q >> 2][q & 3];
            }
            __syncthreads();
            if (part < s) {
#pragma unroll
                for (int q = 0; q < 48; ++q) sum[q >> 2][q & 3] += red[slot][q][lane];
            }
            __syncthreads();
        }
        if (part != 0) return;
    }
    const CurveState st = state[ci];
    // accumulator element r of a lane: row 4 (lane / 16) + r, column lane % 16
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const double sg = side ? -1.0 : 1.0;
            const int k = k0 + 32 * (4 * sub + r) + (side ? 15 - col : 16 + col);
            if (k >= G.nf) continue;
            double z[3][2];
#pragma unroll
            for (int h = 0; h < 3; ++h) {
                z[h][0] = sum[4 * h][r] - sg * sum[4 * h + 3][r];       // CC -+ SS
                z[h][1] = sum[4 * h + 2][r] + sg * sum[4 * h + 1][r];   // SC +- CS
            }
            const double P = gls_power(z[1][0], z[1][1], z[2][0], z[2][1], z[0][0], z[0][1],
                                       st.yy, st.ybar, pp.mode, pp.reg_c, pp.reg_s);
            if (OUT == 0) ((float*)out)[G.out + k] = (float)P;
            else ((double*)out)[G.out + k] = P;
        }
    }
}

// Direct sums at explicit frequencies freqs[out + k] (any spacing): the work of
// lomb_dirsum_custom_frq (cuvarbase/kernels/lomb.cu:167-187).  One frequency
// per lane, each phase reduced mod 1/4 in FP64; WS waves share 64 frequencies,
// every WS-th run of kCusRun points each, and add their FP64 sums in LDS (a
// list of a few thousand frequencies otherwise leaves most compute units
// idle).  The points are the same for every lane of a wave, so they come
// through scalar loads.  Bound by the vector ALU (about 27 instructions per
// point and frequency) of the compute units with the longest curve: 4 curves of
// 500-3,000 points at 4,001 frequencies 33 us, against 145 us with 256
// frequencies per workgroup and no sharing.
constexpr int kCusRun = 4;
template <int WS, int OUT>
__global__ __launch_bounds__(kDirNT) void dirsum_custom_kernel(
    const CurveGeom* __restrict__ geom, const CurveState* __restrict__ state,
    const int32_t* __restrict__ tile_curve, const int32_t* __restrict__ tile_first,
    PointArrays pa, PlanParams pp, const double* __restrict__ freqs, void* __restrict__ out) {
    constexpr int WAVES = kDirNT / kWave;
    __shared__ double red[WS > 1 ? WAVES : 1][WS > 1 ? 6 : 1][kWave];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int part = wv % WS;
    const int ci = tile_curve[blockIdx.x];
    const CurveGeom& G = geom[ci];
    const int N = G.n_obs;
    const int k = tile_first[blockIdx.x] + (wv / WS) * kWave + lane;
    const double f = (k < G.nf) ? 4.0 * freqs[G.out + k] : 0.0;
    const double* const dt = pa.dt + G.pts;
    const float* const pw = pa.w + G.pts;
    const float* const py = pa.yw + G.pts;
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    float a[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto add = [&](int j) {
        const float2 z = expi_turn4(f * dt[j]);
        const float w = pw[j], yw = py[j];
        a[0] += w * z.x;
        a[1] += w * z.y;
        a[2] += w * (z.x * z.x - z.y * z.y);
        a[3] += w * (2.f * z.x * z.y);
        a[4] += yw * z.x;
        a[5] += yw * z.y;
    };
    auto fold = [&]() {
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            acc[q] += (double)a[q];
            a[q] = 0.f;
        }
    };
    int left = 256 / kCusRun;
    int j = part * kCusRun;
    for (; j + kCusRun <= N; j += kCusRun * WS) {
#pragma unroll
        for (int q = 0; q < kCusRun; ++q) add(j + q);
        if (--left == 0) {
            fold();
            left = 256 / kCusRun;
        }
    }
    for (; j < N; ++j) add(j);   // the last, partial run (of one wave)
    fold();
    if constexpr (WS > 1) {
#pragma unroll
        for (int q = 0; q < 6; ++q) red[wv][q][lane] = acc[q];
        __syncthreads();
        if (part != 0) return;
#pragma unroll
        for (int s = 1; s < WS; ++s)
#pragma unroll
            for (int q = 0; q < 6; ++q) acc[q] += red[wv + s][q][lane];
    }
    if (k < G.nf) {
        const CurveState st = state[ci];
        const double P = gls_power(acc[0], acc[1], acc[2], acc[3], acc[4], acc[5], st.yy,
                                   st.ybar, pp.mode, pp.reg_c, pp.reg_s);
        if (OUT == 0) ((float*)out)[G.out + k] = (float)P;
        else ((double*)out)[G.out + k] = P;
    }
}

// The GLS is ill-conditioned where a frequency spans few cycles over the
// baseline (CC SS - CS^2 -> 0): there the FP32 round-off of the NFFT sums,
// largest at the band edge where the lowest frequencies sit, reaches |dP| ~
// 1e-4.  These few frequencies, the leading run of the grid with |f| (t_max -
// t_min) < kLowCycles, are recomputed by direct sums with FP64 phases and FP64
// accumulation.
//
// A workgroup sums kLowGroup consecutive frequencies over a curve's points, or
// over one of S slices of them: a point's phasor at the group's first frequency
// and the phasor of one grid step are evaluated in FP64, the group's other
// frequencies follow by FP64 products (kLowGroup - 1 of them, 1e-16 each).
// Groups and slices are tasks that the curve's workgroups take in turn, so
// however long the run is, every frequency is covered, and the sums of a curve
// do not depend on how many workgroups it got.  Bound by FP64 issue: about 30
// vector instructions per point and frequency (110 with a sine and cosine of
// its own for each) and, for few points, by the chain of loads, exchanges and
// the power.  Measured, against a sine and cosine per point and frequency, one
// wave per frequency (1,024 lanes x 8 workgroups for wide curves) and two
// launches: 2,000 curves of 20-300 points 64 -> 31 us, one of 1,000 points 15
// -> 6 us, 37 of 400-3,000 points 28 -> 12 us, 32 of 100-50,000 points 89 -> 23
// us, one of 200,000 points 32 -> 13 us.
constexpr int kLowNT = 256;
constexpr int kLowSums = 6 * kLowGroup;
constexpr int kLowShort = 256;   // points up to which a wave sums alone

// sums V values over lanes that differ in the bits HI, HI / 2 .. 1 of their
// number: an exchange per value, but each step halves the values a lane holds
// while their number is even.  Afterwards v[0 .. V/8) of a lane are the sums
// number first .. (the same in lanes that differ in the remaining bits);
// returns first
template <int V, int HI>
__device__ __forceinline__ int lane_sum_scatter(double (&v)[V], int lane) {
    static_assert(V % 8 == 0 && V % 16 != 0 && HI >= 4, "three halvings");
    int first = 0;
    int cnt = V;
#pragma unroll
    for (int o = HI; o >= 1; o >>= 1) {
        if (cnt % 2 == 0) {
            cnt /= 2;
            const bool up = (lane & o) != 0;
            first += up ? cnt : 0;
#pragma unroll
            for (int i = 0; i < cnt; ++i) {
                const double send = up ? v[i] : v[cnt + i];
                const double keep = up ? v[cnt + i] : v[i];
                v[i] = keep + __shfl_xor(send, o, kWave);
            }
        } else {
#pragma unroll
            for (int i = 0; i < cnt; ++i) v[i] += __shfl_xor(v[i], o, kWave);
        }
    }
    return first;
}

// adds the points j0, j0 + step .. below j1 of a curve to the sums of the
// kLowGroup frequencies from k0 on
__device__ __forceinline__ void low_points(const CurveGeom& G, const PointArrays& pa, int k0,
                                           int j0, int j1, int step, double (&acc)[kLowSums]) {
    const double f4 = 4.0 * (G.f0 + (double)k0 * G.df), df4 = 4.0 * G.df;
    const double* const dt = pa.dt + G.pts;
    const float* const pw = pa.w + G.pts;
    const float* const py = pa.yw + G.pts;
    double xn = 0.0;
    float wn = 0.f, yn = 0.f;
    if (j0 < j1) {
        xn = dt[j0];
        wn = pw[j0];
        yn = py[j0];
    }
    for (int j = j0; j < j1; j += step) {
        const double x = xn, w = wn, yw = yn;
        if (j + step < j1) {   // the next point, loaded ahead
            xn = dt[j + step];
            wn = pw[j + step];
            yn = py[j + step];
        }
        double2 e = expi64_turn4(f4 * x);
        const double2 r = expi64_turn4(df4 * x);
#pragma unroll
        for (int i = 0; i < kLowGroup; ++i) {
            double* a = acc + 6 * i;
            a[0] += w * e.x;
            a[1] += w * e.y;
            a[2] += w * (e.x * e.x - e.y * e.y);
            a[3] += w * (2.0 * e.x * e.y);
            a[4] += yw * e.x;
            a[5] += yw * e.y;
            e = make_double2(e.x * r.x - e.y * r.y, e.x * r.y + e.y * r.x);
        }
    }
}

// Workgroups: bs for each of the nsmall curves of the list (without a list, the
// curves from first on), then bw for each of the wide ones after them (those with a record in aux may split their points).
template <int OUT>
__global__ __launch_bounds__(kLowNT) void lowfreq_kernel(
    const CurveGeom* __restrict__ geom, const int32_t* __restrict__ list, int first, int nsmall,
    int bs, int bw, const CurveState* __restrict__ state, PointArrays pa, PlanParams pp,
    WideAux* __restrict__ aux, void* __restrict__ out) {
    constexpr int WAVES = kLowNT / kWave;
    __shared__ double red[WAVES][4][kLowSums];
    __shared__ double slices[8][kLowSums];
    __shared__ int last;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = tid / kWave;
    const int bid = blockIdx.x;
    const bool wide = bid >= nsmall * bs;
    const int wi = wide ? (bid - nsmall * bs) / bw : 0;   // which of the wide curves
    const int ci = wide ? nsmall + wi : bid / bs;
    const int c = list ? list[ci] : first + ci;
    const int first_task = wide ? (bid - nsmall * bs) % bw : bid % bs;
    const int nblocks = wide ? bw : bs;
    const CurveGeom& G = geom[c];
    const CurveState st = state[c];
    const int kl = st.klow;
    const int ngroups = (kl + kLowGroup - 1) / kLowGroup;
    const int N = G.n_obs;
    auto store = [&](int k, const double* a) {
        const double P = gls_power(a[0], a[1], a[2], a[3], a[4], a[5], st.yy, st.ybar, pp.mode,
                                   pp.reg_c, pp.reg_s);
        if (OUT == 0) ((float*)out)[G.out + k] = (float)P;
        else ((double*)out)[G.out + k] = P;
    };
    if (N <= kLowShort) {
        // few points: a wave takes four groups, 16 lanes over the points of
        // each (a workgroup for each group spends its time on its barriers)
        constexpr int kRun = 4 * kLowGroup;
        double(*const rw)[kLowSums] = red[wv];
        for (int t = first_task * WAVES + wv; t * kRun < kl; t += nblocks * WAVES) {
            double acc[kLowSums];
#pragma unroll
            for (int q = 0; q < kLowSums; ++q) acc[q] = 0.0;
            const int g = lane >> 4;
            low_points(G, pa, t * kRun + g * kLowGroup, lane & 15, N, 16, acc);
            const int at = lane_sum_scatter<kLowSums, 8>(acc, lane);
            if ((lane & 1) == 0) {
#pragma unroll
                for (int q = 0; q < kLowSums / 8; ++q) rw[g][at + q] = acc[q];
            }
            // (one wave: its LDS accesses are in order)
            __builtin_amdgcn_wave_barrier();
            const int k = t * kRun + lane;
            if (lane < kRun && k < kl) store(k, &rw[lane / kLowGroup][6 * (lane % kLowGroup)]);
            __builtin_amdgcn_wave_barrier();
        }
        return;
    }
    WideAux* const X = (wide && aux) ? aux + wi : nullptr;
    // slices: of at least kLowSlice points, within the record's slots
    int S = 1;
    if (X)
        while (2 * S * ngroups <= kLowSlots && 2 * S * kLowSlice <= N) S *= 2;
    const int per = (N + S - 1) / S;
    for (int task = first_task; task < ngroups * S; task += nblocks) {
        const int g = task / S, z = task % S;
        const int k0 = g * kLowGroup;
        double acc[kLowSums];
#pragma unroll
        for (int q = 0; q < kLowSums; ++q) acc[q] = 0.0;
        low_points(G, pa, k0, z * per + tid, min(N, (z + 1) * per), kLowNT, acc);
        const int at = lane_sum_scatter<kLowSums, 32>(acc, lane);
        if ((lane & 7) == 0) {
#pragma unroll
            for (int q = 0; q < kLowSums / 8; ++q) red[wv][0][at + q] = acc[q];
        }
        __syncthreads();
        if (tid < kLowSums) {
            double v = red[0][0][tid];
#pragma unroll
            for (int q = 1; q < WAVES; ++q) v += red[q][0][tid];
            red[0][0][tid] = v;
            if (S > 1) agent_publish(&X->low[task][tid], v);
        }
        __syncthreads();
        bool done = true;
        if (S > 1) {
            if (tid == 0) last = atomicAdd(&X->low_done[g], 1) == S - 1;
            __syncthreads();
            done = last != 0;
            if (done) {
                // the slices in order, so the sum does not depend on which finished
                // first: kLowParts threads a sum, then those
                constexpr int kLowParts = 8;
                static_assert(kLowParts * kLowSums <= kLowNT, "one slice and sum per thread");
                const int part = tid / kLowSums, q = tid % kLowSums;
                double v = 0.0;
                if (part < kLowParts) {
#pragma unroll 4
                    for (int i = part; i < S; i += kLowParts)
                        v += agent_load(&X->low[g * S + i][q]);
                    slices[part][q] = v;
                }
                __syncthreads();
                if (tid < kLowSums) {
                    v = 0.0;
#pragma unroll
                    for (int i = 0; i < kLowParts; ++i) v += slices[i][tid];
                    red[0][0][tid] = v;
                }
                __syncthreads();
            }
        }
        if (done && tid < kLowGroup && k0 + tid < kl) store(k0 + tid, &red[0][0][6 * tid]);
        __syncthreads();   // red and last are reused by the next task
    }
}

}  // namespace

hipError_t launch_lowfreq(const CurveGeom* d_geom, const int32_t* list, int nsmall, int nwide,
                          const CurveState* state, PointArrays pa, const PlanParams& pp,
                          void* power, int out_f64, WideAux* aux, hipStream_t s) {
    // a workgroup a curve in large batches, up to 16 (four are busy at the
    // common 5 frequencies per 1/baseline) where the device would be idle; 512
    // for a wide curve's slices.  Launches within kMaxLaunchItems
    const int bs = std::max(1, std::min(16, 2048 / std::max(nsmall, 1)));
    constexpr int bw = kLowSlots;
    constexpr int64_t kBlocks = kMaxLaunchItems / kLowNT;
    int s0 = 0, w0 = 0;
    while (s0 < nsmall || w0 < nwide) {
        const int ns = (int)std::min<int64_t>(nsmall - s0, kBlocks / bs);
        // wide curves follow the small ones in the list
        const int nw = s0 + ns < nsmall ? 0
                       : (int)std::min<int64_t>(nwide - w0, (kBlocks - (int64_t)ns * bs) / bw);
        const int f = ns > 0 ? s0 : nsmall + w0;
        const int32_t* l = list ? list + f : nullptr;
        WideAux* const x = aux ? aux + w0 : nullptr;
        const dim3 grid((unsigned)((int64_t)ns * bs + (int64_t)nw * bw));
        if (ns + nw == 0) return hipErrorInvalidValue;
        if (out_f64)
            hipLaunchKernelGGL((lowfreq_kernel<1>), grid, dim3(kLowNT), 0, s, d_geom, l, f, ns,
                               bs, bw, state, pa, pp, x, power);
        else
            hipLaunchKernelGGL((lowfreq_kernel<0>), grid, dim3(kLowNT), 0, s, d_geom, l, f, ns,
                               bs, bw, state, pa, pp, x, power);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        s0 += ns;
        w0 += nw;
    }
    return hipSuccess;
}

// one launch per 2^31 work-items of tiles
template <class F>
static hipError_t for_tile_chunks(int ntiles, F&& launch) {
    const int chunk = (int)(kMaxLaunchItems / kDirNT);
    for (int t0 = 0; t0 < ntiles; t0 += chunk) {
        launch(t0, std::min(chunk, ntiles - t0));
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_dirsum_custom(const CurveGeom* d_geom, const CurveState* state,
                                const int32_t* tile_curve, const int32_t* tile_first,
                                int ntiles, int ws, PointArrays pa, const PlanParams& pp,
                                const double* freqs, void* power, int out_f64, hipStream_t s) {
    return for_tile_chunks(ntiles, [&](int t0, int n) {
#define GLS_CUS(W, O)                                                                           \
    hipLaunchKernelGGL((dirsum_custom_kernel<W, O>), dim3(n), dim3(kDirNT), 0, s, d_geom, state, \
                       tile_curve + t0, tile_first + t0, pa, pp, freqs, power)
#define GLS_CUS_OUT(W)          \
    case W:                     \
        if (out_f64) GLS_CUS(W, 1); \
        else GLS_CUS(W, 0);     \
        break;
        switch (ws) {
            GLS_CUS_OUT(1)
            GLS_CUS_OUT(2)
            GLS_CUS_OUT(4)
            GLS_CUS_OUT(8)
        }
#undef GLS_CUS_OUT
#undef GLS_CUS
    });
}

hipError_t launch_dirsum(const CurveGeom* d_geom, const CurveState* state,
                         const int32_t* tile_curve, const int32_t* tile_first, int ntiles,
                         int ws, PointArrays pa, const PlanParams& pp, void* power, int out_f64,
                         hipStream_t s) {
    return for_tile_chunks(ntiles, [&](int t0, int n) {
#define GLS_DIR(W, O)                                                                    \
    hipLaunchKernelGGL((dirsum_kernel<W, O>), dim3(n), dim3(kDirNT), 0, s, d_geom, state, \
                       tile_curve + t0, tile_first + t0, pa, pp, power)
#define GLS_DIR_OUT(W)          \
    case W:                     \
        if (out_f64) GLS_DIR(W, 1); \
        else GLS_DIR(W, 0);     \
        break;
        switch (ws) {
            GLS_DIR_OUT(1)
            GLS_DIR_OUT(2)
            GLS_DIR_OUT(4)
            GLS_DIR_OUT(8)
        }
#undef GLS_DIR_OUT
#undef GLS_DIR
    });
}

}  // namespace gls
