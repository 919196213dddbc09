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

constexpr int NT = 256;

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
// 1e-4.  These few frequencies are recomputed by direct sums with FP64
// phases and FP64 accumulation.
// Grid (curve, group of 4 frequencies), the groups strided over the
// frequencies from kbegin on: each wave of a block takes one frequency and
// its 64 lanes stride over the curve's points (FP64 phases, FP64 sums), then
// reduce by shuffles.  A block stops at the first group past the curve's low
// frequencies, so however many there are (fine grids have hundreds), every
// one is covered.
constexpr int kLowPerBlock = NT / kWave;
constexpr int kLowGroups = kLowMax / kLowPerBlock;   // blocks per curve

// the six FP64 sums of frequency k over the curve's points and its power
template <int OUT, bool WIDE, int BT, int LANES>
__device__ __forceinline__ void lowfreq_one(const CurveGeom& G, const CurveState& st,
                                            const PointArrays& pa, const PlanParams& pp, int k,
                                            int tid, int lane, int N, double (*red)[6],
                                            void* __restrict__ out) {
    const double f = G.f0 + (double)k * G.df;
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int j = lane; j < N; j += LANES) {
        const double x = f * pa.dt[G.pts + j];
        double sn, cs;
        sincospi(2.0 * (x - rint(x)), &sn, &cs);
        const double w = pa.w[G.pts + j], yw = pa.yw[G.pts + j];
        acc[0] += w * cs;
        acc[1] += w * sn;
        acc[2] += w * (cs * cs - sn * sn);
        acc[3] += w * (2.0 * cs * sn);
        acc[4] += yw * cs;
        acc[5] += yw * sn;
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) acc[q] = wave_sum(acc[q]);
    if (WIDE) {
        const int wv = tid / kWave;
        if ((tid & (kWave - 1)) == 0)
            for (int q = 0; q < 6; ++q) red[wv][q] = acc[q];
        __syncthreads();
        if (tid == 0)
            for (int w = 1; w < BT / kWave; ++w)
                for (int q = 0; q < 6; ++q) acc[q] += red[w][q];
        __syncthreads();   // red is reused by the block's next frequency
    }
    if (lane == 0) {
        const double P = gls_power(acc[0], acc[1], acc[2], acc[3], acc[4], acc[5], st.yy,
                                   st.ybar, pp.mode, pp.reg_c, pp.reg_s);
        if (OUT == 0) ((float*)out)[G.out + k] = (float)P;
        else ((double*)out)[G.out + k] = P;
    }
}

// WIDE: one frequency per 1024-thread block, all its lanes over the points
// (long curves: 16 waves per frequency hide the FP64 latency).
constexpr int kLowWideNT = 1024;
// LOOP: the block strides on over the grid (gridDim.y groups apart) until it
// passes the curve's low run; without it, one group per block (fewer live
// registers: the common case, launched with enough groups for kLowMax
// frequencies, and LOOP launches take any frequencies after those)
template <int OUT, bool WIDE, bool LOOP>
__global__ __launch_bounds__(WIDE ? kLowWideNT : NT) void lowfreq_kernel(
    const CurveGeom* __restrict__ geom, const int32_t* __restrict__ list,
    const CurveState* __restrict__ state, PointArrays pa, PlanParams pp, int kbegin,
    void* __restrict__ out) {
    constexpr int BT = WIDE ? kLowWideNT : NT;     // threads per block
    __shared__ double red[BT / kWave][6];
    constexpr int FPB = WIDE ? 1 : kLowPerBlock;   // frequencies per block
    constexpr int LANES = WIDE ? BT : kWave;       // lanes per frequency
    const int tid = threadIdx.x;
    const int lane = tid % LANES;
    const int c = list[blockIdx.x];
    const CurveGeom& G = geom[c];
    const CurveState& st = state[c];
    int first = kbegin + (int)blockIdx.y * FPB;
    do {
        // frequency k is low if it and every frequency before it span fewer
        // than kLowCycles cycles over the baseline (the leading run of the grid)
        if (first >= G.nf) return;
        if (fabs(G.f0 + (double)first * G.df) * st.tspan >= kLowCycles) return;
        const int k = first + tid / LANES;
        bool active = k < G.nf;
        for (int q = first; q <= k && active; ++q)
            active = fabs(G.f0 + (double)q * G.df) * st.tspan < kLowCycles;
        // uniform per frequency: whole waves (or the block) exit; later groups
        // of this block lie further along the grid, past the run as well
        if (!active) return;
        lowfreq_one<OUT, WIDE, BT, LANES>(G, st, pa, pp, k, tid, lane, G.n_obs, red, out);
        first += (int)gridDim.y * FPB;
    } while (LOOP);
}

// Wide curves with a WideAux record: grid (wide curve, frequency, part);
// each of the kLowSplit workgroups of a low frequency sums one slice of the
// points and stores its six FP64 sums in the record; the last to finish adds
// the slices in order and forms the power.  Frequencies past the low run exit at once.
template <int OUT>
__global__ __launch_bounds__(kLowWideNT) void lowfreq_split_kernel(
    const CurveGeom* __restrict__ geom, const int32_t* __restrict__ list,
    const CurveState* __restrict__ state, PointArrays pa, PlanParams pp,
    WideAux* __restrict__ aux, void* __restrict__ out) {
    __shared__ double red[kLowWideNT / kWave][6];
    const int tid = threadIdx.x;
    const int k = blockIdx.y;
    const int c = list[blockIdx.x];
    const CurveGeom& G = geom[c];
    const CurveState& st = state[c];
    if (k >= min(G.nf, kLowMax)) return;
    const double f = G.f0 + (double)k * G.df;
    if (fabs(f) * st.tspan >= kLowCycles) return;   // the test of lowfreq_kernel<OUT, true>
    const int N = G.n_obs;
    const int per = (N + kLowSplit - 1) / kLowSplit;
    const int j0 = (int)blockIdx.z * per;
    const int j1 = min(N, j0 + per);
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int j = j0 + tid; j < j1; j += kLowWideNT) {
        const double x = f * pa.dt[G.pts + j];
        double sn, cs;
        sincospi(2.0 * (x - rint(x)), &sn, &cs);
        const double w = pa.w[G.pts + j], yw = pa.yw[G.pts + j];
        acc[0] += w * cs;
        acc[1] += w * sn;
        acc[2] += w * (cs * cs - sn * sn);
        acc[3] += w * (2.0 * cs * sn);
        acc[4] += yw * cs;
        acc[5] += yw * sn;
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) acc[q] = wave_sum(acc[q]);
    const int wv = tid / kWave;
    if ((tid & (kWave - 1)) == 0)
        for (int q = 0; q < 6; ++q) red[wv][q] = acc[q];
    __syncthreads();
    if (tid != 0) return;
    for (int w = 1; w < kLowWideNT / kWave; ++w)
        for (int q = 0; q < 6; ++q) acc[q] += red[w][q];
    WideAux& X = aux[blockIdx.x];
    for (int q = 0; q < 6; ++q) X.low[k][blockIdx.z][q] = acc[q];
    __threadfence();
    if (atomicAdd(&X.low_done[k], 1) != kLowSplit - 1) return;
    __threadfence();
    // the slices in order, so the sum does not depend on which finished first
    double sm[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int z = 0; z < kLowSplit; ++z)
        for (int q = 0; q < 6; ++q)
            sm[q] += __hip_atomic_load(&X.low[k][z][q], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
    const double P = gls_power(sm[0], sm[1], sm[2], sm[3], sm[4], sm[5], st.yy, st.ybar,
                               pp.mode, pp.reg_c, pp.reg_s);
    if (OUT == 0) ((float*)out)[G.out + k] = (float)P;
    else ((double*)out)[G.out + k] = P;
}

}  // namespace

hipError_t launch_lowfreq(const CurveGeom* d_geom, const int32_t* small, int nsmall,
                          const int32_t* wide, int nwide, const CurveState* state,
                          PointArrays pa, const PlanParams& pp, void* power, int out_f64,
                          WideAux* aux, hipStream_t s) {
    // the first kLowMax frequencies: one group per block; any further ones
    // (fine grids): a few looping blocks per curve, which exit at once when
    // the low run ends before kLowMax
    constexpr int kMoreGroups = 4;
#define GLS_LOW(OUTV, W, L, GRID, NTH, LIST, KB)                                                \
    hipLaunchKernelGGL((lowfreq_kernel<OUTV, W, L>), GRID, dim3(NTH), 0, s, d_geom, LIST, state, \
                       pa, pp, KB, power)
    if (nsmall > 0) {
        if (out_f64) {
            GLS_LOW(1, false, false, dim3(nsmall, kLowGroups), NT, small, 0);
            GLS_LOW(1, false, true, dim3(nsmall, kMoreGroups), NT, small, kLowMax);
        } else {
            GLS_LOW(0, false, false, dim3(nsmall, kLowGroups), NT, small, 0);
            GLS_LOW(0, false, true, dim3(nsmall, kMoreGroups), NT, small, kLowMax);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (nwide > 0 && aux != nullptr) {
        // the first kLowMax frequencies split over kLowSplit workgroups each
        // (one accumulator slot per frequency in the record)
        const dim3 grid(nwide, kLowMax, kLowSplit);
        if (out_f64)
            hipLaunchKernelGGL((lowfreq_split_kernel<1>), grid, dim3(kLowWideNT), 0, s, d_geom,
                               wide, state, pa, pp, aux, power);
        else
            hipLaunchKernelGGL((lowfreq_split_kernel<0>), grid, dim3(kLowWideNT), 0, s, d_geom,
                               wide, state, pa, pp, aux, power);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    } else if (nwide > 0) {
        if (out_f64) GLS_LOW(1, true, false, dim3(nwide, kLowMax), kLowWideNT, wide, 0);
        else GLS_LOW(0, true, false, dim3(nwide, kLowMax), kLowWideNT, wide, 0);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (nwide > 0) {
        if (out_f64) GLS_LOW(1, true, true, dim3(nwide, kMoreGroups), kLowWideNT, wide, kLowMax);
        else GLS_LOW(0, true, true, dim3(nwide, kMoreGroups), kLowWideNT, wide, kLowMax);
    }
#undef GLS_LOW
    return hipGetLastError();
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
