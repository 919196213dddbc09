// Internal declarations shared by the libgls.so translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/gls.h"
#include "sizes.hpp"
#include "tiles.hpp"

namespace gls {

// ---------------------------------------------------------------------------
// error handling (thread-local message, integer status at the C ABI)
// ---------------------------------------------------------------------------
void set_error(const std::string& msg);
int fail(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);

#define GLS_HIP_TRY(expr)                                                     \
    do {                                                                      \
        hipError_t _e = (expr);                                               \
        if (_e != hipSuccess) return ::gls::hip_fail(_e, #expr);              \
    } while (0)

bool initialised();
int require_init();

// Descriptors as a launch argument (the first of its kernel), at most what the
// runtime takes beside the other arguments; device code reads them where the
// arguments lie, since indexing the parameter would copy it to scratch memory.
constexpr int kMetaArgWords = 224;
struct MetaArg {
    int4 w[kMetaArgWords];
};
#if defined(__HIP_DEVICE_COMPILE__)
__device__ inline const int4* meta_arg_words() {
    return (const int4*)__builtin_amdgcn_kernarg_segment_ptr();
}
#else
__device__ inline const int4* meta_arg_words() { return nullptr; }
#endif

// Asynchronous host-to-device copy of a plan's descriptors: as launch arguments
// where they fit, else through the library's page-locked staging ring
// (allocated by gls_init): the source is copied into the ring on the host and
// a kernel reads the ring, so the call never waits on the runtime's shared
// pageable staging buffer.  Falls back to a plain hipMemcpyAsync for blocks
// larger than half the ring.
hipError_t upload_async(void* dst, const void* src, size_t bytes, hipStream_t s);

// Device address and size of the static scratch array of the current device
// (gls_lomb_execute_static); GLS_E_NOT_INIT before gls_init.
constexpr size_t kScratchBytes = size_t(128) << 20;
int static_scratch(void** ptr);

// Device copy of the ES deconvolution table for (m, beta), uploaded once per
// process and kept until it ends (plans point at it; it is not part of the
// per-execute descriptors).
int es_table_device(int m, float beta, const float** out);

// library-owned streams (default priority) onto which an execute forks the
// independent size buckets of a plan; created on first use
constexpr int kAuxStreams = 3;
hipError_t aux_streams(hipStream_t* out);

constexpr int kMaxGrid = 1 << 24;   // largest grid n (cells)
constexpr int kMinGrid = 1 << 10;   // smallest grid n

// ---------------------------------------------------------------------------
// Inter-pass grid layout (pass 1 writes, pass 2 reads): the rows k1 of a
// grid in blocks of kRowBlock, each block stored row-block-major over the n2
// columns, A[(k1 / R) R n2 + u2 R + k1 % R] (R = kRowBlock).  A pass-1 column
// is then written as R x 8-byte segments and the rows of a pass-2 tile lie in
// one contiguous run per row block (DRAM pages are opened once per tile,
// not once per column).  A grid takes ceil(n1 / R) R n2 cells.  R = 8 (the
// pass-2 tile height of the survey's main buckets) measured 4% faster in pass
// 2 than R = 16 on the survey batch, with pass 1 unchanged.
#ifndef GLS_ROW_BLOCK
#define GLS_ROW_BLOCK 8
#endif
constexpr int kRowBlock = GLS_ROW_BLOCK;
static_assert((kRowBlock & (kRowBlock - 1)) == 0, "the row block is a power of two");
__host__ __device__ inline int64_t grid_cells(int n1, int p2) {
    return (int64_t)((n1 + kRowBlock - 1) / kRowBlock * kRowBlock) << p2;
}

// per-curve plan data (host computed, uploaded once per plan)
// ---------------------------------------------------------------------------
struct CurveGeom {
    int64_t obs;       // first observation index in t / a / b
    int64_t out;       // first output element
    int64_t pts;       // first point slot in the per-point workspace arrays
    int64_t bkt;       // first int of this curve's bucket table (2*(nb+1))
    int64_t grid;      // first float2 of this curve's grids (ngrids * grid_cells)
    double f0;
    double df;
    double n4inv;      // 4 / n: quarter turns per unit of the inter-pass twiddles
    double ybar_in;    // GLS_INPUT_WEIGHTED
    double yy_in;      // GLS_INPUT_WEIGHTED
    int32_t n_obs;
    int32_t nf;        // K, number of output frequencies
    int32_t n;         // grid size n = n1 * n2
    int32_t n1;        // pass-1 column length
    int32_t p2;        // log2 of pass-2 row length n2
    int32_t c1;        // pass-1 columns per tile
    int32_t kc;        // K/2, band centre index
    int32_t ci;        // index of the curve in the plan
    // per-curve constants of the pass kernels, computed on the host (a
    // division or square root in every thread would cost tens of VALU
    // instructions per block)
    float g_binv;      // log2(e) / b        (Gaussian spreading weight)
    float g_norm;      // 1 / sqrt(pi b)
    float g_bpi2;      // b pi^2             (Gaussian deconvolution)
    float ninv;        // 1 / n (FP32)
};

// written by the prep kernel
struct CurveState {
    double tref;       // time origin (min t)
    double ybar;
    double yy;
    double tspan;      // max t - min t
    double tmean;      // mean of the finite t (FP32-coordinate plans only)
    int32_t klow;      // leading frequencies with |f| tspan < kLowCycles
    int32_t pad;
};

// per-point workspace, indexed by CurveGeom::pts + j.  A node record holds a
// point's first cell U, the bits of its fractional offset fr in [0, 1) and of
// its modulated value (re, im) on one grid, so that pass 1 fetches a point
// with one 16-byte load.
struct PointArrays {
    int4* nd0;     // grid 0 (yw at f): node set 1, in bucket order
    int4* nd1;     // grid 1 (w at f): node set 1 (same U, fr as nd0)
    int4* nd2;     // grid 2 (w at 2f): node set 2
    float* w;      float* yw;      // prepared weights (direct method)
    double* dt;                    // t - tref (direct method)
};

struct PlanParams {
    int32_t m;
    int32_t mode;
    double reg_c;
    double reg_s;
    int32_t input_kind;
    int32_t method;
    int32_t kind;      // 0 = lomb, 1 = nfft
    int32_t window;    // GLS_WINDOW_*
    float es_beta;     // ES shape parameter
    int32_t fp32_coords;  // GLS_PRECISION_FP32: FP32 time offsets, cells and phases
    // ES: 1/psi_hat(xi) at xi = i / (2 kEsTab), i = 0 .. kEsTab + 1 (the
    // library's resident device copy for (m, beta), es_table_device)
    const float* es_deconv;
};

constexpr int kEsTab = 16384;   // ES deconvolution table intervals over xi in [0, 1/2]

// tiles of a size bucket (n1, p2): the caller's override (gls_tile_set), else
// the measured table compiled in, else the default rules (tiles.hpp)
struct BucketTiles {
    int c1, cr;
};
// whether this library has a kernel for the tile (tiles_gen.hpp lists them)
bool pass1_tile_built(int n1, int c1);
bool pass2_tile_built(int p2, int cr);

// launchers (defined in the kernel translation units)
// For the NFFT method the preparation of curves of more than kWidePrep points
// (wide curves) is spread over at most kWideBlocks blocks of kWideChunk points or
// a multiple of it each (a reduction, a counting and a scatter pass), with this
// per-curve record in the workspace: the raw-input weight constants and the bucket
// counts of both node sets, one after the other.
constexpr int kWidePrep = 16384;
constexpr int kWideChunk = 1024;
constexpr int kWideBlocks = 1024;
constexpr int kMaxBuckets = 4096;   // n2 / c1 <= 2^12
constexpr double kLowCycles = 3.0;
constexpr int kLowGroup = 4;     // low frequencies summed together by a workgroup
constexpr int kLowSlice = 2048;  // least points of a slice of a wide curve
constexpr int kLowSlots = 512;   // (group, slice) pairs a wide curve may have
// (the record also holds the FP64 sums of each (group, slice) pair of the
// low-frequency kernel, which the last workgroup of a group adds in slice
// order, and how many of a group's slices are done, cleared at every execute)
struct WideAux {
    double ymean;
    double s0inv;
    int32_t hist[2 * kMaxBuckets];    // points per bucket, both node sets
    int32_t taken[2 * kMaxBuckets];   // of those, slots that chunks have reserved
    double low[kLowSlots][6 * kLowGroup];
    int32_t low_done[kLowSlots / 2];   // (two slices or more: at most half the slots)
};
// Per-chunk partial reductions of a wide curve, one slot per chunk, combined in
// chunk order (so the result does not depend on block timing): least t and -t;
// raw input: sum and count of the finite y, sums of 1/dy^2 and of y/dy^2; last
// two, FP32 coordinates only: sum and count of the finite t.  syy: sum of (y -
// ymean - ybar)^2/dy^2 (raw input, from the counting pass).
struct WidePart {
    double v[8];
    double syy;
    double pad;
};
// small: nsmall curves, followed in the same list by the nwide wide ones (wide);
// aux: one WideAux per wide curve (NFFT method), or nullptr to prepare each
// wide curve in one block; part: min(kWideBlocks,
// ceil(wide_max_obs / kWideChunk)) WidePart slots per wide curve; wide_max_obs: the largest n_obs in the wide list;
// max_buckets: the most buckets (n2 / c1) of a curve (NFFT method); in_order:
// the list is 0, 1, 2 ..; meta (or nullptr): the descriptors, meta_words 16-byte
// words that are not in the workspace ws yet: the first launch takes them as an
// argument and stores them there
hipError_t launch_prep(const CurveGeom* d_geom, const int32_t* small, int nsmall,
                       const int32_t* wide, int nwide, CurveState* state,
                       const double* t, const void* a, const void* b,
                       PointArrays pa, int32_t* bkt, const PlanParams& pp,
                       int y_is_f32, WideAux* aux, WidePart* part, int wide_max_obs,
                       int max_buckets, bool in_order, const MetaArg* meta, int meta_words,
                       char* ws, hipStream_t s);
// work-items of one launch of the NFFT passes: the dispatch counts a grid's
// work-items in 32 bits, so a size bucket with more goes out in several
// launches over consecutive curves (max_launch_items(): this, or a smaller
// cap set by gls_launch_items_set)
constexpr int64_t kMaxLaunchItems = (int64_t)1 << 31;
int64_t max_launch_items();
// pass 1 stores a size bucket's grids non-temporally when they exceed this
// (the memory-side cache holds 256 MB)
constexpr int64_t kStreamStoreBytes = (int64_t)96 << 20;
// curves of one plan: the per-curve launches (preparation, low-frequency
// sums, top-k: at most 512 threads per curve) stay within kMaxLaunchItems
constexpr int kMaxPlanCurves = 1 << 22;
// GLS_SPREAD_AUTO spreads a curve in fixed point when it has at least one
// point per kFixedCellsPerPoint grid cells and its pass-1 columns hold at
// least kFixedMinColumn cells (on shorter columns the per-row counting and
// conversion cost more than the integer adds save)
constexpr int kFixedCellsPerPoint = 80;
constexpr int kFixedMinColumn = 64;
// pass 1 and 2 of one size bucket: bgeom holds the geometry of its ncurves
// curves, one after another (a block reads its curve's entry directly)
// (c1: the bucket's pass-1 tile, cr: its pass-2 tile; fix: fixed-point
// spreading; nts: non-temporal grid stores); pass 1's bkt points at the first
// curve's bucket offsets, which the others' follow, 2 (nb + 1) each
hipError_t launch_pass1(int n1, int c1, bool fix, bool nts, const CurveGeom* bgeom, int ncurves,
                        int ngrids, int p2, PointArrays pa, const int32_t* bkt, float2* grids,
                        const PlanParams& pp, hipStream_t s);
hipError_t launch_pass2_lomb(int p2, int cr, int n1, const CurveGeom* bgeom,
                             const CurveState* state, int ncurves, const float2* grids,
                             const PlanParams& pp, void* power, int out_f64,
                             hipStream_t s);
hipError_t launch_pass2_nfft(int p2, int cr, int n1, const CurveGeom* bgeom,
                             const CurveState* state, int ncurves, const float2* grids,
                             const PlanParams& pp, float2* out, hipStream_t s);
// direct sums: workgroups of kDirNT threads, one per tile; a wave takes
// kDirTile consecutive frequencies of a linear grid, or 64 of a frequency
// list, and ws waves (1, 2, 4 or 8) share them, so that a tile has 8 / ws times
// as many
constexpr int kDirNT = 512;
constexpr int kDirTile = 512;
hipError_t launch_dirsum(const CurveGeom* d_geom, const CurveState* state,
                         const int32_t* tile_curve, const int32_t* tile_first,
                         int ntiles, int ws, PointArrays pa,
                         const PlanParams& pp, void* power, int out_f64,
                         hipStream_t s);
// direct FP64 sums for a curve's lowest frequencies, f_k (t_max - t_min) <
// kLowCycles (all of them), overwriting the NFFT powers there; list (or
// nullptr: 0, 1, 2 ..): nsmall curves, then nwide ones, which split their points over workgroups when they
// have records (aux)
hipError_t launch_lowfreq(const CurveGeom* d_geom, const int32_t* list, int nsmall, int nwide,
                          const CurveState* state, PointArrays pa, const PlanParams& pp,
                          void* power, int out_f64, WideAux* aux, hipStream_t s);
hipError_t launch_dirsum_custom(const CurveGeom* d_geom, const CurveState* state,
                                const int32_t* tile_curve, const int32_t* tile_first,
                                int ntiles, int ws, PointArrays pa, const PlanParams& pp,
                                const double* freqs, void* power, int out_f64,
                                hipStream_t s);
hipError_t launch_gaussian_grid(const double* t, const double* y, int n_obs,
                                int ng, int m, double b, double tmin,
                                double tmax, double spp, float* grid,
                                hipStream_t s);
hipError_t launch_topk(const CurveGeom* d_geom, int ncurves, const float* power,
                       const uint8_t* mask, int k, float* top_power,
                       int32_t* top_index, hipStream_t s);

}  // namespace gls
