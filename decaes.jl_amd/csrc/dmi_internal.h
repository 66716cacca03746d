// Internal host/device interface between the C ABI (dmi_api.cpp) and the gfx950 kernels (dmi_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace dmi {

constexpr int kWave = 64;
constexpr int kMaxT2 = 64;        // one lane per T2 column
constexpr int kMaxEcho = 124;     // lane-per-state EPG window (ETL/2 + 2 states)
constexpr int kMaxAngles = 64;    // one lane per flip-angle grid point
constexpr int kTikhCache = 8;     // NNLSTikhonovRegProblemCache size (src/lsqnonneg.jl:396)
constexpr int kLcurveCap = 32;    // L-curve cache entries per voxel: at most 28 are used (4 + 24 bracket moves)
// legacy = true: interpolating splines of at most 64 points (the flip-angle grid; the chi2 doubling search has at
// most 2 + kLegacyMaxDoublings), knots and coefficients in LDS
constexpr int kSplineMaxPts = 64;
constexpr int kSplineKnots = kSplineMaxPts + 8;                 // m + k + 1 <= 68, rounded up to keep 16-byte alignment
constexpr int kSplineLds = kSplineKnots + kSplineMaxPts;        // doubles
constexpr int kLegacyMaxDoublings = 24;                         // chi2 legacy: mu <= 1e-3 * 2^24 (2^24 + 1 samples)
constexpr long long kSplineMaxSamples = (1ll << 24) + 1;        // longest sample grid a legacy scan walks

// Column stride of the column-major bases in device memory (grid bases, fixed basis, the voxel's basis): m rounded
// up to even, so every column starts 16-byte aligned and is copied into LDS with 16-byte global-to-LDS loads.
__host__ __device__ inline int basis_ld(int m) { return (m + 1) & ~1; }

// Static scratch of the allocation-free entry point, in doubles: a header (launch counters), the T2 and angle grids,
// four grid-basis arrays at the device limits (row-major As, dAs; column-major AsT, dAsT), a voxel-list chunk
// (int64) and the per-workgroup slots of the voxel kernel.
constexpr int64_t kNoAllocHeader = 32;
constexpr int64_t kNoAllocGrid = 3 * 64;
constexpr int64_t kNoAllocBasis = (int64_t)kMaxAngles * kMaxT2 * kMaxEcho;   // kMaxEcho is even: basis_ld = m
constexpr int64_t kNoAllocVox = 262144;                                      // voxels selected per chunk
// 40 MiB of slots: at 56 x 60 they hold 1254 voxels, at 64 x 64 1057, of the 2048 the register-resident kernel keeps resident
constexpr int64_t kNoAllocSlots = 5242880;
constexpr int64_t kNoAllocOffGrid = kNoAllocHeader;
constexpr int64_t kNoAllocOffBasis = kNoAllocOffGrid + kNoAllocGrid;
constexpr int64_t kNoAllocOffVox = kNoAllocOffBasis + 4 * kNoAllocBasis;
constexpr int64_t kNoAllocOffRedo = kNoAllocOffVox + kNoAllocVox;                // the chunk's voxels left to the second kernel
constexpr int64_t kNoAllocOffSlots = kNoAllocOffRedo + kNoAllocVox;
constexpr int64_t kNoAllocDoubles = kNoAllocOffSlots + kNoAllocSlots;
constexpr int kNoAllocMaxDevices = 64;

enum StatusBits : int {
    kStatusNnlsMaxIter = 2,
};

enum VoxelMode : int { kModeSearch = 0, kModeB1 = 1, kModeFixed = 2 };

struct GridParams {
    int m, n, K;
    int fp32;             // 1: FP32 recursion (mixed precision)
    int general;          // 1: RefConAngle != 180 (general refocusing train)
    double beta;          // RefConAngle
    double E1;            // exp(-(TE/2)/T1)
    const double *E2;     // n: exp(-(TE/2)/T2_j)
    const double *alphas; // K
    double *As;           // K x m x n, row-major per angle
    double *dAs;          // K x m x n or nullptr
    double *AsT;          // K x n columns of stride basis_ld(m) (column-major per angle)
};

struct T2mapParams {
    int m, n, K, mineval, reg, mode, general;
    int fp32;             // 1: FP32 EPG recursion for the voxel basis (mixed precision)
    int lda, mw;          // workspace: mw = m + n rows, column-major; rows [0, rl) in LDS with column stride lda
    int rl, gld;          // rows [rl, mw) in the workgroup's global slot, column stride gld (rl >= mw: all in LDS)
    int rs;               // register-resident solves with rs rows per lane (a size class), or 0: memory-resident
    int save_resnorm, save_decaycurve, save_regparam, save_basis;
    int legacy;           // legacy = true: spline surrogate for the flip angle, chi2 doubling search
    int64_t V;            // voxels in the volume
    int64_t nvox;         // voxels above threshold (with nvox_dev: an upper bound, the length of the voxel list)
    const unsigned int *nvox_dev;  // or nullptr; else the count of voxels above threshold, read on the device
    double E1, beta, chi2factor, noiselevel, setflip;
    const double *image;  // (V, m) column-major
    const int64_t *vox;   // nvox linear indices
    unsigned int *counter;
    const double *E2;     // n
    const double *logT2;  // n
    const double *alphas; // K
    const double *AsT;    // K grid bases, n columns of stride basis_ld(m) each
    const double *dAsT;   // d/dalpha, same layout
    const double *Afixed; // the SetFlipAngle basis, n columns of stride basis_ld(m)
    const double *As;     // K grid bases, row-major m x n (the register-resident kernel solves on these)
    const double *AfixedR;// the SetFlipAngle basis, row-major m x n
    int64_t *redo;        // register-resident kernel: voxels left to the memory-resident one
    unsigned int *redo_count;
    const double *alpha_in;
    double *scratch;      // per-workgroup slots
    int64_t slot_stride;  // doubles per slot
    double *dist, *gdn, *ggm, *gva, *fnr, *snr, *alpha, *resnorm, *decaycurve, *mu, *chi2f, *decaybasis;
    unsigned long long *counters; // [0] fp64 flops, [1] nnls solves, [2] fp32 flops
    int *status;          // [0] kStatus* flags, [1] voxels put on the redo list
};

// Device words of one T2map call, together so that one fill clears them and one copy reads them: the smallest calls are
// some 20 microseconds of kernels, and a further copy to the host costs them about 10 (median of calls of 1 to 256 voxels
// with 16 to 64 bins: 3% of the call).
struct CallWords {
    unsigned long long counters[4];  // T2mapParams.counters, [3] voxels without outputs
    int status[4];                   // T2mapParams.status
    unsigned counter[4];             // voxels selected, then the launches' own (t2map_launch_raw)
};
static_assert(sizeof(CallWords) == 64 && sizeof(CallWords) <= sizeof(double) * kNoAllocHeader, "");

struct T2partParams {
    int n;
    int64_t V;
    int sp0, sp1, mp0, mp1;   // inclusive 0-based window ranges
    const double *logT2;      // n
    const double *weights;    // n or nullptr (sigmoid)
    const double *dist;
    double *sfr, *sgm, *mfr, *mgm;
};

// LDS of one register-resident workgroup (dmi_nnls_reg.h), offsets and total in doubles: the solution x at 0, the
// right-hand side, the Tikhonov cache's mu, norms and residuals, and the solver's region: the triangular factor packed
// by column (position j's rows [0, j] at T + j (j + 1) / 2), a column in transit, three vectors of kRegStage rows. GCV's Gram
// matrix (odd column stride) takes the region between solves.
constexpr int kRegStage = 144;
struct RegLayout {
    int b, c, T, tmp, stg, total;
};
__host__ __device__ inline RegLayout reg_layout(int m, int n, bool gram) {
    RegLayout l;
    const int ne = (n + 1) & ~1, N = m < n ? m : n;
    l.b = ne;
    l.c = l.b + ((m + n + 1) & ~1);
    l.T = l.c + 3 * kTikhCache;
    l.tmp = l.T + ((n * (n + 1) / 2 + 1) & ~1);
    l.stg = l.tmp + ne;
    l.total = l.stg + 3 * kRegStage;
    const int g = l.T + ((N * (N | 1) + 1) & ~1);
    if (gram && l.total < g) l.total = g;
    // the triangular solve reads 64 rows from the start of every column
    const int r = l.T + n * (n - 1) / 2 + 64;
    if (l.total < r) l.total = r;
    return l;
}

int t2map_lda(int m, int n);
// LDS of one voxel workgroup; K (the flip-angle grid size of the launch) takes no LDS; legacy adds the spline knots
// and coefficients
size_t t2map_lds_bytes(int m, int n, int lda, int K, int legacy);
int64_t t2map_slot_doubles(int m, int n, int gld);

hipError_t launch_grid_basis(const GridParams &p, hipStream_t s);
hipError_t launch_transpose(const double *src, double *dst, int m, int n, int K, hipStream_t s);
// voxels I in [v0, v1) with image[I] > thr (image[I] is echo 1 of voxel I)
hipError_t launch_select(const double *image, int64_t v0, int64_t v1, double thr, int64_t *vox, unsigned int *count,
                         hipStream_t s);
// fills bytes / 4 32-bit words with v
hipError_t launch_fill(void *p, size_t bytes, unsigned int v, hipStream_t s);
// This device's address of the static scratch (looked up once per device with the device made current).
hipError_t noalloc_scratch(int device, double **ptr);
hipError_t launch_t2map(const T2mapParams &p, int grid, size_t lds, hipStream_t s);
hipError_t launch_t2part(const T2partParams &p, hipStream_t s);
// Float32 <-> Float64 element-wise conversion (Float32 entry points)
hipError_t launch_widen(const float *src, double *dst, int64_t n, hipStream_t s);
hipError_t launch_narrow(const double *src, float *dst, int64_t n, hipStream_t s);
// split: of the voxel kernel built for the split schedule (rows beyond an LDS cutoff in the global slot)
hipError_t t2map_occupancy(int reg, int legacy, int *blocks_per_cu, size_t lds, bool split = false);
// the voxel kernel of the split schedule, from dmi_kernels_split.hip (launch_t2map calls it when p.rl < p.mw)
hipError_t launch_t2map_split(const T2mapParams &p, int grid, size_t lds, hipStream_t s);
hipError_t t2map_occupancy_split(int reg, int legacy, int *blocks_per_cu, size_t lds);
// the register-resident voxel kernel of size class S (kRegClasses), one unit per class from dmi_kernels_reg.hip
// Size classes of the register-resident kernel. Solves without regularization have m rows. A Tikhonov solve's window holds
// the m rows and the appended rows whose columns have left the active set again, and up to 3 registers are lost to the
// window's alignment; a solve that outgrows its class sends the voxel to the memory-resident kernel. Sixteen rows beyond m
// are enough for chi2 and mdp (no voxel of 524,288 with 32, 48, 56 and 64 echoes and 40 to 64 bins outgrew them) and gcv
// (one). The L-curve's solves at low mu remove more columns: with sixteen 9, 17 and 24 of 131,072 voxels each at 48, 56 and
// 64 echoes did, all but two of them with more than 40 bins, with 20 or more none of 655,360. One such voxel doubles the time of
// a call of a few hundred voxels (64 voxels of 56 x 64: 11.0 ms, 5.6 in the next class) and adds 6 ms to a 240x240 slice
// (56 x 60: 87.0 ms, 81.1; 48 x 60: 78.8 and 74.5), so those trains take 20 where a class holds them; with up to 40
// bins the larger class is the slower one (48 x 40: 51.3 ms, 52.4). 61 to 64 echoes keep 16 rows: their class is the largest.
constexpr int kRegClasses[] = {48, 64, 72, 80};
inline int t2map_reg_class(int m, int n, int reg) {
    const bool wide = reg == 1 && n > 40;  // the L-curve
    for (int extra : {wide ? 20 : 16, 16})
        for (int s : kRegClasses)
            if (s >= m + (reg == 0 ? 0 : extra)) return s;
    return 0;
}
hipError_t t2map_occupancy_reg(int rs, int reg, int *blocks_per_cu, size_t lds);
template <int S> hipError_t launch_t2map_reg(const T2mapParams &p, int grid, size_t lds, hipStream_t s);
template <int S> hipError_t t2map_reg_occupancy(int reg, int *blocks_per_cu, size_t lds);

}  // namespace dmi
