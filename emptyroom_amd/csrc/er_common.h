// er_common.h -- definitions shared by the host runtime and the gfx950
// kernels: the Widom point stream, the per-framework device view and the
// work-item descriptor of the tiled energy kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace er {

// ---------------------------------------------------------------------------
// Widom point stream.  Philox4x32-10 (Salmon et al., SC'11) keyed by the job
// seed; insertion i uses counter (lo(i), hi(i), stream, 0) and maps the first
// three output words to (w + 1) * 2^-32, i.e. fractional coordinates in
// (0, 1] like curand_uniform_double in src/doHenry.h:53-55.  Stream 0 is the
// direct-sum Widom run, stream 1 the grid-interpolated one.
// ---------------------------------------------------------------------------
__host__ __device__ inline void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                              uint32_t k0, uint32_t k1, uint32_t out[4]) {
    const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;
    const uint32_t W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        uint64_t p0 = (uint64_t)M0 * c0;
        uint64_t p1 = (uint64_t)M1 * c2;
        uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
        uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c0 = n0;
        c1 = (uint32_t)p1;
        c2 = n2;
        c3 = (uint32_t)p0;
        k0 += W0;
        k1 += W1;
    }
    out[0] = c0;
    out[1] = c1;
    out[2] = c2;
    out[3] = c3;
}

__host__ __device__ inline void widom_point(uint64_t seed, uint32_t stream, uint64_t i,
                                            double f[3]) {
    uint32_t w[4];
    philox4x32_10((uint32_t)i, (uint32_t)(i >> 32), stream, 0u, (uint32_t)seed,
                  (uint32_t)(seed >> 32), w);
    const double inv2_32 = 2.3283064365386962890625e-10;  // 2^-32, exact
    f[0] = ((double)w[0] + 1.0) * inv2_32;
    f[1] = ((double)w[1] + 1.0) * inv2_32;
    f[2] = ((double)w[2] + 1.0) * inv2_32;
}

// ---------------------------------------------------------------------------
// Device data of one uploaded framework.
// ---------------------------------------------------------------------------

// Pair parameters of one (guest, framework-atom-type) combination after
// Lorentz-Berthelot mixing: sig2 = sigma_ij^2, eps4 = 4 eps_ij.  rclose is the
// distance below which a pair is evaluated on the FP64 path.
// c3 = -eps4 sigma^6 and c6 = eps4 sigma^12 scale the sums of r^-6 and r^-12.
struct alignas(16) TypeParams {
    double sig2;
    double eps4;
    double rclose;
    double c3, c6;
    double pad;
};

// Work kinds of the tiled energy kernel.
enum JobKind : int { JOB_GRID = 0, JOB_WIDOM = 1 };
// Output modes: FP32 grid (FP32 far-pair LJ, FP64 close pairs and
// accumulation), FP64 grid (every pair on the FP64 path), in-cutoff count.
enum OutMode : int { OUT_F32 = 0, OUT_F64 = 1, OUT_COUNT = 2 };

// One job of the tiled energy kernel: a grid over the unit cell or the Widom
// insertions of one framework.  Plain-old-data, copied to device memory.
struct JobDev {
    double t[9];        // fractional -> Cartesian, row-major (src/Framework.cc:124-132)
    double rc2;         // r_c^2
    double rc;          // r_c
    double min_r2;      // r^2 clamp: 1e-24 grid, 1e-32 Widom
    const double4 *near;      // image atoms near the cell, grouped by type (x, y, z, r_FP64)
    const int *type_begin;    // ntypes + 1 offsets into near
    const TypeParams *types;  // ntypes
    int ntypes;
    int kind;           // JobKind
    int mode;           // OutMode
    int interp;         // grid: the far field of 2 x 2 x 2 tiles from nodes (see grid_block)
    // grid
    int n[3];           // grid points per axis, endpoints included
    int tile[3];        // tile extent in points
    int ntiles[3];      // tiles per axis
    int region[3];      // tiles per region (work item) per axis
    int nregions[3];    // regions per axis
    void *out;          // float*, double* or uint32_t* by mode; index k + j*nz + i*ny*nz
    // Widom
    int nbins[3];       // insertion bins per fractional axis
    int parts;          // > 0: an energy is summed in so many parts (see eval_range)
    int shared;         // with parts: they are shared out to waves (see k_parts), and an
                        // item is a quarter of a cell, or with 2 parts a cell
    int pad0;
    const uint32_t *sorted;     // insertion indices ordered by bin
    const uint32_t *bin_start;  // nbins_total + 1 offsets into sorted
    uint64_t seed;
    uint32_t stream;
    uint32_t pad2;
    double *e_out;      // FP64 energy per insertion index
    double sat_e;       // > 0: stop at a partial energy this high (800 T; see k_tiles)
    double fs_floor;    // far and shell pairs (beyond r_FP64 of every point) add at least
                        // -fs_floor * eps_ij each (<= 1)
    // point boxes (fractional half-extents per axis): a full grid tile's or a
    // bin's, and a full wave quadrant's of a grid tile; a partial one lies in
    // the full one centred on it
    double cell_box[3];
    double wave_box[3];
    // radii of the spheres around them, with the classification margin; inv[d]
    // is the fractional step of a grid point (1 / (n - 1)) or a bin (1 / nbins)
    double cell_R, wave_R;
    double inv[3];
    // scheduling
    long long item_begin;  // first global work item of this job
    long long n_items;     // grid tiles or Widom bins of this job in this launch
    long long local0;      // first tile / bin of the job covered by this launch
};

// One Widom binning job: insertion points of (seed, stream) sorted into a
// regular grid of fractional bins.  Plain-old-data; kernels take an array.
// A job of many bins is sorted in two steps: into `ngroups` groups of `group`
// consecutive bins, then each group into its bins (group = 1: one step).
struct BinJob {
    uint64_t seed;
    uint64_t n;            // insertions
    uint32_t stream;
    int nb[3];             // bins per fractional axis
    int group;             // bins per group
    int ngroups;           // ceil(bins / group)
    uint32_t *count;       // group counts (zeroed by k_bin_zero)
    uint32_t *start;       // nbins + 1 exclusive prefix sums
    uint32_t *cursor;      // ngroups + 1 fill cursors; a group's end after the scatter
    uint32_t *sorted;      // n insertion indices, grouped by bin
    uint2 *tmp;            // two steps: n (bin in its group, insertion) pairs, grouped
    long long block0;      // first binning block of this job in a launch
    long long gblock0;     // first second-step block (one per group) of this job
};

// Slot `at` of a run that begins at `begin`.  In 64 bits: a job may have 2^32 - 1
// insertions, and the slots a wave looks at past the end of its last run lie beyond.
__host__ __device__ inline uint64_t run_slot(uint32_t begin, uint64_t at) { return begin + at; }

// Kernel launch geometry.
constexpr int kWG = 256;      // threads per workgroup (4 wave64)
constexpr int kMaxSeg = 64;   // list segments per fill pass
constexpr int kMaxTypes = 64; // pair types a region sub-list can index
constexpr int kBinWG = 1024;      // threads of a binning scatter block
constexpr int kBinChunkMax = 16384;  // insertions per binning block, at most
constexpr int kBinGroups = 1024;  // groups of a Widom job that is binned in two steps
constexpr int kBinDirectMax = 4096;  // bins up to which a job is binned in one step
constexpr int kBinGroupMax = 15360;  // bins a group may hold (the second step's LDS counts)
constexpr int kBinLdsKeys = 7168;    // keys a binning block histograms in LDS (28 KiB), and so
                                     // most groups of a job; bins accordingly:
constexpr long long kBinsMax = (long long)kBinLdsKeys * kBinGroupMax;
constexpr int kRegionRecords = 8192;  // entries of one workgroup's region sub-list (near-list
                                      // indices, 32 KiB)
constexpr int kBlockList = 6144;  // of these, entries of a block's list (see grid_block)
// Margin (Angstrom) applied to every list classification so that FP64 rounding
// of radii and distances can never misclassify a pair.
constexpr double kMargin = 1e-6;
constexpr int kNodes = 8;        // Chebyshev nodes per axis of a block of 2 x 2 x 2 grid tiles
constexpr double kNodeReach = 8.0;  // far atoms of a block lie at least this many times its
                                    // half-extent away from every point
constexpr int kNodeRecords = kNodes * kNodes * kNodes * 8 / 32;  // LDS records the values take
constexpr long long kNodeMinBlocks = 1024;  // see use_nodes
constexpr double kNodeMinFar = 120.0;
// cells up to which the points of a wave are shared by eight / four / two waves; waves
// up to which jobs of a batch do so (see batch_create)
constexpr long long kPartCells8 = 128, kPartCells4 = 320, kPartCells2 = 512;
constexpr double kPartWaves = 1900.0;
constexpr long long kMinGridItems = 2048;  // regions per grid before regions shrink

}  // namespace er
