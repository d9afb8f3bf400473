// er_kernels.hip -- gfx950 kernels for the guest-framework Lennard-Jones
// energy grid (src/computegridsheet.h:30-99) and Widom insertion
// (src/doHenry.h:29-135).
//
// Layout in HBM, per framework:
//   atoms   : AtomDev[n]           fractional coordinates + type, grouped by type
//   near    : double4[]            Cartesian FP64 image atoms T(f_a + n) that can
//                                  lie within r_c of the unit cell, grouped by type,
//                                  reference enumeration order inside a type
//   types   : TypeParams[ntypes]   mixed sigma^2, 4 eps, FP64 switch radius
// The tiled kernel (k_tiles) is persistent: each workgroup takes work items
// (a region of grid tiles or of Widom bins) from a device counter, gathers the
// near-list indices of the region's candidates into its scratch slice, then
// per tile (a box of grid points, or one bin's insertions) keeps the image
// atoms within r_c + R_tile in LDS, split into far records (inside the cutoff
// and beyond the FP64 switch radius for every point: no test, FP32
// reciprocal powers), shell records (cutoff test) and near records (FP64
// pair arithmetic).  Every lane evaluates its points against the LDS list
// with the record broadcast from LDS and the pair parameters in registers;
// in FP32 and FP64 grid tiles each wave first re-sorts the shell records
// against its own, smaller point box.  A Widom bin of at most one chunk of
// insertions keeps their points and partial energies in registers across
// its LDS passes.  Fine FP32 grids take the far field of blocks of tiles from
// interpolation nodes (grid_block).  Jobs of a few hundred cells sum an energy in
// parts, which several waves make at once where the device is idle (k_parts).
#include "er_kernels.h"

#include <float.h>
#include <limits.h>

#include <type_traits>

// No implicit multiply-add contraction in this file: every FMA below is
// written out, so the arithmetic of a pair (and so every energy) is fixed by
// the source and does not depend on how the compiler schedules one template
// instance against another (1, 2 or 4 points per lane give bit-identical
// energies for the same list).  Coordinates (frac_to_cart) then round like
// the oracle's and the reference's host code: separate products and sums.
#pragma clang fp contract(off)

namespace er {

namespace {

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The same pointer, unknown to the compiler: what is read through it is read
// again instead of being held in registers around a loop.
template <class T>
__device__ __forceinline__ T *reread(T *p) {
    asm volatile("" : "+s"(p));
    return p;
}

__device__ __forceinline__ int lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ void frac_to_cart(const double *t, double fx, double fy, double fz,
                                             double &x, double &y, double &z) {
    x = t[0] * fx + t[1] * fy + t[2] * fz;
    y = t[3] * fx + t[4] * fy + t[5] * fz;
    z = t[6] * fx + t[7] * fy + t[8] * fz;
}

// ---------------------------------------------------------------------------
// Near-image list
// ---------------------------------------------------------------------------

struct NearItem {
    bool valid;
    int type;
    double gx, gy, gz;  // fractional position of the image atom
};

__device__ __forceinline__ NearItem near_item(const NearPlan &p, int blk, int tid) {
    NearItem it;
    it.valid = false;
    int t = 0;
    while (t + 1 < p.ntypes && p.type_block0[t + 1] <= blk) ++t;
    it.type = t;
    const int a0 = p.type_atom0[t];
    const int cnt = p.type_atom0[t + 1] - a0;
    const long long q = (long long)(blk - p.type_block0[t]) * kWG + tid;
    if (cnt <= 0 || q >= (long long)cnt * p.n_images) return it;
    const int m = (int)(q / cnt);
    const int a = a0 + (int)(q % cnt);
    const int nb = 2 * p.rep[1] + 1, nc = 2 * p.rep[2] + 1;
    const int ii = m / (nb * nc) - p.rep[0];
    const int jj = (m / nc) % nb - p.rep[1];
    const int kk = m % nc - p.rep[2];
    const AtomDev at = p.atoms[a];
    // src/computegridsheet.h:61-63
    it.gx = at.fx + 1.0 * ii;
    it.gy = at.fy + 1.0 * jj;
    it.gz = at.fz + 1.0 * kk;
    it.valid = it.gx >= -p.ext[0] && it.gx <= 1.0 + p.ext[0] && it.gy >= -p.ext[1] &&
               it.gy <= 1.0 + p.ext[1] && it.gz >= -p.ext[2] && it.gz <= 1.0 + p.ext[2];
    return it;
}

__global__ __launch_bounds__(kWG) void k_near_count(NearPlan p, uint32_t *block_count) {
    __shared__ int s_w[kWG / 64];
    const int tid = threadIdx.x;
    NearItem it = near_item(p, blockIdx.x, tid);
    uint64_t m = __ballot(it.valid);
    if ((tid & 63) == 0) s_w[tid >> 6] = __popcll(m);
    __syncthreads();
    if (tid == 0) block_count[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

__global__ __launch_bounds__(kWG) void k_near_write(NearPlan p, const uint32_t *block_off,
                                                    double4 *near) {
    __shared__ int s_w[kWG / 64];
    const int tid = threadIdx.x, wave = tid >> 6;
    NearItem it = near_item(p, blockIdx.x, tid);
    uint64_t m = __ballot(it.valid);
    if ((tid & 63) == 0) s_w[wave] = __popcll(m);
    __syncthreads();
    if (it.valid) {
        int off = block_off[blockIdx.x] + lanes_below(m);
        for (int w = 0; w < wave; ++w) off += s_w[w];
        double x, y, z;
        frac_to_cart(p.t, it.gx, it.gy, it.gz, x, y, z);
        near[off] = make_double4(x, y, z, p.types[it.type].rclose);
    }
}

// Single-workgroup exclusive scan of n uint32 values; out[n] = total.
__device__ void block_exclusive_scan(const uint32_t *in, long long n, uint32_t *out,
                                     uint32_t *out2) {
    __shared__ uint32_t s_part[kWG];
    __shared__ uint32_t s_carry;
    const int tid = threadIdx.x;
    if (tid == 0) s_carry = 0;
    __syncthreads();
    const int per = 8;
    for (long long base = 0; base < n; base += (long long)kWG * per) {
        uint32_t v[per];
        uint32_t sum = 0;
        for (int k = 0; k < per; ++k) {
            long long i = base + (long long)tid * per + k;
            v[k] = (i < n) ? in[i] : 0u;
            sum += v[k];
        }
        s_part[tid] = sum;
        __syncthreads();
        // Hillis-Steele inclusive scan over the 256 partial sums
        for (int d = 1; d < kWG; d <<= 1) {
            uint32_t add = (tid >= d) ? s_part[tid - d] : 0u;
            __syncthreads();
            s_part[tid] += add;
            __syncthreads();
        }
        uint32_t run = s_carry + s_part[tid] - sum;
        for (int k = 0; k < per; ++k) {
            long long i = base + (long long)tid * per + k;
            if (i < n) {
                out[i] = run;
                if (out2) out2[i] = run;
            }
            run += v[k];
        }
        __syncthreads();
        if (tid == kWG - 1) s_carry += s_part[kWG - 1];
        __syncthreads();
    }
    if (tid == 0) {
        out[n] = s_carry;
        if (out2) out2[n] = s_carry;
    }
}

__global__ __launch_bounds__(kWG) void k_near_offsets(NearPlan p, const uint32_t *block_count,
                                                      uint32_t *block_off, int *type_begin) {
    block_exclusive_scan(block_count, p.nblocks, block_off, nullptr);
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int t = 0; t < p.ntypes; ++t) type_begin[t] = (int)block_off[p.type_block0[t]];
        type_begin[p.ntypes] = (int)block_off[p.nblocks];
    }
}

// ---------------------------------------------------------------------------
// Widom binning
// ---------------------------------------------------------------------------

__device__ __forceinline__ uint32_t widom_bin(const double f[3], const int nb[3]) {
    int b[3];
    for (int d = 0; d < 3; ++d) {
        int v = (int)(f[d] * nb[d]);  // f in (0,1]
        b[d] = v < nb[d] ? v : nb[d] - 1;
    }
    return (uint32_t)((b[0] * nb[1] + b[1]) * nb[2] + b[2]);
}

// Batched binning.  A job's keys are its bins, or, when it has many, groups of
// consecutive bins.  Each block takes `chunk` consecutive insertion indices of
// one job, histograms their keys in LDS and touches global memory once per key
// it saw: the count pass adds its counts, the scatter pass reserves a range of
// the key's slots and hands them out through LDS atomics.  A grouped job's
// scatter writes (bin in the group, insertion) pairs, which a last pass, one
// block per group, sorts into bins.  The order inside a bin is therefore
// arbitrary; no result depends on it (every insertion of a bin sees the same
// candidate list, and sums run over insertion indices).
//
// A Philox point costs ~20 quarter-rate multiplies, so only the count pass
// makes the points; it leaves each insertion's bin for the scatter pass in the
// one of `sorted` and `tmp` that the scatter does not write.
//
// The groups keep the histogram at a few KiB and the scattered runs long:
// 1.73e7 insertions of 36036 bins took 711 us to count and 1364 us to scatter
// with one global atomic per insertion; now 64 us to count (the points), 67 us
// to scatter and 67 us to sort the groups.  The scatter is bound by its stores:
// written straight from the lanes they took 241 us.  16 jobs of 1e6 insertions
// and ~2080 bins each (one step): 48 + 159 us before, 51 + 69 us now.
__device__ __forceinline__ int bin_job_of(const BinJob *__restrict__ jobs, int njobs,
                                          long long blk) {
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].block0 <= blk) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(kWG) void k_bin_zero(const BinJob *__restrict__ jobs) {
    const BinJob &J = jobs[blockIdx.x];
    for (int b = threadIdx.x; b < J.ngroups; b += kWG) J.count[b] = 0u;
}

__global__ __launch_bounds__(kWG) void k_bin_count(const BinJob *__restrict__ jobs, int njobs,
                                                   int chunk) {
    extern __shared__ uint32_t s_hist[];
    const int j = bin_job_of(jobs, njobs, blockIdx.x);
    const BinJob &J = jobs[j];
    const uint64_t i0 = (uint64_t)(blockIdx.x - J.block0) * (uint64_t)chunk;
    const uint64_t i1 = i0 + (uint64_t)chunk < J.n ? i0 + (uint64_t)chunk : J.n;
    const uint32_t group = (uint32_t)J.group;
    uint32_t *__restrict__ keys = group > 1 ? J.sorted : reinterpret_cast<uint32_t *>(J.tmp);
    for (int b = threadIdx.x; b < J.ngroups; b += kWG) s_hist[b] = 0u;
    __syncthreads();
    for (uint64_t i = i0 + threadIdx.x; i < i1; i += kWG) {
        double f[3];
        widom_point(J.seed, J.stream, i, f);
        const uint32_t bin = widom_bin(f, J.nb);
        keys[i] = bin;
        atomicAdd(&s_hist[group > 1 ? bin / group : bin], 1u);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < J.ngroups; b += kWG)
        if (s_hist[b]) atomicAdd(&J.count[b], s_hist[b]);
}

__global__ __launch_bounds__(kWG) void k_bin_scan(const BinJob *__restrict__ jobs) {
    const BinJob &J = jobs[blockIdx.x];
    block_exclusive_scan(J.count, J.ngroups, J.cursor, J.group > 1 ? nullptr : J.start);
}

// A thread holds the keys of its PER insertions: they are read once, with PER
// loads in flight.  The block sorts its insertions by key in LDS before it
// writes them, so that a wave's store covers a few runs of consecutive slots
// instead of 64 separate lines.
template <int PER>
__global__ __launch_bounds__(kBinWG) void k_bin_scatter(const BinJob *__restrict__ jobs,
                                                        int njobs) {
    extern __shared__ uint32_t s_hist[];
    __shared__ uint32_t s_part[kBinWG / 64];
    constexpr int chunk = PER * kBinWG;
    const int tid = threadIdx.x;
    const int j = bin_job_of(jobs, njobs, blockIdx.x);
    const BinJob &J = jobs[j];
    const uint64_t i0 = (uint64_t)(blockIdx.x - J.block0) * (uint64_t)chunk;
    const int cnt = (int)(J.n - i0 < (uint64_t)chunk ? J.n - i0 : (uint64_t)chunk);
    const uint32_t group = (uint32_t)J.group;
    const int nk = J.ngroups;
    const uint32_t *__restrict__ keys =
        (group > 1 ? J.sorted : reinterpret_cast<const uint32_t *>(J.tmp)) + i0;
    uint32_t bin[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int l = q * kBinWG + tid;
        bin[q] = keys[l < cnt ? l : 0];
    }
    // s_hist[nk]: counts, then first slots in the block's order; s_dst[nk]:
    // first slot in the job's order; s_key, s_loc[chunk]: the sorted insertions
    uint32_t *s_dst = s_hist + nk;
    uint32_t *s_loc = s_dst + nk;
    uint16_t *s_key = reinterpret_cast<uint16_t *>(s_loc + chunk);
    for (int b = tid; b < nk; b += kBinWG) s_hist[b] = 0u;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q)
        if (q * kBinWG + tid < cnt)
            atomicAdd(&s_hist[group > 1 ? bin[q] / group : bin[q]], 1u);
    __syncthreads();
    // exclusive scan of the counts (consecutive keys per thread), each key's
    // share of the job's slots reserved on the way
    const int per = (nk + kBinWG - 1) / kBinWG;
    const int p0 = tid * per < nk ? tid * per : nk, p1 = p0 + per < nk ? p0 + per : nk;
    uint32_t sum = 0;
    for (int b = p0; b < p1; ++b) sum += s_hist[b];
    uint32_t inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t v = __shfl_up(inc, d, 64);
        if ((tid & 63) >= d) inc += v;
    }
    if ((tid & 63) == 63) s_part[tid >> 6] = inc;
    __syncthreads();
    uint32_t run = inc - sum;
    for (int w = 0; w < (tid >> 6); ++w) run += s_part[w];
    for (int b = p0; b < p1; ++b) {
        const uint32_t c = s_hist[b];
        s_hist[b] = run;
        // dst - first: what a slot in the block's order is moved by
        if (c) s_dst[b] = atomicAdd(&J.cursor[b], c) - run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int l = q * kBinWG + tid;
        if (l >= cnt) continue;
        const uint32_t key = group > 1 ? bin[q] / group : bin[q];
        const uint32_t slot = atomicAdd(&s_hist[key], 1u);
        s_key[slot] = (uint16_t)key;
        // bin in the group (< kBinGroupMax < 2^14) and insertion in the chunk (< 2^14)
        s_loc[slot] = (uint32_t)l | ((bin[q] - key * group) << 14);
    }
    __syncthreads();
    for (int l = tid; l < cnt; l += kBinWG) {
        const uint32_t v = s_loc[l], pos = s_dst[s_key[l]] + (uint32_t)l;
        const uint32_t ins = (uint32_t)i0 + (v & 0x3fffu);
        if (group > 1) J.tmp[pos] = make_uint2(v >> 14, ins);
        else J.sorted[pos] = ins;
    }
}

// Second step of grouped jobs: block = one group, whose pairs lie between the
// cursors its neighbour and itself ended at.  A thread keeps its first kFinePer pairs
// (all of them in a group of up to 20480, as 1024 groups of 2e7 insertions have) for
// the second pass, which then reads nothing: 1.73e7 insertions took 80 us with both
// passes reading, 67 us now (138 MB read, 69 MB written).
constexpr int kFinePer = 20;
__global__ __launch_bounds__(kBinWG) void k_bin_fine(const BinJob *__restrict__ jobs, int njobs) {
    extern __shared__ uint32_t s_cnt[];
    __shared__ uint32_t s_part[kBinWG / 64];
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].gblock0 <= blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const BinJob &J = jobs[lo];
    const int g = (int)(blockIdx.x - J.gblock0);
    if (J.group <= 1 || g >= J.ngroups) return;
    const int tid = threadIdx.x;
    const int nbt = J.nb[0] * J.nb[1] * J.nb[2], b0 = g * J.group;
    const int nb = b0 + J.group < nbt ? J.group : nbt - b0;
    const uint32_t e0 = g > 0 ? J.cursor[g - 1] : 0u, e1 = J.cursor[g];
    uint2 v[kFinePer];
#pragma unroll
    for (int q = 0; q < kFinePer; ++q) {
        const uint64_t e = run_slot(e0, q * kBinWG + tid);
        v[q] = J.tmp[e < e1 ? e : 0u];
    }
    for (int b = tid; b < nb; b += kBinWG) s_cnt[b] = 0u;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kFinePer; ++q)
        if (run_slot(e0, q * kBinWG + tid) < e1) atomicAdd(&s_cnt[v[q].x], 1u);
    for (uint64_t e = run_slot(e0, kFinePer * kBinWG + tid); e < e1; e += kBinWG)
        atomicAdd(&s_cnt[J.tmp[e].x], 1u);
    __syncthreads();
    // exclusive scan of the group's bins: per consecutive counts per thread
    const int per = (nb + kBinWG - 1) / kBinWG;
    const int p0 = tid * per < nb ? tid * per : nb, p1 = p0 + per < nb ? p0 + per : nb;
    uint32_t sum = 0;
    for (int b = p0; b < p1; ++b) sum += s_cnt[b];
    uint32_t inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t u = __shfl_up(inc, d, 64);
        if ((tid & 63) >= d) inc += u;
    }
    if ((tid & 63) == 63) s_part[tid >> 6] = inc;
    __syncthreads();
    uint32_t run = e0 + inc - sum;
    for (int w = 0; w < (tid >> 6); ++w) run += s_part[w];
    for (int b = p0; b < p1; ++b) {
        const uint32_t c = s_cnt[b];
        s_cnt[b] = run;
        J.start[b0 + b] = run;
        run += c;
    }
    if (g == J.ngroups - 1 && tid == 0) J.start[nbt] = (uint32_t)J.n;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kFinePer; ++q)
        if (run_slot(e0, q * kBinWG + tid) < e1)
            J.sorted[atomicAdd(&s_cnt[v[q].x], 1u)] = v[q].y;
    for (uint64_t e = run_slot(e0, kFinePer * kBinWG + tid); e < e1; e += kBinWG) {
        const uint2 u = J.tmp[e];
        J.sorted[atomicAdd(&s_cnt[u.x], 1u)] = u.y;
    }
}

__global__ void k_fill_u64(unsigned long long *p, unsigned long long v, long long n) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

// The descriptors of a job that runs alone, by value: one launch writes them and
// clears the counters, in place of a copy per descriptor and a fill per counter.
// With the sums written to pinned memory a Henry run is 7 launches (8 if its bins are
// grouped) and no copy, two launches and three copies less: 1e5 insertions, 200 atoms
// 128 -> 97 us.
struct Setup {
    JobDev job;
    BinJob bin;
    JobDev *d_job;
    BinJob *d_bin;  // nullptr: no binning
    unsigned long long *counter;
};

template <class T>
__device__ __forceinline__ void copy_words(T *to, const T &from) {
    static_assert(sizeof(T) % sizeof(uint32_t) == 0, "whole words");
    const uint32_t *f = reinterpret_cast<const uint32_t *>(&from);
    for (unsigned i = threadIdx.x; i < sizeof(T) / sizeof(uint32_t); i += kWG)
        reinterpret_cast<uint32_t *>(to)[i] = f[i];
}

__global__ __launch_bounds__(kWG) void k_setup(const Setup a) {
    copy_words(a.d_job, a.job);
    if (threadIdx.x == 0) *a.counter = 0ull;
    if (!a.d_bin) return;
    copy_words(a.d_bin, a.bin);
    for (int b = threadIdx.x; b < a.bin.ngroups; b += kWG) a.bin.count[b] = 0u;
}

// ---------------------------------------------------------------------------
// Tiled energy kernel
// ---------------------------------------------------------------------------

enum : int { CAT_NONE = 0, CAT_FAR = 1, CAT_SHELL = 2, CAT_NEAR = 3 };

// Ints per list segment: type, far begin, shell begin, near begin.  The types of
// a pass are consecutive, so a segment ends where the next begins; the entry
// after the last holds the pass's counts, and in place of the type whether a near
// pair may need the clamp of r^2.
constexpr int kSegInts = 4;
constexpr int kClampBit = 1 << 16;

// Pairs per point summed in FP32 (far and shell pairs of one type) before the
// sum is scaled and added to the FP64 energy.
constexpr int kFlushPairs = 16;

struct Tile {
    double cx, cy, cz, R;
};

__device__ __forceinline__ Tile tile_sphere(const double *t, const double lo[3],
                                            const double hi[3]) {
    Tile s;
    frac_to_cart(t, 0.5 * (lo[0] + hi[0]), 0.5 * (lo[1] + hi[1]), 0.5 * (lo[2] + hi[2]), s.cx,
                 s.cy, s.cz);
    const double h[3] = {0.5 * (hi[0] - lo[0]), 0.5 * (hi[1] - lo[1]), 0.5 * (hi[2] - lo[2])};
    double r2 = 0.0;
    for (int c = 0; c < 4; ++c) {  // opposite corners are equally far
        double x, y, z;
        frac_to_cart(t, h[0], c & 2 ? h[1] : -h[1], c & 1 ? h[2] : -h[2], x, y, z);
        const double q = x * x + y * y + z * z;
        r2 = q > r2 ? q : r2;
    }
    s.R = sqrt(r2) * (1.0 + 1e-12) + kMargin;
    return s;
}

// i / (n - 1), correctly rounded (src/writegrid.cu:122-127 divides): the quotient
// from the rounded reciprocal, corrected by its exact remainder.  Equal to the
// division for every 0 <= i < n <= 65536, in 3 instead of ~12 instructions.
__device__ __forceinline__ double grid_frac(const JobDev *__restrict__ J, int d, int i) {
    const double q = (double)i * J->inv[d];
    return fma(fma(-q, (double)(J->n[d] - 1), (double)i), J->inv[d], q);
}

// Sphere around the grid points i0 .. i1 of a tile (or of a wave's part of one);
// R: the radius if they are a full one's (J->cell_R, J->wave_R).
__device__ __forceinline__ Tile points_sphere(const JobDev *__restrict__ J, const int i0[3],
                                              const int i1[3], bool full, double R) {
    if (!full) {  // at the far faces of the grid only
        double lo[3], hi[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo[d] = grid_frac(J, d, i0[d]);
            hi[d] = grid_frac(J, d, i1[d]);
        }
        return tile_sphere(J->t, lo, hi);
    }
    Tile s;
    frac_to_cart(J->t, 0.5 * (i0[0] + i1[0]) * J->inv[0], 0.5 * (i0[1] + i1[1]) * J->inv[1],
                 0.5 * (i0[2] + i1[2]) * J->inv[2], s.cx, s.cy, s.cz);
    s.R = R;
    return s;
}

// Sphere around cell tc (a full tile's points, or less at the far faces, with the
// full tile's radius; or a bin).
__device__ __forceinline__ Tile cell_sphere(const JobDev *__restrict__ J, const int tc[3]) {
    double f[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        double i = tc[d] + 0.5;
        if (J->kind == JOB_GRID) {
            const int a = tc[d] * J->tile[d], e = a + J->tile[d];
            i = 0.5 * (a + (e < J->n[d] ? e : J->n[d]) - 1);
        }
        f[d] = i * J->inv[d];
    }
    Tile s;
    frac_to_cart(J->t, f[0], f[1], f[2], s.cx, s.cy, s.cz);
    s.R = J->cell_R;
    return s;
}

// Split of the LDS list: [0, capA) holds far records (from 0 upwards) and
// shell records (from capA-1 downwards); [capA, cap) holds near records.
template <int MATH>
__host__ __device__ __forceinline__ int near_region_start(int cap) {
    if (MATH == MATH_FP64) return cap - kWG;  // near: atoms within R of the tile centre
    if (MATH == MATH_COUNT || MATH == MATH_OVERLAP) return cap - kWG;  // no near records
    return mixed_far_shell_cap(cap);
}

// Stream the near list of job J from (cur_t, cur_pos) into the LDS list until
// it is exhausted or a region is full, classifying each image atom by its
// distance d to the tile centre: far (every point of the tile is inside the
// cutoff and beyond the FP64 switch radius), shell (beyond the switch radius
// but possibly outside the cutoff), near (possibly inside the switch radius).
// Records hold the atom relative to the tile centre and its squared distance,
// (a - c, |a - c|^2), and keep the source order, so the list (and every sum
// over it) depends only on the tile and the source.  The source is the near
// list src, position p holding src[p], or, with sidx, a sub-list of it,
// position p holding src[sidx[p]].  Returns the number of segments (one per
// type, in the source's order) written to seg.
//
// Chunks of 256 records run across type boundaries (a record carries its type's
// switch radius): six types of 50 records take two rounds of loads, ballots and
// barriers instead of six.  With the cells' radii made on the host and the
// quotients of grid_frac this took a Henry run of 1.73e7 insertions in a 424-atom
// cell (36036 bins) from 2.52 to 2.27 ms and a 4.9e7-point grid of 2400 atoms from
// 7.77 to 6.71 ms, where the setup of a tile cost a third of its instructions.
template <int MATH, int WG>
__device__ int fill_list(const JobDev *__restrict__ J, const double4 *__restrict__ src,
                         const uint32_t *__restrict__ sidx, const int *__restrict__ tbeg,
                         const Tile &tl, int &cur_t, int &cur_pos,
                         int cap, double4 *__restrict__ L, int *__restrict__ seg,
                         int *__restrict__ s_cnt) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ntypes = J->ntypes;
    const double rc = J->rc;
    const int capA = near_region_start<MATH>(cap);
    const int capN = cap - capA;
    // Squared-distance forms of the tests on d = |image atom - tile centre|:
    //   some point may be inside r_c:     d - R <  r_c             (in2)
    //   every point is inside r_c:        d + R <  r_c             (far2)
    //   some point may be inside r_FP64:  d - R <= r_FP64          (near, per type)
    // each widened by kMargin so FP64 rounding cannot misclassify.
    const double in2 = (rc + tl.R + kMargin) * (rc + tl.R + kMargin);
    const double far_r = rc - tl.R - kMargin;
    const double far2 = far_r > 0.0 ? far_r * far_r : -1.0;
    // the clamp of r^2 (at most 1e-24 A^2) can matter only if some point may lie
    // within kMargin of the atom, d <= R + kMargin.  FP64 grids: those are the near
    // records; the others: a pass that keeps none of them is evaluated without it
    const double clamp2 = (tl.R + kMargin) * (tl.R + kMargin);
    // The cell's points lie in a parallelepiped around the centre:
    // J->cell_box[d] times cell vector t_d on either side (a bin's box; a
    // full tile's, which holds a partial edge tile's around that tile's own
    // centre).  A shell record at v from the centre with |v|^2 - h(v) >
    // (r_c + m)|v|, h(v) = sum_d cell_box_d |t_d . v|, is beyond r_c of every
    // point (|a - x| >= |v| - h(v)/|v|) and adds exactly 0: it is not kept.
    // (FP32 and FP64 grid tiles re-test their shell records per wave, against
    // the wave's smaller box, which makes this test redundant there)
    const bool wave_lists = J->kind == JOB_GRID && (MATH == MATH_MIXED || MATH == MATH_FP64);
    const double *hb = J->cell_box;
    const double rout = rc + kMargin, rout2 = rout * rout;
    const double *tm = J->t;
    while (cur_t + 1 < ntypes && uniform(tbeg[cur_t + 1]) <= cur_pos) ++cur_t;
    const int first_t = cur_t;
    // a pass takes at most kMaxSeg types
    const int last_t = first_t + kMaxSeg < ntypes ? first_t + kMaxSeg : ntypes;
    const int end = uniform(tbeg[last_t]);
    int nf = 0, ns = 0, nn = 0, nseg = 1, clamp = 0;
    if (tid == 0) {
        seg[0] = first_t;
        seg[1] = seg[2] = seg[3] = 0;
    }
    while (cur_pos < end) {
        const int idx = cur_pos + tid;
        int cat = CAT_NONE;
        double4 A = make_double4(0.0, 0.0, 0.0, 0.0);
        if (idx < end) {
            const double4 S = src[sidx ? (int)sidx[idx] : idx];
            const double dx = S.x - tl.cx, dy = S.y - tl.cy, dz = S.z - tl.cz;
            const double d2 = dx * dx + dy * dy + dz * dz;
            A = make_double4(dx, dy, dz, d2);
            if (d2 < in2) {
                const double rn = S.w + tl.R + kMargin;
                if (MATH == MATH_FP64 && d2 <= clamp2) cat = CAT_NEAR;
                else if (MATH == MATH_MIXED && d2 <= rn * rn) cat = CAT_NEAR;
                else cat = (MATH != MATH_OVERLAP && d2 < far2) ? CAT_FAR : CAT_SHELL;
                if (cat == CAT_SHELL && !wave_lists) {
                    const double h = hb[0] * fabs(tm[0] * dx + tm[3] * dy + tm[6] * dz) +
                                     hb[1] * fabs(tm[1] * dx + tm[4] * dy + tm[7] * dz) +
                                     hb[2] * fabs(tm[2] * dx + tm[5] * dy + tm[8] * dz);
                    const double g = d2 - h;
                    if (g > 0.0 && g * g > rout2 * d2) cat = CAT_NONE;
                }
            }
        }
        const uint64_t bf = __ballot(cat == CAT_FAR);
        const uint64_t bs = __ballot(cat == CAT_SHELL);
        const uint64_t bn = __ballot(cat == CAT_NEAR);
        const bool at = MATH == MATH_MIXED && __ballot(cat == CAT_NEAR && A.w <= clamp2);
        if (lane == 0) {
            s_cnt[3 * wave] = __popcll(bf);
            s_cnt[3 * wave + 1] = __popcll(bs);
            s_cnt[3 * wave + 2] = __popcll(bn) | (at ? kClampBit : 0);
        }
        __syncthreads();
        int of = nf, os = ns, on = nn, tf = 0, ts = 0, tn = 0;
#pragma unroll
        for (int w = 0; w < WG / 64; ++w) {
            const int cf = s_cnt[3 * w], cs = s_cnt[3 * w + 1];
            const int cn = s_cnt[3 * w + 2] & ~kClampBit;
            clamp |= s_cnt[3 * w + 2] & kClampBit;
            if (w < wave) {
                of += cf;
                os += cs;
                on += cn;
            }
            tf += cf;
            ts += cs;
            tn += cn;
        }
        // types that begin in this chunk: the counts before their first record
        while (first_t + nseg < last_t) {
            const int p = uniform(tbeg[first_t + nseg]) - cur_pos;
            if (p >= WG) break;
            if (wave == p >> 6 && lane == 0) {
                const uint64_t below = (1ull << (p & 63)) - 1ull;
                int *g = seg + kSegInts * nseg;
                g[0] = first_t + nseg;
                g[1] = of + __popcll(bf & below);
                g[2] = os + __popcll(bs & below);
                g[3] = on + __popcll(bn & below);
            }
            ++nseg;
        }
        // A pass takes the kept records in source order up to the first one
        // that does not fit (far + shell share [0, capA), near [capA, cap)),
        // so its content depends only on the sequence of kept records, not on
        // the source's chunking: a region sub-list and the near list give the
        // same passes.  Records after that one may also be written (into
        // slots past the final counts, never read in this pass).
        const int fs_before = of + os + lanes_below(bf | bs);
        const int n_before = on + lanes_below(bn);
        const bool fits = (cat == CAT_FAR || cat == CAT_SHELL) ? fs_before < capA
                          : cat == CAT_NEAR                    ? n_before < capN
                                                               : true;
        if (fits && cat == CAT_FAR) L[of + lanes_below(bf)] = A;
        if (fits && cat == CAT_SHELL) L[capA - 1 - (os + lanes_below(bs))] = A;
        if (fits && cat == CAT_NEAR) L[capA + on + lanes_below(bn)] = A;  // A: (a - c, |a - c|^2)
        const uint64_t bx = __ballot(!fits);
        if (lane == 0) {
            // this wave's first record that does not fit, and the counts before it
            int *x = s_cnt + 3 * (WG / 64) + 4 * wave;
            if (bx) {
                const int l = __builtin_ctzll(bx);
                const uint64_t below = (1ull << l) - 1ull;
                x[0] = l;
                x[1] = of + __popcll(bf & below);
                x[2] = os + __popcll(bs & below);
                x[3] = on + __popcll(bn & below);
            } else {
                x[0] = 64;
            }
        }
        __syncthreads();
        int stop = -1;
#pragma unroll
        for (int w = WG / 64 - 1; w >= 0; --w)
            if (s_cnt[3 * (WG / 64) + 4 * w] < 64) stop = w;
        if (stop >= 0) {
            const int *x = s_cnt + 3 * (WG / 64) + 4 * stop;
            nf = uniform(x[1]);
            ns = uniform(x[2]);
            nn = uniform(x[3]);
            cur_pos += 64 * stop + uniform(x[0]);
            // types that begin at or after the stop belong to the next pass
            while (nseg > 1 && uniform(tbeg[first_t + nseg - 1]) >= cur_pos) --nseg;
            break;
        }
        nf = uniform(nf + tf);
        ns = uniform(ns + ts);
        nn = uniform(nn + tn);
        cur_pos += WG;
    }
    if (cur_pos >= end) {
        cur_pos = end;
        cur_t = last_t;
        // (types whose records all lie before the end have begun; empty ones at
        // the very end may not have)
    } else {
        cur_t = first_t + nseg - 1;
    }
    if (tid == 0) {
        int *g = seg + kSegInts * nseg;
        g[0] = clamp;
        g[1] = nf;
        g[2] = ns;
        g[3] = nn;
    }
    return nseg;
}

// r^2 from this lane's points to record A (both relative to the tile centre):
// the expanded form |a|^2 + |p|^2 - 2 p.a with the z, y, x terms in that
// order.  With XL the lane's points share y and z (grid points that differ
// only in i, on a cell whose first vector lies along x), so the z and y terms
// are formed once per record; the result is bit-identical to the per-point
// form, since the shared terms are the same operations on the same values.
template <int PPL, bool XL>
__device__ __forceinline__ void pair_r2(const double4 &A, const double (&mx)[PPL],
                                        const double (&my)[PPL], const double (&mz)[PPL],
                                        const double (&p2)[PPL], double (&r2)[PPL]) {
    if (XL) {
        const double yz = fma(my[0], A.y, fma(mz[0], A.z, A.w));
#pragma unroll
        for (int q = 0; q < PPL; ++q) r2[q] = fma(mx[q], A.x, yz) + p2[q];
    } else {
#pragma unroll
        for (int q = 0; q < PPL; ++q)
            r2[q] = fma(mx[q], A.x, fma(my[q], A.y, fma(mz[q], A.z, A.w))) + p2[q];
    }
}

// Shell records [sb, se) of a segment (record k at Ls[-k]) against this
// wave's sphere wsph (centre relative to the tile centre, radius wsph.w):
// records beyond r_c + w of it are out of the cutoff for all of the wave's
// points and dropped, those within r_c - w are inside it for all of them (no
// cutoff test).  The wave's points lie in a parallelepiped around that
// centre, J->wave_box[d] times cell vector t_d on either side; for a record
// at v from the centre every point x has |a - x| >= (a - x).v/|v| >=
// |v| - h(v)/|v|, h(v) = sum_d wave_box_d |t_d . v|, so a record with
// |v|^2 - h(v) > (r_c + m)|v| is out of the cutoff for every point as well
// and is dropped: it added exactly 0 to every sum.  (The matching bound
// |a - x|^2 <= |v|^2 + 2 h(v) + w^2 would move a few records from the
// shell to the far list; it measured no gain.)  The wave writes its own
// list of LDS byte offsets (from the start of the list, capA - 1 - k
// records), order kept: the nwf wave-far ones from the front of wl, the nws
// still-shell ones from wl[wcap - 1] down (se - sb <= wcap entries).
__device__ __forceinline__ void wave_shell_lists(const JobDev *__restrict__ J,
                                                 const double4 *__restrict__ Ls, int capA,
                                                 int wcap, int sb, int se, const double4 &wsph,
                                                 uint16_t *__restrict__ wl, int &nwf, int &nws) {
    const int lane = threadIdx.x & 63;
    const double rin = J->rc + wsph.w + kMargin, rfar = J->rc - wsph.w - kMargin;
    const double in2 = rin * rin, far2 = rfar > 0.0 ? rfar * rfar : -1.0;
    const double rout = J->rc + kMargin, rout2 = rout * rout;
    const double *t = J->t, *wb = J->wave_box;
    nwf = 0;
    nws = 0;
    for (int k0 = sb; k0 < se; k0 += 64) {
        const int k = k0 + lane;
        int cat = 0;
        if (k < se) {
            const double4 A = Ls[-k];
            const double dx = A.x - wsph.x, dy = A.y - wsph.y, dz = A.z - wsph.z;
            const double d2 = dx * dx + dy * dy + dz * dz;
            cat = d2 < in2 ? (d2 < far2 ? 1 : 2) : 0;
            if (cat == 2) {
                const double h = wb[0] * fabs(t[0] * dx + t[3] * dy + t[6] * dz) +
                                 wb[1] * fabs(t[1] * dx + t[4] * dy + t[7] * dz) +
                                 wb[2] * fabs(t[2] * dx + t[5] * dy + t[8] * dz);
                const double g = d2 - h;
                if (g > 0.0 && g * g > rout2 * d2) cat = 0;
            }
        }
        const uint64_t bf = __ballot(cat == 1), bs = __ballot(cat == 2);
        const uint16_t off = (uint16_t)((capA - 1 - k) * (int)sizeof(double4));
        if (cat == 1) wl[nwf + lanes_below(bf)] = off;
        if (cat == 2) wl[wcap - 1 - (nws + lanes_below(bs))] = off;
        nwf = uniform(nwf + __popcll(bf));
        nws = uniform(nws + __popcll(bs));
    }
    // the lists are read back by every lane of this wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- sums in parts ----------------------------------------------------------
//
// Jobs of few cells (JobDev::parts) sum an energy in parts, so that several waves
// can share a point's records (k_parts) and one wave can make the same sum, to the
// bit, where the device is full without that (k_tiles).  The records of a pass form
// groups of one segment and kind: 16 far or shell records (the FP32 sums' groups), 8
// near ones.  Part v of `parts` has the groups [v G / parts, (v + 1) G / parts) of the
// pass's G, and a pass adds its parts in order.  A grid's groups are numbered segment
// by segment.  A Widom pass has its near groups first, in parts of their own, so that
// saturated insertions can stop before the others.
constexpr int kNearGroup = 8;
constexpr int kShellGroup = kFlushPairs;

__device__ __forceinline__ int groups_of(int n, int size) { return (n + size - 1) / size; }

__device__ __forceinline__ int part_begin(int v, int groups, int parts) {
    return (v * groups) >> (parts == 8 ? 3 : parts == 4 ? 2 : 1);
}

// Groups of a pass: near ones (x) and others (y).  wn(s): segment s's wave-far and
// (high half) wave-shell records, or just its shell records.
template <class WN>
__device__ __forceinline__ int2 count_groups(const int *__restrict__ seg, int nseg, WN wn) {
    int2 n = make_int2(0, 0);
    for (int s = 0; s < nseg; ++s) {
        const int *g = seg + kSegInts * s;
        const int w = wn(s);
        n.x += groups_of(uniform(g[kSegInts + 3]) - uniform(g[3]), kNearGroup);
        n.y += groups_of(uniform(g[kSegInts + 1]) - uniform(g[1]), kShellGroup) +
               groups_of(w & 0xffff, kShellGroup) + groups_of(w >> 16, kShellGroup);
    }
    return make_int2(uniform(n.x), uniform(n.y));
}

// What eval_list does about parts: nothing, ...
struct NoParts {
    static constexpr bool on = false, one = false;
};

// ... sums them one after the other: e, the energies of the current part, is added to
// sum where the next part begins, ...  (u, v and next are wave-uniform, which the
// compiler does not see by itself: 5% of the kernel's VALU instructions.)
template <int P>
struct PartSums {
    static constexpr bool on = true, one = false;
    double (&sum)[P];
    int groups, parts;
    int u = 0, v = 0, next = 0;  // next group, next part, its first group
    __device__ __forceinline__ PartSums(double (&s)[P], int g, int p)
        : sum(s), groups(g), parts(p) {}
    __device__ __forceinline__ bool ended() const { return uniform(u) == uniform(next); }
    // up to n groups of one part begin here
    __device__ __forceinline__ int run(double (&e)[P], int n) {
        u = uniform(u);
        next = uniform(next);
        if (u == next) {
            flush(e);
            v = uniform(v);
            while (next <= u) next = part_begin(++v, groups, parts);
        }
        const int r = n < next - u ? n : next - u;
        u += r;
        return r;
    }
    __device__ __forceinline__ void flush(double (&e)[P]) {
#pragma unroll
        for (int q = 0; q < P; ++q) {
            sum[q] += e[q];
            e[q] = 0.0;
        }
    }
};

// ... or makes one of them, the groups [lo, hi).
struct OnePart {
    static constexpr bool on = true, one = true;
    int lo, hi;
    int u = 0;
    __device__ __forceinline__ OnePart(int v, int groups, int parts)
        : lo(part_begin(v, groups, parts)), hi(part_begin(v + 1, groups, parts)) {}
    // whether the next n groups are not the part's
    __device__ __forceinline__ bool skip(int n) {
        if (u + n > lo && u < hi) return false;
        u = uniform(u + n);
        return true;
    }
    // records [b, e) in groups of `size`: those of the part
    __device__ __forceinline__ void clip(int &b, int &e, int size) {
        const int count = groups_of(e - b, size);
        const int first = lo > u ? lo - u : 0, end = hi - u < count ? hi - u : count;
        u = uniform(u + count);
        if (end < count) e = b + size * (end > 0 ? end : 0);
        b += size * first;
    }
};

// Energies (or in-cutoff counts) of this lane's PPL points against the LDS
// list.  Points and records are relative to the tile centre c.
//   Far pairs (inside r_c and beyond the FP64 switch radius for every point
//   of the tile): r^2 = |a|^2 + |p|^2 - 2 p.a in FP64 (three FMAs and an add;
//   |a| <= r_c + R keeps the cancellation below 13x), then in FP32
//   u = 1/r^2, and per point the sums S3 = sum u^3 and S6 = sum u^6 over at
//   most kFlushPairs pairs of one type, flushed into the FP64 energy as
//   4 eps (sigma^12 S6 - sigma^6 S3).  sigma and eps stay FP64, so their
//   rounding adds no error common to every pair of a type.
//   Shell pairs: the same, behind the strict FP64 test r^2 < r_c^2.
//   Near pairs (every pair of an FP64 grid): the same FP64 r^2, the
//   reference's clamp and strict cutoff test, FP64 LJ with a Newton-refined
//   reciprocal (one step for FP32 grids and Widom, two for FP64 grids).
// XL: see pair_r2.
// ws (MIXED and FP64 grid tiles, wave-uniform): this wave's points lie in the
// sphere wsph (centre relative to the tile centre, radius w), smaller than
// the tile's, and in the parallelepiped of J->wave_box around the same
// centre; each segment's shell records are then re-classified against them
// into the wave's own lists of LDS byte offsets wl (wave_shell_lists).
// phase (wave-uniform): 0 every record, per segment far, shell, near; 1 only
// the near records; 2 only the far and shell records.
// pb: see "sums in parts".  With parts the wave's shell lists are there already, a
// segment's at its shell offset, and lane s of `lengths` holds their lengths.
template <int PPL, int MATH, bool XL, int NEAR = 1, class PB = NoParts>
__device__ __forceinline__ void eval_list(const JobDev *__restrict__ J,
                                          const double4 *__restrict__ L, int cap,
                                          const int *__restrict__ seg, int nseg,
                                          const double (&px)[PPL], const double (&py)[PPL],
                                          const double (&pz)[PPL], double (&acc)[PPL],
                                          double R, bool ws = false,
                                          double4 wsph = make_double4(0.0, 0.0, 0.0, 0.0),
                                          uint16_t *__restrict__ wl = nullptr, int phase = 0,
                                          PB pb = PB(), int lengths = 0) {
    const bool do_fs = phase != 1, do_near = phase != 2;
    const bool clamp = MATH == MATH_MIXED && do_near && uniform(seg[kSegInts * nseg]) != 0;
    const double rc2 = J->rc2, min_r2 = J->min_r2;
    const int capA = near_region_start<MATH>(cap);
    const double4 *__restrict__ Ls = L + capA - 1;  // shell k at Ls[-k]
    const double4 *__restrict__ Ln = L + capA;      // near k at Ln[k]
    double mx[PPL], my[PPL], mz[PPL], p2[PPL];
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
        mx[q] = -2.0 * px[q];
        my[q] = -2.0 * py[q];
        mz[q] = -2.0 * pz[q];
        p2[q] = px[q] * px[q] + py[q] * py[q] + pz[q] * pz[q];
    }
    for (int s = 0; s < nseg; ++s) {
        const int *g = seg + kSegInts * s;
        const int t = uniform(g[0]);
        const int fb = uniform(g[1]), fe = uniform(g[kSegInts + 1]);
        const int sb = uniform(g[2]), se = uniform(g[kSegInts + 2]);
        const int nb = uniform(g[3]), ne = uniform(g[kSegInts + 3]);
        if (fe - fb + se - sb + ne - nb == 0) continue;
        if constexpr (PB::one) {
            const int w = ws ? __builtin_amdgcn_readlane(lengths, s) : (se - sb) << 16;
            const int fs = groups_of(fe - fb, kShellGroup) + groups_of(w & 0xffff, kShellGroup) +
                           groups_of(w >> 16, kShellGroup);
            if (pb.skip((do_fs ? fs : 0) + (do_near ? groups_of(ne - nb, kNearGroup) : 0)))
                continue;
        }
        const TypeParams P = J->types[t];
        if (MATH == MATH_OVERLAP) {
            // src/computegridsheet.h:154: overlap iff r^2 < sigma_ij^2 (every
            // record is a shell record: the cutoff is sigma_max)
            const double sig2 = P.sig2;
            for (int k = sb; k < se; ++k) {
                double r2[PPL];
                pair_r2<PPL, XL>(Ls[-k], mx, my, mz, p2, r2);
#pragma unroll
                for (int q = 0; q < PPL; ++q) acc[q] += r2[q] < sig2 ? 1.0 : 0.0;
            }
            continue;
        }
        if (MATH == MATH_COUNT) {
            if (!do_fs) continue;  // counting lists hold no near records
#pragma unroll
            for (int q = 0; q < PPL; ++q) acc[q] += (double)(fe - fb);
            for (int k = sb; k < se; ++k) {
                double r2[PPL];
                pair_r2<PPL, XL>(Ls[-k], mx, my, mz, p2, r2);
#pragma unroll
                for (int q = 0; q < PPL; ++q) acc[q] += r2[q] < rc2 ? 1.0 : 0.0;
            }
            continue;
        }
        if (MATH == MATH_MIXED) {
            const double c6 = P.c6, c3 = P.c3;
            auto far_pair = [&](const double4 &A, float (&s3)[PPL], float (&s6)[PPL]) {
                double r2[PPL];
                pair_r2<PPL, XL>(A, mx, my, mz, p2, r2);
#pragma unroll
                for (int q = 0; q < PPL; ++q) {
                    const float w = __builtin_amdgcn_rcpf((float)r2[q]);
                    const float w2 = w * w, w3 = w2 * w;
                    s3[q] = __builtin_fmaf(w2, w, s3[q]);
                    s6[q] = __builtin_fmaf(w3, w3, s6[q]);
                }
            };
            auto shell_pair = [&](const double4 &A, float (&s3)[PPL], float (&s6)[PPL]) {
                double r2[PPL];
                pair_r2<PPL, XL>(A, mx, my, mz, p2, r2);
#pragma unroll
                for (int q = 0; q < PPL; ++q) {
                    const float w = __builtin_amdgcn_rcpf((float)r2[q]);
                    float w3 = w * w * w;
                    w3 = r2[q] < rc2 ? w3 : 0.0f;  // src/computegridsheet.h:79
                    s3[q] += w3;
                    s6[q] = __builtin_fmaf(w3, w3, s6[q]);
                }
            };
            // far records [fb, fe), then shell records [sb, se): FP32 sums of
            // kFlushPairs pairs per point (blocks of 8 unrolled records),
            // then flushed into the FP64 energy
            auto blocks = [&](int b, int e, auto &&pair_at) {
                if constexpr (PB::one) pb.clip(b, e, kShellGroup);
                for (int r = b; r < e; r += kFlushPairs) {
                    if constexpr (PB::on && !PB::one) pb.run(acc, 1);
                    float a3[PPL], a6[PPL];
#pragma unroll
                    for (int q = 0; q < PPL; ++q) a3[q] = a6[q] = 0.0f;
                    const int re = r + kFlushPairs < e ? r + kFlushPairs : e;
#pragma unroll 1
                    for (int h = r; h < re; h += 8) {
                        if (h + 8 <= re) {
#pragma unroll
                            for (int u = 0; u < 8; ++u) pair_at(h + u, a3, a6);
                        } else {
                            for (int k = h; k < re; ++k) pair_at(k, a3, a6);
                        }
                    }
#pragma unroll
                    for (int q = 0; q < PPL; ++q)
                        acc[q] = fma(c6, (double)a6[q], fma(c3, (double)a3[q], acc[q]));
                }
            };
            if (do_fs)
                blocks(fb, fe, [&](int k, float (&s3)[PPL], float (&s6)[PPL]) {
                    far_pair(L[k], s3, s6);
                });
            if (!do_fs) {
            } else if (ws) {
                int nwf, nws, first = 0, last = capA - 1;  // (entries of wl)
                if constexpr (PB::on) {
                    const int w = __builtin_amdgcn_readlane(lengths, s);
                    nwf = w & 0xffff;
                    nws = w >> 16;
                    first = sb;
                    last = se - 1;
                } else {
                    wave_shell_lists(J, Ls, capA, capA, sb, se, wsph, wl, nwf, nws);
                }
                const char *__restrict__ Lb = reinterpret_cast<const char *>(L);
                auto rec = [&](int e) {
                    return *reinterpret_cast<const double4 *>(Lb + wl[e]);
                };
                blocks(0, nwf, [&](int e, float (&s3)[PPL], float (&s6)[PPL]) {
                    far_pair(rec(first + e), s3, s6);
                });
                blocks(0, nws, [&](int e, float (&s3)[PPL], float (&s6)[PPL]) {
                    shell_pair(rec(last - e), s3, s6);
                });
            } else {
                blocks(sb, se, [&](int k, float (&s3)[PPL], float (&s6)[PPL]) {
                    shell_pair(Ls[-k], s3, s6);
                });
            }
            if (!do_near) continue;
            // Near pairs of an FP32 grid or Widom run: the expanded FP64 r^2 of
            // the far pairs (|a| <= r_FP64 + R keeps it exact to ~1e-14 A^2),
            // the reference's clamp and strict cutoff, u = 1/r^2 from the FP32
            // reciprocal and one Newton step (~1e-14 relative), and FP64 sums
            // of u^3 and u^6 scaled by 4 eps sigma^6 / sigma^12 per segment.
            double b3[PPL], b6[PPL];
            // A near record lies within r_FP64 + R of the tile centre, so
            // within r_FP64 + 2R of every point: when that is inside r_c the
            // strict cutoff test (src/computegridsheet.h:79) passes for every
            // pair and is skipped.
            const bool all_in = P.rclose + 2.0 * R + 3.0 * kMargin < J->rc;
            // Most passes hold no record that a point may sit on (kClampBit): without
            // the clamp two points take 27 instead of 30 VALU instructions a record.
            // Grid tiles have NEAR = 2 records in flight (4.9e7 points, 2400 atoms: 6.48 ms
            // with one, 6.37 with two); bins one (a Henry run of 1.7e7: 2.11, 2.15 ms).
            auto near_pairs = [&](int nb, int ne, auto clamp, auto test) {
#pragma unroll NEAR
                for (int k = nb; k < ne; ++k) {
                    double r2[PPL];
                    pair_r2<PPL, XL>(Ln[k], mx, my, mz, p2, r2);
#pragma unroll
                    for (int q = 0; q < PPL; ++q) {
                        // src/computegridsheet.h:77 (r^2 is never NaN, so fmax is the clamp)
                        const double rr = decltype(clamp)::value ? fmax(r2[q], min_r2) : r2[q];
                        double y = (double)__builtin_amdgcn_rcpf((float)rr);
                        y = fma(fma(-rr, y, 1.0), y, y);
                        double y3 = y * y * y;
                        if (decltype(test)::value) y3 = rr < rc2 ? y3 : 0.0;  // :79
                        b3[q] += y3;
                        b6[q] = fma(y3, y3, b6[q]);
                    }
                }
            };
            using no = std::integral_constant<bool, false>;
            using yes = std::integral_constant<bool, true>;
            auto near_run = [&](int nb, int ne) {
#pragma unroll
                for (int q = 0; q < PPL; ++q) b3[q] = b6[q] = 0.0;
                if (!all_in) near_pairs(nb, ne, yes(), yes());
                else if (clamp) near_pairs(nb, ne, yes(), no());
                else near_pairs(nb, ne, no(), no());
#pragma unroll
                for (int q = 0; q < PPL; ++q) acc[q] = fma(c6, b6[q], fma(c3, b3[q], acc[q]));
            };
            if constexpr (PB::on && !PB::one) {
                for (int k = nb; k < ne;) {
                    const int e = k + kNearGroup * pb.run(acc, groups_of(ne - k, kNearGroup));
                    near_run(k, e < ne ? e : ne);
                    k = e;
                }
            } else {
                int b = nb, e = ne;
                if constexpr (PB::one) pb.clip(b, e, kNearGroup);
                near_run(b, e);
            }
            continue;
        }
        // FP64 grids: every pair in FP64.  The expanded FP64 r^2 of the near
        // pairs of FP32 grids, u = 1/r^2 from the FP32 reciprocal refined in
        // FP64, FP64 sums of u^3 and u^6 scaled by 4 eps sigma^6 / sigma^12
        // per segment.  Far records (inside r_c for every point, farther than
        // kMargin from all) need neither the clamp nor the cutoff test, shell
        // records only the test, near records (an atom within R of the tile
        // centre) both.
        // One Newton step: the FP32 reciprocal of the rounded r^2 is within
        // e0 <= 2^-24 + 2^-23 of 1/r^2, and y + y (1 - r^2 y) leaves 1/r^2
        // (1 - e0^2) plus one FP64 rounding, so u is low by at most 3.2e-14
        // relative and a pair's energy is off by at most 2e-13 of |4 eps
        // sigma^12 u^6| + |4 eps sigma^6 u^3| -- the size of the rounding the
        // expanded r^2 already leaves (|a|^2 + |p|^2 - 2 p.a cancels ~13 FP64
        // ulps of |a|^2).  Near records take two steps.
        const double c6 = P.c6, c3 = P.c3;
        double b3[PPL], b6[PPL];
#pragma unroll
        for (int q = 0; q < PPL; ++q) b3[q] = b6[q] = 0.0;
        auto fp64_pair = [&](const double4 &A, auto clamp, auto test) {
            double r2[PPL];
            pair_r2<PPL, XL>(A, mx, my, mz, p2, r2);
#pragma unroll
            for (int q = 0; q < PPL; ++q) {
                const double rr = decltype(clamp)::value ? fmax(r2[q], min_r2) : r2[q];  // :77
                double y = (double)__builtin_amdgcn_rcpf((float)rr);
                y = fma(fma(-rr, y, 1.0), y, y);
                double y3 = y * y * y;
                if (decltype(test)::value) y3 = rr < rc2 ? y3 : 0.0;  // src/computegridsheet.h:79
                b3[q] += y3;
                b6[q] = fma(y3, y3, b6[q]);
            }
        };
        using no = std::integral_constant<bool, false>;
        using yes = std::integral_constant<bool, true>;
        auto scale = [&]() {
#pragma unroll
            for (int q = 0; q < PPL; ++q) {
                acc[q] = fma(c6, b6[q], fma(c3, b3[q], acc[q]));
                b3[q] = b6[q] = 0.0;
            }
        };
        // a run of records of one kind, in parts if the sums are
        auto run = [&](int n, auto group, auto &&add) {
            constexpr int G = decltype(group)::value;
            if constexpr (PB::on && !PB::one) {
                for (int k = 0; k < n;) {
                    if (pb.ended()) scale();
                    const int e = k + G * pb.run(acc, groups_of(n - k, G));
                    add(k, e < n ? e : n);
                    k = e;
                }
            } else {
                int b = 0, e = n;
                if constexpr (PB::one) pb.clip(b, e, G);
                add(b, e);
            }
        };
        using shells = std::integral_constant<int, kShellGroup>;
        // (NEAR records in flight: a 173^3-point grid of 424 atoms takes 745 us with one,
        // 662 with two, 663 with four)
        run(fe - fb, shells(), [&](int b, int e) {
#pragma unroll NEAR
            for (int k = b; k < e; ++k) fp64_pair(L[fb + k], no(), no());
        });
        // wave lists of an FP64 tile hold as many entries as an FP32 tile's
        // (the far + shell part of the FP32 list), which keeps four
        // workgroups per CU; a segment with more shell records than that
        // takes the tile-level path
        const int wcap = mixed_far_shell_cap(cap);
        if (ws && (PB::on || se - sb <= wcap)) {
            // shell records against the wave's own sphere (as for FP32
            // grids): wave-far ones need no cutoff test, those beyond r_c of
            // every point of the wave contribute exactly 0 and are skipped
            int nwf, nws, first = 0, last = wcap - 1;  // (entries of wl)
            if constexpr (PB::on) {
                const int w = __builtin_amdgcn_readlane(lengths, s);
                nwf = w & 0xffff;
                nws = w >> 16;
                first = sb;
                last = se - 1;
            } else {
                wave_shell_lists(J, Ls, capA, wcap, sb, se, wsph, wl, nwf, nws);
            }
            const char *__restrict__ Lb = reinterpret_cast<const char *>(L);
            run(nwf, shells(), [&](int b, int e) {
#pragma unroll NEAR
                for (int k = b; k < e; ++k)
                    fp64_pair(*reinterpret_cast<const double4 *>(Lb + wl[first + k]), no(), no());
            });
            run(nws, shells(), [&](int b, int e) {
#pragma unroll NEAR
                for (int k = b; k < e; ++k)
                    fp64_pair(*reinterpret_cast<const double4 *>(Lb + wl[last - k]), no(), yes());
            });
        } else {
            run(se - sb, shells(), [&](int b, int e) {
                for (int k = b; k < e; ++k) fp64_pair(Ls[-(sb + k)], no(), yes());
            });
        }
        // Near records (an atom within R of the tile centre, where a grid
        // point may sit on the atom): r^2 from the FP64 differences, as
        // src/computegridsheet.h:71-75 forms it, so that a point on an atom
        // gives exactly 0 and the reference's clamp (the expanded form would
        // leave a rounding residue of either sign there).
        run(ne - nb, std::integral_constant<int, kNearGroup>(), [&](int b, int e) {
            for (int k = nb + b; k < nb + e; ++k) {
                const double4 A = Ln[k];
#pragma unroll
                for (int q = 0; q < PPL; ++q) {
                    const double dx = px[q] - A.x, dy = py[q] - A.y, dz = pz[q] - A.z;
                    const double rr = fmax(dx * dx + dy * dy + dz * dz, min_r2);  // :77
                    double y = (double)__builtin_amdgcn_rcpf((float)rr);
                    y = fma(fma(-rr, y, 1.0), y, y);
                    y = fma(fma(-rr, y, 1.0), y, y);
                    double y3 = y * y * y;
                    y3 = rr < rc2 ? y3 : 0.0;  // src/computegridsheet.h:79
                    b3[q] += y3;
                    b6[q] = fma(y3, y3, b6[q]);
                }
            }
        });
        scale();
    }
    if constexpr (PB::on && !PB::one) pb.flush(acc);
}

// ---- far field of a block of tiles from nodes -------------------------------
//
// Lagrange weights of the kNodes Chebyshev nodes x_a = cos((2 a + 1) pi / 16) at
// the m equally spaced points of an axis whose first and last lie at -1 and 1
// (m = 1: at 0): w[m][i][a].
struct NodeWeights {
    double x[kNodes];
    double w[17][16][kNodes];
};

constexpr NodeWeights make_node_weights() {
    NodeWeights t{};
    const double c[4] = {0.98078528040323044912618, 0.83146961230254523707878,
                         0.55557023301960222474283, 0.19509032201612826784829};
    for (int a = 0; a < 4; ++a) {
        t.x[a] = c[a];
        t.x[kNodes - 1 - a] = -c[a];
    }
    for (int m = 1; m <= 16; ++m)
        for (int i = 0; i < m; ++i) {
            const double z = m > 1 ? (2.0 * i - (m - 1)) / (m - 1) : 0.0;
            for (int a = 0; a < kNodes; ++a) {
                double p = 1.0, q = 1.0;
                for (int b = 0; b < kNodes; ++b)
                    if (b != a) {
                        p *= z - t.x[b];
                        q *= t.x[a] - t.x[b];
                    }
                t.w[m][i][a] = p / q;
            }
        }
    return t;
}

static __device__ const NodeWeights kNodeWeights = make_node_weights();

// A block's node values (LDS, [a][b][c]) and where a tile lies in it.
struct BlockNodes {
    const double *value = nullptr;  // nullptr: no nodes
    int points[3] = {1, 1, 1};      // grid points of the block per axis (at most 16)
    int first[3] = {0, 0, 0};       // the tile's first point in the block
};

// This lane's two points (il + 4 q, jl, kl) of an 8 x 8 x 8 tile: the block's
// interpolated far field, one axis after the other; g and h: 512 doubles each.
__device__ __forceinline__ void node_energies(const BlockNodes &bn, int il, int jl, int kl,
                                              double *__restrict__ g, double *__restrict__ h,
                                              double (&e)[2]) {
    auto row = [&](int d, int l) {
        const int i = bn.first[d] + l;
        return kNodeWeights.w[bn.points[d]][i < bn.points[d] ? i : bn.points[d] - 1];
    };
    double w[kNodes];
    const double *r = row(2, kl);
#pragma unroll
    for (int c = 0; c < kNodes; ++c) w[c] = r[c];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const double *v = bn.value + ((il + 4 * q) * kNodes + jl) * kNodes;
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < kNodes; ++c) s = fma(w[c], v[c], s);
        g[((il + 4 * q) * kNodes + jl) * 8 + kl] = s;
    }
    __syncthreads();
    r = row(1, jl);
#pragma unroll
    for (int b = 0; b < kNodes; ++b) w[b] = r[b];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const double *v = g + (il + 4 * q) * kNodes * 8 + kl;
        double s = 0.0;
#pragma unroll
        for (int b = 0; b < kNodes; ++b) s = fma(w[b], v[b * 8], s);
        h[((il + 4 * q) * 8 + jl) * 8 + kl] = s;
    }
    __syncthreads();
    double v[kNodes];
#pragma unroll
    for (int a = 0; a < kNodes; ++a) v[a] = h[(a * 8 + jl) * 8 + kl];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        r = row(0, il + 4 * q);
        e[q] = 0.0;
#pragma unroll
        for (int a = 0; a < kNodes; ++a) e[q] = fma(r[a], v[a], e[q]);
    }
}

// Energies of one grid tile (tile coordinates tc), candidates streamed from
// src / tbeg (the framework's near list, or a region's sub-list of it).
// (PARTS: sums in parts, see there; such jobs have the quadrant layout)
template <int PPL, int MATH, bool PARTS = false>
__device__ void grid_tile(const JobDev *__restrict__ J, const int tc[3],
                          const double4 *__restrict__ src, const uint32_t *__restrict__ sidx,
                          const int *__restrict__ tbeg, int cap,
                          double4 *__restrict__ s_list, int *__restrict__ s_seg,
                          int *__restrict__ s_cnt, uint16_t *__restrict__ s_wl,
                          const BlockNodes nodes = BlockNodes()) {
    const int tid = threadIdx.x;
    int i0[3], i1[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        i0[d] = tc[d] * J->tile[d];
        const int e = i0[d] + J->tile[d];
        i1[d] = (e < J->n[d] ? e : J->n[d]) - 1;
    }
    const int t0 = J->tile[0], t1 = J->tile[1], t2 = J->tile[2];
    const Tile tl = points_sphere(J, i0, i1,
                                  i1[0] - i0[0] == t0 - 1 && i1[1] - i0[1] == t1 - 1 &&
                                      i1[2] - i0[2] == t2 - 1,
                                  J->cell_R);
    double px[PPL], py[PPL], pz[PPL], acc[PPL];
    long long oidx[PPL];
    bool ok[PPL];
    // Quadrant layout (see quadrant_tile): wave w owns the (j, k) quadrant
    // (w & 1, w >> 1) of the tile and all of its i; lane l holds points
    // i = il + q * t0 / PPL.  Otherwise point p = tid + 256 q of the tile in
    // k-fastest order.
    const int wave = tid >> 6, lane = tid & 63;
    const bool quad = (MATH == MATH_MIXED || MATH == MATH_FP64) &&
                      quadrant_tile(J->tile, PPL, near_region_start<MATH>(cap));
    const int h1 = t1 / 2, h2 = t2 / 2;
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
        int gi, gj, gk;
        if (quad) {
            gi = i0[0] + lane / (h1 * h2) + q * (t0 / PPL);
            gj = i0[1] + (wave & 1) * h1 + (lane / h2) % h1;
            gk = i0[2] + (wave >> 1) * h2 + lane % h2;
        } else {
            const int p = q * kWG + tid;
            gi = i0[0] + p / (t1 * t2);
            gj = i0[1] + (p / t2) % t1;
            gk = i0[2] + p % t2;
        }
        ok[q] = gi <= i1[0] && gj <= i1[1] && gk <= i1[2];
        if (!ok[q]) {
            gi = i0[0];
            gj = i0[1];
            gk = i0[2];
        }
        frac_to_cart(J->t, grid_frac(J, 0, gi), grid_frac(J, 1, gj), grid_frac(J, 2, gk), px[q],
                     py[q], pz[q]);
        px[q] -= tl.cx;
        py[q] -= tl.cy;
        pz[q] -= tl.cz;
        oidx[q] = (long long)gk + (long long)gj * J->n[2] + (long long)gi * J->n[1] * J->n[2];
        acc[q] = 0.0;
    }
    // A lane's points differ only in i (quadrant layout, or p = tid + 256 q
    // with t1 * t2 dividing 256), so on a cell whose first vector lies along
    // x (t_yx = t_zx = 0, as cell parameters give it) only in x.
    const bool xl = PPL > 1 && (quad || kWG % (t1 * t2) == 0) && J->t[3] == 0.0 &&
                    J->t[6] == 0.0;
    // The sphere around this wave's valid points (quadrant layout): its
    // index box is the tile's i range times the quadrant's j and k ranges.
    bool ws = false, idle = false;
    double4 wsph = make_double4(0.0, 0.0, 0.0, 0.0);
    if (quad) {
        const int jb = i0[1] + (wave & 1) * h1, kb = i0[2] + (wave >> 1) * h2;
        const int je = jb + h1 - 1 < i1[1] ? jb + h1 - 1 : i1[1];
        const int ke = kb + h2 - 1 < i1[2] ? kb + h2 - 1 : i1[2];
        idle = jb > i1[1] || kb > i1[2];  // no point of this wave is on the grid
        if (!idle) {
            const int w0[3] = {i0[0], jb, kb}, w1[3] = {i1[0], je, ke};
            const Tile w = points_sphere(J, w0, w1,
                                         i1[0] - i0[0] == t0 - 1 && je - jb == h1 - 1 &&
                                             ke - kb == h2 - 1,
                                         J->wave_R);
            wsph = make_double4(w.cx - tl.cx, w.cy - tl.cy, w.cz - tl.cz, w.R);
            ws = true;
        }
    }
    int cur_t = 0, cur_pos = uniform(tbeg[0]);
    do {
        const int nseg =
            fill_list<MATH, kWG>(J, src, sidx, tbeg, tl, cur_t, cur_pos, cap, s_list, s_seg, s_cnt);
        __syncthreads();
        if constexpr (PARTS) {
            // the wave's shell lists of every segment, their lengths in lane s
            const int capA = near_region_start<MATH>(cap);
            int lengths = 0;
            for (int s = 0; s < nseg && !idle; ++s) {
                const int sb = uniform(s_seg[kSegInts * s + 2]),
                          se = uniform(s_seg[kSegInts * (s + 1) + 2]);
                int nwf = 0, nws = 0;
                if (se > sb)
                    wave_shell_lists(J, s_list + capA - 1, capA, se - sb, sb, se, wsph,
                                     s_wl + sb, nwf, nws);
                if (lane == s) lengths = nwf | nws << 16;
            }
            const int2 groups = count_groups(s_seg, nseg, [&](int s) {
                return __builtin_amdgcn_readlane(lengths, s);
            });
            double e[PPL], sum[PPL];
#pragma unroll
            for (int q = 0; q < PPL; ++q) e[q] = sum[q] = 0.0;
            const PartSums<PPL> pb(sum, groups.x + groups.y, uniform(J->parts));
            if (idle) {
            } else if (xl) {
                eval_list<PPL, MATH, true, 2>(J, s_list, cap, s_seg, nseg, px, py, pz, e, tl.R, ws,
                                              wsph, s_wl, 0, pb, lengths);
            } else {
                eval_list<PPL, MATH, false, 2>(J, s_list, cap, s_seg, nseg, px, py, pz, e, tl.R,
                                               ws, wsph, s_wl, 0, pb, lengths);
            }
#pragma unroll
            for (int q = 0; q < PPL; ++q) acc[q] += sum[q];
        } else if (!idle) {
            if (xl)
                eval_list<PPL, MATH, true, 2>(J, s_list, cap, s_seg, nseg, px, py, pz, acc, tl.R,
                                              ws, wsph, s_wl);
            else
                eval_list<PPL, MATH, false, 2>(J, s_list, cap, s_seg, nseg, px, py, pz, acc, tl.R,
                                               ws, wsph, s_wl);
        }
        __syncthreads();
    } while (cur_t < J->ntypes);
    if constexpr (MATH == MATH_MIXED && PPL == 2) {
        if (nodes.value) {  // 8 x 8 x 8 tile in the quadrant layout (see use_nodes)
            double far[2], *g = reinterpret_cast<double *>(s_list);
            node_energies(nodes, lane >> 4, (wave & 1) * 4 + ((lane >> 2) & 3),
                          (wave >> 1) * 4 + (lane & 3), g, g + 512, far);
            acc[0] += far[0];
            acc[1] += far[1];
        }
    }
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
        if (!ok[q]) continue;
        if (MATH == MATH_COUNT) {
            ((uint32_t *)J->out)[oidx[q]] = (uint32_t)acc[q];
        } else if (MATH == MATH_OVERLAP) {
            // src/computegridsheet.h:159-162
            ((double *)J->out)[oidx[q]] = acc[q] > 0.0 ? 0.0 : 1.0;
        } else if (J->mode == OUT_F64) {
            ((double *)J->out)[oidx[q]] = acc[q];
        } else {
            const double v = acc[q] < (double)FLT_MAX ? acc[q] : (double)FLT_MAX;
            ((float *)J->out)[oidx[q]] = (float)v;
        }
    }
}

// Sub-list of the near list for a region of tiles: every image atom within
// r_c + R of the region centre c, where R bounds |c_t - c| + R_t over the
// region's tiles.  Any atom a tile's own fill would keep (d_t - R_t < r_c)
// therefore lies in the sub-list, and the sub-list keeps the near-list order,
// so every tile builds exactly the list it would build from the near list.
// The sub-list holds near-list indices (4 bytes a record): the records
// themselves are read from the near list, which every workgroup on a
// framework shares (it stays in L2), while each workgroup's sub-list is its
// own.  Returns false (and builds nothing usable) if the sub-list exceeds
// cap_s.
__device__ bool build_region_list(const JobDev *__restrict__ J, double cx, double cy, double cz,
                                  double in2, uint32_t *__restrict__ out, int cap_s,
                                  int *__restrict__ rbeg, int *__restrict__ s_cnt) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ntypes = J->ntypes, end = uniform(J->type_begin[ntypes]);
    int n = 0, t = 0;
    for (int pos = 0; pos < end; pos += kWG) {
        const int idx = pos + tid;
        bool keep = false;
        if (idx < end) {
            const double4 A = J->near[idx];
            const double dx = A.x - cx, dy = A.y - cy, dz = A.z - cz;
            keep = dx * dx + dy * dy + dz * dz < in2;
        }
        const uint64_t bk = __ballot(keep);
        if (lane == 0) s_cnt[wave] = __popcll(bk);
        __syncthreads();
        int off = n, tot = 0;
#pragma unroll
        for (int w = 0; w < kWG / 64; ++w) {
            if (w < wave) off += s_cnt[w];
            tot += s_cnt[w];
        }
        __syncthreads();
        if (n + tot > cap_s) return false;  // uniform
        if (keep) out[off + lanes_below(bk)] = (uint32_t)idx;
        // types that begin in this chunk
        for (; t < ntypes; ++t) {
            const int p = uniform(J->type_begin[t]) - pos;
            if (p >= kWG) break;
            if (wave == p >> 6 && lane == 0)
                rbeg[t] = off + __popcll(bk & ((1ull << (p & 63)) - 1ull));
        }
        n = uniform(n + tot);
    }
    for (; t <= ntypes; ++t)
        if (tid == 0) rbeg[t] = n;
    // the sub-list is read back by the waves of this workgroup only
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return true;
}

// A block of up to 2 x 2 x 2 tiles of 8 x 8 x 8 points (first tile b0, bn tiles
// per axis) of a fine FP32 grid.  An atom inside r_c of every point of the
// block and at least kNodeReach half-extents away from it gives a smooth field
// there: its pairs are evaluated at 8 x 8 x 8 Chebyshev nodes of the block's
// box, and the sum is interpolated to the block's 4096 points (node_energies) -- an
// eighth of the pairs.  Every other atom of the source goes into a list of the
// block (blist, in the source's order), from which the tiles are computed
// directly, as without nodes.  Direct tiles are bound by VALU issue (98% of the
// cycles), and at 0.1 A half of what they issue is for such pairs: a grid of
// 1.48e7 points and 3000 atoms (0.21 atoms/A^3) issued 5.0e9 wave instructions
// in 10.3 ms and with nodes 3.5e9 in 7.2 ms (6.6 ms now); one of 4.9e7 points and
// 2400 atoms (0.05 atoms/A^3) took 10.6, then 7.8 ms (6.4 now).
//
// Accuracy: an atom at D from the middle of a segment of half-length h through
// the box has a Chebyshev interpolation error on it of at most
// 2 C(13, 5) (h / 2 D)^8 of its own r^-6 (the Gegenbauer coefficients of
// |D - x|^-6; C(19, 11) for r^-12); with D >= 8 h that is 6e-7 for an atom on the
// segment's own axis and 10 to 100 times less elsewhere.  Against direct FP64
// sums over the far atoms of blocks at 0.1 A (0.12 atoms/A^3, cells of 65 to 112
// degrees, far fields of 300 to 2000 K): 4e-7 to 3e-6 K rms, 2e-5 K at most,
// less than the FP32 arithmetic of the same pairs rounds off.  The nodes' pairs are
// evaluated in FP64 like those of an FP64 grid: interpolated FP32 sums were up to 8%
// further off (rms) than direct tiles, FP64 ones are 8 to 40% nearer
// (|E| < 1000 K, 0.07 to 0.12 A), for 3 to 5% of the grid's time.
//
// Returns no nodes if the block's list does not fit kBlockList entries, which
// depends on the block alone.
__device__ BlockNodes grid_block(const JobDev *__restrict__ J, const int b0[3], const int bn[3],
                           const double4 *__restrict__ src, const uint32_t *__restrict__ sidx,
                           const int *__restrict__ tbeg, uint32_t *__restrict__ blist,
                           int *__restrict__ bbeg, int cap,
                           double4 *__restrict__ s_list, int *__restrict__ s_seg,
                           int *__restrict__ s_cnt) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const double *t = J->t;
    BlockNodes nodes;
    double lo[3], hi[3], half[3], h = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int i0 = b0[d] * J->tile[d], e = i0 + bn[d] * J->tile[d];
        const int i1 = (e < J->n[d] ? e : J->n[d]) - 1;
        nodes.points[d] = i1 - i0 + 1;
        lo[d] = 1.0 * i0 / (J->n[d] - 1);
        hi[d] = 1.0 * i1 / (J->n[d] - 1);
        half[d] = 0.5 * (hi[d] - lo[d]);
        const double hd = half[d] * sqrt(t[d] * t[d] + t[3 + d] * t[3 + d] + t[6 + d] * t[6 + d]);
        h = hd > h ? hd : h;
    }
    const Tile bs = tile_sphere(t, lo, hi);
    const double in2 = (J->rc + bs.R + kMargin) * (J->rc + bs.R + kMargin);
    const double far_r = J->rc - bs.R - kMargin;
    const double far2 = far_r > 0.0 ? far_r * far_r : -1.0;
    // this lane's nodes (a = wave + 4 q, b, c), relative to the block's centre
    double px[2], py[2], pz[2], acc[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        frac_to_cart(t, half[0] * kNodeWeights.x[wave + 4 * q],
                     half[1] * kNodeWeights.x[lane >> 3], half[2] * kNodeWeights.x[lane & 7],
                     px[q], py[q], pz[q]);
        acc[q] = 0.0;
    }
    const bool xl = t[3] == 0.0 && t[6] == 0.0;
    const int ntypes = J->ntypes, end = uniform(tbeg[ntypes]);
    const double reach = (kNodeReach * h) + bs.R + kMargin, reach2 = reach * reach;
    // far records and types first_t .. first_t + nseg - 1 in the list; kept records;
    // types begun (first_t + nseg)
    int nf = 0, nb = 0, first_t = 0, nseg = 0, nt = 0;
    // The first `take` far records at the nodes; what is left of the list is moved to
    // its front.  A pass ends at a number of kept records, not where a chunk of the
    // source does, so the sums depend on the records alone.
    auto evaluate = [&](int take) {
        __syncthreads();
        int ns = nseg;  // types that begin before `take`
        while (ns > 1 && uniform(s_seg[kSegInts * (ns - 1) + 1]) >= take) --ns;
        const int left = nf - take, segs = nseg - ns + 1;
        const double4 rest = s_list[tid < left ? take + tid : 0];
        const int begin = tid < segs ? s_seg[kSegInts * (ns - 1 + tid) + 1] - take : 0;
        __syncthreads();
        if (tid == 0) s_seg[kSegInts * ns + 1] = take;
        __syncthreads();
        if (xl)
            eval_list<2, MATH_FP64, true, 2>(J, s_list, cap, s_seg, ns, px, py, pz, acc, bs.R);
        else
            eval_list<2, MATH_FP64, false, 2>(J, s_list, cap, s_seg, ns, px, py, pz, acc, bs.R);
        __syncthreads();
        first_t += ns - 1;
        if (tid < left) s_list[tid] = rest;
        if (tid < segs) {
            s_seg[kSegInts * tid] = first_t + tid;
            s_seg[kSegInts * tid + 1] = begin > 0 ? begin : 0;
        }
        nf = left;
        nseg = segs;
    };
    const int pass = cap - kWG;  // far records of a pass; one more chunk fits behind them
    for (int i = tid; i <= kMaxSeg; i += kWG)
        s_seg[kSegInts * i + 2] = s_seg[kSegInts * i + 3] = 0;  // no shell, no near records
    for (int pos = 0; pos < end; pos += kWG) {
        const int idx = pos + tid;
        int at = 0;
        bool far = false, keep = false;
        double4 A = make_double4(0.0, 0.0, 0.0, 0.0);
        if (idx < end) {
            at = sidx ? (int)sidx[idx] : idx;
            const double4 S = src[at];
            const double dx = S.x - bs.cx, dy = S.y - bs.cy, dz = S.z - bs.cz;
            const double d2 = dx * dx + dy * dy + dz * dz;
            const double rn = S.w + bs.R + kMargin;
            A = make_double4(dx, dy, dz, d2);
            far = d2 < far2 && d2 > reach2 && d2 > rn * rn;
            keep = d2 < in2 && !far;
        }
        const uint64_t bf = __ballot(far), bk = __ballot(keep);
        if (lane == 0) {
            s_cnt[2 * wave] = __popcll(bf);
            s_cnt[2 * wave + 1] = __popcll(bk);
        }
        __syncthreads();
        int of = nf, ok = nb, tf = 0, tk = 0;
#pragma unroll
        for (int w = 0; w < kWG / 64; ++w) {
            const int cf = s_cnt[2 * w], ck = s_cnt[2 * w + 1];
            if (w < wave) {
                of += cf;
                ok += ck;
            }
            tf += cf;
            tk += ck;
        }
        __syncthreads();
        if (nb + tk > kBlockList) return BlockNodes();  // uniform
        if (far) s_list[of + lanes_below(bf)] = A;
        if (keep) blist[ok + lanes_below(bk)] = (uint32_t)at;
        // types that begin in this chunk
        for (; nt < ntypes; ++nt) {
            const int p = uniform(tbeg[nt]) - pos;
            if (p >= kWG) break;
            if (wave == p >> 6 && lane == 0) {
                const uint64_t below = (1ull << (p & 63)) - 1ull;
                bbeg[nt] = ok + __popcll(bk & below);
                s_seg[kSegInts * nseg] = nt;
                s_seg[kSegInts * nseg + 1] = of + __popcll(bf & below);
            }
            ++nseg;
        }
        nf = uniform(nf + tf);
        nb = uniform(nb + tk);
        if (nf >= pass) evaluate(pass);
    }
    for (; nt <= ntypes; ++nt)
        if (tid == 0) bbeg[nt] = nb;
    if (nf > 0) evaluate(nf);
    // the list's last kNodeRecords records hold the values while the block's
    // tiles are computed (with a list shorter by as much)
    double *value = reinterpret_cast<double *>(s_list + cap - kNodeRecords);
#pragma unroll
    for (int q = 0; q < 2; ++q) value[(wave + 4 * q) * 64 + lane] = acc[q];
    nodes.value = value;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return nodes;
}

constexpr bool parts_math(int math) { return math == MATH_IN_PARTS || math == MATH_IN_PARTS_FP64; }

template <int PPL, int VARIANT>
__global__ __launch_bounds__(kWG, VARIANT == MATH_NODES || parts_math(VARIANT) ? 4 : 1)
void k_tiles(const JobDev *__restrict__ jobs, int njobs, long long total_items,
             unsigned long long *__restrict__ counter, int cap, uint32_t *__restrict__ scratch,
             int scratch_cap) {
    constexpr bool PARTS = parts_math(VARIANT);
    constexpr int MATH = VARIANT == MATH_IN_PARTS        ? MATH_MIXED
                         : VARIANT == MATH_IN_PARTS_FP64 ? MATH_FP64
                                                         : VARIANT;
    extern __shared__ double4 s_list[];
    __shared__ int s_seg[kSegInts * (kMaxSeg + 1)];
    __shared__ int s_cnt[7 * (kWG / 64)];  // fill: 3 counts + 4 stop fields per wave
    __shared__ int s_rbeg[kMaxTypes + 1], s_bbeg[MATH == MATH_NODES ? kMaxTypes + 1 : 1];
    __shared__ long long s_item;
    const int tid = threadIdx.x;
    uint32_t *__restrict__ slice =
        scratch ? scratch + (size_t)blockIdx.x * (size_t)scratch_cap : nullptr;
    // per-wave shell offset lists after the LDS list (FP32 and FP64 grids)
    uint16_t *__restrict__ s_wl = (MATH == MATH_MIXED || MATH == MATH_FP64 || MATH == MATH_NODES)
        ? reinterpret_cast<uint16_t *>(s_list + cap) +
              (tid >> 6) * (PARTS ? near_region_start<MATH>(cap) : mixed_far_shell_cap(cap))
        : nullptr;

    for (;;) {
        if (tid == 0) s_item = (long long)atomicAdd(counter, 1ull);
        __syncthreads();
        const long long item = s_item;
        __syncthreads();
        if (item >= total_items) break;
        int jl = 0, jh = njobs - 1;
        while (jl < jh) {
            const int mid = (jl + jh + 1) >> 1;
            if (jobs[mid].item_begin <= item) jl = mid;
            else jh = mid - 1;
        }
        const JobDev *__restrict__ J = jobs + jl;
        const long long local = item - J->item_begin + J->local0;

        // ---- one region of cells (grid tiles or Widom bins); index
        //      k + j * nz + i * ny * nz over the job's regions ----
        const bool grid = J->kind == JOB_GRID;
        int ncell[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) ncell[d] = grid ? J->ntiles[d] : J->nbins[d];
        long long rem = local;
        int rg[3], t0[3], tn[3];
        rg[2] = (int)(rem % J->nregions[2]);
        rem /= J->nregions[2];
        rg[1] = (int)(rem % J->nregions[1]);
        rg[0] = (int)(rem / J->nregions[1]);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            t0[d] = rg[d] * J->region[d];
            const int e = t0[d] + J->region[d];
            tn[d] = (e < ncell[d] ? e : ncell[d]) - t0[d];
        }
        const int nt = tn[0] * tn[1] * tn[2];
        auto cell_of = [&](int ti, int tc[3]) {
            tc[0] = t0[0] + ti / (tn[1] * tn[2]);
            tc[1] = t0[1] + (ti / tn[2]) % tn[1];
            tc[2] = t0[2] + ti % tn[2];
        };
        const double4 *src = J->near;
        const uint32_t *sidx = nullptr;
        const int *tbeg = J->type_begin;
        // (a lone block of 2 x 2 x 2 tiles streams the near list itself)
        const bool lone = MATH == MATH_NODES && tn[0] <= 2 && tn[1] <= 2 && tn[2] <= 2;
        if (nt > 1 && !lone && slice && J->ntypes <= kMaxTypes) {
            // region centre: middle of its first and last cell's centres, which
            // all others lie between; R: to the corner of that box, and a cell's
            // radius
            int tc[3];
            cell_of(0, tc);
            const Tile ca = cell_sphere(J, tc);
            cell_of(nt - 1, tc);
            const Tile cb = cell_sphere(J, tc);
            const double cx = 0.5 * (ca.cx + cb.cx), cy = 0.5 * (ca.cy + cb.cy),
                         cz = 0.5 * (ca.cz + cb.cz);
            double r2 = 0.0;
            for (int c = 0; c < 4; ++c) {
                double h[3], x, y, z;
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const double w = (tn[d] - 1) * (grid ? J->tile[d] : 1) * J->inv[d];
                    h[d] = (d == 1 && (c & 2)) || (d == 2 && (c & 1)) ? -0.5 * w : 0.5 * w;
                }
                frac_to_cart(J->t, h[0], h[1], h[2], x, y, z);
                const double q = x * x + y * y + z * z;
                r2 = q > r2 ? q : r2;
            }
            const double R = (sqrt(r2) + J->cell_R) * (1.0 + 1e-12) + kMargin;
            const double rr = J->rc + R + kMargin;
            const int room = MATH == MATH_NODES ? scratch_cap - kBlockList : scratch_cap;
            if (build_region_list(J, cx, cy, cz, rr * rr, slice, room, s_rbeg, s_cnt)) {
                sidx = slice;
                tbeg = s_rbeg;
            }
        }
        if constexpr (MATH == MATH_NODES) {
            // regions of a grid with nodes hold whole blocks of 2 x 2 x 2 tiles; a
            // block's list has the end of the slice
            uint32_t *const blist = slice + (scratch_cap - kBlockList);
            for (int bi = 0; bi < tn[0]; bi += 2)
                for (int bj = 0; bj < tn[1]; bj += 2)
                    for (int bk = 0; bk < tn[2]; bk += 2) {
                        const int b0[3] = {t0[0] + bi, t0[1] + bj, t0[2] + bk};
                        const int bn[3] = {bi + 1 < tn[0] ? 2 : 1, bj + 1 < tn[1] ? 2 : 1,
                                           bk + 1 < tn[2] ? 2 : 1};
                        BlockNodes nodes = grid_block(reread(J), b0, bn, src, sidx, tbeg, blist,
                                                      s_bbeg, cap, s_list, s_seg, s_cnt);
                        const uint32_t *bidx = nodes.value ? blist : sidx;
                        const int *bbeg = nodes.value ? s_bbeg : tbeg;
                        for (int ti = 0; ti < bn[0] * bn[1] * bn[2]; ++ti) {
                            const int o0 = ti / (bn[1] * bn[2]), o1 = (ti / bn[2]) % bn[1],
                                      o2 = ti % bn[2];
                            const int tc[3] = {b0[0] + o0, b0[1] + o1, b0[2] + o2};
                            nodes.first[0] = 8 * o0;
                            nodes.first[1] = 8 * o1;
                            nodes.first[2] = 8 * o2;
                            grid_tile<PPL, MATH_MIXED>(reread(J), tc, src, bidx, bbeg,
                                                       cap - kNodeRecords, s_list, s_seg, s_cnt,
                                                       s_wl, nodes);
                        }
                    }
            continue;
        } else {
            for (int ti = 0; ti < nt; ++ti) {
                int tc[3];
                cell_of(ti, tc);
                if (grid) {
                    grid_tile<PPL, MATH, PARTS>(J, tc, src, sidx, tbeg, cap, s_list, s_seg, s_cnt,
                                                s_wl);
                    continue;
                }
                // ---- one Widom bin: every insertion whose point falls in it ----
                // (at most 2 per lane: bins hold a few hundred insertions).  A
                // chunk's slots are c + q*256 + tid; a wave none of whose lanes
                // holds a second slot evaluates one point per lane, and a wave
                // with no slot at all skips the chunk (the energies do not depend
                // on the points per lane).  Each pass adds its near records, then
                // its far and shell records, to the insertion's energy.
                //
                // Saturation (J->sat_e > 0, jobs whose energies only feed the
                // Boltzmann sums): no pair energy is below -eps_ij, and none of a
                // far or shell record (beyond r_FP64 of every point) below
                // -fs_floor eps_ij, so once an insertion's partial energy plus
                // those floors for every record not yet evaluated (-eps_ij of its
                // type for records not yet classified) reaches sat_e = 800 T, its exact
                // energy is at least 800 T as well, exp(-E/T) is exactly 0 in
                // FP64 for both, and neither sum changes.  A wave whose valid insertions are all
                // saturated stops evaluating them; the stored partial energy
                // (>= 800 T) then stands in for the exact one.
                constexpr int PW = PPL > 2 ? 2 : PPL;
                // One pass of this wave's P points (px.., valid where ok) over the
                // LDS list: the near records, then, unless every valid point is
                // saturated by then, the far and shell records.  out = prev + the
                // pass's terms (the terms alone in the first pass).  Returns false,
                // out untouched, if the points were saturated before the pass:
                // their stored energies stand.
                auto one_pass = [&](auto pw, const auto &px, const auto &py, const auto &pz,
                                    const auto &ok, const auto &prev, auto &out, const Tile &tl,
                                    int nseg, bool first, double lb_near, double lb_fs,
                                    double lb_later) {
                    constexpr int P = decltype(pw)::value;
                    double acc[P];
#pragma unroll
                    for (int q = 0; q < P; ++q) acc[q] = 0.0;
                    const bool sat = J->sat_e > 0.0;
                    auto saturated = [&](double lb) {
                        bool all = true;
#pragma unroll
                        for (int q = 0; q < P; ++q)
                            if (ok[q]) all = all && prev[q] + acc[q] + lb >= J->sat_e;
                        return __all(all) != 0;
                    };
                    if (sat && !first && saturated(lb_near + lb_fs + lb_later)) return false;
                    if constexpr (PARTS) {
                        auto wn = [&](int s) {
                            return (uniform(s_seg[kSegInts * (s + 1) + 2]) -
                                    uniform(s_seg[kSegInts * s + 2])) << 16;
                        };
                        // (e: the current part, zero again after each call)
                        double e[P];
#pragma unroll
                        for (int q = 0; q < P; ++q) e[q] = 0.0;
                        const int parts = uniform(J->parts);
                        const int2 groups = count_groups(s_seg, nseg, wn);
                        eval_list<P, MATH, false>(
                            J, s_list, cap, s_seg, nseg, px, py, pz, e, tl.R, false,
                            make_double4(0.0, 0.0, 0.0, 0.0), nullptr, 1,
                            PartSums<P>(acc, groups.x, parts));
                        if (!(sat && saturated(lb_fs + lb_later)))
                            eval_list<P, MATH, false>(
                                J, s_list, cap, s_seg, nseg, px, py, pz, e, tl.R, false,
                                make_double4(0.0, 0.0, 0.0, 0.0), nullptr, 2,
                                PartSums<P>(acc, groups.y, parts));
                    } else {
                        eval_list<P, MATH, false>(J, s_list, cap, s_seg, nseg, px, py, pz, acc,
                                                  tl.R, false, make_double4(0.0, 0.0, 0.0, 0.0),
                                                  nullptr, 1);
                        if (!(sat && saturated(lb_fs + lb_later)))
                            eval_list<P, MATH, false>(
                                J, s_list, cap, s_seg, nseg, px, py, pz, acc, tl.R, false,
                                make_double4(0.0, 0.0, 0.0, 0.0), nullptr, 2);
                    }
#pragma unroll
                    for (int q = 0; q < P; ++q) out[q] = first ? acc[q] : prev[q] + acc[q];
                    return true;
                };
                // A chunk of up to P * 256 of the bin's insertions, slots
                // c + q * 256 + tid: points generated and energies loaded and
                // stored for this pass.
                auto chunk = [&](auto pw, uint64_t c, uint64_t end, const Tile &tl, int nseg,
                                 bool first, double lb_near, double lb_fs, double lb_later) {
                    constexpr int P = decltype(pw)::value;
                    double px[P], py[P], pz[P], prev[P], out[P];
                    uint32_t ins[P];
                    bool ok[P];
#pragma unroll
                    for (int q = 0; q < P; ++q) {
                        const uint64_t p = c + (uint64_t)(q * kWG + tid);
                        ok[q] = p < end;
                        ins[q] = J->sorted[ok[q] ? p : c];
                        double f[3];
                        widom_point(J->seed, J->stream, ins[q], f);
                        frac_to_cart(J->t, f[0], f[1], f[2], px[q], py[q], pz[q]);
                        px[q] -= tl.cx;
                        py[q] -= tl.cy;
                        pz[q] -= tl.cz;
                        prev[q] = first ? 0.0 : J->e_out[ins[q]];
                    }
                    if (!one_pass(pw, px, py, pz, ok, prev, out, tl, nseg, first, lb_near, lb_fs,
                                  lb_later))
                        return;
#pragma unroll
                    for (int q = 0; q < P; ++q)
                        if (ok[q]) J->e_out[ins[q]] = out[q];
                };
                // A bin whose insertions fit one chunk (at most PW * 256, most
                // bins) keeps each lane's points and partial energies in
                // registers across the passes and writes the energies once; the
                // passes add the same terms in the same order as the chunked
                // form, which stores and reloads them after every pass.
                auto resident = [&](auto pw, const double (&X)[PW], const double (&Y)[PW],
                                    const double (&Z)[PW], const bool (&OK)[PW], double (&T)[PW],
                                    const Tile &tl, int nseg, bool first, double lb_near,
                                    double lb_fs, double lb_later) {
                    constexpr int P = decltype(pw)::value;
                    double px[P], py[P], pz[P], prev[P], out[P];
                    bool ok[P];
#pragma unroll
                    for (int q = 0; q < P; ++q) {
                        px[q] = X[q];
                        py[q] = Y[q];
                        pz[q] = Z[q];
                        ok[q] = OK[q];
                        prev[q] = first ? 0.0 : T[q];
                    }
                    if (!one_pass(pw, px, py, pz, ok, prev, out, tl, nseg, first, lb_near, lb_fs,
                                  lb_later))
                        return;
#pragma unroll
                    for (int q = 0; q < P; ++q) T[q] = out[q];
                };
                const int b = (tc[0] * J->nbins[1] + tc[1]) * J->nbins[2] + tc[2];
                const uint32_t s0 = J->bin_start[b], s1 = J->bin_start[b + 1];
                if (s0 == s1) continue;
                const Tile tl = cell_sphere(J, tc);
                // one chunk: this wave's points per lane (wave-uniform; 0 for a
                // wave with no slot); several chunks: -1.  Only the FP32-grid /
                // Widom pair math keeps bins resident: Widom jobs never run with
                // the other variants, whose registers the resident state would
                // only crowd (FP64 grids would drop to three waves per SIMD).
                const uint64_t wv0 = s0 + (uint64_t)(tid & ~63);
                const int mode = (MATH != MATH_MIXED || s1 - s0 > (uint32_t)(PW * kWG)) ? -1
                                 : wv0 >= s1                     ? 0
                                 : (PW > 1 && wv0 + kWG >= s1)   ? 1
                                                                 : PW;
                double rx[PW], ry[PW], rz[PW], rt[PW];
                uint32_t rins[PW];
                bool rok[PW];
#pragma unroll
                for (int q = 0; q < PW; ++q) {
                    rx[q] = ry[q] = rz[q] = rt[q] = 0.0;
                    rins[q] = 0;
                    rok[q] = false;
                    if (q < mode) {
                        const uint64_t p = s0 + (uint64_t)(q * kWG + tid);
                        rok[q] = p < s1;
                        rins[q] = J->sorted[rok[q] ? p : s0];
                        double f[3];
                        widom_point(J->seed, J->stream, rins[q], f);
                        frac_to_cart(J->t, f[0], f[1], f[2], rx[q], ry[q], rz[q]);
                        rx[q] -= tl.cx;
                        ry[q] -= tl.cy;
                        rz[q] -= tl.cz;
                    }
                }
                int cur_t = 0, cur_pos = uniform(tbeg[0]);
                bool first = true;
                do {
                    const int nseg = fill_list<MATH, kWG>(J, src, sidx, tbeg, tl, cur_t, cur_pos,
                                                          cap, s_list, s_seg, s_cnt);
                    __syncthreads();
                    // -eps_ij for every record of this pass (near; far and shell)
                    // and every source record after it
                    double lb_near = 0.0, lb_fs = 0.0, lb_later = 0.0;
                    if (J->sat_e > 0.0) {
                        for (int sg = 0; sg < nseg; ++sg) {
                            const int *g = s_seg + kSegInts * sg, *e = g + kSegInts;
                            const double eps = 0.25 * J->types[uniform(g[0])].eps4;
                            lb_fs -= eps * J->fs_floor *
                                     (double)(uniform(e[1]) - uniform(g[1]) + uniform(e[2]) -
                                              uniform(g[2]));
                            lb_near -= eps * (double)(uniform(e[3]) - uniform(g[3]));
                        }
                        // source records after this pass, each at -eps of its type:
                        // the rest of the current type, then every later type
                        if (cur_t < J->ntypes) {
                            lb_later = -0.25 * J->types[cur_t].eps4 *
                                       (double)(uniform(tbeg[cur_t + 1]) - cur_pos);
                            for (int u = cur_t + 1; u < J->ntypes; ++u)
                                lb_later -= 0.25 * J->types[u].eps4 *
                                            (double)(uniform(tbeg[u + 1]) - uniform(tbeg[u]));
                        }
                    }
                    if (mode == PW)
                        resident(std::integral_constant<int, PW>(), rx, ry, rz, rok, rt, tl, nseg,
                                 first, lb_near, lb_fs, lb_later);
                    else if (PW > 1 && mode == 1)
                        resident(std::integral_constant<int, 1>(), rx, ry, rz, rok, rt, tl, nseg,
                                 first, lb_near, lb_fs, lb_later);
                    for (uint64_t c = s0; mode < 0 && c < s1; c += (uint64_t)(PW * kWG)) {
                        const uint64_t w0 = c + (uint64_t)(tid & ~63);  // wave-uniform
                        if (w0 >= s1) continue;
                        if (PW > 1 && w0 + kWG >= s1)
                            chunk(std::integral_constant<int, 1>(), c, s1, tl, nseg, first, lb_near,
                                  lb_fs, lb_later);
                        else
                            chunk(std::integral_constant<int, PW>(), c, s1, tl, nseg, first,
                                  lb_near, lb_fs, lb_later);
                    }
                    first = false;
                    __syncthreads();
                } while (cur_t < J->ntypes);
#pragma unroll
                for (int q = 0; q < PW; ++q)
                    if (q < mode && rok[q]) J->e_out[rins[q]] = rt[q];
            }
        }
    }
}

// ---- small jobs -----------------------------------------------------------
//
// A grid or Widom run of a few dozen cells leaves most of the device idle: the
// launch takes as long as one workgroup's chain of fills and pairs, with one
// wave on a SIMD to wait for every LDS read and every FP64 result.  Such jobs
// (JobDev::parts) give each cell four workgroups of eight waves, or of four when
// the device would not hold them all at once.  A workgroup has the 128 points of
// one wave of grid_tile or of a bin (two per lane), makes the same lists, and each
// of its waves makes one part of a pass's sums (see "sums in parts").  For grids up
// to twice as many cells as CUs a workgroup of eight waves has a whole cell, two
// waves for each of its four quarters, which share the list: up to four waves on a
// SIMD instead of two, in one round.
//
// us a call, one workgroup of four waves per cell / eight waves a quarter / four:
// FP32 grid of 8 cells, 400 atoms 115 / 50 / 65, 64 cells 88 / 42 / 56, 216 cells
// 83 / 77 / 61, 343 cells 87 / - / 88; Henry run of 1e3 insertions (2 bins), 1500
// atoms 720 / 205 / 304, 2e4 (42) 360 / 111 / 184, 1e5 (209) 300 / 231 / 175, 1.5e5
// (313) 322 / - / 250, 2e5 (417) 343 / - / 373.  Four waves a cell / two waves a
// quarter: FP32 grid of 343 cells, 400 atoms 83 / 69, 512 cells 83 / 71, 729 cells
// 95 / 101; FP64 95 / 79, 95 / 80, 109 / 109.
//
// In company (a batch whose jobs fill the device, see batch_create) the four
// workgroups of a cell only repeat its fills: 256 grids of 0.5 A took 8.4 ms, 4.0 ms
// in k_tiles<., MATH_IN_PARTS>, whose one wave a quarter makes the parts one after
// the other (3.9 ms without parts); 256 Henry runs of 1e5 insertions 13.0 and 6.3 ms,
// a step of both 21.5 and 10.3.

template <int MATH, int WAVES, int PARTS>
__global__ __launch_bounds__(64 * WAVES * PARTS, 4) void k_parts(const JobDev *__restrict__ jobs,
                                                                 int njobs, int cap) {
    constexpr int WG = 64 * WAVES * PARTS;
    extern __shared__ double4 s_list[];
    __shared__ int s_seg[kSegInts * (kMaxSeg + 1)];
    __shared__ int s_wn_all[PARTS][2 * kMaxSeg];
    __shared__ int s_cnt[7 * (WG / 64)];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const long long item = blockIdx.x;
    int jl = 0, jh = njobs - 1;
    while (jl < jh) {
        const int mid = (jl + jh + 1) >> 1;
        if (jobs[mid].item_begin <= item) jl = mid;
        else jh = mid - 1;
    }
    const JobDev *__restrict__ J = jobs + jl;
    const long long local = item - J->item_begin + J->local0;
    const int part = PARTS == 4 ? uniform(wave / WAVES) : (int)(local & 3);
    const int pwave = uniform(wave & (WAVES - 1));  // of the part's waves
    const bool grid = MATH == MATH_FP64 || PARTS == 4 || J->kind == JOB_GRID;
    const int *nc = grid ? J->ntiles : J->nbins;
    int tc[3];
    const long long cell = PARTS == 4 ? local : local >> 2;
    tc[2] = (int)(cell % nc[2]);
    tc[1] = (int)((cell / nc[2]) % nc[1]);
    tc[0] = (int)(cell / ((long long)nc[1] * nc[2]));
    const int capA = near_region_start<MATH>(cap);
    uint16_t *__restrict__ s_wl =
        reinterpret_cast<uint16_t *>(s_list + cap) + (PARTS == 4 ? part * capA : 0);
    int *s_wn = s_wn_all[PARTS == 4 ? part : 0];

    // a tile: the part's quadrant, as a wave of grid_tile has it; a bin: the
    // insertions a wave of k_tiles has of each 512
    int i0[3] = {0, 0, 0}, i1[3] = {0, 0, 0};
    const int h1 = J->tile[1] / 2, h2 = J->tile[2] / 2;
    uint32_t s0 = 0, s1 = 0;
    bool idle = false;
    Tile tl;
    double4 wsph = make_double4(0.0, 0.0, 0.0, 0.0);
    if (grid) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            i0[d] = tc[d] * J->tile[d];
            const int e = i0[d] + J->tile[d];
            i1[d] = (e < J->n[d] ? e : J->n[d]) - 1;
        }
        const int jb = i0[1] + (part & 1) * h1, kb = i0[2] + (part >> 1) * h2;
        const int je = jb + h1 - 1 < i1[1] ? jb + h1 - 1 : i1[1];
        const int ke = kb + h2 - 1 < i1[2] ? kb + h2 - 1 : i1[2];
        idle = jb > i1[1] || kb > i1[2];  // no point of the part is on the grid
        if (PARTS == 1 && idle) return;
        tl = points_sphere(J, i0, i1,
                           i1[0] - i0[0] == J->tile[0] - 1 && i1[1] - i0[1] == J->tile[1] - 1 &&
                               i1[2] - i0[2] == J->tile[2] - 1,
                           J->cell_R);
        const int w0[3] = {i0[0], idle ? i0[1] : jb, idle ? i0[2] : kb};
        const int w1[3] = {i1[0], idle ? i0[1] : je, idle ? i0[2] : ke};
        const Tile w = points_sphere(J, w0, w1,
                                     i1[0] - i0[0] == J->tile[0] - 1 && je - jb == h1 - 1 &&
                                         ke - kb == h2 - 1,
                                     J->wave_R);
        wsph = make_double4(w.cx - tl.cx, w.cy - tl.cy, w.cz - tl.cz, w.R);
    } else {
        const int b = (tc[0] * nc[1] + tc[1]) * nc[2] + tc[2];
        s0 = J->bin_start[b];
        s1 = J->bin_start[b + 1];
        tl = cell_sphere(J, tc);
    }
    const bool xl = grid && J->t[3] == 0.0 && J->t[6] == 0.0;
    // (a grid's part is one round; a bin has one for every 512 insertions)
    for (uint64_t c = run_slot(s0, 64 * part); grid || c < s1; c += 512) {
        double px[2], py[2], pz[2];
        double total = 0.0;  // of point pwave of the part's two
        long long at[2];
        bool ok[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (grid) {
                int gi = i0[0] + lane / (h1 * h2) + q * (J->tile[0] / 2);
                int gj = i0[1] + (part & 1) * h1 + (lane / h2) % h1;
                int gk = i0[2] + (part >> 1) * h2 + lane % h2;
                ok[q] = gi <= i1[0] && gj <= i1[1] && gk <= i1[2];
                if (!ok[q]) {
                    gi = i0[0];
                    gj = i0[1];
                    gk = i0[2];
                }
                frac_to_cart(J->t, grid_frac(J, 0, gi), grid_frac(J, 1, gj), grid_frac(J, 2, gk),
                             px[q], py[q], pz[q]);
                at[q] = (long long)gk + (long long)gj * J->n[2] +
                        (long long)gi * J->n[1] * J->n[2];
            } else {
                const uint64_t slot = c + lane + 256 * q;
                ok[q] = slot < s1;
                at[q] = J->sorted[ok[q] ? slot : c];
                double f[3];
                widom_point(J->seed, J->stream, (uint64_t)at[q], f);
                frac_to_cart(J->t, f[0], f[1], f[2], px[q], py[q], pz[q]);
            }
            px[q] -= tl.cx;
            py[q] -= tl.cy;
            pz[q] -= tl.cz;
        }
        int cur_t = 0, cur_pos = uniform(J->type_begin[0]);
        do {
            const int nseg = fill_list<MATH, WG>(J, J->near, nullptr, J->type_begin, tl,
                                                      cur_t, cur_pos, cap, s_list, s_seg, s_cnt);
            __syncthreads();
            if (grid) {
                // each segment's shell records against the part's points, a wave
                // per segment
                for (int s = pwave; s < nseg; s += WAVES) {
                    const int sb = uniform(s_seg[kSegInts * s + 2]),
                              se = uniform(s_seg[kSegInts * (s + 1) + 2]);
                    int nwf = 0, nws = 0;
                    if (se > sb && !idle)
                        wave_shell_lists(J, s_list + capA - 1, capA, se - sb, sb, se, wsph,
                                         s_wl + sb, nwf, nws);
                    if (lane == 0) {
                        s_wn[2 * s] = nwf;
                        s_wn[2 * s + 1] = nws;
                    }
                }
                __syncthreads();
            }
            // this wave's part of the groups (Widom: of the near ones, and of the others)
            double e[2] = {0.0, 0.0}, far[2] = {0.0, 0.0};
            const double4 none = make_double4(0.0, 0.0, 0.0, 0.0);
            if (!grid) {
                auto wn = [&](int s) {
                    return (uniform(s_seg[kSegInts * (s + 1) + 2]) -
                            uniform(s_seg[kSegInts * s + 2])) << 16;
                };
                const int2 groups = count_groups(s_seg, nseg, wn);
                eval_list<2, MATH, false, 4>(J, s_list, cap, s_seg, nseg, px, py, pz, e, tl.R,
                                             false, none, nullptr, 1,
                                             OnePart(pwave, groups.x, WAVES));
                eval_list<2, MATH, false, 4>(J, s_list, cap, s_seg, nseg, px, py, pz, far, tl.R,
                                             false, none, nullptr, 2,
                                             OnePart(pwave, groups.y, WAVES));
            } else if (!idle) {
                const int lengths =
                    lane < nseg ? s_wn[2 * lane] | s_wn[2 * lane + 1] << 16 : 0;
                const int2 groups = count_groups(s_seg, nseg, [&](int s) {
                    return __builtin_amdgcn_readlane(lengths, s);
                });
                const OnePart part(pwave, groups.x + groups.y, WAVES);
                if (xl)
                    eval_list<2, MATH, true, 4>(J, s_list, cap, s_seg, nseg, px, py, pz, e, tl.R,
                                                true, none, s_wl, 0, part, lengths);
                else
                    eval_list<2, MATH, false, 4>(J, s_list, cap, s_seg, nseg, px, py, pz, e,
                                                 tl.R, true, none, s_wl, 0, part, lengths);
            }
            __syncthreads();
            // the parts of the pass, added in order
            double *red = reinterpret_cast<double *>(s_list);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                red[(2 * wave + q) * 64 + lane] = e[q];
                if (!grid) red[(2 * (wave + WG / 64) + q) * 64 + lane] = far[q];
            }
            __syncthreads();
            if (pwave < 2) {
                const double *r = red + (2 * (PARTS == 4 ? part * WAVES : 0) + pwave) * 64 + lane;
                double sum = 0.0;
                for (int w = 0; w < WAVES; ++w) sum += r[128 * w];
                for (int w = 0; w < WAVES && !grid; ++w) sum += r[128 * (w + WG / 64)];
                total += sum;
            }
            // (the next fill meets two barriers before it writes the list)
        } while (cur_t < J->ntypes);
        if (pwave < 2) {
            const long long o = pwave == 0 ? at[0] : at[1];
            if (pwave == 0 ? ok[0] : ok[1]) {
                if (!grid) J->e_out[o] = total;
                else if (J->mode == OUT_F64) ((double *)J->out)[o] = total;
                else
                    ((float *)J->out)[o] =
                        (float)(total < (double)FLT_MAX ? total : (double)FLT_MAX);
            }
        }
        if (grid) return;
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Reductions
// ---------------------------------------------------------------------------

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Block g of G sums exp(-E/T) (src/doHenry.h:107) and E exp(-E/T) over the
// contiguous insertion range [g n / G, (g+1) n / G) in a fixed order (thread
// stride, then a fixed shuffle tree and the four wave sums in order).  About 70
// VALU instructions a value, most of them the division and the exponential: as 240
// blocks, one wave per SIMD, 1.73e7 energies took 110 us; 39 us now (3.5 TB/s).
__device__ __forceinline__ void widom_partial_block(const double *e, long long n,
                                                   double temperature, long long g, long long G,
                                                   double2 *partials, double *s_b,
                                                   double *s_eb) {
    const long long lo = g * n / G, hi = (g + 1) * n / G;
    double sb = 0.0, seb = 0.0;
    for (long long i = lo + threadIdx.x; i < hi; i += kWG) {
        const double E = e[i];
        const double bz = exp(-E / temperature);
        sb += bz;
        seb += (bz == 0.0) ? 0.0 : E * bz;
    }
    sb = wave_sum(sb);
    seb = wave_sum(seb);
    if ((threadIdx.x & 63) == 0) {
        s_b[threadIdx.x >> 6] = sb;
        s_eb[threadIdx.x >> 6] = seb;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        partials[g] = make_double2((s_b[0] + s_b[1]) + (s_b[2] + s_b[3]),
                                   (s_eb[0] + s_eb[1]) + (s_eb[2] + s_eb[3]));
}

// One block of kWG threads: thread t sums partials t, t + kWG, ... in order,
// then a fixed shuffle tree per wave and the wave sums in order -- the same
// summation order on every run.
__device__ __forceinline__ void widom_final_block(const double2 *partials, int nblk, double *out,
                                                  double *s_b, double *s_eb) {
    double sb = 0.0, seb = 0.0;
#pragma unroll 16
    for (int g = threadIdx.x; g < nblk; g += kWG) {
        sb += partials[g].x;
        seb += partials[g].y;
    }
    sb = wave_sum(sb);
    seb = wave_sum(seb);
    if ((threadIdx.x & 63) == 0) {
        s_b[threadIdx.x >> 6] = sb;
        s_eb[threadIdx.x >> 6] = seb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[0] = (s_b[0] + s_b[1]) + (s_b[2] + s_b[3]);
        out[1] = (s_eb[0] + s_eb[1]) + (s_eb[2] + s_eb[3]);
    }
}

__global__ __launch_bounds__(kWG) void k_widom_partials(const double *e, long long n,
                                                        double temperature, double2 *partials) {
    __shared__ double s_b[kWG / 64], s_eb[kWG / 64];
    widom_partial_block(e, n, temperature, blockIdx.x, gridDim.x, partials, s_b, s_eb);
}

__global__ __launch_bounds__(kWG) void k_widom_final(const double2 *partials, int nblk,
                                                     double *out) {
    __shared__ double s_b[kWG / 64], s_eb[kWG / 64];
    widom_final_block(partials, nblk, out, s_b, s_eb);
}

// Every Widom run of a batch in one launch: block b serves run b / kReduceBlocks.
__global__ __launch_bounds__(kWG) void k_widom_partials_many(const WidomReduce *runs) {
    __shared__ double s_b[kWG / 64], s_eb[kWG / 64];
    const WidomReduce &R = runs[blockIdx.x / kReduceBlocks];
    const int g = blockIdx.x % kReduceBlocks, G = reduce_blocks(R.n);
    if (g >= G) return;
    widom_partial_block(R.e, R.n, R.temperature, g, G, R.partials, s_b, s_eb);
}

__global__ __launch_bounds__(kWG) void k_widom_final_many(const WidomReduce *runs) {
    __shared__ double s_b[kWG / 64], s_eb[kWG / 64];
    const WidomReduce &R = runs[blockIdx.x];
    widom_final_block(R.partials, reduce_blocks(R.n), R.out, s_b, s_eb);
}

__global__ __launch_bounds__(kWG) void k_sum_u32(const uint32_t *v, long long n,
                                                 unsigned long long *out) {
    unsigned long long s = 0;
    for (long long i = (long long)blockIdx.x * kWG + threadIdx.x; i < n;
         i += (long long)gridDim.x * kWG)
        s += v[i];
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(out, s);
}

__global__ __launch_bounds__(kWG) void k_sum_f64_counts(const double *v, long long n,
                                                        unsigned long long *out) {
    unsigned long long s = 0;
    for (long long i = (long long)blockIdx.x * kWG + threadIdx.x; i < n;
         i += (long long)gridDim.x * kWG)
        s += (unsigned long long)v[i];
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(out, s);
}

int grid_blocks(long long n, int per_block, int cap_blocks) {
    long long b = (n + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > cap_blocks) b = cap_blocks;
    return (int)b;
}

template <int PPL, int MATH>
hipError_t launch_tiles_t(const JobDev *jobs, int njobs, long long total, unsigned long long *ctr,
                          int wgs, int cap, uint32_t *scratch, int scratch_cap, hipStream_t s) {
    hipLaunchKernelGGL((k_tiles<PPL, MATH>), dim3(wgs), dim3(kWG),
                       tiles_lds_bytes(cap, MATH), s, jobs, njobs, total, ctr, cap, scratch,
                       scratch_cap);
    return hipGetLastError();
}

template <int PPL, int MATH>
int occupancy_t(int cap) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_tiles<PPL, MATH>, kWG,
                                                     tiles_lds_bytes(cap, MATH)) !=
        hipSuccess)
        return 1;
    return n > 0 ? n : 1;
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

hipError_t launch_near_count(const NearPlan &p, uint32_t *block_count, hipStream_t s) {
    if (p.nblocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_near_count, dim3(p.nblocks), dim3(kWG), 0, s, p, block_count);
    return hipGetLastError();
}

hipError_t launch_near_offsets(const NearPlan &p, const uint32_t *block_count,
                               uint32_t *block_off, int *type_begin, hipStream_t s) {
    hipLaunchKernelGGL(k_near_offsets, dim3(1), dim3(kWG), 0, s, p, block_count, block_off,
                       type_begin);
    return hipGetLastError();
}

hipError_t launch_near_write(const NearPlan &p, const uint32_t *block_off, double4 *near,
                             hipStream_t s) {
    if (p.nblocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_near_write, dim3(p.nblocks), dim3(kWG), 0, s, p, block_off, near);
    return hipGetLastError();
}

hipError_t launch_setup(const JobDev &job, JobDev *d_job, unsigned long long *counter,
                        const BinJob *bin, BinJob *d_bin, hipStream_t s) {
    Setup a;
    a.job = job;
    a.bin = bin ? *bin : BinJob{};
    a.d_job = d_job;
    a.d_bin = bin ? d_bin : nullptr;
    a.counter = counter;
    hipLaunchKernelGGL(k_setup, dim3(1), dim3(kWG), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_fill_u64(unsigned long long *p, unsigned long long v, long long n,
                           hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_u64, dim3(grid_blocks(n, kWG, 4096)), dim3(kWG), 0, s, p, v, n);
    return hipGetLastError();
}

int bin_blocks(uint64_t n, int chunk) { return (int)((n + (uint64_t)chunk - 1) / (uint64_t)chunk); }

// Insertions per binning block: long chunks give long runs per key and few
// global atomics, but a launch needs ~1000 blocks, and a block zeroes and
// flushes its whole histogram, which a chunk of 2 insertions per key pays for.
int bin_chunk(uint64_t total_insertions, long long max_keys) {
    int chunk = kBinWG;
    while (chunk < kBinChunkMax &&
           ((uint64_t)chunk * 1024 < total_insertions || chunk < 2 * max_keys))
        chunk <<= 1;
    return chunk;
}

void bin_groups(long long nbins, int *group, int *ngroups) {
    long long g = 1;
    if (nbins > kBinDirectMax) g = (nbins + kBinGroups - 1) / kBinGroups;
    if (g > kBinGroupMax) g = kBinGroupMax;
    *group = (int)g;
    *ngroups = (int)((nbins + g - 1) / g);
}

hipError_t launch_bin_all(const BinJob *jobs, int njobs, long long total_blocks, int chunk,
                          long long max_keys, int max_group, long long total_groups,
                          bool cleared, hipStream_t s) {
    if (njobs <= 0 || total_blocks <= 0) return hipSuccess;
    if (chunk < kBinWG || chunk > kBinChunkMax || (chunk & (chunk - 1)) ||
        total_blocks > (1LL << 31) - 1 || max_keys <= 0 || max_keys > kBinLdsKeys ||
        max_group < 1 ||
        max_group > kBinGroupMax || total_groups < 0 || total_groups > (1LL << 31) - 1)
        return hipErrorInvalidValue;
    const size_t lds_bytes = sizeof(uint32_t) * (size_t)max_keys;
    if (!cleared) hipLaunchKernelGGL(k_bin_zero, dim3(njobs), dim3(kWG), 0, s, jobs);
    hipLaunchKernelGGL(k_bin_count, dim3((unsigned)total_blocks), dim3(kWG), lds_bytes, s, jobs,
                       njobs, chunk);
    hipLaunchKernelGGL(k_bin_scan, dim3(njobs), dim3(kWG), 0, s, jobs);
    const size_t scatter_lds = 2 * lds_bytes + 6 * (size_t)chunk;
#define ER_SCATTER(P)                                                                          \
    if (chunk == P * kBinWG) {                                                                 \
        static const bool lds_ok =                                                             \
            hipFuncSetAttribute((const void *)k_bin_scatter<P>,                                \
                                hipFuncAttributeMaxDynamicSharedMemorySize,                    \
                                8 * kBinLdsKeys + 6 * P * kBinWG) == hipSuccess;               \
        if (!lds_ok) return hipErrorInvalidValue;                                              \
        hipLaunchKernelGGL(k_bin_scatter<P>, dim3((unsigned)total_blocks), dim3(kBinWG),       \
                           scatter_lds, s, jobs, njobs);                                       \
    }
    ER_SCATTER(1) ER_SCATTER(2) ER_SCATTER(4) ER_SCATTER(8) ER_SCATTER(16)
#undef ER_SCATTER
    if (total_groups > 0)
        hipLaunchKernelGGL(k_bin_fine, dim3((unsigned)total_groups), dim3(kBinWG),
                           sizeof(uint32_t) * (size_t)max_group, s, jobs, njobs);
    return hipGetLastError();
}

size_t tiles_lds_bytes(int cap, int math) {
    size_t b = (size_t)cap * sizeof(double4);
    if (math == MATH_MIXED || math == MATH_FP64 || math == MATH_NODES || math == MATH_IN_PARTS)
        b += (size_t)(kWG / 64) * mixed_far_shell_cap(cap) * sizeof(uint16_t);
    if (math == MATH_IN_PARTS_FP64)
        b += (size_t)(kWG / 64) * near_region_start<MATH_FP64>(cap) * sizeof(uint16_t);
    return (b + 15) & ~(size_t)15;
}

static hipError_t launch_parts(int math, const JobDev *jobs, int njobs, long long total,
                               int cap, hipStream_t s) {
    if (total <= 0) return hipSuccess;
    if (cap < 2 * kWG || total > (1LL << 31) - 1) return hipErrorInvalidValue;
    // a list of shell offsets for each part of the workgroup
#define ER_PARTS(V, M, W, P)                                                                  \
    if (math == V) {                                                                          \
        const size_t lds = (size_t)cap * sizeof(double4) +                                    \
                           (size_t)P * near_region_start<M>(cap) * sizeof(uint16_t);          \
        hipLaunchKernelGGL((k_parts<M, W, P>), dim3((unsigned)total), dim3(64 * W * P),       \
                           (lds + 15) & ~(size_t)15, s, jobs, njobs, cap);                    \
    }
    ER_PARTS(MATH_PARTS8, MATH_MIXED, 8, 1)
    ER_PARTS(MATH_PARTS8_FP64, MATH_FP64, 8, 1)
    ER_PARTS(MATH_PARTS4, MATH_MIXED, 4, 1)
    ER_PARTS(MATH_PARTS4_FP64, MATH_FP64, 4, 1)
    ER_PARTS(MATH_PARTS2, MATH_MIXED, 2, 4)
    ER_PARTS(MATH_PARTS2_FP64, MATH_FP64, 2, 4)
#undef ER_PARTS
    return hipGetLastError();
}

hipError_t launch_tiles(int math, int ppl, const JobDev *jobs, int njobs, long long total,
                        unsigned long long *ctr, int wgs, int cap, uint32_t *scratch,
                        int scratch_cap, hipStream_t s) {
    if (total <= 0) return hipSuccess;
    if (math >= MATH_PARTS8 && math <= MATH_PARTS2_FP64)
        return launch_parts(math, jobs, njobs, total, cap, s);
    if (cap < 2 * kWG || wgs <= 0) return hipErrorInvalidValue;
    if (scratch && scratch_cap < kWG) return hipErrorInvalidValue;
    if (math == MATH_NODES &&
        (!scratch || scratch_cap < kBlockList + kWG || cap < 2 * kWG + kNodeRecords))
        return hipErrorInvalidValue;
#define ER_TILES(P, M)                                                                     \
    if (ppl == P && math == M)                                                             \
        return launch_tiles_t<P, M>(jobs, njobs, total, ctr, wgs, cap, scratch, scratch_cap, s);
    ER_TILES(1, MATH_MIXED) ER_TILES(2, MATH_MIXED) ER_TILES(4, MATH_MIXED)
    ER_TILES(1, MATH_FP64) ER_TILES(2, MATH_FP64) ER_TILES(4, MATH_FP64)
    ER_TILES(1, MATH_COUNT) ER_TILES(2, MATH_COUNT) ER_TILES(4, MATH_COUNT)
    ER_TILES(1, MATH_OVERLAP) ER_TILES(2, MATH_OVERLAP) ER_TILES(4, MATH_OVERLAP)
    ER_TILES(2, MATH_NODES)
    if (parts_math(math)) ppl = 2;  // (insertions have the same energies whatever it is)
    ER_TILES(2, MATH_IN_PARTS) ER_TILES(2, MATH_IN_PARTS_FP64)
#undef ER_TILES
    return hipErrorInvalidValue;
}

int tiles_occupancy(int math, int ppl, int cap) {
#define ER_OCC(P, M) \
    if (ppl == P && math == M) return occupancy_t<P, M>(cap);
    ER_OCC(1, MATH_MIXED) ER_OCC(2, MATH_MIXED) ER_OCC(4, MATH_MIXED)
    ER_OCC(1, MATH_FP64) ER_OCC(2, MATH_FP64) ER_OCC(4, MATH_FP64)
    ER_OCC(1, MATH_COUNT) ER_OCC(2, MATH_COUNT) ER_OCC(4, MATH_COUNT)
    ER_OCC(1, MATH_OVERLAP) ER_OCC(2, MATH_OVERLAP) ER_OCC(4, MATH_OVERLAP)
    ER_OCC(2, MATH_NODES)
    if (parts_math(math)) ppl = 2;
    ER_OCC(2, MATH_IN_PARTS) ER_OCC(2, MATH_IN_PARTS_FP64)
#undef ER_OCC
    return 1;
}

hipError_t launch_widom_partials(const double *e, long long n, double temperature,
                                 double2 *partials, hipStream_t s) {
    hipLaunchKernelGGL(k_widom_partials, dim3(reduce_blocks(n)), dim3(kWG), 0, s, e, n, temperature,
                       partials);
    return hipGetLastError();
}

hipError_t launch_widom_reduce_many(const WidomReduce *runs, int nruns, hipStream_t s) {
    if (nruns <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_widom_partials_many, dim3((unsigned)nruns * kReduceBlocks), dim3(kWG), 0,
                       s, runs);
    hipLaunchKernelGGL(k_widom_final_many, dim3((unsigned)nruns), dim3(kWG), 0, s, runs);
    return hipGetLastError();
}

hipError_t launch_widom_final(const double2 *partials, int nblk, double *out, hipStream_t s) {
    hipLaunchKernelGGL(k_widom_final, dim3(1), dim3(kWG), 0, s, partials, nblk, out);
    return hipGetLastError();
}

hipError_t launch_sum_u32(const uint32_t *v, long long n, unsigned long long *out, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sum_u32, dim3(grid_blocks(n, kWG, 2048)), dim3(kWG), 0, s, v, n, out);
    return hipGetLastError();
}

hipError_t launch_sum_f64_counts(const double *v, long long n, unsigned long long *out,
                                 hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sum_f64_counts, dim3(grid_blocks(n, kWG, 2048)), dim3(kWG), 0, s, v, n,
                       out);
    return hipGetLastError();
}

}  // namespace er
