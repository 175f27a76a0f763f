// Projection in range order, for arc projection of points onto lines that share
// an origin (sector and pyramid scans).
//
// With a common origin a point's distance |p - o|, and with it its radial bin,
// its radial table cell and its sub-sample phase, is the same for every line.
// The points are therefore sorted by bin once per dataset and origin, and a bin
// of a line is a sum over consecutive points: no two waves ever add to the same
// bin, so the sums live in registers and the kernel has no atomics at all.
//
//   sort      range_count_kernel, range_scan_kernel, range_scatter_kernel: a
//             counting sort into 32-byte records (RangeRec) with the bin, the
//             distance and the phase rotation already evaluated.
//   project   a wave owns a patch of up to 64 lines near one another in direction
//             (one line per lane) and a run of bins.  It tests 64 points at a time
//             (one per lane) against the patch's bounds, and walks the points that
//             can reach the patch one by one: the point's values go to scalar
//             registers, every lane evaluates its own line's weight, and a register
//             per lane collects the bin until the points move on to the next bin.
//             Four finished bins of a line are stored at a time.
//   table     a workgroup's waves share a window of bins.  The radial cells of a
//             lookup-table beam that the window's distances can use are staged in
//             LDS, cut to the samples above the weight cutoff, each sample with its
//             radial difference: the eight corners of a lookup are four LDS reads.
//
// What bounds it: VALU issue.  A (point, patch) visit is about 50 instructions for 64
// lines with a table and 30 with a Gaussian.  1M points, 4096 lines, table 256 x 64 x 64:
// 7.3M visits, 46 % of the lanes' lines in reach, 448.8M wave instructions in 1.71M cycles on
// 1024 SIMDs, one in 3.9 cycles, 0.69 of the rate at which fused multiply-adds issue on this
// card (LDS waits are few).  A Gaussian sector (509 lines x 333k points), whose 7680 waves end
// unevenly: one in 6.1 cycles, 0.43.  The tile kernel waits on the table
// gathers' cache lines (one L1 miss a pair) and on float LDS atomics (a lane in three
// cycles) instead.  Frame times, tile kernel -> range order, frames of three simulators
// in flight with one convolution kernel: that volume 1.91 -> 0.83 ms (with that of
// convolve_fixed.hip 0.77), with phase delay (two atomics a pair there, one more register here)
// 2.91 -> 1.05 (1.00); 768 lines x 200k points 0.174 -> 0.072 (0.060); Gaussian sectors of 509
// lines x 333k points 0.173 -> 0.051 (0.046), 128 x 100k 0.0229 -> 0.0138 (0.0127).
// 64 lines a patch because a lane is a line: patches of 32 lines, two points at a time,
// would visit 0.8 as often and need three instructions for each value read of a lane.
//
// Compiled with -ffp-contract=off (see proj_math.h): bins, distances and the beam
// coordinates round as in the tile kernel.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "proj_math.h"
#include "sim_device.h"

namespace bcsim_hip {

// ---- sort ----------------------------------------------------------------------

// Bin of point i among its distance's points, or -1 (outside every line).
__device__ __forceinline__ int range_bin(const ProjCommon& c, const float4& p, float ox, float oy, float oz, float3& d,
                                         float& absd, double& ti) {
    d = make_float3(p.x - ox, p.y - oy, p.z - oz);
    absd = sqrt_distance(d.x * d.x + d.y * d.y + d.z * d.z);
    return radial_bin(c, absd, ti);
}

// Adds the points of each bin to count; rank[i]: point i's place among its bin's.
__global__ __launch_bounds__(256) void range_count_kernel(ProjCommon c, FixedSet s, int* __restrict__ count,
                                                          int* __restrict__ rank) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= s.n) return;
    const LineGeom& L = c.lines[0];
    float3 d;
    float absd;
    double ti;
    const int bin = range_bin(c, s.pts[i], L.ox, L.oy, L.oz, d, absd, ti);
    rank[i] = bin >= 0 ? atomicAdd(&count[bin], 1) : -1;
}

// start[b] = points of the bins before b; the counts go back to zero for the next sort.
__global__ __launch_bounds__(1024) void range_scan_kernel(int* __restrict__ count, int* __restrict__ start) {
    constexpr int Q = kRangeBins / 1024;
    __shared__ int wsum[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int4* mine = reinterpret_cast<int4*>(count + threadIdx.x * Q);
    int v[Q], sum = 0;
#pragma unroll
    for (int q = 0; q < Q / 4; q++) {
        const int4 c = mine[q];
        v[4 * q] = c.x, v[4 * q + 1] = c.y, v[4 * q + 2] = c.z, v[4 * q + 3] = c.w;
        sum += c.x + c.y + c.z + c.w;
        mine[q] = make_int4(0, 0, 0, 0);
    }
    int incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(incl, d);
        if (lane >= d) incl += t;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int run = incl - sum;
    for (int w = 0; w < wave; w++) run += wsum[w];
    if (threadIdx.x == 0) start[0] = 0;
#pragma unroll
    for (int q = 0; q < Q; q++) start[1 + threadIdx.x * Q + q] = (run += v[q]);
}

__global__ __launch_bounds__(256) void range_scatter_kernel(ProjCommon c, FixedSet s, const int* __restrict__ start,
                                                            const int* __restrict__ rank,
                                                            RangeRec* __restrict__ recs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= s.n || rank[i] < 0) return;
    const LineGeom& L = c.lines[0];
    const float4 p = s.pts[i];
    float3 d;
    float absd;
    double ti;
    const int bin = range_bin(c, p, L.ox, L.oy, L.oz, d, absd, ti);
    float si, co;
    sincosf((float)((double)bin - ti) * c.phase_per_sample, &si, &co);
    float4* dst = reinterpret_cast<float4*>(recs + start[bin] + rank[i]);
    dst[0] = make_float4(d.x, d.y, d.z, p.w);
    dst[1] = make_float4(absd, __int_as_float(bin), co, si);
}

// ---- projection ----------------------------------------------------------------

__device__ __forceinline__ float read_lane(float v, int k) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}

// x*a + y*b + z*c with fused multiply-adds, for the bounds tests.
__device__ __forceinline__ float dot_fused(float x, float y, float z, float a, float b, float c) {
    return __builtin_fmaf(x, a, __builtin_fmaf(y, b, z * c));
}

// max(x, 0) of a number as one integer instruction (fmaxf also quiets NaNs).
__device__ __forceinline__ float at_least_0(float x) { return __int_as_float(max(__float_as_int(x), 0)); }

// Records (r, l, e) of the table that a window can look up, and the slices it holds.
struct RangeRegion {
    int s0, ns;          // first slice and number of slices
    int l0, l1, e0, e1;  // inclusive record ranges; empty: l1 < l0
};

__device__ __forceinline__ RangeRegion range_region(const ProfileParams& P, float r_lo, float r_hi, int max_slices) {
    // a thousandth of a cell (and more for long tables) covers the rounding of a point's cell
    const float m = 1e-3f + 2e-6f * (float)P.nr;
    const float top = (float)(P.nr - 2);
    const float t0 = fminf(fmaxf(floorf((r_lo - P.r_min) * P.inv_dr - m), 0.0f), top);
    const float t1 = fminf(fmaxf(floorf((r_hi - P.r_min) * P.inv_dr + m), 0.0f), top);
    RangeRegion g;
    g.s0 = (int)t0;
    g.ns = min((int)t1 - g.s0 + 2, max_slices);
    g.l0 = 0, g.l1 = P.nl - 2, g.e0 = 0, g.e1 = P.ne - 2;
    if (P.slice_box) {
        int4 u = P.slice_box[g.s0];
        for (int s = 1; s < g.ns - 1; s++) {
            const int4 b = P.slice_box[g.s0 + s];
            u = make_int4(min(u.x, b.x), max(u.y, b.y), min(u.z, b.z), max(u.w, b.w));
        }
        g.l0 = max(g.l0, u.x), g.l1 = min(g.l1, u.y), g.e0 = max(g.e0, u.z), g.e1 = min(g.e1, u.w);
        if (g.e1 < g.e0) g.l1 = g.l0 - 1;
    }
    return g;
}

// Four consecutive bins of one line, stored together (16 bytes, 4-byte aligned).
typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));

// Four bins (b .. b + 3) of a line's run of n bins, real parts h and imaginary parts g;
// dst: the run's first bin in memory.
template <bool PHASE, bool ADD>
__device__ __forceinline__ void put_bin(float* d, float h, float g) {
    d[0] = ADD ? d[0] + h : h;
    if (PHASE) d[1] = ADD ? d[1] + g : g;
}
template <bool PHASE, bool ADD>
__device__ __forceinline__ void put_quad(float* dst, int b, int n, float h0, float h1, float h2, float h3, float g0,
                                         float g1, float g2, float g3) {
    constexpr int E = PHASE ? 2 : 1;
    float* d = dst + b * E;
    if (!ADD && b + 4 <= n) {
        *reinterpret_cast<Quad*>(d) = PHASE ? Quad{h0, g0, h1, g1} : Quad{h0, h1, h2, h3};
        if (PHASE) *reinterpret_cast<Quad*>(d + 4) = Quad{h2, g2, h3, g3};
        return;
    }
    put_bin<PHASE, ADD>(d, h0, g0);
    if (b + 1 < n) put_bin<PHASE, ADD>(d + E, h1, g1);
    if (b + 2 < n) put_bin<PHASE, ADD>(d + 2 * E, h2, g2);
    if (b + 3 < n) put_bin<PHASE, ADD>(d + 3 * E, h3, g3);
}

template <bool PHASE, bool LUT, bool ADD, bool COUNT>
__global__ __launch_bounds__(1024, 8) void project_range_kernel(ProjCommon c, CullParams cp, RangeLaunch R,
                                                                float* __restrict__ out,
                                                                unsigned long long* __restrict__ stats) {
    // Windows are dealt to the XCDs round-robin (workgroups are), and one XCD runs the
    // patches of a window one after another: their points and slices stay in its L2.
    const int windows = (c.num_rf + R.window_bins - 1) / R.window_bins;
    const int groups = (R.n_patches + R.group - 1) / R.group;
    const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
    // Far windows first: they hold the most points, and the short ones fill the tail.
    const int window = windows - 1 - ((turn / groups) * 8 + xcd);
    if (window < 0) return;
    const int patch0 = (turn % groups) * R.group;
    const int b0 = window * R.window_bins;
    const int nb = min(R.window_bins, c.num_rf - b0);
    constexpr bool SINGLE = false, PARTS = false;
    constexpr int part_lo = 0, part_hi = 0, subs = 1;
    constexpr double* sums = nullptr;
#include "range_window.inc"
}

template <bool PHASE, bool LUT, bool ADD, bool COUNT>
static hipError_t launch_range_t(const ProjCommon& c, const CullParams& cp, const RangeLaunch& R, float* out,
                                 unsigned long long* stats, hipStream_t stream) {
    auto k = project_range_kernel<PHASE, LUT, ADD, COUNT>;
    const size_t lds = LUT ? range_lds_bytes(R) : 0;
    hipError_t e = allow_lds((const void*)k, lds);
    if (e != hipSuccess) return e;
    const int windows = (c.num_rf + R.window_bins - 1) / R.window_bins;
    hipLaunchKernelGGL(k, dim3(8 * ((R.n_patches + R.group - 1) / R.group) * ((windows + 7) / 8)), dim3(R.block), lds, stream, c, cp, R, out,
                       stats);
    return hipGetLastError();
}

// The crowded blocks of bins (more than R.split points), which project_range_kernel left at zero:
// a block's points in up to kRangeParts parts, a workgroup takes one part and a few patches, each
// patch by several waves where there are fewer patches than waves.  The waves' sums meet in LDS
// as doubles; a bin then takes one float atomic a part.
// What it is for: a wave of project_range_kernel walks all points of a run, one after another
// (0.17 us a point with a Gaussian, 0.2 with a table).  Points crowded at some distances leave
// the chip to a few such waves.  Frames by the runs alone, with the parts, and by the tile kernel
// (which takes over where that is much the faster): 128 lines x 100k points within 1 mm of depth
// 641 / 48 / 34 us, 512 x 200k 604 / 101 / 101, with a table 3495 / 142 / 205, 64 x 20k points at
// one depth 3344 / 39 / 27.
template <bool PHASE, bool LUT, bool COUNT>
__global__ __launch_bounds__(512, 4) void project_range_parts_kernel(ProjCommon c, CullParams cp, RangeLaunch R,
                                                                     float* __restrict__ out,
                                                                     unsigned long long* __restrict__ stats) {
    constexpr int E = PHASE ? 2 : 1, SUMS = kRangePartPatches * kRangePatch * kRangeBlock * E;
    constexpr bool SINGLE = false, PARTS = true, ADD = true;
    extern __shared__ __attribute__((aligned(16))) float2 cells[];  // the staged cells, then the sums
    double* sums = reinterpret_cast<double*>(reinterpret_cast<char*>(cells) + (LUT ? range_lds_bytes(R) : 0));
    __shared__ unsigned wave_items[8];
    __shared__ unsigned item_of[2];
    const int groups = (R.n_patches + kRangePartPatches - 1) / kRangePartPatches;
    const int blocks = (c.num_rf + kRangeBlock - 1) / kRangeBlock;
    unsigned base = 0, next = blockIdx.x;  // items of the blocks before; this workgroup's next item
    for (int q0 = 0; q0 < blocks; q0 += 512) {
        // items of each thread's block, and of those before it
        const int q = q0 + (int)threadIdx.x;
        unsigned n = 0;
        if (q < blocks) {
            const int len = R.start[kRangeBlock * q + kRangeBlock] - R.start[kRangeBlock * q];
            if (len > R.split) n = (unsigned)range_parts(len) * (unsigned)groups;
        }
        unsigned incl = n;
        for (int d = 1; d < 64; d <<= 1) {
            const unsigned t = __shfl_up(incl, d);
            if ((int)(threadIdx.x & 63) >= d) incl += t;
        }
        if ((threadIdx.x & 63) == 63) wave_items[threadIdx.x >> 6] = incl;
        __syncthreads();
        unsigned total = 0, before = base + incl - n;
        for (int w = 0; w < 8; w++) {
            total += wave_items[w];
            if (w < (int)(threadIdx.x >> 6)) before += wave_items[w];
        }
        __syncthreads();
        for (; next < base + total; next += gridDim.x) {
            if (next >= before && next < before + n) item_of[0] = (unsigned)q, item_of[1] = next - before;
            for (int i = threadIdx.x; i < SUMS; i += 512) sums[i] = 0.0;
            __syncthreads();
            const int b0 = kRangeBlock * (int)__builtin_amdgcn_readfirstlane(item_of[0]);
            const int item = (int)__builtin_amdgcn_readfirstlane(item_of[1]);
            const int nb = min(kRangeBlock, c.num_rf - b0), patch0 = item % groups * kRangePartPatches;
            const int begin = R.start[b0], end = R.start[b0 + nb];
            // parts of the whole block, whose last bins may lie beyond the line
            const int len = R.start[b0 + kRangeBlock] - begin;
            const int each = (len - 1) / range_parts(len) + 1;
            const int part_lo = min(begin + item / groups * each, end), part_hi = min(part_lo + each, end);
            const int patches = min(kRangePartPatches, R.n_patches - patch0);
            const int subs = max(1, 8 / patches);
            {
#include "range_window.inc"
            }
            __syncthreads();
            for (int i = threadIdx.x; i < patches * kRangePatch * kRangeBlock * E; i += 512) {
                const int bin = i / E % kRangeBlock, line = i / E / kRangeBlock;
                const RangePatch& p = R.patches[patch0 + line / kRangePatch];
                const float v = (float)sums[i];
                if (line % kRangePatch < p.n && bin < nb && v != 0.0f)
                    unsafeAtomicAdd(out + ((size_t)p.line[line % kRangePatch] * c.num_rf + b0 + bin) * E + i % E, v);
            }
            __syncthreads();  // the next item reuses the LDS
        }
        base += total;
    }
}

template <bool PHASE, bool LUT, bool COUNT>
static hipError_t launch_parts_t(const ProjCommon& c, const CullParams& cp, const RangeLaunch& R, float* out,
                                 unsigned long long* stats, hipStream_t stream) {
    auto k = project_range_parts_kernel<PHASE, LUT, COUNT>;
    const size_t lds = (LUT ? range_lds_bytes(R) : 0) + range_part_lds_bytes(PHASE);
    const hipError_t e = allow_lds((const void*)k, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(kRangePartGrid), dim3(512), lds, stream, c, cp, R, out, stats);
    return hipGetLastError();
}

// The runs of many jobs' patches, for Gaussian beams.  A job's items share its runs, far ones
// first: 16 waves an item, in workgroups of four (nothing in LDS ties them together).
template <bool PHASE>
__global__ __launch_bounds__(256, 8) void project_range_batch_kernel(const ProjJob* __restrict__ jobs,
                                                                     const int2* __restrict__ items) {
    const int2 w = items[blockIdx.x >> 2];
    const ProjJob& J = jobs[__builtin_amdgcn_readfirstlane(w.x)];
    const ProjCommon& c = J.c;
    const CullParams& cp = J.cp;
    const RangeLaunch& R = J.g.range;
    float* __restrict__ out = J.bins;
    constexpr bool LUT = false, ADD = false, COUNT = false, SINGLE = true, PARTS = false;
    constexpr int part_lo = 0, part_hi = 0, subs = 1;
    constexpr double* sums = nullptr;
    constexpr unsigned long long* stats = nullptr;
    const int turn = __builtin_amdgcn_readfirstlane((blockIdx.x & 3) * 4 + (threadIdx.x >> 6));
    const int all_runs = (c.num_rf + R.run_bins - 1) / R.run_bins;
    for (int u0 = 16 * __builtin_amdgcn_readfirstlane(w.y) + turn; u0 < all_runs * R.n_patches; u0 += 16 * J.blocks_per_slice) {
        const int b0 = (all_runs - 1 - u0 / R.n_patches) * R.run_bins;
        const int nb = min(R.run_bins, c.num_rf - b0), patch0 = u0 % R.n_patches;
#include "range_window.inc"
    }
}

hipError_t launch_range_batch(bool phase, const ProjJob* jobs, const int2* items, int n_items, hipStream_t stream) {
    if (phase) hipLaunchKernelGGL(project_range_batch_kernel<true>, dim3(4 * n_items), dim3(256), 0, stream, jobs, items);
    else hipLaunchKernelGGL(project_range_batch_kernel<false>, dim3(4 * n_items), dim3(256), 0, stream, jobs, items);
    return hipGetLastError();
}

hipError_t launch_range_sort(const ProjCommon& c_in, const FixedSet& s, const RangeLaunch& R, hipStream_t stream) {
    ProjCommon c = c_in;
    c.num_rf = kRangeBins;  // every bin a line of any length can have
    const dim3 grid((s.n + 255) / 256), block(256);
    hipLaunchKernelGGL(range_count_kernel, grid, block, 0, stream, c, s, R.count, R.rank);
    hipLaunchKernelGGL(range_scan_kernel, dim3(1), dim3(1024), 0, stream, R.count, R.start);
    hipLaunchKernelGGL(range_scatter_kernel, grid, block, 0, stream, c, s, R.start, R.rank, R.recs);
    return hipGetLastError();
}

static hipError_t launch_runs(const ProjCommon& c, const CullParams& cp, const RangeLaunch& R, float* out, bool phase,
                              bool lut, int accumulate, unsigned long long* stats, hipStream_t stream) {
#define BCSIM_RANGE(P, U)                                                                  \
    return stats ? (accumulate ? launch_range_t<P, U, true, true>(c, cp, R, out, stats, stream)   \
                               : launch_range_t<P, U, false, true>(c, cp, R, out, stats, stream)) \
                 : (accumulate ? launch_range_t<P, U, true, false>(c, cp, R, out, stats, stream)  \
                               : launch_range_t<P, U, false, false>(c, cp, R, out, stats, stream))
    if (phase) {
        if (lut) BCSIM_RANGE(true, true);
        BCSIM_RANGE(true, false);
    }
    if (lut) BCSIM_RANGE(false, true);
    BCSIM_RANGE(false, false);
#undef BCSIM_RANGE
}

hipError_t launch_project_range(const ProjCommon& c, const CullParams& cp, const RangeLaunch& R, float* out,
                                bool phase, bool lut, int accumulate, unsigned long long* stats, hipStream_t stream) {
    const hipError_t e = launch_runs(c, cp, R, out, phase, lut, accumulate, stats, stream);
    if (e != hipSuccess || !R.split) return e;
#define BCSIM_PARTS(P, U)                                                     \
    return stats ? launch_parts_t<P, U, true>(c, cp, R, out, stats, stream)   \
                 : launch_parts_t<P, U, false>(c, cp, R, out, stats, stream)
    if (phase) {
        if (lut) BCSIM_PARTS(true, true);
        BCSIM_PARTS(true, false);
    }
    if (lut) BCSIM_PARTS(false, true);
    BCSIM_PARTS(false, false);
#undef BCSIM_PARTS
}

}  // namespace bcsim_hip
