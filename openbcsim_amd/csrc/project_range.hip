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
// lines with a table and 30 with a Gaussian, at about 4.4 cycles a wave instruction
// (1M points, 4096 lines, table 256 x 64 x 64: 7.3M visits, 46 % of the lanes' lines in
// reach; the VALU busy for 0.95 of the kernel).  The tile kernel waits on the table
// gathers' cache lines (one L1 miss a pair) and on float LDS atomics (a lane in three
// cycles) instead.  Frame times, tile kernel -> range order, frames of three simulators
// in flight: that volume 1.91 -> 0.82 ms, with phase delay (two atomics a pair there, one
// more register here) 2.91 -> 1.05 ms; 768 lines x 200k points 0.174 -> 0.072; Gaussian
// sectors of 509 lines x 333k points 0.173 -> 0.051, 128 x 100k 0.0229 -> 0.0134.
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

// One wave: the run of wn bins from b0 on of a patch's lines.  LUT: the table's region G that the
// run can look up is in LDS at `cells`.
template <bool PHASE, bool LUT, bool ADD, bool COUNT>
__device__ __forceinline__ void range_unit(const ProjCommon& c, const CullParams& cp, const RangeLaunch& R,
                                           const RangePatch& patch, int b0, int wn, const RangeRegion& G, int row,
                                           int plane, const float2* cells, float* __restrict__ out, unsigned* counts) {
    constexpr int E = PHASE ? 2 : 1;
    // A Gaussian beam's bins were exact integer sums: doubles keep them so to 1e-16.
    using Acc = typename std::conditional<LUT, float, double>::type;
    const int lane = threadIdx.x & 63;
    const ProfileParams& P = c.prof;
    const char* cell_bytes = reinterpret_cast<const char*>(cells);
    const bool small_x = P.g_cut <= kExpMinusMax;
    const float r_far = (float)(b0 + wn) * cp.r_per_bin;
    const int i1 = R.start[b0 + wn];
    int i0 = R.start[b0];
    const float lx = patch.axes[0][lane], ly = patch.axes[1][lane], lz = patch.axes[2][lane];
    const float ex = patch.axes[3][lane], ey = patch.axes[4][lane], ez = patch.axes[5][lane];
    const int line = patch.line[lane];
    float* dst = lane < patch.n ? out + ((size_t)line * c.num_rf + b0) * E : nullptr;
    // the patch's bounds: a line's coordinate differs from the patch axis's by at most
    // the distance times the largest difference of the axes (a relative 1e-5 for rounding)
    const float m_r = r_far * (patch.dr + 1e-5f), m_l = r_far * (patch.dl + 1e-5f), m_e = r_far * (patch.de + 1e-5f);
    // the window's beam support, and the square of its largest distance from a beam's axis
    const float l_lo = P.l_min + ((float)G.l0 - 1.01f) * cp.lut_dl, l_hi = P.l_min + ((float)G.l1 + 1.01f) * cp.lut_dl;
    const float e_lo = P.e_min + ((float)G.e0 - 1.01f) * cp.lut_de, e_hi = P.e_min + ((float)G.e1 + 1.01f) * cp.lut_de;
    const float l_far = fmaxf(fabsf(l_lo), fabsf(l_hi)), e_far = fmaxf(fabsf(e_lo), fabsf(e_hi));
    const float reach2 = LUT ? l_far * l_far + e_far * e_far : cp.g_max / fminf(cp.g_a, cp.g_b);
    // (A) One point per lane: can it reach a line of the patch (hit), and could one that it
    // reaches see it behind the origin (behind)?  A line that sees a point within its support
    // sees it at least sqrt(distance^2 - reach^2) before or behind the origin.
    struct Seen {
        bool hit, behind;
    };
    const auto test = [&](const float4& p, const float4& q) {
        const float rc = dot_fused(p.x, p.y, p.z, patch.rx, patch.ry, patch.rz);
        const float lc = dot_fused(p.x, p.y, p.z, patch.lx, patch.ly, patch.lz);
        const float ec = dot_fused(p.x, p.y, p.z, patch.ex, patch.ey, patch.ez);
        const float along = 0.9999f * __builtin_amdgcn_sqrtf(fmaxf(0.0f, q.x * q.x - 1.001f * reach2));
        bool hit = rc > -m_r;
        if (LUT) {
            const float tr = (q.x - P.r_min) * P.inv_dr;
            hit = hit && lc > l_lo - m_l && lc < l_hi + m_l && ec > e_lo - m_e && ec < e_hi + m_e &&
                  G.l1 >= G.l0 && tr > -1.0f && tr < (float)(P.nr - 1);
        } else {
            const float dl = fmaxf(0.0f, fabsf(lc) - m_l), de = fmaxf(0.0f, fabsf(ec) - m_e);
            hit = hit && !(cp.g_a * dl * dl + cp.g_b * de * de >= cp.g_max);
        }
        // points within about a sample of the origin may fall into bin 0 on the far side of it
        const bool at_origin = __float_as_int(q.y) <= 1;
        return Seen{hit || at_origin, at_origin || !(rc > m_r - along)};
    };
    // The sums of the bin at hand of this lane's line, and its four bins finished last:
    // scalars of their own (a struct of them ends up in scratch memory).
    Acc re = Acc(0), im = Acc(0);
    float h0 = 0, h1 = 0, h2 = 0, h3 = 0, g0 = 0, g1 = 0, g2 = 0, g3 = 0;
    int cur = 0;  // the bin at hand, of the run
    const auto advance = [&](int to) {
#pragma unroll 1
        for (; cur < to; cur++) {
            h0 = h1, h1 = h2, h2 = h3, h3 = (float)re;
            if (PHASE) g0 = g1, g1 = g2, g2 = g3, g3 = (float)im;
            re = im = Acc(0);
            if ((cur & 3) == 3 && dst) put_quad<PHASE, ADD>(dst, cur - 3, wn, h0, h1, h2, h3, g0, g1, g2, g3);
        }
    };
    bool far_side = false;
    unsigned n_evals = 0, n_adds = 0, n_pairs = 0;
    const float4* recs = reinterpret_cast<const float4*>(R.recs);
    float4 a{}, b{};
    if (i0 < i1) {
        const int i = min(i0 + lane, i1 - 1);
        a = recs[2 * (size_t)i];
        b = recs[2 * (size_t)i + 1];
    }
    for (; i0 < i1; i0 += 64) {
        const bool in = i0 + lane < i1;
        const float4 p = a, q = b;
        if (i0 + 64 < i1) {  // the next 64 points, while these are projected
            const int i = min(i0 + 64 + lane, i1 - 1);
            a = recs[2 * (size_t)i];
            b = recs[2 * (size_t)i + 1];
        }
        const int bin = __float_as_int(q.y) - b0;
        const Seen seen = test(p, q);
        float fr = 0.0f;
        int off = 0;
        if (LUT) {
            const float tr = (q.x - P.r_min) * P.inv_dr;
            const int r0 = (int)tr;  // truncates: a coordinate in (-1, 0) reads slice 0 alone
            fr = fmaxf(tr - (float)r0, 0.0f);
            off = 8 * min(max(r0 - G.s0, 0), G.ns - 2) * plane;  // bytes
        }
        far_side = far_side || __any(in && seen.hit && seen.behind);  // for the end
        unsigned long long mask = __ballot(in && seen.hit && !seen.behind);
        // (B) one line per lane: the points one by one
        while (mask) {
            const int k = __builtin_ctzll(mask);
            mask &= mask - 1;
            const float dx = read_lane(p.x, k), dy = read_lane(p.y, k), dz = read_lane(p.z, k);
            const float amp = read_lane(p.w, k);
            const int lb = __builtin_amdgcn_readlane(bin, k);
            if (lb != cur) advance(lb);
            if (COUNT) n_pairs++;
            // for a Gaussian beam fused: the weight is smooth (a table's edge is not)
            const float l = LUT ? dx * lx + dy * ly + dz * lz : dot_fused(dx, dy, dz, lx, ly, lz);
            const float e = LUT ? dx * ex + dy * ey + dz * ez : dot_fused(dx, dy, dz, ex, ey, ez);
            // w, turned by the phase rotation of the point in lane k
            const auto add = [&](float w) {
                re += (Acc)(PHASE ? w * read_lane(q.z, k) : w);
                if (PHASE) im += (Acc)(w * read_lane(q.w, k));
            };
            float w = 0.0f;
            bool ok;
            if (LUT) {
                const float tl = (l - P.l_min) * P.inv_dl, te = (e - P.e_min) * P.inv_de;
                const unsigned il = (unsigned)((int)tl - G.l0), ie = (unsigned)((int)te - G.e0);
                ok = il <= (unsigned)(G.l1 - G.l0) && ie <= (unsigned)(G.e1 - G.e0);
                if (ok) {
                    const float fl = __builtin_amdgcn_fractf(at_least_0(tl)), fe = __builtin_amdgcn_fractf(at_least_0(te));
                    const float f = read_lane(fr, k);
                    const float2* s = reinterpret_cast<const float2*>(
                        cell_bytes + (__umul24(ie, 8u * row) + (unsigned)__builtin_amdgcn_readlane(off, k) + 8u * il));
                    const float2 s00 = s[0], s10 = s[1], s01 = s[row], s11 = s[row + 1];
                    const float c00 = __builtin_fmaf(f, s00.y, s00.x), c10 = __builtin_fmaf(f, s10.y, s10.x);
                    const float c01 = __builtin_fmaf(f, s01.y, s01.x), c11 = __builtin_fmaf(f, s11.y, s11.x);
                    w = lerp(lerp(c00, c10, fl), lerp(c01, c11, fl), fe);
                    w = fabsf(w) < P.w_cut ? 0.0f : w * amp;
                    add(w);
                }
            } else {
                const float x = l * l * P.inv_tsl + e * e * P.inv_tse;
                ok = !(x > P.g_cut);
                if (ok) {
                    w = (small_x ? exp_minus(x) : expf(-x)) * amp;
                    add(w);
                }
            }
            if (COUNT) {
                n_evals += ok ? 1u : 0u;
                n_adds += w != 0.0f ? (unsigned)E : 0u;
            }
        }
    }
    advance((wn + 3) & ~3);
    if (far_side) {
        // The points set aside, by the tile kernel's rule: the side of the origin that a line
        // sees a point on decides its distance and bin.  Their bins are this wave's, or bin 0
        // from bin 1 (both in the line's first run), and stored by now.
        for (i0 = R.start[b0]; i0 < i1; i0 += 64) {
            const int i = min(i0 + lane, i1 - 1);
            const float4 p = recs[2 * (size_t)i], q = recs[2 * (size_t)i + 1];
            const Seen seen = test(p, q);
            unsigned long long mask = __ballot(i0 + lane < i1 && seen.hit && seen.behind);
            while (mask) {
                const int k = __builtin_ctzll(mask);
                mask &= mask - 1;
                if (COUNT) n_pairs++;
                const float dx = read_lane(p.x, k), dy = read_lane(p.y, k), dz = read_lane(p.z, k);
                const LineGeom& L = c.lines[line];
                const Local o{dx * L.rx + dy * L.ry + dz * L.rz, dx * lx + dy * ly + dz * lz,
                              dx * ex + dy * ey + dz * ez};
                const float r = copysignf(read_lane(q.x, k), o.r);
                int bn = __builtin_amdgcn_readlane(__float_as_int(q.y), k);
                float si = read_lane(q.w, k);
                if (signbit(r)) {
                    // the far side: bin 0, or none.  Its sub-sample delay is that of the near side
                    // negated, or the same half sample where the near side rounds up to bin 1.
                    if (bn == 0) si = -si;
                    double ti;
                    bn = bn <= 1 ? radial_bin(c, r, ti) : -1;
                }
                if (bn < 0 || !dst) continue;
                Tally t;
                const float w =
                    (LUT ? lut_weight(P, r, o.l, o.e, t) : gauss_weight(P, o.l, o.e, t)) * read_lane(p.w, k);
                if (COUNT) n_evals += t.evals, n_adds += w != 0.0f ? (unsigned)E : 0u;
                if (w == 0.0f) continue;
                float* d = dst + (bn - b0) * E;
                d[0] += PHASE ? w * read_lane(q.z, k) : w;
                if (PHASE) d[1] += w * si;
            }
        }
    }
    if (COUNT) {
        if (dst) atomicAdd(&counts[0], n_evals), atomicAdd(&counts[1], n_adds);
        if (lane == 0) atomicAdd(&counts[2], n_pairs);
    }
}

template <bool PHASE, bool LUT, bool ADD, bool COUNT>
__global__ __launch_bounds__(1024, 8) void project_range_kernel(ProjCommon c, CullParams cp, RangeLaunch R,
                                                                float* __restrict__ out,
                                                                unsigned long long* __restrict__ stats) {
    extern __shared__ __attribute__((aligned(16))) float2 cells[];
    __shared__ unsigned counts[3];
    __shared__ int next_unit;
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
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    if (COUNT && threadIdx.x < 3) counts[threadIdx.x] = 0;

    const ProfileParams& P = c.prof;
    RangeRegion G{};
    int row = 0, plane = 0;  // LDS pitch of a table row, and of a radial cell
    if (LUT) {
        G = range_region(P, ((float)b0 - 0.5f) * cp.r_per_bin, ((float)(b0 + nb) - 0.5f) * cp.r_per_bin, R.max_slices);
        const int nl = G.l1 - G.l0 + 2, ne = G.e1 - G.e0 + 2;
        row = nl | 1;
        plane = row * ne;
        if (G.l1 >= G.l0) {
            const int rows = (G.ns - 1) * ne;
            for (int q = wave; q < rows; q += nwaves) {
                const int s = q / ne, e = q - s * ne;
                const float* src = R.table + ((size_t)(G.s0 + s) * P.ne + (G.e0 + e)) * P.nl + G.l0;
                const float* up = src + P.ne * P.nl;
                float2* dst = cells + s * plane + e * row;
                for (int l = lane; l < nl; l += 64) dst[l] = make_float2(src[l], up[l] - src[l]);
            }
        }
    }
    if (threadIdx.x == 0) next_unit = nwaves;
    __syncthreads();

    const int runs = (nb + R.run_bins - 1) / R.run_bins;
    const int units = runs * min(R.group, R.n_patches - patch0);
    const auto claim = [&] {  // the wave's next unit: they differ in how many points reach a patch
        int u = 0;
        if (lane == 0) u = atomicAdd(&next_unit, 1);
        return __builtin_amdgcn_readfirstlane(u);
    };
    for (int u = wave; u < units; u = claim()) {
        const int w0 = (u % runs) * R.run_bins;  // the run's first bin in the window
        range_unit<PHASE, LUT, ADD, COUNT>(c, cp, R, R.patches[patch0 + u / runs], b0 + w0, min(R.run_bins, nb - w0), G,
                                           row, plane, cells, out, counts);
    }
    if (COUNT) {
        __syncthreads();
        if (threadIdx.x < 3) atomicAdd(&stats[threadIdx.x], (unsigned long long)counts[threadIdx.x]);
    }
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

// The runs of many jobs' patches, for Gaussian beams.  A job's items share its runs, far ones
// first: 16 waves an item, in workgroups of four (nothing in LDS ties them together).
template <bool PHASE>
__global__ __launch_bounds__(256, 8) void project_range_batch_kernel(const ProjJob* __restrict__ jobs,
                                                                     const int2* __restrict__ items) {
    const int2 w = items[blockIdx.x >> 2];
    const ProjJob& J = jobs[__builtin_amdgcn_readfirstlane(w.x)];
    const RangeLaunch& R = J.g.range;
    const int wave = __builtin_amdgcn_readfirstlane((blockIdx.x & 3) * 4 + (threadIdx.x >> 6));
    const int runs = (J.c.num_rf + R.run_bins - 1) / R.run_bins, units = runs * R.n_patches;
    for (int u = 16 * __builtin_amdgcn_readfirstlane(w.y) + wave; u < units; u += 16 * J.blocks_per_slice) {
        const int b0 = (runs - 1 - u / R.n_patches) * R.run_bins;
        range_unit<PHASE, false, false, false>(J.c, J.cp, R, R.patches[u % R.n_patches], b0,
                                               min(R.run_bins, J.c.num_rf - b0), RangeRegion{}, 0, 0, nullptr, J.bins,
                                               nullptr);
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

hipError_t launch_project_range(const ProjCommon& c, const CullParams& cp, const RangeLaunch& R, float* out,
                                bool phase, bool lut, int accumulate, unsigned long long* stats, hipStream_t stream) {
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

}  // namespace bcsim_hip
