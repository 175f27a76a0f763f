// What a frame in range order costs its busiest wave (project_range.hip): how many points crowd
// into a few bins, told from a sample of a dataset's points.  Host code.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <vector>

namespace bcsim_hip {

// Positions of some points of a dataset, evenly spaced in its z-curve order; control-point major
// for splines (cps of them a point).  Fewer of splines, whose sample is looked at for every frame
// at another time (1024 take 8 us of the host's).
struct PointSample {
    static constexpr size_t kPoints = 1024, kSplines = 256;
    size_t n = 0;        // sampled points
    double each = 0.0;   // points of the dataset that one stands for
    int cps = 1;
    std::vector<float> x, y, z;  // [cps][n]

    // Index in [0, points) of each sampled point.
    static std::vector<size_t> choose(size_t points, size_t most) {
        const size_t n = std::min(points, most);
        std::vector<size_t> at(n);
        for (size_t i = 0; i < n; i++) at[i] = (size_t)((double)i * (double)points / (double)n);
        return at;
    }
    void resize(size_t points, size_t most, int cps_) {
        n = std::min(points, most);
        each = n ? (double)points / (double)n : 0.0;
        cps = cps_;
        x.assign(n * (size_t)cps, 0.f), y = z = x;
    }
};

// A cone of lines from one origin: mean axes and how far the lines' lie from them, and the beam's
// reach across them (metres).
struct ScanCone {
    float r[4], l[4], e[4];
    float beam_l, beam_e;
};

// The sample's points seen by a scan, by distance: cells of 2^k blocks of `block` bins.
struct RangeCrowd {
    static constexpr int kLevels = 13;
    double seen = 0.0;               // points of the dataset that the scan can see
    double fullest[kLevels] = {};    // points in the fullest cell of 2^k blocks, surely

    // Points in the fullest `bins` consecutive bins, about: a cell's points spread over it.
    double heaviest(double bins, int block) const {
        double most = 0.0;
        for (int k = 0; k < kLevels; k++) most = std::max(most, fullest[k] * std::min(1.0, bins / (double)(block << k)));
        return most;
    }
};

// (ox, oy, oz): the scan's origin; basis: weights of the control points lo .. lo + count - 1.
// A cell of m sampled points counts as m - 2 sqrt(m): a uniform phantom's fullest cells of a few
// points do not look crowded (1200 frames of uniform points, shells and mixtures: 6 % of the
// uniform ones called crowded by m alone, none so).
inline RangeCrowd range_crowd(const PointSample& s, int lo, int count, const float* basis, float ox, float oy, float oz,
                              const ScanCone& cone, float bins_per_metre, int num_rf, int block) {
    RangeCrowd out;
    const int finest = s.n > 512 ? 0 : 2;  // few points: cells of four blocks tell as much
    const int width = block << finest;
    int n = (num_rf + width - 1) / width;
    std::vector<int> cell(n + 1, 0);  // the last one takes what the scan does not see
    const float to_cell = 1.0f / (float)width, none = (float)n;
    // a few points at a time, in loops without branches
    constexpr size_t kStep = 128;
    float x[kStep], y[kStep], z[kStep], d[kStep], at[kStep];
    for (size_t i0 = 0; i0 < s.n; i0 += kStep) {
        const size_t m = std::min(kStep, s.n - i0);
        for (size_t i = 0; i < m; i++) x[i] = -ox, y[i] = -oy, z[i] = -oz;
        for (int q = 0; q < count; q++) {
            const size_t from = (size_t)(lo + q) * s.n + i0;
            const float *px = &s.x[from], *py = &s.y[from], *pz = &s.z[from], w = basis[q];
            for (size_t i = 0; i < m; i++) x[i] += px[i] * w, y[i] += py[i] * w, z[i] += pz[i] * w;
        }
        for (size_t i = 0; i < m; i++) d[i] = std::sqrt(x[i] * x[i] + y[i] * y[i] + z[i] * z[i]);
        for (size_t i = 0; i < m; i++) {
            const float r = x[i] * cone.r[0] + y[i] * cone.r[1] + z[i] * cone.r[2];
            const float l = x[i] * cone.l[0] + y[i] * cone.l[1] + z[i] * cone.l[2];
            const float e = x[i] * cone.e[0] + y[i] * cone.e[1] + z[i] * cone.e[2];
            const float bin = d[i] * bins_per_metre + 0.5f;
            const bool in = (r > -d[i] * cone.r[3]) & (std::fabs(l) < d[i] * cone.l[3] + cone.beam_l) &
                            (std::fabs(e) < d[i] * cone.e[3] + cone.beam_e) & (bin < (float)num_rf);
            at[i] = in ? bin * to_cell : none;
        }
        for (size_t i = 0; i < m; i++) cell[std::min((int)at[i], n)]++;
    }
    const int seen = (int)s.n - cell[n];
    cell[n] = 0;
    out.seen = seen * s.each;
    for (int k = finest; k < RangeCrowd::kLevels; k++) {
        int most = 0;
        for (int i = 0; i < n; i++) most = std::max(most, cell[i]);
        out.fullest[k] = std::max(0.0, most - 2.0 * std::sqrt((double)most)) * s.each;
        if (n <= 1) break;
        if (n & 1) cell[n] = 0;
        n = (n + 1) / 2;
        for (int i = 0; i < n; i++) cell[i] = cell[2 * i] + cell[2 * i + 1];
    }
    return out;
}

}  // namespace bcsim_hip
