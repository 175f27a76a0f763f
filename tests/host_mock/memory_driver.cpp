// Test infrastructure (CPU only): the host code around the projection in range order
// under the mock runtime of mock_hip.cpp, with device allocations and copies that fail
// on request.  The mock is compiled with its hipMalloc, hipMemcpy and
// launch_project_tile renamed (mock_*); the ones here inject the failures and check
// what a range-order launch reads before they pass the call on.
//   usage: memory_driver <scenario>
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <random>
#include <string>
#include <vector>
#include <unistd.h>

#include "../../include/bcsim_c.h"
#include "../../openbcsim_amd/csrc/sim_device.h"

using namespace bcsim_hip;

extern "C" hipError_t mock_hipMalloc(void** ptr, size_t size);
extern "C" hipError_t mock_hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind kind);
namespace bcsim_hip {
hipError_t mock_launch_project_tile(const ProjCommon& c, const CullParams& cp, const FixedSet* fixed,
                                    const SplineSet* spline, const ChunkBox* boxes, int nchunks, void* bins, bool arc,
                                    bool phase, bool lut, bool shared_origin, const TileLaunch& cfg, hipStream_t s);
}

#define REQUIRE(x)                                                                                 \
    do {                                                                                           \
        if (!(x)) {                                                                                \
            fprintf(stderr, "FAIL %s:%d %s (%s)\n", __FILE__, __LINE__, #x, bcsim_last_error());    \
            _exit(1);                                                                              \
        }                                                                                          \
    } while (0)
#define CHK(x) REQUIRE((x) == BCSIM_OK)

// ---- failures: the allocation or copy for which the predicate holds fails
static std::function<bool(size_t)> fail_malloc, fail_copy;
static int mallocs = 0;  // allocations of count_bytes
static size_t count_bytes = 0;

extern "C" hipError_t hipMalloc(void** ptr, size_t size) {
    mallocs += size == count_bytes;
    if (fail_malloc && fail_malloc(size)) {
        *ptr = nullptr;
        return hipErrorOutOfMemory;
    }
    return mock_hipMalloc(ptr, size);
}
extern "C" hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind kind) {
    if (fail_copy && fail_copy(n)) return hipErrorUnknown;
    return mock_hipMemcpy(dst, src, n, kind);
}

static bool under_capture = false;
extern "C" hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* status) {
    *status = under_capture ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}

static bool live(const void* p) {
    hipPointerAttribute_t a;
    return p && hipPointerGetAttributes(&a, p) == hipSuccess;
}

static int range_launches = 0;  // projections in range order
static const void* last_records = nullptr;  // of the last one
static float table_value = 0.0f;  // what every sample of the profile's table is

namespace bcsim_hip {
hipError_t launch_project_tile(const ProjCommon& c, const CullParams& cp, const FixedSet* fixed, const SplineSet* spline,
                               const ChunkBox* boxes, int nchunks, void* bins, bool arc, bool phase, bool lut,
                               bool shared_origin, const TileLaunch& cfg, hipStream_t s) {
    const RangeLaunch& R = cfg.range;
    if (R.recs) {
        REQUIRE(live(R.recs) && live(R.start) && !spline);
        REQUIRE(live(fixed->pts));
        if (R.sort) REQUIRE(live(R.count) && live(R.rank));
        if (R.sort != 2) {
            range_launches++;
            last_records = R.recs;
            REQUIRE(live(R.patches) && R.n_patches > 0);
            if (lut) {
                REQUIRE(live(R.table));
                const int n = c.prof.nr * c.prof.nl * c.prof.ne;
                REQUIRE(R.table[0] == table_value && R.table[n - 1] == table_value);
            }
        }
    }
    return mock_launch_project_tile(c, cp, fixed, spline, boxes, nchunks, bins, arc, phase, lut, shared_origin, cfg, s);
}
}  // namespace bcsim_hip

// ---- simulators
struct Scan {
    std::vector<float> o, d, l, t;
    float len = 0.05f;
};
static Scan sector(int n, float x0 = 0.0f) {
    Scan s;
    for (int k = 0; k < n; k++) {
        const double a = -0.6 + 1.2 * k / (n - 1);
        s.o.insert(s.o.end(), {x0, 0, 0});
        s.d.insert(s.d.end(), {(float)sin(a), 0, (float)cos(a)});
        s.l.insert(s.l.end(), {(float)cos(a), 0, (float)-sin(a)});
        s.t.push_back(0);
    }
    return s;
}
static void set_scan(bcsim_sim* s, const Scan& q, bool at_once = false) {
    CHK(bcsim_set_scan_sequence(s, (int)q.t.size(), q.o.data(), q.d.data(), q.l.data(), q.t.data(), q.len, at_once));
}
static std::vector<float> box_points(size_t n) {
    std::mt19937 rng(3);
    std::uniform_real_distribution<float> u(0, 1);
    std::vector<float> p;
    for (size_t i = 0; i < n; i++)
        p.insert(p.end(), {0.05f * u(rng) - 0.025f, 0.004f * u(rng) - 0.002f, 0.005f + 0.04f * u(rng), u(rng) - 0.5f});
    return p;
}
static bcsim_sim* simulator(int lines, size_t points) {
    bcsim_sim* s;
    CHK(bcsim_create("gpu", &s));
    std::vector<float> pulse(55, 0.5f);
    CHK(bcsim_set_excitation(s, pulse.data(), 55, 27, 50e6f, 2.5e6f));
    set_scan(s, sector(lines));
    if (points) {
        const std::vector<float> p = box_points(points);
        CHK(bcsim_add_fixed_scatterers(s, p.data(), points));
    }
    CHK(bcsim_set_analytical_profile(s, 1e-3f, 1e-3f));
    return s;
}
static bcsim_status set_table(bcsim_sim* s, int nr) {
    std::vector<float> t((size_t)nr * 24 * 24, 1.0f / nr);
    const bcsim_status st =
        bcsim_set_lut_profile(s, 0, 0.05f, -0.01f, 0.01f, -0.01f, 0.01f, t.data(), nr, 24, 24);
    if (st == BCSIM_OK) table_value = 1.0f / nr;
    return st;
}
static std::string plan(bcsim_sim* s) {
    char b[2048];
    CHK(bcsim_get_parameter(s, "launch_plan", b, sizeof b));
    return b;
}
// One frame; whether it ran in range order.
static bool ranged(bcsim_sim* s) {
    int L, S;
    CHK(bcsim_get_output_shape(s, &L, &S));
    std::vector<float> out((size_t)L * S * 2);
    const int before = range_launches;
    CHK(bcsim_simulate_lines(s, out.data(), (size_t)L * S, &L, &S));
    const bool r = plan(s).find("range order") != std::string::npos;
    REQUIRE(!r || range_launches > before);  // (trials launch it too)
    return r;
}

// A table whose samples or quads do not fit, or whose copies fail, leaves the profile
// that was there; without room for the samples alone the frames run the tile kernel.
static void table_failures() {
    bcsim_sim* s = simulator(128, 20000);
    CHK(set_table(s, 16));
    REQUIRE(ranged(s));
    int k = 0;
    fail_malloc = [&](size_t) { return ++k == 1; };  // the quads
    REQUIRE(set_table(s, 20) == BCSIM_ERR_OUT_OF_MEMORY);
    fail_malloc = nullptr;
    REQUIRE(ranged(s));  // with the old table
    for (int copy : {1, 2}) {
        k = 0;
        fail_copy = [&](size_t) { return ++k == copy; };
        REQUIRE(set_table(s, 20) == BCSIM_ERR_DEVICE);
        fail_copy = nullptr;
        REQUIRE(ranged(s));
    }
    k = 0;
    fail_malloc = [&](size_t) { return ++k == 2; };  // the samples
    CHK(set_table(s, 20));
    fail_malloc = nullptr;
    REQUIRE(!ranged(s));
    CHK(set_table(s, 20));
    REQUIRE(ranged(s));
    CHK(bcsim_destroy(s));
}

// Without room for the constant-length transforms' twiddles, the patches, or a range order
// the frames run the kernels that do without them.
static void optional_buffers() {
    for (size_t bytes : {conv_roots_size(12, false, 0) * sizeof(float2), 2 * sizeof(RangePatch)}) {
        bcsim_sim* s = simulator(128, 20000);
        int failed = 0;
        fail_malloc = [&](size_t n) { return n == bytes && ++failed; };
        const bool in_order = ranged(s);
        fail_malloc = nullptr;
        REQUIRE(failed > 0 && in_order == (bytes != 2 * sizeof(RangePatch)));
        REQUIRE(ranged(s));  // there is room again
        CHK(bcsim_destroy(s));
    }
    bcsim_sim* s = simulator(128, 20000);
    fail_malloc = [&](size_t n) { return n > 20000 * sizeof(RangeRec) && n < 21000 * sizeof(RangeRec) + 200000; };
    REQUIRE(!ranged(s));
    fail_malloc = nullptr;
    REQUIRE(ranged(s));
    CHK(bcsim_destroy(s));
}

// Points that crowd: few lines and points are projected in parts, many by the tile kernel;
// uniform points, and points beyond the lines, in range order as they are.
static std::vector<float> shell_points(size_t n, float radius, float share) {
    std::vector<float> p = box_points(n);
    std::mt19937 rng(4);
    std::uniform_real_distribution<float> u(-0.6f, 0.6f);
    for (size_t i = 0; i < (size_t)(share * n); i++) {
        const float a = u(rng);
        p[4 * i] = radius * sinf(a), p[4 * i + 1] = 0, p[4 * i + 2] = radius * cosf(a);
    }
    return p;
}
static void crowds() {
    struct Case {
        int lines;
        size_t n;
        float radius, share;
        bool table, in_order, parts;
    };
    for (const Case& q : {Case{128, 100000, 0.03f, 0.0f, false, true, false}, Case{128, 100000, 0.03f, 0.0f, true, true, false},
                          Case{40, 8000, 0.03f, 1.0f, false, true, true}, Case{40, 8000, 0.03f, 1.0f, true, true, true},
                          Case{128, 400000, 0.03f, 1.0f, false, false, false}, Case{64, 100000, 0.03f, 0.3f, true, true, true},
                          Case{128, 100000, 0.2f, 0.5f, false, true, false}}) {
        bcsim_sim* s = simulator(q.lines, 0);
        const std::vector<float> p = shell_points(q.n, q.radius, q.share);
        CHK(bcsim_add_fixed_scatterers(s, p.data(), q.n));
        if (q.table) CHK(set_table(s, 16));
        const bool in_order = ranged(s);
        const bool parts = plan(s).find("in parts") != std::string::npos;
        if (in_order != q.in_order || parts != q.parts) fprintf(stderr, "%d lines %zu points: %s", q.lines, q.n, plan(s).c_str());
        REQUIRE(in_order == q.in_order && parts == q.parts);
        // the same points as splines at one time: sorted every frame, which crowds slow down too
        if (q.lines == 128 && !q.table) {
            std::vector<float> cp, amp;
            for (size_t i = 0; i < q.n; i++) {
                for (int k = 0; k < 4; k++) cp.insert(cp.end(), {p[4 * i], p[4 * i + 1], p[4 * i + 2]});
                amp.push_back(p[4 * i + 3]);
            }
            const float knots[] = {0, 0, 0, 0, 1, 1, 1, 1};
            CHK(bcsim_clear_fixed_scatterers(s));
            CHK(bcsim_add_spline_scatterers(s, 3, knots, 8, cp.data(), amp.data(), q.n, 4));
            Scan wide = sector(256);
            for (auto& t : wide.t) t = 0.4f;
            set_scan(s, wide, true);
            REQUIRE(ranged(s) == (q.share == 0.0f || q.radius > 0.05f));
        }
        CHK(bcsim_destroy(s));
    }
    // few points on many long lines, whose bins are the frame
    for (size_t n : {size_t(200), size_t(60000)}) {
        bcsim_sim* s = simulator(2500, n);
        Scan deep = sector(2500);
        deep.len = 0.15f;
        set_scan(s, deep);
        REQUIRE(ranged(s) == (n > 200));
        CHK(bcsim_destroy(s));
    }
    // many points on short lines, evenly over the sector's area: nothing crowds
    for (int lines : {40, 400}) {
        std::mt19937 rng(5);
        std::uniform_real_distribution<float> u(0, 1);
        std::vector<float> p;
        for (int i = 0; i < 400000; i++) {
            const float r = 0.025f * sqrtf(u(rng)), a = 1.2f * u(rng) - 0.6f;
            p.insert(p.end(), {r * sinf(a), 0.01f * (u(rng) - 0.5f) * r, r * cosf(a), 1.0f});
        }
        bcsim_sim* s = simulator(lines, 0);
        CHK(bcsim_add_fixed_scatterers(s, p.data(), p.size() / 4));
        CHK(set_table(s, 24));
        Scan shallow = sector(lines);
        shallow.len = 0.025f;
        set_scan(s, shallow);
        REQUIRE(ranged(s) && plan(s).find("in parts") == std::string::npos);
        CHK(bcsim_destroy(s));
    }
}

// Orders of a dataset: four, the one longest unused giving way to an origin that stays.
static void origins() {
    const size_t n = 20000;
    bcsim_sim* s = simulator(64, n);
    count_bytes = n * sizeof(RangeRec) + (2 * kRangeBins + 4 + n) * sizeof(int);
    const auto at = [&](float x) {
        set_scan(s, sector(64, x));
        return ranged(s);
    };
    const auto allocated = [&] {
        const int k = mallocs;
        mallocs = 0;
        return k;
    };
    (void)allocated();
    // demodulation frequencies without phase delay: one order, which serves phase delay too
    std::vector<float> pulse(55, 0.5f);
    for (int k = 1; k <= 6; k++) {
        CHK(bcsim_set_excitation(s, pulse.data(), 55, 27, 50e6f, k * 1e6f));
        REQUIRE(ranged(s));
    }
    REQUIRE(allocated() == 1);
    CHK(bcsim_set_parameter(s, "phase_delay", "on"));
    CHK(bcsim_set_excitation(s, pulse.data(), 55, 27, 50e6f, 1e6f));
    REQUIRE(ranged(s) && allocated() == 0);
    CHK(bcsim_set_parameter(s, "phase_delay", "off"));
    for (float x : {0.001f, 0.002f, 0.003f}) REQUIRE(at(x));
    REQUIRE(allocated() == 3);
    // a fifth origin: from its second frame on, in the place of the first one
    REQUIRE(!at(0.004f) && at(0.004f) && at(0.004f) && allocated() == 1);
    REQUIRE(at(0.001f) && at(0.002f) && at(0.003f) && allocated() == 0);
    // more origins by turns than orders: those that have one keep it, nothing is sorted again
    for (int turn = 0; turn < 4; turn++) {
        for (float x : {0.001f, 0.002f, 0.003f, 0.004f}) REQUIRE(at(x));
        REQUIRE(!at(0.0f));
    }
    REQUIRE(allocated() == 0);
    // an origin that wanders: nothing is sorted, the others keep their orders
    for (int k = 0; k < 20; k++) REQUIRE(!at(0.01f + 0.0001f * k));
    REQUIRE(at(0.001f) && at(0.002f) && at(0.003f) && at(0.004f) && allocated() == 0);
    // a batch's tables name orders: they stay while it lives
    bcsim_batch* b;
    CHK(bcsim_batch_create(&b));
    CHK(bcsim_batch_add(b, s, nullptr));  // at 0.004
    size_t total = 0;
    int jobs = 0;
    CHK(bcsim_batch_get_layout(b, &total, &jobs, nullptr, nullptr, nullptr, 0));
    void* out = nullptr;
    REQUIRE(hipMalloc(&out, total * 8) == hipSuccess);
    CHK(bcsim_batch_simulate_device(b, out, total));
    (void)allocated();
    REQUIRE(!at(0.02f) && at(0.02f) && !at(0.021f) && at(0.021f) && !at(0.022f) && at(0.022f) && allocated() == 3);
    REQUIRE(!at(0.023f) && at(0.023f) && allocated() == 1);  // for 0.02's: 0.004's is the batch's
    REQUIRE(at(0.004f) && allocated() == 0);
    CHK(bcsim_batch_synchronize(b));
    CHK(bcsim_batch_destroy(b));
    CHK(bcsim_destroy(s));
    hipFree(out);
}

// Orders that captured frames name: a graph of them can be replayed whatever scans came since.
static void captured_frames() {
    const size_t n = 20000;
    for (bool noalloc : {true, false}) {
        bcsim_sim* s = simulator(64, n);
        count_bytes = n * sizeof(RangeRec) + (2 * kRangeBins + 4 + n) * sizeof(int);
        const auto at = [&](float x) {
            set_scan(s, sector(64, x));
            return ranged(s);
        };
        int nl = 0, ns = 0;
        CHK(bcsim_get_output_shape(s, &nl, &ns));
        void *out = nullptr, *stream = nullptr;
        REQUIRE(hipMalloc(&out, (size_t)nl * ns * 8) == hipSuccess);
        CHK(bcsim_get_stream(s, &stream));
        const hipStream_t st = static_cast<hipStream_t>(stream);
        const auto capture = [&] {
            hipGraph_t g = nullptr;
            hipGraphExec_t e = nullptr;
            under_capture = true;
            REQUIRE(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) == hipSuccess);
            CHK((noalloc ? bcsim_simulate_lines_device_noalloc : bcsim_simulate_lines_device)(s, out, (size_t)nl * ns, &nl, &ns));
            REQUIRE(hipStreamEndCapture(st, &g) == hipSuccess);
            under_capture = false;
            REQUIRE(hipGraphInstantiate(&e, g, nullptr, nullptr, 0) == hipSuccess);
            REQUIRE(hipGraphDestroy(g) == hipSuccess);
            return e;
        };
        REQUIRE(at(0.0f));
        const hipGraphExec_t first = capture();
        const void* records = last_records;
        // four more origins that stay: three orders, then the one longest unused of those three
        for (float x : {0.001f, 0.002f, 0.003f}) REQUIRE(at(x));
        REQUIRE(!at(0.004f) && at(0.004f) && !at(0.005f) && at(0.005f) && !at(0.006f) && at(0.006f));
        // one that is seen again under capture waits for nothing and allocates nothing
        REQUIRE(!at(0.007f));
        mallocs = range_launches = 0;
        const hipGraphExec_t fifth = capture();
        REQUIRE(mallocs == 0 && range_launches == 0);
        // the captured one is there still, and the same
        REQUIRE(live(records) && at(0.0f) && mallocs == 0 && last_records == records);
        REQUIRE(hipGraphLaunch(first, st) == hipSuccess && hipGraphLaunch(fifth, st) == hipSuccess);
        CHK(bcsim_synchronize(s));
        REQUIRE(hipGraphExecDestroy(first) == hipSuccess && hipGraphExecDestroy(fifth) == hipSuccess);
        CHK(bcsim_destroy(s));
        hipFree(out);
    }
}

// A server counts the orders and the samples of its tables, sorts none that its budget has no
// room for, and gives one back for a request that needs the room.
static void server_budget() {
    const size_t n = 40000, order = n * sizeof(RangeRec) + (2 * kRangeBins + 4 + n) * sizeof(int);
    count_bytes = order;
    const Scan small = sector(24), large = sector(320);
    const auto stat = [](bcsim_server* v, const char* key) {
        double x = 0;
        size_t k = 0;
        CHK(bcsim_server_get_stats(v, key, &x, 1, &k));
        return x;
    };
    for (bool room : {false, true}) {
        bcsim_sim* s = simulator(64, n);
        bcsim_server* v;
        CHK(bcsim_server_create(&v));
        CHK(bcsim_server_set_parameter(v, "memory_budget_bytes", "1000000000"));
        CHK(bcsim_server_add_phantom(v, s, nullptr));
        int gs, gl, L, S;
        CHK(bcsim_server_add_geometry(v, 24, small.o.data(), small.d.data(), small.l.data(), small.len, &gs));
        CHK(bcsim_server_add_geometry(v, 320, large.o.data(), large.d.data(), large.l.data(), large.len, &gl));
        CHK(bcsim_server_get_output_shape(v, 0, gl, &L, &S));
        const double resident = stat(v, "resident_bytes");
        const auto frame = [&](int lines) { return lines * (S * 4.0 + S * 8.0 + 64) + 4096 * 16.0 + S * 8.0; };
        const double budget = resident + (room ? frame(320) + 200000 : frame(24) + 0.5 * order);
        char text[32];
        snprintf(text, sizeof text, "%.0f", budget);
        CHK(bcsim_server_set_parameter(v, "memory_budget_bytes", text));
        std::vector<float> out((size_t)L * S * 2);
        const auto serve = [&](int g) {
            uint64_t id;
            CHK(bcsim_server_submit(v, 0, g, 0.0f, out.data(), out.size() / 2, &id));
            CHK(bcsim_server_wait(v, id, -1, nullptr, nullptr, nullptr));
        };
        mallocs = 0;
        serve(gs);
        serve(gs);
        REQUIRE(mallocs == (room ? 1 : 0));
        REQUIRE(stat(v, "used_bytes") >= resident + (room ? order : 0) && stat(v, "used_bytes") <= budget);
        if (room) {
            REQUIRE(budget - resident < frame(320) + order);
            serve(gl);  // the order gives way
            REQUIRE(stat(v, "used_bytes") <= budget && stat(v, "resident_bytes") == resident);
            serve(gs);
        }
        CHK(bcsim_server_destroy(v));
        CHK(bcsim_destroy(s));
    }
    bcsim_sim* s = simulator(64, n);
    bcsim_server* v;
    CHK(bcsim_server_create(&v));
    CHK(bcsim_server_add_phantom(v, s, nullptr));
    const double plain = stat(v, "resident_bytes");
    CHK(set_table(s, 16));
    CHK(bcsim_server_add_phantom(v, s, nullptr));
    REQUIRE(stat(v, "resident_bytes") - plain == 16 * 24 * 24 * (8 * 4 + 4));
    CHK(bcsim_server_destroy(v));
    CHK(bcsim_destroy(s));
}

// Tuned choices are kept for the kernels that they were tried with.
static void tuned_radix() {
    int fours = 0;
    for (int lines : {9, 17, 33, 65, 129, 257, 513}) {
        bcsim_sim *noisy = simulator(lines, 500), *plain = simulator(lines, 500);
        CHK(bcsim_set_parameter(noisy, "noise_amplitude", "0.5"));
        for (bcsim_sim* s : {noisy, plain}) {
            CHK(bcsim_set_parameter(s, "autotune", "on"));
            (void)ranged(s);
        }
        fours += plan(noisy).find("radix=4") != std::string::npos;  // (by random times)
        REQUIRE(plan(plain).find("radix=8") != std::string::npos);
        CHK(bcsim_destroy(noisy));
        CHK(bcsim_destroy(plain));
    }
    REQUIRE(fours > 0);
}

static std::string tuned(bcsim_sim* s) {
    static char b[1 << 20];
    CHK(bcsim_get_parameter(s, "autotune_report", b, sizeof b));
    return b;
}
static int count(const std::string& text, const char* word) {
    int n = 0;
    for (size_t at = text.find(word); at != std::string::npos; at = text.find(word, at + 1)) n++;
    return n;
}
static Scan parallel(int n) {
    Scan s = sector(n);
    for (int k = 0; k < n; k++) {
        s.o[3 * k] = -0.01f + 0.02f * k / (n - 1);
        for (int a = 0; a < 3; a++) s.d[3 * k + a] = a == 2, s.l[3 * k + a] = a == 0;
    }
    return s;
}
// Lines of one origin and others run different kernels: each class is tried.
static void tuned_shapes_by_origin() {
    bcsim_sim* s = simulator(12, 5000);
    CHK(bcsim_set_parameter(s, "autotune", "on"));
    (void)ranged(s);
    REQUIRE(count(tuned(s), "tile/fixed/") == 1);
    set_scan(s, parallel(12));
    (void)ranged(s);
    REQUIRE(count(tuned(s), "tile/fixed/") == 2);
    set_scan(s, sector(12, 0.01f));
    (void)ranged(s);
    REQUIRE(count(tuned(s), "tile/fixed/") == 2);
    CHK(bcsim_destroy(s));
}

// With tuning on, range order is tried beside the shapes, and what was faster runs.
static void tuned_order() {
    int in_order = 0, shapes = 0;
    for (int lines : {17, 33, 65, 129, 257}) {
        bcsim_sim* s = simulator(lines, 8000);
        CHK(bcsim_set_parameter(s, "autotune", "on"));
        const bool r = ranged(s);  // by random times
        REQUIRE(count(tuned(s), "[order]=") == in_order + shapes + 1);
        REQUIRE(count(tuned(s), "ms with range order") == in_order + (r ? 1 : 0));
        REQUIRE(ranged(s) == r && count(tuned(s), "[order]=") == in_order + shapes + 1);
        (r ? in_order : shapes)++;
        CHK(bcsim_destroy(s));
    }
    REQUIRE(shapes > 0);
}

// A batch tries shapes only for jobs that run them, with the bins that they will have.
static void batch_shapes() {
    std::vector<bcsim_sim*> sims;
    bcsim_batch* b;
    CHK(bcsim_batch_create(&b));
    for (int lines : {20, 40, 80}) {
        sims.push_back(simulator(lines, 8000));  // range order
        sims.push_back(simulator(lines, 8000));
        set_scan(sims.back(), parallel(lines));
        sims.push_back(simulator(lines, 8000));
        set_scan(sims.back(), parallel(lines));
        CHK(set_table(sims.back(), 16));
    }
    for (bcsim_sim* s : sims) CHK(bcsim_batch_add(b, s, nullptr));
    size_t total = 0;
    int jobs = 0;
    CHK(bcsim_batch_get_layout(b, &total, &jobs, nullptr, nullptr, nullptr, 0));
    void* out = nullptr;
    REQUIRE(hipMalloc(&out, total * 8) == hipSuccess);
    CHK(bcsim_batch_simulate_device(b, out, total));
    CHK(bcsim_batch_synchronize(b));
    const std::string report = tuned(sims[0]);
    REQUIRE(count(report, "tile=fixed/") == 6 && count(report, "tile/") == 0 && count(report, "arc-shared") == 0);
    for (size_t at = 0; at < report.size(); at = report.find('\n', at) + 1) {
        const std::string line = report.substr(at, report.find('\n', at) - at);
        if (line.find("tile=") != 0) continue;
        REQUIRE(count(line, line.find("/gauss/") != std::string::npos ? ",float]=" : ",fixed]=") == 0);
    }
    CHK(bcsim_batch_destroy(b));
    for (bcsim_sim* s : sims) CHK(bcsim_destroy(s));
    hipFree(out);
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    const std::vector<std::pair<std::string, void (*)()>> all = {
        {"table_failures", table_failures}, {"optional_buffers", optional_buffers}, {"crowds", crowds}, {"origins", origins},
        {"captured_frames", captured_frames},
        {"server_budget", server_budget}, {"tuned_radix", tuned_radix},
        {"tuned_shapes_by_origin", tuned_shapes_by_origin}, {"tuned_order", tuned_order},
        {"batch_shapes", batch_shapes}};
    for (auto& e : all)
        if (e.first == what) {
            e.second();
            fprintf(stderr, "DONE %s\n", what.c_str());
            fflush(stderr);
            _exit(0);
        }
    fprintf(stderr, "unknown scenario\n");
    return 2;
}
