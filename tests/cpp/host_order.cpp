// The host side of the library (pl_api.cpp) without a GPU: in the place of the HIP runtime and of the kernel
// launches there is a record of what was enqueued where, with a clock per stream that follows events and
// waits (F. Mattern, Virtual Time and Global States of Distributed Systems, 1989).  Two launches that
// touch the same array, one of them writing, must be ordered by it whatever the streams do.
//
// Usage: host_order.bin SCENARIO; 0 when it holds, 1 and what does not otherwise.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "permutohedral_lattice.h"
#include "pl_kernels.h"

namespace {

int g_failures = 0;
void expect(bool ok, const std::string &what) {
    if (ok) return;
    std::printf("%s\n", what.c_str());
    g_failures += 1;
}

// ------------------------------------------------------------------------------------------------
// Streams, events, and who touched an array last
// ------------------------------------------------------------------------------------------------
using Clock = std::map<int, long>;   // how far along each stream
void join(Clock &a, const Clock &b) {
    for (const auto &[stream, time] : b)
        if (a[stream] < time) a[stream] = time;
}

struct Stream {
    int id;
    Clock clock;
    bool capturing = false;
};
std::map<void *, Stream> g_streams;   // by handle
int g_stream_ids = 0;
std::map<void *, Clock> g_events;
Clock g_host;                         // what the host has waited for

Stream &stream_of(hipStream_t s) {
    auto found = g_streams.find((void *)s);
    if (found == g_streams.end()) found = g_streams.emplace((void *)s, Stream{++g_stream_ids, {}}).first;
    return found->second;
}
hipStream_t named_stream(long name) {
    hipStream_t s = (hipStream_t)(name * 64);
    stream_of(s);
    return s;
}

struct Access {
    int stream;
    long time;
    std::string by;
};
struct Array {
    std::vector<Access> reads, writes;
};
std::map<const void *, Array> g_arrays;
std::vector<std::string> g_launches;
std::string g_fail_next;   // the launch of this name fails, once
long g_allocated = 0;      // device arrays in existence
unsigned g_rows_of_sums = 0;                // what the lists of a merging build report
std::map<const void *, size_t> g_sizes;     // of arrays from alloc_if_allowed

hipError_t launch(const char *name, hipStream_t s, const std::vector<const void *> &reads,
                  const std::vector<const void *> &writes) {
    if (g_fail_next == name) {
        g_fail_next.clear();
        return hipErrorInvalidValue;
    }
    g_launches.push_back(name);
    Stream &stream = stream_of(s);
    if (stream.capturing) return hipSuccess;
    join(stream.clock, g_host);
    const Access now{stream.id, ++stream.clock[stream.id], name};
    auto behind = [&](const std::vector<Access> &before) {
        for (const Access &a : before)
            expect(stream.clock[a.stream] >= a.time, std::string(name) + " does not wait for " + a.by);
    };
    for (const void *p : reads)
        if (p) behind(g_arrays[p].writes), g_arrays[p].reads.push_back(now);
    for (const void *p : writes)
        if (p) behind(g_arrays[p].writes), behind(g_arrays[p].reads), g_arrays[p].writes.push_back(now);
    return hipSuccess;
}
bool launched(const char *name) {
    for (const auto &l : g_launches)
        if (l == name) return true;
    return false;
}

plk::Points64 g_points64;             // of the last build of doubles
const float *g_values[2];             // value tables of the lattice blurred last in a joint pass

// What a build counts in must be zero when it starts (it and the passes behind it then zero the other set)
void count_in(plk::Counters *counters, const plk::CreatedLists &lists) {
    static const plk::Counters zero{};
    expect(std::memcmp(counters, &zero, sizeof(zero)) == 0, "a build counts in counters that are not zero");
    counters->vertices = counters->segment_count[0].n = 100;
    if (lists.foreign_rows) return;
    expect(lists.chunk_count[0] == 0, "a build counts in chunk sums that are not zero");
    lists.chunk_count[0] = 100;
}

void report(plk::HostReport to) {
    to.status->num_vertices = 100;
    to.status->flags = 0;
    to.status->max_segment = 100;
    to.status->n_segments = 0;
    to.status->foreign_rows = 0;
    to.status->sequence = to.sequence;
}

}  // namespace

// ------------------------------------------------------------------------------------------------
// The HIP runtime
// ------------------------------------------------------------------------------------------------
extern "C" {
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return g_allocated += 1, hipHostMalloc(p, n, 0); }
hipError_t hipFree(void *p) { return g_allocated -= p != nullptr, hipHostFree(p); }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
    return std::memcpy(to, from, n), hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    static long made = 1000;
    return *s = named_stream(++made), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return g_streams.erase((void *)s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return join(g_host, stream_of(s).clock), hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *status) {
    *status = stream_of(s).capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { return *d = 0, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    if (!g_events.count((void *)e)) return hipErrorInvalidHandle;
    return join(stream_of(s).clock, g_events[(void *)e]), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
    static long made = 0;
    *e = (hipEvent_t)(++made * 64);
    return g_events[(void *)*e] = {}, hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    return g_events.erase((void *)e) ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (!g_events.count((void *)e)) return hipErrorInvalidHandle;
    expect(!stream_of(s).capturing, "an event is recorded on a stream that is being captured");
    join(stream_of(s).clock, g_host);
    return g_events[(void *)e] = stream_of(s).clock, hipSuccess;
}
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipErrorInvalidValue; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidValue; }
}

// ------------------------------------------------------------------------------------------------
// The launches
// ------------------------------------------------------------------------------------------------
namespace plk {

int key_field_bits(int pd) { return 60 / pd > 16 ? 16 : 60 / pd; }
PointMap make_point_map(int N, int n_dims, const int *dims) {
    PointMap m{};
    m.N = N;
    m.mode = n_dims == 2 ? 2 : 0;
    m.dims[0] = 1;
    m.dims[1] = n_dims == 2 ? dims[0] : 1;
    m.dims[2] = n_dims == 2 ? dims[1] : N;
    m.n_blocks = (unsigned)(N + 255) / 256u;
    return m;
}
bool build_can_splat(int vd) { return vd <= 4; }
bool blur_can_take_three_axes(int vd) { return vd <= 4; }
size_t vertex_list_scan_blocks(int) { return 1; }
size_t vertex_list_max_chunks(int, size_t rows) { return rows; }
size_t vertex_list_max_long(size_t rows) { return rows; }
bool slice_pairs_take(int, int, int) { return true; }

hipError_t clear_table(uint64_t *keys, uint32_t, hipStream_t s) { return launch("clear_table", s, {}, {keys}); }
hipError_t fill_zero(float *p, size_t n, hipStream_t s) {
    const hipError_t e = launch("fill_zero", s, {}, {p});
    if (e == hipSuccess) std::memset(p, 0, n * sizeof(float));
    return e;
}
hipError_t fill_ranges(FillRanges ranges, hipStream_t s) {
    std::vector<const void *> written;
    for (const auto &r : ranges.range) written.push_back(r.words_at);
    return launch("fill_ranges", s, {}, written);
}
hipError_t build(int, const PointFeatures &, const PointMap &, const ScaleFactor &, uint64_t *keys, uint32_t,
                 Counters *counters, ReplayEntry *replay, int, int, const float *, int, float *, const CreatedLists &lists,
                 const RegionSource &, const InBuildNumbering *, bool, hipStream_t s) {
    const hipError_t e = launch("build", s, {}, {keys, replay});
    if (e == hipSuccess) count_in(counters, lists);
    return e;
}
hipError_t build_joint(int, int n, const BuildWork *work, const ScaleFactor &, int, int, int, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i) {
        e = launch("build_joint", s, {}, {work[i].cell_keys, work[i].replay});
        if (e == hipSuccess) count_in(work[i].counters, work[i].lists);
    }
    return e;
}
hipError_t build_f64(int, const Points64 &points, const PointMap &, uint64_t *keys, uint32_t, Counters *,
                     ReplayEntry *replay, int, const CreatedLists &, const RegionSource &, const InBuildNumbering *,
                     int, const double *, int, double *, bool, hipStream_t s) {
    g_points64 = points;
    return launch("build_f64", s, {}, {keys, replay});
}
hipError_t number_vertices(int, const PointMap &, const CreatedLists &, int *next_chunk_count, unsigned n_chunks,
                           const VertexTables &, float *values, int, float *, Counters *, Counters *next_counters,
                           HostReport to, bool, hipStream_t s) {
    report(to);
    *next_counters = Counters{};
    std::memset(next_chunk_count, 0, n_chunks * sizeof(int));
    return launch("number_vertices", s, {}, {values});
}
hipError_t number_vertices_joint(int pd, int n, const BuildWork *work, int vd, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i)
        e = number_vertices(pd, work[i].map, work[i].lists, work[i].next_chunk_count, work[i].n_chunks, work[i].vertices,
                            work[i].values, vd, nullptr, work[i].counters, work[i].next_counters, work[i].report_to, false, s);
    return e;
}
hipError_t neighbours(int, const VertexTables &vertices, const Counters *, const uint64_t *keys, uint32_t, int,
                      const CreatedLists *, unsigned, void *values, int, bool, Counters *to_report,
                      Counters *next_counters, HostReport to, bool, hipStream_t s) {
    if (to_report) {
        report(to);
        *next_counters = Counters{};
    }
    return launch("neighbours", s, {keys}, {vertices.neighbours, values});
}
hipError_t neighbours_joint(int pd, int n, const BuildWork *work, int vd, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i)
        e = neighbours(pd, work[i].vertices, work[i].counters, work[i].cell_keys, 0, 0, nullptr, 0, work[i].values, vd, false,
                       work[i].numbering.n_segments ? work[i].counters : nullptr, work[i].next_counters, work[i].report_to,
                       false, s);
    return e;
}
hipError_t build_vertex_lists(int, const PointMap &, ReplayEntry *replay, const int *, int, const VertexLists &lists,
                              unsigned *info, unsigned sequence, hipStream_t s) {
    info[0] = lists.map.tile_vertices.table ? g_rows_of_sums : 0u;
    info[1] = 1;
    info[2] = sequence;
    return launch("build_vertex_lists", s, {replay}, {lists.entries});
}
hipError_t splat_gather(int vd, const VertexLists &lists, unsigned, unsigned, const float *input, int, float *values,
                        hipStream_t s) {
    if (g_rows_of_sums && lists.map.tile_vertices.table)
        expect(g_sizes[lists.chunks.partial_rows] >= sizeof(float) * g_rows_of_sums * tile_row_floats(vd),
               "the rows of sums have no room");
    return launch("splat_gather", s, {lists.entries, input}, {values});
}
hipError_t splat_gather_many(int, int, int n, const GatherWork *work, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i)
        e = launch("splat_gather_many", s, {work[i].entries, work[i].input}, {work[i].values});
    return e;
}
hipError_t splat_tile(int, int, const PointMap &, const float *input, int, const ReplayEntry *replay, float *values, int,
                      hipStream_t s) {
    return launch("splat_tile", s, {input, replay}, {values});
}
hipError_t splat_joint(int, int, int n, const PointsWork *work, int, int, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i)
        e = launch("splat_joint", s, {work[i].input, work[i].replay}, {work[i].values});
    return e;
}
hipError_t blur_joint(int vd, int n, const BlurWork *work, hipStream_t s) { return blur_many(vd, n, work, s); }
hipError_t slice_joint(int, int, int n, const PointsWork *work, int, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i)
        e = launch("slice_joint", s, {work[i].replay, work[i].values}, {work[i].output});
    return e;
}
hipError_t splat_f64(int, int, const PointMap &, const double *input, int, ReplayEntry *replay, const double *,
                     const int *, double *values, int, hipStream_t s) {
    return launch("splat_f64", s, {input, replay}, {values});
}
hipError_t blur_many(int, int n, const BlurWork *work, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i) {
        g_values[0] = work[i].src;
        g_values[1] = work[i].dst;
        e = launch("blur_many", s, {work[i].src, work[i].nbr_first}, {work[i].dst, work[i].reset_cell_keys});
    }
    return e;
}
hipError_t blur_two_axes(int, const Counters *, int, const float *src, float *dst, const int2 *, const int2 *,
                         uint64_t *reset, const int *, int, hipStream_t s) {
    return launch("blur_two_axes", s, {src}, {dst, reset});
}
hipError_t blur_axis(int, const Counters *, int, const float *src, float *dst, const int2 *, uint64_t *reset,
                     const int *, int, hipStream_t s) {
    return launch("blur_axis", s, {src}, {dst, reset});
}
hipError_t blur_two_axes_f64(int, const Counters *, int, const double *src, double *dst, const int2 *, const int2 *,
                             uint64_t *reset, const int *, int, hipStream_t s) {
    return launch("blur_two_axes_f64", s, {src}, {dst, reset});
}
hipError_t blur_axis_f64(int, const Counters *, int, const double *src, double *dst, const int2 *, uint64_t *reset,
                         const int *, int, hipStream_t s) {
    return launch("blur_axis_f64", s, {src}, {dst, reset});
}
hipError_t slice(int, int, const PointMap &, const ReplayEntry *replay, const int *, const float *values,
                 float *output, int, hipStream_t s) {
    return launch("slice", s, {replay, values}, {output});
}
hipError_t slice_f64(int, int, const PointMap &, const ReplayEntry *replay, const double *, const int *,
                     const double *values, double *output, int, hipStream_t s) {
    return launch("slice_f64", s, {replay, values}, {output});
}
hipError_t slice_pairs(int, int, int, int n, const SlicePair *work, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess; ++i)
        e = launch("slice_pairs", s, {work[i].replay_a, work[i].replay_b, work[i].values_a, work[i].values_b,
                                      work[i].logits}, {work[i].output});
    return e;
}
hipError_t mean_field_update(float *q, const float *logits, const float *, const float *, size_t, int, hipStream_t s) {
    return launch("mean_field_update", s, {logits}, {q});
}
hipError_t compute_positions_f64(const double *reference, double *positions, int, int, int, const SpatialDims &, double,
                                 double, hipStream_t s) {
    return launch("compute_positions_f64", s, {reference}, {positions});
}
hipError_t export_values(const float *values, int, const VertexNumbers &, float *out, hipStream_t s) {
    return launch("export_values", s, {values}, {out});
}

}  // namespace plk

// ------------------------------------------------------------------------------------------------
// Scenarios
// ------------------------------------------------------------------------------------------------
namespace {

constexpr int kH = 16, kW = 32, kClasses = 6, kItems = 2;

// two images' lattices: image i on the streams own[2 i], own[2 i + 1]
struct Pairs {
    pl_handle bilateral[kItems], spatial[kItems];
    float *q, *logits, *messages;
    float guide[kH * kW * 3];
    const int dims[2] = {kH, kW};
    explicit Pairs(const std::vector<hipStream_t> &own) {
        for (int i = 0; i < kItems; ++i) {
            expect(pl_create(5, kClasses + 1, kH * kW, own[2 * i], nullptr, &bilateral[i]) == PL_OK, "pl_create");
            expect(pl_create(2, kClasses + 1, kH * kW, own[2 * i + 1], nullptr, &spatial[i]) == PL_OK, "pl_create");
        }
        build();
        const size_t bytes = sizeof(float) * kItems * kH * kW * kClasses;
        for (float **p : {&q, &logits, &messages}) (void)hipMalloc((void **)p, bytes);
    }
    void build() {
        for (int i = 0; i < kItems; ++i) {
            expect(pl_build_image(bilateral[i], guide, 3, 2, dims, 8.0f, 0.1f) == PL_OK, "pl_build_image");
            expect(pl_build_image(spatial[i], nullptr, 0, 2, dims, 3.0f, 1.0f) == PL_OK, "pl_build_image");
        }
    }
    // (arrays of their own for every call: only the lattices tie the calls together)
    int infer(hipStream_t s) {
        (void)hipMalloc((void **)&q, 4);
        return pl_mean_field_infer(kItems, bilateral, spatial, q, logits, 2, s);
    }
    int send(hipStream_t s) {
        (void)hipMalloc((void **)&messages, 4);
        return pl_mean_field_messages(kItems, bilateral, spatial, messages, logits, 0, s);
    }
};

std::vector<hipStream_t> four_streams() {
    return {named_stream(1), named_stream(2), named_stream(3), named_stream(4)};
}

// the value tables are read on a lattice's own stream, then the stream used last goes on
void read_on_the_own_stream() {
    Pairs p(four_streams());
    const hipStream_t t = named_stream(9);
    expect(p.infer(t) == PL_OK, "infer");
    for (int i = 0; i < kItems; ++i) {
        for (const pl_handle h : {p.bilateral[i], p.spatial[i]}) {
            float *out = nullptr;
            (void)hipMalloc((void **)&out, 4);
            expect(pl_debug_values(h, out) == PL_OK, "pl_debug_values");
        }
    }
    expect(p.infer(t) == PL_OK, "infer");
}

// the replay of a captured apply, which the library does not see, on a lattice's own stream
void replay_on_the_own_stream() {
    Pairs p(four_streams());
    const hipStream_t t = named_stream(9), own = named_stream(4);
    stream_of(own).capturing = true;
    expect(pl_apply(p.spatial[1], p.messages, p.logits, 0) == PL_OK, "pl_apply");
    stream_of(own).capturing = false;
    for (int turn = 0; turn < 3; ++turn) {
        // (the lattice blurred last is the last spatial one)
        expect(p.send(t) == PL_OK, "messages");
        (void)launch("a replayed graph", own, {}, {g_values[0], g_values[1]});
    }
}

// lattices that share a stream, called on another, on their own, and on the other again
void one_stream_for_all() {
    const hipStream_t own = named_stream(1), t = named_stream(9);
    Pairs p({own, own, own, own});
    for (const hipStream_t s : {t, own, t, own, own, t}) expect(p.send(s) == PL_OK, "messages");
}

// a stream ends, and another is given its handle
void handle_given_out_again() {
    Pairs p(four_streams());
    expect(p.send(named_stream(9)) == PL_OK, "messages");
    (void)hipStreamDestroy((hipStream_t)(9l * 64));
    expect(p.send(named_stream(9)) == PL_OK, "messages");
}

void two_callers_and_builds() {
    Pairs p(four_streams());
    for (int turn = 0; turn < 4; ++turn) {
        const hipStream_t s = named_stream(8 + turn % 2);
        expect(p.infer(s) == PL_OK && p.send(s) == PL_OK, "infer and messages");
        if (turn == 1) p.build();
        if (turn == 2) {
            float *out = nullptr;
            (void)hipMalloc((void **)&out, 4);
            expect(pl_apply(p.spatial[1], out, p.logits, 0) == PL_OK, "pl_apply");
        }
    }
}

// calls with some of the lattices, in changing order and company, some destroyed in between: the events that
// they refer to are one another's
void changing_company() {
    for (int destroyed = 0; destroyed <= 4; ++destroyed) {
        Pairs p(four_streams()), other({named_stream(5), named_stream(5), named_stream(1), named_stream(6)});
        auto call = [&](const std::vector<pl_handle> &bilateral, const std::vector<pl_handle> &spatial, long stream) {
            float *out = nullptr;
            (void)hipMalloc((void **)&out, 4);
            expect(pl_mean_field_messages((int)bilateral.size(), bilateral.data(), spatial.data(), out, p.logits, 0,
                                          named_stream(stream)) == PL_OK, "messages");
        };
        const pl_handle *a = p.bilateral, *b = p.spatial, *c = other.bilateral, *d = other.spatial;
        call({a[0], a[1]}, {b[0], b[1]}, 9);
        call({c[0], a[1]}, {b[1], d[1]}, 8);
        call({a[0]}, {b[0]}, 2);
        call({a[1], a[0], c[1]}, {d[0], b[0], b[1]}, 9);
        call({c[0], c[1]}, {d[1], d[0]}, 7);
        float *out = nullptr;
        (void)hipMalloc((void **)&out, 4);
        expect(pl_apply(a[1], out, p.logits, 0) == PL_OK, "pl_apply");
        call({a[1]}, {d[1]}, 3);
        const pl_handle all[] = {a[0], a[1], b[0], c[0]};
        for (int i = 0; i < destroyed; ++i) expect(pl_destroy(all[i]) == PL_OK, "pl_destroy");
        if (destroyed < 1) call({a[0], c[0]}, {b[1], d[0]}, 8);
        if (destroyed < 2) call({a[1]}, {b[0]}, 9);
        if (destroyed < 4) call({c[0]}, {d[1]}, 8);
        call({c[1]}, {b[1]}, 7);
        call({c[1]}, {d[0]}, 9);
        for (int i = destroyed; i < 4; ++i) (void)pl_destroy(all[i]);
        for (const pl_handle h : {b[1], c[1], d[0], d[1]}) (void)pl_destroy(h);
        expect(g_events.empty(), "events are left");
        g_arrays.clear();   // (freed memory comes back as other arrays)
    }
}

// a lattice's own stream is being captured: nothing may be recorded there, nothing is enqueued
void own_stream_captured() {
    Pairs p(four_streams());
    expect(p.send(named_stream(9)) == PL_OK, "messages");
    stream_of(named_stream(3)).capturing = true;
    const size_t before = g_launches.size();
    expect(p.send(named_stream(9)) == PL_EUNSUPPORTED, "messages while a lattice's stream is captured");
    stream_of(named_stream(3)).capturing = false;
    stream_of(named_stream(9)).capturing = true;
    expect(p.infer(named_stream(9)) == PL_EUNSUPPORTED, "infer on a stream that is captured");
    expect(g_launches.size() == before, "something was enqueued");
}

// the launch that would have emptied the hash cells fails: the next build empties the table
void failed_blur() {
    Pairs p(four_streams());
    g_fail_next = "blur_many";
    expect(p.send(named_stream(9)) == PL_EHIP, "a launch failed");
    g_launches.clear();
    p.build();
    expect(launched("clear_table"), "the table is taken to be empty");
}

// the op of doubles leaves no pointer to its reference image in its lattice
void no_pointer_kept() {
    const int dims[2] = {kH, kW};
    double *in = nullptr, *out = nullptr, *reference = nullptr, *positions = nullptr;
    for (double **p : {&in, &out, &reference, &positions}) (void)hipMalloc((void **)p, sizeof(double) * kH * kW * 5);
    expect(pl_lattice_filter_op_f64(in, reference, out, 1, 2, dims, 2, 3, 1, 8.0f, 0.1f, 1.0f, 0, nullptr, nullptr) ==
               PL_OK, "the op");
    expect(g_points64.reference == reference, "the features come from the reference image");
    // (the pooled lattice is filtered from a positions array by an op whose points are no grid of tiles)
    const int flat[1] = {kH * kW};
    expect(pl_lattice_filter_op_f64(in, reference, out, 1, 1, flat, 2, 4, 1, 8.0f, 0.1f, 1.0f, 0, nullptr, nullptr) ==
               PL_OK, "the op on a list");
    expect(g_points64.positions && !g_points64.reference, "the reference image of a call that has returned");
}

// a batch that cannot be enqueued whole -- the memory of one of its lattices is refused, or a launch fails --
// leaves lattices whose next builds are like any other
bool g_refuse = false;
void *alloc_if_allowed(void *, size_t bytes) {
    if (g_refuse) return nullptr;
    void *p = std::calloc(1, bytes);
    g_sizes[p] = bytes;
    return p;
}
void free_any(void *, void *p) {
    g_sizes.erase(p);
    std::free(p);
}
void failed_batch() {
    const hipStream_t s = named_stream(1);
    const int dims[2] = {kH, kW};
    const pl_alloc alloc{alloc_if_allowed, free_any, nullptr};
    for (const int channels : {3, kClasses}) {
        const size_t bytes = sizeof(float) * 2 * kH * kW * kClasses;
        float *in = nullptr, *out = nullptr, *guide = nullptr;
        for (float **p : {&in, &out, &guide}) (void)hipMalloc((void **)p, bytes);
        pl_handle h[2];
        expect(pl_create(5, channels + 1, kH * kW, s, nullptr, &h[0]) == PL_OK, "pl_create");
        expect(pl_create(5, channels + 1, kH * kW, s, &alloc, &h[1]) == PL_OK, "pl_create");
        auto alone = [&](int i) { return pl_filter_image(h[i], out, in, guide, 3, 2, dims, 8.0f, 0.1f, 0); };
        auto together = [&]() { return pl_filter_images(2, h, out, in, guide, 3, 2, dims, 8.0f, 0.1f, 0); };
        expect(alone(0) == PL_OK && alone(0) == PL_OK, "the first");
        g_refuse = true;
        for (int turn = 0; turn < 3; ++turn) {
            expect(together() == PL_ENOMEM, "a batch without the memory for its second lattice");
            if (turn != 1) expect(alone(0) == PL_OK, "the first after it");
        }
        g_refuse = false;
        expect(together() == PL_OK && together() == PL_OK, "the batch with memory");
        for (const char *launch : {"build_joint", "neighbours", "blur_many", "slice_joint"}) {
            g_fail_next = launch;
            expect(together() == PL_EHIP, std::string(launch) + " failed");
            expect(alone(1) == PL_OK && together() == PL_OK && alone(0) == PL_OK, std::string("after ") + launch);
        }
        for (const char *launch : {"build", "neighbours", "blur_two_axes"}) {
            g_fail_next = launch;
            expect(alone(0) == PL_EHIP, std::string(launch) + " failed");
            expect(alone(0) == PL_OK && together() == PL_OK, std::string("after ") + launch);
        }
        for (const pl_handle l : h) (void)pl_destroy(l);
        g_arrays.clear();
    }
}

// batches of one shape whose passes can be enqueued together and whose cannot, in turn: the same lattices
void batches_either_way() {
    const int dims[2] = {kH, kW}, flat[1] = {kH * kW};
    const hipStream_t s = named_stream(1);
    float *in = nullptr, *out = nullptr, *reference = nullptr;
    for (float **p : {&in, &out, &reference}) (void)hipMalloc((void **)p, sizeof(float) * 4 * kH * kW * 4);
    long first = 0;
    for (const char *turn = "jjssjsjj"; *turn; ++turn) {
        g_launches.clear();
        const int rc = *turn == 'j' ? pl_lattice_filter_op(in, reference, out, 3, 2, dims, 3, 3, 1, 8.0f, 0.1f, 1.0f, 0, s, nullptr)
                                    : pl_lattice_filter_op(in, reference, out, 3, 1, flat, 3, 4, 1, 8.0f, 0.1f, 1.0f, 0, s, nullptr);
        expect(rc == PL_OK, "the op");
        expect(launched("build_joint") == (*turn == 'j') && launched("build") == (*turn == 's'), "how it was enqueued");
        (void)launch("the caller's", s, {out}, {in, reference});
        if (!first) first = g_allocated;
        expect(g_allocated == first, "more lattices than items in flight");
    }
}

// the rows of sums that a build's lists turn out to have are given room when the build ends; where there is
// none, the lattice has to be built again
void more_rows_of_sums() {
    const hipStream_t s = named_stream(1);
    const int dims[2] = {kH, kW};
    const pl_alloc alloc{alloc_if_allowed, free_any, nullptr};
    const size_t bytes = sizeof(float) * kH * kW * kClasses;
    float *in = nullptr, *out = nullptr, *guide = nullptr;
    for (float **p : {&in, &out, &guide}) (void)hipMalloc((void **)p, bytes);
    pl_handle h = nullptr;
    expect(pl_create(5, kClasses + 1, kH * kW, s, &alloc, &h) == PL_OK, "pl_create");
    auto build = [&]() { return pl_build_image(h, guide, 3, 2, dims, 8.0f, 0.1f); };
    for (unsigned rows : {1u, 5000u, 40000u, 70u, 50000u}) {
        g_rows_of_sums = rows;
        expect(build() == PL_OK && pl_apply(h, out, in, 0) == PL_OK, "a build and an apply");
    }
    g_rows_of_sums = 90000u;
    g_refuse = true;
    expect(build() == PL_ENOMEM && pl_apply(h, out, in, 0) == PL_ESTATE, "no memory for the rows");
    g_refuse = false;
    expect(build() == PL_OK && pl_apply(h, out, in, 0) == PL_OK, "with memory again");
    (void)pl_destroy(h);
    expect(g_sizes.empty(), "memory is left");
}

}  // namespace

int main(int argc, char **argv) {
    const std::map<std::string, std::function<void()>> scenarios{
        {"read_on_the_own_stream", read_on_the_own_stream},
        {"replay_on_the_own_stream", replay_on_the_own_stream},
        {"one_stream_for_all", one_stream_for_all},
        {"handle_given_out_again", handle_given_out_again},
        {"two_callers_and_builds", two_callers_and_builds},
        {"changing_company", changing_company},
        {"own_stream_captured", own_stream_captured},
        {"failed_blur", failed_blur},
        {"no_pointer_kept", no_pointer_kept},
        {"failed_batch", failed_batch},
        {"batches_either_way", batches_either_way},
        {"more_rows_of_sums", more_rows_of_sums},
    };
    const auto found = scenarios.find(argc > 1 ? argv[1] : "");
    if (found == scenarios.end()) {
        for (const auto &s : scenarios) std::printf("%s\n", s.first.c_str());
        return 2;
    }
    found->second();
    return g_failures ? 1 : 0;
}
