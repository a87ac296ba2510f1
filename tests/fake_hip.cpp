// fake_hip.cpp -- a HIP runtime and kernel launches for tests of the host code
// (nuosc_capi.cpp, nuosc_xfer.cpp) without a GPU, with errors on request.
//
// Work on a stream is queued and runs when the stream or an event on it is
// waited for, so what a call leaves behind can be counted.  A state copy or a
// record array holds one number in its first 8 bytes: a state's number grows by
// 1 with every step, records carry the number of the state they belong to, and
// a kernel that is given records of another state counts as a mistake.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "nuosc_dev.h"

using namespace nuosc;
using Op = std::function<void()>;

struct ihipGraph { std::vector<Op> ops; };
struct hipGraphExec { std::vector<Op> ops; };
struct ihipStream_t {
    int device = 0;
    std::vector<Op> queue;
    ihipGraph* capture = nullptr;
};
struct ihipEvent_t {
    int device = 0;
    ihipStream_t* stream = nullptr;
    double at = 0;
};

namespace {
std::recursive_mutex mu;
double now_ms = 0;
long long mistakes = 0, device_bytes = 0, graphs = 0;
unsigned host_flags = 0, event_flags = 0;
std::map<std::string, int> fail_in;          // call or kernel -> fails at the n-th from now
std::map<std::string, long long> count;      // how often it ran
std::map<void*, size_t> device_mem;
std::vector<ihipStream_t*> streams;
double best_zlen[kLone + 1] = {};
int last_zlen[kLone + 1] = {};
std::vector<BatchMember> batch_members;
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;

hipError_t err(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
bool fails(const char* what) {
    std::lock_guard<std::recursive_mutex> g(mu);
    ++count[what];
    auto it = fail_in.find(what);
    if (it == fail_in.end() || --it->second > 0) return false;
    fail_in.erase(it);
    return true;
}
void run(ihipStream_t* s) {
    std::lock_guard<std::recursive_mutex> g(mu);
    if (std::find(streams.begin(), streams.end(), s) == streams.end()) return;   // (an event's, gone)
    std::vector<Op> q;
    q.swap(s->queue);
    for (Op& op : q) op();
}
void submit(ihipStream_t* s, Op op) {
    std::lock_guard<std::recursive_mutex> g(mu);
    if (s->capture) s->capture->ops.push_back(op);
    else s->queue.push_back(op);
}
// a launch checks the last error, as hipGetLastError() after a real one does
hipError_t launch(const char* name, ihipStream_t* s, double ms, Op op) {
    if (fails(name) || fails("launch")) return hipErrorLaunchFailure;
    submit(s, [=] { now_ms += ms; op(); });
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
double& tag(const void* p) { return *(double*)p; }
void expect(bool ok) { mistakes += !ok; }
}  // namespace

extern "C" {

void fake_reset() {
    std::lock_guard<std::recursive_mutex> g(mu);
    fail_in.clear();
    count.clear();
    mistakes = 0;
    last = hipSuccess;
    current = 0;
    for (double& b : best_zlen) b = 0;
}
void fake_fail(const char* what, int nth) { fail_in[what] = nth; }
long long fake_count(const char* what) { return count[what]; }
long long fake_mistakes() { return mistakes; }
long long fake_device_bytes() { return device_bytes; }
long long fake_graphs() { return graphs; }
unsigned fake_host_flags() { return host_flags; }
unsigned fake_event_flags() { return event_flags; }
int fake_pending() {
    size_t n = 0;
    for (ihipStream_t* s : streams) n += s->queue.size();
    return (int)n;
}
void fake_best_zlen(int pair, double z) { best_zlen[pair] = z; }
int fake_last_zlen(int pair) { return last_zlen[pair]; }

const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "ok" : "error"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipSetDevice(int d) { return current = d, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = current, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset((void*)p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    std::lock_guard<std::recursive_mutex> g(mu);
    *s = new ihipStream_t;
    (*s)->device = current;
    streams.push_back(*s);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    run(s);
    std::lock_guard<std::recursive_mutex> g(mu);
    streams.erase(std::find(streams.begin(), streams.end(), s));
    delete s;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return run(s), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
    if (fails("hipEventCreate")) return err(hipErrorOutOfMemory);
    *e = new ihipEvent_t;
    (*e)->device = current;
    event_flags = flags;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = new ihipEvent_t;
    (*e)->device = current;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    if (e->stream) run(e->stream);
    delete e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (e->device != s->device) return err(hipErrorInvalidHandle);
    e->stream = s;
    submit(s, [=] { e->at = now_ms; });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (e->stream) run(e->stream);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { return *ms = (float)(b->at - a->at), hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    if (fails("hipMalloc")) return err(hipErrorOutOfMemory);
    std::lock_guard<std::recursive_mutex> g(mu);
    *p = std::calloc(1, std::max<size_t>(n, 8));
    device_mem[*p] = n;
    device_bytes += (long long)n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    for (ihipStream_t* s : std::vector<ihipStream_t*>(streams)) run(s);
    std::lock_guard<std::recursive_mutex> g(mu);
    device_bytes -= (long long)device_mem.at(p);
    device_mem.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    if (fails("hipHostMalloc")) return err(hipErrorOutOfMemory);
    *p = std::malloc(n);
    host_flags = flags;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    submit(st, [=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
    expect(!st->capture);
    submit(st, [=] { std::memset(d, v, n); });
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    run(s);
    s->capture = new ihipGraph;
    ++graphs;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    *g = s->capture;
    s->capture = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    *x = nullptr;
    if (fails("hipGraphInstantiate")) return hipErrorOutOfMemory;
    *x = new hipGraphExec{g->ops};
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
    if (fails("hipGraphLaunch")) return hipErrorLaunchFailure;
    for (const Op& op : x->ops) submit(s, op);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    --graphs;
    delete g;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return delete x, hipSuccess; }

}  // extern "C"

namespace nuosc {

int rows_per_wave(int) { return 1; }
int waves_per_block(int) { return 4; }
int dirs_per_chunk(int) { return 64; }
bool buffer_addressable(const Geometry&, int) { return true; }
bool flavor3_addressable(const Geometry&, int) { return true; }
int ana_blocks(const Geometry&) { return 1; }
StagePlan plan_stage_zlen(const Geometry& g, int zlen) { return StagePlan{std::min(zlen, g.nz), 1, 1, 1, 1}; }
StagePlan plan_stage(const Geometry& g, int) { return plan_stage_zlen(g, 64); }
int pair_waves(const Geometry&, int, int zlen) { return zlen; }
// planned lengths of the pair kernels: 15, 25, 15, 20; of a batch: 24
int plan_pair_zlen(const Geometry& g, int, int pair, int) { return std::min(g.nz, pair == 2 ? 25 : (pair == kLone ? 20 : 15)); }
int plan_batch_zlen(const std::vector<Geometry>&, int, int) { return 24; }
// a kernel takes 1 ms where its segments have the best length, longer elsewhere
static double pair_ms(int pair, int zlen) {
    last_zlen[pair] = zlen;
    return 1.0 + std::abs(zlen - best_zlen[pair]) / (pair == 2 ? 5.0 : 10.0);   // (pair 2 the longer)
}
static int zlen_of(const int* z, int pair) { return z[pair - 1]; }
[[maybe_unused]] static int zlen_of(int z, int) { return z; }

template <typename T>
hipError_t launch_init(const Geometry&, int, const double*, const double*, const double*, const double*, double,
                       uint64_t seed, T* y, hipStream_t s) {
    return launch("init", s, 1, [=] { tag(y) = (double)seed; });
}
template <typename T>
hipError_t launch_analysis(const Geometry&, const T*, const double*, const double*, double*, double* out, hipStream_t s) {
    return launch("analysis", s, 1, [=] { std::fill(out, out + kNAna, 1.0); });
}
template <typename T>
hipError_t launch_ghosted(const Geometry&, int, int, const T* y, int, double* dst, hipStream_t s) {
    return launch("ghosted", s, 1, [=] { *dst = tag(y); });
}
template <typename T>
hipError_t launch_pack(const Geometry&, const T* y, int, long long, long long cnt, double* dst, hipStream_t s) {
    return launch("pack", s, 1, [=] { std::fill(dst, dst + cnt, tag(y)); });
}
template <typename T>
hipError_t launch_unpack(const Geometry&, const double* src, T* y, int, long long, long long, hipStream_t s) {
    return launch("unpack", s, 1, [=] { tag(y) = *src; });
}
template <typename T>
hipError_t launch_p3_slice(const Geometry&, const T* y, const double*, const int*, const int*, int, long long, long long cnt,
                           double* dst, hipStream_t s) {
    return launch("p3", s, 1, [=] { std::fill(dst, dst + cnt, tag(y)); });
}
template <typename T>
hipError_t launch_xghosts(const Geometry&, T*, hipStream_t s) { return launch("xghosts", s, 1, [] {}); }
template <typename T>
hipError_t launch_open_ghosts(const Geometry&, T*, const double*, const double*, const Inflow&, const double*, double,
                              hipStream_t s) {
    return launch("open_ghosts", s, 1, [] {});
}
template <typename T>
hipError_t launch_renorm(const Geometry&, T* y, const double*, const double*, hipStream_t s) {
    return launch("renorm", s, 1, [=] { tag(y) += 1000; });
}
template <typename T>
hipError_t launch_moments(const Geometry&, const T* y, double* part, hipStream_t s) {
    return launch("moments", s, 1, [=] { tag(part) = tag(y); });
}
template <typename T>
hipError_t launch_moments3(const Geometry&, const T* y, double* tot, hipStream_t s) {
    return launch("moments", s, 1, [=] { tag(tot) = tag(y); });
}
hipError_t launch_moment_totals(const Geometry&, bool, const double* part, double* tot, hipStream_t s) {
    return launch("totals", s, 1, [=] { tag(tot) = tag(part); });
}
hipError_t launch_moment_totals3(const Geometry&, const double* part, double* tot, hipStream_t s) {
    return launch("totals", s, 1, [=] { tag(tot) = tag(part); });
}
hipError_t launch_advance_time(double* t, double dt, hipStream_t s) { return launch("time", s, 1, [=] { *t += dt; }); }

// stages: the inputs' and outputs' numbers of RK4 (1-4) and SSP-RK3 (5-7)
static void stage(int st, const void* yin, const void* u, void* w, void* yout, const double* mtot, double* mpart) {
    expect(tag(mtot) == tag(yin));
    switch (st) {
        case 0: return;
        case 1: case 5: tag(yout) = tag(yin) + 0.25; break;
        case 2: tag(w) = tag(u); tag(yout) = tag(u) + 0.5; break;
        case 3: case 6: tag(yout) = tag(u) + 0.75; break;
        case 4: tag(yout) = tag(w) + 1; break;
        default: tag(yout) = tag(u) + 1; break;
    }
    tag(mpart) = tag(yout);
}
template <typename T>
hipError_t launch_stage(int st, const Geometry&, const Physics&, const StagePlan&, const T* yin, const T* u, T* w, T* yout,
                        const double* mtot, double* mpart, double, double, hipStream_t s, double, double) {
    return launch("stage", s, 1, [=] { stage(st, yin, u, w, yout, mtot, mpart); });
}
template <typename T>
hipError_t launch_stage3(int st, const Geometry&, const Physics&, const T* yin, const T* u, T* w, T* yout, const double* mtot,
                         double* mpart, double, double, hipStream_t s, double, double) {
    return launch("stage", s, 1, [=] { stage(st, yin, u, w, yout, mtot, mpart); });
}

static void predict(int pair, const PairBuffers& b) {
    const bool first = pair == 1 || pair == 3;
    expect(tag(b.tot) == tag(first ? b.u : b.y3));
    tag(first ? b.mu : b.m3) = tag(b.tot);
}
static void pair_kernel(int pair, int esize, const PairBuffers& b) {
    const bool first = pair == 1 || pair == 3;
    if (first) tag(b.y3) = tag(b.u) + 0.5;
    else tag(b.unew) = tag(b.u) + 1;
    if (esize == 4 && pair == 1) tag(b.a) = tag(b.u);
    if (esize == 4 && pair == 2) expect(tag(b.a) == tag(b.u));
    tag(b.part) = tag(first ? b.y3 : b.unew);
}
template <typename T>
hipError_t launch_pair(int pair, const Geometry&, const Physics&, int zlen, const PairBuffers& b, double, hipStream_t s) {
    const PairBuffers c = b;
    return launch("pair", s, pair_ms(pair, zlen), [=] { pair_kernel(pair, sizeof(T), c); });
}
hipError_t launch_pair_predict(int pair, const Geometry&, const Physics&, const PairBuffers& b, double, hipStream_t s) {
    const PairBuffers c = b;
    return launch("predict", s, 1, [=] { predict(pair, c); });
}
hipError_t launch_pair_totals(const Geometry&, bool, const PairBuffers& b, hipStream_t s) {
    const PairBuffers c = b;
    return launch("pair_totals", s, 1, [=] { tag(c.tot) = tag(c.part); });
}
template <typename T>
hipError_t launch_pair_ghosts(int, const Geometry&, const PairBuffers&, const double*, const double*, const Inflow&,
                              const double*, double, hipStream_t s) {
    return launch("pair_ghosts", s, 1, [] {});
}
template <typename T>
hipError_t launch_pair_sums(const Geometry&, const T* y, double* part, hipStream_t s) {
    return launch("pair_sums", s, 1, [=] { tag(part) = tag(y); });
}

hipError_t batch_build(BatchTables& t, const std::vector<BatchMember>& ms, int esize, int launch_form, hipStream_t) {
    if (fails("batch_build")) return hipErrorOutOfMemory;
    t.esize = esize;
    t.launch = launch_form;
    t.nblocks[0] = (int)ms.size();
    batch_members = ms;
    return hipSuccess;
}
void batch_free(BatchTables&) {}
static PairBuffers flipped(PairBuffers b, int flip) {
    if (flip) std::swap(b.u, b.unew);
    return b;
}
hipError_t batch_pair(const BatchTables& t, int pair, int flip, hipStream_t s) {
    const std::vector<BatchMember> ms = batch_members;
    const int esize = t.esize;
    double ms_all = 0;
    for (const BatchMember& m : ms) ms_all += pair_ms(pair, zlen_of(m.zlen, pair));
    return launch("batch_pair", s, ms_all, [=] {
        for (const BatchMember& m : ms) pair_kernel(pair, esize, flipped(m.b, flip));
    });
}
hipError_t batch_step(const BatchTables& t, int flip, hipStream_t s) {
    const std::vector<BatchMember> ms = batch_members;
    for (int pair = 1; pair <= 2; ++pair) {
        hipError_t e = launch("predict", s, 1, [=] { for (const BatchMember& m : ms) predict(pair, flipped(m.b, flip)); });
        if (e == hipSuccess) e = batch_pair(t, pair, flip, s);
        if (e == hipSuccess)
            e = launch("pair_totals", s, 1, [=] { for (const BatchMember& m : ms) tag(m.b.tot) = tag(m.b.part); });
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
static std::vector<StageMember> stage_members;
hipError_t stage_batch_build(StageBatch& t, const std::vector<StageMember>& ms, int, int, hipStream_t) {
    t.nblocks = (int)ms.size();
    stage_members = ms;
    return hipSuccess;
}
void stage_batch_free(StageBatch&) {}
hipError_t stage_batch_step(const StageBatch&, int nstages, hipStream_t s) {
    const std::vector<StageMember> ms = stage_members;
    return launch("stage_batch", s, 1, [=] {
        for (const StageMember& m : ms) {
            expect(tag(m.mu) == tag(m.u));
            tag(m.ya) = tag(m.u) + 0.25;
            if (nstages == 4) tag(m.mu) = tag(m.u) += 1;
        }
    });
}

#define INST(T)                                                                                                          \
    template hipError_t launch_init<T>(const Geometry&, int, const double*, const double*, const double*, const double*, \
                                       double, uint64_t, T*, hipStream_t);                                               \
    template hipError_t launch_analysis<T>(const Geometry&, const T*, const double*, const double*, double*, double*,    \
                                           hipStream_t);                                                                 \
    template hipError_t launch_ghosted<T>(const Geometry&, int, int, const T*, int, double*, hipStream_t);               \
    template hipError_t launch_pack<T>(const Geometry&, const T*, int, long long, long long, double*, hipStream_t);      \
    template hipError_t launch_unpack<T>(const Geometry&, const double*, T*, int, long long, long long, hipStream_t);    \
    template hipError_t launch_p3_slice<T>(const Geometry&, const T*, const double*, const int*, const int*, int,        \
                                           long long, long long, double*, hipStream_t);                                  \
    template hipError_t launch_xghosts<T>(const Geometry&, T*, hipStream_t);                                             \
    template hipError_t launch_open_ghosts<T>(const Geometry&, T*, const double*, const double*, const Inflow&,          \
                                              const double*, double, hipStream_t);                                       \
    template hipError_t launch_renorm<T>(const Geometry&, T*, const double*, const double*, hipStream_t);                \
    template hipError_t launch_moments<T>(const Geometry&, const T*, double*, hipStream_t);                              \
    template hipError_t launch_moments3<T>(const Geometry&, const T*, double*, hipStream_t);                             \
    template hipError_t launch_stage<T>(int, const Geometry&, const Physics&, const StagePlan&, const T*, const T*, T*,  \
                                        T*, const double*, double*, double, double, hipStream_t, double, double);        \
    template hipError_t launch_stage3<T>(int, const Geometry&, const Physics&, const T*, const T*, T*, T*, const double*, \
                                         double*, double, double, hipStream_t, double, double);                          \
    template hipError_t launch_pair<T>(int, const Geometry&, const Physics&, int, const PairBuffers&, double, hipStream_t); \
    template hipError_t launch_pair_ghosts<T>(int, const Geometry&, const PairBuffers&, const double*, const double*,    \
                                              const Inflow&, const double*, double, hipStream_t);                        \
    template hipError_t launch_pair_sums<T>(const Geometry&, const T*, double*, hipStream_t);
INST(double)
INST(float)

}  // namespace nuosc
