// stub_device.cpp -- a HIP runtime of host threads, and stand-ins for the
// kernel launchers, for tests of the engine's host code without a device.
//
// A stream is a thread that runs its queue in order; events, waits on events of
// other streams, captured graphs and asynchronous copies behave as the runtime's
// do.  The kernels are replaced by work that is easy to check: a target has
// S = W / 4 splits, its outputs are placed in the pool like k_plan does, and its
// rows hold a value made from the target and the submission.
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <sys/mman.h>
#include <thread>
#include <vector>

#include "../../eagleimp_amd/csrc/eimp_launch.h"
#include "stub_device.h"

StubState stub;

namespace {
using Work = std::function<void()>;
struct Event {
    std::mutex m;
    std::condition_variable cv;
    uint64_t recorded = 0, done = 0;
};
struct Graph {
    std::vector<Work> work;
};
struct Stream {
    std::mutex m;
    std::condition_variable cv, idle;
    std::deque<Work> q;
    bool busy = false, quit = false;
    Graph *capture = nullptr;
    std::thread th;
    Stream() : th([this] { loop(); }) {}
    ~Stream() {
        {
            std::lock_guard<std::mutex> l(m);
            quit = true;
        }
        cv.notify_all();
        th.join();
    }
    void loop() {
        for (;;) {
            Work w;
            {
                std::unique_lock<std::mutex> l(m);
                cv.wait(l, [&] { return quit || !q.empty(); });
                if (q.empty()) return;
                w = std::move(q.front());
                q.pop_front();
                busy = true;
            }
            w();
            {
                std::lock_guard<std::mutex> l(m);
                busy = false;
                if (q.empty()) idle.notify_all();
            }
        }
    }
    void push(Work w) {
        if (capture) {
            capture->work.push_back(std::move(w));
            return;
        }
        {
            std::lock_guard<std::mutex> l(m);
            q.push_back(std::move(w));
        }
        cv.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> l(m);
        idle.wait(l, [&] { return q.empty() && !busy; });
    }
};
Stream *st(hipStream_t s) { return reinterpret_cast<Stream *>(s); }
Event *ev(hipEvent_t e) { return reinterpret_cast<Event *>(e); }
std::mutex map_mu;
std::map<void *, size_t> maps;  // device allocations
std::map<void *, size_t> pinned;
}  // namespace

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *c) {
    *c = 1;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = *t = 1ull << 38;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s) {
    *p = const_cast<void *>(s);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    void *m = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> l(map_mu);
    maps[m] = n;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> l(map_mu);
    munmap(p, maps.at(p));
    maps.erase(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned int) {
    if (stub.fail_host_malloc) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    std::lock_guard<std::mutex> l(map_mu);
    pinned[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::lock_guard<std::mutex> l(map_mu);
    pinned.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    *a = hipPointerAttribute_t{};
    a->type = hipMemoryTypeUnregistered;
    std::lock_guard<std::mutex> l(map_mu);
    auto it = pinned.upper_bound(const_cast<void *>(p));
    if (it != pinned.begin() && (--it, (const char *)p < (const char *)it->first + it->second))
        a->type = hipMemoryTypeHost;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int) {
    *s = reinterpret_cast<hipStream_t>(new Stream);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    delete st(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    st(s)->wait();
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t q) {
    if (k == hipMemcpyHostToDevice) {
        // pageable sources are read before the call returns
        hipPointerAttribute_t a;
        (void)hipPointerGetAttributes(&a, s);
        if (a.type == hipMemoryTypeUnregistered) {
            std::vector<char> c((const char *)s, (const char *)s + n);
            st(q)->push([=] { std::memcpy(d, c.data(), n); });
            return hipSuccess;
        }
    }
    stub.copies++;
    st(q)->push([=] {
        if (k == hipMemcpyDeviceToHost && stub.copy_us)
            std::this_thread::sleep_for(std::chrono::microseconds(stub.copy_us));
        std::memcpy(d, s, n);
        if (k == hipMemcpyDeviceToHost) stub.copies_done++;
    });
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t q) {
    st(q)->push([=] { std::memset(d, v, n); });
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
    delete ev(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Event *E = ev(e);
    uint64_t n;
    {
        std::lock_guard<std::mutex> l(E->m);
        n = ++E->recorded;
    }
    st(s)->push([=] {
        // notified under the lock: a waiter may destroy the event afterwards
        std::lock_guard<std::mutex> l(E->m);
        E->done = n;
        E->cv.notify_all();
    });
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned int) {
    Event *E = ev(e);
    uint64_t n;
    {
        std::lock_guard<std::mutex> l(E->m);
        n = E->recorded;
        if (E->done >= n) return hipSuccess;
    }
    st(s)->push([=] {
        std::unique_lock<std::mutex> l(E->m);
        E->cv.wait(l, [&] { return E->done >= n; });
    });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    Event *E = ev(e);
    std::unique_lock<std::mutex> l(E->m);
    const uint64_t n = E->recorded;
    E->cv.wait(l, [&] { return E->done >= n; });
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    std::lock_guard<std::mutex> l(ev(e)->m);
    return ev(e)->done >= ev(e)->recorded ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 1.f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    st(s)->wait();
    st(s)->capture = new Graph;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
    *g = reinterpret_cast<hipGraph_t>(st(s)->capture);
    st(s)->capture = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
    *x = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph *>(g)));
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
    stub.graphs++;
    for (const Work &w : reinterpret_cast<Graph *>(x)->work) st(s)->push(w);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    delete reinterpret_cast<Graph *>(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t g) {
    delete reinterpret_cast<Graph *>(g);
    return hipSuccess;
}
}  // extern "C"

namespace eimp {
namespace {
hipError_t none() { return hipSuccess; }
void pause_us(uint32_t us) {
    if (us) std::this_thread::sleep_for(std::chrono::microseconds(us));
}
// rows of a target: a value of the target's window, K and row
uint32_t row_word(const TgtDev &T, uint64_t i) { return (uint32_t)(i * 2654435761u + T.W * 97u + T.K); }
void fill(const TgtDev &T) {
    if (!T.Mp) return;
    for (uint64_t i = 0; i < 2ull * T.Mp * T.RS; i++) T.out[i] = row_word(T, i);
    for (uint32_t r = 0; r < T.Mp; r++) T.count0[r] = (int32_t)(r ^ T.W);
}
}  // namespace
hipError_t launch_gather(const GatherArgs &a, void *dst, hipStream_t s) {
    if (stub.fail_gather >= 0 && stub.gathers == stub.fail_gather) return hipErrorLaunchFailure;
    stub.gathers++;
    st(s)->push([=] {
        pause_us(stub.gather_us);
        for (uint32_t i = 0; i < a.n; i++) std::memcpy((char *)dst + a.off[i], a.src[i], a.bytes[i]);
    });
    return hipSuccess;
}
hipError_t launch_site_to_hap(const PanelDev &, uint64_t *, hipStream_t) { return none(); }
hipError_t launch_panel_mono(const PanelDev &, uint64_t *, uint64_t *, hipStream_t) { return none(); }
hipError_t launch_distance(const PanelDev &, const TgtDev *, const uint32_t *, uint32_t, hipStream_t) {
    return none();
}
hipError_t launch_select(const PanelDev &, const TgtDev *, uint32_t, hipStream_t) { return none(); }
hipError_t launch_monos(const PanelDev &, const TgtDev *, const uint32_t *, uint32_t, uint32_t, uint32_t,
                        hipStream_t) {
    return none();
}
hipError_t launch_splits(const PanelDev &, const TgtDev *tg, uint32_t n, hipStream_t s) {
    st(s)->push([=] {
        for (uint32_t t = 0; t < n; t++) {
            tg[t].stats[0] = tg[t].W / 4;
            tg[t].stats[1] = 1;
        }
    });
    return hipSuccess;
}
hipError_t launch_bits_to_list(const TgtDev *, uint32_t, uint32_t, int, hipStream_t) { return none(); }
hipError_t launch_cref(const PanelDev &, const TgtDev *, const CrefItem *, uint32_t, uint32_t, bool,
                       hipStream_t) {
    return none();
}
uint32_t cref_max_k() { return 65536 - 64; }
hipError_t launch_digest_count0(const TgtDev *, uint32_t, hipStream_t) { return none(); }
hipError_t launch_cref_rows(const TgtDev *, uint32_t, uint32_t Mp, uint64_t *rows, uint32_t rw, hipStream_t s) {
    st(s)->push([=] { std::memset(rows, 0, (size_t)Mp * rw * 8); });
    return hipSuccess;
}
hipError_t launch_digest_rows(const TgtDev *tg, const uint32_t *d_n, uint32_t, uint64_t *dig, hipStream_t s) {
    st(s)->push([=] {
        for (uint32_t t = 0; t < *d_n; t++) {
            for (uint64_t i = 0; i < 2ull * tg[t].Mp * tg[t].RS; i++) dig[2 * t] += dig_word(i, tg[t].out[i]);
            for (uint32_t r = 0; r < tg[t].Mp; r++) dig[2 * t + 1] += dig_count0(r, tg[t].count0[r]);
        }
    });
    return hipSuccess;
}
size_t pbwt_big_lds_bytes(uint32_t) { return 1024; }
uint32_t pbwt_big_max_k() { return 1u << 19; }
hipError_t launch_pbwt_big(const BigItem *, uint32_t, uint32_t, hipStream_t) { return none(); }
static const int kNt[] = {256, 256, 512, 512, 1024, 512, 1024}, kCpw[] = {8, 16, 20, 32, 24, 20, 24};
int pbwt_variant_count() { return 7; }
int pbwt_variant_threads(int v) { return kNt[v]; }
int pbwt_variant_cpw(int v) { return kCpw[v]; }
uint32_t pbwt_variant_maxk(int v) { return (uint32_t)(kNt[v] * kCpw[v]); }
size_t pbwt_lds_bytes(int v, uint32_t Kpad) {
    return (int)((Kpad + kNt[v] - 1) / kNt[v]) > kCpw[v] ? ~(size_t)0 : 5u * Kpad + 8192;
}
hipError_t pbwt_prepare(int v, size_t, int *occ) {
    if (occ) *occ = kNt[v] == 512 ? 3 : kNt[v] == 1024 ? 1 : 4;
    return hipSuccess;
}
hipError_t launch_order(int v, const TgtDev *, const OrderItem *, bool, uint32_t, const uint32_t *, uint32_t *,
                        uint16_t *, size_t, hipStream_t) {
    stub.order_variant = v;
    return none();
}
hipError_t launch_dense(int, const TgtDev *, uint32_t, const uint16_t *, int32_t *, size_t, hipStream_t) {
    return none();
}
hipError_t launch_rows(const TgtDev *tg, const uint32_t *d_n, uint32_t n, const uint32_t *, RowItem *, uint32_t *,
                       uint32_t, uint64_t, uint32_t, hipStream_t s) {
    st(s)->push([=] {
        pause_us(stub.build_us);
        for (uint32_t t = 0; t < (d_n ? *d_n : n); t++) fill(tg[t]);
    });
    return hipSuccess;
}
hipError_t launch_prep_dev(int cls, const PanelDev &P, const TgtDev *tg, const uint32_t *d_n, uint32_t, uint32_t,
                           uint32_t, hipStream_t s) {
    (void)P;
    if (cls != 3) return hipSuccess;
    st(s)->push([=] {
        pause_us(stub.prep_us);
        for (uint32_t t = 0; t < *d_n; t++) {
            tg[t].stats[0] = tg[t].W / 4;
            tg[t].stats[1] = 1;
        }
    });
    return hipSuccess;
}
hipError_t launch_plan(TgtDev *tg, BatchDev *B, const PlanArgs &A, hipStream_t s) {
    st(s)->push([=] {
        uint64_t off = 0;
        for (uint32_t t = 0; t < B->n; t++) {
            TgtDev &T = tg[t];
            const uint32_t Mp = 2 * T.stats[0] + 1, Kpad = (T.K + 63) / 64 * 64, RS = row_stride(T.K, A.layout);
            const uint64_t cb = region_cref_bytes(Mp, Kpad), c0b = region_c0_bytes(Mp), ob = region_out_bytes(Mp, RS);
            const bool fit = off + cb + c0b + ob <= A.pool_cap;
            T.S = T.stats[0];
            T.stats[2] = fit ? 0u : 1u;
            T.Mp = fit ? Mp : 0u;
            T.Kpad = Kpad;
            T.RS = RS;
            T.cref = (uint16_t *)(A.pool + off);
            T.count0 = (int32_t *)(A.pool + off + cb);
            T.out = (uint32_t *)(A.pool + off + cb + c0b);
            off += cb + c0b + ob;
        }
    });
    return hipSuccess;
}
hipError_t launch_digest_count0_dev(const TgtDev *, const uint32_t *, uint32_t, hipStream_t) { return none(); }
size_t cref_lds_bytes(const PanelDev &, uint32_t) { return 1024; }
hipError_t cref_persist_prepare(const PanelDev &, uint32_t, int *occ) {
    occ[0] = occ[1] = 2;
    return hipSuccess;
}
bool cref_ident_ok(const PanelDev &) { return true; }
hipError_t launch_site_blocks(const PanelDev &, uint64_t, uint32_t, uint16_t *, hipStream_t) { return none(); }
hipError_t launch_cref_persist(const PanelDev &, const TgtDev *, BatchDev *, const uint32_t *, const uint32_t *,
                               uint32_t, const uint32_t *, hipStream_t) {
    return none();
}
}  // namespace eimp

uint64_t stub_digest(uint32_t W, uint32_t K, uint32_t layout) {
    eimp::TgtDev T{};
    T.W = W;
    T.K = K;
    T.Mp = 2 * (W / 4) + 1;
    T.RS = eimp::row_stride(K, layout);
    uint64_t d = 0;
    for (uint64_t i = 0; i < 2ull * T.Mp * T.RS; i++) d += eimp::dig_word(i, eimp::row_word(T, i));
    return d;
}
