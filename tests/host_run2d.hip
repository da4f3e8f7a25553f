// The host side of the resident 2D steps (vti_run2d.hip) over a runtime that
// is made up here: allocations are host memory, launches are only recorded and
// refused as the scenario asks.  No device is touched and no kernel runs.
// test_host_run2d.py builds it with the device passes left out and runs one
// scenario (argv[1]) a time; a failed condition names itself and ends it.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <thread>

#include "../geophysics_amd/csrc/vti_run2d.hip"

#define CHECK(x)                                        \
    do {                                                \
        if (!(x)) {                                     \
            std::printf("line %d: %s\n", __LINE__, #x); \
            std::exit(1);                               \
        }                                               \
    } while (0)

// ---- the runtime ------------------------------------------------------------
struct Launched {
    const void *kernel;
    int grid, block;
    size_t lds;
};
static std::vector<Launched> g_launched;
static std::map<const void *, int> g_lds_max;       // the attribute of each function
static std::function<void()> g_after_attribute;     // what another thread does after this one's set
static std::vector<hipError_t> g_refuse;            // what the next launches return, hipSuccess: as usual
static std::vector<std::string> g_order;            // launches, events and waits, with their streams
static bool g_busy = false;                         // the latest noted launch is under way
static hipStream_t g_capturing = nullptr;
static int g_mask = 256;                            // CUs that a stream may use
static bool g_no_memory = false;
static int g_cus = 256, g_lds = 163840;

extern "C" {
char __hip_fatbin[64];
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return !g_no_memory && (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c)
{
    *c = s && s == g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? g_cus : (a == hipDeviceAttributeMaxSharedMemoryPerBlock ? g_lds : 1);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int v)
{
    g_lds_max[f] = v;
    std::function<void()> other;
    other.swap(g_after_attribute);
    if (other) other();
    return hipSuccess;
}
static std::string named(const char *what, hipStream_t s) { return what + std::to_string((size_t)s); }
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t lds, hipStream_t s)
{
    if (!g_refuse.empty()) {
        const hipError_t e = g_refuse.front();
        g_refuse.erase(g_refuse.begin());
        if (e != hipSuccess) return e;
    }
    if (!g_lds_max.count(f) || (int)lds > g_lds_max[f] || (int)lds > g_lds) return hipErrorInvalidValue;
    g_launched.push_back({f, (int)g.x, (int)b.x, lds});
    g_order.push_back(named("launch ", s));
    return hipSuccess;
}
hipError_t hipExtStreamGetCUMask(hipStream_t, uint32_t n, uint32_t *m)
{
    for (int k = 0; k < (int)n * 32; ++k)
        if (k < g_mask) m[k / 32] |= 1u << k % 32;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(1);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t s)
{
    g_order.push_back(named("record ", s));
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return g_busy ? hipErrorNotReady : hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned)
{
    g_order.push_back(named("wait ", s));
    return hipSuccess;
}
hipError_t hipDeviceGetPCIBusId(char *p, int n, int)
{
    std::snprintf(p, n, "host-%d", (int)getpid());   // no device's
    return hipSuccess;
}
hipError_t hipDeviceGet(hipDevice_t *d, int)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetUuid(hipUUID *u, hipDevice_t)
{
    *u = hipUUID{};
    return hipSuccess;
}
}

namespace vti {
int fail(int code, const std::string &) { return code; }
hipError_t launch_zero(float *p, size_t n, hipStream_t)
{
    std::memset(p, 0, n * sizeof(float));
    return hipSuccess;
}
VtiState main_state(vti_ctx *c)
{
    VtiState s;
    for (int k = 0; k < 11; ++k) s.f[k] = c->f[k];
    return s;
}

// ---- scenarios --------------------------------------------------------------
struct Ctx : vti_ctx {   // a 2D context, its padded size
    Ctx(int nnx, int nnz)
    {
        cfg.ndim = 2;
        cfg.mode = VTI_MODE_GPU_REF;
        cfg.dt = 1e-3f;
        cfg.dx = cfg.dy = cfg.dz = 10.0f;
        g = Grid{nnx, 1, nnz, (nnz + 31) / 32 * 32, 0};
        g.ldxy = (long long)g.ldz * nnx;
        nvol = (size_t)g.ldxy;
        nnmax = std::max(nnx, nnz);
    }
    ~Ctx() { run2d_free(this); }
};

// Two threads whose tiles of one kernel need different amounts of LDS: the
// smaller one's launch comes, if it can, between the larger one's attribute and
// launch.
void lds_attribute()
{
    Ctx large(1440, 543), small(1340, 543);
    int r = -1;
    std::thread other;
    g_after_attribute = [&] {
        other = std::thread([&] { r = run2d_steps(&small, 0, 32); });
        std::this_thread::sleep_for(std::chrono::milliseconds(200));
    };
    const int q = run2d_steps(&large, 0, 32);
    other.join();
    CHECK(q == 1 && r == 1 && g_launched.size() == 2);
    CHECK(g_launched[0].kernel == g_launched[1].kernel && g_launched[0].lds != g_launched[1].lds);
    for (const auto &m : g_lds_max) CHECK(m.second == g_lds - (int)kStaticLds);
}

// A refused launch leaves that call to the per-step kernels and no later one.
void refused_step()
{
    Ctx c(440, 440);
    g_refuse = {hipErrorOutOfMemory};
    CHECK(run2d_steps(&c, 0, 32) == 0);
    CHECK(run2d_steps(&c, 32, 16) == 1 && g_launched.size() == 1);
}

hipStream_t stream(int k) { return reinterpret_cast<hipStream_t>((size_t)k); }

// No two resident launches under way at once: those of one stream follow each
// other by themselves, without events; those of several by events, the launch
// that was under way when the second stream came included; a stream that its
// context has left is not touched again.
void launch_order()
{
    using Order = std::vector<std::string>;
    Ctx a(440, 440), c(240, 240);
    a.stream = stream(1);
    c.stream = stream(1);
    CHECK(run2d_steps(&a, 0, 32) == 1 && run2d_steps(&c, 0, 32) == 1 && run2d_steps(&a, 0, 32) == 1);
    CHECK((g_order == Order{"launch 1", "launch 1", "launch 1"}));
    {
        Ctx b(440, 440);
        b.stream = stream(2);
        g_order.clear();
        g_capturing = stream(1);        // no event there, so not now
        CHECK(run2d_steps(&b, 0, 32) == 0 && g_order.empty());
        g_capturing = nullptr;
        CHECK(run2d_steps(&b, 0, 32) == 1 && run2d_steps(&b, 0, 32) == 1);
        CHECK((g_order == Order{"record 1", "wait 2", "launch 2", "record 2", "launch 2", "record 2"}));
        g_order.clear();
        CHECK(run2d_steps(&c, 0, 32) == 1);
        CHECK((g_order == Order{"wait 1", "launch 1", "record 1"}));
        run2d_leave(&b);            // vti_set_stream
        b.stream = stream(3);
        g_order.clear();
        CHECK(run2d_steps(&a, 0, 32) == 1 && run2d_steps(&b, 0, 32) == 1);
        CHECK((g_order == Order{"launch 1", "record 1", "wait 3", "launch 3", "record 3"}));
    }
    g_order.clear();                // stream 3 has gone
    CHECK(run2d_steps(&a, 0, 32) == 1);
    CHECK((g_order == Order{"launch 1"}));
}

// A short call does not wait for another stream's launch, a long one and a
// program do.
void short_calls()
{
    Ctx a(440, 440), b(440, 440);
    a.stream = stream(1);
    b.stream = stream(2);
    CHECK(run2d_steps(&a, 0, 32) == 1 && run2d_steps(&b, 0, 32) == 1);
    g_busy = true;
    CHECK(run2d_steps(&a, 0, 23) == 0 && run2d_steps(&b, 0, 23) == 1);   // b's own
    g_order.clear();
    CHECK(run2d_steps(&a, 0, 24) == 1 && g_order.front() == "wait 1");
    g_busy = false;
    CHECK(run2d_steps(&b, 0, 8) == 1);
}

// Another process that has the device's resident launches (its name, bound
// here), and a stream that may not use all CUs: the per-step kernels.
void shared_device()
{
    sockaddr_un n{};
    n.sun_family = AF_UNIX;
    const int len = std::snprintf(n.sun_path + 1, sizeof n.sun_path - 1, "vti-resident-host-%d-%032d", (int)getpid(), 0);
    const int fd = socket(AF_UNIX, SOCK_STREAM, 0);
    const socklen_t size = (socklen_t)(offsetof(sockaddr_un, sun_path) + 1 + len);
    auto held = [&] { return bind(fd, reinterpret_cast<sockaddr *>(&n), size) != 0; };
    CHECK(!held());
    Ctx a(440, 440);
    CHECK(run2d_steps(&a, 0, 32) == 0 && g_launched.empty());
    close(fd);
    CHECK(run2d_steps(&a, 0, 32) == 1);
    {
        Ctx b(440, 440);
        CHECK(run2d_steps(&b, 0, 32) == 1);
        run2d_free(&a);
    }
    const int again = socket(AF_UNIX, SOCK_STREAM, 0);    // given back with the last object
    CHECK(bind(again, reinterpret_cast<sockaddr *>(&n), size) == 0);
    close(again);
    g_mask = 255;
    Ctx c(440, 440);
    CHECK(run2d_steps(&c, 0, 32) == 0);
    g_mask = 256;
    CHECK(run2d_steps(&c, 0, 32) == 1);
}

struct Group : Run2dGroup {   // shots of two parts
    std::vector<Run2dShot> shots;
    std::vector<Run2dOp> ops{Run2dOp{1, 0, 8, 1, 0, 0, 0}};
    std::vector<long long> offs = std::vector<long long>(8, 0);
    Group()
    {
        for (int nnx : {2441, 2401}) {
            Run2dShot b{};
            b.nnx = b.M = nnx;
            b.nnz = 543;
            b.ldz = 544;
            shots.push_back(b);
        }
        CHECK(run2d_group_make(*this, run2d_parts(shots, 0), shots, false, 8, nullptr) == 1);
        CHECK(parts.part.size() == 2);
    }
    ~Group() { run2d_group_free(*this); }
    int run() { return run2d_group_run(*this, ops, offs, 1, nullptr); }
};

// A program refused before its first part has run nothing, one refused later
// has; both leave the group alone until the next set of shots.
void refused_program()
{
    Group g;
    CHECK(g.run() == 1 && g_launched.size() == 2);
    g_refuse = {hipErrorOutOfMemory};
    CHECK(g.run() == 0 && g.run() == 0 && g_launched.size() == 2);
    CHECK(run2d_group_set(g, g.shots, nullptr) == VTI_OK && g.run() == 1 && g_launched.size() == 4);
    g_refuse = {hipSuccess, hipErrorOutOfMemory};
    CHECK(g.run() == 2 && g.run() == 0 && g_launched.size() == 5);
    g.offs.resize(1 << 16);   // a program larger than the group's share of memory, and none to be had
    g.ops[0].n = 1 << 16;
    CHECK(run2d_group_set(g, g.shots, nullptr) == VTI_OK);
    g_no_memory = true;
    CHECK(g.run() == 0 && g.run() == 0 && g_launched.size() == 5);
    g_no_memory = false;
    CHECK(run2d_group_set(g, g.shots, nullptr) == VTI_OK && g.run() == 1 && g_launched.size() == 7);
}

// An exchange that never came is reported once, by the check after the program
// that missed it; the object then keeps the per-step kernels.
void missed_exchange()
{
    Group g;
    CHECK(g.run() == 1 && run2d_group_check(g, nullptr) == VTI_OK);
    CHECK(g.run() == 1);
    *g.dead = 1;   // as a workgroup does
    CHECK(run2d_group_check(g, nullptr) == VTI_ERR_HIP);
    CHECK(run2d_group_set(g, g.shots, nullptr) == VTI_OK && g.run() == 0);
    CHECK(run2d_group_check(g, nullptr) == VTI_OK);
}

// The parts of a list of shots by a plain search, every number of shots and
// every cost anew.
Run2dParts plain_parts(const std::vector<Run2dShot> &shots, const Device2d &d)
{
    Run2dParts r;
    const int ns = (int)shots.size();
    std::vector<std::vector<Cut>> cuts[kRtmShapes];
    for (int j = 0; j < kRtmShapes; ++j)
        for (const Run2dShot &s : shots) {
            cuts[j].emplace_back();
            cuts_of(s.nnx, s.nnz, false, j, d.cus, d.lds, cuts[j].back());
            if (j == kRtmShapes - 1)
                for (Cut &c : cuts[j].back()) c.cost *= 2.0;
        }
    for (int first = 0; first < ns;) {
        double rate = 1e300, cells = 0.0;
        Run2dPart part{};
        std::vector<Cut> taken;
        for (int n = 1; first + n <= ns; ++n) {
            cells += (double)shots[first + n - 1].nnx * shots[first + n - 1].nnz;
            double least = 1e300;
            int shape = 0;
            std::vector<Cut> pick;
            for (int j = 0; j < kRtmShapes; ++j) {
                std::vector<double> costs;
                for (int s = 0; s < n; ++s)
                    for (const Cut &c : cuts[j][first + s]) costs.push_back(c.cost);
                std::sort(costs.begin(), costs.end());
                auto fit = [&](double c) {
                    std::vector<Cut> p;
                    int tiles = 0;
                    for (int s = 0; s < n; ++s) {
                        const auto &l = cuts[j][first + s];
                        const auto i = std::find_if(l.begin(), l.end(), [&](const Cut &x) { return x.cost <= c; });
                        if (i == l.end() || (tiles += i->tiles) > d.cus) return std::vector<Cut>{};
                        p.push_back(*i);
                    }
                    return p;
                };
                const auto i = std::partition_point(costs.begin(), costs.end(), [&](double c) { return fit(c).empty(); });
                if (i == costs.end() || *i >= least) continue;
                least = *i;
                shape = j;
                pick = fit(*i);
            }
            if (pick.empty()) break;
            if ((least + 4000.0) / cells >= rate) continue;
            rate = (least + 4000.0) / cells;
            part = Run2dPart{first, n, shape, 0, 0};
            taken = pick;
        }
        if (taken.empty()) return Run2dParts{};
        for (const Cut &c : taken) {
            r.gx.push_back(c.gx);
            r.gz.push_back(c.gz);
            r.tile0.push_back(part.ntile);
            part.ntile += c.tiles;
            part.lds = std::max(part.lds, c.lds);
        }
        r.part.push_back(part);
        first += part.n;
    }
    return r;
}

// The plans are those of the plain search, on a whole and on a smaller device,
// with shots that no launch holds among them; every cut covers its grid with
// tiles that the kernel can hold; and a large batch is planned much faster.
void plans()
{
    unsigned seed = 7;
    auto draw = [&](int lo, int hi) { return lo + (int)((seed = seed * 1664525u + 1013904223u) >> 8) % (hi - lo); };
    double plain = 0.0, quick = 0.0;
    for (int t = 0; t < 24; ++t) {
        g_cus = t % 3 == 2 ? 64 : 256;
        std::vector<Run2dShot> shots;
        const int n = draw(1, 40), large = t % 4 == 3 ? 2500 : 900;
        for (int k = 0; k < n; ++k) {
            Run2dShot b{};
            b.nnx = draw(16, k % 5 ? 500 : large);
            b.nnz = draw(16, k % 5 ? 300 : large);
            if (k && k % 3 == 0) {      // grids that occur again
                b.nnx = shots[0].nnx;
                b.nnz = shots[0].nnz;
            }
            shots.push_back(b);
        }
        if (t == 23) shots.assign(200, shots[0]);
        Device2d d;
        CHECK(device_2d(0, d));
        auto clock = [] { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); };
        const double t0 = clock();
        const Run2dParts a = plain_parts(shots, d);
        const double t1 = clock();
        const Run2dParts b = run2d_parts(shots, 0);
        if (t == 23) {
            plain = t1 - t0;
            quick = clock() - t1;
        }
        CHECK(a.gx == b.gx && a.gz == b.gz && a.tile0 == b.tile0 && a.part.size() == b.part.size());
        for (size_t k = 0; k < a.part.size(); ++k) {
            const Run2dPart &p = a.part[k], &q = b.part[k];
            CHECK(p.first == q.first && p.n == q.n && p.shape == q.shape && p.ntile == q.ntile && p.lds == q.lds);
            CHECK(q.ntile <= d.cus && q.lds + kStaticLds <= (size_t)d.lds);
            for (int s = q.first; s < q.first + q.n; ++s) {
                const Run2dShot &g = shots[s];
                const int nt = kShapes[q.shape].nt, nu = kShapes[q.shape].nu;
                int cells = 0;
                for (int i = 0; i < b.gx[s] * b.gz[s]; ++i) {
                    const Tile w = tile_of(g.nnx, g.nnz, b.gx[s], b.gz[s], i / b.gz[s], i % b.gz[s]);
                    CHECK(w.nx >= std::min(7, g.nnx - 8) && w.nz >= 8 && w.nx + 14 <= nt);
                    CHECK((w.nx + nu - 1) / nu * w.nz <= nt && 4 * (size_t)Lds<false>(w.nx, w.nz).total <= q.lds);
                    cells += w.nx * w.nz;
                }
                CHECK(cells == (g.nnx - 8) * ((g.nnz - 8 + 3) / 4 * 4));
            }
        }
        for (bool tti : {false, true}) {
            const Plan2d one = plan_one(shots[0], tti, d);
            double least = 1e300;
            std::vector<Cut> c;
            for (int k = 0; k < kNumShapes; ++k) {
                cuts_of(shots[0].nnx, shots[0].nnz, tti, k, d.cus, d.lds, c);
                for (const Cut &x : c) least = std::min(least, x.cost);
            }
            CHECK(one.cost == least && one.cut.empty() == (least == 1e300));
        }
    }
    std::printf("200 shots: %.2f ms, plain search %.2f ms\n", 1e3 * quick, 1e3 * plain);
    CHECK(quick < 0.2 * plain);
}

}  // namespace vti

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> all = {{"lds_attribute", vti::lds_attribute},
                                                       {"refused_step", vti::refused_step},
                                                       {"launch_order", vti::launch_order},
                                                       {"short_calls", vti::short_calls},
                                                       {"shared_device", vti::shared_device},
                                                       {"refused_program", vti::refused_program},
                                                       {"missed_exchange", vti::missed_exchange},
                                                       {"plans", vti::plans}};
    const auto s = all.find(argc > 1 ? argv[1] : "");
    CHECK(s != all.end());
    s->second();
    std::printf("ok\n");
    return 0;
}
