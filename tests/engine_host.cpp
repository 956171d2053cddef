// The engine's host logic on a device that is host memory: hipMalloc and its
// like are defined here (the executable's definitions come before the HIP
// runtime's for the library too), no kernel runs, and every launch ends every
// problem.  Each scenario prints what failed and returns 1; test_engine_host.py
// builds and runs them.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "../include/suli_ps.h"
#include "../suli_amd/csrc/ps_engine.h"

using namespace sps;

namespace {

constexpr int kSlots = 256;   // of a context

struct Device {
    size_t limit = (size_t)-1, held = 0;
    std::map<void *, size_t> blocks;
    std::vector<size_t> refused;
    std::map<size_t, int> given;   // how many of a size
    // as the runtime's: kept until it is read, successful calls leave it
    hipError_t last = hipSuccess;
    CgScalars *status = nullptr;
    int slots = kSlots;
    int launches = 0, waits = 0;
    int skip_copies = 0, fail_copies = 0;   // asynchronous copies: pass these, then fail these
} dev;

hipError_t fault(hipError_t e)
{
    dev.last = e;
    return e;
}

int bad = 0;
#define CHECK(cond)                                                     \
    do {                                                                \
        if (!(cond)) std::printf("line %d: %s\n", __LINE__, #cond), bad = 1; \
    } while (0)

}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    *p = nullptr;
    if (dev.held + n > dev.limit) {
        dev.refused.push_back(n);
        return fault(hipErrorOutOfMemory);
    }
    *p = std::calloc(n, 1);
    dev.blocks[*p] = n;
    ++dev.given[n];
    dev.held += n;
    if (n == sizeof(CgScalars) * dev.slots) dev.status = static_cast<CgScalars *>(*p);
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    auto it = dev.blocks.find(p);
    if (it == dev.blocks.end()) return p ? fault(hipErrorInvalidValue) : hipSuccess;
    dev.held -= it->second;
    dev.blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::calloc(n, 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (dev.fail_copies > 0 && dev.skip_copies-- <= 0) return --dev.fail_copies, fault(hipErrorInvalidValue);
    std::memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    std::memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n)
{
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
// what a launch statement calls around hipLaunchKernel
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t)
{
    ++dev.launches;
    for (int i = 0; dev.status && i < dev.slots; ++i) dev.status[i].final_ = 1;
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = dev.last;
    dev.last = hipSuccess;
    return e;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidSymbol; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    ++dev.waits;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.f;
    return hipSuccess;
}
}

namespace {

constexpr int kN = 40;   // 40^3 cells: a problem of the multigrid iteration

suli_ps_grid grid(int n = kN)
{
    suli_ps_grid g{};
    g.nx = g.ny = g.nz = n;
    g.ccx0 = g.ccy0 = 1;
    g.t_press = 1;
    g.dx = g.dy = g.dz = g.dt = 1.0;
    return g;
}

SolveOpts fp64()
{
    SolveOpts o;
    o.stop_rule = SULI_PS_STOP_RELATIVE;
    return o;
}

double field[(kN + 3) * (kN + 3) * (kN + 3)];

struct Bench {
    Engine eng;
    hipStream_t s = nullptr;
    Bench()
    {
        hipStreamCreateWithFlags(&s, 0);
        CHECK(eng.init(s, kSlots) == 0);
        eng.set_graphs(false);
    }
    int admit(int *slot = nullptr, const SolveOpts &o = fp64())
    {
        int si = -1;
        const int rc = eng.admit(grid(), SetupIn{}, field, o, 0, &si);
        if (slot) *slot = si;
        return rc;
    }
};

const size_t tables = 1 << 20;   // room for the launch tables
const size_t plain = problem_bytes(kN, kN, kN, false);
const size_t multi = state_bytes(kN, kN, kN, fp64());

// Room for plain CG's state but not for the multigrid iteration's: plain CG,
// and no error left behind.
void fallback()
{
    Bench b;
    CHECK(multi > plain + tables);
    dev.limit = dev.held + plain + tables;
    int si = -1;
    CHECK(b.admit(&si) == 0);
    CHECK(si == 0 && b.eng.slot(0).bytes == plain && !b.eng.slot(0).mg);
    CHECK(dev.refused.size() == 2 && hipGetLastError() == hipSuccess);
    CHECK(b.eng.run_all(false) == 0);
}

// A block that only fits once the pool's cached ones are given back.
void cached()
{
    Bench b;
    SolveOpts o = fp64();
    o.keep_null = true;   // plain CG
    int si = -1;
    CHECK(b.admit(&si, o) == 0 && b.eng.run_all(false) == 0);
    b.eng.release(si);
    dev.limit = dev.held - plain + multi + tables;
    CHECK(b.admit(&si) == 0 && b.eng.slot(si).mg);
    CHECK(b.eng.run_all(false) == 0);
}

// A set-up that fails on the way leaves no problem behind, and its slot and memory
// serve the next one.
void failed_setup()
{
    Bench b;
    for (int n : {0, 1}) {   // the scalars' copy to the device, the descriptor's
        CHECK(b.admit() == 0);   // (takes slot 0)
        dev.skip_copies = n;
        dev.fail_copies = 1;
        int si = -1;
        CHECK(b.admit(&si) == SULI_PS_EHIP && si < 0);
        CHECK(dev.fail_copies == 0 && b.eng.active_count() == 1 && !b.eng.slot(1).used);
        CHECK(hipGetLastError() != hipSuccess);
        const size_t held = dev.held;
        CHECK(b.admit(&si) == 0 && si == 1);
        CHECK(dev.held == held);   // the failed one's block
        CHECK(b.eng.run_all(false) == 0);
        b.eng.release(0);
        b.eng.release(1);
    }
}

// Beside another problem, one whose multigrid state does not fit waits for memory
// instead of taking plain CG's.
void beside()
{
    Bench b;
    dev.limit = dev.held + multi + plain + tables;
    int si = -1;
    CHECK(b.admit() == 0);
    CHECK(b.admit(&si) == SULI_PS_ENOMEM && si < 0);
    CHECK(b.eng.run_all(false) == 0);
    b.eng.release(0);
    CHECK(b.admit(&si) == 0 && b.eng.slot(si).mg);
    CHECK(b.eng.run_all(false) == 0);
}

// A batch that does not fit at once is solved in parts, every problem by the
// iteration that it takes alone.
void batch()
{
    suli_ps_opts o{};
    o.precision = SULI_PS_FP64;
    o.stop_rule = SULI_PS_STOP_RELATIVE;
    o.tol = 1e-8;
    o.no_graphs = 1;
    suli_ps_ctx *ctx = suli_ps_create(&o);
    CHECK(ctx);
    dev.limit = dev.held + 2 * multi + plain + tables;
    dev.given.clear();
    suli_ps_problem p[5] = {};
    for (auto &q : p) {
        q.grid = grid();
        q.u = q.v = q.w = q.rho = q.prd1 = field;
        q.stats.status = -1;
    }
    CHECK(suli_ps_graddin_batch_dev(ctx, p, 5) == 0);
    for (auto &q : p) CHECK(q.stats.status == 0);
    CHECK(!dev.given.count(plain) && dev.given[multi] == 2);
    // none fits
    dev.limit = 0;
    suli_ps_destroy(ctx);
    dev.limit = (size_t)-1;
    ctx = suli_ps_create(&o);
    dev.limit = dev.held;
    CHECK(suli_ps_graddin_batch_dev(ctx, p, 2) == SULI_PS_ENOMEM);
    suli_ps_destroy(ctx);
}

// A chunk length chosen for plain CG's steps does not queue as many multigrid steps,
// of up to a dozen launches each, past the end of a solve.
void chunk()
{
    int launches[3], k = 0;
    for (int steps : {0, 1, 512}) {
        Bench b;
        b.eng.set_chunk(steps);
        CHECK(b.admit() == 0 && b.eng.slot(0).mg);
        const int before = dev.launches;
        CHECK(b.eng.run_all(false) == 0);
        launches[k++] = dev.launches - before;
    }
    CHECK(launches[1] <= launches[0] && launches[2] == launches[0]);
}

// The masked problems of a batch share one wait for the counts of their fluid parts.
void masks()
{
    static uint8_t solid[kN * kN * kN];
    int waits[2], k = 0;
    for (int count : {1, 8}) {
        suli_ps_opts o{};
        o.precision = SULI_PS_MIXED;
        o.stop_rule = SULI_PS_STOP_RELATIVE;
        o.tol = 1e-8;
        suli_ps_ctx *ctx = suli_ps_create(&o);
        suli_ps_problem p[8] = {};
        for (auto &q : p) {
            q.grid = grid();
            q.u = q.v = q.w = q.rho = q.prd1 = field;
            q.solid = solid;
        }
        for (int i = 1; i < count; i += 2) p[i].solid = nullptr;
        const int before = dev.waits;
        CHECK(suli_ps_graddin_batch_dev(ctx, p, count) == 0);
        waits[k++] = dev.waits - before;
        suli_ps_destroy(ctx);
    }
    CHECK(waits[1] == waits[0]);
}

}  // namespace

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> scenarios = {
        {"fallback", fallback},         {"cached", cached}, {"failed_setup", failed_setup},
        {"beside", beside},             {"batch", batch},   {"chunk", chunk},
        {"masks", masks},
    };
    const auto it = scenarios.find(argc > 1 ? argv[1] : "");
    if (it == scenarios.end()) return 2;
    it->second();
    return bad;
}
