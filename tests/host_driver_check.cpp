// The host side of the C ABI (psp_amd/csrc/psp_hip.cpp) against a HIP runtime
// made of host memory, without a GPU:
//   host_driver_check fused|oom|retry|memory|several nx ny nz [precision]
// The kernels' launch wrappers here compute nothing; they check that every
// array they are given lies in live memory and is as large as the kernel needs,
// and count.
//  fused: which calls factor, allocate and run which panel solves when the
//         fused launches are switched on after Initialize;
//  oom:   the same without the memory for their layout;
//  retry: Initialize after a first one whose n-th allocation failed, for
//         every n;
//  memory: the most memory that Initialize holds;
//  several: what several factored contexts hold.
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "kernels.hpp"
#include "psp_hip.h"

using namespace psp_amd;

static int fails = 0;
static void need(bool ok, const char* what, long a = 0, long b = 0)
{
    if (ok) return;
    std::fprintf(stderr, "FAIL %s (%ld, %ld)\n", what, a, b);
    if (++fails > 20) std::exit(1);
}

// ---- device memory -----------------------------------------------------------
static std::map<char*, size_t> live;
static size_t used = 0, most = 0, smallest = 0, capacity = (size_t)-1;
static long allocs = 0, frees = 0, failAt = -1;  // failAt: allocations (of at least
                                                 // `smallest` bytes) until all fail
static bool failed = false;
static std::mutex mu;
static hipError_t lastError = hipSuccess;

static hipError_t Set(hipError_t e)
{
    if (e != hipSuccess) lastError = e;
    return e;
}

static void Live(const void* p, double bytes, const char* what)
{
    std::lock_guard<std::mutex> lock(mu);
    auto it = live.upper_bound((char*)p);
    if (p && it != live.begin()) {
        --it;
        if ((char*)p + (size_t)bytes <= it->first + it->second) return;
    }
    need(bytes <= 0, what, (long)(size_t)p, (long)bytes);
}

hipError_t hipMalloc(void** p, size_t n)
{
    std::lock_guard<std::mutex> lock(mu);
    ++allocs;
    if (used + n > capacity || (n >= smallest && failAt == 0)) {
        failed = true;
        return Set(hipErrorOutOfMemory);
    }
    if (n >= smallest && failAt > 0) --failAt;
    *p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (*p == MAP_FAILED) std::abort();
    live[(char*)*p] = n;
    used += n;
    most = std::max(most, used);
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    std::lock_guard<std::mutex> lock(mu);
    ++frees;
    auto it = live.find((char*)p);
    need(p == nullptr || it != live.end(), "free of no allocation");
    if (it == live.end()) return hipSuccess;
    used -= it->second;
    munmap(p, it->second);
    live.erase(it);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t)
{
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void* d, int, size_t n, hipStream_t)
{
    Live(d, (double)n, "memset");  // (new memory is zero)
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s)
{
    *p = (void*)s;
    live[(char*)s] = (size_t)64 << 20;
    return hipSuccess;
}

// ---- the rest of the runtime ---------------------------------------------------
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError()
{
    const hipError_t e = lastError;
    lastError = hipSuccess;
    return e;
}
static char token;
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)&token, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = (hipGraph_t)&token, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    return *e = (hipGraphExec_t)&token, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)&token, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }

// ---- launches ------------------------------------------------------------------
static std::atomic<long> factorizations{0}, merged{0}, fusedSolves{0}, couplings{0};
static std::atomic<bool> slow{false};

namespace psp_amd {
bool XcdRoundRobin(hipStream_t) { return true; }
void PrimeSolveOccupancy() {}
int ReducePartials(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(512, (n + 255) / 256)); }
int64_t ArnoldiPartials(int64_t np, int k, int m) { return 2 * (int64_t)std::min(m, 64) * ReducePartials(np) * k; }
int64_t ArnoldiGram(int k, int m) { return (int64_t)std::min(m, 64) * std::min(m, 64) * k; }
int32_t* SliceCounters(const ClassDev& c, const ClassPlan&, int, int) { return c.bredc; }
bool FusedApplies(const ClassDev& c, const ClassPlan& plan, int k, int64_t)
{
    return c.nqueues > 0 && plan.qcut >= 0 && k >= 8 && k <= 16;
}
void LaunchFillZero(void* p, int64_t n, hipStream_t) { Live(p, (double)n, "fill"); }
void LaunchFillZeroRows(void* p, int64_t n, int rows, int64_t stride, hipStream_t)
{
    if (rows > 0) Live(p, (double)stride * (rows - 1) + n, "fill rows");
}

template <typename T>
static double Eb(const ClassDev& c)
{
    return (double)sizeof(cx<T>) * c.npanels;
}
template <typename T>
static void Factors(const ClassDev& c, bool u)
{
    Live(c.L, Eb<T>(c) * c.fstore, "L");
    if (u) Live(c.U, Eb<T>(c) * c.ustore, "U");
}
template <typename T>
void LaunchScatterOrig(const ClassDev& c, const StencilArgs&, const double*, double, hipStream_t)
{
    ++factorizations;
    if (slow) std::this_thread::sleep_for(std::chrono::milliseconds(50));
    Factors<T>(c, true);
    Live(c.T, Eb<T>(c) * c.tstore, "T");
    Live(c.F, Eb<T>(c) * c.fentries, "F");
}
template <typename T>
void LaunchExtendAdd(const ClassDev& c, int, int, hipStream_t) { Factors<T>(c, true); }
template <typename T>
void LaunchLdlDiag(const ClassDev& c, int, int, int, hipStream_t) { Factors<T>(c, false); }
template <typename T>
void LaunchLdlTrsm(const ClassDev& c, int, int, int, hipStream_t) { Factors<T>(c, false); }
template <typename T>
void LaunchGemm(const ClassDev& c, int, int n, hipStream_t)
{
    if (n > 0) Factors<T>(c, true);
}
template <typename T>
void LaunchInvDiag(const ClassDev& c, int, hipStream_t) { Factors<T>(c, false); }
template <typename T>
void LaunchPack(const ClassDev& c, int, int, hipStream_t)
{
    Factors<T>(c, true);
    Live(c.F, Eb<T>(c) * c.fentries, "F");
}
template <typename T>
void LaunchCompose(const ClassDev& c, int, int, hipStream_t)
{
    Live(c.U, Eb<T>(c) * c.ustore, "E");
    Live(c.F, Eb<T>(c) * c.fentries, "F");
}
template <typename T>
void LaunchTransposeScale(const ClassDev& c, hipStream_t)
{
    Factors<T>(c, false);
    Live(c.LT, Eb<T>(c) * c.fstore, "LT");
}
template <typename T>
void LaunchFoldBack(const ClassDev& c, hipStream_t s) { LaunchTransposeScale<T>(c, s); }
template <typename T>
void LaunchPanelSolve(const ClassDev& c, const ClassPlan& plan, int b, void* V, void* P, int k,
                      hipStream_t, MvProfile*, int, int)
{
    ++merged;
    need(b >= 0 && b < c.npanels, "panel", b);
    Live(c.F, Eb<T>(c) * c.fentries, "F");
    Live(V, sizeof(cx<T>) * (double)VecRows(plan).total * k, "solve vector");
    Live(P, sizeof(cx<T>) * 64.0 * plan.bslots * k, "partial sums");
}
template <typename T>
void LaunchPanelSolveFused(const ClassDev& c, const ClassPlan& plan, int b, void* Xp, void* W,
                           void* P, void* G, int k, hipStream_t, MvProfile*, int32_t* sync)
{
    ++fusedSolves;
    need(b >= 0 && b < c.npanels, "panel", b);
    Factors<T>(c, false);
    Live(c.LT, Eb<T>(c) * c.fstore, "LT");
    const double e = sizeof(cx<T>) * (double)k, pad = kSolvePad + 2;
    Live(Xp, e * (c.n + pad), "panel vector");
    Live(W, e * (c.wstore + pad), "work vectors");
    Live(G, e * (2 * c.wstore + pad), "slot copies");
    Live(P, e * 64 * plan.maxSlots, "partial sums");
    Live(sync, 4.0 * c.nsync, "fused state");
}
template <typename T>
void LaunchCopyIn(const PanelMap& m, const c128*, void* X, int k, int, int, int, int, int,
                  hipStream_t, int32_t*, int)
{
    Live(X, sizeof(cx<T>) * (double)m.n * k, "copy in");
}
template <typename T>
void LaunchCopyOut(const PanelMap& m, c128*, const void* X, int k, int, int, int, int, int, int,
                   hipStream_t, const StencilArgs*, const double*, int)
{
    Live(X, sizeof(cx<T>) * (double)m.n * k, "copy out");
}
template <typename T>
void LaunchPassOn(const StencilArgs&, const double*, c128*, int, const PassPanel& o, const PassPanel& i,
                  int, int, hipStream_t)
{
    ++couplings;
    Live(o.X, 1, "pass out");
    Live(i.X, 1, "pass in");
}
template <typename T>
void LaunchZeroSetPlane(const PanelMap& m, const StencilArgs&, const double*, const c128*, void* X,
                        int k, int, int, hipStream_t, int32_t*, int)
{
    Live(X, sizeof(cx<T>) * (double)m.n * k, "zero set");
}
template <typename T>
void LaunchSolveBatch(int, int, const BatchBlock*, int, const BatchSolveSeg*, const int32_t*, hipStream_t) {}
template <typename T>
void LaunchReduceBatch(int, const BatchBlock*, int, const BatchSolveSeg*, const int32_t*, hipStream_t) {}
template <typename T>
void LaunchCopyBatch(int, const BatchBlock*, int, const BatchCopySeg*, const int32_t*, hipStream_t) {}
void LaunchSpmv(const StencilArgs&, const double*, const c128*, const c128*, c128*, int, int, hipStream_t) {}
void LaunchArnoldi(const c128*, int, int, c128*, int64_t, int, c128*, c128*, double*, c128*, double*, hipStream_t) {}
void LaunchColNorm2(const c128*, int64_t, int, double*, double*, hipStream_t) {}
void LaunchScaleCols(const double*, const c128*, c128*, int64_t, int, hipStream_t) {}
void LaunchUpdateX(const c128*, const c128*, const c128*, int, int64_t, int, c128*, hipStream_t) {}
void LaunchAdjointGrad(const StencilArgs&, const c128*, const c128*, int, double*, int, hipStream_t) {}

#define BOTH(f, ...)                 \
    template void f<float>(__VA_ARGS__); \
    template void f<double>(__VA_ARGS__);
BOTH(LaunchScatterOrig, const ClassDev&, const StencilArgs&, const double*, double, hipStream_t)
BOTH(LaunchExtendAdd, const ClassDev&, int, int, hipStream_t)
BOTH(LaunchLdlDiag, const ClassDev&, int, int, int, hipStream_t)
BOTH(LaunchLdlTrsm, const ClassDev&, int, int, int, hipStream_t)
BOTH(LaunchGemm, const ClassDev&, int, int, hipStream_t)
BOTH(LaunchInvDiag, const ClassDev&, int, hipStream_t)
BOTH(LaunchPack, const ClassDev&, int, int, hipStream_t)
BOTH(LaunchCompose, const ClassDev&, int, int, hipStream_t)
BOTH(LaunchTransposeScale, const ClassDev&, hipStream_t)
BOTH(LaunchFoldBack, const ClassDev&, hipStream_t)
BOTH(LaunchPanelSolve, const ClassDev&, const ClassPlan&, int, void*, void*, int, hipStream_t, MvProfile*, int, int)
BOTH(LaunchPanelSolveFused, const ClassDev&, const ClassPlan&, int, void*, void*, void*, void*, int,
     hipStream_t, MvProfile*, int32_t*)
BOTH(LaunchCopyIn, const PanelMap&, const c128*, void*, int, int, int, int, int, int, hipStream_t, int32_t*, int)
BOTH(LaunchCopyOut, const PanelMap&, c128*, const void*, int, int, int, int, int, int, int, hipStream_t,
     const StencilArgs*, const double*, int)
BOTH(LaunchPassOn, const StencilArgs&, const double*, c128*, int, const PassPanel&, const PassPanel&, int, int,
     hipStream_t)
BOTH(LaunchZeroSetPlane, const PanelMap&, const StencilArgs&, const double*, const c128*, void*, int, int, int,
     hipStream_t, int32_t*, int)
BOTH(LaunchSolveBatch, int, int, const BatchBlock*, int, const BatchSolveSeg*, const int32_t*, hipStream_t)
BOTH(LaunchReduceBatch, int, const BatchBlock*, int, const BatchSolveSeg*, const int32_t*, hipStream_t)
BOTH(LaunchCopyBatch, int, const BatchBlock*, int, const BatchCopySeg*, const int32_t*, hipStream_t)
}  // namespace psp_amd

// ---- the checks ------------------------------------------------------------------
static psp_hip_desc desc;
static std::vector<double> vel;
static std::vector<std::complex<double>> block;

static psp_hip_ctx* Context()
{
    psp_hip_ctx* c = nullptr;
    if (psp_hip_create(&desc, &c) != PSP_HIP_OK) std::exit(2);
    return c;
}

static int Factor(psp_hip_ctx* c) { return psp_hip_factor(c, vel.data(), PSP_HIP_LDL_SELINV_1D, nullptr); }

struct Counts {
    long f, m, q, a, r;
};
// what one call does: factorizations, merged and fused panel solves,
// allocations and frees
template <class F>
static Counts Of(const char* what, psp_hip_ctx* c, const F& call)
{
    const Counts t{factorizations, merged, fusedSolves, allocs, frees};
    const int st = call();
    need(st == PSP_HIP_OK, what, st);
    if (st) std::fprintf(stderr, "  %s\n", psp_hip_last_error(c));
    return {factorizations - t.f, merged - t.m, fusedSolves - t.q, allocs - t.a, frees - t.r};
}

static void fused()
{
    psp_hip_ctx* c = Context();
    need(Factor(c) == PSP_HIP_OK, "Initialize");
    const int solves = 2 * psp_hip_num_panels(c) - 1;
    const long once = factorizations;
    psp_hip_set_option(c, PSP_HIP_OPT_SOLVE_FUSED, 1);
    void* B = block.data();
    Counts n = Of("noalloc", c, [&] { return psp_hip_precondition_noalloc(c, B, 8); });
    need(n.f == 0 && n.a == 0 && n.r == 0 && n.m == solves && n.q == 0, "noalloc", n.f, n.a);
    n = Of("Multiply", c, [&] { return psp_hip_multiply(c, B, B, 8); });
    need(n.f == 0 && n.a == 0, "Multiply", n.f, n.a);
    n = Of("gradient", c, [&] { return psp_hip_adjoint_gradient(c, B, B, 8, vel.data(), 0); });
    need(n.f == 0 && n.a == 0, "gradient", n.f, n.a);
    for (int k : {3, 7, 17}) {  // the fused launches take 8 to 16
        n = Of("sweep", c, [&] { return psp_hip_precondition(c, B, k); });
        need(n.f == 0 && n.m == solves && n.q == 0, "sweep without fused launches", n.f, n.q);
    }
    n = Of("first fused sweep", c, [&] { return psp_hip_precondition(c, B, 8); });
    need(n.f == once && n.q > 0, "factors in the fused layout", n.f, n.q);
    n = Of("fused sweep", c, [&] { return psp_hip_precondition(c, B, 12); });
    need(n.f == 0 && n.q > 0, "kept", n.f, n.q);
    n = Of("noalloc", c, [&] { return psp_hip_precondition_noalloc(c, B, 8); });
    need(n.f == 0 && n.a == 0 && n.r == 0 && n.q > 0, "noalloc, fused", n.a, n.q);
    psp_hip_destroy(c);
}

static void oom()
{
    // (the workspace's are smaller without slices)
    const size_t big = block.size() * sizeof(block[0]) * (desc.precision ? 1 : 2);
    for (int n = 0;; ++n) {
        psp_hip_ctx* c = Context();
        psp_hip_set_option(c, PSP_HIP_OPT_SOLVE_MAX_SPLIT, 1);
        psp_hip_set_option(c, PSP_HIP_OPT_SOLVE_MIN_TILES, 1);
        psp_hip_set_option(c, PSP_HIP_OPT_SWEEP_GRAPH, 0);
        need(Factor(c) == PSP_HIP_OK, "Initialize");
        const int solves = 2 * psp_hip_num_panels(c) - 1;
        const size_t resident = used;
        psp_hip_set_option(c, PSP_HIP_OPT_SOLVE_FUSED, 1);
        void* B = block.data();
        smallest = big;
        failAt = n;
        Counts t = Of("panel solve", c, [&] { return psp_hip_solve_panel(c, B, 9, 1); });
        const bool short_ = failed;
        failed = false;
        failAt = -1;
        smallest = 0;
        if (short_) {
            need(t.f == 0 && t.m == 1 && t.q == 0, "merged solves serve", n, t.f);
            t = Of("noalloc", c, [&] { return psp_hip_precondition_noalloc(c, B, 8); });
            need(t.f == 0 && t.m == solves, "noalloc", n);
            t = Of("Multiply", c, [&] { return psp_hip_multiply(c, B, B, 9); });
            psp_hip_set_option(c, PSP_HIP_OPT_SOLVE_FUSED, 0);  // frees the workspace
            need(used <= resident, "memory given back", n, (long)(used - resident));
            psp_hip_set_option(c, PSP_HIP_OPT_SOLVE_FUSED, 1);
        }
        t = Of("sweep", c, [&] { return psp_hip_precondition(c, B, 9); });
        need((t.f > 0) == short_ && t.q > 0, "fused solves with the memory back", n, t.f);
        psp_hip_destroy(c);
        if (!short_) break;
        need(n < 20, "big allocations");
    }
}

static void retry()
{
    for (int n = 0;; ++n) {
        psp_hip_ctx* c = Context();
        failAt = n;
        const int st = Factor(c);
        const bool short_ = failed;
        failed = false;
        failAt = -1;
        need(st == (short_ ? PSP_HIP_ERR_MEMORY : PSP_HIP_OK), "Initialize", n, st);
        if (short_) need(Factor(c) == PSP_HIP_OK, "Initialize again", n);
        Of("sweep", c, [&] { return psp_hip_precondition(c, block.data(), 8); });
        psp_hip_destroy(c);
        need(used == 0, "given back", n, (long)used);
        if (!short_) break;
    }
}

// Bytes of the factors of all panels as two plain copies, and of the scratch of
// their updates and inverses.
static void plainSizes(double* factors, double* scratch, double* folded)
{
    Plan plan;
    std::string msg;
    if (BuildPlan(desc, plan, msg) != PSP_HIP_OK) std::exit(2);
    const double eb = desc.precision == PSP_HIP_FRONTS_FP32 ? 8 : 16;
    *factors = *scratch = *folded = 0;
    std::vector<int> panels(3, 0);
    for (int p = 0; p < plan.geo.numPanels; ++p) ++panels[plan.geo.cls(p)];
    for (int cl = 0; cl < 3; ++cl) {
        if (!plan.present[cl]) continue;
        const ClassPlan& C = plan.cls[cl];
        *factors += 2 * eb * panels[cl] * C.fstore;
        *scratch += eb * panels[cl] * (C.ustore + C.tstore);
        *folded += eb * panels[cl] * 256.0 * (C.nblocks + 1);
        // the pieces of a depth group's E do not overlap
        for (const auto& g : C.groups) {
            std::vector<std::pair<int64_t, int64_t>> e;
            for (size_t t = 0; t < C.nodes.size(); ++t)
                if (C.nodes[t].depth >= g[0] && C.nodes[t].depth <= g[1] && C.nodes[t].size > 0)
                    e.push_back({C.foldNodes[t].e, (int64_t)C.nodes[t].size * C.nodes[t].usize});
            std::sort(e.begin(), e.end());
            for (size_t i = 0; i < e.size(); ++i)
                need(e[i].first + e[i].second <= (i + 1 < e.size() ? e[i + 1].first : C.estore),
                     "E", cl, (long)i);
        }
    }
}

static void memory()
{
    double factors, scratch, folded;
    plainSizes(&factors, &scratch, &folded);
    psp_hip_ctx* c = Context();
    need(Factor(c) == PSP_HIP_OK && Factor(c) == PSP_HIP_OK, "Initialize");
    const double peak = (double)most;
    psp_hip_finalize(c);
    const double plan = (double)used;
    std::printf("GB: at most %.2f, as plain copies %.2f\n", (peak - plan) / 1e9, (factors + scratch) / 1e9);
    need(peak - plan <= factors + scratch, "memory of Initialize");
    psp_hip_destroy(c);
    need(used == 0, "given back", (long)used);
}

// Contexts with factors at the same time, one after another and on threads.
static void several()
{
    double factors, scratch, folded;
    plainSizes(&factors, &scratch, &folded);
    const double slack = 1 << 16;
    psp_hip_ctx* c[3] = {Context(), Context(), Context()};
    need(Factor(c[0]) == PSP_HIP_OK, "Initialize");
    psp_hip_finalize(c[0]);
    const double plan = (double)used;
    for (psp_hip_ctx* x : c) need(Factor(x) == PSP_HIP_OK, "Initialize");
    need(used <= 3 * (plan + folded) + factors / 2 + slack, "one L", (long)used);
    // an allocation that needs L's memory gets it
    capacity = used;
    Of("sweep", c[1], [&] { return psp_hip_precondition(c[1], block.data(), 8); });
    need(failed && used <= 3 * (plan + folded) + factors / 4, "memory of L", (long)used);
    capacity = (size_t)-1;
    failed = false;
    need(Factor(c[2]) == PSP_HIP_OK, "Initialize again");
    for (psp_hip_ctx* x : c) psp_hip_finalize(x);
    need(used <= 3 * plan + slack, "given back", (long)used);
    slow = true;
    std::vector<std::thread> threads;
    for (psp_hip_ctx* x : c) threads.emplace_back([x] { need(Factor(x) == PSP_HIP_OK, "Initialize"); });
    for (std::thread& t : threads) t.join();
    need(used <= 3 * (plan + folded) + factors / 2 + slack, "scratch of threads", (long)used);
    for (psp_hip_ctx* x : c) psp_hip_destroy(x);
    need(used == 0, "given back", (long)used);
}

int main(int argc, char** argv)
{
    if (argc < 5) return 2;
    desc.nx = std::atoi(argv[2]);
    desc.ny = std::atoi(argv[3]);
    desc.nz = std::atoi(argv[4]);
    desc.precision = argc > 5 ? std::atoi(argv[5]) : 0;
    const double h = 1.0 / (std::max(desc.nx, std::max(desc.ny, desc.nz)) + 1);
    desc.wx = (desc.nx + 1) * h;
    desc.wy = (desc.ny + 1) * h;
    desc.wz = (desc.nz + 1) * h;
    desc.omega = 30.0;
    desc.bx = desc.by = desc.bz = 5;
    desc.sigmax = desc.sigmay = desc.sigmaz = 1.5;
    desc.damping = 7.0;
    desc.planesPerPanel = 4;
    desc.cutoff = 12;
    const size_t N = (size_t)desc.nx * desc.ny * desc.nz;
    vel.assign(N, 2.0);
    block.assign(N * 32, {1.0, 0.0});
    const std::string mode = argv[1];
    if (mode == "fused")
        fused();
    else if (mode == "oom")
        oom();
    else if (mode == "retry")
        retry();
    else if (mode == "memory")
        memory();
    else if (mode == "several")
        several();
    else
        return 2;
    std::printf("%s: %ld allocations, %ld factorizations\n", mode.c_str(), allocs,
                factorizations.load());
    return fails ? 1 : 0;
}
