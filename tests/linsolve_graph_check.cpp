// LinSolver's kept graphs.  They are built for a system that comes again or takes long.  After a failed build the solver reports the failure, holds nothing of it, and the next
// system replays graphs of its own size only; and the form of an iteration (two launches or five) follows the rows and non-zeros of each system, whatever
// was solved before on the same arrays.  The HIP calls that ls_solve_device makes are stand-ins: a graph is a
// record of its first kernel argument (the system's size) and its launches, and one chosen call fails.
#include "../shiokaze_amd/csrc/shkz_linsolve.hip"
#include "host_hip.hpp"

#include <cstdio>

int shkz_set_error(int code, const char *) { return code; }

namespace {
struct Graph {
    int n = 0, nodes = 0;
};
int live_execs = 0, wrong_launches = 0, launches = 0, want_n = 0, polls = 0, nnz = 0, chunks = 2, builds_done = 0, direct = 0;
int calls_left = -1;  // the call that fails (counted over the building calls), -1: none
bool fails() { return calls_left >= 0 && calls_left-- == 0; }
}  // namespace

extern "C" {
hipError_t hipGraphCreate(hipGraph_t *g, unsigned) {
    if (fails()) return hipErrorOutOfMemory;
    *g = (hipGraph_t) new Graph;
    return hipSuccess;
}
hipError_t hipGraphAddKernelNode(hipGraphNode_t *node, hipGraph_t g, const hipGraphNode_t *, size_t,
                                 const hipKernelNodeParams *p) {
    if (fails()) return hipErrorOutOfMemory;
    const int n = *(const int *)p->kernelParams[0];
    if (!((Graph *)g)->n) ((Graph *)g)->n = n;
    ++((Graph *)g)->nodes;
    *node = (hipGraphNode_t)g;
    return hipSuccess;
}
hipError_t hipGraphInstantiateWithFlags(hipGraphExec_t *e, hipGraph_t g, unsigned long long) {
    if (fails()) return hipErrorOutOfMemory;
    *e = (hipGraphExec_t) new Graph(*(Graph *)g);
    ++live_execs;
    ++builds_done;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    delete (Graph *)g;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    if (!e) return hipErrorInvalidValue;
    delete (Graph *)e;
    --live_execs;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    ++launches;
    wrong_launches += !e || ((Graph *)e)->n != want_n;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *, size_t, hipMemcpyKind, hipStream_t) {
    auto *s = (LsScalars *)dst;
    std::memset(s, 0, sizeof(*s));
    s->maxit = 1000;
    s->nnz = nnz;
    s->done = polls >= chunks;
    s->iter = LS_BUILD_AFTER * polls++;  // the second chunk: replayed, and long enough for the longer graph
    s->r0 = 1.0;
    s->rinf = 0.9;
    s->tol = 1e-6;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
    ++direct;
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
}

static int solve(shkz_linsolver &L, int n) {
    static double memory[1 << 12];
    const LsArrays D{(const int *)memory, (const int *)memory + 1, memory, memory, memory + 100, memory + 200, memory + 300,
                     memory + 400, memory + 500, memory + 600, memory + 700, memory + 800, memory + 900,
                     (LsScalars *)(memory + 1000)};
    shkz_linsolve_params prm;
    shkz_linsolve_default_params(&prm);
    shkz_linsolve_result res;
    polls = 0;
    want_n = n;
    return ls_solve_device(&L, nullptr, D, n, &prm, &res, true);
}

static int after_failed_builds() {
    int bad = 0, builds = 0;
    for (int n : {100, LS_FOLD_ROWS + 100}) {  // both forms of an iteration
        for (int fail_at = 0;; ++fail_at) {
            shkz_linsolver L;
            LsScalars host;
            L.host_s = &host;
            launches = wrong_launches = live_execs = 0;
            const int first = solve(L, n);
            calls_left = fail_at;
            const int other = solve(L, n - 1);
            const bool failed = calls_left < 0;
            calls_left = -1;
            if (!failed) break;  // fewer building calls than that
            ++builds;
            const int held = live_execs;
            const int again = solve(L, n);
            if (first != SHKZ_OK || other != SHKZ_ERR_DEVICE || held != 0 || again != SHKZ_OK || live_execs != 2 ||
                wrong_launches || !launches || L.built.n != n) {
                ++bad;
                std::printf("n=%d, failure at call %d: %d %d %d, held %d, live %d, %d of %d launches of another graph\n", n, fail_at,
                            first, other, again, held, live_execs, wrong_launches, launches);
            }
        }
    }
    std::printf("%d failed builds, %d went wrong\n", builds, bad);
    if (!bad && builds > 4) std::printf("OK\n");
    return bad;
}

static int forms() {
    int bad = 0;
    // the form: four launches for two iterations, or five for one
    shkz_linsolver L;
    LsScalars host;
    L.host_s = &host;
    const int rows = 1000, most = LS_FOLD_ROWS;
    const struct {
        int n, nnz, nodes;
    } systems[] = {{rows, 7 * rows, 4},  {rows, 640 * rows, 4},     {rows, 640 * rows + 1, 5}, {rows, 7 * rows, 4},
                   {most, 7 * most, 4},  {most, 10 << 20, 4},       {most, (10 << 20) + 1, 5},  {most + 1, 7 * most, 5},
                   {1, 1, 4},            {most, 2147483647, 5}};
    for (const auto &x : systems) {
        nnz = x.nnz;
        wrong_launches = 0;
        const int rc = solve(L, x.n);
        const int nodes = L.exec ? ((Graph *)L.exec)->nodes : 0, longer = L.exec_many ? ((Graph *)L.exec_many)->nodes : 0;
        if (rc != SHKZ_OK || wrong_launches || nodes != x.nodes || longer != 8 * x.nodes) {
            ++bad;
            std::printf("n=%d with %d non-zeros: %d, graphs of %d and %d launches\n", x.n, x.nnz, rc, nodes, longer);
        }
    }
    if (!bad) std::printf("OK\n");
    return bad;
}

// Systems that converge within the first chunk: launched directly at first sight, replayed when they come again.
static int short_solves() {
    int bad = 0;
    chunks = 1;
    shkz_linsolver L;
    LsScalars host;
    L.host_s = &host;
    const struct {
        int n;
        bool replayed, built;
    } solves[] = {{100, false, false}, {100, true, true},  {100, true, false}, {99, false, false}, {100, true, false},
                  {99, false, false},  {99, true, true},   {99, true, false},  {100, false, false}, {100, true, true},
                  {LS_FOLD_ROWS + 5, false, false}, {LS_FOLD_ROWS + 5, true, true}};
    for (const auto &x : solves) {
        launches = wrong_launches = builds_done = direct = 0;
        const int rc = solve(L, x.n);
        const bool by_launches = direct > 8;  // (the set-up is launched in any case)
        if (rc != SHKZ_OK || wrong_launches || (launches > 0) != x.replayed || by_launches == x.replayed ||
            builds_done != (x.built ? 2 : 0)) {
            ++bad;
            std::printf("n=%d: %d, %d replays (%d wrong), %d launches, %d graphs built\n", x.n, rc, launches, wrong_launches, direct,
                        builds_done);
        }
    }
    if (!bad) std::printf("OK\n");
    return bad;
}

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    return what == "form" ? forms() : what == "short" ? short_solves() : after_failed_builds();
}
