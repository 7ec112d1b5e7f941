// Host stand-in for the HIP runtime and the kernel launchers, linked with the library's host sources
// so that tests can see what the host runtime does without a GPU: device memory is host memory
// counted against a capacity, with a limit on one block; launches succeed, do nothing and leave
// their arguments behind.  The time between two events is the waves of the sweeps launched in
// between, so a traversal with fewer waves is a faster one.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>

#include "gpe_internal.h"

using namespace gpe;

namespace {

struct Counts {
    long long allocs, host_allocs, copies, used, waves;
} g_n;
long long g_capacity = 1ll << 40, g_max_block = 1ll << 40;
std::map<void *, size_t> &g_blocks = *new std::map<void *, size_t>;
SweepArgs g_sweep;
ObsArgs g_obs;
int g_obs_blocks = 1024;

hipError_t take(void **p, size_t n)
{
    if ((long long)n > g_max_block || g_n.used + (long long)n > g_capacity) return hipErrorOutOfMemory;
    *p = calloc(1, n ? n : 1);
    g_blocks[*p] = n;
    g_n.used += (long long)n;
    g_n.allocs += 1;
    return hipSuccess;
}

hipError_t give(void *p)
{
    if (!p) return hipSuccess;
    const auto it = g_blocks.find(p);
    if (it == g_blocks.end()) abort();  // freed twice, or never allocated
    g_n.used -= (long long)it->second;
    g_blocks.erase(it);
    free(p);
    return hipSuccess;
}

}  // namespace

extern "C" {

// what the tests see
void stand_in_limits(long long capacity, long long max_block) { g_capacity = capacity, g_max_block = max_block; }
void stand_in_counts(long long out[5]) { memcpy(out, &g_n, sizeof g_n); }
// waves and workgroups of the last reduction, its segments a chunk, chunks a wave and launched workgroups
void stand_in_reduction(long long out[12])
{
    const Geometry &g = g_obs.g;
    const long long v[12] = {g.nx, g.ny, g.nz, g.V, g.ty, g.rows, g.nseg, g.waves, g.ntile, g_obs.segs, g_obs.per, g_obs.blocks};
    memcpy(out, v, sizeof v);
}
void stand_in_resident(int blocks) { g_obs_blocks = blocks; }
// rows, x per lane, tile rows, waves and exchange of the last sweep
void stand_in_sweep(long long out[5])
{
    const Geometry &g = g_sweep.g;
    const long long v[5] = {g.rows, g.xpl, g.ty, g.waves, g.exchange};
    memcpy(out, v, sizeof v);
}

hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return take(p, n); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipFreeAsync(void *p, hipStream_t) { return give(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    g_n.host_allocs += 1;
    return (*p = calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *avail, size_t *total)
{
    *avail = (size_t)(g_capacity - g_n.used), *total = (size_t)g_capacity;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    g_n.copies += 1;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }

hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = (hipEvent_t)calloc(1, sizeof(long long));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    *(long long *)e = g_n.waves;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)(*(long long *)b - *(long long *)a);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = (hipStream_t)malloc(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

int gpe_get_state_noalloc(gpe_ctx *, int, double *) { return GPE_EDEVICE; }

}  // extern "C"

namespace gpe {

hipError_t launch_sweep(int, int, int, const SweepArgs &a, hipStream_t)
{
    g_sweep = a;
    g_n.waves += a.g.waves;
    return hipSuccess;
}
hipError_t launch_observables(int, int, const ObsArgs &a, hipStream_t)
{
    g_obs = a;
    return hipSuccess;
}
hipError_t observables_resident(int, int, int, int *blocks)
{
    *blocks = g_obs_blocks;
    return hipSuccess;
}
hipError_t launch_adjoint(int, int, const AdjArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_advance_base(int *, int, hipStream_t) { return hipSuccess; }
hipError_t launch_set_base(int *, int, hipStream_t) { return hipSuccess; }
hipError_t launch_aux(int, int, const AuxArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_ensemble_sweep(int, int, int, int, const EnsembleArgs &, int, hipStream_t) { return hipSuccess; }
hipError_t launch_fill_tf(int, const Geometry &, const Tables &, const Physics &, int, const FillArgs &, void *, hipStream_t)
{
    return hipSuccess;
}
hipError_t launch_finalize(const double *, int, int, int, double *, double *, hipStream_t) { return hipSuccess; }
hipError_t launch_finalize_few(const double *, int, int, int, double *, double *, hipStream_t) { return hipSuccess; }
hipError_t launch_local_fields(int, int, const Geometry &, const Tables &, const void *, int, double *, hipStream_t)
{
    return hipSuccess;
}
hipError_t launch_noise(int, int, const Geometry &, const Tables &, void *, double, unsigned long long, hipStream_t)
{
    return hipSuccess;
}
hipError_t launch_norm(int, int, const NormArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_norm_scale(const double *, int, double, double *, double *, hipStream_t) { return hipSuccess; }
hipError_t launch_objective(int, int, const ObjArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_pack(int, const Geometry &, const Tables &, int, const double *, void *, hipStream_t) { return hipSuccess; }
hipError_t launch_unpack(int, const Geometry &, const Tables &, int, const void *, double *, hipStream_t) { return hipSuccess; }
hipError_t launch_phase_copy(int, const void *, void *, long long, double, double, hipStream_t) { return hipSuccess; }
hipError_t launch_project(int, int, const Geometry &, void *, int, double, hipStream_t) { return hipSuccess; }
hipError_t launch_scale(int, void *, long long, double, const double *, hipStream_t) { return hipSuccess; }
hipError_t launch_stream(int, const void *, void *, long long, hipStream_t) { return hipSuccess; }
hipError_t launch_sum_tables(const double *, int, int, int, double *, long long, hipStream_t) { return hipSuccess; }

}  // namespace gpe
