// Host runtime of libgpe: contexts, device memory, lattice tables, field ramps and the
// sweep loop behind the C ABI declared in include/gpe.h.
#include "gpe.h"
#include "gpe_internal.h"
#include "lattice_tables.h"

#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <cstdio>
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <string>
#include <tuple>
#include <vector>

using namespace gpe;

namespace {

struct Ramp {
    std::vector<double> q_val, q_dur, b_val, b_dur;
    std::vector<int> q_type, b_type;
    double tau = 1.0, time_scale = 1.0;
    double scale_q = 1.0, scale_b = 1.0, qscale_q = 0.0, qscale_b = 0.0;
    bool active = false;
};

// One channel of the piecewise ramp (getSignal, Spin1GpeBCC/AliceRingRamps.h:80-138).
void ramp_channel(const std::vector<double> &val, const std::vector<double> &dur, const std::vector<int> &type,
                  int width, double tau, double t, double *out)
{
    const int n = (int)dur.size();
    if (n == 0) {
        for (int k = 0; k < width; ++k) out[k] = 0.0;
        return;
    }
    int idx = 0;
    for (; idx < n; ++idx) {
        const double tin = t - dur[idx];
        if (tin < 0) break;
        t = tin;
    }
    if (idx >= n) {
        for (int k = 0; k < width; ++k) out[k] = val[(n - 1) * width + k];
        return;
    }
    for (int k = 0; k < width; ++k) {
        const double prev = idx > 0 ? val[(idx - 1) * width + k] : 0.0;
        const double cur = val[idx * width + k];
        switch (type[idx]) {
        case 1: out[k] = prev + t * (cur - prev) / dur[idx]; break;
        case 2: out[k] = prev + (cur - prev) * std::sqrt(t / dur[idx]); break;
        case 3: out[k] = prev + (cur - prev) * (1.0 - std::exp(-t / tau)); break;
        default: out[k] = cur; break;
        }
    }
}

}  // namespace

// Device memory a context keeps between calls that need a lot of it (the adjoint's levels): the
// driver clears what is freed, so freeing and allocating gigabytes on every call costs from
// nothing to seconds (4.6 GB in one block: 134 ms a call once the first few have gone through; in
// blocks of 75 MB 17 ms; 18 GB up to 5 s), the kernels of a 200-sweep call on spin-1 BCC 64^3 25 ms.
// Idle workspaces are given back when an allocation of the library fails, when less than half of
// the device would stay free, and with their context.
struct Workspace {
    void *p = nullptr;
    size_t bytes = 0;
    int device = 0;
    bool busy = false;
    std::vector<void *> loose;  // buffers of the current call where one block for all does not fit
};

struct gpe_ctx {
    Workspace ws;    // guarded by g_ws_mutex
    gpe_config cfg{};
    const LatticeTable *lat = nullptr;
    Geometry g{};    // one x per lane: observables, packing, adjoint
    Geometry gs{};   // the sweep's geometry (1 or 2 x per lane)
    Geometry gr{};   // the reductions' geometry (one x per lane over row groups)
    int gr_segs = 1;    // 64-slot segments of a row group that a wave of it takes
    int red_blocks = 1; // workgroups of a reduction: as many as run at once
    Physics ph{};
    int fp64 = 0;
    size_t elem_bytes = 0;   // bytes of one complex element
    long long level_elems = 0;
    hipStream_t stream = nullptr;
    hipStream_t copy_stream = nullptr;  // uploads beside the sweeps (adjoint target), made on first use
    int device = 0;
    void *level[2] = {nullptr, nullptr};
    // tables: one block, which d_scalars and d_red share
    char *d_tables = nullptr;
    int *d_abi = nullptr, *d_nface = nullptr, *d_facex = nullptr;  // d_abi: V places, then their inverse
    int *d_oface = nullptr, *d_nfwd = nullptr;  // the observables' faces (ObsArgs)
    double *d_ow = nullptr;
    float *d_w32 = nullptr, *d_wsum32 = nullptr, *d_pos32 = nullptr;
    double *d_w64 = nullptr, *d_wsum64 = nullptr, *d_pos64 = nullptr, *d_dv = nullptr;
    // fields per sweep (the adjoint's; made on first use)
    FieldRec *d_fields = nullptr;
    int fields_cap = 0;
    FieldRec *h_fields = nullptr;  // pinned staging
    // reductions
    double *d_partials = nullptr;
    double *d_scalars = nullptr;   // [0..15] results / scales
    double *d_red = nullptr;       // FIN_SCRATCH doubles: first-stage results of launch_finalize
    double *h_red = nullptr;       // pinned: results the host reads (FIN_WIDTH_MAX doubles)
    // static field and ramp
    double bq = 0, bb[3] = {0, 0, 0}, bqq = 0, bbq[3] = {0, 0, 0};
    Ramp ramp;
    // time bookkeeping
    double t0 = 0.0;
    long long sweeps = 0;
    bool level1_valid = false;
    // timing
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_ms_per_sweep = 0.0;
    std::string err;
};

namespace {

int fail(gpe_ctx *c, int code, const char *what)
{
    if (c) c->err = what;
    return code;
}

int hip_fail(gpe_ctx *c, hipError_t e, const char *where)
{
    if (c) {
        c->err = std::string(where) + ": " + hipGetErrorString(e);
    }
    return GPE_EDEVICE;
}

#define HIPCALL(ctx, call)                                     \
    do {                                                       \
        hipError_t e_ = (call);                                \
        if (e_ != hipSuccess) return hip_fail(ctx, e_, #call); \
    } while (0)

std::mutex &g_ws_mutex = *new std::mutex;  // never destroyed: a context may outlive static objects
std::set<Workspace *> &g_workspaces = *new std::set<Workspace *>;  // those that hold memory

void drop_workspace(Workspace *w)  // with g_ws_mutex held
{
    if (!w->p) return;
    (void)hipFree(w->p);
    w->p = nullptr;
    w->bytes = 0;
    g_workspaces.erase(w);
}

void drop_loose(Workspace *w)  // the context's own call
{
    for (void *p : w->loose) (void)hipFree(p);
    w->loose.clear();
}

// Give back the device's idle workspaces; whether there were any.
bool drop_idle_workspaces(int device)
{
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    bool any = false;
    for (auto it = g_workspaces.begin(); it != g_workspaces.end();) {
        Workspace *w = *it++;
        if (w->busy || w->device != device) continue;
        drop_workspace(w);
        any = true;
    }
    return any;
}

// The library's device memory: hipMalloc (hipMallocAsync with a stream); where that fails, again
// after the device's idle workspaces are given back.
hipError_t device_malloc(void **out, size_t bytes, int device)
{
    const hipError_t e = hipMalloc(out, bytes);
    if (e == hipSuccess || !drop_idle_workspaces(device)) return e;
    (void)hipGetLastError();
    return hipMalloc(out, bytes);
}

hipError_t device_malloc(void **out, size_t bytes, int device, hipStream_t stream)
{
    const hipError_t e = hipMallocAsync(out, bytes, stream);
    if (e == hipSuccess || !drop_idle_workspaces(device)) return e;
    (void)hipGetLastError();
    return hipMallocAsync(out, bytes, stream);
}

// Buffers of these sizes from the context's workspace, until end_workspace: one block, or where that
// does not fit (one allocation has to be contiguous and below the driver's limit) each on its own.
hipError_t begin_workspace(gpe_ctx *c, const std::vector<size_t> &sizes, std::vector<void *> &out)
{
    Workspace &w = c->ws;
    size_t bytes = 0;
    for (size_t n : sizes) bytes += (n + 255) / 256 * 256;
    out.assign(sizes.size(), nullptr);
    const auto cut = [&](char *p) {
        for (size_t i = 0; i < sizes.size(); ++i) {
            out[i] = p;
            p += (sizes[i] + 255) / 256 * 256;
        }
    };
    {
        std::lock_guard<std::mutex> lk(g_ws_mutex);
        if (w.bytes >= bytes) {
            w.busy = true;
            cut((char *)w.p);
            return hipSuccess;
        }
        drop_workspace(&w);
    }
    void *p = nullptr;
    hipError_t e = device_malloc(&p, bytes, c->device);
    if (e == hipSuccess) {
        std::lock_guard<std::mutex> lk(g_ws_mutex);
        w.p = p;
        w.bytes = bytes;
        w.device = c->device;
        w.busy = true;
        g_workspaces.insert(&w);
        cut((char *)p);
        return hipSuccess;
    }
    (void)hipGetLastError();
    w.loose.reserve(sizes.size());
    for (size_t i = 0; i < sizes.size(); ++i) {
        e = device_malloc(&out[i], sizes[i] > 0 ? sizes[i] : 1, c->device);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            drop_loose(&w);
            return e;
        }
        w.loose.push_back(out[i]);
    }
    return hipSuccess;
}

// `to` takes over the workspace of `from` (both idle).
void move_workspace(Workspace *from, Workspace *to)
{
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    if (!from->p) return;
    drop_workspace(to);
    *to = *from;
    g_workspaces.erase(from);
    g_workspaces.insert(to);
    *from = Workspace{};
}

// The work on the workspace has ended (its streams synchronised): keep it or give it back.
void end_workspace(gpe_ctx *c)
{
    drop_loose(&c->ws);
    size_t avail = 0, total = 0;
    const bool known = hipMemGetInfo(&avail, &total) == hipSuccess;
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    c->ws.busy = false;
    if (!known || avail < total / 2) drop_workspace(&c->ws);
}

// Wait for an event: poll for up to SPIN_US, then block.  A blocking wait of more than about 20 us
// sleeps and wakes 20 us late (10 sweeps of a small box, 42 us of work: 84 us a call, 65 polled).
// Shorter waits spin inside hipStreamSynchronize, which is cheaper than an event of their own.
constexpr double SPIN_US = 1000.0;

hipError_t wait_event(hipEvent_t ev)
{
    const auto t0 = std::chrono::steady_clock::now();
    hipError_t e = hipEventQuery(ev);
    if (e != hipErrorNotReady) return e;
    while ((e = hipEventQuery(ev)) == hipErrorNotReady) {
        const std::chrono::duration<double, std::micro> us = std::chrono::steady_clock::now() - t0;
        if (us.count() > SPIN_US) break;
    }
    (void)hipGetLastError();  // "not ready" is no error of ours
    return e == hipErrorNotReady ? hipEventSynchronize(ev) : e;
}

double sweep_dt(const gpe_ctx *c) { return c->cfg.scheme == GPE_SCHEME_STAGGERED ? 0.5 * c->cfg.dt : c->cfg.dt; }

FieldRec field_at(const gpe_ctx *c, double t)
{
    FieldRec f{};
    f.trap_on = t < c->ph.trap_off_time;
    f.sigma = 1.0;
    if (c->cfg.expansion_rate != 0.0 && t > c->cfg.expansion_start)
        f.sigma = 1.0 + c->cfg.expansion_rate * (t - c->cfg.expansion_start);
    if (c->ramp.active) {
        const Ramp &r = c->ramp;
        double sq, sb[3];
        const double tr = t * r.time_scale;
        ramp_channel(r.q_val, r.q_dur, r.q_type, 1, r.tau, tr, &sq);
        ramp_channel(r.b_val, r.b_dur, r.b_type, 3, r.tau, tr, sb);
        f.bq = r.scale_q * sq;
        f.bqq = r.qscale_q * sq;
        for (int k = 0; k < 3; ++k) {
            f.bb[k] = r.scale_b * sb[k];
            f.bbq[k] = r.qscale_b * sb[k];
        }
    } else {
        f.bq = c->bq;
        f.bqq = c->bqq;
        for (int k = 0; k < 3; ++k) {
            f.bb[k] = c->bb[k];
            f.bbq[k] = c->bbq[k];
        }
    }
    f.fbq = (float)f.bq;
    f.fbqq = (float)f.bqq;
    for (int k = 0; k < 3; ++k) {
        f.fbb[k] = (float)f.bb[k];
        f.fbbq[k] = (float)f.bbq[k];
    }
    f.fsigma = (float)f.sigma;
    f.fksc = (float)(1.0 / (f.sigma * f.sigma));
    return f;
}

// FP32 mirror of the physics constants (after any change to c->ph).
void physics_to_float(Physics &ph)
{
    PhysicsF &f = ph.f;
    for (int k = 0; k < 3; ++k) {
        f.cell[k] = (float)ph.cell[k];
        f.p0[k] = (float)ph.p0[k];
        f.trap2[k] = (float)ph.trap2[k];
        f.center[k] = (float)ph.center[k];
    }
    f.trap_offset = (float)ph.trap_offset;
    f.c0 = (float)ph.c0;
    f.c1 = (float)ph.c1;
    f.c2 = (float)ph.c2;
    f.alpha = (float)ph.alpha;
    f.quad_sign = (float)ph.quad_sign;
    f.q = (float)ph.q;
}

bool quad_active(const gpe_ctx *c)
{
    if (c->cfg.ncomp == 1) return false;
    if (c->ramp.active) return c->ramp.qscale_q != 0.0 || c->ramp.qscale_b != 0.0;
    return c->bqq != 0.0 || c->bbq[0] != 0.0 || c->bbq[1] != 0.0 || c->bbq[2] != 0.0;
}

Tables tables(const gpe_ctx *c)
{
    Tables t;
    t.abi = c->d_abi;
    t.place = c->d_abi + c->g.V;
    t.w32 = c->d_w32;
    t.w64 = c->d_w64;
    t.wsum32 = c->d_wsum32;
    t.wsum64 = c->d_wsum64;
    t.pos32 = c->d_pos32;
    t.pos64 = c->d_pos64;
    t.dv = c->d_dv;
    t.nface = c->d_nface;
    t.facex = c->d_facex;
    return t;
}

int ensure_fields(gpe_ctx *c, int n)
{
    if (n <= c->fields_cap) return GPE_OK;
    int cap = c->fields_cap ? c->fields_cap : 1024;
    while (cap < n) cap *= 2;
    if (c->d_fields) {
        HIPCALL(c, hipStreamSynchronize(c->stream));
        (void)hipFree(c->d_fields);
        (void)hipHostFree(c->h_fields);
        c->d_fields = nullptr;
        c->h_fields = nullptr;
        c->fields_cap = 0;
    }
    HIPCALL(c, device_malloc((void **)&c->d_fields, sizeof(FieldRec) * cap, c->device));
    HIPCALL(c, hipHostMalloc((void **)&c->h_fields, sizeof(FieldRec) * cap, hipHostMallocDefault));
    c->fields_cap = cap;
    return GPE_OK;
}

// Upload the fields of sweeps [first, first + n) to d_fields[0..n).
int upload_fields(gpe_ctx *c, long long first, int n)
{
    int rc = ensure_fields(c, n);
    if (rc) return rc;
    HIPCALL(c, hipStreamSynchronize(c->stream));  // staging buffer may still feed a copy
    const double sdt = sweep_dt(c);
    for (int k = 0; k < n; ++k) c->h_fields[k] = field_at(c, c->t0 + (double)(first + k) * sdt);
    HIPCALL(c, hipMemcpyAsync(c->d_fields, c->h_fields, sizeof(FieldRec) * n, hipMemcpyHostToDevice, c->stream));
    return GPE_OK;
}

FastDiv make_fast_div(unsigned d)
{
    FastDiv f;
    f.d = d;
    unsigned l = 0;
    while ((1ull << l) < d) ++l;
    f.l = l;
    f.m = d <= 1 ? 1u : (unsigned)((((1ull << 32) * ((1ull << l) - d)) / d) + 1);
    return f;
}

// Lanes of a traversal's waves that carry values: rows * pairs pair slots in whole waves.
static double lane_use(int rows, int pairs)
{
    const int slots = rows * pairs;
    return (double)slots / (64.0 * ((slots + 63) / 64));
}

// pack (FP64 sweeps, one x per lane): whether the rows of a tile are one group instead of one row per
// wave.  It gains lanes, and it costs:
//   * rows of whole 128-byte lines (8 values) start waves on them, others inside lines that the
//     neighbouring wave touches too: spinors of large cells have the most of these;
//   * a box of one tile has no group whose y neighbours are all inside, and a Cube of fewer than 2 waves
//     a SIMD wants the waves rather than the lanes;
//   * the unknowns of a cell now meet a tile of rows apart, which has to stay in an XCD's 4 MiB L2 (C15
//     spin-2 of 200 values, 17 MB: 0.84 of one row's speed, 104 values, 9 MB: 0.94).
// Measured at 8 rows a tile over 1016 boxes (six lattices, 1, 3 and 5 components, 14-200 values a line,
// 8.7e4-7e6 unknowns): packed always 1.044 times the speed of one row a wave in the mean, 385 boxes of
// them slower (to 0.64); by this rule 1.083 and 7 (to 0.94); by the best choice for each 1.087.
constexpr double PACK_BYTES = 5.3e6;

// Times the lanes of one row a wave that packing has to fill to pay.
double pack_pays(const Geometry &g)
{
    const bool few = g.V == 1 && (long long)g.ny * g.nz * ((g.nx + 63) / 64) < 2000;
    if (g.ny <= g.ty || few) return 1.9;
    return g.nx % 8 == 0 ? 1.2 : (g.V > 12 && g.C > 1 ? 1.9 : 1.5);
}

bool pack_rows(const Geometry &g)
{
    return g.ty > 1 && lane_use(g.ty, g.nx) >= pack_pays(g) * lane_use(1, g.nx) &&
           16.0 * g.V * g.C * g.ty * g.lx <= PACK_BYTES;
}

// Segments, tiles, waves and workgroups of a traversal from nx, ny, nz, V, ty and xpl.
// Wave indices must stay below 2^31 (the decode's divisions).
bool finish_geometry(Geometry &g, bool pack = false)
{
    g.ty = g.ty < g.ny ? g.ty : g.ny;
    g.pairs = g.xpl == 2 ? (g.nx + 1) / 2 : g.nx;
    // x pairs: one row per wave leaves lanes idle unless a line holds a multiple of 128 values.
    // Lines of <= 64 (<= 32) values: the wave's pair slots spread over a group of 2 (4) rows of
    // the tile (a group size that divides the tile's rows).  Unit cells of <= 12 unknowns: the
    // group of 1-8 rows (dividing the tile's rows) with the best lane use when it fills at least
    // 5% more lanes (BCC 70^3 +9%, FCC 45^3 +7%, scalar FCC 160^3 +17%, spin-2 Cube 293^3 +8%,
    // spin-1 BCC 192^3 +3%; scalar Cube 293^3 -2%).  Larger cells (A15, C15, Z) take a group
    // only where it packs >= 90% of the lanes: groups of 4 rows (85%) cost A15 82^3 and Z 68^3
    // spin-2 5-7%, while 3 rows of A15's 41 pairs (96%, tiles of 6 or 12 rows) gain 6-8% and 7
    // rows of Z's 34 pairs (93%, tiles of 14) 5%; the tile heights with such divisors are
    // autotuner candidates.
    int rows = 1;
    if (g.xpl == 2 && g.slabs && g.ty > 1 && ((g.ty * g.lx) % 16 == 0 || g.ty >= g.ny)) {
        // slab layout, tiles of rows holding a multiple of 16 values (or one tile): the tile is
        // the group, one contiguous run of pairs from a 128-byte boundary
        rows = g.ty;
    } else if (g.xpl == 2) {
        const int want = g.nx <= 32 ? 4 : (g.nx <= 64 ? 2 : 1);
        while (rows < want && g.ty % (2 * rows) == 0) rows *= 2;
        const double floor_use = g.V <= 12 ? 0.0 : 0.9;
        double best = lane_use(rows, g.pairs) + 0.05;
        for (int r = 2; r <= 8; ++r)
            if (g.ty % r == 0 && lane_use(r, g.pairs) >= floor_use && lane_use(r, g.pairs) > best + 1e-9) {
                best = lane_use(r, g.pairs);
                rows = r;
            }
    } else if (pack && pack_rows(g)) {
        rows = g.ty;
    }
    g.rows = rows;
    g.tyr = g.ty / rows;
    g.nseg = rows > 1 ? (rows * g.pairs + 63) / 64 : (g.nx + 64 * g.xpl - 1) / (64 * g.xpl);
    g.ntile = (g.ny + g.ty - 1) / g.ty;
    g.waves = (long long)g.ntile * g.tyr * g.nz * g.V * g.nseg;
    g.exchange = g.rings && exchange_ok(g.deg, g.C) && (g.nseg == 1 || g.v_inner);
    const long long blocks = (g.waves + 3) / 4;
    if (blocks >= (1ll << 29)) return false;  // wave indices below 2^31 (the decode's divisions)
    g.blocks = (int)blocks;
    g.f_nseg = make_fast_div((unsigned)g.nseg);
    g.f_V = make_fast_div((unsigned)g.V);
    g.f_ty = make_fast_div((unsigned)g.tyr);
    g.f_nz = make_fast_div((unsigned)g.nz);
    g.f_pairs = make_fast_div((unsigned)g.pairs);
    return true;
}

// Tile height of an untuned sweep: 8 rows, or the lowest height up to 32 that fills the most lanes
// where that is a tenth more.  Lines of a few dozen values fill waves only in some heights, and a
// low last tile leaves whole waves empty on the XCDs that have it (20 rows of A15's 10 pairs: 52%
// of the lanes in tiles of 8, 78% in one tile; FCC 19^3 49% and 99%).  Taller tiles have to keep
// a plane's rows in an XCD's L2 with room for its neighbours (TILE_BYTES: C15 57^3 spin-2 588 us
// at 8 rows, 700 at 24), and large cells' tiles to start on 128-byte boundaries (A15 41^3 49 -> 51).
// FP64 boxes of 14-104 values a line (520 of them): 1.17 times the speed of one row a wave in tiles of 8, where the
// best of ten heights for each would give 1.21.
constexpr double TILE_BYTES = 2.6e6;

int default_tile(const Geometry &g0, int elem_bytes, bool pack)
{
    const auto use = [&](int ty) {
        Geometry g = g0;
        g.ty = ty;
        if (!finish_geometry(g, pack)) return 0.0;
        const int slots = g.xpl == 2 ? g.pairs : g.nx;
        const double lanes = (double)g.ny * slots / (64.0 * g.ntile * g.tyr * g.nseg);
        return pack && g.rows > 1 ? lanes / 1.3 : lanes;  // packed lanes are worth less, in the mean by that
    };
    const int lo = std::min(8, g0.ny), hi = std::min(32, g0.ny);
    int ty = lo;
    double best = use(lo) * 1.1;
    for (int t = lo + 1; t <= hi; ++t) {
        if ((double)t * g0.lx * g0.V * g0.C * elem_bytes > TILE_BYTES) break;
        if (g0.V > 12 && t < g0.ny && (t * g0.lx) % 16 != 0) continue;
        if (use(t) > best + 1e-9) {
            best = use(t);
            ty = t;
        }
    }
    return ty;
}

// Traversal of a reduction over a level: one x per lane, the rows of a tile as one group whose
// slots (row, x) fill whole waves.  The tile is the lowest of 8-32 rows whose waves carry within
// 3% of the most values (57-value lines, 57 rows: 19 rows 99% against 8 rows 87%, and one row
// a wave 89%; 16-value lines one row a wave 25%).  A wave takes a chunk of the group's segments:
// all of them where the groups alone give every wave of the launch one, fewer in smaller boxes.
// Needs a finished g.  Its groups are never more than g's waves, and where they are split into chunks there
// are at most 4 blocks of these (more than g's waves in some small boxes: 57x11 rows of a plane 18 for
// 16), so wave indices stay below 2^31 where g's do.
Geometry reduce_geometry(const Geometry &g, int blocks, int *segs)
{
    Geometry r = g;
    r.xpl = 1;
    r.v_inner = 0;
    r.pairs = g.nx;
    const auto segments = [&](int rows) { return ((long long)rows * g.nx + 63) / 64; };
    const auto use = [&](int ty) {  // values per lane slot of the waves that hold any
        const long long waves = (g.ny / ty) * segments(ty) + (g.ny % ty ? segments(g.ny % ty) : 0);
        return (double)g.ny * g.nx / (64.0 * waves);
    };
    const int lo = std::min(8, g.ny), hi = std::min(32, g.ny);
    double best = 0.0;
    for (int ty = lo; ty <= hi; ++ty) best = std::max(best, use(ty));
    for (r.ty = lo; use(r.ty) < best - 0.03;) ++r.ty;
    r.rows = r.ty;
    r.tyr = 1;
    r.ntile = (g.ny + r.ty - 1) / r.ty;
    const long long groups = (long long)r.ntile * g.nz * g.V, each = segments(r.ty);
    const long long parts = std::min(each, std::max(1ll, 4 * blocks / groups));
    *segs = (int)((each + parts - 1) / parts);
    r.nseg = (int)((each + *segs - 1) / *segs);
    r.waves = groups * r.nseg;
    r.blocks = (int)((r.waves + 3) / 4);
    r.f_nseg = make_fast_div((unsigned)r.nseg);
    r.f_ty = make_fast_div(1u);
    r.f_pairs = make_fast_div((unsigned)g.nx);
    return r;
}

// Layout of a configuration's levels and its default traversal (one x per lane, tiles of 8 rows,
// XCD remap), before finish_geometry.
Geometry base_geometry(const gpe_config &cfg)
{
    Geometry g{};
    g.nx = cfg.nx;
    g.ny = cfg.ny;
    g.nz = cfg.nz;
    g.V = kLattices[cfg.lattice].V;
    g.deg = kLattices[cfg.lattice].deg;
    g.rings = kLattices[cfg.lattice].rings;
    g.C = cfg.ncomp;
    g.xpl = 1;
    g.ty = cfg.ny < 8 ? cfg.ny : 8;
    // x-lines start on 128-byte boundaries unless that pads a line by more than 1/20 (the padding
    // is fetched and written in part with every line), then on 16 / 32 bytes (an even number of
    // values, which keeps the x-pair accesses 16-byte aligned).  Spin-2 FP32, even against
    // 128-byte lines: BCC 115^3 (11% padding) +8.5%, BCC 118^3 (8.5%) +5%, A15 76^3 (5.3%) +2.4%;
    // lines padded by less ran 1-3% faster with the 128-byte start.
    const long long align = cfg.precision == GPE_FP64 ? 8 : 16;
    g.lx = ((long long)cfg.nx + align - 1) / align * align;
    if (20 * g.lx > 21 * (long long)cfg.nx) g.lx = ((long long)cfg.nx + 1) / 2 * 2;
    // FP32 lines whose even length is not a whole number of 128-byte lines: component slabs of
    // contiguous rows of that even length, whose row groups start on 128-byte boundaries
    // (finish_geometry) with no padding fetched (Cube 293^3: +2-3% against 304-value x-lines)
    const long long even = ((long long)cfg.nx + 1) / 2 * 2;
    g.slabs = cfg.precision != GPE_FP64 && even % align != 0;
    if (g.slabs) g.lx = even;
    if (g.slabs) {
        const long long ls = ((long long)cfg.ny * g.lx + align - 1) / align * align;
        g.ys = g.lx;
        g.cs = ls;
        g.vs = (long long)cfg.ncomp * ls;
        g.zs = g.vs * g.V;
    } else {
        g.cs = g.lx;
        g.vs = (long long)cfg.ncomp * g.lx;
        g.ys = g.vs * g.V;
        g.zs = g.ys * cfg.ny;
    }
    g.xcd_remap = 1;
    g.v_inner = g.rings && exchange_ok(g.deg, g.C);  // rings of four in a workgroup
    return g;
}

// The same of an untuned sweep: its x values per lane and tile height.
Geometry untuned_geometry(const gpe_config &cfg)
{
    Geometry g = base_geometry(cfg);
    const int fp64 = cfg.precision == GPE_FP64;
    g.xpl = default_xpl(fp64, g.deg, cfg.ncomp, cfg.nx);
    g.ty = default_tile(g, fp64 ? 16 : 8, fp64);
    return g;
}

// Arguments of one sweep at time t of the run.
SweepArgs sweep_args(gpe_ctx *c, double t, const void *cur, void *next, double coef)
{
    SweepArgs a;
    a.g = c->gs;
    a.tb = tables(c);
    a.ph = c->ph;
    a.cur = cur;
    a.next = next;
    a.prev = nullptr;
    a.field = field_at(c, t);
    a.fields = nullptr;
    a.order = 0;
    a.quad = quad_active(c) ? 1 : 0;
    a.loss = c->cfg.alpha != 0.0 ? 1 : 0;
    a.coef = coef;
    a.scale_in = nullptr;
    a.partials = c->d_partials;
    return a;
}

// Reduction partials: AUX_COUNT doubles a workgroup of the one-x-per-lane traversal, one of the
// sweep's (norm partials), OBS_COUNT of a reduction's.
size_t partials_bytes(const gpe_ctx *c)
{
    const size_t per_block = sizeof(double) * AUX_COUNT * (size_t)std::max(c->g.blocks, c->gs.blocks);
    return std::max(per_block, sizeof(double) * OBS_COUNT * RED_BLOCKS_MAX);
}

// Sums over a level (gpe_observables_t) into d_scalars[8...] and the pinned h_red.
hipError_t reduce_observables(gpe_ctx *c, int level, double t)
{
    const FieldRec f = field_at(c, t);
    const Physics &ph = c->ph;
    ObsArgs oa;
    oa.g = c->gr;
    oa.tb = tables(c);
    oa.face = c->d_oface;
    oa.w = c->d_ow;
    oa.nfwd = c->d_nfwd;
    oa.psi = c->level[level];
    oa.quad = quad_active(c);
    ObsConsts &k = oa.k;
    const bool trap_on = t < ph.trap_off_time;
    const double sign = c->cfg.ncomp == 5 ? -1.0 : 1.0;
    k.sig = f.sigma;
    k.ik = -1.0 / (f.sigma * f.sigma);
    k.off = trap_on ? ph.trap_offset : 0.0;
    k.bq = sign * f.bq;
    k.bqq = f.bqq;
    for (int a = 0; a < 3; ++a) {
        k.p0[a] = ph.p0[a];
        k.cell[a] = f.sigma * ph.cell[a];
        k.ht[a] = trap_on ? 0.5 * ph.trap2[a] : 0.0;
        k.center[a] = ph.center[a];
        k.bb[a] = sign * f.bb[a];
        k.bbq[a] = f.bbq[a];
    }
    k.quad_sign = ph.quad_sign;
    k.q = ph.q;
    k.hc0 = 0.5 * ph.c0;
    k.hc1 = 0.5 * ph.c1;
    k.c2_10 = ph.c2 / 10.0;
    oa.segs = c->gr_segs;
    oa.per = (c->gr.blocks + c->red_blocks - 1) / c->red_blocks;
    oa.blocks = ((c->gr.blocks + oa.per - 1) / oa.per + 7) / 8 * 8;
    oa.partials = c->d_partials;
    hipError_t e = launch_observables(c->fp64, c->cfg.ncomp, oa, c->stream);
    if (e == hipSuccess)
        e = launch_finalize_few(c->d_partials, oa.blocks, OBS_COUNT, OBS_MAXDENS, c->d_scalars + 8, c->h_red,
                                c->stream);
    return e;
}

// Time of a level.
double time_of(const gpe_ctx *c, int level) { return c->t0 + (double)(c->sweeps - level) * sweep_dt(c); }

int check_level(gpe_ctx *c, int level)
{
    if (level != 0 && level != 1) return fail(c, GPE_EINVAL, "level must be 0 or 1");
    return GPE_OK;
}

}  // namespace

namespace gpe {

int ctx_view(gpe_ctx *c, CtxView *out)
{
    if (!c || !out) return GPE_EINVAL;
    out->g = c->g;
    out->tb = tables(c);
    out->fp64 = c->fp64;
    out->ncomp = c->cfg.ncomp;
    out->device = c->device;
    out->stream = c->stream;
    out->level[0] = c->level[0];
    out->level[1] = c->level[1];
    return GPE_OK;
}

int ctx_fail(gpe_ctx *c, int code, const char *what) { return fail(c, code, what); }

}  // namespace gpe

extern "C" {

int gpe_lattice_values(int lattice)
{
    if (lattice < 0 || lattice > 5) return GPE_EINVAL;
    return kLattices[lattice].V;
}

const char *gpe_last_error(const gpe_ctx *ctx)
{
    if (!ctx) return "null context";
    return ctx->err.c_str();
}

int gpe_create(const gpe_config *cfg, gpe_ctx **out)
{
    if (!cfg || !out) return GPE_EINVAL;
    *out = nullptr;
    if (cfg->lattice < 0 || cfg->lattice > 5) return GPE_EINVAL;
    if (cfg->ncomp != 1 && cfg->ncomp != 3 && cfg->ncomp != 5) return GPE_EINVAL;
    if (cfg->precision != GPE_FP32 && cfg->precision != GPE_FP64) return GPE_EINVAL;
    if (cfg->scheme != GPE_SCHEME_LEAPFROG3 && cfg->scheme != GPE_SCHEME_STAGGERED) return GPE_EINVAL;
    if (cfg->nx < 1 || cfg->ny < 1 || cfg->nz < 1) return GPE_EINVAL;
    if (!(cfg->block_scale > 0.0) || !(cfg->dt > 0.0)) return GPE_EINVAL;
    if (!(cfg->expansion_rate >= 0.0)) return GPE_EINVAL;
    gpe_ctx *c = new (std::nothrow) gpe_ctx();
    if (!c) return GPE_ENOMEM;
    c->cfg = *cfg;
    c->lat = &kLattices[cfg->lattice];
    c->fp64 = cfg->precision == GPE_FP64;
    c->elem_bytes = c->fp64 ? 16 : 8;

    Geometry &g = c->g;
    g = base_geometry(*cfg);
    c->gs = untuned_geometry(*cfg);
    if (!finish_geometry(g) || !finish_geometry(c->gs, c->fp64)) {
        delete c;
        return GPE_EINVAL;
    }
    // 32-bit index arithmetic in the kernels: offsets within a z plane and to its neighbours
    // (line_index, the per-face line offsets, row strides: below 4 zs) and line numbers
    // ((z ny + y) V + v)
    if (4 * g.zs >= (1ll << 31) || (long long)g.nz * g.ny * g.V >= (1ll << 31)) {
        delete c;
        return GPE_EINVAL;
    }
    c->level_elems = g.nz * g.zs;

    Physics &ph = c->ph;
    for (int k = 0; k < 3; ++k) ph.cell[k] = cfg->block_scale * c->lat->block_width[k];
    for (int k = 0; k < 3; ++k) {
        ph.p0[k] = cfg->p0[k];
        ph.trap[k] = cfg->trap[k];
        ph.trap2[k] = cfg->trap[k] * cfg->trap[k];
        ph.center[k] = cfg->center[k];
    }
    ph.trap_offset = cfg->trap_offset;
    ph.trap_off_time = cfg->trap_off_time;
    ph.c0 = cfg->c0;
    ph.c1 = cfg->c1;
    ph.c2 = cfg->c2;
    ph.alpha = cfg->alpha;
    ph.quad_sign = cfg->quad_sign;
    ph.q = cfg->q;
    physics_to_float(ph);

    int rc = GPE_OK;
    hipError_t e;
    if ((e = hipGetDevice(&c->device)) != hipSuccess) rc = hip_fail(c, e, "hipGetDevice");
    if (!rc && (e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking)) != hipSuccess)
        rc = hip_fail(c, e, "hipStreamCreate");
    if (!rc && (e = observables_resident(c->fp64, cfg->ncomp, c->device, &c->red_blocks)) != hipSuccess)
        rc = hip_fail(c, e, "occupancy");
    c->gr = reduce_geometry(g, c->red_blocks, &c->gr_segs);
    const size_t lbytes = (size_t)c->level_elems * c->elem_bytes;
    for (int l = 0; l < 2 && !rc; ++l) {
        if ((e = device_malloc(&c->level[l], lbytes, c->device)) != hipSuccess)
            rc = GPE_ENOMEM;
        else if ((e = hipMemsetAsync(c->level[l], 0, lbytes, c->stream)) != hipSuccess)
            rc = hip_fail(c, e, "hipMemset");
    }
    // tables: weights w_f = -1/2 hodge_f / s^2 (Spin1GpeBCC.cu:859,1169)
    const int V = g.V, deg = g.deg;
    const double s = cfg->block_scale;
    std::vector<double> w64(V * deg), wsum64(V, 0.0), pos64(3 * V), dv(V);
    std::vector<float> w32(V * deg), wsum32(V), pos32(3 * V);
    std::vector<int> nface(V), facex(2 * V * deg), oface(2 * V * deg), nfwd(V);
    std::vector<double> ow(V * deg);
    // place p of a cell on the device holds the table's unknown order[p]
    const int *order = c->lat->order;
    std::vector<int> place(V);
    for (int p = 0; p < V; ++p) place[order[p]] = p;
    for (int v = 0; v < V; ++v) {
        const int src = order[v] * deg;
        int nf = deg;  // pad faces (zero Hodge weight) trail the real ones
        while (nf > 0 && c->lat->hodge[src + nf - 1] == 0.0) --nf;
        nface[v] = nf;
        // rings: the faces to places v ^ 1 and v ^ 3 of the same cell lead, the others follow in the
        // table's order
        std::vector<int> row;
        for (int k = 0; k < (c->lat->rings ? 2 : 0); ++k)
            for (int f = 0; f < nf; ++f) {
                const int pk = c->lat->face[src + f];
                if ((pk & 63) == 21 && place[pk >> 8] == (v ^ (k ? 3 : 1))) {
                    row.push_back(f);
                    break;
                }
            }
        for (int f = 0; f < deg; ++f)
            if (std::find(row.begin(), row.end(), f) == row.end()) row.push_back(f);
        for (int f = 0; f < deg; ++f) {
            const int tab = c->lat->face[src + row[f]];
            const int pk = (tab & 63) | (place[tab >> 8] << 8);
            const long long dy = ((pk >> 2) & 3) - 1, dz = ((pk >> 4) & 3) - 1, t = pk >> 8;
            facex[2 * (v * deg + f)] = pk;
            // |offset| < 3 zs, checked against the int range at creation
            facex[2 * (v * deg + f) + 1] = (int)(dz * g.zs + dy * g.ys + (t - v) * g.vs);
            const double w = -0.5 * c->lat->hodge[src + row[f]] / (s * s);
            w64[v * deg + f] = w;
            w32[v * deg + f] = (float)w;
        }
        for (int f = 0; f < deg; ++f) wsum64[v] += -0.5 * c->lat->hodge[src + f] / (s * s);
        wsum32[v] = (float)wsum64[v];
        // the observables' order: faces to a higher address (offset between the two unknowns, dx
        // included), the others, then the pad faces
        int o = v * deg;
        for (int pass = 0; pass < 3; ++pass) {
            for (int f = 0; f < deg; ++f) {
                const int pk = facex[2 * (v * deg + f)], off = facex[2 * (v * deg + f) + 1];
                const int kind = f >= nf ? 2 : (off + (pk & 3) - 1 > 0 ? 0 : 1);
                if (kind != pass) continue;
                oface[2 * o] = pk;
                oface[2 * o + 1] = off;
                ow[o++] = w64[v * deg + f];
            }
            if (pass == 0) nfwd[v] = o - v * deg;
        }
        for (int k = 0; k < 3; ++k) {
            pos64[3 * v + k] = s * c->lat->pos[3 * order[v] + k];
            pos32[3 * v + k] = (float)pos64[3 * v + k];
        }
        dv[v] = s * s * s * c->lat->vol[order[v]];
    }
    std::vector<int> abi(order, order + V);
    abi.insert(abi.end(), place.begin(), place.end());
    // the tables in one allocation and one copy, with the small results behind them: copies of their own
    // (11 us each) and the pinned records of the adjoint's fields, now made by the call that uses them (27 us
    // and 250 to free), made it 410 us to set up and tear down a run of 8x6x5 cells, 127 so
    std::vector<char> image;
    std::vector<std::pair<void *, size_t>> at;  // a table's pointer and its place
    const auto put = [&](void *dst, const void *src, size_t bytes) {
        at.emplace_back(dst, image.size());
        image.insert(image.end(), (const char *)src, (const char *)src + bytes);
        image.resize((image.size() + 255) / 256 * 256);
    };
    put(&c->d_abi, abi.data(), sizeof(int) * 2 * V);
    put(&c->d_nface, nface.data(), sizeof(int) * V);
    put(&c->d_facex, facex.data(), sizeof(int) * 2 * V * deg);
    put(&c->d_oface, oface.data(), sizeof(int) * 2 * V * deg);
    put(&c->d_ow, ow.data(), sizeof(double) * V * deg);
    put(&c->d_nfwd, nfwd.data(), sizeof(int) * V);
    put(&c->d_w32, w32.data(), sizeof(float) * V * deg);
    put(&c->d_w64, w64.data(), sizeof(double) * V * deg);
    put(&c->d_wsum32, wsum32.data(), sizeof(float) * V);
    put(&c->d_wsum64, wsum64.data(), sizeof(double) * V);
    put(&c->d_pos32, pos32.data(), sizeof(float) * 3 * V);
    put(&c->d_pos64, pos64.data(), sizeof(double) * 3 * V);
    put(&c->d_dv, dv.data(), sizeof(double) * V);
    const size_t scalar_bytes = sizeof(double) * 64, red_bytes = sizeof(double) * FIN_SCRATCH;
    if (!rc && device_malloc((void **)&c->d_tables, image.size() + scalar_bytes + red_bytes, c->device) != hipSuccess)
        rc = GPE_ENOMEM;
    if (!rc) {
        for (const auto &t : at) {
            const void *p = c->d_tables + t.second;
            std::memcpy(t.first, &p, sizeof p);
        }
        c->d_scalars = (double *)(c->d_tables + image.size());
        c->d_red = c->d_scalars + 64;
        e = hipMemcpy(c->d_tables, image.data(), image.size(), hipMemcpyHostToDevice);
        if (e != hipSuccess) rc = hip_fail(c, e, "hipMemcpy tables");
    }
    if (!rc && device_malloc((void **)&c->d_partials, partials_bytes(c), c->device) != hipSuccess) rc = GPE_ENOMEM;
    if (!rc && hipHostMalloc((void **)&c->h_red, sizeof(double) * FIN_WIDTH_MAX, hipHostMallocDefault) != hipSuccess)
        rc = GPE_ENOMEM;
    if (!rc && (e = hipEventCreate(&c->ev0)) != hipSuccess) rc = hip_fail(c, e, "hipEventCreate");
    if (!rc && (e = hipEventCreate(&c->ev1)) != hipSuccess) rc = hip_fail(c, e, "hipEventCreate");
    if (!rc && (e = hipStreamSynchronize(c->stream)) != hipSuccess) rc = hip_fail(c, e, "create sync");
    if (rc) {
        gpe_destroy(c);
        return rc;
    }
    *out = c;
    return GPE_OK;
}

int gpe_destroy(gpe_ctx *c)
{
    if (!c) return GPE_EINVAL;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    {
        std::lock_guard<std::mutex> lk(g_ws_mutex);
        drop_workspace(&c->ws);
    }
    for (int l = 0; l < 2; ++l)
        if (c->level[l]) (void)hipFree(c->level[l]);
    void *ptrs[] = {c->d_tables, c->d_fields, c->d_partials};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (c->h_fields) (void)hipHostFree(c->h_fields);
    if (c->h_red) (void)hipHostFree(c->h_red);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    if (c->copy_stream) (void)hipStreamDestroy(c->copy_stream);
    delete c;
    return GPE_OK;
}

static int set_state_impl(gpe_ctx *c, int level, const double *psi, double t, hipMemcpyKind kind)
{
    if (!c) return GPE_EINVAL;
    if (!psi) return fail(c, GPE_EINVAL, "null state pointer");
    int rc = check_level(c, level);
    if (rc) return rc;
    const Geometry &g = c->g;
    const size_t nbytes = (size_t)c->cfg.ncomp * g.nz * g.ny * g.nx * g.V * 2 * sizeof(double);
    const double *src = psi;
    double *staging = nullptr;
    if (kind == hipMemcpyHostToDevice) {
        HIPCALL(c, device_malloc((void **)&staging, nbytes, c->device, c->stream));
        HIPCALL(c, hipMemcpyAsync(staging, psi, nbytes, hipMemcpyHostToDevice, c->stream));
        src = staging;
    }
    hipError_t e = launch_pack(c->fp64, g, tables(c), c->cfg.ncomp, src, c->level[level], c->stream);
    if (staging) (void)hipFreeAsync(staging, c->stream);
    if (e != hipSuccess) return hip_fail(c, e, "pack");
    HIPCALL(c, hipStreamSynchronize(c->stream));
    if (level == 0) {
        c->t0 = t;
        c->sweeps = 0;
        c->level1_valid = false;
    } else {
        c->level1_valid = true;
    }
    return GPE_OK;
}

int gpe_set_state(gpe_ctx *c, int level, const double *psi, double t)
{
    return set_state_impl(c, level, psi, t, hipMemcpyHostToDevice);
}

int gpe_set_state_device(gpe_ctx *c, int level, const double *dpsi, double t)
{
    return set_state_impl(c, level, dpsi, t, hipMemcpyDeviceToDevice);
}

static int get_state_impl(gpe_ctx *c, int level, double *psi, bool host)
{
    if (!c) return GPE_EINVAL;
    if (!psi) return fail(c, GPE_EINVAL, "null state pointer");
    int rc = check_level(c, level);
    if (rc) return rc;
    const Geometry &g = c->g;
    const size_t nbytes = (size_t)c->cfg.ncomp * g.nz * g.ny * g.nx * g.V * 2 * sizeof(double);
    double *dst = psi;
    double *staging = nullptr;
    if (host) {
        HIPCALL(c, device_malloc((void **)&staging, nbytes, c->device, c->stream));
        dst = staging;
    }
    hipError_t e = launch_unpack(c->fp64, g, tables(c), c->cfg.ncomp, c->level[level], dst, c->stream);
    if (e != hipSuccess) return hip_fail(c, e, "unpack");
    if (host) {
        HIPCALL(c, hipMemcpyAsync(psi, staging, nbytes, hipMemcpyDeviceToHost, c->stream));
        (void)hipFreeAsync(staging, c->stream);
    }
    HIPCALL(c, hipStreamSynchronize(c->stream));
    return GPE_OK;
}

int gpe_get_state(gpe_ctx *c, int level, double *psi) { return get_state_impl(c, level, psi, true); }
int gpe_get_state_device(gpe_ctx *c, int level, double *dpsi) { return get_state_impl(c, level, dpsi, false); }

int gpe_set_field(gpe_ctx *c, double bq, const double bb[3], double bq_quad, const double bb_quad[3])
{
    if (!c) return GPE_EINVAL;
    c->ramp.active = false;
    c->bq = bq;
    c->bqq = bq_quad;
    for (int k = 0; k < 3; ++k) {
        c->bb[k] = bb ? bb[k] : 0.0;
        c->bbq[k] = bb_quad ? bb_quad[k] : 0.0;
    }
    return GPE_OK;
}

int gpe_set_ramp(gpe_ctx *c, const gpe_ramp *r)
{
    if (!c) return GPE_EINVAL;
    if (!r) {
        c->ramp.active = false;
        return GPE_OK;
    }
    if (r->nq < 0 || r->nb < 0) return fail(c, GPE_EINVAL, "negative segment count");
    if ((r->nq && (!r->q_val || !r->q_dur || !r->q_type)) || (r->nb && (!r->b_val || !r->b_dur || !r->b_type)))
        return fail(c, GPE_EINVAL, "null ramp array");
    Ramp &d = c->ramp;
    d.q_val.assign(r->q_val, r->q_val + r->nq);
    d.q_dur.assign(r->q_dur, r->q_dur + r->nq);
    d.q_type.assign(r->q_type, r->q_type + r->nq);
    d.b_val.assign(r->b_val, r->b_val + 3 * r->nb);
    d.b_dur.assign(r->b_dur, r->b_dur + r->nb);
    d.b_type.assign(r->b_type, r->b_type + r->nb);
    for (int t : d.q_type)
        if (t < 0 || t > 3) return fail(c, GPE_EINVAL, "bad ramp segment type");
    for (int t : d.b_type)
        if (t < 0 || t > 3) return fail(c, GPE_EINVAL, "bad ramp segment type");
    d.tau = r->tau;
    d.time_scale = r->time_scale;
    d.scale_q = r->scale_q;
    d.scale_b = r->scale_b;
    d.qscale_q = r->qscale_q;
    d.qscale_b = r->qscale_b;
    d.active = true;
    return GPE_OK;
}

int gpe_start(gpe_ctx *c, int mode, double mu)
{
    if (!c) return GPE_EINVAL;
    const double sdt = sweep_dt(c);
    if (mode == GPE_START_EULER) {
        SweepArgs a = sweep_args(c, time_of(c, 0), c->level[0], c->level[1], sdt);
        hipError_t e = launch_sweep(c->fp64, c->cfg.ncomp, MODE_EULER, a, c->stream);
        if (e != hipSuccess) return hip_fail(c, e, "forward Euler");
        std::swap(c->level[0], c->level[1]);
        c->sweeps += 1;
    } else if (mode == GPE_START_PHASE) {
        // psi(t - sdt) = exp(+i mu sdt) psi(t)  (GPBlocks.cpp:516-523)
        hipError_t e = launch_phase_copy(c->fp64, c->level[0], c->level[1], c->level_elems, std::cos(mu * sdt),
                                         std::sin(mu * sdt), c->stream);
        if (e != hipSuccess) return hip_fail(c, e, "phase start");
    } else if (mode == GPE_START_COPY) {
        HIPCALL(c, hipMemcpyAsync(c->level[1], c->level[0], (size_t)c->level_elems * c->elem_bytes,
                                  hipMemcpyDeviceToDevice, c->stream));
    } else {
        return fail(c, GPE_EINVAL, "unknown start mode");
    }
    c->level1_valid = true;
    HIPCALL(c, hipStreamSynchronize(c->stream));
    return GPE_OK;
}

int gpe_step(gpe_ctx *c, int nsteps)
{
    if (!c) return GPE_EINVAL;
    if (nsteps < 0) return fail(c, GPE_EINVAL, "negative step count");
    if (!c->level1_valid) return fail(c, GPE_ESTATE, "second time level not set: call gpe_start");
    if (nsteps == 0) return GPE_OK;
    const int per = c->cfg.scheme == GPE_SCHEME_STAGGERED ? 2 : 1;
    const long long total = (long long)nsteps * per;
    const double coef = 2.0 * sweep_dt(c);
    HIPCALL(c, hipEventRecord(c->ev0, c->stream));
    for (long long k = 0; k < total; ++k) {
        // the field travels in the kernel's arguments: nothing to upload, and one load less in the
        // sweep's chain of scalar loads
        SweepArgs a = sweep_args(c, time_of(c, 0), c->level[0], c->level[1], coef);
        a.order = (int)(c->sweeps & 1);
        hipError_t e = launch_sweep(c->fp64, c->cfg.ncomp, MODE_UPDATE, a, c->stream);
        if (e != hipSuccess) return hip_fail(c, e, "sweep launch");
        std::swap(c->level[0], c->level[1]);
        c->sweeps += 1;
        if ((k & 0xffff) == 0xffff) HIPCALL(c, hipStreamSynchronize(c->stream));  // bounds the queue
    }
    HIPCALL(c, hipEventRecord(c->ev1, c->stream));
    HIPCALL(c, wait_event(c->ev1));
    float ms = 0.f;
    HIPCALL(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms_per_sweep = ms / (double)total;
    return GPE_OK;
}

int gpe_itp(gpe_ctx *c, int nsteps, double dt_itp)
{
    if (!c) return GPE_EINVAL;
    if (nsteps < 0 || !(dt_itp > 0.0)) return fail(c, GPE_EINVAL, "bad ITP arguments");
    double *scale[2] = {c->d_scalars + 1, c->d_scalars + 2};
    // initial scale from the norm of level 0
    NormArgs na;
    na.g = c->gr;
    na.psi = c->level[0];
    na.dv = c->d_dv;
    na.segs = c->gr_segs;
    na.per = (c->gr.blocks + c->red_blocks - 1) / c->red_blocks;
    na.blocks = ((c->gr.blocks + na.per - 1) / na.per + 7) / 8 * 8;
    na.partials = c->d_partials;
    hipError_t e = launch_norm(c->fp64, c->cfg.ncomp, na, c->stream);
    if (e == hipSuccess) e = launch_norm_scale(c->d_partials, na.blocks, 1.0, scale[0], c->d_red, c->stream);
    if (e != hipSuccess) return hip_fail(c, e, "ITP initial norm");
    SweepArgs a = sweep_args(c, time_of(c, 0), nullptr, nullptr, dt_itp);
    for (int i = 0; i < nsteps; ++i) {
        a.cur = c->level[0];
        a.next = c->level[1];
        a.scale_in = scale[i & 1];
        a.order = i & 1;
        e = launch_sweep(c->fp64, c->cfg.ncomp, MODE_ITP, a, c->stream);
        if (e == hipSuccess)
            e = launch_norm_scale(c->d_partials, c->gs.blocks, 1.0, scale[(i + 1) & 1], c->d_red, c->stream);
        if (e != hipSuccess) return hip_fail(c, e, "ITP step");
        std::swap(c->level[0], c->level[1]);
    }
    e = launch_scale(c->fp64, c->level[0], c->level_elems, 1.0, scale[nsteps & 1], c->stream);
    if (e != hipSuccess) return hip_fail(c, e, "ITP final scale");
    c->level1_valid = false;
    HIPCALL(c, hipStreamSynchronize(c->stream));
    return GPE_OK;
}

int gpe_observables(gpe_ctx *c, int level, gpe_observables_t *out)
{
    if (!c) return GPE_EINVAL;
    if (!out) return fail(c, GPE_EINVAL, "null output");
    int rc = check_level(c, level);
    if (rc) return rc;
    const double t = time_of(c, level);
    const hipError_t e = reduce_observables(c, level, t);
    if (e != hipSuccess) return hip_fail(c, e, "observables");
    HIPCALL(c, hipStreamSynchronize(c->stream));
    const double *h = c->h_red;
    out->norm = h[OBS_NORM];
    out->energy = h[OBS_ENERGY];
    out->expect_h = h[OBS_EXPECT_H];
    out->magnetization[0] = h[OBS_MX];
    out->magnetization[1] = h[OBS_MY];
    out->magnetization[2] = h[OBS_MZ];
    out->max_density = h[OBS_MAXDENS];
    out->time = t;
    out->finite = (h[OBS_NONFINITE] == 0.0 && std::isfinite(h[OBS_NORM]) && std::isfinite(h[OBS_ENERGY])) ? 1 : 0;
    out->spin = h[OBS_SPIN];
    out->moment[0] = h[OBS_RX];
    out->moment[1] = h[OBS_RY];
    out->moment[2] = h[OBS_RZ];
    out->ref_spin = h[OBS_REF_SPIN];
    out->ref_magnetization_z = h[OBS_REF_MZ];
    return out->finite ? GPE_OK : fail(c, GPE_ERANGE, "non-finite value in the state");
}

// ------------------------------------------------------------------ observable series --

// The reference's time-series file (Spin1GpeBCC.cu:1497-1504, 1659-1712): eight MATLAB
// vectors that each saved file extends ("times = [times, ...];"), one column per append.
struct gpe_series {
    std::vector<double> col[8];  // times, Bq, Bz, Spin, mag_x, mag_y, mag_z, norm
};

int gpe_series_create(gpe_series **out)
{
    if (!out) return GPE_EINVAL;
    *out = new (std::nothrow) gpe_series();
    return *out ? GPE_OK : GPE_ENOMEM;
}

int gpe_series_destroy(gpe_series *s)
{
    delete s;
    return GPE_OK;
}

int gpe_series_append(gpe_series *s, gpe_ctx *c, int level)
{
    if (!s || !c) return GPE_EINVAL;
    gpe_observables_t o;
    const int rc = gpe_observables(c, level, &o);
    if (rc && rc != GPE_ERANGE) return rc;
    const FieldRec f = field_at(c, o.time);
    const double v[8] = {o.time * (c->ramp.active ? c->ramp.time_scale : 1.0),
                         f.bq,
                         f.bb[0] + f.bb[1] + f.bb[2],
                         o.ref_spin,
                         o.magnetization[0],
                         o.magnetization[1],
                         o.ref_magnetization_z,
                         o.norm};
    for (int k = 0; k < 8; ++k) s->col[k].push_back(v[k]);
    return rc;
}

int gpe_series_save(gpe_series *s, const char *path)
{
    if (!s || !path) return GPE_EINVAL;
    static const char *const names[8] = {"times", "Bq", "Bz", "Spin", "mag_x", "mag_y", "mag_z", "norm"};
    FILE *f = std::fopen(path, "w");
    if (!f) return GPE_EINVAL;
    bool ok = true;
    for (int k = 0; k < 8 && ok; ++k) {
        ok = std::fprintf(f, "%s = [%s", names[k], names[k]) > 0;
        for (double x : s->col[k]) ok = ok && std::fprintf(f, ", %.18f", x) > 0;
        ok = ok && std::fprintf(f, "];\n") > 0;
    }
    ok = (std::fclose(f) == 0) && ok;
    if (!ok) return GPE_EDEVICE;
    for (auto &v : s->col) v.clear();  // the next file starts a new series, as the reference's does
    return GPE_OK;
}

// k_aux over a level with an optional device reference state; h[0] = maximum, h[1] = sum.
static int aux_reduce(gpe_ctx *c, int level, const double *dref, double pre, double pim, double h[AUX_COUNT])
{
    const double t = time_of(c, level);
    AuxArgs aa;
    aa.g = c->g;
    aa.tb = tables(c);
    aa.ph = c->ph;
    aa.psi = c->level[level];
    aa.ref = (const double2 *)dref;
    aa.phase_re = pre;
    aa.phase_im = pim;
    aa.field = field_at(c, t);
    aa.partials = c->d_partials;
    hipError_t e = launch_aux(c->fp64, c->cfg.ncomp, aa, c->stream);
    if (e == hipSuccess) e = launch_finalize(c->d_partials, c->g.blocks, AUX_COUNT, AUX_MAXHAM, c->d_scalars + 8, c->d_red, c->stream);
    if (e != hipSuccess) return hip_fail(c, e, "local reduction");
    HIPCALL(c, hipMemcpyAsync(h, c->d_scalars + 8, sizeof(double) * AUX_COUNT, hipMemcpyDeviceToHost, c->stream));
    HIPCALL(c, hipStreamSynchronize(c->stream));
    return GPE_OK;
}

int gpe_max_hamiltonian(gpe_ctx *c, int level, double *out)
{
    if (!c) return GPE_EINVAL;
    if (!out) return fail(c, GPE_EINVAL, "null output");
    if (c->cfg.ncomp == 5) return fail(c, GPE_EINVAL, "the Hamiltonian bound is defined for scalar and spin-1 states");
    int rc = check_level(c, level);
    if (rc) return rc;
    double h[AUX_COUNT];
    if ((rc = aux_reduce(c, level, nullptr, 1.0, 0.0, h))) return rc;
    *out = h[AUX_MAXHAM];
    return std::isfinite(*out) ? GPE_OK : fail(c, GPE_ERANGE, "non-finite value in the state");
}

int gpe_weighted_diff_device(gpe_ctx *c, int level, const double *dref, double phase_re, double phase_im, double *out)
{
    if (!c) return GPE_EINVAL;
    if (!dref || !out) return fail(c, GPE_EINVAL, "null reference state or output");
    int rc = check_level(c, level);
    if (rc) return rc;
    double h[AUX_COUNT];
    if ((rc = aux_reduce(c, level, dref, phase_re, phase_im, h))) return rc;
    *out = h[AUX_WDIFF];
    return GPE_OK;
}

int gpe_weighted_diff(gpe_ctx *c, int level, const double *ref, double phase_re, double phase_im, double *out)
{
    if (!c) return GPE_EINVAL;
    if (!ref || !out) return fail(c, GPE_EINVAL, "null reference state or output");
    int rc = check_level(c, level);
    if (rc) return rc;
    const size_t bytes = 2 * sizeof(double) * (size_t)c->cfg.ncomp * c->cfg.nx * c->cfg.ny * c->cfg.nz * c->g.V;
    double *d = nullptr;
    if (device_malloc((void **)&d, bytes, c->device) != hipSuccess)
        return fail(c, GPE_ENOMEM, "reference state does not fit");
    hipError_t e = hipMemcpyAsync(d, ref, bytes, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) rc = gpe_weighted_diff_device(c, level, d, phase_re, phase_im, out);
    else rc = hip_fail(c, e, "reference upload");
    (void)hipStreamSynchronize(c->stream);
    (void)hipFree(d);
    return rc;
}

int gpe_field_width(int kind)
{
    switch (kind) {
    case GPE_FIELD_DENSITY: return 1;
    case GPE_FIELD_SPIN: return 3;
    case GPE_FIELD_SPIN_NORM: return 1;
    case GPE_FIELD_UV_THETA: return 7;
    default: return GPE_EINVAL;
    }
}

int gpe_local_fields(gpe_ctx *c, int level, int kind, double *out)
{
    if (!c) return GPE_EINVAL;
    const int width = gpe_field_width(kind);
    if (width < 0) return fail(c, GPE_EINVAL, "unknown field kind");
    if (!out) return fail(c, GPE_EINVAL, "null output");
    if (kind == GPE_FIELD_UV_THETA && c->cfg.ncomp != 3) return fail(c, GPE_EINVAL, "u, v, theta need spin-1");
    int rc = check_level(c, level);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * (size_t)width * (size_t)c->cfg.nx * c->cfg.ny * c->cfg.nz * c->g.V;
    double *d = nullptr;
    if (device_malloc((void **)&d, bytes, c->device) != hipSuccess)
        return fail(c, GPE_ENOMEM, "field map does not fit");
    hipError_t e = launch_local_fields(c->fp64, c->cfg.ncomp, c->g, tables(c), c->level[level], kind, d, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(out, d, bytes, hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    (void)hipFree(d);
    return e == hipSuccess ? GPE_OK : hip_fail(c, e, "local fields");
}

int gpe_scale(gpe_ctx *c, int level, double factor)
{
    if (!c) return GPE_EINVAL;
    int rc = check_level(c, level);
    if (rc) return rc;
    hipError_t e = launch_scale(c->fp64, c->level[level], c->level_elems, factor, nullptr, c->stream);
    if (e != hipSuccess) return hip_fail(c, e, "scale");
    HIPCALL(c, hipStreamSynchronize(c->stream));
    return GPE_OK;
}

int gpe_sync(gpe_ctx *c)
{
    if (!c) return GPE_EINVAL;
    HIPCALL(c, hipStreamSynchronize(c->stream));
    return GPE_OK;
}

int gpe_time(const gpe_ctx *c, double *t, long long *sweeps)
{
    if (!c) return GPE_EINVAL;
    if (t) *t = c->t0 + (double)c->sweeps * sweep_dt(c);
    if (sweeps) *sweeps = c->sweeps;
    return GPE_OK;
}

int gpe_fill_thomas_fermi(gpe_ctx *c, double g, double mu, const double *weights, double noise, unsigned long long seed,
                          double t)
{
    if (!c) return GPE_EINVAL;
    if (!(g > 0.0) || !weights || noise < 0.0) return fail(c, GPE_EINVAL, "bad Thomas-Fermi fill arguments");
    FillArgs f;
    f.mu = mu;
    f.g = g;
    f.amp = noise;
    f.seed = seed;
    for (int k = 0; k < 10; ++k) f.w[k] = k < 2 * c->cfg.ncomp ? weights[k] : 0.0;
    hipError_t e = launch_fill_tf(c->fp64, c->g, tables(c), c->ph, c->cfg.ncomp, f, c->level[0], c->stream);
    if (e != hipSuccess) return hip_fail(c, e, "fill");
    HIPCALL(c, hipStreamSynchronize(c->stream));
    c->t0 = t;
    c->sweeps = 0;
    c->level1_valid = false;
    return GPE_OK;
}

int gpe_set_trap(gpe_ctx *c, const double trap[3])
{
    if (!c || !trap) return GPE_EINVAL;
    for (int k = 0; k < 3; ++k) {
        c->cfg.trap[k] = trap[k];
        c->ph.trap[k] = trap[k];
        c->ph.trap2[k] = trap[k] * trap[k];
    }
    physics_to_float(c->ph);
    return GPE_OK;
}

int gpe_get_config(const gpe_ctx *c, gpe_config *out)
{
    if (!c || !out) return GPE_EINVAL;
    *out = c->cfg;
    return GPE_OK;
}

int gpe_set_time(gpe_ctx *c, double t0, long long sweeps)
{
    if (!c) return GPE_EINVAL;
    if (sweeps < 0 || !std::isfinite(t0)) return fail(c, GPE_EINVAL, "bad clock");
    c->t0 = t0;
    c->sweeps = sweeps;
    return GPE_OK;
}

int gpe_clock(const gpe_ctx *c, double *t0, long long *sweeps)
{
    if (!c) return GPE_EINVAL;
    if (t0) *t0 = c->t0;
    if (sweeps) *sweeps = c->sweeps;
    return GPE_OK;
}

int gpe_project_spinor(gpe_ctx *c, int level, int phase, double param)
{
    if (!c) return GPE_EINVAL;
    int rc = check_level(c, level);
    if (rc) return rc;
    const int C = c->cfg.ncomp;
    const bool spin1 = C == 3 && (phase == GPE_PHASE_POLAR || phase == GPE_PHASE_FERRO || phase == GPE_PHASE_MIXED);
    const bool spin2 = C == 5 && (phase == GPE_PHASE_FERRO || (phase >= GPE_PHASE_UN && phase <= GPE_PHASE_CYCLIC));
    if (!spin1 && !spin2) return fail(c, GPE_EINVAL, "phase does not exist for this component count");
    if (phase == GPE_PHASE_MIXED && !(param >= 0.0 && param <= 1.0)) return fail(c, GPE_EINVAL, "mix outside [0, 1]");
    hipError_t e = launch_project(c->fp64, C, c->g, c->level[level], phase, param, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    return e == hipSuccess ? GPE_OK : hip_fail(c, e, "spinor projection");
}

int gpe_add_noise(gpe_ctx *c, int level, double amplitude, unsigned long long seed)
{
    if (!c) return GPE_EINVAL;
    int rc = check_level(c, level);
    if (rc) return rc;
    if (!(amplitude >= 0.0)) return fail(c, GPE_EINVAL, "negative noise amplitude");
    hipError_t e = launch_noise(c->fp64, c->cfg.ncomp, c->g, tables(c), c->level[level], amplitude, seed, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    return e == hipSuccess ? GPE_OK : hip_fail(c, e, "noise");
}

int gpe_set_knot_ramp(gpe_ctx *c, int n, const double *knots, double duration, double bq)
{
    if (!c) return GPE_EINVAL;
    if (n < 2 || !knots || !(duration > 0.0)) return fail(c, GPE_EINVAL, "need >= 2 knots and a positive duration");
    std::vector<double> bval(3 * (size_t)n, 0.0), bdur(n), qval{bq}, qdur{1e300};
    std::vector<int> btype(n), qtype{0};
    for (int j = 0; j < n; ++j) {
        bval[3 * j + 2] = knots[j];
        bdur[j] = j == 0 ? 0.0 : duration / (n - 1);
        btype[j] = j == 0 ? 0 : 1;
    }
    gpe_ramp r{};
    r.nq = 1;
    r.q_val = qval.data();
    r.q_dur = qdur.data();
    r.q_type = qtype.data();
    r.nb = n;
    r.b_val = bval.data();
    r.b_dur = bdur.data();
    r.b_type = btype.data();
    r.tau = 1.0;
    r.time_scale = 1.0;
    r.scale_q = r.scale_b = 1.0;
    r.qscale_q = r.qscale_b = 0.0;
    return gpe_set_ramp(c, &r);
}

// Ramp sensitivities: the ramp value is linear in the segment values, so
// d value(t) / d val[j] = value(t) evaluated with val = e_j.
static double ramp_basis(const std::vector<double> &dur, const std::vector<int> &type, double tau, double t, int j)
{
    std::vector<double> e(dur.size(), 0.0);
    e[j] = 1.0;
    double out;
    ramp_channel(e, dur, type, 1, tau, t, &out);
    return out;
}

// The adjoint of an FP32 context with FP64 psi and mu: the run (configuration, fields, ramp,
// clock and level 0) is copied into a temporary FP64 context, the adjoint taken there, and the
// final two levels copied back.
static int adjoint_fp64_copy(gpe_ctx *c, const gpe_adjoint_spec *spec, gpe_adjoint_result *res)
{
    gpe_config cfg = c->cfg;
    cfg.precision = GPE_FP64;
    gpe_ctx *d = nullptr;
    int rc = gpe_create(&cfg, &d);
    if (rc) return fail(c, rc, "the FP64 copy of the run does not fit");
    d->ramp = c->ramp;
    d->bq = c->bq;
    d->bqq = c->bqq;
    for (int k = 0; k < 3; ++k) {
        d->bb[k] = c->bb[k];
        d->bbq[k] = c->bbq[k];
    }
    const size_t abi = (size_t)cfg.ncomp * c->g.nz * c->g.ny * c->g.nx * c->g.V * 2 * sizeof(double);
    double *tmp = nullptr;
    if (device_malloc((void **)&tmp, abi, c->device) != hipSuccess) {
        gpe_destroy(d);
        return fail(c, GPE_ENOMEM, "staging for the FP64 copy does not fit");
    }
    const double t0 = c->t0;
    rc = gpe_get_state_device(c, 0, tmp);
    if (!rc) rc = gpe_set_state_device(d, 0, tmp, t0);
    gpe_adjoint_spec s64 = *spec;
    s64.fp64_trajectory = 0;
    if (!rc) {
        move_workspace(&c->ws, &d->ws);
        rc = gpe_adjoint(d, &s64, res);
        if (rc) c->err = "FP64 copy: " + d->err;
        move_workspace(&d->ws, &c->ws);
    }
    if (!rc) rc = gpe_get_state_device(d, 0, tmp);
    if (!rc) rc = gpe_set_state_device(c, 0, tmp, t0);
    if (!rc) rc = gpe_get_state_device(d, 1, tmp);
    if (!rc) rc = gpe_set_state_device(c, 1, tmp, t0);
    if (!rc) {
        c->sweeps = d->sweeps;
        c->level1_valid = true;
    } else {
        c->level1_valid = false;
    }
    (void)hipFree(tmp);
    gpe_destroy(d);
    return rc;
}

int gpe_adjoint(gpe_ctx *c, const gpe_adjoint_spec *spec, gpe_adjoint_result *res)
{
    if (!c) return GPE_EINVAL;
    if (!spec || !res) return fail(c, GPE_EINVAL, "null adjoint spec or result");
    if (c->cfg.scheme != GPE_SCHEME_LEAPFROG3) return fail(c, GPE_EINVAL, "adjoint needs the 3-level scheme");
    if (c->cfg.alpha != 0.0) return fail(c, GPE_EINVAL, "adjoint needs alpha = 0");
    if (c->cfg.expansion_rate != 0.0) return fail(c, GPE_EINVAL, "adjoint needs a static grid (expansion_rate = 0)");
    if (c->ramp.active && (c->ramp.qscale_q != 0.0 || c->ramp.qscale_b != 0.0))
        return fail(c, GPE_EINVAL, "adjoint does not differentiate a ramped quadratic field");
    const int N = spec->nsweeps, K = spec->checkpoint_every;
    if (N < 1 || K < 2) return fail(c, GPE_EINVAL, "need nsweeps >= 1 and checkpoint_every >= 2");
    if (spec->objective < 0 || spec->objective > 2) return fail(c, GPE_EINVAL, "unknown objective");
    if (spec->objective == GPE_OBJ_OVERLAP && !spec->target) return fail(c, GPE_EINVAL, "overlap needs a target");
    if (c->sweeps != 0) return fail(c, GPE_ESTATE, "adjoint must start right after gpe_set_state");
    if (spec->fp64_trajectory && !c->fp64) return adjoint_fp64_copy(c, spec, res);

    const size_t lbytes = (size_t)c->level_elems * c->elem_bytes;
    const int nck = (N + K - 1) / K;
    const Geometry &g = c->g;
    const size_t abi = (size_t)c->cfg.ncomp * g.nz * g.ny * g.nx * g.V * 2 * sizeof(double);
    const bool overlap = spec->objective == GPE_OBJ_OVERLAP;
    // per-sweep sensitivity partials of up to Q consecutive adjoint sweeps, summed in one launch
    // (one two-stage finalize per sweep cost ~15% of the backward pass in launches)
    // the adjoint sweeps run on the forward sweep's traversal (x pairs in FP32)
    const int adj_blocks = c->gs.blocks;
    const size_t sweep_part = (size_t)ADJ_COUNT * adj_blocks;
    const int Q = (int)std::max<size_t>(1, std::min<size_t>((size_t)K, ((size_t)256 << 20) / (sweep_part * 8)));
    // every buffer of the run in the context's workspace
    const int nseg = std::min(K, N);  // levels of the longest segment
    const int nlevels = 2 * nck + std::max(nseg - 2, 0) + 2 + (overlap ? 1 : 0);
    std::vector<size_t> sizes(nlevels, lbytes);
    sizes.push_back(overlap ? abi : 0);
    sizes.push_back(sizeof(double) * ADJ_COUNT * (size_t)N);
    sizes.push_back(sizeof(double) * ADJ_COUNT * (size_t)g.blocks);
    sizes.push_back(sizeof(double) * sweep_part * Q);
    std::vector<void *> bufs;
    if (begin_workspace(c, sizes, bufs) != hipSuccess) return fail(c, GPE_ENOMEM, "adjoint buffers do not fit");
    const auto release = [&]() {
        (void)hipStreamSynchronize(c->stream);
        if (c->copy_stream) (void)hipStreamSynchronize(c->copy_stream);
        end_workspace(c);
    };
    size_t taken = 0;
    const auto next = [&]() { return bufs[taken++]; };
    std::vector<void *> ck(2 * nck), seg(std::max(nseg, 2), nullptr);
    for (void *&p : ck) p = next();
    for (int i = 2; i < nseg; ++i) seg[i] = next();  // seg[0], seg[1] alias checkpoints
    void *mu[2];
    for (void *&p : mu) p = next();
    void *target = overlap ? next() : nullptr;
    double *staging = (double *)next(), *d_steps = (double *)next(), *d_part = (double *)next();
    double *d_qpart = (double *)next();
    int rc = GPE_OK;
    res->checkpoint_bytes = (double)lbytes * 2 * nck;
    res->segment_bytes = (double)lbytes * nseg;
    hipError_t e = hipSuccess;
    // on a failure the buffers are freed and the levels hold an intermediate state: the
    // context needs gpe_set_state (and gpe_start) before it steps again
#define ADJ_CHECK(call, what)                 \
    do {                                      \
        e = (call);                           \
        if (e != hipSuccess) {                \
            release();                        \
            c->level1_valid = false;          \
            return hip_fail(c, e, what);      \
        }                                     \
    } while (0)

    const double sdt = sweep_dt(c);
    rc = upload_fields(c, 0, N);
    if (rc) {
        release();
        return rc;
    }
    // ---- forward pass, keeping (psi_jK, psi_jK+1)
    ADJ_CHECK(hipEventRecord(c->ev0, c->stream), "adjoint");
    // where psi_m is written: the last segment's levels stay where the reverse pass reads them, so it
    // recomputes nothing there, the others' first two in their checkpoints, the rest alternate
    // between the context's levels
    const int klast = (nck - 1) * K;
    void *const even = c->level[0], *const odd = c->level[1];
    const auto at = [&](int m) -> void * {
        if (m < N && m >= klast && m - klast >= 2) return seg[m - klast];
        if (m < N && m % K < 2) return ck[2 * (m / K) + m % K];
        return m & 1 ? odd : even;
    };
    ADJ_CHECK(hipMemcpyAsync(ck[0], even, lbytes, hipMemcpyDeviceToDevice, c->stream), "checkpoint");
    for (int k = 0; k < N; ++k) {  // produces psi_{k+1}
        SweepArgs a = sweep_args(c, c->t0 + k * sdt, at(k), at(k + 1), k == 0 ? sdt : 2.0 * sdt);
        a.order = k & 1;
        if (k > 0 && at(k - 1) != at(k + 1)) a.prev = at(k - 1);
        ADJ_CHECK(launch_sweep(c->fp64, c->cfg.ncomp, k == 0 ? MODE_EULER : MODE_UPDATE, a, c->stream), "forward sweep");
    }
    // psi_N in level 0, psi_{N-1} in level 1
    c->level[0] = at(N);
    c->level[1] = c->level[0] == even ? odd : even;
    ADJ_CHECK(hipMemcpyAsync(c->level[1], at(N - 1), lbytes, hipMemcpyDeviceToDevice, c->stream), "psi_{N-1}");
    c->sweeps = N;
    c->level1_valid = true;
    ADJ_CHECK(hipEventRecord(c->ev1, c->stream), "adjoint");
    if (overlap) {  // the host's copy of the target goes up while the forward sweeps run
        if (!c->copy_stream)
            ADJ_CHECK(hipStreamCreateWithFlags(&c->copy_stream, hipStreamNonBlocking), "copy stream");
        ADJ_CHECK(hipMemcpyAsync(staging, spec->target, abi, hipMemcpyHostToDevice, c->copy_stream), "target");
        ADJ_CHECK(launch_pack(c->fp64, g, tables(c), c->cfg.ncomp, staging, target, c->copy_stream), "pack target");
        ADJ_CHECK(hipStreamSynchronize(c->copy_stream), "target");
    }
    ADJ_CHECK(hipEventSynchronize(c->ev1), "adjoint");
    float fms = 0.f;
    ADJ_CHECK(hipEventElapsedTime(&fms, c->ev0, c->ev1), "adjoint");
    res->forward_ms = fms;

    // ---- objective and mu_N
    ADJ_CHECK(hipEventRecord(c->ev0, c->stream), "adjoint");
    ObjArgs oa;
    oa.g = c->g;
    oa.tb = tables(c);
    oa.ph = c->ph;
    oa.field = field_at(c, c->t0 + N * sdt);
    oa.psi = c->level[0];
    oa.target = target;
    oa.grad = mu[1];
    oa.scalars = c->d_scalars + 32;
    oa.partials = d_part;
    ADJ_CHECK(hipMemsetAsync(mu[0], 0, lbytes, c->stream), "clear mu");
    double J = 0.0;
    double explicit_mom[4] = {0, 0, 0, 0};  // energy: sum dv r_a^2 n, s sum dv (dx Fx + dy Fy - 2 dz Fz)
    double explicit_mag[3] = {0, 0, 0};
    if (overlap) {
        oa.mode = OBJ_PARTIALS;
        ADJ_CHECK(launch_objective(c->fp64, c->cfg.ncomp, oa, c->stream), "overlap");
        ADJ_CHECK(launch_finalize(d_part, g.blocks, 2, -1, c->d_scalars + 32, c->d_red, c->stream), "overlap sum");
        oa.mode = OBJ_OVERLAP;
        ADJ_CHECK(launch_objective(c->fp64, c->cfg.ncomp, oa, c->stream), "overlap grad");
        double ov[2];
        ADJ_CHECK(hipMemcpyAsync(ov, c->d_scalars + 32, sizeof(ov), hipMemcpyDeviceToHost, c->stream), "adjoint");
        ADJ_CHECK(hipStreamSynchronize(c->stream), "adjoint");
        J = ov[0] * ov[0] + ov[1] * ov[1];
    } else {
        gpe_observables_t o;
        int orc = gpe_observables(c, 0, &o);
        if (orc) {
            release();
            return orc;
        }
        if (spec->objective == GPE_OBJ_ENERGY) {
            J = o.energy;
            for (int k = 0; k < 3; ++k) explicit_mag[k] = o.magnetization[k];
            oa.mode = OBJ_EXPLICIT;
            ADJ_CHECK(launch_objective(c->fp64, c->cfg.ncomp, oa, c->stream), "explicit terms");
            ADJ_CHECK(launch_finalize(d_part, c->g.blocks, 4, -1, c->d_scalars + 40, c->d_red, c->stream), "explicit sums");
            ADJ_CHECK(hipMemcpyAsync(explicit_mom, c->d_scalars + 40, sizeof(explicit_mom), hipMemcpyDeviceToHost,
                                      c->stream), "adjoint");
            ADJ_CHECK(hipStreamSynchronize(c->stream), "adjoint");
            // H psi_N at the time of psi_N into mu[1], then scaled by 2 dv
            SweepArgs a = sweep_args(c, c->t0 + N * sdt, c->level[0], mu[1], 0.0);
            ADJ_CHECK(launch_sweep(c->fp64, c->cfg.ncomp, MODE_HPSI, a, c->stream), "H psi");
            oa.mode = OBJ_ENERGY;
        } else {
            J = o.magnetization[2];
            oa.mode = OBJ_MAGZ;
        }
        ADJ_CHECK(launch_objective(c->fp64, c->cfg.ncomp, oa, c->stream), "objective grad");
    }
    res->objective = J;

    // ---- backward pass over the segments, recomputing psi inside each
    // A = mu_{k+2}, B = mu_{k+1}
    void *A = mu[0], *B = mu[1];
    for (int j = nck - 1; j >= 0; --j) {
        const int klo = j * K, khi = std::min((j + 1) * K - 1, N - 1);
        seg[0] = ck[2 * j];
        seg[1] = ck[2 * j + 1];
        for (int m = klo + 1; m < khi && j < nck - 1; ++m) {  // psi_{m+1} = psi_{m-1} - 2i dt H psi_m
            SweepArgs a = sweep_args(c, c->t0 + m * sdt, seg[m - klo], seg[m + 1 - klo], 2.0 * sdt);
            a.prev = seg[m - 1 - klo];
            a.order = m & 1;
            ADJ_CHECK(launch_sweep(c->fp64, c->cfg.ncomp, MODE_UPDATE, a, c->stream), "recompute");
        }
        int qhi = khi, nq = 0;  // pending sweeps qhi, qhi - 1, ... in slots 0, 1, ...
        for (int k = khi; k >= klo; --k) {
            AdjArgs aa;
            aa.g = c->gs;
            aa.tb = tables(c);
            aa.ph = c->ph;
            aa.psi = seg[k - klo];
            aa.mu1 = B;
            aa.mu2 = A;
            aa.fields = c->d_fields;
            aa.sweep = k;
            aa.order = k & 1;
            aa.quad = quad_active(c);
            aa.coef = 2.0 * sdt;
            aa.partials = d_qpart + sweep_part * nq;
            ADJ_CHECK(launch_adjoint(c->fp64, c->cfg.ncomp, aa, c->stream), "adjoint sweep");
            if (++nq == Q || k == klo) {
                ADJ_CHECK(launch_sum_tables(d_qpart, nq, adj_blocks, ADJ_COUNT, d_steps + (size_t)ADJ_COUNT * qhi,
                                            -(long long)ADJ_COUNT, c->stream),
                          "adjoint sums");
                qhi = k - 1;
                nq = 0;
            }
            std::swap(A, B);
        }
    }
    std::vector<double> steps((size_t)ADJ_COUNT * N);
    ADJ_CHECK(hipMemcpyAsync(steps.data(), d_steps, sizeof(double) * steps.size(), hipMemcpyDeviceToHost, c->stream), "adjoint");
    ADJ_CHECK(hipEventRecord(c->ev1, c->stream), "adjoint");
    ADJ_CHECK(hipEventSynchronize(c->ev1), "adjoint");
    float bms = 0.f;
    ADJ_CHECK(hipEventElapsedTime(&bms, c->ev0, c->ev1), "adjoint");
    res->backward_ms = bms;
    release();

    // ---- chain rule to the parameters (FP64 on the host)
    for (int a = 0; a < 3; ++a) {
        res->grad_trap[a] = 0.0;
        res->grad_static_bb[a] = 0.0;
    }
    res->grad_static_bq = 0.0;
    const Ramp &r = c->ramp;
    if (res->grad_ramp_q)
        for (size_t j = 0; j < r.q_dur.size(); ++j) res->grad_ramp_q[j] = 0.0;
    if (res->grad_ramp_b)
        for (size_t j = 0; j < 3 * r.b_dur.size(); ++j) res->grad_ramp_b[j] = 0.0;
    for (int k = 0; k < N; ++k) {
        const double *p = &steps[(size_t)ADJ_COUNT * k];
        const double w = (k == 0) ? sdt : 2.0 * sdt;
        for (int a = 0; a < 3; ++a) res->grad_trap[a] += w * p[ADJ_WX + a];
        if (!r.active) {
            for (int a = 0; a < 3; ++a) res->grad_static_bb[a] += w * p[ADJ_BX + a];
            res->grad_static_bq += w * p[ADJ_BQ];
        } else {
            const double tr = (c->t0 + k * sdt) * r.time_scale;
            if (res->grad_ramp_q)
                for (size_t j = 0; j < r.q_dur.size(); ++j)
                    res->grad_ramp_q[j] += w * r.scale_q * ramp_basis(r.q_dur, r.q_type, r.tau, tr, (int)j) * p[ADJ_BQ];
            if (res->grad_ramp_b)
                for (size_t j = 0; j < r.b_dur.size(); ++j) {
                    const double phi = ramp_basis(r.b_dur, r.b_type, r.tau, tr, (int)j);
                    if (phi == 0.0) continue;
                    for (int a = 0; a < 3; ++a) res->grad_ramp_b[3 * j + a] += w * r.scale_b * phi * p[ADJ_BX + a];
                }
        }
    }
    if (spec->objective == GPE_OBJ_ENERGY) {
        // explicit dependence of E[psi_N] on the parameters at t_N
        const double tN = c->t0 + N * sdt;
        if (tN < c->ph.trap_off_time)
            for (int a = 0; a < 3; ++a) res->grad_trap[a] += c->ph.trap[a] * explicit_mom[a];
        if (c->cfg.ncomp > 1) {
            const double s = c->cfg.ncomp == 3 ? 1.0 : -1.0;
            if (!r.active) {
                for (int a = 0; a < 3; ++a) res->grad_static_bb[a] += s * explicit_mag[a];
                res->grad_static_bq += explicit_mom[3];
            } else {
                const double tr = tN * r.time_scale;
                if (res->grad_ramp_q)
                    for (size_t j = 0; j < r.q_dur.size(); ++j)
                        res->grad_ramp_q[j] += r.scale_q * ramp_basis(r.q_dur, r.q_type, r.tau, tr, (int)j) * explicit_mom[3];
                if (res->grad_ramp_b)
                    for (size_t j = 0; j < r.b_dur.size(); ++j) {
                        const double phi = ramp_basis(r.b_dur, r.b_type, r.tau, tr, (int)j);
                        for (int a = 0; a < 3; ++a) res->grad_ramp_b[3 * j + a] += r.scale_b * phi * s * explicit_mag[a];
                    }
            }
        }
    }
#undef ADJ_CHECK
    return GPE_OK;
}

int gpe_release_workspace(gpe_ctx *c)
{
    if (!c) return GPE_EINVAL;
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    drop_workspace(&c->ws);
    return GPE_OK;
}

// ------------------------------------------------------------------------- ensembles ---

// Members sharing (face degree, x per lane) form a group launched by one specialised kernel.
struct EnsembleGroup {
    int deg, form;      // face degree and lane_form of every member
    int first, count;   // members [first, first + count) of the sorted member list
    int blocks;         // workgroups of the group's launch
};

struct gpe_ensemble {
    std::vector<gpe_ctx *> m;          // sorted by group
    std::vector<Geometry> trav;        // each member's sweep traversal when the ensemble was made
    std::vector<std::pair<int, int>> span;  // each member's first workgroup and workgroups in its launch
    std::vector<EnsembleGroup> groups;
    EnsembleMember *d = nullptr;  // records and fields of the current call (up_bytes)
    char *up = nullptr;           // their pinned staging
    size_t up_bytes = 0;
    int *d_base = nullptr;
    int ncomp = 0, fp64 = 0, per = 1;
    hipStream_t stream = nullptr;
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    int graph_sweeps = 0;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_ms = 0.0, unknowns = 0.0;
    std::string err;
};

static int ens_fail(gpe_ensemble *e, int code, const std::string &what)
{
    if (e) e->err = what;
    return code;
}

int gpe_ensemble_create(gpe_ctx *const *members, int n, gpe_ensemble **out)
{
    if (!members || n < 1 || !out) return GPE_EINVAL;
    *out = nullptr;
    gpe_ctx *c0 = members[0];
    for (int i = 0; i < n; ++i) {
        gpe_ctx *c = members[i];
        if (!c) return GPE_EINVAL;
        if (c->cfg.ncomp != c0->cfg.ncomp || c->fp64 != c0->fp64 || c->cfg.scheme != c0->cfg.scheme ||
            c->device != c0->device)
            return GPE_EINVAL;
        if (!c->level1_valid) return GPE_ESTATE;
    }
    gpe_ensemble *e = new (std::nothrow) gpe_ensemble();
    if (!e) return GPE_ENOMEM;
    e->m.assign(members, members + n);
    std::stable_sort(e->m.begin(), e->m.end(), [](const gpe_ctx *a, const gpe_ctx *b) {
        const auto key = [](const Geometry &g) {
            return std::make_tuple(g.deg, lane_form(g.xpl, g.rows), g.blocks >= ENS_SOLO_BLOCKS);
        };
        return key(a->gs) < key(b->gs);
    });
    e->ncomp = c0->cfg.ncomp;
    e->fp64 = c0->fp64;
    e->per = c0->cfg.scheme == GPE_SCHEME_STAGGERED ? 2 : 1;
    int begin = 0;
    bool prev_solo = false;
    for (int i = 0; i < n; ++i) {
        const gpe_ctx *c = e->m[i];
        const int form = lane_form(c->gs.xpl, c->gs.rows);
        const bool solo = c->gs.blocks >= ENS_SOLO_BLOCKS;
        if (i == 0 || solo || prev_solo || c->gs.deg != e->groups.back().deg || form != e->groups.back().form ||
            e->groups.back().count == ENS_GROUP_MAX) {
            e->groups.push_back(EnsembleGroup{c->gs.deg, form, i, 0, 0});
            begin = 0;
        }
        prev_solo = solo;
        e->groups.back().count += 1;
        e->span.emplace_back(begin, c->gs.blocks);
        begin += (c->gs.blocks + 7) / 8 * 8;
        e->groups.back().blocks = begin;
        e->trav.push_back(c->gs);
        e->unknowns += (double)c->cfg.nx * c->cfg.ny * c->cfg.nz * c->g.V;
    }
    int rc = GPE_OK;
    if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess) rc = GPE_EDEVICE;
    if (!rc && device_malloc((void **)&e->d_base, sizeof(int) * 4, c0->device) != hipSuccess) rc = GPE_ENOMEM;
    if (!rc && (hipEventCreate(&e->ev0) != hipSuccess || hipEventCreate(&e->ev1) != hipSuccess)) rc = GPE_EDEVICE;
    if (rc) {
        gpe_ensemble_destroy(e);
        return rc;
    }
    *out = e;
    return GPE_OK;
}

int gpe_ensemble_destroy(gpe_ensemble *e)
{
    if (!e) return GPE_EINVAL;
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    if (e->gexec) (void)hipGraphExecDestroy(e->gexec);
    if (e->graph) (void)hipGraphDestroy(e->graph);
    if (e->d) (void)hipFree(e->d);
    if (e->up) (void)hipHostFree(e->up);
    if (e->d_base) (void)hipFree(e->d_base);
    if (e->ev0) (void)hipEventDestroy(e->ev0);
    if (e->ev1) (void)hipEventDestroy(e->ev1);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
    return GPE_OK;
}

const char *gpe_ensemble_last_error(const gpe_ensemble *e) { return e ? e->err.c_str() : "null ensemble"; }

#define ENSCALL(e, call)                                                                      \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess) return ens_fail(e, GPE_EDEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

int gpe_ensemble_step(gpe_ensemble *e, int nsteps, int graph_sweeps)
{
    if (!e) return GPE_EINVAL;
    if (nsteps < 0) return ens_fail(e, GPE_EINVAL, "negative step count");
    const int nsw = nsteps * e->per;
    if (nsw == 0) return GPE_OK;
    if (graph_sweeps < 0 || (graph_sweeps > 0 && (graph_sweeps % 2 != 0 || nsw % graph_sweeps != 0)))
        return ens_fail(e, GPE_EINVAL, "graph_sweeps must be even and divide the sweep count");
    for (size_t i = 0; i < e->m.size(); ++i) {
        gpe_ctx *c = e->m[i];
        if (!c->level1_valid) return ens_fail(e, GPE_ESTATE, "member not started");
        const Geometry &t = e->trav[i];
        if (c->gs.blocks != t.blocks || c->gs.xpl != t.xpl || c->gs.rows != t.rows || c->gs.ty != t.ty ||
            c->gs.xcd_remap != t.xcd_remap || c->gs.v_inner != t.v_inner)
            return ens_fail(e, GPE_ESTATE, "member traversal changed after the ensemble was created");
        ENSCALL(e, hipStreamSynchronize(c->stream));
    }
    // the members' records and the fields of all their sweeps go up in one copy: members first, then
    // member i's fields at i nsw
    const size_t rec = (sizeof(EnsembleMember) * e->m.size() + 255) / 256 * 256;
    const size_t bytes = rec + sizeof(FieldRec) * e->m.size() * (size_t)nsw;
    if (bytes > e->up_bytes) {
        if (e->d) (void)hipFree(e->d);
        if (e->up) (void)hipHostFree(e->up);
        e->d = nullptr;
        e->up = nullptr;
        e->up_bytes = 0;
        if (e->gexec) (void)hipGraphExecDestroy(e->gexec);  // captured with the old records' address
        e->gexec = nullptr;
        ENSCALL(e, device_malloc((void **)&e->d, bytes, e->m[0]->device));
        ENSCALL(e, hipHostMalloc((void **)&e->up, bytes, hipHostMallocDefault));
        e->up_bytes = bytes;
    }
    EnsembleMember *h = (EnsembleMember *)e->up;
    FieldRec *hf = (FieldRec *)(e->up + rec);
    const FieldRec *df = (const FieldRec *)((const char *)e->d + rec);
    for (size_t i = 0; i < e->m.size(); ++i) {
        gpe_ctx *c = e->m[i];
        const double coef = 2.0 * sweep_dt(c), sdt = sweep_dt(c);
        h[i].begin = e->span[i].first;
        h[i].blocks = e->span[i].second;
        for (int p = 0; p < 2; ++p) {
            h[i].args[p] = sweep_args(c, time_of(c, 0), c->level[p], c->level[1 - p], coef);
            h[i].args[p].fields = df + i * nsw;
        }
        for (int k = 0; k < nsw; ++k) hf[i * nsw + k] = field_at(c, c->t0 + (double)(c->sweeps + k) * sdt);
    }
    ENSCALL(e, hipMemcpyAsync(e->d, e->up, bytes, hipMemcpyHostToDevice, e->stream));
    // one launch per group per sweep; groups are independent of each other
    auto launch_group = [&](const EnsembleGroup &gr, int k, const int *base, hipStream_t st) -> hipError_t {
        EnsembleArgs a;
        a.members = e->d + gr.first;
        a.nmember = gr.count;
        a.parity = k & 1;
        a.sweep = k;
        a.sweep_base = base;
        for (int i = 0; i < gr.count; ++i) a.begin[i] = e->span[gr.first + i].first;
        return launch_ensemble_sweep(e->fp64, e->ncomp, gr.deg, gr.form, a, gr.blocks, st);
    };
    auto launch_all = [&](int k, const int *base) -> hipError_t {
        for (const EnsembleGroup &gr : e->groups) {
            hipError_t err = launch_group(gr, k, base, e->stream);
            if (err != hipSuccess) return err;
        }
        return hipSuccess;
    };
    // K sweeps of every group, one group after another: chains of independent groups forked
    // onto concurrent streams ran 3% slower (their kernels share each XCD's L2)
    auto capture_chains = [&](int K) -> hipError_t {
        hipError_t err = hipSuccess;
        for (size_t g = 0; g < e->groups.size() && err == hipSuccess; ++g)
            for (int k = 0; k < K && err == hipSuccess; ++k) err = launch_group(e->groups[g], k, e->d_base, e->stream);
        return err;
    };
    ENSCALL(e, hipEventRecord(e->ev0, e->stream));
    if (graph_sweeps > 0) {
        if (!e->gexec || e->graph_sweeps != graph_sweeps) {
            if (e->gexec) (void)hipGraphExecDestroy(e->gexec);
            if (e->graph) (void)hipGraphDestroy(e->graph);
            e->gexec = nullptr;
            e->graph = nullptr;
            ENSCALL(e, hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
            hipError_t cap = capture_chains(graph_sweeps);
            if (cap == hipSuccess) cap = launch_advance_base(e->d_base, graph_sweeps, e->stream);
            hipGraph_t captured = nullptr;
            const hipError_t end = hipStreamEndCapture(e->stream, &captured);
            if (cap != hipSuccess || end != hipSuccess) {
                if (captured) (void)hipGraphDestroy(captured);
                return ens_fail(e, GPE_EDEVICE, std::string("graph capture: ") +
                                                    hipGetErrorString(cap != hipSuccess ? cap : end));
            }
            e->graph = captured;
            ENSCALL(e, hipGraphInstantiate(&e->gexec, e->graph, nullptr, nullptr, 0));
            e->graph_sweeps = graph_sweeps;
        }
        ENSCALL(e, launch_set_base(e->d_base, 0, e->stream));
        for (int r = 0; r < nsw / graph_sweeps; ++r) ENSCALL(e, hipGraphLaunch(e->gexec, e->stream));
    } else {
        for (int k = 0; k < nsw; ++k) ENSCALL(e, launch_all(k, nullptr));
    }
    ENSCALL(e, hipEventRecord(e->ev1, e->stream));
    ENSCALL(e, wait_event(e->ev1));
    float ms = 0.f;
    ENSCALL(e, hipEventElapsedTime(&ms, e->ev0, e->ev1));
    e->last_ms = ms / nsw;
    for (gpe_ctx *c : e->m) {
        if (nsw & 1) std::swap(c->level[0], c->level[1]);
        c->sweeps += nsw;
    }
    return GPE_OK;
}

int gpe_ensemble_timing(const gpe_ensemble *e, double *ms_per_sweep, double *unknowns)
{
    if (!e) return GPE_EINVAL;
    if (ms_per_sweep) *ms_per_sweep = e->last_ms;
    if (unknowns) *unknowns = e->unknowns;
    return GPE_OK;
}

// ------------------------------------------------------------------------ autotuning ---

// Apply a traversal to both geometries; on failure (a workgroup count past the 2^29 limit of
// the decode) both are left as they were and false is returned.  flags: bit 0 the XCD remap,
// bit 1 the unknown v inside the x segment in the traversal order.
static bool set_traversal(gpe_ctx *c, int ty, int flags, int xpl)
{
    Geometry g = c->g, gs = c->gs;
    gs.xpl = xpl;
    for (Geometry *p : {&g, &gs}) {
        p->ty = ty;
        p->xcd_remap = flags & 1;
        p->v_inner = (flags >> 1) & 1;
        if (!finish_geometry(*p, p == &gs && c->fp64)) return false;
    }
    c->g = g;
    c->gs = gs;
    return true;
}

// Apply a traversal with room for its reduction partials; where that fails the context keeps the
// traversal and the partials it had.
static int change_traversal(gpe_ctx *c, int ty, int flags, int xpl)
{
    const Geometry g = c->g, gs = c->gs;
    const size_t before = partials_bytes(c);
    if (!set_traversal(c, ty, flags, xpl))
        return fail(c, GPE_EINVAL, "traversal needs more workgroups than the decode supports");
    if (partials_bytes(c) <= before) return GPE_OK;
    double *grown = nullptr;
    hipError_t e = device_malloc((void **)&grown, partials_bytes(c), c->device);
    const int code = e == hipSuccess ? GPE_EDEVICE : GPE_ENOMEM;
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) {
        if (grown) (void)hipFree(grown);
        c->g = g;
        c->gs = gs;
        return fail(c, code, "partials");
    }
    (void)hipFree(c->d_partials);
    c->d_partials = grown;
    return GPE_OK;
}

int gpe_set_traversal(gpe_ctx *c, int tile_rows, int xcd_remap, int x_per_lane)
{
    if (!c) return GPE_EINVAL;
    if (tile_rows < 1 || tile_rows > 1024 || xcd_remap < 0 || xcd_remap > 3 || (x_per_lane != 1 && x_per_lane != 2))
        return fail(c, GPE_EINVAL, "bad traversal");
    if (x_per_lane == 2 && !pair_lanes_ok(c->fp64, c->g.deg, c->cfg.ncomp))
        return fail(c, GPE_EINVAL, "two x per lane needs FP32");
    return change_traversal(c, tile_rows, xcd_remap, x_per_lane);
}

int gpe_traversal(const gpe_ctx *c, int *tile_rows, int *xcd_remap, int *x_per_lane)
{
    if (!c) return GPE_EINVAL;
    if (tile_rows) *tile_rows = c->gs.ty;
    if (xcd_remap) *xcd_remap = c->gs.xcd_remap | (c->gs.v_inner << 1);
    if (x_per_lane) *x_per_lane = c->gs.xpl;
    return GPE_OK;
}

static bool plan_arguments_ok(const gpe_config *cfg, int tile_rows, int xcd_remap, int x_per_lane, gpe_traversal_plan *out)
{
    if (!cfg || !out) return false;
    if (cfg->lattice < 0 || cfg->lattice > 5 || (cfg->ncomp != 1 && cfg->ncomp != 3 && cfg->ncomp != 5)) return false;
    if (cfg->precision != GPE_FP32 && cfg->precision != GPE_FP64) return false;
    if (cfg->nx < 1 || cfg->ny < 1 || cfg->nz < 1) return false;
    if (tile_rows < 1 || tile_rows > 1024 || xcd_remap < 0 || xcd_remap > 3) return false;
    return x_per_lane == 1 || (x_per_lane == 2 && pair_lanes_ok(cfg->precision == GPE_FP64, kLattices[cfg->lattice].deg, cfg->ncomp));
}

static void write_plan(const Geometry &g, gpe_traversal_plan *out)
{
    out->nx = g.nx;
    out->ny = g.ny;
    out->nz = g.nz;
    out->V = g.V;
    out->C = g.C;
    out->x_per_lane = g.xpl;
    out->rows = g.rows;
    out->pairs = g.pairs;
    out->nseg = g.nseg;
    out->tile_rows = g.ty;
    out->row_groups = g.tyr;
    out->ntile = g.ntile;
    out->xcd_remap = g.xcd_remap | (g.v_inner << 1);
    out->lx = g.lx;
    out->slabs = g.slabs;
    out->ys = g.ys;
    out->vs = g.vs;
    out->cs = g.cs;
    out->zs = g.zs;
    out->waves = g.waves;
    out->blocks = g.blocks;
    const FastDiv *d[5] = {&g.f_nseg, &g.f_V, &g.f_ty, &g.f_nz, &g.f_pairs};
    unsigned *o[5] = {out->div_nseg, out->div_V, out->div_rows, out->div_nz, out->div_pairs};
    for (int k = 0; k < 5; ++k) {
        o[k][0] = d[k]->d;
        o[k][1] = d[k]->m;
        o[k][2] = d[k]->l;
    }
}

static int plan(const gpe_config *cfg, int tile_rows, int xcd_remap, int x_per_lane, bool pack, gpe_traversal_plan *out)
{
    Geometry g = base_geometry(*cfg);
    g.ty = tile_rows;
    g.xcd_remap = xcd_remap & 1;
    g.v_inner = (xcd_remap >> 1) & 1;
    g.xpl = x_per_lane;
    if (!finish_geometry(g, pack)) return GPE_EINVAL;
    write_plan(g, out);
    return GPE_OK;
}

int gpe_plan_traversal(const gpe_config *cfg, int tile_rows, int xcd_remap, int x_per_lane, gpe_traversal_plan *out)
{
    if (!plan_arguments_ok(cfg, tile_rows, xcd_remap, x_per_lane, out)) return GPE_EINVAL;
    return plan(cfg, tile_rows, xcd_remap, x_per_lane, false, out);
}

int gpe_plan_sweep(const gpe_config *cfg, int tile_rows, int xcd_remap, int x_per_lane, gpe_traversal_plan *out)
{
    const bool untuned = tile_rows == 0;
    if (!plan_arguments_ok(cfg, untuned ? 1 : tile_rows, untuned ? 0 : xcd_remap, untuned ? 1 : x_per_lane, out))
        return GPE_EINVAL;
    const int fp64 = cfg->precision == GPE_FP64;
    if (!untuned) return plan(cfg, tile_rows, xcd_remap, x_per_lane, fp64, out);
    Geometry g = untuned_geometry(*cfg);
    if (!finish_geometry(g, fp64)) return GPE_EINVAL;
    write_plan(g, out);
    return GPE_OK;
}

typedef std::tuple<int, int, int, int, int, int> TuneKey;
static std::map<TuneKey, std::tuple<int, int, int>> g_tune_cache;  // rows, remap, x per lane
static std::mutex g_tune_mutex;

int gpe_autotune(gpe_ctx *c, int trial_sweeps, int *tile_rows, int *xcd_remap, int *x_per_lane, double *ms_out)
{
    if (!c) return GPE_EINVAL;
    if (trial_sweeps < 0) return fail(c, GPE_EINVAL, "negative trial sweeps");
    const TuneKey key(c->cfg.lattice, c->cfg.ncomp, c->fp64, c->cfg.nx, c->cfg.ny, c->cfg.nz);
    int best_ty = c->gs.ty, best_remap = c->gs.xcd_remap | (c->gs.v_inner << 1), best_xpl = c->gs.xpl;
    double best_ms = -1.0;
    bool chosen = trial_sweeps > 0;  // otherwise the context keeps what it has
    {
        std::lock_guard<std::mutex> lk(g_tune_mutex);
        auto it = g_tune_cache.find(key);
        if (it != g_tune_cache.end()) {
            std::tie(best_ty, best_remap, best_xpl) = it->second;
            trial_sweeps = 0;
            chosen = true;
        }
    }
    if (trial_sweeps > 0) {
        const size_t lbytes = (size_t)c->level_elems * c->elem_bytes;
        // scratch copies of the two levels, freed when the trials end (also on failure), when
        // the context's traversal on entry is restored too (the winner is applied below)
        struct Trial {
            gpe_ctx *c;
            Geometry g, gs;
            void *s0 = nullptr, *s1 = nullptr;
            ~Trial()
            {
                if (s0 || s1) (void)hipStreamSynchronize(c->stream);
                if (s0) (void)hipFree(s0);
                if (s1) (void)hipFree(s1);
                c->g = g;
                c->gs = gs;
            }
        } trial{c, c->g, c->gs};
        if (device_malloc(&trial.s0, lbytes, c->device) != hipSuccess ||
            device_malloc(&trial.s1, lbytes, c->device) != hipSuccess)
            return fail(c, GPE_ENOMEM, "autotune scratch does not fit");
        HIPCALL(c, hipMemcpyAsync(trial.s0, c->level[0], lbytes, hipMemcpyDeviceToDevice, c->stream));
        HIPCALL(c, hipMemcpyAsync(trial.s1, c->level[1], lbytes, hipMemcpyDeviceToDevice, c->stream));
        // tile heights: powers of two, and multiples of 3, 5, 6 and 7 rows, which are
        // candidates only where their row groups are not powers of two; and the whole plane
        // (one tile: each XCD a range of planes that share their y neighbours in its L2;
        // FP32 A15 82^3 one component +17%, spin-2 +8%, Cube 293^3 one component +11%)
        // the height of an untuned sweep comes first, whatever it is: without it the fastest candidate
        // can be slower than not tuning (lanes used, untuned against the best other candidate: FCC 19^3
        // spin-1 99% and 74%, A15 9x11x9 86% and 43%, FP64 FCC 17^3 90% and 50%)
        std::vector<int> tys = {1, 2, 4, 8, 16, 32, 3, 6, 12, 24, 5, 10, 20, 7, 14, 28};
        if (c->g.ny > 32 && c->g.ny <= 1024) tys.push_back(c->g.ny);
        const Geometry untuned = untuned_geometry(c->cfg);
        const int untuned_ty = untuned.ty;
        tys.erase(std::remove(tys.begin(), tys.end(), untuned_ty), tys.end());
        tys.insert(tys.begin(), untuned_ty);
        const int nxpl = pair_lanes_ok(c->fp64, c->g.deg, c->cfg.ncomp) ? 2 : 1;
        for (int xpl = 1; xpl <= nxpl; ++xpl)
        for (int ty : tys) {
            if (ty > c->g.ny && ty != 1) continue;
            const bool any_rows = (ty & (ty - 1)) == 0 || (ty == untuned_ty && xpl == untuned.xpl);
            // flags: XCD remap, and the unknown inside the x segment (only where lines span several waves)
            for (int remap = 0; remap < 4; ++remap) {
                if (!set_traversal(c, ty, remap, xpl)) continue;  // too many workgroups: not a candidate
                if (!any_rows && (xpl == 1 || (c->gs.rows & (c->gs.rows - 1)) == 0)) continue;
                if ((remap & 2) && c->gs.nseg == 1) continue;
                void *cur = trial.s0, *nxt = trial.s1;
                for (int k = 0; k < trial_sweeps + 2; ++k) {
                    if (k == 2) HIPCALL(c, hipEventRecord(c->ev0, c->stream));
                    SweepArgs a = sweep_args(c, time_of(c, 0), cur, nxt, 2.0 * sweep_dt(c));
                    a.order = k & 1;
                    hipError_t e = launch_sweep(c->fp64, c->cfg.ncomp, MODE_UPDATE, a, c->stream);
                    if (e != hipSuccess) return hip_fail(c, e, "autotune sweep");
                    std::swap(cur, nxt);
                }
                HIPCALL(c, hipEventRecord(c->ev1, c->stream));
                HIPCALL(c, hipEventSynchronize(c->ev1));
                float ms = 0.f;
                HIPCALL(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
                const double per = ms / trial_sweeps;
                if (best_ms < 0 || per < best_ms) {
                    best_ms = per;
                    best_ty = c->g.ty;
                    best_remap = remap;
                    best_xpl = xpl;
                }
            }
        }
        std::lock_guard<std::mutex> lk(g_tune_mutex);
        g_tune_cache[key] = std::make_tuple(best_ty, best_remap, best_xpl);
    }
    const int rc = chosen ? change_traversal(c, best_ty, best_remap, best_xpl) : GPE_OK;
    if (rc) return rc;
    if (tile_rows) *tile_rows = best_ty;
    if (xcd_remap) *xcd_remap = best_remap;
    if (x_per_lane) *x_per_lane = best_xpl;
    if (ms_out) *ms_out = best_ms;
    return GPE_OK;
}

int gpe_stream_bandwidth(long long bytes, int reps, double *copy_gbs, double *update_gbs)
{
    if (bytes < (1 << 20) || reps < 1) return GPE_EINVAL;
    bytes = bytes / 16 * 16;
    void *a = nullptr, *b = nullptr;
    hipStream_t s = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = GPE_OK;
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) rc = GPE_EDEVICE;
    if (!rc && (device_malloc(&a, bytes, device) != hipSuccess || device_malloc(&b, bytes, device) != hipSuccess))
        rc = GPE_ENOMEM;
    if (!rc && (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess || hipEventCreate(&e0) != hipSuccess ||
                hipEventCreate(&e1) != hipSuccess))
        rc = GPE_EDEVICE;
    if (!rc && (hipMemsetAsync(a, 0, bytes, s) != hipSuccess || hipMemsetAsync(b, 0, bytes, s) != hipSuccess))
        rc = GPE_EDEVICE;
    double *out[2] = {copy_gbs, update_gbs};
    const double moved[2] = {2.0 * bytes, 3.0 * bytes};
    for (int kind = 0; kind < 2 && !rc; ++kind) {
        bool ok = launch_stream(kind, a, b, bytes / 16, s) == hipSuccess && hipEventRecord(e0, s) == hipSuccess;
        for (int r = 0; r < reps && ok; ++r) ok = launch_stream(kind, a, b, bytes / 16, s) == hipSuccess;
        ok = ok && hipEventRecord(e1, s) == hipSuccess && hipEventSynchronize(e1) == hipSuccess;
        float ms = 0.f;
        ok = ok && hipEventElapsedTime(&ms, e0, e1) == hipSuccess;
        if (!ok) rc = GPE_EDEVICE;
        else if (out[kind]) *out[kind] = moved[kind] * reps / (ms * 1e-3) / 1e9;
    }
    if (s) (void)hipStreamSynchronize(s);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (a) (void)hipFree(a);
    if (b) (void)hipFree(b);
    if (s) (void)hipStreamDestroy(s);
    return rc;
}

int gpe_last_step_timing(const gpe_ctx *c, double *ms_per_sweep, double *bytes_per_sweep)
{
    if (!c) return GPE_EINVAL;
    if (ms_per_sweep) *ms_per_sweep = c->last_ms_per_sweep;
    if (bytes_per_sweep) {
        const double n = (double)c->cfg.nx * c->cfg.ny * c->cfg.nz * c->g.V;
        *bytes_per_sweep = n * 3.0 * c->cfg.ncomp * 2.0 * (c->fp64 ? 8.0 : 4.0);
    }
    return GPE_OK;
}

}  // extern "C"
