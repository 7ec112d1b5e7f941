// HIP kernels of the DEC Gross-Pitaevskii step for CDNA4 (gfx950).
//
// One sweep = one pass over every unknown of a time level:
//     next += coef * (-i) H(cur)           (3-level leapfrog, Spin1GpeBCC.cu:793-917;
//                                           staggered half-step, GPBlocks.cpp:560-606)
// with H = -1/2 L + V(r) + c0 n [-i alpha n^2] + (c1 F +- B).f + singlet + quadratic Zeeman.
//
// Work mapping: a wave owns 64 consecutive x of one (z, y, unknown v) line of the device
// layout (gpe_internal.h), so the face table row, the neighbour line (z+dz, y+dy, target)
// and the field are wave-uniform (scalar loads), and each neighbour access is one
// contiguous 64-lane load shifted by dx.  Out-of-box neighbours are folded into the face
// weight (weight 0 and a clamped in-bounds address), so the sweep has no branches.
// Workgroups are remapped so that each XCD walks a contiguous slab of the traversal
// order (y-tiles, then z, then rows of the tile): the z +- 1 and y +- 1 rows a wave needs
// were fetched into the same XCD's L2 by its neighbours shortly before.
#include "gpe_device.h"

namespace gpe {

// ------------------------------------------------------------------------- the sweep --

// Physics and field constants of one sweep in the sweep's precision: the FP32 copies made on
// the host for FP32 (no per-wave conversions), the FP64 values for FP64.
template <typename R>
struct LocalConsts {
    R cell[3], p0[3], trap2[3], trap_offset, center[3], c0, c1, c2, alpha, quad_sign, q;
    R bq, bb[3], bqq, bbq[3], sigma, ksc;
};

template <typename R>
__device__ __forceinline__ LocalConsts<R> local_consts(const Physics &ph, const const_ptr<FieldRec> fr)
{
    LocalConsts<R> k;
    if constexpr (std::is_same<R, float>::value) {
        const PhysicsF &f = ph.f;
        for (int i = 0; i < 3; ++i) {
            k.cell[i] = f.cell[i];
            k.p0[i] = f.p0[i];
            k.trap2[i] = f.trap2[i];
            k.center[i] = f.center[i];
            k.bb[i] = fr->fbb[i];
            k.bbq[i] = fr->fbbq[i];
        }
        k.trap_offset = f.trap_offset;
        k.c0 = f.c0;
        k.c1 = f.c1;
        k.c2 = f.c2;
        k.alpha = f.alpha;
        k.quad_sign = f.quad_sign;
        k.q = f.q;
        k.bq = fr->fbq;
        k.bqq = fr->fbqq;
        k.sigma = fr->fsigma;
        k.ksc = fr->fksc;
    } else {
        for (int i = 0; i < 3; ++i) {
            k.cell[i] = ph.cell[i];
            k.p0[i] = ph.p0[i];
            k.trap2[i] = ph.trap2[i];
            k.center[i] = ph.center[i];
            k.bb[i] = fr->bb[i];
            k.bbq[i] = fr->bbq[i];
        }
        k.trap_offset = ph.trap_offset;
        k.c0 = ph.c0;
        k.c1 = ph.c1;
        k.c2 = ph.c2;
        k.alpha = ph.alpha;
        k.quad_sign = ph.quad_sign;
        k.q = ph.q;
        k.bq = fr->bq;
        k.bqq = fr->bqq;
        k.sigma = fr->sigma;
        k.ksc = 1.0 / (fr->sigma * fr->sigma);
    }
    return k;
}

// One x value per lane (FP64, and FP32 where the neighbour pairs would not fit).
// ROWS: the wave's lanes lie in a group of g.rows consecutive y rows of one (z, v), as in
// sweep_body_pair: y0 is the group's first row and a lane's offsets are from its line.
template <typename R, int C, int DEG, int MODE, bool ROWS, int NIN, typename Field>
__device__ __forceinline__ void sweep_body_single(const SweepArgs &a, const Field &field, int b, int nb)
{
    using V2 = vec2_t<R>;
    const Geometry &g = a.g;
    const LaneCoord lc = lane_coord<ROWS>(g, b, nb);
    double part = 0.0;

    if (lc.valid) {
        const int x = lc.x, v = lc.v, y = lc.y, z = lc.z;
        const bool act = lc.act;
        const int xc = lc.at;  // the lane's offset from the line of row y0 (its own x, clamped into the box)
        const V2 *__restrict__ cur = (const V2 *)a.cur;
        V2 *__restrict__ nxt = (V2 *)a.next;
        const V2 *__restrict__ prv = (const V2 *)(a.prev ? a.prev : a.next);
        const long long cstride = comp_stride(g);  // elements between components of a line
        const long long own_line = line_index(g, 0, z, lc.y0, v);

        // issue every load of the wave before any use: own values, psi_{k-1}, and the
        // DEG neighbour lines (wave-uniform line bases, per-lane 32-bit offsets)
        R pr[C], pi[C], qr[C], qi[C], ar[C], ai[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const V2 o = cur[own_line + c * cstride + xc];
            pr[c] = o.x;
            pi[c] = o.y;
            ar[c] = 0;
            ai[c] = 0;
        }
        if constexpr (MODE == MODE_UPDATE) {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const V2 o = nt_load<R>(&prv[own_line + c * cstride + xc]);
                qr[c] = o.x;
                qi[c] = o.y;
            }
        }
        const int2 *fx = (const int2 *)a.tb.facex + v * DEG;  // (packed face, line offset) pairs
        int face[DEG], fd[DEG];
#pragma unroll
        for (int f = 0; f < DEG; ++f) {
            const int2 e = fx[f];
            face[f] = e.x;
            fd[f] = e.y;
        }
        const R *wt = table_w<R>(a.tb) + v * DEG;
        R wu[DEG];    // weight: 0 when the neighbour's y or z is outside the box (wave-uniform unless ROWS)
        bool xok[DEG];
        int dxf[DEG];
        const V2 *nbase[DEG];
        int noff[DEG];
        face_lanes<R, DEG, ROWS>(g, lc, cur + own_line, face, fd, wt, wu, xok, dxf, nbase, noff);
        // degree-8 tables pad some unknowns with zero-weight faces: skip their loads
        const int nf = DEG == 8 ? a.tb.nface[v] : DEG;
        V2 nb[DEG - NIN][C];
#pragma unroll
        for (int f = NIN; f < DEG; ++f)
#pragma unroll
            for (int c = 0; c < C; ++c) {
                if (f < nf) {
                    nb[f - NIN][c] = nbase[f][c * cstride + noff[f]];
                } else {
                    nb[f - NIN][c].x = 0;
                    nb[f - NIN][c].y = 0;
                }
            }
        // stencil: sum_f w_f psi_t(f); out-of-box neighbours carry weight 0.  Same-x faces need
        // no per-lane test (a live lane's own x is inside the box): wave-uniform weight.
        if constexpr (NIN > 0) {
            __shared__ V2 ex[4][C][64];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                V2 o;
                o.x = pr[c];
                o.y = pi[c];
                ex[threadIdx.x >> 6][c][threadIdx.x & 63] = o;
            }
            exchange_barrier();
#pragma unroll
            for (int f = 0; f < NIN; ++f)
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const V2 o = ex[exchange_wave(f)][c][threadIdx.x & 63];
                    ar[c] += wt[f] * o.x;
                    ai[c] += wt[f] * o.y;
                }
        }
#pragma unroll
        for (int f = NIN; f < DEG; ++f) {
            const R w = (dxf[f] == 0 || xok[f]) ? wu[f] : (R)0;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                ar[c] += w * nb[f - NIN][c].x;
                ai[c] += w * nb[f - NIN][c].y;
            }
        }
        const R wsum = table_wsum<R>(a.tb)[v];
        const Physics &ph = a.ph;
        const const_ptr<FieldRec> fr = field();
        const LocalConsts<R> k = local_consts<R>(ph, fr);
        R hr[C], hi[C];
        R sc = (R)1;
        if constexpr (MODE == MODE_ITP) sc = (R)(*a.scale_in);
        const R sig = k.sigma;        // expanding grid: lengths x sigma
        const R ksc = sc * k.ksc;     // Laplacian / sigma^2
#pragma unroll
        for (int c = 0; c < C; ++c) {
            hr[c] = ksc * (ar[c] - wsum * pr[c]);
            hi[c] = ksc * (ai[c] - wsum * pi[c]);
            pr[c] *= sc;
            pi[c] *= sc;
        }
        // position, trap and field
        const R *pos = table_pos<R>(a.tb) + 3 * v;
        const R rx = k.p0[0] + sig * (k.cell[0] * (R)x + pos[0]);
        const R ry = k.p0[1] + sig * (k.cell[1] * (R)y + pos[1]);
        const R rz = k.p0[2] + sig * (k.cell[2] * (R)z + pos[2]);
        R vtrap = 0;
        if (fr->trap_on)
            vtrap = (R)0.5 * (k.trap2[0] * rx * rx + k.trap2[1] * ry * ry + k.trap2[2] * rz * rz) + k.trap_offset;
        R Bx = 0, By = 0, Bz = 0, Qx = 0, Qy = 0, Qz = 0;
        if constexpr (C > 1) {
            const R dxr = rx - k.center[0], dyr = ry - k.center[1], dzr = rz - k.center[2];
            Bx = k.bq * dxr + k.bb[0];
            By = k.bq * dyr + k.bb[1];
            Bz = (R)-2 * k.bq * dzr + k.bb[2];
            Qx = k.bqq * dxr + k.bbq[0];
            Qy = k.bqq * dyr + k.bbq[1];
            Qz = (R)-2 * k.bqq * dzr + k.bbq[2];
        }
        add_local_h<R, C>(pr, pi, vtrap, Bx, By, Bz, Qx, Qy, Qz, k.c0, k.c1, k.c2, k.alpha, k.quad_sign, k.q,
                          a.quad, a.loss, hr, hi);

        const R coef = (R)a.coef;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const long long idx = own_line + c * cstride + xc;
            V2 o;
            if constexpr (MODE == MODE_UPDATE) {
                o.x = qr[c] + coef * hi[c];
                o.y = qi[c] - coef * hr[c];
            } else if constexpr (MODE == MODE_EULER) {
                o.x = pr[c] + coef * hi[c];
                o.y = pi[c] - coef * hr[c];
            } else if constexpr (MODE == MODE_ITP) {
                o.x = pr[c] - coef * hr[c];
                o.y = pi[c] - coef * hi[c];
                if (act) part += (double)o.x * (double)o.x + (double)o.y * (double)o.y;
            } else {
                o.x = hr[c];
                o.y = hi[c];
            }
            if (act) nt_store<R>(o, &nxt[idx]);
        }
        if constexpr (MODE == MODE_ITP) part *= a.tb.dv[v];
    } else if constexpr (NIN > 0) {
        exchange_barrier();
    }

    if constexpr (MODE == MODE_ITP) {
        __shared__ double red[4];
        part = wave_sum(part);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = part;
        __syncthreads();
        if (threadIdx.x == 0) a.partials[b] = (red[0] + red[1]) + (red[2] + red[3]);
    }
}

// Two consecutive x values per lane (FP32): every access is one 16-byte load or store of a
// pair of complex values.  Lane l of segment s owns x0 = 128 s + 2 l and x0 + 1.  A
// neighbour pair starts at x0 + dx, which is 8-byte aligned only; the start is clamped to
// [0, lx - 2] (inside the line, so inside the allocation) and the two values are shifted
// back into place, and any value outside the box (x, y or z) is replaced by zero by a
// select, so the line padding x >= nx is never used whatever it holds.
// ROWS: the wave's pairs lie in a group of g.rows consecutive y rows of one (z, v); a lane's
// row is then a per-lane offset from the group's first row y0, a lane past the group or the box
// is clamped to the group's last row in the box and masked, and a neighbour row outside the
// box gets weight 0 per lane.
typedef float f4a __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(8)));
typedef float f2n __attribute__((ext_vector_type(2)));

template <int C, int DEG, int MODE, bool ROWS, int NIN, typename Field>
__device__ __forceinline__ void sweep_body_pair(const SweepArgs &a, const Field &field, int b, int nb)
{
    const Geometry &g = a.g;
    int x0, v, y0, z, r = 0;
    bool valid;
    if constexpr (ROWS) {
        const RowCoord rc = decode_rows<2>(g, b, nb);
        x0 = rc.x, v = rc.v, y0 = rc.y0, z = rc.z, r = rc.r, valid = rc.valid;
    } else {
        const WaveCoord wc = decode(g, b, nb);
        x0 = wc.x, v = wc.v, y0 = wc.y, z = wc.z, valid = wc.valid;
    }
    double part = 0.0;

    if (valid) {
        // the lane's row: y0 (+ r under ROWS, clamped into the box) at element offset roff
        bool rowok = true;
        int y = y0, roff = 0;
        const int rowstride = (int)g.ys;  // elements between rows y and y + 1
        int ylo = y0, yhi = y0;           // the rows of the wave's lanes
        if constexpr (ROWS) {
            const int nrow = g.ny - y0 < g.rows ? g.ny - y0 : g.rows;  // the group's rows in the box
            rowok = r < nrow;
            const int rr = rowok ? r : nrow - 1;
            y = y0 + rr;
            roff = rr * rowstride;
            // a lane's row grows with its lane number: lanes 0 and 63 bound the wave's rows
            const int r0 = __builtin_amdgcn_readfirstlane(rr), r63 = __builtin_amdgcn_readlane(rr, 63);
            ylo = y0 + r0;
            yhi = y0 + r63;
        }
        const bool act0 = rowok && x0 < g.nx, act1 = rowok && x0 + 1 < g.nx;
        const int xc = x0 < g.nx ? x0 : ((g.nx - 1) & ~1);  // even, so xc + 1 <= lx - 1
        const int lo = roff + xc;                            // lane offset from the row-y0 line
        const float2 *__restrict__ cur = (const float2 *)a.cur;
        float2 *__restrict__ nxt = (float2 *)a.next;
        const float2 *__restrict__ prv = (const float2 *)(a.prev ? a.prev : a.next);
        const long long cstride = comp_stride(g);
        const long long own_line = line_index(g, 0, z, y0, v);
        const int lxm2 = (int)g.lx - 2;

        float pr[2][C], pi[2][C], qr[2][C], qi[2][C], ar[2][C], ai[2][C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const f4a o = *(const f4a *)(cur + own_line + c * cstride + lo);
            pr[0][c] = o.x;
            pi[0][c] = o.y;
            pr[1][c] = o.z;
            pi[1][c] = o.w;
            ar[0][c] = ar[1][c] = 0.f;
            ai[0][c] = ai[1][c] = 0.f;
        }
        if constexpr (MODE == MODE_UPDATE) {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const f4a o = __builtin_nontemporal_load((const f4a *)(prv + own_line + c * cstride + lo));
                qr[0][c] = o.x;
                qi[0][c] = o.y;
                qr[1][c] = o.z;
                qi[1][c] = o.w;
            }
        }
        // packed face and own-line-to-neighbour-line offset side by side: one scalar load
        const int2 *fx = (const int2 *)a.tb.facex + v * DEG;
        int face[DEG], fd[DEG];
#pragma unroll
        for (int f = 0; f < DEG; ++f) {
            const int2 e = fx[f];
            face[f] = e.x;
            fd[f] = e.y;
        }
        const float *wt = a.tb.w32 + v * DEG;
        const float2 *nbase[DEG];
        int sh[DEG], dxf[DEG], scf[DEG];
        float wf[DEG];
        bool ok0[DEG], ok1[DEG];
#pragma unroll
        for (int f = 0; f < DEG; ++f) {
            const int dx = (face[f] & 3) - 1;
            dxf[f] = dx;
            const int s0 = xc + dx;
            const int sc = s0 < 0 ? 0 : (s0 > lxm2 ? lxm2 : s0);
            scf[f] = sc;
            sh[f] = s0 - sc;  // -1, 0 or +1
            ok0[f] = (unsigned)(x0 + dx) < (unsigned)g.nx;
            ok1[f] = (unsigned)(x0 + 1 + dx) < (unsigned)g.nx;
        }
        // a wave whose rows and plane are all inside [1, n - 2] has every y / z neighbour inside
        // the box: its neighbour lines are the own line plus the per-face offsets of the table
        if (z >= 1 && z <= g.nz - 2 && ylo >= 1 && yhi <= g.ny - 2) {
            const float2 *own = cur + own_line;
#pragma unroll
            for (int f = 0; f < DEG; ++f) {
                wf[f] = wt[f];
                nbase[f] = own + (fd[f] + roff + scf[f]);  // one 32-bit lane offset
            }
        } else {
#pragma unroll
            for (int f = 0; f < DEG; ++f) {
                const int pk = face[f];
                const int dy = ((pk >> 2) & 3) - 1, dz = ((pk >> 4) & 3) - 1, t = pk >> 8;
                int zn = z + dz, yn = y + dy;
                const bool inside = (unsigned)zn < (unsigned)g.nz && (unsigned)yn < (unsigned)g.ny;
                wf[f] = inside ? wt[f] : 0.f;  // wave-uniform unless ROWS: y / z outside the box
                if constexpr (ROWS) {
                    // row-y0 line of (zn, t), the lane's own row when the neighbour is outside
                    if ((unsigned)zn >= (unsigned)g.nz) zn = z;
                    nbase[f] = cur + line_index(g, 0, zn, y0, t) + (roff + (inside ? dy * rowstride : 0) + scf[f]);
                } else {
                    if (!inside) {
                        zn = z;
                        yn = y;
                    }
                    nbase[f] = cur + line_index(g, 0, zn, yn, t) + scf[f];
                }
            }
        }
        // degree-8 tables (FCC) pad the 4-face unknowns with 4 zero-weight faces: skip their
        // loads.  With 5 components the degree-8 faces go in two batches
        // of 4, so a wave holds one batch of neighbour pairs at a time (the second batch, loaded
        // after the first is summed and only by 8-face waves, cannot be hoisted past the
        // wave-uniform test): 159 instead of 228 VGPRs, 3 waves per SIMD instead of 2, +6-12% on
        // FCC boxes of 96-128 blocks; pairs over row groups of slab rows +1-1.5% on FCC 45-100^3.
        // Fewer components gain nothing from it.
        const int nf = DEG == 8 ? a.tb.nface[v] : DEG;
        constexpr int FB = (DEG == 8 && C == 5) ? 4 : DEG;
#pragma unroll
        for (int f0 = 0; f0 < DEG; f0 += FB) {
            if (f0 > 0 && f0 >= nf) break;
            constexpr int N0 = NIN;  // (exchanging tables have one batch)
            f4u nbv[FB - N0][C];
#pragma unroll
            for (int k = N0; k < FB; ++k)
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if (f0 + k < nf)
                        nbv[k - N0][c] = *(const f4u *)(nbase[f0 + k] + c * cstride);
                    else
                        nbv[k - N0][c] = (f4u)(0.f);
                }
            if constexpr (NIN > 0) {
                static_assert(NIN == 0 || FB == DEG, "one batch");
                __shared__ f4a ex[4][C][64];
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    f4a o;
                    o.x = pr[0][c];
                    o.y = pi[0][c];
                    o.z = pr[1][c];
                    o.w = pi[1][c];
                    ex[threadIdx.x >> 6][c][threadIdx.x & 63] = o;
                }
                exchange_barrier();
#pragma unroll
                for (int f = 0; f < NIN; ++f)
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        const f4a e = ex[exchange_wave(f)][c][threadIdx.x & 63];
                        ar[0][c] += wt[f] * e.x;
                        ai[0][c] += wt[f] * e.y;
                        ar[1][c] += wt[f] * e.z;
                        ai[1][c] += wt[f] * e.w;
                    }
            }
#pragma unroll
            for (int k = N0; k < FB; ++k) {
                const int f = f0 + k;
                const float w = wf[f];
                if (dxf[f] == 0) {
                    // same x: the pair is (x0, x0 + 1) unshifted; a live value's x is inside the
                    // box (the second value of a lone last x is never stored): no per-lane masks
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        const f4u e = nbv[k - N0][c];
                        ar[0][c] += w * e.x;
                        ai[0][c] += w * e.y;
                        ar[1][c] += w * e.z;
                        ai[1][c] += w * e.w;
                    }
                } else {
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        const f4u e = nbv[k - N0][c];
                        // values at x0 + dx and x0 + 1 + dx from the clamped pair
                        float n0r = sh[f] == 0 ? e.x : e.z, n0i = sh[f] == 0 ? e.y : e.w;
                        float n1r = sh[f] == 0 ? e.z : e.x, n1i = sh[f] == 0 ? e.w : e.y;
                        n0r = (ok0[f] && sh[f] >= 0) ? n0r : 0.f;
                        n0i = (ok0[f] && sh[f] >= 0) ? n0i : 0.f;
                        n1r = (ok1[f] && sh[f] <= 0) ? n1r : 0.f;
                        n1i = (ok1[f] && sh[f] <= 0) ? n1i : 0.f;
                        ar[0][c] += w * n0r;
                        ai[0][c] += w * n0i;
                        ar[1][c] += w * n1r;
                        ai[1][c] += w * n1i;
                    }
                }
            }
        }
        const float wsum = a.tb.wsum32[v];
        float sc = 1.f;
        if constexpr (MODE == MODE_ITP) sc = (float)(*a.scale_in);
        const Physics &ph = a.ph;
        const PhysicsF &pf = ph.f;
        const const_ptr<FieldRec> fr = field();
        const float sig = fr->fsigma;        // expanding grid: lengths x sigma
        const float ksc = sc * fr->fksc;     // Laplacian / sigma^2
        const float *pos = a.tb.pos32 + 3 * v;
        const float ry = pf.p0[1] + sig * (pf.cell[1] * (float)y + pos[1]);
        const float rz = pf.p0[2] + sig * (pf.cell[2] * (float)z + pos[2]);
        const bool trap_on = fr->trap_on != 0;
        const float coef = (float)a.coef;
        float2 out[2][C];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            float hr[C], hi[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                hr[c] = ksc * (ar[e][c] - wsum * pr[e][c]);
                hi[c] = ksc * (ai[e][c] - wsum * pi[e][c]);
                pr[e][c] *= sc;
                pi[e][c] *= sc;
            }
            const float rx = pf.p0[0] + sig * (pf.cell[0] * (float)(x0 + e) + pos[0]);
            float vtrap = 0.f;
            if (trap_on)
                vtrap = 0.5f * (pf.trap2[0] * rx * rx + pf.trap2[1] * ry * ry + pf.trap2[2] * rz * rz) +
                        pf.trap_offset;
            float Bx = 0, By = 0, Bz = 0, Qx = 0, Qy = 0, Qz = 0;
            if constexpr (C > 1) {
                const float dxr = rx - pf.center[0], dyr = ry - pf.center[1], dzr = rz - pf.center[2];
                Bx = fr->fbq * dxr + fr->fbb[0];
                By = fr->fbq * dyr + fr->fbb[1];
                Bz = -2.f * fr->fbq * dzr + fr->fbb[2];
                Qx = fr->fbqq * dxr + fr->fbbq[0];
                Qy = fr->fbqq * dyr + fr->fbbq[1];
                Qz = -2.f * fr->fbqq * dzr + fr->fbbq[2];
            }
            add_local_h<float, C>(pr[e], pi[e], vtrap, Bx, By, Bz, Qx, Qy, Qz, pf.c0, pf.c1, pf.c2, pf.alpha,
                                  pf.quad_sign, pf.q, a.quad, a.loss, hr, hi);
            const bool live = e == 0 ? act0 : act1;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                float2 o;
                if constexpr (MODE == MODE_UPDATE) {
                    o.x = qr[e][c] + coef * hi[c];
                    o.y = qi[e][c] - coef * hr[c];
                } else if constexpr (MODE == MODE_EULER) {
                    o.x = pr[e][c] + coef * hi[c];
                    o.y = pi[e][c] - coef * hr[c];
                } else if constexpr (MODE == MODE_ITP) {
                    o.x = pr[e][c] - coef * hr[c];
                    o.y = pi[e][c] - coef * hi[c];
                    if (live) part += (double)o.x * (double)o.x + (double)o.y * (double)o.y;
                } else {
                    o.x = hr[c];
                    o.y = hi[c];
                }
                out[e][c] = o;
            }
        }
        // one 16-byte store per live lane: the lone last x of an odd-length line also writes its
        // partner slot x = nx, which is line padding (lines have an even length), never read as a
        // value -- every load of it is masked by a select and every reduction and copy to the ABI
        // stops at nx.  (A separate 8-byte store for that lane made every wave run both store
        // paths: odd-length lines ran 8-10% slower.)
#pragma unroll
        for (int c = 0; c < C; ++c) {
            float2 *dst = nxt + own_line + c * cstride + lo;
            if (act0) {
                f4a o;
                o.x = out[0][c].x;
                o.y = out[0][c].y;
                o.z = out[1][c].x;
                o.w = out[1][c].y;
                __builtin_nontemporal_store(o, (f4a *)dst);
            }
        }
        if constexpr (MODE == MODE_ITP) part *= a.tb.dv[v];
    } else if constexpr (NIN > 0) {
        exchange_barrier();
    }

    if constexpr (MODE == MODE_ITP) {
        __shared__ double red[4];
        part = wave_sum(part);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = part;
        __syncthreads();
        if (threadIdx.x == 0) a.partials[b] = (red[0] + red[1]) + (red[2] + red[3]);
    }
}

// X: the lane form (lane_form).
// field: gives the sweep's FieldRec.
template <typename R, int C, int DEG, int MODE, int X, int NIN, typename Field>
__device__ __forceinline__ void sweep_body(const SweepArgs &a, const Field &field, int b, int nb)
{
    if constexpr (X == 3)
        sweep_body_pair<C, DEG, MODE, true, NIN>(a, field, b, nb);
    else if constexpr (X == 2)
        sweep_body_pair<C, DEG, MODE, false, NIN>(a, field, b, nb);
    else
        sweep_body_single<R, C, DEG, MODE, X == 4, NIN>(a, field, b, nb);
}

template <typename R, int C, int DEG, int MODE, int X, int NIN>
__global__ __launch_bounds__(256) void k_sweep(SweepArgs a)
{
    // loaded as early as can be: kept for after the neighbours it costs large boxes 2-3% (FCC 128^3 spin-1
    // 342 -> 351 us a sweep).  Its head lies on a line of the arguments that every wave reads (BCC 30^3
    // 4.4 -> 4.2, FCC 30^3 spin-1 7.8 -> 7.1)
    const auto field = []() { return args_at<FieldRec>(offsetof(SweepArgs, field)); };
    sweep_body<R, C, DEG, MODE, X, NIN>(a, field, sweep_order(a.g, blockIdx.x, gridDim.x, a.order), gridDim.x);
}

// One leapfrog sweep of every member of an ensemble group in a single launch (a group: the
// members sharing component count, face degree and lanes per x, so the kernel is as
// specialised as a single run's).  Member m owns workgroups [begin_m, begin_m + blocks_m)
// (begin_m a multiple of 8, so the XCD remap of the member's own range stays valid); its
// arguments for parity p are m.args[p].  Without the exchange between waves that a single run's BCC
// sweeps make: with the arguments in memory it takes 121 registers for 94 (4 waves a SIMD for 5).  us a
// sweep of one of two members, with -> without: FP32 spin-1 128^3 335 -> 319, spin-2 96^3 251 -> 215, FP64
// spin-1 96^3 308 -> 282, spin-2 64^3 130 either way.
template <typename R, int C, int DEG, int X>
__global__ __launch_bounds__(256) void k_ensemble_sweep(EnsembleArgs e)
{
    // parity-1 sweeps take the whole launch in reverse (members included), keeping each
    // workgroup's XCD, so a sweep starts on the member the previous one ended with
    const int b = e.parity ? reverse_in_xcd(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    int lo = 0, hi = e.nmember - 1;
    while (lo < hi) {  // last member with begin <= b
        const int mid = (lo + hi + 1) >> 1;
        if (e.begin[mid] <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    const EnsembleMember &m = e.members[lo];
    const int local = b - e.begin[lo];
    if (local >= m.blocks) return;  // padding workgroup (uniform)
    const SweepArgs &a = m.args[e.parity];
    const int sweep = e.sweep + (e.sweep_base ? *e.sweep_base : 0);
    const auto field = [&]() { return (const_ptr<FieldRec>)(unsigned long long)(a.fields + sweep); };
    sweep_body<R, C, DEG, MODE_UPDATE, X, 0>(a, field, local, m.blocks);
}

__global__ void k_advance_base(int *base, int by)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *base += by;
}

__global__ void k_set_base(int *base, int value)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *base = value;
}

// ------------------------------------------------------------------------ observables --

// A wave's part of a reduction (reduce_geometry): a chunk of the 64-slot segments of one group of
// y rows of (z, v); slot p of the group is row p / nx, x = p mod nx.
struct RedCoord {
    int v, z, y0, nrow;  // the group's first row and its rows in the box
    unsigned slot0;      // the chunk's first slot
};

__device__ __forceinline__ bool decode_reduce(const Geometry &g, int segs, unsigned w, RedCoord &rc)
{
    if ((long long)w >= g.waves) return false;
    int chunk;
    const unsigned q1 = split_v_seg(g, w, &rc.v, &chunk);
    const unsigned q2 = fast_div(q1, g.f_nz);
    rc.z = (int)(q1 - q2 * (unsigned)g.nz);
    rc.y0 = (int)q2 * g.ty;
    rc.nrow = g.ny - rc.y0 < g.rows ? g.ny - rc.y0 : g.rows;
    rc.slot0 = (unsigned)(chunk * segs * 64);
    return true;
}

// FP64 observables of a level.  Spin-1 128^3 FP32 issues 98 M vector instructions (159 us at 4 cycles a wave
// and SIMD) and misses L2 for 1.18 GB, twice the level (177 us at the copy rate), which 4 waves a SIMD
// overlap in part: 282 us of kernel time, 770 us with one unknown a lane and an exchange per wave of 64.  So:
//   * a lane keeps its 14 sums over all the unknowns it takes and the wave exchanges them once;
//   * the kinetic energy is summed over the faces, each once: with dv_i w_ij = dv_j w_ji (the dual
//     volumes are solved from it) Re sum_i dv_i psi_i* sum_j w_ij (psi_j - psi_i) is
//     -sum over faces of dv_i w_ij |psi_i - psi_j|^2, and -dv_i w_ij |psi_i|^2 for a face at the
//     box's boundary.  A face belongs to the unknown that finds the other one at a higher address
//     (the first nfwd[v] of its row of the table), so a lane loads two neighbours, not four;
//   * the decode serves all segments of the wave's chunk.
// U segments go together (two for one component, 202 -> 208 us on Cube 293^3 with one; three
// components lose a wave a SIMD with two, 296 -> 316 us): the own values and the first four faces'
// neighbours are in flight at once.  Tables, weights and constants are read again in every step
// (scalar loads, fresh()): kept across the loop they take more scalar registers than there are, and
// the spills cost more (447 us).
template <typename R, int C, int U>
__global__ __launch_bounds__(256) void k_observables(ObsArgs a)
{
    using V2 = vec2_t<R>;
    const Geometry &g = a.g;
    const unsigned wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // XCD k (blocks k, k + 8, ...: gridDim.x is a multiple of 8) has a contiguous range of the
    // traversal, which its workgroups walk side by side: the rows and planes a wave needs are what
    // the others read at the same time (each workgroup on a range of its own read a level 2.4 times)
    const unsigned each = gridDim.x >> 3;
    const unsigned first = ((blockIdx.x & 7u) * each * (unsigned)a.per + (blockIdx.x >> 3)) * 4u + wid;
    const V2 *__restrict__ psi = (const V2 *)a.psi;
    const long long cstride = comp_stride(g);
    const int deg = g.deg;
    constexpr int FB = 4;
    double acc[OBS_COUNT];
#pragma unroll
    for (int i = 0; i < OBS_COUNT; ++i) acc[i] = 0.0;
    bool bad = false;

    for (int j = 0; j < a.per; ++j) {
        RedCoord rc;
        if (!decode_reduce(g, a.segs, first + 4u * each * (unsigned)j, rc)) break;
        const int v = rc.v, z = rc.z;
        const V2 *base = psi + line_index(g, 0, z, rc.y0, v);  // the group's first row
        // every y / z neighbour of the group inside the box
        const bool inner = z >= 1 && z <= g.nz - 2 && rc.y0 >= 1 && rc.y0 + rc.nrow <= g.ny - 1;
        const int nfwd = fresh(a.nfwd + v)[0], nf = fresh(a.tb.nface + v)[0];
        const unsigned rows = (unsigned)rc.nrow, slots = rows * (unsigned)g.nx;
        const unsigned end = rc.slot0 + 64u * (unsigned)a.segs < slots ? rc.slot0 + 64u * (unsigned)a.segs : slots;
        for (unsigned s = rc.slot0; s < end; s += 64u * U) {
            int x[U], y[U], at[U];
            bool live[U];
            const const_ptr<int2> fx = fresh((const int2 *)a.face + v * deg);
            int2 face[FB];
#pragma unroll
            for (int f = 0; f < FB; ++f) {
                face[f].x = fx[f].x;
                face[f].y = fx[f].y;
            }
            V2 own[U][C], nb[U][FB][C];
            double ekin[U];
            // whether a face's neighbour is inside the box
            auto inside = [&](int u, int pk) {
                const int dx = (pk & 3) - 1, dy = ((pk >> 2) & 3) - 1, dz = ((pk >> 4) & 3) - 1;
                return (unsigned)(x[u] + dx) < (unsigned)g.nx && (unsigned)(z + dz) < (unsigned)g.nz &&
                       (unsigned)(y[u] + dy) < (unsigned)g.ny;
            };
            // an outside neighbour reads the lane's own value: |psi_i - psi_i|^2 adds nothing
            auto load = [&](int u, int f, int2 e) {
                int off = at[u] + e.y + (e.x & 3) - 1;
                if (!inner || (e.x & 3) != 1) off = inside(u, e.x) ? off : at[u];
#pragma unroll
                for (int c = 0; c < C; ++c) nb[u][f][c] = base[c * cstride + off];
            };
            auto face_energy = [&](int u, int f, double w) {
                double d2 = 0;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const double dr = (double)own[u][c].x - (double)nb[u][f][c].x;
                    const double di = (double)own[u][c].y - (double)nb[u][f][c].y;
                    d2 += dr * dr;
                    d2 += di * di;
                }
                ekin[u] += w * d2;
            };
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const unsigned p = s + 64u * u + (threadIdx.x & 63);
                const unsigned r = fast_div(p, g.f_pairs);
                live[u] = p < end;
                const unsigned rr = live[u] ? r : 0;  // a slot past the group reads the first row
                x[u] = live[u] ? (int)(p - r * (unsigned)g.nx) : 0;
                y[u] = rc.y0 + (int)rr;
                at[u] = (int)rr * (int)g.ys + x[u];
                ekin[u] = 0;
#pragma unroll
                for (int c = 0; c < C; ++c) own[u][c] = base[c * cstride + at[u]];
            }
#pragma unroll
            for (int f = 0; f < FB; ++f) {
                if (f >= nfwd) break;
#pragma unroll
                for (int u = 0; u < U; ++u) load(u, f, face[f]);
            }
            const const_ptr<double> wt = fresh(a.w + v * deg);
#pragma unroll
            for (int f = 0; f < FB; ++f) {
                if (f >= nfwd) break;
#pragma unroll
                for (int u = 0; u < U; ++u) face_energy(u, f, wt[f]);
            }
            for (int f = FB; f < nfwd; ++f) {  // unknowns that own more faces (degree 6 and 8)
                int2 e;
                e.x = fx[f].x;
                e.y = fx[f].y;
#pragma unroll
                for (int u = 0; u < U; ++u) load(u, 0, e);
#pragma unroll
                for (int u = 0; u < U; ++u) face_energy(u, 0, wt[f]);
            }
            const const_ptr<ObsConsts> k = fresh_args<ObsConsts>(offsetof(ObsArgs, k));
            const const_ptr<double> pos = fresh(a.tb.pos64 + 3 * v);
            const double dv = fresh(a.tb.dv + v)[0];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                double pr[C], pi[C], q[C], n = 0;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    pr[c] = own[u][c].x;
                    pi[c] = own[u][c].y;
                    q[c] = pr[c] * pr[c] + pi[c] * pi[c];
                    n += q[c];
                }
                // faces of the box's boundary, whichever unknown would own them
                for (int f = 0; f < nf; ++f) {
                    const int pk = fx[f].x;
                    if (inner && (pk & 3) == 1) continue;
                    ekin[u] += (inside(u, pk) ? 0.0 : wt[f]) * n;
                }
                const double rx = k->p0[0] + k->sig * pos[0] + k->cell[0] * x[u];
                const double ry = k->p0[1] + k->sig * pos[1] + k->cell[1] * y[u];
                const double rz = k->p0[2] + k->sig * pos[2] + k->cell[2] * z;
                // e = part + half, <H> density = part + 2 half: interactions count twice
                double trap = k->off + k->ht[0] * rx * rx;
                trap += k->ht[1] * ry * ry;
                trap += k->ht[2] * rz * rz;
                double part = k->ik * ekin[u] + trap * n;
                double half = k->hc0 * n * n;
                if (!live[u]) continue;
                if constexpr (C > 1) {
                    const double dxr = rx - k->center[0], dyr = ry - k->center[1], dzr = rz - k->center[2];
                    double Fx, Fy, Fz;
                    spin_density<double, C>(pr, pi, Fx, Fy, Fz);
                    const double fxy = Fx * Fx + Fy * Fy, f2 = fxy + Fz * Fz;
                    part += (k->bq * dxr + k->bb[0]) * Fx;
                    part += (k->bq * dyr + k->bb[1]) * Fy;
                    part += (k->bb[2] - 2 * k->bq * dzr) * Fz;
                    half += k->hc1 * f2;
                    if constexpr (C == 5) {
                        const double thr = 2 * (pr[0] * pr[4] - pi[0] * pi[4]) - 2 * (pr[1] * pr[3] - pi[1] * pi[3]) +
                                           (pr[2] * pr[2] - pi[2] * pi[2]);
                        const double thi = 2 * (pr[0] * pi[4] + pi[0] * pr[4]) - 2 * (pr[1] * pi[3] + pi[1] * pr[3]) +
                                           2 * pr[2] * pi[2];
                        half += k->c2_10 * (thr * thr + thi * thi);
                    }
                    if (a.quad) {
                        const double Qx = k->bqq * dxr + k->bbq[0], Qy = k->bqq * dyr + k->bbq[1];
                        const double Qz = -2 * k->bqq * dzr + k->bbq[2];
                        double tr[C], ti[C], m2 = 0;
                        spin_dot<double, C>(Qx, Qy, Qz, pr, pi, tr, ti);
#pragma unroll
                        for (int c = 0; c < C; ++c) m2 += tr[c] * tr[c] + ti[c] * ti[c];
                        part += k->quad_sign * m2;
                    }
                    if constexpr (C == 3)
                        part += k->q * (q[0] + q[2]);
                    else
                        part += k->q * (4 * (q[0] + q[4]) + (q[1] + q[3]));
                    // the reference's local spin (localAvgSpinAndDensity, Spin1GpeBCC.cu:235-271;
                    // Spin2GpeBCC.cu 214-262 applies the same spin-1 expressions to m = 1, 0, -1): x, y of
                    // the spinor divided by sqrt(n), z = |psi_1|^2 - |psi_-1|^2 undivided; its integrals
                    // weight it by n (integrateSpinAndDensity, Spin1GpeBCC.cu:992-1020).  n |(sx, sy, z)|
                    // with sx, sy = (the undivided x, y) / n is |(x, y, n z)|: no division, and unknowns
                    // with n = 0 add nothing.
                    double sxy = fxy, zr = n * Fz;
                    if constexpr (C == 5) {
                        const double sx = (pr[1] * pr[2] + pi[1] * pi[2]) + (pr[2] * pr[3] + pi[2] * pi[3]);
                        const double sy = (pr[1] * pi[2] - pi[1] * pr[2]) + (pr[2] * pi[3] - pi[2] * pr[3]);
                        sxy = 2 * (sx * sx + sy * sy);
                        zr = n * (q[1] - q[3]);
                    }
                    acc[OBS_MX] += Fx * dv;
                    acc[OBS_MY] += Fy * dv;
                    acc[OBS_MZ] += Fz * dv;
                    acc[OBS_SPIN] += sqrt(f2) * dv;
                    acc[OBS_REF_SPIN] += sqrt(sxy + zr * zr) * dv;
                    acc[OBS_REF_MZ] += zr * dv;
                }
                const double nd = n * dv, e = part + half;
                bad = bad || !isfinite(e);  // a non-finite n makes e non-finite
                acc[OBS_NORM] += nd;
                acc[OBS_ENERGY] += e * dv;
                acc[OBS_EXPECT_H] += (e + half) * dv;
                acc[OBS_MAXDENS] = fmax(acc[OBS_MAXDENS], n);
                acc[OBS_RX] += nd * rx;
                acc[OBS_RY] += nd * ry;
                acc[OBS_RZ] += nd * rz;
            }
        }
    }
    acc[OBS_NONFINITE] = bad ? 1.0 : 0.0;
    __shared__ double red[4][OBS_COUNT];
    const double dens = wave_max(acc[OBS_MAXDENS]);
    wave_sum_n<OBS_COUNT>(acc);
    acc[OBS_MAXDENS] = dens;
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int i = 0; i < OBS_COUNT; ++i) red[threadIdx.x >> 6][i] = acc[i];
    }
    __syncthreads();
    if (threadIdx.x < OBS_COUNT) {
        const int i = threadIdx.x;
        double r;
        if (i == OBS_MAXDENS)
            r = fmax(fmax(red[0][i], red[1][i]), fmax(red[2][i], red[3][i]));
        else
            r = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
        a.partials[(long long)blockIdx.x * OBS_COUNT + i] = r;
    }
}

// FP64 norm of a level (OBS_NORM alone) over the same traversal: one read of the level.
template <typename R, int C>
__global__ __launch_bounds__(256) void k_norm(NormArgs a)
{
    using V2 = vec2_t<R>;
    const Geometry &g = a.g;
    const unsigned wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned each = gridDim.x >> 3;
    const unsigned first = ((blockIdx.x & 7u) * each * (unsigned)a.per + (blockIdx.x >> 3)) * 4u + wid;
    const long long cstride = comp_stride(g);
    double sum = 0.0;
    for (int j = 0; j < a.per; ++j) {
        RedCoord rc;
        if (!decode_reduce(g, a.segs, first + 4u * each * (unsigned)j, rc)) break;
        const V2 *base = (const V2 *)a.psi + line_index(g, 0, rc.z, rc.y0, rc.v);
        const unsigned slots = (unsigned)rc.nrow * (unsigned)g.nx;
        const unsigned end = rc.slot0 + 64u * (unsigned)a.segs < slots ? rc.slot0 + 64u * (unsigned)a.segs : slots;
        double n = 0.0;
#pragma unroll 4
        for (unsigned p = rc.slot0 + (threadIdx.x & 63); p < end; p += 64u) {
            const unsigned r = fast_div(p, g.f_pairs);
            const int at = (int)r * (int)g.ys + (int)(p - r * (unsigned)g.nx);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const V2 o = base[c * cstride + at];
                n += (double)o.x * (double)o.x;
                n += (double)o.y * (double)o.y;
            }
        }
        sum += n * a.dv[rc.v];
    }
    __shared__ double red[4];
    sum = wave_sum(sum);
    if ((threadIdx.x & 63) == 0) red[wid] = sum;
    __syncthreads();
    if (threadIdx.x == 0) a.partials[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Two local reductions over a level, one x per lane:
//   max over unknowns of the local Hamiltonian bound (Spin1GpeBCC.cu:144-189): with
//   p = V(r) + c0 n and B = B(r, t) + c1 <F> (<F> = psi^dag f psi, not divided by n),
//   max(p + |Bx| / sqrt2, p + |By| / sqrt2, p + |Bz|); a scalar state gives V + c0 n;
//   sum over unknowns of dv |a|^2 |psi - a|^2 with a = phase * ref (Spin1GpeBCC.cu:436-461
//   with the volume factor of its integrate reduction, :1622-1631; spin-2: the same sum,
//   RelativisticSpin2Gpe.cu:227).  Spin-2 has no Hamiltonian bound: its column holds V + c0 n.
template <typename R, int C>
__global__ __launch_bounds__(256) void k_aux(AuxArgs a)
{
    using V2 = vec2_t<R>;
    const Geometry &g = a.g;
    const WaveCoord wc = decode(g);
    double hmax = -INFINITY, wsum = 0.0;
    if (wc.valid && wc.x < g.nx) {
        const int x = wc.x, v = wc.v, y = wc.y, z = wc.z;
        const V2 *__restrict__ psi = (const V2 *)a.psi;
        double pr[C], pi[C];
        double n = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const V2 o = psi[line_index(g, c, z, y, v) + x];
            pr[c] = o.x;
            pi[c] = o.y;
            n += pr[c] * pr[c] + pi[c] * pi[c];
        }
        const Physics &ph = a.ph;
        const double *pos = a.tb.pos64 + 3 * v;
        const double sig = a.field.sigma;
        const double rx = ph.p0[0] + sig * (ph.cell[0] * x + pos[0]);
        const double ry = ph.p0[1] + sig * (ph.cell[1] * y + pos[1]);
        const double rz = ph.p0[2] + sig * (ph.cell[2] * z + pos[2]);
        double vtrap = 0;
        if (a.field.trap_on)
            vtrap = 0.5 * (ph.trap2[0] * rx * rx + ph.trap2[1] * ry * ry + ph.trap2[2] * rz * rz) + ph.trap_offset;
        const double p = vtrap + ph.c0 * n;
        hmax = p;
        if constexpr (C == 3) {
            const double tr = (pr[0] * pr[1] + pi[0] * pi[1]) + (pr[1] * pr[2] + pi[1] * pi[2]);
            const double ti = (pr[0] * pi[1] - pi[0] * pr[1]) + (pr[1] * pi[2] - pi[1] * pr[2]);
            const double s2 = 1.4142135623730951;
            const double Fx = s2 * tr, Fy = s2 * ti;
            const double Fz = (pr[0] * pr[0] + pi[0] * pi[0]) - (pr[2] * pr[2] + pi[2] * pi[2]);
            const double Bx = a.field.bq * (rx - ph.center[0]) + a.field.bb[0] + ph.c1 * Fx;
            const double By = a.field.bq * (ry - ph.center[1]) + a.field.bb[1] + ph.c1 * Fy;
            const double Bz = -2 * a.field.bq * (rz - ph.center[2]) + a.field.bb[2] + ph.c1 * Fz;
            hmax = fmax(p + fabs(Bx) / s2, fmax(p + fabs(By) / s2, p + fabs(Bz)));
        }
        if (a.ref) {
            const long long line = (long long)g.nx * g.V;
            const long long plane = line * g.ny, comp = plane * g.nz;
            const long long at = (long long)z * plane + (long long)y * line + (long long)x * g.V + a.tb.abi[v];
            double an = 0, dn = 0;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const double2 r = a.ref[(long long)c * comp + at];
                const double ar = a.phase_re * r.x - a.phase_im * r.y;
                const double ai = a.phase_re * r.y + a.phase_im * r.x;
                an += ar * ar + ai * ai;
                dn += (pr[c] - ar) * (pr[c] - ar) + (pi[c] - ai) * (pi[c] - ai);
            }
            wsum = an * dn * a.tb.dv[v];
        }
    }
    __shared__ double red[4][AUX_COUNT];
    const double m = wave_max(hmax), s = wave_sum(wsum);
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6][AUX_MAXHAM] = m;
        red[threadIdx.x >> 6][AUX_WDIFF] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a.partials[(long long)blockIdx.x * AUX_COUNT + AUX_MAXHAM] =
            fmax(fmax(red[0][AUX_MAXHAM], red[1][AUX_MAXHAM]), fmax(red[2][AUX_MAXHAM], red[3][AUX_MAXHAM]));
        a.partials[(long long)blockIdx.x * AUX_COUNT + AUX_WDIFF] =
            (red[0][AUX_WDIFF] + red[1][AUX_WDIFF]) + (red[2][AUX_WDIFF] + red[3][AUX_WDIFF]);
    }
}

// --------------------------------------------------------------------- small kernels --

// Deterministic two-stage reduction of per-workgroup partials (n rows x width columns; column
// maxcol takes the maximum, the others the sum): stage 1 gives each of up to FIN_BLOCKS
// workgroups a fixed contiguous chunk of rows, stage 2 reduces the chunk results in one
// workgroup.  Fixed chunks, strides and trees: the same inputs give the same bits.
constexpr int FIN_BLOCKS = 256;

__device__ __forceinline__ double fin_op(bool is_max, double a, double b) { return is_max ? fmax(a, b) : a + b; }

__global__ __launch_bounds__(256) void k_finalize_stage(const double *partials, int n, int width, int maxcol,
                                                        int chunk, double *out)
{
    __shared__ double red[256];
    const int lo = blockIdx.x * chunk;
    const int hi = min(n, lo + chunk);
    for (int col = 0; col < width; ++col) {
        const bool is_max = col == maxcol;
        double acc = is_max ? -INFINITY : 0.0;
        for (int i = lo + (int)threadIdx.x; i < hi; i += 256) acc = fin_op(is_max, acc, partials[(long long)i * width + col]);
        red[threadIdx.x] = acc;
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if ((int)threadIdx.x < st) red[threadIdx.x] = fin_op(is_max, red[threadIdx.x], red[threadIdx.x + st]);
            __syncthreads();
        }
        if (threadIdx.x == 0) out[(long long)blockIdx.x * width + col] = red[0];
        __syncthreads();
    }
}

// The reduction of at most RED_BLOCKS_MAX records in one workgroup, a wave a column: the fixed lane
// stride and butterfly give the same bits for the same inputs.  The results go to `out` and, for
// a host that reads them, straight to its pinned buffer (a copy of 112 bytes after the kernel cost
// 8 us of a 20 us small-box call).
__global__ __launch_bounds__(1024) void k_finalize_few(const double *partials, int n, int width, int maxcol,
                                                       double *out, double *host)
{
    const int col = threadIdx.x >> 6;
    if (col >= width) return;
    const bool is_max = col == maxcol;
    double acc = is_max ? -INFINITY : 0.0;
#pragma unroll 8
    for (int i = threadIdx.x & 63; i < n; i += 64) acc = fin_op(is_max, acc, partials[(long long)i * width + col]);
    acc = is_max ? wave_max(acc) : wave_sum(acc);
    if ((threadIdx.x & 63) == 0) {
        out[col] = acc;
        if (host) host[col] = acc;
    }
}

// Column sums of `nslot` independent partial tables, one workgroup per table: table s holds n
// records of `width` doubles and its sums go to out + s * out_stride.  A fixed stride order
// and tree, so identical inputs give identical bits.
__global__ __launch_bounds__(256) void k_sum_tables(const double *partials, int n, int width, double *out,
                                                    long long out_stride)
{
    __shared__ double red[256];
    const double *tab = partials + (long long)blockIdx.x * n * width;
    double *dst = out + (long long)blockIdx.x * out_stride;
    for (int col = 0; col < width; ++col) {
        double acc = 0.0;
        for (int i = (int)threadIdx.x; i < n; i += 256) acc += tab[(long long)i * width + col];
        red[threadIdx.x] = acc;
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
            __syncthreads();
        }
        if (threadIdx.x == 0) dst[col] = red[0];
        __syncthreads();
    }
}

// out = sqrt(target / sum of the n partial norms), one workgroup: fixed strides and trees.  41472
// partials (FP64 BCC 96^3) in one launch instead of a two-stage sum and a scale kernel.
__global__ __launch_bounds__(1024) void k_norm_scale(const double *partials, int n, double target, double *out)
{
    __shared__ double red[16];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    int i = threadIdx.x;
    for (; i + 3 * 1024 < n; i += 4 * 1024)
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[k] += partials[i + k * 1024];
    for (int k = 0; i < n; i += 1024, ++k) acc[k] += partials[i];
    const double w = wave_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
    __syncthreads();
    if (threadIdx.x < 64) {
        const double sum = wave_sum(threadIdx.x < 16 ? red[threadIdx.x] : 0.0);
        if (threadIdx.x == 0) out[0] = sqrt(target / sum);
    }
}

template <typename R>
__global__ __launch_bounds__(256) void k_scale(vec2_t<R> *psi, long long n, double factor, const double *dfactor)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const R f = (R)(dfactor ? *dfactor : factor);
    vec2_t<R> o = psi[i];
    o.x *= f;
    o.y *= f;
    psi[i] = o;
}

template <typename R>
__global__ __launch_bounds__(256) void k_phase_copy(const vec2_t<R> *src, vec2_t<R> *dst, long long n, double pre,
                                                     double pim)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const vec2_t<R> s = src[i];
    vec2_t<R> o;
    o.x = (R)(pre * (double)s.x - pim * (double)s.y);
    o.y = (R)(pre * (double)s.y + pim * (double)s.x);
    dst[i] = o;
}

// Counter-based uniform variate in [0, 1) from (seed, index, stream): a 64-bit mix
// (splitmix64 finaliser) of the counter, so every unknown draws independently of the
// traversal and of the launch shape.
__device__ __forceinline__ double hash_uniform(unsigned long long seed, unsigned long long idx, unsigned s)
{
    unsigned long long z = seed * 0x9E3779B97F4A7C15ull + idx * 0xD1B54A32D192ED03ull + (unsigned long long)s * 0x94D049BB133111EBull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = z ^ (z >> 31);
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// psi_c = sqrt(max(mu - V, 0) / g) (w_c + amp * eps_c), eps_c uniform in the unit disk: multiplicative
// noise for one component with w = 1, spinor noise around the spinor w otherwise.
template <typename R>
__global__ __launch_bounds__(256) void k_fill_tf(Geometry g, Tables tb, Physics ph, int ncomp, FillArgs f, void *psi)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long total = (long long)g.nz * g.ny * g.V * g.nx;
    if (i >= total) return;
    long long r = i;
    const int x = (int)(r % g.nx);
    r /= g.nx;
    const int v = (int)(r % g.V);
    r /= g.V;
    const int y = (int)(r % g.ny);
    const int z = (int)(r / g.ny);
    const double *pos = tb.pos64 + 3 * v;
    const double rx = ph.p0[0] + ph.cell[0] * x + pos[0];
    const double ry = ph.p0[1] + ph.cell[1] * y + pos[1];
    const double rz = ph.p0[2] + ph.cell[2] * z + pos[2];
    const double V = 0.5 * (ph.trap2[0] * rx * rx + ph.trap2[1] * ry * ry + ph.trap2[2] * rz * rz) + ph.trap_offset;
    const double a = sqrt(fmax(f.mu - V, 0.0) / f.g);
    const unsigned long long node = (((unsigned long long)z * g.ny + y) * g.nx + x) * g.V + tb.abi[v];
    vec2_t<R> *out = (vec2_t<R> *)psi;
    for (int c = 0; c < ncomp; ++c) {
        double er = 0, ei = 0;
        if (f.amp != 0.0) {
            const double rad = sqrt(hash_uniform(f.seed, node, 2 * c));
            const double ang = 6.283185307179586 * hash_uniform(f.seed, node, 2 * c + 1);
            er = rad * cos(ang);
            ei = rad * sin(ang);
        }
        vec2_t<R> o;  // a (w_c + amp eps_c)
        o.x = (R)(a * (f.w[2 * c] + f.amp * er));
        o.y = (R)(a * (f.w[2 * c + 1] + f.amp * ei));
        out[line_index(g, c, z, y, v) + x] = o;
    }
}

// Unknown (x, v, y, z) of flat index i, x fastest: consecutive lanes take consecutive x of one
// line of the device layout.
struct Unknown {
    int x, v, y, z;
};

__device__ __forceinline__ Unknown unknown_of(const Geometry &g, long long i)
{
    Unknown u;
    u.x = (int)(i % g.nx);
    i /= g.nx;
    u.v = (int)(i % g.V);
    i /= g.V;
    u.y = (int)(i % g.ny);
    u.z = (int)(i / g.ny);
    return u;
}

// Spinor phase projection keeping the density n of every unknown (phases of gpe.h
// GPE_PHASE_*): spin-1 polar (0, sqrt n, 0), ferromagnetic (sqrt n, 0, 0), mixed
// (sqrt(n mix), sqrt(n (1 - mix)), 0) (Spin1GpeBCC.cu:463-551); spin-2 UN, horizontal and vertical
// BN, cyclic with the relative phase `param` (Spin2GpeBCC.cu:417-558), ferromagnetic.  The
// density is summed over m = F..-F and the amplitudes formed as in the reference.
template <typename R, int C>
__global__ __launch_bounds__(256) void k_project(Geometry g, vec2_t<R> *psi, int phase, double param)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)g.nz * g.ny * g.V * g.nx) return;
    const Unknown u = unknown_of(g, i);
    double n = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const vec2_t<R> o = psi[line_index(g, c, u.z, u.y, u.v) + u.x];
        const double re = o.x, im = o.y;
        n += re * re + im * im;
    }
    double outr[C], outi[C];
#pragma unroll
    for (int c = 0; c < C; ++c) outr[c] = outi[c] = 0.0;
    const double cp = cos(param), sp = sin(param);
    if constexpr (C == 3) {
        if (phase == 0) {
            outr[1] = sqrt(n);
        } else if (phase == 1) {
            outr[0] = sqrt(n);
        } else {
            outr[0] = sqrt(n * param);
            outr[1] = sqrt(n * (1.0 - param));
        }
    } else {
        if (phase == 1) {
            outr[0] = sqrt(n);
        } else if (phase == 3) {
            outr[2] = sqrt(n);
        } else if (phase == 4 || phase == 5) {
            const double a = sqrt(n / 2);
            const int lo = phase == 4 ? 0 : 1;
            outr[lo] = a;
            outr[4 - lo] = cp * a;
            outi[4 - lo] = sp * a;
        } else {
            const double a2 = sqrt(n * 1 / 3), a1 = sqrt(n * 2 / 3);
            outr[0] = a2;
            outr[3] = cp * a1;
            outi[3] = sp * a1;
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
        vec2_t<R> o;
        o.x = (R)outr[c];
        o.y = (R)outi[c];
        psi[line_index(g, c, u.z, u.y, u.v) + u.x] = o;
    }
}

// psi_m += amp sqrt(n) eps_m, eps_m uniform in the unit disk from the counter hash of (seed,
// unknown in ABI order, 2m / 2m + 1) -- the variates of k_fill_tf -- n the density before.
template <typename R, int C>
__global__ __launch_bounds__(256) void k_noise(Geometry g, const int *abi, vec2_t<R> *psi, double amp, unsigned long long seed)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)g.nz * g.ny * g.V * g.nx) return;
    const Unknown u = unknown_of(g, i);
    const unsigned long long node = (((unsigned long long)u.z * g.ny + u.y) * g.nx + u.x) * g.V + abi[u.v];
    double pr[C], pi[C], n = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const vec2_t<R> o = psi[line_index(g, c, u.z, u.y, u.v) + u.x];
        pr[c] = o.x;
        pi[c] = o.y;
        n += pr[c] * pr[c] + pi[c] * pi[c];
    }
    const double a = amp * sqrt(n);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const double rad = sqrt(hash_uniform(seed, node, 2 * c));
        const double ang = 6.283185307179586 * hash_uniform(seed, node, 2 * c + 1);
        vec2_t<R> o;
        o.x = (R)(pr[c] + a * rad * cos(ang));
        o.y = (R)(pi[c] + a * rad * sin(ang));
        psi[line_index(g, c, u.z, u.y, u.v) + u.x] = o;
    }
}

hipError_t launch_project(int fp64, int ncomp, const Geometry &g, void *psi, int phase, double param, hipStream_t s)
{
    const unsigned grid = (unsigned)(((long long)g.nz * g.ny * g.V * g.nx + 255) / 256);
    if (ncomp == 3) {
        if (fp64) hipLaunchKernelGGL((k_project<double, 3>), dim3(grid), dim3(256), 0, s, g, (double2 *)psi, phase, param);
        else hipLaunchKernelGGL((k_project<float, 3>), dim3(grid), dim3(256), 0, s, g, (float2 *)psi, phase, param);
    } else if (ncomp == 5) {
        if (fp64) hipLaunchKernelGGL((k_project<double, 5>), dim3(grid), dim3(256), 0, s, g, (double2 *)psi, phase, param);
        else hipLaunchKernelGGL((k_project<float, 5>), dim3(grid), dim3(256), 0, s, g, (float2 *)psi, phase, param);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_noise(int fp64, int ncomp, const Geometry &g, const Tables &tb, void *psi, double amp, unsigned long long seed,
                        hipStream_t s)
{
    const unsigned grid = (unsigned)(((long long)g.nz * g.ny * g.V * g.nx + 255) / 256);
#define NZ(R, C) hipLaunchKernelGGL((k_noise<R, C>), dim3(grid), dim3(256), 0, s, g, tb.abi, (vec2_t<R> *)psi, amp, seed)
    if (fp64) {
        if (ncomp == 1) NZ(double, 1); else if (ncomp == 3) NZ(double, 3); else NZ(double, 5);
    } else {
        if (ncomp == 1) NZ(float, 1); else if (ncomp == 3) NZ(float, 3); else NZ(float, 5);
    }
#undef NZ
    return hipGetLastError();
}

hipError_t launch_fill_tf(int fp64, const Geometry &g, const Tables &tb, const Physics &ph, int ncomp, const FillArgs &f,
                          void *psi, hipStream_t s)
{
    const long long total = (long long)g.nz * g.ny * g.V * g.nx;
    const unsigned grid = (unsigned)((total + 255) / 256);
    if (fp64)
        hipLaunchKernelGGL(k_fill_tf<double>, dim3(grid), dim3(256), 0, s, g, tb, ph, ncomp, f, psi);
    else
        hipLaunchKernelGGL(k_fill_tf<float>, dim3(grid), dim3(256), 0, s, g, tb, ph, ncomp, f, psi);
    return hipGetLastError();
}

// Per-unknown field maps in ABI order (z, y, x, v), `width` doubles each.
//   FIELD_DENSITY    n = sum_m |psi_m|^2
//   FIELD_SPIN       <F> = psi^dag F psi / n (0 where n = 0)
//   FIELD_SPIN_NORM  |psi^dag F psi|
//   FIELD_UV_THETA   spin-1 Cartesian vector a = (psi_-1 - psi_1, -i (psi_-1 + psi_1), sqrt2 psi_0) / sqrt2
//                    = m + i n; theta = atan2(-2 m.n, |m|^2 - |n|^2) / 2 in [0, pi) makes u = Re(a e^{i theta}),
//                    v = Im(a e^{i theta}) orthogonal; (u, v) ordered so that |u| >= |v|; out = u, v, theta.
template <typename R, int C>
__global__ __launch_bounds__(256) void k_local_fields(Geometry g, const int *place, const vec2_t<R> *psi, int kind, double *out)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long total = (long long)g.nz * g.ny * g.nx * g.V;
    if (i >= total) return;
    long long r = i;
    const int v = place[(int)(r % g.V)];
    r /= g.V;
    const int x = (int)(r % g.nx);
    r /= g.nx;
    const int y = (int)(r % g.ny);
    const int z = (int)(r / g.ny);
    double pr[C], pi[C];
    double n = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const vec2_t<R> o = psi[line_index(g, c, z, y, v) + x];
        pr[c] = o.x;
        pi[c] = o.y;
        n += pr[c] * pr[c] + pi[c] * pi[c];
    }
    if (kind == FIELD_DENSITY) {
        out[i] = n;
        return;
    }
    if (kind == FIELD_UV_THETA) {
        if constexpr (C == 3) {
            const double s = 0.7071067811865476;
            const double m[3] = {s * (pr[2] - pr[0]), s * (pi[2] + pi[0]), pr[1]};
            const double q[3] = {s * (pi[2] - pi[0]), -s * (pr[2] + pr[0]), pi[1]};
            const double mq = m[0] * q[0] + m[1] * q[1] + m[2] * q[2];
            const double mm = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
            const double qq = q[0] * q[0] + q[1] * q[1] + q[2] * q[2];
            double th = 0.5 * atan2(-2.0 * mq, mm - qq);
            if (th < 0) th += 3.141592653589793;
            const double ct = cos(th), st = sin(th);
            double u[3], w[3], uu = 0, ww = 0;
            for (int k = 0; k < 3; ++k) {
                u[k] = m[k] * ct - q[k] * st;
                w[k] = m[k] * st + q[k] * ct;
                uu += u[k] * u[k];
                ww += w[k] * w[k];
            }
            double *o = out + 7 * i;
            const bool keep = uu >= ww;
            for (int k = 0; k < 3; ++k) {
                o[k] = keep ? u[k] : w[k];
                o[3 + k] = keep ? w[k] : u[k];
            }
            o[6] = th;
        }
        return;
    }
    double F[3] = {0, 0, 0};
    if constexpr (C > 1) {
        double tr[C], ti[C];
        for (int a = 0; a < 3; ++a) {
            spin_dot<double, C>(a == 0, a == 1, a == 2, pr, pi, tr, ti);
            for (int c = 0; c < C; ++c) F[a] += pr[c] * tr[c] + pi[c] * ti[c];
        }
    }
    if (kind == FIELD_SPIN_NORM) {
        out[i] = sqrt(F[0] * F[0] + F[1] * F[1] + F[2] * F[2]);
    } else {
        const double inv = n > 0 ? 1.0 / n : 0.0;
        for (int a = 0; a < 3; ++a) out[3 * i + a] = F[a] * inv;
    }
}

hipError_t launch_local_fields(int fp64, int ncomp, const Geometry &g, const Tables &tb, const void *psi, int kind, double *out,
                               hipStream_t s)
{
    const long long total = (long long)g.nz * g.ny * g.nx * g.V;
    const unsigned grid = (unsigned)((total + 255) / 256);
#define LF(R, C) hipLaunchKernelGGL((k_local_fields<R, C>), dim3(grid), dim3(256), 0, s, g, tb.place, (const vec2_t<R> *)psi, kind, out)
    if (fp64) {
        if (ncomp == 1) LF(double, 1); else if (ncomp == 3) LF(double, 3); else LF(double, 5);
    } else {
        if (ncomp == 1) LF(float, 1); else if (ncomp == 3) LF(float, 3); else LF(float, 5);
    }
#undef LF
    return hipGetLastError();
}

// Streaming reference kernels for the achievable HBM rate: a copy and an in-place
// read-2-write-1 update (the sweep's own HBM pattern), 16-byte non-temporal accesses.
typedef float f4s __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_stream_copy(const f4s *__restrict__ a, f4s *__restrict__ b, long long n)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) __builtin_nontemporal_store(__builtin_nontemporal_load(&a[i]), &b[i]);
}

__global__ __launch_bounds__(256) void k_stream_update(const f4s *__restrict__ a, f4s *b, long long n, float s)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) __builtin_nontemporal_store(__builtin_nontemporal_load(&b[i]) + s * a[i], &b[i]);
}

hipError_t launch_stream(int kind, const void *a, void *b, long long n16, hipStream_t s)
{
    const unsigned grid = (unsigned)((n16 + 255) / 256);
    if (kind == 0)
        hipLaunchKernelGGL(k_stream_copy, dim3(grid), dim3(256), 0, s, (const f4s *)a, (f4s *)b, n16);
    else
        hipLaunchKernelGGL(k_stream_update, dim3(grid), dim3(256), 0, s, (const f4s *)a, (f4s *)b, n16, 0.5f);
    return hipGetLastError();
}

// ABI order (c, z, y, x, v) in FP64 <-> device layout.  A workgroup turns a run of 2^lg consecutive
// cells of one component round in LDS: the ABI side is one contiguous run, a device line is read or
// written 2^lg values at a time.  With one ABI value a thread, whose device address is a line away
// from its neighbour's, the cache bound it; now bytes do (spin-1 128^3 FP32 out 425 -> 312 us, 5.8
// TB/s, in 450 -> 325; C15 57^3 spin-2 1290 -> 527, 5.7 TB/s, and 1240 -> 840, where 32 cells are short
// pieces of unaligned lines; BCC 96^3 FP64 195 -> 181 and 240 -> 169).  A cell takes an odd number of
// places in LDS, so lanes that hold one unknown of consecutive cells meet no bank twice.
constexpr int PACK_BATCH = 4;  // values a thread has in flight

template <typename R, bool PACK>
__global__ __launch_bounds__(256) void k_pack(Geometry g, const int *__restrict__ abi_of, int lg,
                                              const double2 *__restrict__ abi_in, double2 *__restrict__ abi_out,
                                              const vec2_t<R> *__restrict__ dev_in, vec2_t<R> *__restrict__ dev_out)
{
    using V2 = vec2_t<R>;
    extern __shared__ double2 pack_lds[];
    const int nb = 1 << lg, odd = g.V | 1;
    V2 *tile = (V2 *)pack_lds;                 // [cell][unknown]
    int *off = (int *)(tile + nb * odd);       // a cell's device offset in its component and plane z0
    int *order = off + nb;                     // the ABI's unknown at each device place
    const long long cells = (long long)g.nz * g.ny * g.nx;
    const long long q0 = (long long)blockIdx.x << lg;
    const int n = (int)(cells - q0 < nb ? cells - q0 : nb);
    const unsigned plane = (unsigned)(g.ny * g.nx);  // < 2^31 (Geometry::zs)
    const long long z0 = q0 / plane;
    const unsigned at = (unsigned)(q0 - z0 * plane);
    const unsigned y0 = at / (unsigned)g.nx, x0 = at - y0 * (unsigned)g.nx;
    for (int k = threadIdx.x; k < n; k += 256) {
        const unsigned row = (x0 + k) / (unsigned)g.nx, x = x0 + k - row * (unsigned)g.nx;
        const unsigned dz = (y0 + row) / (unsigned)g.ny, y = y0 + row - dz * (unsigned)g.ny;
        off[k] = (int)(dz * (unsigned)g.zs + y * (unsigned)g.ys + x);
    }
    for (int p = threadIdx.x; p < g.V; p += 256) order[p] = abi_of[p];
    __syncthreads();
    const long long dev0 = z0 * g.zs + (long long)blockIdx.y * g.cs;
    const long long abi0 = ((long long)blockIdx.y * cells + q0) * g.V;
    const int vs = (int)g.vs, pad = odd - g.V;
    const int nabi = n * g.V, ndev = g.V << lg;
    if constexpr (PACK) {
        for (int i0 = threadIdx.x; i0 < nabi; i0 += 256 * PACK_BATCH) {
            double2 s[PACK_BATCH];
#pragma unroll
            for (int j = 0; j < PACK_BATCH; ++j)
                s[j] = nt_load<double>(&abi_in[abi0 + (i0 + 256 * j < nabi ? i0 + 256 * j : 0)]);
#pragma unroll
            for (int j = 0; j < PACK_BATCH; ++j) {
                const int i = i0 + 256 * j;
                V2 o;
                o.x = (R)s[j].x;
                o.y = (R)s[j].y;
                if (i < nabi) tile[i + pad * (int)fast_div((unsigned)i, g.f_V)] = o;
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < ndev; i += 256) {
            const int k = i & (nb - 1), p = i >> lg;
            if (k < n) dev_out[dev0 + off[k] + p * vs] = tile[k * odd + order[p]];
        }
    } else {
        for (int i0 = threadIdx.x; i0 < ndev; i0 += 256 * PACK_BATCH) {
            V2 s[PACK_BATCH];
#pragma unroll
            for (int j = 0; j < PACK_BATCH; ++j) {
                const int i = i0 + 256 * j, k = i & (nb - 1), p = i >> lg;
                s[j] = dev_in[dev0 + (i < ndev && k < n ? off[k] + p * vs : 0)];
            }
#pragma unroll
            for (int j = 0; j < PACK_BATCH; ++j) {
                const int i = i0 + 256 * j, k = i & (nb - 1), p = i >> lg;
                if (i < ndev && k < n) tile[k * odd + order[p]] = s[j];
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < nabi; i += 256) {
            const V2 s = tile[i + pad * (int)fast_div((unsigned)i, g.f_V)];
            nt_store<double>(make_double2((double)s.x, (double)s.y), &abi_out[abi0 + i]);
        }
    }
}

// One ABI value a thread (pack_direct): no table, no barrier between a value's load and its store.
template <typename R, bool PACK>
__global__ __launch_bounds__(256) void k_pack_values(Geometry g, const int *__restrict__ place, const double2 *__restrict__ abi_in,
                                                     double2 *__restrict__ abi_out, const vec2_t<R> *__restrict__ dev_in,
                                                     vec2_t<R> *__restrict__ dev_out)
{
    const long long values = (long long)g.nz * g.ny * g.nx * g.V;
    const long long n = (long long)blockIdx.x * 256 + threadIdx.x;
    if (n >= values) return;
    const long long q = n / g.V, row = q / g.nx;
    const int p = place[(int)(n - q * g.V)], x = (int)(q - row * g.nx);
    const int z = (int)(row / g.ny), y = (int)(row - (long long)z * g.ny);
    const long long d = line_index(g, blockIdx.y, z, y, p) + x, i = blockIdx.y * values + n;
    if constexpr (PACK) {
        const double2 s = abi_in[i];
        vec2_t<R> o;
        o.x = (R)s.x;
        o.y = (R)s.y;
        dev_out[d] = o;
    } else {
        const vec2_t<R> s = dev_in[d];
        abi_out[i] = make_double2((double)s.x, (double)s.y);
    }
}

// ------------------------------------------------------------------------- launchers --

static inline unsigned grid1(long long n) { return (unsigned)((n + 255) / 256); }

template <typename R, int C, int DEG, int X, int NIN>
static hipError_t sweep_mode_n(int mode, const SweepArgs &a, hipStream_t s)
{
    dim3 grid(a.g.blocks), block(256);
    void (*k)(SweepArgs) = nullptr;
    switch (mode) {
    case MODE_UPDATE: k = k_sweep<R, C, DEG, MODE_UPDATE, X, NIN>; break;
    case MODE_EULER: k = k_sweep<R, C, DEG, MODE_EULER, X, NIN>; break;
    case MODE_ITP: k = k_sweep<R, C, DEG, MODE_ITP, X, NIN>; break;
    case MODE_HPSI: k = k_sweep<R, C, DEG, MODE_HPSI, X, NIN>; break;
    default: return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(k, grid, block, 0, s, a);
    return hipGetLastError();
}

template <typename R, int C, int DEG, int X>
static hipError_t sweep_mode_x(int mode, const SweepArgs &a, hipStream_t s)
{
    if constexpr (exchange_ok(DEG, C)) {
        if (a.g.exchange) return sweep_mode_n<R, C, DEG, X, 2>(mode, a, s);
    }
    return sweep_mode_n<R, C, DEG, X, 0>(mode, a, s);
}

template <typename R, int C, int DEG>
static hipError_t sweep_mode(int mode, const SweepArgs &a, hipStream_t s)
{
    const int form = lane_form(a.g.xpl, a.g.rows);
    if (form == 1) return sweep_mode_x<R, C, DEG, 1>(mode, a, s);
    if constexpr (std::is_same<R, double>::value) {
        if (form == 4) return sweep_mode_x<R, C, DEG, 4>(mode, a, s);
    }
    if constexpr (pair_lanes_ok(std::is_same<R, double>::value, DEG, C)) {
        if (form == 2) return sweep_mode_x<R, C, DEG, 2>(mode, a, s);
        if (form == 3) return sweep_mode_x<R, C, DEG, 3>(mode, a, s);
    }
    return hipErrorInvalidValue;
}

template <typename R, int C>
static hipError_t sweep_deg(int mode, const SweepArgs &a, hipStream_t s)
{
    switch (a.g.deg) {
    case 4: return sweep_mode<R, C, 4>(mode, a, s);
    case 6: return sweep_mode<R, C, 6>(mode, a, s);
    case 8: return sweep_mode<R, C, 8>(mode, a, s);
    default: return hipErrorInvalidValue;
    }
}

template <typename R>
static hipError_t sweep_comp(int ncomp, int mode, const SweepArgs &a, hipStream_t s)
{
    switch (ncomp) {
    case 1: return sweep_deg<R, 1>(mode, a, s);
    case 3: return sweep_deg<R, 3>(mode, a, s);
    case 5: return sweep_deg<R, 5>(mode, a, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_sweep(int fp64, int ncomp, int mode, const SweepArgs &a, hipStream_t s)
{
    return fp64 ? sweep_comp<double>(ncomp, mode, a, s) : sweep_comp<float>(ncomp, mode, a, s);
}

typedef void (*ObsKernel)(ObsArgs);

static ObsKernel observables_kernel(int fp64, int ncomp)
{
    switch (ncomp) {
    case 1: return fp64 ? k_observables<double, 1, 2> : k_observables<float, 1, 2>;
    case 3: return fp64 ? k_observables<double, 3, 1> : k_observables<float, 3, 1>;
    case 5: return fp64 ? k_observables<double, 5, 1> : k_observables<float, 5, 1>;
    default: return nullptr;
    }
}

hipError_t observables_resident(int fp64, int ncomp, int device, int *blocks)
{
    int per = 0, cus = 0;
    const ObsKernel f = observables_kernel(fp64, ncomp);
    if (!f) return hipErrorInvalidValue;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void *)f, 256, 0);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    const int n = per * cus;
    *blocks = n < 1 ? 1 : (n > RED_BLOCKS_MAX ? RED_BLOCKS_MAX : n);
    return e;
}

hipError_t launch_observables(int fp64, int ncomp, const ObsArgs &a, hipStream_t s)
{
    const ObsKernel f = observables_kernel(fp64, ncomp);
    if (!f) return hipErrorInvalidValue;
    hipLaunchKernelGGL(f, dim3(a.blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <typename R>
static hipError_t aux_comp(int ncomp, const AuxArgs &a, hipStream_t s)
{
    dim3 grid(a.g.blocks), block(256);
    switch (ncomp) {
    case 1: hipLaunchKernelGGL((k_aux<R, 1>), grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL((k_aux<R, 3>), grid, block, 0, s, a); break;
    case 5: hipLaunchKernelGGL((k_aux<R, 5>), grid, block, 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_aux(int fp64, int ncomp, const AuxArgs &a, hipStream_t s)
{
    return fp64 ? aux_comp<double>(ncomp, a, s) : aux_comp<float>(ncomp, a, s);
}

template <typename R, int C, int DEG, int X>
static hipError_t ens_n(const EnsembleArgs &e, int blocks, hipStream_t s)
{
    hipLaunchKernelGGL((k_ensemble_sweep<R, C, DEG, X>), dim3(blocks), dim3(256), 0, s, e);
    return hipGetLastError();
}

template <typename R, int C, int DEG>
static hipError_t ens_x(int form, const EnsembleArgs &e, int blocks, hipStream_t s)
{
    if (form == 1) return ens_n<R, C, DEG, 1>(e, blocks, s);
    if constexpr (std::is_same<R, double>::value) {
        if (form == 4) return ens_n<R, C, DEG, 4>(e, blocks, s);
    }
    if constexpr (pair_lanes_ok(std::is_same<R, double>::value, DEG, C)) {
        if (form == 2) return ens_n<R, C, DEG, 2>(e, blocks, s);
        if (form == 3) return ens_n<R, C, DEG, 3>(e, blocks, s);
    }
    return hipErrorInvalidValue;
}

template <typename R, int C>
static hipError_t ens_deg(int deg, int form, const EnsembleArgs &e, int blocks, hipStream_t s)
{
    switch (deg) {
    case 4: return ens_x<R, C, 4>(form, e, blocks, s);
    case 6: return ens_x<R, C, 6>(form, e, blocks, s);
    case 8: return ens_x<R, C, 8>(form, e, blocks, s);
    default: return hipErrorInvalidValue;
    }
}

template <typename R>
static hipError_t ens_comp(int ncomp, int deg, int form, const EnsembleArgs &e, int blocks, hipStream_t s)
{
    switch (ncomp) {
    case 1: return ens_deg<R, 1>(deg, form, e, blocks, s);
    case 3: return ens_deg<R, 3>(deg, form, e, blocks, s);
    case 5: return ens_deg<R, 5>(deg, form, e, blocks, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_ensemble_sweep(int fp64, int ncomp, int deg, int form, const EnsembleArgs &e, int blocks,
                                 hipStream_t s)
{
    return fp64 ? ens_comp<double>(ncomp, deg, form, e, blocks, s)
                : ens_comp<float>(ncomp, deg, form, e, blocks, s);
}

hipError_t launch_advance_base(int *base, int by, hipStream_t s)
{
    hipLaunchKernelGGL(k_advance_base, dim3(1), dim3(64), 0, s, base, by);
    return hipGetLastError();
}

hipError_t launch_set_base(int *base, int value, hipStream_t s)
{
    hipLaunchKernelGGL(k_set_base, dim3(1), dim3(64), 0, s, base, value);
    return hipGetLastError();
}

hipError_t launch_finalize(const double *partials, int n, int width, int maxcol, double *out, double *scratch,
                           hipStream_t s)
{
    if (n <= 0 || width <= 0 || width > FIN_WIDTH_MAX) return hipErrorInvalidValue;
    int nb = (n + 1023) / 1024;
    if (nb > FIN_BLOCKS) nb = FIN_BLOCKS;
    if (nb == 1) {
        hipLaunchKernelGGL(k_finalize_stage, dim3(1), dim3(256), 0, s, partials, n, width, maxcol, n, out);
        return hipGetLastError();
    }
    const int chunk = (n + nb - 1) / nb;
    nb = (n + chunk - 1) / chunk;
    hipLaunchKernelGGL(k_finalize_stage, dim3(nb), dim3(256), 0, s, partials, n, width, maxcol, chunk, scratch);
    hipLaunchKernelGGL(k_finalize_stage, dim3(1), dim3(256), 0, s, (const double *)scratch, nb, width, maxcol, nb,
                       out);
    return hipGetLastError();
}

hipError_t launch_finalize_few(const double *partials, int n, int width, int maxcol, double *out, double *host,
                               hipStream_t s)
{
    if (n <= 0 || n > RED_BLOCKS_MAX || width <= 0 || width > FIN_WIDTH_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_finalize_few, dim3(1), dim3(64 * FIN_WIDTH_MAX), 0, s, partials, n, width, maxcol, out, host);
    return hipGetLastError();
}

hipError_t launch_sum_tables(const double *partials, int nslot, int n, int width, double *out, long long out_stride,
                             hipStream_t s)
{
    if (nslot <= 0 || n <= 0 || width <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sum_tables, dim3(nslot), dim3(256), 0, s, partials, n, width, out, out_stride);
    return hipGetLastError();
}

hipError_t launch_norm_scale(const double *partials, int n, double target, double *out, double *scratch, hipStream_t s)
{
    if (n <= 0) return hipErrorInvalidValue;
    if (n > NORM_ONE_MAX) {
        const int chunk = (n + FIN_BLOCKS - 1) / FIN_BLOCKS, nb = (n + chunk - 1) / chunk;
        hipLaunchKernelGGL(k_finalize_stage, dim3(nb), dim3(256), 0, s, partials, n, 1, -1, chunk, scratch);
        partials = scratch;
        n = nb;
    }
    hipLaunchKernelGGL(k_norm_scale, dim3(1), dim3(1024), 0, s, partials, n, target, out);
    return hipGetLastError();
}

hipError_t launch_norm(int fp64, int ncomp, const NormArgs &a, hipStream_t s)
{
    void (*k)(NormArgs) = nullptr;
    switch (ncomp) {
    case 1: k = fp64 ? k_norm<double, 1> : k_norm<float, 1>; break;
    case 3: k = fp64 ? k_norm<double, 3> : k_norm<float, 3>; break;
    case 5: k = fp64 ? k_norm<double, 5> : k_norm<float, 5>; break;
    default: return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(k, dim3(a.blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_scale(int fp64, void *psi, long long nelem, double factor, const double *dfactor, hipStream_t s)
{
    if (nelem <= 0) return hipSuccess;
    if (fp64)
        hipLaunchKernelGGL(k_scale<double>, dim3(grid1(nelem)), dim3(256), 0, s, (double2 *)psi, nelem, factor, dfactor);
    else
        hipLaunchKernelGGL(k_scale<float>, dim3(grid1(nelem)), dim3(256), 0, s, (float2 *)psi, nelem, factor, dfactor);
    return hipGetLastError();
}

hipError_t launch_phase_copy(int fp64, const void *src, void *dst, long long nelem, double pre, double pim,
                             hipStream_t s)
{
    if (nelem <= 0) return hipSuccess;
    if (fp64)
        hipLaunchKernelGGL(k_phase_copy<double>, dim3(grid1(nelem)), dim3(256), 0, s, (const double2 *)src,
                           (double2 *)dst, nelem, pre, pim);
    else
        hipLaunchKernelGGL(k_phase_copy<float>, dim3(grid1(nelem)), dim3(256), 0, s, (const float2 *)src,
                           (float2 *)dst, nelem, pre, pim);
    return hipGetLastError();
}

// Where one ABI value a thread is faster than the turn in LDS.  us a call of the smallest and of larger levels,
// through LDS and direct:
//   * cells of one unknown, whose two sides are runs of lines already: Cube 150^3 FP64 in 30 and 26;
//   * levels of few workgroups, whose time is one chain of latencies: C15 6x5x6 FP64 in 14.8 and 13.1, out
//     15.1 and 12.9.  The lines meet at 2e5-3e5 values in and 4e5-6e5 out for every cell size;
//   * on the way in, levels of smaller cells that the caches hold, where a line's pieces meet in L2: BCC 48^3
//     spin-1 FP64 35 and 31, 96^3 210 and 247; of 1.6e6-7e6 values A15 FP64 4-8% slower through LDS, BCC
//     FP32 1-4%; A15 FP32 9-14% faster, Z and C15 2-59% faster.
template <typename R, bool PACK>
static bool pack_direct(const Geometry &g, long long values)
{
    if (g.V == 1 || values < (PACK ? 1 << 18 : 1 << 19)) return true;
    return PACK && values < (8 << 20) && g.V <= (sizeof(R) == 8 ? 46 : 12);
}

// Cells per workgroup: 64 (fewer where those of a large cell fill more than 24 KiB or a
// small box has under 128 workgroups, but 16 cells), and more, in
// a tile of up to 40 KiB, while there are workgroups enough to hide a tile's load before its store.
// Measured: tiles of up to 64 KiB, BCC 96^3 FP64 out 181 -> 256 us; of up to 32 KiB, C15 57^3 spin-2 in
// 840 -> 930; 16 cells of FCC 30^3 spin-1 in 20 us, 64 16; 256 of FCC 60^3 spin-1 in 45, 64 41.
template <typename R, bool PACK>
static hipError_t pack(const Geometry &g, const Tables &tb, int ncomp, const double *abi_in, double *abi_out, const void *dev_in,
                       void *dev_out, hipStream_t s)
{
    const long long cells = (long long)g.nz * g.ny * g.nx;
    const long long values = cells * g.V;
    if (pack_direct<R, PACK>(g, ncomp * values)) {
        hipLaunchKernelGGL((k_pack_values<R, PACK>), dim3(grid1(values), (unsigned)ncomp), dim3(256), 0, s, g, tb.place,
                           (const double2 *)abi_in, (double2 *)abi_out, (const vec2_t<R> *)dev_in, (vec2_t<R> *)dev_out);
        return hipGetLastError();
    }
    const size_t cell = (size_t)(g.V | 1) * sizeof(vec2_t<R>);
    int lg = 6;
    while (lg > 4 && ((cell << lg) > 24576 || ncomp * (cells >> lg) < 128)) --lg;
    while (lg < 10 && (cell << (lg + 1)) <= 40960 && ncomp * ((cells >> (lg + 1)) + 1) >= 8192) ++lg;
    const size_t lds = (cell << lg) + (sizeof(int) << lg) + sizeof(int) * (size_t)g.V;
    const dim3 grid((unsigned)((cells + (1 << lg) - 1) >> lg), (unsigned)ncomp);
    hipLaunchKernelGGL((k_pack<R, PACK>), grid, dim3(256), lds, s, g, tb.abi, lg, (const double2 *)abi_in, (double2 *)abi_out,
                       (const vec2_t<R> *)dev_in, (vec2_t<R> *)dev_out);
    return hipGetLastError();
}

hipError_t launch_pack(int fp64, const Geometry &g, const Tables &tb, int ncomp, const double *abi, void *dev, hipStream_t s)
{
    return fp64 ? pack<double, true>(g, tb, ncomp, abi, nullptr, nullptr, dev, s)
                : pack<float, true>(g, tb, ncomp, abi, nullptr, nullptr, dev, s);
}

hipError_t launch_unpack(int fp64, const Geometry &g, const Tables &tb, int ncomp, const void *dev, double *abi, hipStream_t s)
{
    return fp64 ? pack<double, false>(g, tb, ncomp, nullptr, abi, dev, nullptr, s)
                : pack<float, false>(g, tb, ncomp, nullptr, abi, dev, nullptr, s);
}

}  // namespace gpe
