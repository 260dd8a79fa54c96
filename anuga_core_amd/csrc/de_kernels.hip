// HIP kernels of the DE step for gfx950 (FP64 and mixed FP32/FP64).
//
// One thread per triangle, triangles in a locality order (bisection tiles or
// RCM), DE_BLOCK-thread workgroups remapped XCD-contiguous. Per Euler substep:
//   de_extrapolate  protect + velocity + dry-neighbour zeroing + limited
//                   second-order edge values (sw_domain_orig.c:1215-1281,
//                   :1994-2680). Reads the raw centroid state and never
//                   writes it: the protect / zeroing outcome goes to a flag
//                   byte, so the step's initial state doubles as the RK2 backup.
//   de_flux         per-triangle gather of its three edge fluxes in local edge
//                   order (bit-identical to the reference's compute-once-and-
//                   mirror loop, sw_domain_orig.c:765-1150), boundary states
//                   evaluated in place, CFL timestep and boundary inflow as
//                   per-block partials. In the later Runge-Kutta substeps the
//                   kernel also applies friction, the update,
//                   fix_negative_cells and the substep's combination with the
//                   step's initial state, since dt is already known.
//   de_update       friction + update + fix_negative_cells
//                   (sw_domain_orig.c:2805-2838, quantity.c:772-822,
//                   sw_domain_orig.c:2890-2910).
//                   In device-controlled steps it forms the timestep too.
//   de_reduce_chunks, de_reduce, de_finish_step  fixed-order reduction of the
//                   per-block partials; the last also ends the step.
//   de_xflux,       extrapolation and flux fused over compact tiles (the
//   de_xflux_mixed  bisection order): a workgroup extrapolates its
//                   triangles and their halo into LDS and gathers the fluxes
//                   from there, with the same device functions as the
//                   separate kernels, so the same bits.
// No atomics touch the state, so every run is bitwise reproducible.
//
// Every kernel is a template on T, the type of the extrapolation,
// reconstruction and flux arithmetic: double for the FP64 path (bit-comparable
// with the reference), float for the mixed path. The conserved state, the
// update, the wet/dry thresholds, the CFL reduction and the volume stay FP64
// in both.
#include "de_device.h"
#include "de_pow.h"


// ---------------------------------------------------------------------------
// geometry access, per precision
// ---------------------------------------------------------------------------
template <class T> struct DeGeo;
template <> struct DeGeo<double> {
    using X = DeGeoX64;
    using F = DeGeoF64;
};
template <> struct DeGeo<float> {
    using X = DeGeoX32;
    using F = DeGeoF32;
};

// the step's centroid state after protect + momentum zeroing, from the flag
struct DeCentroid {
    double w, uh, vh, z;
};

__device__ __forceinline__ DeCentroid de_centroid(const DeQ q, unsigned f)
{
    DeCentroid c;
    c.z = q.z;
    c.w = (f & DE_F_CLAMP) ? q.z : q.w;
    c.uh = (f & DE_F_KEEP) ? q.uh : 0.0;
    c.vh = (f & DE_F_KEEP) ? q.vh : 0.0;
    return c;
}

// ---------------------------------------------------------------------------
// extrapolation
// ---------------------------------------------------------------------------
// The extrapolation of one triangle k (sw_domain_orig.c:1215-1281,
// :1994-2680): its protected centroid cell, the protect / momentum flag,
// protect's added mass and the limited jumps from the centroid to its three
// edges. Shared by the extrapolation kernel and the tiled fused kernel, so
// both produce the same bits.
template <class T>
struct DeExtrap {
    DeCell c;
    T jw[3], jh[3], ju[3], jv[3];
    bool constant, gw, gu, gv;
    unsigned flag;
    double mass;
    double z;   // the centroid bed
};

// The extrapolation geometry of triangle k from its vertices, as
// general_mesh.py forms the arrays the reference's extrapolation reads
// (:599-626 edge midpoints 0.5 (Va + Vb); sw_domain_orig.c:2112-2135 their
// offsets from the stored centroid).
struct DeVerts {
    double2 v0, v1, v2;
};

__device__ __forceinline__ void de_vertex_offsets(const double2 c, const DeVerts &w,
                                                  double dxv[3], double dyv[3])
{
    const double2 v0 = w.v0, v1 = w.v1, v2 = w.v2;
    dxv[0] = 0.5 * (v1.x + v2.x) - c.x;
    dyv[0] = 0.5 * (v1.y + v2.y) - c.y;
    dxv[1] = 0.5 * (v2.x + v0.x) - c.x;
    dyv[1] = 0.5 * (v2.y + v0.y) - c.y;
    dxv[2] = 0.5 * (v0.x + v1.x) - c.x;
    dyv[2] = 0.5 * (v0.y + v1.y) - c.y;
}

// Outward normal and length of an edge from va to vb (general_mesh.py:202-232:
// of the edge opposite vertex i, (x, y) = V[i+2] - V[i+1],
// l = sqrt(x^2 + y^2), normal (y / l, -(x / l))).
__device__ __forceinline__ void de_vertex_normal(const double2 va, const double2 vb, double &n1,
                                                 double &n2, double &len)
{
    const double xn = vb.x - va.x, yn = vb.y - va.y;
    len = sqrt(xn * xn + yn * yn);
    n1 = yn / len;
    n2 = -(xn / len);
}

// Edge offsets and the gradient's auxiliary geometry of triangle k from the
// stored record: the six numbers of DeGeoX64 (FP64), or formed from the FP32
// surrogate offsets.
template <class T>
struct DeStoredGeo {
    typename DeGeo<T>::X g;
    __device__ __forceinline__ DeStoredGeo(const DeMesh &m, int k, T dxv[3], T dyv[3])
        : g(static_cast<const typename DeGeo<T>::X *>(m.gx)[k])
    {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            dxv[i] = g.dxv[i];
            dyv[i] = g.dyv[i];
        }
    }
    __device__ __forceinline__ void aux(T &dx1, T &dx2, T &dy1, T &dy2, T &area2, T &inv) const
    {
        if constexpr (sizeof(T) == 8) {
            dx1 = g.aux[0];
            dx2 = g.aux[1];
            dy1 = g.aux[2];
            dy2 = g.aux[3];
            area2 = g.aux[4];
            inv = g.aux[5];
        } else {
            dx1 = g.rx[1] - g.rx[0];
            dx2 = g.rx[2] - g.rx[0];
            dy1 = g.ry[1] - g.ry[0];
            dy2 = g.ry[2] - g.ry[0];
            area2 = dy2 * dx1 - dy1 * dx2;
            inv = de_rcp(area2);
        }
    }
    __device__ __forceinline__ void line(bool e0, bool e1, T &dx2, T &dy2) const
    {
        if constexpr (sizeof(T) == 8) {
            dx2 = g.aux[1];
            dy2 = g.aux[3];
        } else {
            // selects on named copies: a select between members would load
            // from a selected address, so the record would sit in scratch
            const T x0 = g.rx[0], x1 = g.rx[1], x2 = g.rx[2];
            const T y0 = g.ry[0], y1 = g.ry[1], y2 = g.ry[2];
            const T dx1 = e0 ? x0 : (e1 ? x1 : x2);
            const T dy1 = e0 ? y0 : (e1 ? y1 : y2);
            const T area2 = dx1 * dx1 + dy1 * dy1;
            dx2 = de_rcp(area2);
            dy2 = dx2 * dy1;
            dx2 *= dx1;
        }
    }
};

// The same from the centroids: the surrogate centroids c0, c1, c2 (ck, its
// own, where an edge is a boundary edge).
struct DeCentroidGeo {
    double2 ck, c0, c1, c2;
    // the surrogate centroids' triangle (sw_domain_orig.c:2130-2160)
    __device__ __forceinline__ void aux(double &dx1, double &dx2, double &dy1, double &dy2,
                                        double &area2, double &inv) const
    {
        dx1 = c1.x - c0.x;
        dx2 = c2.x - c0.x;
        dy1 = c1.y - c0.y;
        dy2 = c2.y - c0.y;
        area2 = dy2 * dx1 - dy1 * dx2;
        inv = 1.0 / area2;
    }
    // toward the one interior neighbour (sw_domain_orig.c:2421-2450)
    __device__ __forceinline__ void line(bool e0, bool e1, double &dx2, double &dy2) const
    {
        const double x0 = c0.x, x1 = c1.x, x2 = c2.x, y0 = c0.y, y1 = c1.y, y2 = c2.y;
        const double cx = e0 ? x0 : (e1 ? x1 : x2), cy = e0 ? y0 : (e1 ? y1 : y2);
        const double ddx = cx - ck.x, ddy = cy - ck.y;
        const double a2 = ddx * ddx + ddy * ddy;
        dx2 = 1.0 / a2;
        dy2 = dx2 * ddy;
        dx2 *= ddx;
    }
};

// The limited jumps of a triangle whose own cell is x.c, from its surrogate
// neighbours' cells; v, nbound: its neighbour record.
template <class T, class Geo>
__device__ __forceinline__ void de_extrap_jumps(const DeParams &p, const int v[3], int nbound,
                                                const DeCell nb[3], const T dxv[3],
                                                const T dyv[3], const Geo &geo, int *err,
                                                DeExtrap<T> &x)
{
    const double mah = p.mah;
    const DeCell &c = x.c;
    T(&jw)[3] = x.jw, (&jh)[3] = x.jh, (&ju)[3] = x.ju, (&jv)[3] = x.jv;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        jw[i] = T(0.0);
        jh[i] = T(0.0);
        ju[i] = T(0.0);
        jv[i] = T(0.0);
    }
    bool &constant = x.constant, &gw = x.gw, &gu = x.gu, &gv = x.gv;
    constant = (nbound == 3);
    gw = gu = gv = true;   // false: beta == 0, edge = centroid value
    if (nbound <= 1) {
        T dx1, dx2, dy1, dy2, area2, inv_area2;
        geo.aux(dx1, dx2, dy1, dy2, area2, inv_area2);
        if (area2 <= T(0.0)) {
            constant = true;
        } else {
            const T a_tmp = T(0.3), b_tmp = T(0.1);
            const T c_tmp = T(1.0) / (a_tmp - b_tmp);
            const T d_tmp = T(1.0) - (c_tmp * a_tmp);
            const T tmah = T(mah);
            const T hc = T(c.h), h0 = T(nb[0].h), h1 = T(nb[1].h), h2 = T(nb[2].h);
            const T hmin = fmin(fmin(h0, fmin(h1, h2)), hc);
            const T hmax = fmax(fmax(h0, fmax(h1, h2)), hc);
            T hfactor = fmax(T(0.0), fmin(de_div(c_tmp * fmax(hmin, T(0.0)), fmax(hc, T(1.0e-06))) + d_tmp,
                                          fmin(de_div(c_tmp * fmax(hc, T(0.0)), fmax(hmax, T(1.0e-06))) + d_tmp,
                                               T(1.0))));
            hfactor = fmin(de_div(T(1.2) * fmax(hmin - tmah, T(0.0)), fmax(hmin, T(0.0)) + T(1.0) * tmah),
                           hfactor);

            T beta = T(p.bwd) + (T(p.bw) - T(p.bwd)) * hfactor;
            gw = beta > T(0.0);
            if (gw) {
                de_aux_jumps<T>(c.w, nb[0].w, nb[1].w, nb[2].w, dx1, dx2, dy1, dy2, inv_area2,
                                dxv, dyv, beta, jw);
                de_aux_jumps<T>(c.h, nb[0].h, nb[1].h, nb[2].h, dx1, dx2, dy1, dy2, inv_area2,
                                dxv, dyv, beta, jh);
            }
            beta = T(p.buhd) + (T(p.buh) - T(p.buhd)) * hfactor;
            gu = beta > T(0.0);
            if (gu)
                de_aux_jumps<T>(c.u, nb[0].u, nb[1].u, nb[2].u, dx1, dx2, dy1, dy2, inv_area2,
                                dxv, dyv, beta, ju);
            beta = T(p.bvhd) + (T(p.bvh) - T(p.bvhd)) * hfactor;
            gv = beta > T(0.0);
            if (gv)
                de_aux_jumps<T>(c.v, nb[0].v, nb[1].v, nb[2].v, dx1, dx2, dy1, dy2, inv_area2,
                                dxv, dyv, beta, jv);
        }
    } else if (nbound == 2) {
        // the first edge whose surrogate is not k itself (sw_domain_orig.c:2421-2439)
        // selects rather than indexing, so the register arrays stay in registers
        const bool e0 = v[0] >= 0, e1 = v[1] >= 0, e2 = v[2] >= 0;
        if (!(e0 || e1 || e2)) {
            atomicOr(err, DE_ERR_NO_NEIGHBOUR);
            constant = true;
        } else {
            // field-wise selects on named copies: indexing the array here
            // would place it in private (scratch) memory
            const DeCell a0 = nb[0], a1 = nb[1], a2 = nb[2];
            DeCell n1;
            n1.w = e0 ? a0.w : (e1 ? a1.w : a2.w);
            n1.h = e0 ? a0.h : (e1 ? a1.h : a2.h);
            n1.u = e0 ? a0.u : (e1 ? a1.u : a2.u);
            n1.v = e0 ? a0.v : (e1 ? a1.v : a2.v);
            T dx2, dy2;
            geo.line(e0, e1, dx2, dy2);
            const T bw = T(p.bw);
            de_line_jumps<T>(c.w, n1.w, dx2, dy2, dxv, dyv, bw, jw);
            de_line_jumps<T>(c.h, n1.h, dx2, dy2, dxv, dyv, bw, jh);
            de_line_jumps<T>(c.u, n1.u, dx2, dy2, dxv, dyv, bw, ju);
            de_line_jumps<T>(c.v, n1.v, dx2, dy2, dxv, dyv, bw, jv);
        }
    }
}

// The whole extrapolation of triangle k, its neighbours gathered from memory.
// vk, qk: its neighbour record and state, loaded by the caller.
template <class T>
__device__ __forceinline__ void de_extrap_cell(const DeMesh &m, const DeParams &p,
                                               const DeQ *__restrict__ q, int k, int4 vk,
                                               DeQ qk, int *err, DeExtrap<T> &x)
{
    const double mah = p.mah;
    const int v[3] = {vk.x, vk.y, vk.z};
    const int nbound = vk.w;
    x.z = qk.z;
    int sur[3];
#pragma unroll
    for (int i = 0; i < 3; i++) sur[i] = v[i] >= 0 ? (v[i] >> 2) : k;
    // surrogate neighbours: one record each
    DeQ qs[3];
#pragma unroll
    for (int i = 0; i < 3; i++) qs[i] = q[sur[i]];
    double hs[3];
#pragma unroll
    for (int i = 0; i < 3; i++) hs[i] = de_height(qs[i].w, qs[i].z);

    // protect + velocity of triangle k (sw_domain_orig.c:1245-1276, :2014-2064)
    const bool clamp = de_clamped(qk.w, qk.z, mah);
    DeCell &c = x.c;
    c.w = clamp ? qk.z : qk.w;
    c.h = de_height(c.w, qk.z);
    bool dry_k = true;
#pragma unroll
    for (int i = 0; i < 3; i++) dry_k = dry_k && (v[i] < 0 || hs[i] < mah);
    const bool keep = (c.h > mah) && !dry_k;
    c.u = 0.0;
    c.v = 0.0;
    if (keep) {
        const double inv = 1.0 / c.h;
        c.u = qk.uh * inv;
        c.v = qk.vh * inv;
    }
    x.mass = clamp ? (qk.z - qk.w) * m.area[k] : 0.0;
    x.flag = (clamp ? DE_F_CLAMP : 0u) | (keep ? DE_F_KEEP : 0u);

    // the same for the surrogate neighbours. A wet neighbour n keeps its
    // velocity unless all of its own neighbours are dry; k is one of
    // them, so the heights of n's other neighbours are needed only when
    // k itself is dry (a boundary edge's surrogate is k: its test is dry_k)
    DeCell nb[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const bool cl = de_clamped(qs[i].w, qs[i].z, mah);
        nb[i].w = cl ? qs[i].z : qs[i].w;
        nb[i].h = hs[i];
        nb[i].u = 0.0;
        nb[i].v = 0.0;
        if (hs[i] > mah) {
            bool dry = v[i] < 0 ? dry_k : (c.h < mah);
            if (v[i] >= 0 && dry) {
                const int4 vs = m.nb[sur[i]];
                const int vv[3] = {vs.x, vs.y, vs.z};
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    if (vv[r] >= 0) {
                        const DeQ t = q[vv[r] >> 2];
                        dry = dry && (de_height(t.w, t.z) < mah);
                    }
                }
            }
            if (!dry) {
                const double inv = 1.0 / hs[i];
                nb[i].u = qs[i].uh * inv;
                nb[i].v = qs[i].vh * inv;
            }
        }
    }

    // limited jumps from the centroid to the edges, per quantity
    T dxv[3], dyv[3];
    const DeStoredGeo<T> geo(m, k, dxv, dyv);
    de_extrap_jumps<T>(p, v, nbound, nb, dxv, dyv, geo, err, x);
}

// the same, loading triangle k's records
template <class T>
__device__ __forceinline__ void de_extrap_cell(const DeMesh &m, const DeParams &p,
                                               const DeQ *__restrict__ q, int k, int *err,
                                               DeExtrap<T> &x)
{
    de_extrap_cell<T>(m, p, q, k, m.nb[k], q[k], err, x);
}

// FP64 edge values of edge i (compile-time i, or a select on a run-time one):
// edge = centroid + limited jump; the beta == 0 and constant branches copy the
// centroid value (sw_domain_orig.c:2278-2283)
__device__ __forceinline__ void de_edge64(const DeExtrap<double> &x, int i, double &ew,
                                          double &eh, double &euh, double &evh)
{
    const double jw = i == 0 ? x.jw[0] : (i == 1 ? x.jw[1] : x.jw[2]);
    const double jh = i == 0 ? x.jh[0] : (i == 1 ? x.jh[1] : x.jh[2]);
    const double ju = i == 0 ? x.ju[0] : (i == 1 ? x.ju[1] : x.ju[2]);
    const double jv = i == 0 ? x.jv[0] : (i == 1 ? x.jv[1] : x.jv[2]);
    ew = (x.constant || !x.gw) ? x.c.w : x.c.w + jw;
    eh = (x.constant || !x.gw) ? x.c.h : x.c.h + jh;
    const double eu = (x.constant || !x.gu) ? x.c.u : x.c.u + ju;
    const double ev = (x.constant || !x.gv) ? x.c.v : x.c.v + jv;
    euh = eu * eh;
    evh = ev * eh;
}

// Mixed-path edge record of edge i (compile-time i): FP32 stage and depth
// jumps and edge momenta, referred to the FP64 centroid depth x.c.h
__device__ __forceinline__ float4 de_edge32(const DeExtrap<float> &x, int i)
{
    const float jw = i == 0 ? x.jw[0] : (i == 1 ? x.jw[1] : x.jw[2]);
    const float jh = i == 0 ? x.jh[0] : (i == 1 ? x.jh[1] : x.jh[2]);
    const float ju = i == 0 ? x.ju[0] : (i == 1 ? x.ju[1] : x.ju[2]);
    const float jv = i == 0 ? x.jv[0] : (i == 1 ? x.jv[1] : x.jv[2]);
    const float hw = x.constant ? 0.f : jw;
    const float hh = x.constant ? 0.f : jh;
    const float eh = float(x.c.h + double(hh));
    const float eu = float(x.c.u + (x.constant ? 0.0 : double(ju)));
    const float ev = float(x.c.v + (x.constant ? 0.0 : double(jv)));
    return make_float4(hw, hh, eu * eh, ev * eh);
}

template <class T>
__global__ void __launch_bounds__(DE_BLOCK)
de_extrapolate(DeMesh m, DeParams p, const DeQ *__restrict__ q, void *__restrict__ E,
               unsigned char *__restrict__ flags, double *__restrict__ part_mass,
               DeControl *ctl)
{
    __shared__ double red[DE_BLOCK / 64];
    const int lb = xcd_block();
    DeControl *cb = de_ctl(ctl, m.scen, lb);
    if (cb->done) return;
    int *err = &cb->status;
    const int N = m.N;
    const int k = lb * DE_BLOCK + threadIdx.x;
    double mass = 0.0;

    if (k < cb->kend) {
        DeExtrap<T> x;
        de_extrap_cell<T>(m, p, q, k, err, x);
        mass = x.mass;
        flags[k] = x.flag;
        if constexpr (sizeof(T) == 8) {
            // FP64 edge values: four [edge][triangle] arrays (w, h, uh, vh)
            double *__restrict__ ow = reinterpret_cast<double *>(E);
            double *__restrict__ oh = ow + 3 * (size_t)N;
            double *__restrict__ ouh = ow + 6 * (size_t)N;
            double *__restrict__ ovh = ow + 9 * (size_t)N;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                double ew, eh, euh, evh;
                de_edge64(x, i, ew, eh, euh, evh);
                const int ki = i * N + k;
                ow[ki] = ew;
                oh[ki] = eh;
                ouh[ki] = euh;
                ovh[ki] = evh;
            }
        } else {
            DeEdgeRec32 rec;
#pragma unroll
            for (int i = 0; i < 3; i++) rec.e[i] = de_edge32(x, i);
            rec.hc = x.c.h;
            rec.pad = 0.0;
            reinterpret_cast<DeEdgeRec32 *>(E)[k] = rec;
        }
    }

    // block partial of protect's added mass
    mass = de_wave_sum(mass);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) red[wv] = mass;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = red[0];
        for (int i = 1; i < DE_BLOCK / 64; i++) t += red[i];
        part_mass[lb] = t;
    }
}

// Write the protect / momentum-zeroing outcome back into the centroid state
// (what the reference's distribute_to_vertices_and_edges leaves behind).
__global__ void __launch_bounds__(DE_BLOCK)
de_materialize(int N, DeQ *q, const unsigned char *__restrict__ flags)
{
    const int k = xcd_block() * DE_BLOCK + threadIdx.x;
    if (k >= N) return;
    const unsigned f = flags[k];
    if (f & DE_F_CLAMP) q[k].w = q[k].z;
    if (!(f & DE_F_KEEP)) {
        q[k].uh = 0.0;
        q[k].vh = 0.0;
    }
}

// ---------------------------------------------------------------------------
// friction + update + fix_negative_cells for one triangle
// ---------------------------------------------------------------------------
__device__ __forceinline__ double de_update_one(double q, double ex, double si, double dt,
                                                int *err)
{
    // quantity.c:786-812
    if (q == 0.0) si = 0.0;
    else si /= q;
    q += dt * ex;
    const double den = 1.0 - dt * si;
    if (den <= 0.0) {
        atomicOr(err, DE_ERR_SEMI_IMPLICIT);
        return q;
    }
    return q / den;
}

// bed terms of sloped friction for one triangle
struct DeSlope {
    bool on;
    double zs, zmean;
};

// The vertex beds of the last extrapolation (edge bed z_e = w_e - h_e, vertex
// = sum of the two other edges minus the opposite one, sw_domain_orig.c:2660-2668)
// and their plane's gradient (_gradient, anuga/utilities/util_ext.h:52-92).
__device__ __forceinline__ DeSlope de_sloped_bed(const double *__restrict__ E, int N, int k,
                                                 const double *__restrict__ vx)
{
    const double *Ew = E, *Eh = E + 3 * (size_t)N;
    double ze[3];
#pragma unroll
    for (int i = 0; i < 3; i++) ze[i] = Ew[i * N + k] - Eh[i * N + k];
    const double z0 = ze[1] + ze[2] - ze[0];
    const double z1 = ze[0] + ze[2] - ze[1];
    const double z2 = ze[0] + ze[1] - ze[2];
    const double *x = vx + 6 * (size_t)k;
    const double x0 = x[0], y0 = x[1], x1 = x[2], y1 = x[3], x2 = x[4], y2 = x[5];
    const double det = (y2 - y0) * (x1 - x0) - (y1 - y0) * (x2 - x0);
    double a = (y2 - y0) * (z1 - z0) - (y1 - y0) * (z2 - z0);
    a /= det;
    double b = (x1 - x0) * (z2 - z0) - (x2 - x0) * (z1 - z0);
    b /= det;
    DeSlope s;
    s.on = true;
    s.zs = sqrt(1.0 + a * a + b * b);
    s.zmean = (z0 + z1 + z2) * (1.0 / 3.0);
    return s;
}

// The semi-implicit Manning coefficient S of one triangle:
// _manning_friction_flat with eps = minimum_allowed_height (friction.py:64-72),
// or _manning_friction_sloped (sw_domain_orig.c:2840-2888): depth over the
// mean vertex bed and the slope factor sqrt(1 + |grad z|^2). False where the
// reference adds nothing (n <= eps or a depth below eps).
__device__ __forceinline__ bool de_manning_S(const DeCentroid &c, double eta, const DeParams &p,
                                             const DeSlope &sl, double &S)
{
    if (!(eta > p.mah)) return false;
    const double h = c.w - (sl.on ? sl.zmean : c.z);
    if (!(h >= p.mah)) return false;
    S = sl.on ? -p.g * eta * eta * sl.zs * sqrt((c.uh * c.uh + c.vh * c.vh))
              : -p.g * eta * eta * sqrt((c.uh * c.uh + c.vh * c.vh));
    S /= de_pow_7_3(h);
    return true;
}

__device__ __forceinline__ DeQ de_advance(const DeCentroid c, double eta, double exw, double exuh,
                                          double exvh, double dt, const DeParams &p, int *err,
                                          unsigned long long *nneg,
                                          const DeSlope sl = DeSlope{false, 0.0, 0.0})
{
    double si_uh = 0.0, si_vh = 0.0, S;
    if (de_manning_S(c, eta, p, sl, S)) {
        si_uh += S * c.uh;
        si_vh += S * c.vh;
    }
    DeQ r;
    r.w = de_update_one(c.w, exw, 0.0, dt, err);
    r.uh = de_update_one(c.uh, exuh, si_uh, dt, err);
    r.vh = de_update_one(c.vh, exvh, si_vh, dt, err);
    r.z = c.z;
    // _orig_fix_negative_cells (every triangle is a full triangle here)
    if (r.w - c.z < 0.0) {
        atomicAdd(nneg, 1ull);
        r.w = c.z;
        r.uh = 0.0;
        r.vh = 0.0;
    }
    return r;
}

// The Runge-Kutta combination of substep SUBSTEP of the advanced state r with
// the step's initial state b (saxpy_centroid_values, quantity.c:752-769, with
// the weights of generic_domain.py:2018-2045 and :2053-2179):
// 1: rk2 end, 0.5 r + 0.5 b; 2: rk3 middle, 0.25 r + 0.75 b;
// 3: rk3 end, (2 r + 1 b) / 3.
template <int SUBSTEP>
__device__ __forceinline__ DeQ de_rk_combine(const DeQ &r, const DeQ &b)
{
    DeQ o;
    if constexpr (SUBSTEP == 1) {
        o.w = 0.5 * r.w + 0.5 * b.w;
        o.uh = 0.5 * r.uh + 0.5 * b.uh;
        o.vh = 0.5 * r.vh + 0.5 * b.vh;
    } else if constexpr (SUBSTEP == 2) {
        o.w = 0.25 * r.w + 0.75 * b.w;
        o.uh = 0.25 * r.uh + 0.75 * b.uh;
        o.vh = 0.25 * r.vh + 0.75 * b.vh;
    } else {
        o.w = (2.0 * r.w + 1.0 * b.w) / 3.0;
        o.uh = (2.0 * r.uh + 1.0 * b.uh) / 3.0;
        o.vh = (2.0 * r.vh + 1.0 * b.vh) / 3.0;
    }
    o.z = b.z;
    return o;
}

// ---------------------------------------------------------------------------
// riverwalls
// ---------------------------------------------------------------------------
// Blend the edge flux (normal frame, per unit length) towards the
// Villemonte-corrected weir discharge Qfactor 2/3 H sqrt(2/3 g H) (1 - Q2/Q1)^0.385,
// returning to the shallow-water flux between submergence s1 and s2 or
// tailwater-head / weir-height h1 and h2; the momentum fluxes take the mass
// flux's scaling (at most 10). sw_domain_orig.c:671-763, operation for operation.
__device__ __forceinline__ void de_weir_adjust(double ef[3], double hl, double hr, double g,
                                               double weir_height, const DeRiverwall &rw,
                                               double &speed)
{
    const double two3 = 2.0 / 3.0;
    const double minhd = fmin(hl, hr), maxhd = fmax(hl, hr);
    const double q1 = rw.qfactor * two3 * maxhd * sqrt(two3 * g * maxhd);
    const double q2 = rw.qfactor * two3 * minhd * sqrt(two3 * g * minhd);
    const double q_ratio = q2 / fmax(q1, 1.0e-100);
    const double h_ratio = minhd / fmax(maxhd, 1.0e-100);
    const double head_ratio = minhd / fmax(weir_height, 1.0e-100);
    double q = q1 * de_pow_0385(1.0 - q_ratio);
    if (hr > hl) q *= -1.0;
    if ((h_ratio < rw.s2) & (head_ratio < rw.h2)) {
        const double w1 = fmin(fmax(h_ratio - rw.s1, 0.0) / (rw.s2 - rw.s1), 1.0);
        const double w2 = fmin(fmax(head_ratio - rw.h1, 0.0) / (rw.h2 - rw.h1), 1.0);
        const double blended = (q * (1.0 - w1) + w1 * ef[0]) * (1.0 - w2) + w2 * ef[0];
        double scale = (fabs(ef[0]) > 1.0e-100) ? blended / ef[0] : 0.0;
        scale = fmax(scale, 0.0);
        ef[0] = blended;
        ef[1] *= fmin(scale, 10.0);
        ef[2] *= fmin(scale, 10.0);
    }
    if (fabs(ef[0]) > 0.0) speed = sqrt(g * (maxhd + weir_height)) + fabs(ef[0] / (maxhd + 1.0e-12));
}

// The weir on a riverwall edge: only where the crest stands above both cells'
// beds and either side's first-order head over z_half is positive
// (sw_domain_orig.c:905-968). wn, zn: the neighbour's centroid stage and bed
// (interior edges); on a boundary edge the right head is hc + zr - z_half.
__device__ __forceinline__ void de_riverwall_weir(const DeRiverwall &rw, double g, bool interior,
                                                  double wk, double zc, double hc, double wn,
                                                  double zn, double zl, double zr,
                                                  double z_half, double ef[3], double &speed)
{
    const double weir_height = fmax(rw.elev - fmin(zl, zr), 0.0);
    if (!(rw.elev > fmax(zc, zn))) return;
    const double hl = fmax(wk - z_half, 0.0);
    const double hr = interior ? fmax(wn - z_half, 0.0) : fmax(hc + zr - z_half, 0.0);
    if (!((hl > 0.0) || (hr > 0.0))) return;
    de_weir_adjust(ef, hl, hr, g, weir_height, rw, speed);
}

// ---------------------------------------------------------------------------
// flux
// ---------------------------------------------------------------------------
// One edge's terms of triangle k's flux sums (the body of the reference's
// edge loop, sw_domain_orig.c:828-1004, for the half-edge (k, i)): own edge
// values ql0 (stage), hle (depth), ql1, ql2 (momenta); for an interior edge
// (vi >= 0) the neighbour's at the shared edge, for a boundary edge the
// boundary state evaluated here. Adds to the sums sw, sx, sy, the boundary
// inflow and the CFL bound. Shared by the flux kernel and the tiled fused
// kernel, so both produce the same bits. fnb: where the neighbour's flag is
// (GENERAL walls; NULL: flags[n]).
template <class T, int SUBSTEP, bool GENERAL>
__device__ __forceinline__ void de_edge_terms(const DeMesh &m, const DeParams &p,
                                              const DeBoundary &bc, const DeQ *q,
                                              const unsigned char *__restrict__ flags, int N,
                                              int k, int i, int vi, const DeCentroid &c, T hc,
                                              T zc, T ql0, T hle, T ql1, T ql2, T qr0, T hre,
                                              T qr1, T qr2, T ef[3], T &pg, T &speed,
                                              const unsigned char *fnb = nullptr)
{
    const T g = T(p.g), eps = T(p.eps);
    const T zl = ql0 - hle;
    const T n1 = m.nx[i * N + k], n2 = m.ny[i * N + k];
    T zr;
    if (vi >= 0) {
        zr = qr0 - hre;
    } else {
        const int j = -vi - 1;
        const int kind = bc.kind[j];
        const double *bv = bc.val + (size_t)de_bc_slot<SUBSTEP>() * bc.sstride;
        if (kind == 0) {          // reflective
            const T r1 = -ql1 * n1 - ql2 * n2;
            const T r2 = -ql1 * n2 + ql2 * n1;
            qr0 = ql0;
            qr1 = n1 * r1 - n2 * r2;
            qr2 = n2 * r1 + n1 * r2;
        } else if (kind == 1) {   // transmissive
            qr0 = ql0;
            qr1 = ql1;
            qr2 = ql2;
        } else if (kind == 2) {   // Dirichlet (constant or time-dependent)
            qr0 = T(bv[j]);
            qr1 = T(bv[bc.M + j]);
            qr2 = T(bv[2 * bc.M + j]);
        } else if (kind == 3) {   // transmissive from centroid values
            qr0 = T(c.w);
            qr1 = T(c.uh);
            qr2 = T(c.vh);
        } else if (kind == 4) {   // stage set, normal momentum kept, tangential 0
            const T nq = n1 * ql1 + n2 * ql2;
            qr0 = T(bv[j]);
            qr1 = nq * n1;
            qr2 = nq * n2;
        } else if (kind == 5) {   // transmissive stage, zero momentum
            qr0 = ql0;
            qr1 = T(0.0);
            qr2 = T(0.0);
        } else {                  // stage set, momentum transmissive
            qr0 = T(bv[j]);
            qr1 = ql1;
            qr2 = ql2;
        }
        zr = zl;
        hre = fmax(qr0 - zr, T(0.0));
    }
    T z_half = fmax(zl, zr);
    int wall = -1;
    bool mirrored = false;
    if constexpr (GENERAL) {
        // the wall is a thin bed step between the two half-edges
        // (sw_domain_orig.c:880-893)
        if (m.rw) {
            wall = m.rw[i * N + k];
            if (wall >= 0) z_half = fmax(m.rwd[wall].elev, z_half);
        }
        if (p.low_froude && vi >= 0) mirrored = m.caller[vi >> 2] < m.caller[k];
    }
    const T h_left = fmax(hle + zl - z_half, T(0.0));
    const T h_right = fmax(hre + zr - z_half, T(0.0));
    T pflux;
    if constexpr (GENERAL)
        de_flux_central<T>(ql0, ql1, ql2, qr0, qr1, qr2, h_left, h_right, hle, hre, n1,
                           n2, eps, z_half, g, ef, speed, pflux, p.low_froude, mirrored);
    else
        de_flux_central<T>(ql0, ql1, ql2, qr0, qr1, qr2, h_left, h_right, hle, hre, n1,
                           n2, eps, z_half, g, ef, speed, pflux);
    if constexpr (GENERAL) {
        if (wall >= 0) {
            double wn = 0.0, zn = c.z;
            if (vi >= 0) {
                const int n = vi >> 2;
                // the neighbour's protect flag: from the flag array, or from
                // the fused kernel's LDS (fnb), where a halo neighbour's is
                const DeCentroid cn = de_centroid(q[n], fnb ? *fnb : flags[n]);
                wn = cn.w;
                zn = cn.z;
            }
            de_riverwall_weir(m.rwd[wall], p.g, vi >= 0, c.w, c.z, hc, wn, zn, zl, zr,
                              z_half, ef, speed);
        }
    }
    const T length = m.len[i * N + k];
    ef[0] *= length;
    ef[1] *= length;
    ef[2] *= length;
    pg = length * (-g * T(0.5) * (h_left * h_left - hle * hle - (hle + hc) * (zl - zc)) + pflux);
}

// de_edge_terms added to triangle k's sums (sw_domain_orig.c:1107-1132, the
// edge's flux, then its pressure terms along the normal), the boundary inflow
// and the CFL bound
template <class T, int SUBSTEP, bool GENERAL>
__device__ __forceinline__ void de_edge_flux(const DeMesh &m, const DeParams &p,
                                             const DeBoundary &bc, const DeQ *q,
                                             const unsigned char *__restrict__ flags, int N,
                                             int k, int i, int vi, const DeCentroid &c, T hc,
                                             T zc, T ql0, T hle, T ql1, T ql2, T qr0, T hre,
                                             T qr1, T qr2, double &sw, double &sx, double &sy,
                                             double &bflux, double &dtmin,
                                             const unsigned char *fnb = nullptr)
{
    T ef[3], pg, speed;
    de_edge_terms<T, SUBSTEP, GENERAL>(m, p, bc, q, flags, N, k, i, vi, c, hc, zc, ql0, hle, ql1,
                                       ql2, qr0, hre, qr1, qr2, ef, pg, speed, fnb);
    const T n1 = m.nx[i * N + k], n2 = m.ny[i * N + k];
    sw += double(-ef[0]);
    sx += double(-ef[1]);
    sy += double(-ef[2]);
    if (vi < 0) bflux += double(-ef[0]);
    sx -= double(n1 * pg);
    sy -= double(n2 * pg);
    if (SUBSTEP == 0 && double(speed) > p.eps) {
        const double t = 1.0 / fmax(double(speed), p.eps);
        dtmin = fmin(dtmin, m.radius[k] * t);
    }
}

// SUBSTEP 0: writes explicit updates; SUBSTEP > 0: advances with the
// scenario's dt and writes de_rk_combine<SUBSTEP>(advanced, bk) to out (out
// may be bk, or q itself: each thread reads its own q and bk before writing).
// STAGE: substep 0 writes the explicit updates and advances with dt to out.
// GENERAL: the instantiation for riverwalls, low_froude 1/2 and sloped
// friction (runtime switches), so that the common kernel carries none of
// their registers.
template <class T, int SUBSTEP, bool GENERAL = false, bool STAGE = false>
__global__ void __launch_bounds__(DE_BLOCK)
de_flux(DeMesh m, DeParams p, const DeQ *q, const double *__restrict__ eta,
        const T *__restrict__ E, DeBoundary bc, const unsigned char *__restrict__ flags,
        double *__restrict__ exw, double *__restrict__ exuh, double *__restrict__ exvh,
        const DeQ *bk, DeQ *out, DeControl *ctl,
        const DeControl *dctl, double *__restrict__ part_dt,
        double *__restrict__ part_bf, unsigned long long *__restrict__ nneg)
{
    __shared__ double red_dt[DE_BLOCK / 64];
    __shared__ double red_bf[DE_BLOCK / 64];
    const int lb = xcd_block();
    DeControl *cb = de_ctl(ctl, m.scen, lb);
    if (cb->done) return;
    int *err = &cb->status;
    const double dt = SUBSTEP || STAGE ? dctl[cb - ctl].dt : 0.0;
    const int N = m.N;
    const int k = lb * DE_BLOCK + threadIdx.x;
    double dtmin = 1.0e100, bflux = 0.0;

    if (k < cb->kend) {
        const DeCentroid c = de_centroid(q[k], flags[k]);
        const int4 vk = m.nb[k];
        const int v[3] = {vk.x, vk.y, vk.z};
        const T *__restrict__ Ew = E;
        const T *__restrict__ Eh = E + 3 * (size_t)N;
        const T *__restrict__ Euh = E + 6 * (size_t)N;
        const T *__restrict__ Evh = E + 9 * (size_t)N;
        const T hc = T(de_height(c.w, c.z));
        const T zc = T(c.z);
        double sw = 0.0, sx = 0.0, sy = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int ki = i * N + k;
            const T ql0 = Ew[ki], hle = Eh[ki], ql1 = Euh[ki], ql2 = Evh[ki];
            T qr0 = T(0.0), qr1 = T(0.0), qr2 = T(0.0), hre = T(0.0);
            if (v[i] >= 0) {
                const int nm = (v[i] & 3) * N + (v[i] >> 2);
                qr0 = Ew[nm];
                qr1 = Euh[nm];
                qr2 = Evh[nm];
                hre = Eh[nm];
            }
            de_edge_flux<T, SUBSTEP, GENERAL>(m, p, bc, q, flags, N, k, i, v[i], c, hc, zc, ql0,
                                              hle, ql1, ql2, qr0, hre, qr1, qr2, sw, sx, sy,
                                              bflux, dtmin);
        }
        const double inv_area = 1.0 / m.area[k];
        sw *= inv_area;
        sx *= inv_area;
        sy *= inv_area;
        if (SUBSTEP == 0) {
            exw[k] = sw;
            exuh[k] = sx;
            exvh[k] = sy;
            if constexpr (STAGE)
                out[k] = de_advance(c, eta[k], sw, sx, sy, dt, p, err, nneg);
        } else {
            DeSlope sl{false, 0.0, 0.0};
            if constexpr (GENERAL)
                if (p.sloped) sl = de_sloped_bed((const double *)E, N, k, m.vx);
            const DeQ r = de_advance(c, eta[k], sw, sx, sy, dt, p, err, nneg, sl);
            out[k] = de_rk_combine<SUBSTEP>(r, bk[k]);
        }
    }

    dtmin = de_wave_min(dtmin);
    bflux = de_wave_sum(bflux);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        red_dt[wv] = dtmin;
        red_bf[wv] = bflux;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = red_dt[0], b = red_bf[0];
        for (int i = 1; i < DE_BLOCK / 64; i++) {
            a = fmin(a, red_dt[i]);
            b += red_bf[i];
        }
        part_dt[lb] = a;
        part_bf[lb] = b;
    }
}

// ---------------------------------------------------------------------------
// local flux updating (euler steps, FP64, the common options)
// ---------------------------------------------------------------------------
// compute_fluxes with local flux updating (sw_domain_orig.c:765-1150 with the
// skip test at :829): each triangle evaluates those of its half-edges whose
// update flag is set (both halves of an edge carry the same flag, and each
// half's terms are the bits the reference mirrors to it), stores their terms,
// edge timesteps and the call number, and sums the stored terms of all three
// edges, fresh or not (:1107-1139). The CFL partials cover the evaluated
// edges; the inflow partials every boundary edge's stored flux.
__global__ void __launch_bounds__(DE_BLOCK)
de_flux_lts(DeMesh m, DeParams p, const DeQ *q, const double *__restrict__ E, DeBoundary bc,
            const unsigned char *__restrict__ flags, double *__restrict__ exw,
            double *__restrict__ exuh, double *__restrict__ exvh, DeLts lt, int call,
            DeControl *ctl, double *__restrict__ part_dt, double *__restrict__ part_bf)
{
    __shared__ double red_dt[DE_BLOCK / 64];
    __shared__ double red_bf[DE_BLOCK / 64];
    const int lb = xcd_block();
    DeControl *cb = de_ctl(ctl, m.scen, lb);
    if (cb->done) return;
    const int N = m.N;
    const int k = lb * DE_BLOCK + threadIdx.x;
    double dtmin = 1.0e100, bflux = 0.0;

    if (k < cb->kend) {
        const DeCentroid c = de_centroid(q[k], flags[k]);
        const int4 vk = m.nb[k];
        const int v[3] = {vk.x, vk.y, vk.z};
        const double *__restrict__ Ew = E;
        const double *__restrict__ Eh = E + 3 * (size_t)N;
        const double *__restrict__ Euh = E + 6 * (size_t)N;
        const double *__restrict__ Evh = E + 9 * (size_t)N;
        const double hc = de_height(c.w, c.z);
        const double zc = c.z;
        double sw = 0.0, sx = 0.0, sy = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int ki = i * N + k;
            double e0, e1, e2, pg;
            if (lt.unf[ki]) {
                const double ql0 = Ew[ki], hle = Eh[ki], ql1 = Euh[ki], ql2 = Evh[ki];
                double qr0 = 0.0, qr1 = 0.0, qr2 = 0.0, hre = 0.0;
                if (v[i] >= 0) {
                    const int nm = (v[i] & 3) * N + (v[i] >> 2);
                    qr0 = Ew[nm];
                    qr1 = Euh[nm];
                    qr2 = Evh[nm];
                    hre = Eh[nm];
                }
                double ef[3], speed;
                de_edge_terms<double, 0, false>(m, p, bc, q, flags, N, k, i, v[i], c, hc, zc,
                                                ql0, hle, ql1, ql2, qr0, hre, qr1, qr2, ef, pg,
                                                speed);
                e0 = -ef[0];
                e1 = -ef[1];
                e2 = -ef[2];
                const double t = 1.0 / fmax(speed, p.eps);
                const double et = m.radius[k] * t;
                lt.e0[ki] = e0;
                lt.e1[ki] = e1;
                lt.e2[ki] = e2;
                lt.pg[ki] = pg;
                lt.et[ki] = et;
                lt.acf[ki] = call;
                if (speed > p.eps) dtmin = fmin(dtmin, et);
            } else {
                e0 = lt.e0[ki];
                e1 = lt.e1[ki];
                e2 = lt.e2[ki];
                pg = lt.pg[ki];
            }
            const double n1 = m.nx[ki], n2 = m.ny[ki];
            sw += e0;
            sx += e1;
            sy += e2;
            if (v[i] < 0) bflux += e0;
            sx -= n1 * pg;
            sy -= n2 * pg;
        }
        const double inv_area = 1.0 / m.area[k];
        exw[k] = sw * inv_area;
        exuh[k] = sx * inv_area;
        exvh[k] = sy * inv_area;
    }

    dtmin = de_wave_min(dtmin);
    bflux = de_wave_sum(bflux);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        red_dt[wv] = dtmin;
        red_bf[wv] = bflux;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = red_dt[0], b = red_bf[0];
        for (int i = 1; i < DE_BLOCK / 64; i++) {
            a = fmin(a, red_dt[i]);
            b += red_bf[i];
        }
        part_dt[lb] = a;
        part_bf[lb] = b;
    }
}

// The update frequency derived from an edge pair's timesteps
// (sw_domain_orig.c:573-600): int(min(et / dt, M)) of each side, the smaller,
// clamped to [1, M] and rounded down to a power of two.
__device__ __forceinline__ int de_lts_frequency(double et_a, double et_b, bool pair, int M,
                                                double timestep)
{
    const double notSoFast = 1.0;
    long long f = (long long)fmin((et_a / timestep) * notSoFast, M * 1.0);
    if (pair) f = (long long)fmin((double)(long long)fmin(et_b / timestep * notSoFast, M * 1.0),
                                  (double)f);
    if (f < 1) f = 1;
    if (f > M) f = M;
    for (long long ii = 2; ii < M; ii *= 2)
        if (f > ii && f < 2 * ii) f = ii;
    return (int)f;
}

// _compute_flux_update_frequency, part 1 (sw_domain_orig.c:540-608), for
// triangle k's half-edges; cyc is the step count modulo M. The two halves of
// an edge hold the same frequency and already_computed_flux, so each half
// replays the reference's two visits of the pair on its own copy: with a
// positive call number the first visit derives the frequency and flips the
// sign, and a second visit, made only if the new frequency divides cyc,
// flips it back; with a negative one the first visit flips and the second
// flips back and derives it; 0 (never evaluated) changes nothing. A boundary
// edge has one visit: it flips the sign and derives the frequency if the sign
// was positive. Then part 2's first loop (:618-628): tmin[k], the smallest of
// the three.
__global__ void __launch_bounds__(DE_BLOCK)
de_lts_part1(int kend, int N, const int4 *__restrict__ nb, DeLts lt, long long cyc, int M,
             double timestep)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= kend) return;
    const int4 vk = nb[k];
    const int v[3] = {vk.x, vk.y, vk.z};
    int fmin3 = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const int ki = i * N + k;
        int f = lt.fuf[ki];
        if ((cyc & (long long)(f - 1)) == 0) {
            int a = lt.acf[ki];
            bool derive;
            if (v[i] >= 0) {
                derive = a != 0;
            } else {
                derive = a > 0;
                a = -a;
            }
            if (derive) {
                const double etb = v[i] >= 0 ? lt.et[(v[i] & 3) * N + (v[i] >> 2)] : 0.0;
                f = de_lts_frequency(lt.et[ki], etb, v[i] >= 0, M, timestep);
                if (v[i] >= 0 && a > 0 && (cyc & (long long)(f - 1)) != 0) a = -a;
                lt.fuf[ki] = f;
            }
            lt.acf[ki] = a;
        }
        fmin3 = i == 0 ? f : min(fmin3, f);
    }
    lt.tmin[k] = fmin3;
}

// part 2's second loop (:636-656): each half-edge takes the smaller of its
// two triangles' minima, and is evaluated on the next call when its frequency
// divides the next step count.
__global__ void __launch_bounds__(DE_BLOCK)
de_lts_part2(int kend, int N, const int4 *__restrict__ nb, DeLts lt, long long cyc_next)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= kend) return;
    const int4 vk = nb[k];
    const int v[3] = {vk.x, vk.y, vk.z};
    const int tk = lt.tmin[k];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const int ki = i * N + k;
        const int f = v[i] >= 0 ? min(tk, lt.tmin[v[i] >> 2]) : tk;
        lt.fuf[ki] = f;
        lt.unf[ki] = (cyc_next & (long long)(f - 1)) == 0 ? 1 : 0;
    }
}

// initial state: nothing stored, every edge evaluated, frequency 1, edge
// timesteps 1e100 (shallow_water_domain.py:404-426)
__global__ void __launch_bounds__(DE_BLOCK)
de_lts_init(int n3, DeLts lt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    lt.e0[i] = 0.0;
    lt.e1[i] = 0.0;
    lt.e2[i] = 0.0;
    lt.pg[i] = 0.0;
    lt.et[i] = 1.0e100;
    lt.fuf[i] = 1;
    lt.acf[i] = 0;
    lt.unf[i] = 1;
}

// Tiled fused extrapolation + flux (FP64, any SUBSTEP; out never aliases q).
// GENERAL: riverwalls, low_froude 1/2 and sloped friction, with the tile's
// and the halo's protect flags in LDS for the walls' neighbour centroids;
// with sloped friction each triangle also writes its edge stage and depth to
// Eg, which the sloped update and the later substeps' friction read. A workgroup extrapolates its tile's DE_BLOCK triangles and
// its halo (the neighbour triangles outside the tile, each once) into LDS, then each thread gathers its triangle's three edge fluxes
// from LDS. The edge values never reach HBM. The arithmetic is
// de_extrap_cell and de_edge_flux, as in de_extrapolate and de_flux, and the
// per-block partials (CFL, boundary inflow, protect mass) are formed in the
// same order, so the results are the same bits. The state read (q) is never
// written by this kernel: later substeps write out, the step's initial state
// (rk2, rk3's last) or a third buffer (rk3's middle).
template <int SUBSTEP, bool GENERAL = false>
__global__ void __launch_bounds__(DE_BLOCK)
de_xflux(DeMesh m, DeParams p, const DeQ *__restrict__ q, const double *__restrict__ eta,
         DeTiles tl, DeBoundary bc, unsigned char *__restrict__ flags, double *__restrict__ exw,
         double *__restrict__ exuh, double *__restrict__ exvh, const DeQ *bk, DeQ *out,
         DeControl *ctl,
         const DeControl *dctl, double *__restrict__ part_dt, double *__restrict__ part_bf,
         double *__restrict__ part_mass, unsigned long long *__restrict__ nneg,
         double *__restrict__ Eg)
{
    // [4 quantities][3 edges][DE_BLOCK] tile edge values, then [4][3][hcap] halo
    extern __shared__ double lds[];
    __shared__ double red_dt[DE_BLOCK / 64], red_bf[DE_BLOCK / 64], red_m[DE_BLOCK / 64];
    const int lb = tl.list ? tl.list[xcd_block()] : xcd_block();
    DeControl *cb = de_ctl(ctl, m.scen, lb);
    if (cb->done) return;
    int *err = &cb->status;
    const double dt = SUBSTEP ? dctl[cb - ctl].dt : 0.0;
    const int N = m.N, t = threadIdx.x;
    const int k0 = lb * DE_BLOCK, k = k0 + t;
    const int kend = cb->kend;
    const int hcap = tl.hcap;
    double *const hl = lds + 12 * DE_BLOCK;
    // GENERAL: the protect flags of the tile's and the halo's triangles
    unsigned char *const lfl = reinterpret_cast<unsigned char *>(hl + 12 * hcap);
    double mass = 0.0, dtmin = 1.0e100, bflux = 0.0;
    unsigned fk = 0;

    if (k < kend) {
        DeExtrap<double> x;
        de_extrap_cell<double>(m, p, q, k, err, x);
        mass = x.mass;
        fk = x.flag;
        flags[k] = (unsigned char)fk;
        if constexpr (GENERAL) lfl[t] = (unsigned char)fk;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double ew, eh, euh, evh;
            de_edge64(x, i, ew, eh, euh, evh);
            lds[(0 + i) * DE_BLOCK + t] = ew;
            lds[(3 + i) * DE_BLOCK + t] = eh;
            lds[(6 + i) * DE_BLOCK + t] = euh;
            lds[(9 + i) * DE_BLOCK + t] = evh;
            if constexpr (GENERAL) {
                // sloped friction reads the triangle's edge stage and depth
                // (its vertex beds) from HBM, in the update and below
                if (p.sloped) {
                    Eg[(size_t)i * N + k] = ew;
                    Eg[3 * (size_t)N + (size_t)i * N + k] = eh;
                }
            }
        }
    }
    // halo triangles: all three edges, so that the edge is chosen by the
    // reader's LDS address (a run-time choice between the registers of x
    // would place x in scratch)
    const int h0 = tl.start[lb], nh = tl.start[lb + 1] - h0;
    for (int j = t; j < nh; j += DE_BLOCK) {
        DeExtrap<double> x;
        de_extrap_cell<double>(m, p, q, tl.halo[h0 + j], err, x);
        if constexpr (GENERAL) lfl[DE_BLOCK + j] = (unsigned char)x.flag;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double ew, eh, euh, evh;
            de_edge64(x, i, ew, eh, euh, evh);
            hl[(0 + i) * hcap + j] = ew;
            hl[(3 + i) * hcap + j] = eh;
            hl[(6 + i) * hcap + j] = euh;
            hl[(9 + i) * hcap + j] = evh;
        }
    }
    __syncthreads();

    if (k < kend) {
        const DeCentroid c = de_centroid(q[k], fk);
        const int4 vk = m.nb[k];
        const int v[3] = {vk.x, vk.y, vk.z};
        const unsigned sl = tl.slot[k];
        const double hc = de_height(c.w, c.z);
        const double zc = c.z;
        double sw = 0.0, sx = 0.0, sy = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const double ql0 = lds[(0 + i) * DE_BLOCK + t], hle = lds[(3 + i) * DE_BLOCK + t];
            const double ql1 = lds[(6 + i) * DE_BLOCK + t], ql2 = lds[(9 + i) * DE_BLOCK + t];
            double qr0 = 0.0, qr1 = 0.0, qr2 = 0.0, hre = 0.0;
            const unsigned char *fnb = nullptr;
            if (v[i] >= 0) {
                const unsigned s = (sl >> (10 * i)) & 1023u;
                const double *src;
                int stride;
                if (s == 1023u) {
                    src = lds + (v[i] & 3) * DE_BLOCK + ((v[i] >> 2) - k0);
                    stride = 3 * DE_BLOCK;
                    if constexpr (GENERAL) fnb = lfl + ((v[i] >> 2) - k0);
                } else {
                    src = hl + (v[i] & 3) * hcap + s;
                    stride = 3 * hcap;
                    if constexpr (GENERAL) fnb = lfl + DE_BLOCK + s;
                }
                qr0 = src[0];
                hre = src[stride];
                qr1 = src[2 * stride];
                qr2 = src[3 * stride];
            }
            de_edge_flux<double, SUBSTEP, GENERAL>(m, p, bc, q, flags, N, k, i, v[i], c, hc, zc,
                                                   ql0, hle, ql1, ql2, qr0, hre, qr1, qr2, sw,
                                                   sx, sy, bflux, dtmin, fnb);
        }
        const double inv_area = 1.0 / m.area[k];
        sw *= inv_area;
        sx *= inv_area;
        sy *= inv_area;
        if (SUBSTEP == 0) {
            exw[k] = sw;
            exuh[k] = sx;
            exvh[k] = sy;
        } else {
            DeSlope sl{false, 0.0, 0.0};
            if constexpr (GENERAL)
                if (p.sloped) sl = de_sloped_bed(Eg, N, k, m.vx);
            const DeQ r = de_advance(c, eta[k], sw, sx, sy, dt, p, err, nneg, sl);
            out[k] = de_rk_combine<SUBSTEP>(r, bk[k]);
        }
    }

    dtmin = de_wave_min(dtmin);
    bflux = de_wave_sum(bflux);
    mass = de_wave_sum(mass);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        red_dt[wv] = dtmin;
        red_bf[wv] = bflux;
        red_m[wv] = mass;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = red_dt[0], b = red_bf[0], cm = red_m[0];
        for (int i = 1; i < DE_BLOCK / 64; i++) {
            a = fmin(a, red_dt[i]);
            b += red_bf[i];
            cm += red_m[i];
        }
        part_dt[lb] = a;
        part_bf[lb] = b;
        part_mass[lb] = cm;
    }
}

// The workgroup's partial results: its smallest CFL timestep, boundary flux
// and protect mass (substep 0), or its boundary flux alone (the later
// substeps' reductions read nothing else). A sum whose lanes are all zero is
// zero without the exchange.
__device__ __forceinline__ double de_wave_sum_nz(double x)
{
    return __ballot(x != 0.0) ? de_wave_sum(x) : 0.0;
}

template <int SUBSTEP>
__device__ __forceinline__ void de_block_partials(double dtmin, double bflux, double mass,
                                                  double *red_dt, double *red_bf, double *red_m,
                                                  double *part_dt, double *part_bf,
                                                  double *part_mass, int lb)
{
    if (SUBSTEP == 0) dtmin = de_wave_min(dtmin);
    bflux = de_wave_sum_nz(bflux);
    if (SUBSTEP == 0) mass = de_wave_sum_nz(mass);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        red_dt[wv] = dtmin;
        red_bf[wv] = bflux;
        red_m[wv] = mass;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = red_dt[0], b = red_bf[0], cm = red_m[0];
        for (int i = 1; i < DE_BLOCK / 64; i++) {
            a = fmin(a, red_dt[i]);
            b += red_bf[i];
            cm += red_m[i];
        }
        if (SUBSTEP == 0) {
            part_dt[lb] = a;
            part_mass[lb] = cm;
        }
        part_bf[lb] = b;
    }
}

// the three 10-bit fields of a word
__device__ __forceinline__ int de_field(unsigned w, int i) { return (int)((w >> (10 * i)) & 1023u); }

// The protected cell of a triangle with state q (sw_domain_orig.c:1245-1276,
// :2014-2064) before the dry-neighbour test: the velocity of a cell deeper
// than mah, which that test may still zero.
__device__ __forceinline__ DeCell de_wet_cell(const DeQ &q, double mah)
{
    DeCell c;
    c.w = de_clamped(q.w, q.z, mah) ? q.z : q.w;
    c.h = de_height(c.w, q.z);
    c.u = 0.0;
    c.v = 0.0;
    if (c.h > mah) {
        const double inv = 1.0 / c.h;
        c.u = q.uh * inv;
        c.v = q.vh * inv;
    }
    return c;
}

// The cells of a tile in LDS: [w, h, u, v, centroid x, y][2 DE_BLOCK]
#define DE_XSTRIDE (2 * DE_BLOCK)
__device__ __forceinline__ void de_put_cell(double *L, int j, const DeCell &v, const double2 &cen)
{
    L[j] = v.w;
    L[DE_XSTRIDE + j] = v.h;
    L[2 * DE_XSTRIDE + j] = v.u;
    L[3 * DE_XSTRIDE + j] = v.v;
    L[4 * DE_XSTRIDE + j] = cen.x;
    L[5 * DE_XSTRIDE + j] = cen.y;
}

// What the extrapolation of a triangle reads of the cells: its own after the
// dry-neighbour test, its surrogate neighbours', and their centroids (VG). v:
// negative on boundary edges (only the signs are used).
struct DeStencil {
    DeCell own, nb[3];
    double2 ck, c0, c1, c2;
    int v[3], nbound;
    bool keep;     // the momentum survives
};

// The stencil st of the triangle with cell `self` from the cells in LDS, as
// de_extrap_cell forms it from the records in memory: the same operations on
// the same values. The triangle's id k (of kp, if given) is read only where
// it is dry.
template <bool VG>
__device__ __forceinline__ void de_read_stencil(const DeMesh &m, const DeParams &p,
                                                const DeQ *__restrict__ q, const int *kp, int k,
                                                unsigned st, int self, const double *L,
                                                DeStencil &x)
{
    const double mah = p.mah;
    x.own.w = L[self];
    x.own.h = L[DE_XSTRIDE + self];
    x.own.u = L[2 * DE_XSTRIDE + self];
    x.own.v = L[3 * DE_XSTRIDE + self];
    int idx[3];
    x.nbound = 0;
    bool dry_k = true;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const int f = de_field(st, i);
        const bool edge = f == 1023;
        x.v[i] = edge ? -1 : 0;
        x.nbound += edge;
        idx[i] = edge ? self : f;
        x.nb[i].w = L[idx[i]];
        x.nb[i].h = L[DE_XSTRIDE + idx[i]];
        x.nb[i].u = L[2 * DE_XSTRIDE + idx[i]];
        x.nb[i].v = L[3 * DE_XSTRIDE + idx[i]];
        dry_k = dry_k && (edge || x.nb[i].h < mah);
    }
    if constexpr (VG) {
        const double *cx = L + 4 * DE_XSTRIDE, *cy = L + 5 * DE_XSTRIDE;
        x.ck = make_double2(cx[self], cy[self]);
        x.c0 = make_double2(cx[idx[0]], cy[idx[0]]);
        x.c1 = make_double2(cx[idx[1]], cy[idx[1]]);
        x.c2 = make_double2(cx[idx[2]], cy[idx[2]]);
    }
    x.keep = x.own.h > mah && !dry_k;
    if (!x.keep) {
        x.own.u = x.own.v = 0.0;
        // a boundary edge's surrogate is the triangle itself
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (x.v[i] < 0) x.nb[i].u = x.nb[i].v = 0.0;
    }
    if (x.own.h < mah && x.nbound < 3) {
        // a wet neighbour keeps its velocity unless all of its own neighbours
        // are dry; this triangle is one, so the others count only here
        const int4 vk = m.nb[kp ? *kp : k];
        const int vn[3] = {vk.x, vk.y, vk.z};
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (vn[i] >= 0 && x.nb[i].h > mah) {
                const int4 vs = m.nb[vn[i] >> 2];
                const int vv[3] = {vs.x, vs.y, vs.z};
                bool dry = true;
#pragma unroll
                for (int r = 0; r < 3; r++)
                    if (vv[r] >= 0) {
                        const DeQ t = q[vv[r] >> 2];
                        dry = dry && (de_height(t.w, t.z) < mah);
                    }
                if (dry) x.nb[i].u = x.nb[i].v = 0.0;
            }
    }
}

// The extrapolation of a stencil; nd: the nodes of word vi (VG), otherwise the
// stored record of triangle k.
template <bool VG>
__device__ __forceinline__ void de_extrap_stencil(const DeMesh &m, const DeParams &p, int k,
                                                  const DeStencil &s, const double2 *nd,
                                                  unsigned vi, int *err, DeExtrap<double> &x)
{
    x.c = s.own;
    double dxv[3], dyv[3];
    if constexpr (VG) {
        const DeVerts tv{nd[de_field(vi, 0)], nd[de_field(vi, 1)], nd[de_field(vi, 2)]};
        de_vertex_offsets(s.ck, tv, dxv, dyv);
        const DeCentroidGeo geo{s.ck, s.c0, s.c1, s.c2};
        de_extrap_jumps<double>(p, s.v, s.nbound, s.nb, dxv, dyv, geo, err, x);
    } else {
        const DeStoredGeo<double> geo(m, k, dxv, dyv);
        de_extrap_jumps<double>(p, s.v, s.nbound, s.nb, dxv, dyv, geo, err, x);
    }
}

// One listed edge of a tile (de_xflux_e): its flux from the tile triangle's
// side, written over the LDS edge values that only this entry reads. he: the
// halo edge it is (its neighbour in the halo), or negative: the neighbour is
// in the tile, and its side's pressure term and CFL bound are formed here too.
template <int SUBSTEP, bool VG>
__device__ __forceinline__ void de_tile_edge(const DeMesh &m, const DeParams &p, unsigned en,
                                             int he, int k0, double *lds, double *hl,
                                             const double *hz, int hecap, const double2 *nd,
                                             const unsigned *vis, double &dtmin)
{
    constexpr int Q = 3 * DE_BLOCK;
    const double g = p.g, eps = p.eps;
    const int N = m.N;
    const int ta = DE_TE_T(en), ia = DE_TE_I(en), nb = DE_TE_N(en), jb = DE_TE_J(en);
    const bool halo = he >= 0;
    const int ka = k0 + ta;
    double *const A = lds + ia * DE_BLOCK + ta;
    double *const R = halo ? hl + he : lds + jb * DE_BLOCK + nb;
    const int rs = halo ? hecap : Q;
    const double ql0 = A[0], hle = A[Q], ql1 = A[2 * Q], ql2 = A[3 * Q];
    const double qr0 = R[0], hre = R[rs], qr1 = R[2 * rs], qr2 = R[3 * rs];
    double n1, n2, length;
    if constexpr (VG) {
        const unsigned w = vis[ta];
        const int a = ia == 2 ? 0 : ia + 1, b = ia == 0 ? 2 : ia - 1;
        de_vertex_normal(nd[de_field(w, a)], nd[de_field(w, b)], n1, n2, length);
    } else {
        n1 = m.nx[ia * N + ka];
        n2 = m.ny[ia * N + ka];
        length = m.len[ia * N + ka];
    }
    // the CFL radii, requested before the flux that decides whether they are
    // used: 206.0 -> 200.7 us substep 0 at 4M triangles
    double ra = 0.0, rb = 0.0;
    if (SUBSTEP == 0) {
        ra = m.radius[ka];
        rb = halo ? ra : m.radius[k0 + nb];
    }
    const double zl = ql0 - hle, zr = qr0 - hre;
    const double z_half = fmax(zl, zr);
    const double h_left = fmax(hle + zl - z_half, 0.0);
    const double h_right = fmax(hre + zr - z_half, 0.0);
    double ef[3], speed, pflux;
    de_flux_central<double>(ql0, ql1, ql2, qr0, qr1, qr2, h_left, h_right, hle, hre, n1, n2,
                            eps, z_half, g, ef, speed, pflux);
    ef[0] *= length;
    ef[1] *= length;
    ef[2] *= length;
    const double hca = hz[ta], zca = hz[DE_BLOCK + ta];
    const double pga = length * (-g * 0.5 * (h_left * h_left - hle * hle -
                                             (hle + hca) * (zl - zca)) + pflux);
    A[0] = -ef[0];
    A[Q] = -ef[1];
    A[2 * Q] = -ef[2];
    A[3 * Q] = n1 * pga;
    R[0] = n2 * pga;
    double tt = 0.0;
    const bool cfl = SUBSTEP == 0 && speed > eps;
    if (cfl) {
        tt = 1.0 / fmax(speed, eps);
        dtmin = fmin(dtmin, ra * tt);
    }
    if (!halo) {
        // the other side: its own depths and bed, the same flux
        const double hcb = hz[nb], zcb = hz[DE_BLOCK + nb];
        const double pgb = length * (-g * 0.5 * (h_right * h_right - hre * hre -
                                                 (hre + hcb) * (zr - zcb)) + pflux);
        R[rs] = n1 * pgb;
        R[2 * rs] = n2 * pgb;
        if (cfl) dtmin = fmin(dtmin, rb * tt);
    }
}

// The fused FP64 kernel with each edge's flux evaluated once (the common
// options: no riverwalls, low_froude 0, flat friction; the mesh's normals and
// lengths mirror exactly across every interior edge). VG: the geometry is
// formed from the vertices. Phases, with a barrier after each:
//  0. the state of the tile, its halo and the halo's neighbours becomes cells
//     in LDS (protected stage, depth, velocity, centroid), each formed once,
//     with the vertices beside them;
//  1. every thread extrapolates its triangle from the cells (de_extrap_jumps,
//     as de_xflux), and one thread per halo edge reads that halo triangle's
//     stencil into registers. The tile's edge values take the cells' place in
//     LDS, one barrier later;
//  2. the first waves extrapolate the halo while each thread of the others
//     evaluates one edge inside the tile, from its lower-numbered side, which
//     also forms the other side's pressure term (the reference's compute-
//     once-and-mirror loop, sw_domain_orig.c:996-1009);
//  3. the tile's remaining edges and the edges to the halo (from the tile's
//     side) in one pass over all the waves;
//  4. each thread gathers its triangle's three edges in local order as
//     de_xflux does: the same operations on the same values, so the same bits
//     (the other side's flux is exactly the negation, its pressure flux and
//     wave speed identical); boundary edges are evaluated here, from the
//     untouched edge values.
// Each listed edge's results overwrite the LDS edge values only it reads.
//
// Bound by instruction issue: the SIMDs issue VALU work some 80% of the time, four
// waves each (105 VGPRs; 34 KB of LDS per workgroup allow four workgroups per
// CU). Against gathering every neighbour's state, centroid and vertices from
// memory in phases 1 and 2 (4M triangles): 826 -> 403 MB of HBM reads per
// launch, 960 -> 274 cache accesses and 1548 -> 1436 VALU instructions per
// wave, 251 -> 212 us (substep 0) and 280 -> 235 us (substep 1); with two
// divisions a limiter and the CFL radii requested early 201 and 227. A workgroup
// of five waves, the fifth for the halo in phase 1, took 410 us: its waves do
// not spread evenly over four SIMDs, so two workgroups fit a CU instead of
// four. 128 triangles per tile: 245 us.
template <int SUBSTEP, bool VG = false>
__global__ void __launch_bounds__(DE_BLOCK, 4)
de_xflux_e(DeMesh m, DeParams p, const DeQ *__restrict__ q, const double *__restrict__ eta,
           DeTileX tx, DeBoundary bc, unsigned char *__restrict__ flags, double *__restrict__ exw,
           double *__restrict__ exuh, double *__restrict__ exvh, const DeQ *bk, DeQ *out,
           DeControl *ctl,
           const DeControl *dctl, double *__restrict__ part_dt, double *__restrict__ part_bf,
           double *__restrict__ part_mass, unsigned long long *__restrict__ nneg)
{
    static_assert(DE_BLOCK >= 128, "the halo and the tile's edges share the workgroup's waves");
    // [6][2 DE_BLOCK] cells, then in their place [4 quantities][3 edges]
    // [DE_BLOCK] tile edge values; [4][hecap] halo edge values; [2][DE_BLOCK]
    // centroid depths and beds; VG: [ncap] nodes, [DE_BLOCK] node words
    extern __shared__ double2 lds16[];
    double *const lds = reinterpret_cast<double *>(lds16);
    __shared__ double red_dt[DE_BLOCK / 64], red_bf[DE_BLOCK / 64], red_m[DE_BLOCK / 64];
    const int lb = xcd_block();
    const int N = m.N, t = threadIdx.x;
    const int k0 = lb * DE_BLOCK, k = k0 + t;
    const int hecap = tx.hecap;
    double *const hl = lds + 12 * DE_BLOCK;
    double *const hz = hl + 4 * hecap;
    double2 *const nd = reinterpret_cast<double2 *>(hz + 2 * DE_BLOCK);
    unsigned *const vis = reinterpret_cast<unsigned *>(nd + tx.ncap);
    const int c0 = tx.cstart[lb], nc = tx.cstart[lb + 1] - c0;
    const int h0 = tx.hstart[lb], nhe = tx.hstart[lb + 1] - h0;
    const int e0 = tx.estart[lb], es = tx.esplit[lb], e1 = tx.estart[lb + 1];

    // every record that phases 0 to 3 need, requested before the control block
    // is read (bounded by the arrays' length, not yet by the scenario's end)
    const int kc = t < nc ? tx.cell[c0 + t] : 0;
    DeQ qk{0.0, 0.0, 0.0, 0.0};
    double2 ck = make_double2(0.0, 0.0);
    unsigned st = 0x3fffffffu, vi = 0;
    if (k < N) {
        qk = q[k];
        ck = m.cen[k];
        st = tx.stencil[k];
        if (VG) vi = tx.nodes[k];
    }
    double2 node = make_double2(0.0, 0.0);
    int n0 = 0, nn = 0;
    if (VG) {
        n0 = tx.nstart[lb];
        nn = tx.nstart[lb + 1] - n0;
        if (t < nn) node = tx.node[n0 + t];
    }
    // phase 2: hw waves take the halo (at most one edge to it per thread),
    // each thread of the others one edge inside the tile
    const int hw = (nhe + 63) >> 6;
    const int e2 = e0 + t - 64 * hw, e3 = min(es, e0 + DE_BLOCK - 64 * hw) + t;
    const bool has2 = t >= 64 * hw && e2 < es;
    const bool hal = t < nhe;
    const unsigned en2 = has2 ? tx.edge[e2] : 0u, en3 = e3 < e1 ? tx.edge[e3] : 0u;
    unsigned hst = 0, hc = 0, hvi = 0;
    if (hal) {
        hst = tx.hstencil[h0 + t];
        hc = tx.hcell[h0 + t];
        if (VG) hvi = tx.hnodes[h0 + t];
    }
    DeQ qc{0.0, 0.0, 0.0, 0.0};
    double2 cc = make_double2(0.0, 0.0);
    if (t < nc) {
        qc = q[kc];
        cc = m.cen[kc];
    }

    DeControl *cb = de_ctl(ctl, m.scen, lb);
    if (cb->done || (tx.crowded && tx.crowded[lb])) return;
    int *err = &cb->status;
    const double dt = SUBSTEP ? dctl[cb - ctl].dt : 0.0;
    const bool on = k < cb->kend;
    double mass = 0.0, dtmin = 1.0e100, bflux = 0.0;
    unsigned fk = 0;
    constexpr int Q = 3 * DE_BLOCK;   // stride between quantities of the tile

    // phase 0
    de_put_cell(lds, t, de_wet_cell(qk, p.mah), ck);
    hz[DE_BLOCK + t] = qk.z;
    if (VG) {
        vis[t] = vi;
        if (t < nn) nd[t] = node;
        for (int j = t + DE_BLOCK; j < nn; j += DE_BLOCK) nd[j] = tx.node[n0 + j];
    }
    if (t < nc) de_put_cell(lds, DE_BLOCK + t, de_wet_cell(qc, p.mah), cc);
    __syncthreads();

    // phase 1
    double ev[4][3];
    if (on) {
        DeStencil s;
        de_read_stencil<VG>(m, p, q, nullptr, k, st, t, lds, s);
        const bool clamp = de_clamped(qk.w, qk.z, p.mah);
        if (clamp) mass = (qk.z - qk.w) * m.area[k];
        fk = (clamp ? DE_F_CLAMP : 0u) | (s.keep ? DE_F_KEEP : 0u);
        flags[k] = (unsigned char)fk;
        hz[t] = s.own.h;
        DeExtrap<double> x;
        de_extrap_stencil<VG>(m, p, k, s, nd, vi, err, x);
#pragma unroll
        for (int i = 0; i < 3; i++) de_edge64(x, i, ev[0][i], ev[1][i], ev[2][i], ev[3][i]);
    }
    DeStencil hs{};
    int kh = 0;
    if (hal) {
        const int *kp = tx.cell + c0 + (int)(hc & 1023u) - DE_BLOCK;
        if (!VG) kh = *kp;
        de_read_stencil<VG>(m, p, q, kp, 0, hst, (int)(hc & 1023u), lds, hs);
    }
    __syncthreads();
    // every cell has been read: the edge values take their place
    if (on) {
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) lds[(3 * r + i) * DE_BLOCK + t] = ev[r][i];
    }
    __syncthreads();

    // phase 2: the halo's extrapolation, and edges inside the tile
    if (hal) {
        DeExtrap<double> x;
        de_extrap_stencil<VG>(m, p, kh, hs, nd, hvi, err, x);
        // a branch per edge: a run-time choice between the registers of x
        // would place x in scratch
        const int jb = (int)(hc >> 10) & 3;
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (i == jb) {
                double ew, eh, euh, evh;
                de_edge64(x, i, ew, eh, euh, evh);
                hl[t] = ew;
                hl[hecap + t] = eh;
                hl[2 * hecap + t] = euh;
                hl[3 * hecap + t] = evh;
            }
    } else if (has2) {
        de_tile_edge<SUBSTEP, VG>(m, p, en2, -1, k0, lds, hl, hz, hecap, nd, vis, dtmin);
    }
    __syncthreads();

    // phase 3: the tile's remaining edges, then the edges to the halo
    if (e3 < e1) {
        de_tile_edge<SUBSTEP, VG>(m, p, en3, e3 - es, k0, lds, hl, hz, hecap, nd, vis, dtmin);
        for (int e = e3 + DE_BLOCK; e < e1; e += DE_BLOCK)
            de_tile_edge<SUBSTEP, VG>(m, p, tx.edge[e], e - es, k0, lds, hl, hz, hecap, nd, vis,
                                      dtmin);
    }
    // phase 4's inputs, requested before the barrier (held from the kernel's
    // start they cost registers in every phase)
    DeQ q3{0.0, 0.0, 0.0, 0.0}, bk_k{0.0, 0.0, 0.0, 0.0};
    double eta_k = 0.0, area_k = 1.0;
    unsigned ac = 0;
    if (on) {
        ac = tx.across[k];
        area_k = m.area[k];
        if (SUBSTEP) {
            q3 = q[k];
            eta_k = eta[k];
            bk_k = bk[k];
        }
    }
    __syncthreads();

    // phase 4: each triangle's three edges in local order
    if (on) {
        double sw = 0.0, sx = 0.0, sy = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double *const A = lds + i * DE_BLOCK + t;
            const int f = de_field(st, i);
            if (f == 1023) {            // a boundary edge
                const DeCentroid c = de_centroid(SUBSTEP ? q3 : q[k], fk);
                const int4 vk = m.nb[k];
                const int vb = i == 0 ? vk.x : (i == 1 ? vk.y : vk.z);
                const double hc = de_height(c.w, c.z);
                de_edge_flux<double, SUBSTEP, false>(m, p, bc, q, flags, N, k, i, vb, c, hc,
                                                     c.z, A[0], A[Q], A[2 * Q], A[3 * Q], 0.0,
                                                     0.0, 0.0, 0.0, sw, sx, sy, bflux, dtmin);
                continue;
            }
            double a0, a1, a2, b1, b2;
            if (f > t) {                // evaluated from this side
                a0 = A[0];
                a1 = A[Q];
                a2 = A[2 * Q];
                b1 = A[3 * Q];
                b2 = f >= DE_BLOCK ? hl[(ac >> (6 + 8 * i)) & 255u]
                                   : lds[((ac >> (2 * i)) & 3u) * DE_BLOCK + f];
            } else {                    // evaluated from the neighbour's side
                const double *O = lds + ((ac >> (2 * i)) & 3u) * DE_BLOCK + f;
                a0 = -O[0];
                a1 = -O[Q];
                a2 = -O[2 * Q];
                b1 = -A[Q];
                b2 = -A[2 * Q];
            }
            sw += a0;
            sx += a1;
            sy += a2;
            sx -= b1;
            sy -= b2;
        }
        const double inv_area = 1.0 / area_k;
        sw *= inv_area;
        sx *= inv_area;
        sy *= inv_area;
        if (SUBSTEP == 0) {
            exw[k] = sw;
            exuh[k] = sx;
            exvh[k] = sy;
        } else {
            const DeQ r = de_advance(de_centroid(q3, fk), eta_k, sw, sx, sy, dt, p, err, nneg);
            out[k] = de_rk_combine<SUBSTEP>(r, bk_k);
        }
    }

    de_block_partials<SUBSTEP>(dtmin, bflux, mass, red_dt, red_bf, red_m, part_dt, part_bf,
                               part_mass, lb);
}

// One edge's terms of triangle k's sums on the mixed path (the body of the
// reference's edge loop, sw_domain_orig.c:828-1004, over FP32 differences):
// own edge record el (dw, dh, uh, vh) and centroid depth hcd; for an interior
// edge the neighbour's record er at the shared edge and its centroid depth
// hcn. Shared by de_flux_mixed and the tiled fused kernel.
template <int SUBSTEP>
__device__ __forceinline__ void de_edge_flux_mixed(const DeParams &p, const DeBoundary &bc,
                                                   const DeGeoF32 *__restrict__ gf,
                                                   const DeCentroid &c,
                                                   double hcd, float hc, int i, int vi,
                                                   float4 el, float4 er, double hcn, double &sw,
                                                   double &sx, double &sy, double &bflux,
                                                   double &dtmin)
{
    const float g = float(p.g), eps = float(p.eps);
    const float hle = float(hcd + double(el.y));
    const float zl = el.x - el.y;
    const float ql1 = el.z, ql2 = el.w;
    const float n1 = gf->nx[i], n2 = gf->ny[i];
    float hre, zr, qr1, qr2, dH = 0.f;
    if (vi >= 0) {
        hre = float(hcn + double(er.y));
        zr = gf->dzc[i] + (er.x - er.y);
        qr1 = er.z;
        qr2 = er.w;
        dH = (float(hcn - hcd) + (er.y - el.y)) + (zr - zl);
    } else {
        const int j = -vi - 1;
        const int kind = bc.kind[j];
        const double *bv = bc.val + (size_t)de_bc_slot<SUBSTEP>() * bc.sstride;
        float wr;                                   // stage above z_c
        if (kind == 0) {          // reflective
            const float r1 = -ql1 * n1 - ql2 * n2;
            const float r2 = -ql1 * n2 + ql2 * n1;
            wr = zl + hle;
            qr1 = n1 * r1 - n2 * r2;
            qr2 = n2 * r1 + n1 * r2;
        } else if (kind == 1) {   // transmissive
            wr = zl + hle;
            qr1 = ql1;
            qr2 = ql2;
        } else if (kind == 2) {   // Dirichlet
            wr = float(bv[j] - c.z);
            qr1 = float(bv[bc.M + j]);
            qr2 = float(bv[2 * bc.M + j]);
        } else if (kind == 3) {   // transmissive from centroid values
            wr = float(c.w - c.z);
            qr1 = float(c.uh);
            qr2 = float(c.vh);
        } else if (kind == 4) {   // stage set, normal momentum kept, tangential 0
            const float nq = n1 * ql1 + n2 * ql2;
            wr = float(bv[j] - c.z);
            qr1 = nq * n1;
            qr2 = nq * n2;
        } else if (kind == 5) {   // transmissive stage, zero momentum
            wr = zl + hle;
            qr1 = 0.f;
            qr2 = 0.f;
        } else {                  // stage set, momentum transmissive
            wr = float(bv[j] - c.z);
            qr1 = ql1;
            qr2 = ql2;
        }
        zr = zl;
        hre = (kind <= 1 || kind == 5) ? fmax(hle, 0.f) : fmax(wr - zr, 0.f);
    }
    const float z_half = fmax(zl, zr);
    const float hl_raw = hle + (zl - z_half);
    const float hr_raw = hre + (zr - z_half);
    const float h_left = fmax(hl_raw, 0.f);
    const float h_right = fmax(hr_raw, 0.f);
    const float diff0 = (vi >= 0 && hl_raw > 0.f && hr_raw > 0.f) ? dH : h_right - h_left;
    float ef[3], speed, pflux;
    de_flux_central_d<float>(ql1, ql2, qr1, qr2, h_left, h_right, hle, hre, n1, n2, eps,
                             diff0, g, ef, speed, pflux);
    const float length = gf->len[i];
    const float dsq = (hl_raw > 0.f) ? (zl - z_half) * (h_left + hle) : -(hle * hle);
    const float pg = length * (-g * 0.5f * (dsq - (hle + hc) * zl) + pflux);
    sw -= double(ef[0] * length);
    sx -= double(ef[1] * length);
    sy -= double(ef[2] * length);
    if (vi < 0) bflux -= double(ef[0] * length);
    sx -= double(n1 * pg);
    sy -= double(n2 * pg);
    if (SUBSTEP == 0 && double(speed) > p.eps)
        dtmin = fmin(dtmin, double(gf->radius) * (1.0 / double(speed)));
}

// Mixed-precision flux. All FP32 arithmetic is on quantities referred to the
// own centroid bed z_c (a local datum): edge bed zl = dw - dh, neighbour edge
// bed zr = (z_n - z_c) + dw' - dh', depths h = h_c + dh formed in FP64 and
// rounded, and the two terms that are differences of depths,
//   fmax(wr, z_half) - fmax(wl, z_half) = h_right - h_left
//   h_left^2 - hle^2 = (zl - z_half)(h_left + hle)   (h_left > 0),
// evaluated from small differences. Equal to the reference's formulas in real
// arithmetic (sw_domain_orig.c:879-1004); sums, CFL and update stay FP64.
template <int SUBSTEP>
__global__ void __launch_bounds__(DE_BLOCK)
de_flux_mixed(DeMesh m, DeParams p, const DeQ *q, const double *__restrict__ eta,
              const DeEdgeRec32 *__restrict__ E, DeBoundary bc,
              const unsigned char *__restrict__ flags, double *__restrict__ exw,
              double *__restrict__ exuh, double *__restrict__ exvh, const DeQ *bk, DeQ *out,
              DeControl *ctl,
              const DeControl *dctl, double *__restrict__ part_dt, double *__restrict__ part_bf,
              unsigned long long *__restrict__ nneg)
{
    __shared__ double red_dt[DE_BLOCK / 64];
    __shared__ double red_bf[DE_BLOCK / 64];
    const int lb = xcd_block();
    DeControl *cb = de_ctl(ctl, m.scen, lb);
    if (cb->done) return;
    int *err = &cb->status;
    const double dt = SUBSTEP ? dctl[cb - ctl].dt : 0.0;
    const int N = m.N;
    const int k = lb * DE_BLOCK + threadIdx.x;
    double dtmin = 1.0e100, bflux = 0.0;

    if (k < cb->kend) {
        const DeCentroid c = de_centroid(q[k], flags[k]);
        const int4 vk = m.nb[k];
        const int v[3] = {vk.x, vk.y, vk.z};
        const DeGeoF32 *gf = static_cast<const DeGeoF32 *>(m.gf) + k;
        const DeEdgeRec32 own = E[k];
        const double hcd = own.hc;
        const float hc = float(hcd);
        double sw = 0.0, sx = 0.0, sy = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            float4 er = make_float4(0.f, 0.f, 0.f, 0.f);
            double hcn = 0.0;
            if (v[i] >= 0) {
                const DeEdgeRec32 *rn = E + (v[i] >> 2);
                er = rn->e[v[i] & 3];
                hcn = rn->hc;
            }
            de_edge_flux_mixed<SUBSTEP>(p, bc, gf, c, hcd, hc, i, v[i], own.e[i], er, hcn, sw, sx,
                                        sy, bflux, dtmin);
        }
        const double inv_area = 1.0 / m.area[k];
        sw *= inv_area;
        sx *= inv_area;
        sy *= inv_area;
        if (SUBSTEP == 0) {
            exw[k] = sw;
            exuh[k] = sx;
            exvh[k] = sy;
        } else {
            const DeQ r = de_advance(c, eta[k], sw, sx, sy, dt, p, err, nneg);
            out[k] = de_rk_combine<SUBSTEP>(r, bk[k]);
        }
    }

    dtmin = de_wave_min(dtmin);
    bflux = de_wave_sum(bflux);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        red_dt[wv] = dtmin;
        red_bf[wv] = bflux;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a2 = red_dt[0], b2 = red_bf[0];
        for (int i = 1; i < DE_BLOCK / 64; i++) {
            a2 = fmin(a2, red_dt[i]);
            b2 += red_bf[i];
        }
        part_dt[lb] = a2;
        part_bf[lb] = b2;
    }
}

// Tiled fused extrapolation + flux on the mixed path (any SUBSTEP): as
// de_xflux, with the FP32 edge records of de_extrapolate<float> and the FP64
// centroid depths in LDS, and the edge terms of de_flux_mixed, so the
// results are the bits of the separate mixed kernels. DE_MIXED_WAVES: the
// waves per SIMD the register allocation aims at (the autotuner's choice;
// 5, with 96 VGPRs and a 12 B spill, ran 4% faster than 4 with 100 VGPRs).
#ifndef DE_MIXED_WAVES
#define DE_MIXED_WAVES 5
#endif
template <int SUBSTEP>
__global__ void __launch_bounds__(DE_BLOCK, DE_MIXED_WAVES)
de_xflux_mixed(DeMesh m, DeParams p, const DeQ *__restrict__ q, const double *__restrict__ eta,
               DeTiles tl, DeBoundary bc, unsigned char *__restrict__ flags,
               double *__restrict__ exw, double *__restrict__ exuh, double *__restrict__ exvh,
               const DeQ *bk, DeQ *out, DeControl *ctl,
               const DeControl *dctl, double *__restrict__ part_dt,
               double *__restrict__ part_bf, double *__restrict__ part_mass,
               unsigned long long *__restrict__ nneg)
{
    // centroid depths [DE_BLOCK] tile then [hcap] halo (double); then the
    // records' components [4][3][DE_BLOCK] tile and [4][3][hcap] halo (float)
    extern __shared__ double lds[];
    __shared__ double red_dt[DE_BLOCK / 64], red_bf[DE_BLOCK / 64], red_m[DE_BLOCK / 64];
    const int lb = xcd_block();
    const int t = threadIdx.x;
    const int k0 = lb * DE_BLOCK, k = k0 + t;
    // the extrapolation's own records, requested before the control block is
    // read (bounded by the arrays' length, not yet by the scenario's end)
    int4 vk1 = make_int4(-1, -1, -1, 3);
    DeQ qk1{0.0, 0.0, 0.0, 0.0};
    if (k < m.N) {
        vk1 = m.nb[k];
        qk1 = q[k];
    }
    DeControl *cb = de_ctl(ctl, m.scen, lb);
    if (cb->done) return;
    int *err = &cb->status;
    const double dt = SUBSTEP ? dctl[cb - ctl].dt : 0.0;
    const int kend = cb->kend;
    const int hcap = tl.hcap;
    double *const hct = lds, *const hch = lds + DE_BLOCK;
    float *const ft = reinterpret_cast<float *>(lds + DE_BLOCK + hcap);
    float *const fh = ft + 12 * DE_BLOCK;
    double mass = 0.0, dtmin = 1.0e100, bflux = 0.0;
    unsigned fk = 0;
    // a halo thread's first halo triangle, loaded now so that its latency
    // hides behind the tile's extrapolation
    const int h0 = tl.start[lb], nh = tl.start[lb + 1] - h0;
    const int kh0 = t < nh ? tl.halo[h0 + t] : 0;

    if (k < kend) {
        DeExtrap<float> x;
        de_extrap_cell<float>(m, p, q, k, vk1, qk1, err, x);
        mass = x.mass;
        fk = x.flag;
        flags[k] = (unsigned char)fk;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const float4 r = de_edge32(x, i);
            ft[(0 + i) * DE_BLOCK + t] = r.x;
            ft[(3 + i) * DE_BLOCK + t] = r.y;
            ft[(6 + i) * DE_BLOCK + t] = r.z;
            ft[(9 + i) * DE_BLOCK + t] = r.w;
        }
        hct[t] = x.c.h;
    }
    for (int j = t; j < nh; j += DE_BLOCK) {
        DeExtrap<float> x;
        de_extrap_cell<float>(m, p, q, j == t ? kh0 : tl.halo[h0 + j], err, x);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const float4 r = de_edge32(x, i);
            fh[(0 + i) * hcap + j] = r.x;
            fh[(3 + i) * hcap + j] = r.y;
            fh[(6 + i) * hcap + j] = r.z;
            fh[(9 + i) * hcap + j] = r.w;
        }
        hch[j] = x.c.h;
    }
    // the flux's own records, requested before the barrier; the whole
    // geometry record is held in registers (the edge loop runs faster with
    // it there than through a pointer)
    DeQ qk2{0.0, 0.0, 0.0, 0.0};
    int4 vk2 = make_int4(-1, -1, -1, 3);
    unsigned sl2 = 0;
    DeGeoF32 gfr{};
    if (k < kend) {
        qk2 = q[k];
        vk2 = m.nb[k];
        sl2 = tl.slot[k];
        gfr = static_cast<const DeGeoF32 *>(m.gf)[k];
    }
    __syncthreads();

    if (k < kend) {
        const DeCentroid c = de_centroid(qk2, fk);
        const int4 vk = vk2;
        const int v[3] = {vk.x, vk.y, vk.z};
        const unsigned sl = sl2;
        const DeGeoF32 *gf = &gfr;
        const double hcd = hct[t];
        const float hc = float(hcd);
        double sw = 0.0, sx = 0.0, sy = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const float4 el = make_float4(ft[(0 + i) * DE_BLOCK + t], ft[(3 + i) * DE_BLOCK + t],
                                          ft[(6 + i) * DE_BLOCK + t], ft[(9 + i) * DE_BLOCK + t]);
            float4 er = make_float4(0.f, 0.f, 0.f, 0.f);
            double hcn = 0.0;
            if (v[i] >= 0) {
                const unsigned s = (sl >> (10 * i)) & 1023u;
                const float *src;
                int stride;
                if (s == 1023u) {
                    const int tn = (v[i] >> 2) - k0;
                    src = ft + (v[i] & 3) * DE_BLOCK + tn;
                    stride = 3 * DE_BLOCK;
                    hcn = hct[tn];
                } else {
                    src = fh + (v[i] & 3) * hcap + s;
                    stride = 3 * hcap;
                    hcn = hch[s];
                }
                er = make_float4(src[0], src[stride], src[2 * stride], src[3 * stride]);
            }
            de_edge_flux_mixed<SUBSTEP>(p, bc, gf, c, hcd, hc, i, v[i], el, er, hcn, sw, sx, sy,
                                        bflux, dtmin);
        }
        const double inv_area = 1.0 / m.area[k];
        sw *= inv_area;
        sx *= inv_area;
        sy *= inv_area;
        if (SUBSTEP == 0) {
            exw[k] = sw;
            exuh[k] = sx;
            exvh[k] = sy;
        } else {
            const DeQ r = de_advance(c, eta[k], sw, sx, sy, dt, p, err, nneg);
            out[k] = de_rk_combine<SUBSTEP>(r, bk[k]);
        }
    }

    de_block_partials<SUBSTEP>(dtmin, bflux, mass, red_dt, red_bf, red_m, part_dt, part_bf,
                               part_mass, lb);
}

// Fixed-order reduction of the per-block partials part[row][nblocks], row
// DE_P_*, into the control blocks. Each scenario's blocks split into
// DE_RCHUNKS contiguous chunks; a chunk's partials are added in a fixed order,
// then the chunk results. The order depends only on the scenario's block
// count. Up to DE_DIRECT_BLOCKS blocks (a chunk of at most 64, one per lane)
// one workgroup per scenario reduces them in a single launch (4.6 us, at any
// such size); above, de_reduce_chunks gives each chunk its own workgroup so
// that many CUs read the partials, and a second stage adds the chunk results.
// Both give the same bits.
#define DE_DIRECT_BLOCKS (64 * DE_RCHUNKS)

// what a reduction leaves in the control block
enum { DE_R_FLUX0 = 0, DE_R_FLUX1, DE_R_MASS, DE_R_VOLUME, DE_R_FLUX2 };

#define DE_RED_THREADS 512
// The sums of NR rows of one scenario's partials, by one workgroup of TH
// threads (every thread gets them): the chunk results are read (CHUNKS) or
// formed here, a wave per chunk and a lane per block.
template <bool CHUNKS, int NR, int TH = DE_RED_THREADS>
__device__ __forceinline__ void de_reduce_rows(const double *__restrict__ src, int nblocks,
                                               const DeControl *cb, int sc, int S,
                                               const int rows[3], double (*res)[DE_RCHUNKS],
                                               double sum[3])
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (!CHUNKS) {
        const int b0 = cb->bbeg, b1 = cb->bend;
        const int len = (b1 - b0 + DE_RCHUNKS - 1) / DE_RCHUNKS;
        constexpr int W = TH / 64, PER = de_wave_passes(W, DE_RCHUNKS);
        double x[PER][3];
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int c = de_wave_chunk(wv, j, W, DE_RCHUNKS);
            const int i = b0 + c * len + lane;
            const bool in = c >= 0 && lane < len && i < b1;
#pragma unroll
            for (int r = 0; r < NR; r++)
                x[j][r] = in ? src[(size_t)rows[r] * nblocks + i] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int c = de_wave_chunk(wv, j, W, DE_RCHUNKS);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const double v = de_wave_sum_nz(x[j][r]);
                if (lane == 0 && c >= 0) res[r][c] = v;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
        double v = 0.0;
        if (lane < DE_RCHUNKS)
            v = CHUNKS ? src[((size_t)rows[r] * S + sc) * DE_RCHUNKS + lane] : res[r][lane];
        sum[r] = __shfl(de_wave_sum_nz(v), 0, 64);
    }
}

// boundary_flux_integral_operator.__call__ (boundary_flux_integral_operator.py:46-62)
__device__ __forceinline__ double de_flux_integral(double integral, double dt, int method,
                                                   double s0, double s1, double s2)
{
    if (method == 1) return integral + dt * s0;
    if (method == 2) return integral + 0.5 * dt * (s0 + s1);
    return integral + 1.0 / 6.0 * dt * (s0 + s1 + 4.0 * s2);
}

// Generic_Domain.update_timestep (generic_domain.py:2349-2415): the timestep
// before the clamps, min(CFL * flux_dt, max_dt), and the step's timestep,
// clamped to the final time and the next yield time. Reads nothing that
// de_commit_timestep writes.
__device__ __forceinline__ double de_cfl_timestep(const DeControl *c, double flux_dt)
{
    const double a = c->cfl * (c->fixed_flux_dt > 0.0 ? c->fixed_flux_dt : flux_dt);
    return (c->max_dt < a) ? c->max_dt : a;
}

__device__ __forceinline__ double de_clamped_timestep(const DeControl *c, double ts)
{
    if (c->t + ts > c->finaltime) ts = c->finaltime - c->t;
    if (c->t + ts > c->yieldtime) ts = c->yieldtime - c->t;
    return ts;
}

// the rest of update_timestep, by one thread of a scenario: the recorded
// extremes, the small-step counter with its first-order switch and its
// exception (returned as DE_ERR_SMALL_TIMESTEP), and the results
__device__ __forceinline__ int de_commit_timestep(DeControl *c, double flux_dt, double ts,
                                                  double dt)
{
    int err = 0;
    c->rec_max = (c->rec_max > ts) ? c->rec_max : ts;      // max(timestep, recorded_max)
    c->rec_min = (c->rec_min < ts) ? c->rec_min : ts;      // min(timestep, recorded_min)
    if (ts < c->min_dt) {
        c->smallsteps += 1;
        if (c->smallsteps > c->max_smallsteps) {
            c->smallsteps = 0;
            if (c->order == 1) err = DE_ERR_SMALL_TIMESTEP;
            else c->order = 1;
        }
    } else {
        c->smallsteps = 0;
        if (c->order == 1 && c->default_order == 2) c->order = 2;
    }
    c->flux_dt = flux_dt;
    c->dt = dt;
    return err;
}

// what the control workgroups of de_update read and write (DE_DT_STEP); of
// the host-sequenced steps the method alone
struct DeStepEnd {
    DeControl *next;
    const double *part;
    double *hist;
    int nblocks, method;
};

// The end of a step at time t + dt: timestep history (one scenario only) and
// the yield / final-time test of _evolve_base (generic_domain.py:1855-1895)
// that turns the scenario's next steps into no-ops; returns DE_ERR_OVERSHOOT
// or 0.
__device__ __forceinline__ int de_end_step(DeControl *c, double t, double dt, double *hist)
{
    c->t = t + dt;
    if (hist && c->nsteps < c->hist_cap) hist[c->nsteps] = dt;
    c->nsteps += 1;
    if (c->t >= c->finaltime - c->eps) {
        c->done = 1;
        return c->t > c->finaltime ? DE_ERR_OVERSHOOT : 0;
    }
    if (c->t >= c->yieldtime) c->done = 2;
    return 0;
}

// The minimum of a scenario's CFL partials, formed by every thread of a
// workgroup of DE_BLOCK threads.
__device__ __forceinline__ double de_block_dt(const double *__restrict__ pdt, int b0, int b1,
                                              double *red)
{
    double m = 1.0e100;
    for (int i = b0 + (int)threadIdx.x; i < b1; i += DE_BLOCK) m = fmin(m, pdt[i]);
    m = de_wave_min(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = red[0];
    for (int i = 1; i < DE_BLOCK / 64; i++) m = fmin(m, red[i]);
    return m;
}

// A scenario's control workgroup in a self-contained step (DE_DT_STEP): the
// next control block from this step's, the timestep and the boundary fluxes
// that are known: of rk2 and rk3 the step's later ones are added one step
// late, from the partials they left (pending), or by de_flush_step. The status
// bits stay where the kernels set them.
__device__ __forceinline__ void de_step_control(const DeControl *__restrict__ c, DeControl *next,
                                                const double *__restrict__ part, int nblocks,
                                                int method, double *hist, double *red,
                                                double (*res)[DE_RCHUNKS])
{
    const bool live = !c->done;
    double m = 0.0, sum[3] = {0.0, 0.0, 0.0};
    if (live) {
        m = de_block_dt(part + (size_t)DE_P_DT * nblocks, c->bbeg, c->bend, red);
        const int rows[3] = {DE_P_BF0, DE_P_BF1, DE_P_BF2};
        de_reduce_rows<false, 3, DE_BLOCK>(part, nblocks, c, 0, 1, rows, res, sum);
    }
    if (threadIdx.x) return;
    DeControl n = *c;
    n.status = next->status;
    if (live) {
        if (n.pending) {
            n.bflux1 = sum[1];
            n.bflux2 = sum[2];
            n.integral = de_flux_integral(n.integral, n.dt, method, n.bflux0, n.bflux1, n.bflux2);
        }
        const double ts = de_cfl_timestep(&n, m), dt = de_clamped_timestep(&n, ts);
        n.status |= de_commit_timestep(&n, m, ts, dt);
        n.bflux0 = sum[0];
        n.pending = method > 1;
        if (method == 1) n.integral = de_flux_integral(n.integral, dt, 1, n.bflux0, 0.0, 0.0);
        n.status |= de_end_step(&n, n.t, dt, hist);
    }
    *next = n;
}

// After the last self-contained step of a run: the boundary fluxes still
// pending, and after an odd number of steps the control blocks of ctl2 back
// into ctl, with the status bits of both.
template <int METHOD>
__global__ void __launch_bounds__(DE_RED_THREADS)
de_flush_step(const double *__restrict__ part, int nblocks, DeControl *ctl, DeControl *ctl2,
              int odd)
{
    __shared__ double res[3][DE_RCHUNKS];
    const int sc = blockIdx.x, S = gridDim.x;
    DeControl *c = ctl + sc;
    const int status = c->status | ctl2[sc].status;
    const int pending = odd ? ctl2[sc].pending : c->pending;
    double sum[3] = {0.0, 0.0, 0.0};
    const int rows[3] = {DE_P_BF0, DE_P_BF1, DE_P_BF2};
    if (METHOD > 1 && pending)
        de_reduce_rows<false, METHOD>(part, nblocks, c, sc, S, rows, res, sum);
    if (threadIdx.x) return;
    if (odd) *c = ctl2[sc];
    c->status = status;
    ctl2[sc].status = 0;
    if (METHOD > 1 && pending) {
        c->bflux1 = sum[1];
        if (METHOD > 2) c->bflux2 = sum[2];
        c->integral = de_flux_integral(c->integral, c->dt, METHOD, c->bflux0, c->bflux1,
                                       c->bflux2);
        c->pending = 0;
    }
}

// where de_update takes the timestep from: the control block, the host (which
// it then records, and for euler advances the boundary flux integral), or update_timestep
// over the minimum of the scenario's per-block CFL partials, read directly (at
// most DE_DIRECT_BLOCKS of them) or as the chunk results of de_reduce_chunks.
// DE_DT_STEP: directly, with the step's whole control in workgroups of its own.
enum { DE_DT_GIVEN = 0, DE_DT_HOST, DE_DT_DIRECT, DE_DT_CHUNKS, DE_DT_STEP };

// friction + update + fix_negative_cells from the explicit updates of substep 0;
// `out` may alias `q` (Euler, in place: each thread reads then writes its own record).
// With DT, every workgroup forms the step's timestep for itself from pdt, the
// CFL partials or chunk results, and the scenario's first one records it: the
// reduction and update_timestep cost no launches of their own. The control
// fields that the others read are not the ones it writes. Each launch in the
// graph of a step takes about 4.6 us however small: with the end of the step
// reduced in de_finish_step, a DE0 step has 3 launches instead of 6 and a DE1
// step 4 instead of 9 (6 above DE_DIRECT_BLOCKS); 120 DE1 steps of 90k
// triangles with two reads went from 16.5 to 10.5 ms, a 40k DE0 run of 205
// steps from 13.7 to 10.3 ms. The minimum's loads and barrier hide behind the
// triangle's own records, requested first: 66.5 us at 4M triangles, 67.0
// without it.
//
// DE_DT_STEP: S more workgroups, behind the others, write each scenario's next
// control block (de_step_control) while these advance their triangles, so that
// a step needs no launch for its end: 18.2 -> 16.7 us a DE0 step of 40k
// triangles, 39.5 -> 36.8 a DE1 step of 90k.
template <bool SLOPED, int DT>
__global__ void __launch_bounds__(DE_BLOCK)
de_update(const int *__restrict__ scen, DeParams p, const DeQ *q, const double *__restrict__ eta,
          const unsigned char *__restrict__ flags, const double *__restrict__ exw,
          const double *__restrict__ exuh, const double *__restrict__ exvh, DeControl *ctl,
          DeQ *out, unsigned long long *__restrict__ nneg, const double *__restrict__ pdt,
          double host_dt, DeStepEnd se, const double *__restrict__ E = nullptr, int N = 0,
          const double *__restrict__ vx = nullptr)
{
    __shared__ double red[DE_BLOCK / 64];
    const int lb = xcd_block();
    if constexpr (DT == DE_DT_STEP) {
        __shared__ double res[3][DE_RCHUNKS];
        if (lb >= se.nblocks) {
            const int s = lb - se.nblocks;
            de_step_control(ctl + s, se.next + s, se.part, se.nblocks, se.method, se.hist, red,
                            res);
            return;
        }
    }
    const int sc = scen ? scen[lb] : 0;
    DeControl *cb = ctl + sc;
    if (cb->done) return;
    const int k = lb * DE_BLOCK + threadIdx.x;
    const bool on = k < cb->kend;
    DeQ qk{0.0, 0.0, 0.0, 0.0};
    unsigned f = 0;
    double n = 0.0, e0 = 0.0, e1 = 0.0, e2 = 0.0;
    if (on) {
        qk = q[k];
        f = flags[k];
        n = eta[k];
        e0 = exw[k];
        e1 = exuh[k];
        e2 = exvh[k];
    }
    double dt;
    if constexpr (DT == DE_DT_GIVEN) {
        dt = cb->dt;
    } else if constexpr (DT == DE_DT_HOST) {
        dt = host_dt;
        if (lb == cb->bbeg && threadIdx.x == 0) {
            cb->dt = dt;
            if (se.method == 1)
                cb->integral = de_flux_integral(cb->integral, dt, 1, cb->bflux0, 0.0, 0.0);
        }
    } else {
        const double m = DT == DE_DT_CHUNKS ? de_block_dt(pdt, sc * DE_RCHUNKS,
                                                          (sc + 1) * DE_RCHUNKS, red)
                                            : de_block_dt(pdt, cb->bbeg, cb->bend, red);
        const double ts = de_cfl_timestep(cb, m);
        dt = de_clamped_timestep(cb, ts);
        if (DT != DE_DT_STEP && lb == cb->bbeg && threadIdx.x == 0) {
            const int e = de_commit_timestep(cb, m, ts, dt);
            if (e) atomicOr(&cb->status, e);
        }
    }
    if (!on) return;
    DeSlope sl{false, 0.0, 0.0};
    if constexpr (SLOPED) sl = de_sloped_bed(E, N, k, vx);
    out[k] = de_advance(de_centroid(qk, f), n, e0, e1, e2, dt, p, &cb->status, nneg, sl);
}

// ---------------------------------------------------------------------------
// per-operation kernels: one kernel per call the reference's Domain makes in
// evolve_one_{euler,rk2,rk3}_step (generic_domain.py:1914-2179), over the
// centroid state q as distribute_to_vertices_and_edges left it. One
// scenario, triangles [0, kend).
// ---------------------------------------------------------------------------
// backup_centroid_values of stage, xmomentum, ymomentum (quantity.c:735-749)
__global__ void __launch_bounds__(DE_BLOCK)
de_backup(int kend, const DeQ *__restrict__ q, DeQ *__restrict__ bk)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k < kend) bk[k] = q[k];
}

// saxpy_centroid_values (quantity.c:752-769): q = a q + b backup
__global__ void __launch_bounds__(DE_BLOCK)
de_saxpy(int kend, double a, double b, DeQ *__restrict__ q, const DeQ *__restrict__ bk)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= kend) return;
    DeQ r = q[k];
    const DeQ s = bk[k];
    r.w = a * r.w + b * s.w;
    r.uh = a * r.uh + b * s.uh;
    r.vh = a * r.vh + b * s.vh;
    q[k] = r;
}

// rk3's closing division of the conserved centroids (generic_domain.py:2167-2170)
__global__ void __launch_bounds__(DE_BLOCK)
de_divide(int kend, double divisor, DeQ *__restrict__ q)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= kend) return;
    DeQ r = q[k];
    r.w = r.w / divisor;
    r.uh = r.uh / divisor;
    r.vh = r.vh / divisor;
    q[k] = r;
}

// compute_forcing_terms: Manning friction added to the momenta's
// semi-implicit updates (manning_friction_implicit, friction.py:22-76). The
// sloped form reads the vertex beds of the last extrapolation (E).
template <bool SLOPED>
__global__ void __launch_bounds__(DE_BLOCK)
de_friction(int kend, DeParams p, const DeQ *__restrict__ q, const double *__restrict__ eta,
            double *__restrict__ si_uh, double *__restrict__ si_vh,
            const double *__restrict__ E = nullptr, int N = 0,
            const double *__restrict__ vx = nullptr)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= kend) return;
    const DeQ r = q[k];
    const DeCentroid c{r.w, r.uh, r.vh, r.z};
    DeSlope sl{false, 0.0, 0.0};
    if constexpr (SLOPED) sl = de_sloped_bed(E, N, k, vx);
    double S;
    if (de_manning_S(c, eta[k], p, sl, S)) {
        si_uh[k] += S * c.uh;
        si_vh[k] += S * c.vh;
    }
}

// Quantity.update of stage, xmomentum and ymomentum (quantity.c:772-822): the
// explicit and semi-implicit updates with timestep dt; the semi-implicit
// updates are reset. Stage has no semi-implicit term.
__global__ void __launch_bounds__(DE_BLOCK)
de_update_centroids(int kend, DeControl *ctl, DeQ *__restrict__ q,
                    const double *__restrict__ exw, const double *__restrict__ exuh,
                    const double *__restrict__ exvh, double *__restrict__ si_uh,
                    double *__restrict__ si_vh)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= kend) return;
    const double dt = ctl->dt;
    int *err = &ctl->status;
    DeQ r = q[k];
    r.w = de_update_one(r.w, exw[k], 0.0, dt, err);
    r.uh = de_update_one(r.uh, exuh[k], si_uh[k], dt, err);
    r.vh = de_update_one(r.vh, exvh[k], si_vh[k], dt, err);
    q[k] = r;
    si_uh[k] = 0.0;
    si_vh[k] = 0.0;
}

// _orig_fix_negative_cells (sw_domain_orig.c:2890-2910); every triangle is full
__global__ void __launch_bounds__(DE_BLOCK)
de_fix_negative(int kend, DeQ *__restrict__ q, unsigned long long *__restrict__ nneg)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= kend) return;
    DeQ r = q[k];
    if (r.w - r.z < 0.0) {
        atomicAdd(nneg, 1ull);
        r.w = r.z;
        r.uh = 0.0;
        r.vh = 0.0;
        q[k] = r;
    }
}

// One workgroup per chunk (blockIdx.x) and scenario (blockIdx.y): the CFL
// minimum if DT, and the sums of NR rows, each to chunks[row][scenario][chunk].
// live: nothing for scenarios that are done.
template <bool DT, int NR>
__global__ void __launch_bounds__(256)
de_reduce_chunks(const double *__restrict__ part, int nblocks, int r0, int r1, int r2, int live,
                 const DeControl *__restrict__ ctl, double *__restrict__ chunks)
{
    __shared__ double red[4][4];
    const int sc = blockIdx.y, c = blockIdx.x, S = gridDim.y;
    const DeControl *cb = ctl + sc;
    if (live && cb->done) return;
    const int rows[3] = {r0, r1, r2};
    double a = 1.0e100, b[3] = {0.0, 0.0, 0.0};
    const int b0 = cb->bbeg, b1 = cb->bend;
    const int len = (b1 - b0 + DE_RCHUNKS - 1) / DE_RCHUNKS;
    const int c0 = b0 + c * len, c1 = min(b1, c0 + len);
    for (int i = c0 + (int)threadIdx.x; i < c1; i += 256) {
        if (DT) a = fmin(a, part[(size_t)DE_P_DT * nblocks + i]);
#pragma unroll
        for (int r = 0; r < NR; r++) b[r] += part[(size_t)rows[r] * nblocks + i];
    }
    if (DT) a = de_wave_min(a);
#pragma unroll
    for (int r = 0; r < NR; r++) b[r] = de_wave_sum(b[r]);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        red[3][wv] = a;
#pragma unroll
        for (int r = 0; r < NR; r++) red[r][wv] = b[r];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const size_t o = (size_t)sc * DE_RCHUNKS + c, n = (size_t)S * DE_RCHUNKS;
        if (DT) {
            for (int k = 1; k < 4; k++) red[3][0] = fmin(red[3][0], red[3][k]);
            chunks[DE_P_DT * n + o] = red[3][0];
        }
#pragma unroll
        for (int r = 0; r < NR; r++) {
            for (int k = 1; k < 4; k++) red[r][0] += red[r][k];
            chunks[rows[r] * n + o] = red[r][0];
        }
    }
}

// A reduction to the control block outside device-controlled steps: MODE
// DE_R_*, of the row (and for DE_R_FLUX0 the CFL timesteps and protect's
// mass). src: the partials, or the chunk results (CHUNKS). integrate: the
// method whose step it completes, or 0.
template <int MODE, bool CHUNKS>
__global__ void __launch_bounds__(DE_RED_THREADS)
de_reduce(const double *__restrict__ src, int nblocks, int row, int integrate, DeControl *ctl)
{
    __shared__ double res[3][DE_RCHUNKS], red[DE_RED_THREADS / 64];
    const int sc = blockIdx.x, S = gridDim.x, t = threadIdx.x;
    DeControl *cb = ctl + sc;
    const bool live = MODE == DE_R_FLUX0 || MODE == DE_R_FLUX1 || MODE == DE_R_FLUX2;
    if (live && cb->done) return;
    double sum[3];
    const int rows[3] = {row, DE_P_MASS, 0};
    de_reduce_rows<CHUNKS, MODE == DE_R_FLUX0 ? 2 : 1>(src, nblocks, cb, sc, S, rows, res, sum);
    if (MODE == DE_R_FLUX0) {
        double a = 1.0e100;
        if (CHUNKS) {
            if (t < DE_RCHUNKS) a = src[((size_t)DE_P_DT * S + sc) * DE_RCHUNKS + t];
        } else {
            for (int i = cb->bbeg + t; i < cb->bend; i += DE_RED_THREADS)
                a = fmin(a, src[(size_t)DE_P_DT * nblocks + i]);
        }
        a = de_wave_min(a);
        if ((t & 63) == 0) red[t >> 6] = a;
        __syncthreads();
        if (t == 0) {
            for (int i = 1; i < DE_RED_THREADS / 64; i++) red[0] = fmin(red[0], red[i]);
            cb->flux_dt = red[0];
            cb->bflux0 = sum[0];
            cb->mass = sum[1];
        }
        return;
    }
    if (t == 0) {
        if (MODE == DE_R_FLUX1) cb->bflux1 = sum[0];
        else if (MODE == DE_R_MASS) cb->mass = sum[0];
        else if (MODE == DE_R_VOLUME) cb->volume = sum[0];
        else cb->bflux2 = sum[0];
        if (integrate)
            cb->integral = de_flux_integral(cb->integral, cb->dt, integrate, cb->bflux0,
                                            cb->bflux1, cb->bflux2);
    }
}

// one thread per scenario for the control kernels below
__device__ __forceinline__ DeControl *de_scenario(DeControl *ctl, int S)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    return s < S ? ctl + s : nullptr;
}

// End of a step that is not self-contained (operators, gauges, more than
// DE_DIRECT_BLOCKS blocks), one workgroup per scenario: the boundary flux sums
// of the METHOD's substeps and their integral (boundary_flux_integral_operator
// .py:39-49), and de_end_step.
template <int METHOD, bool CHUNKS>
__global__ void __launch_bounds__(DE_RED_THREADS)
de_finish_step(const double *__restrict__ src, int nblocks, DeControl *ctl, double *hist)
{
    __shared__ double res[3][DE_RCHUNKS];
    const int sc = blockIdx.x, S = gridDim.x;
    DeControl *c = ctl + sc;
    if (c->done) return;
    double sum[3] = {0.0, 0.0, 0.0};
    const int rows[3] = {DE_P_BF0, DE_P_BF1, DE_P_BF2};
    de_reduce_rows<CHUNKS, METHOD>(src, nblocks, c, sc, S, rows, res, sum);
    if (threadIdx.x) return;
    c->bflux0 = sum[0];
    if (METHOD > 1) c->bflux1 = sum[1];
    if (METHOD > 2) c->bflux2 = sum[2];
    const double dt = c->dt;
    c->integral = de_flux_integral(c->integral, dt, METHOD, sum[0], sum[1], sum[2]);
    const int e = de_end_step(c, c->t, dt, hist);
    if (e) atomicOr(&c->status, e);
}

// host-controlled steps (one scenario): the host computed dt
__global__ void de_set_dt(DeControl *c, double dt)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) c->dt = dt;
}

// host-controlled steps: boundary flux integral after the update
__global__ void de_integrate(DeControl *c, int method)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    c->integral = de_flux_integral(c->integral, c->dt, method, c->bflux0, c->bflux1, c->bflux2);
}

// time-control parameters and state for a run of device-controlled steps
struct DeBatchSetup {
    double t, rec_min, rec_max, cfl, max_dt, min_dt, finaltime, yieldtime, fixed_flux_dt, eps;
    int smallsteps, order, default_order, max_smallsteps, hist_cap, method;
    int stop_reached;  // a scenario already at its final or yield time takes no step
};

__device__ __forceinline__ void de_setup(DeControl *c, const DeBatchSetup &b)
{
    c->t = b.t;
    c->rec_min = b.rec_min;
    c->rec_max = b.rec_max;
    c->cfl = b.cfl;
    c->max_dt = b.max_dt;
    c->min_dt = b.min_dt;
    c->finaltime = b.finaltime;
    c->yieldtime = b.yieldtime;
    c->fixed_flux_dt = b.fixed_flux_dt;
    c->eps = b.eps;
    c->smallsteps = b.smallsteps;
    c->order = b.order;
    c->default_order = b.default_order;
    c->max_smallsteps = b.max_smallsteps;
    c->hist_cap = b.hist_cap;
    c->method = b.method;
    c->nsteps = 0;
    c->gstep = 0;
    c->pending = 0;
    c->done = 0;
    if (b.stop_reached) {
        if (c->t >= c->finaltime - c->eps) c->done = 1;
        else if (c->t >= c->yieldtime) c->done = 2;
    }
}

__global__ void de_setup_batch(DeControl *ctl, int S, const DeBatchSetup *__restrict__ setup)
{
    DeControl *c = de_scenario(ctl, S);
    if (c) de_setup(c, setup[c - ctl]);
}

// a single scenario's, from the kernel's arguments
__global__ void de_setup_one(DeControl *c, DeBatchSetup b)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) de_setup(c, b);
}

// leave device-controlled mode: steps are live again
__global__ void de_clear_done(DeControl *ctl, int S)
{
    DeControl *c = de_scenario(ctl, S);
    if (c) c->done = 0;
}

// clear the error bits of every scenario (a kernel, so that no memset node
// is needed in code a caller may capture)
__global__ void de_clear_status(DeControl *ctl, int S)
{
    DeControl *c = de_scenario(ctl, S);
    if (c) c->status = 0;
}

// the per-block partial of a per-thread value: wave sums, then the block's
// waves in order (the fixed order every volume reduction uses)
__device__ __forceinline__ void de_block_sum(double v, double *__restrict__ part, int lb)
{
    __shared__ double red[DE_BLOCK / 64];
    v = de_wave_sum(v);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) red[wv] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = red[0];
        for (int i = 1; i < DE_BLOCK / 64; i++) t += red[i];
        part[lb] = t;
    }
}

// per-block partial of sum(area * max(w - z, 0)) over the current state
__global__ void __launch_bounds__(DE_BLOCK)
de_volume(const int *__restrict__ scen, const DeControl *ctl, const DeQ *__restrict__ q,
          const double *__restrict__ area, double *__restrict__ part)
{
    const int lb = xcd_block();
    const DeControl *cb = scen ? ctl + scen[lb] : ctl;
    const int k = lb * DE_BLOCK + threadIdx.x;
    double v = 0.0;
    if (k < cb->kend) {
        const DeQ r = q[k];
        v = area[k] * de_height(r.w, r.z);
    }
    de_block_sum(v, part, lb);
}

// the same partials over separate stage, bed and area arrays of N triangles
__global__ void __launch_bounds__(DE_BLOCK)
de_volume_arrays(int N, const double *__restrict__ w, const double *__restrict__ z,
                 const double *__restrict__ area, double *__restrict__ part)
{
    const int lb = xcd_block();
    const int k = lb * DE_BLOCK + threadIdx.x;
    double v = 0.0;
    if (k < N) v = area[k] * de_height(w[k], z[k]);
    de_block_sum(v, part, lb);
}

// a one-scenario control block over triangles [0, N) in nblocks blocks
__global__ void de_control_init(DeControl *c, int N, int nblocks)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    c->kbeg = 0;
    c->kend = N;
    c->bbeg = 0;
    c->bend = nblocks;
    c->done = 0;
    c->status = 0;
    c->volume = 0.0;
}

__global__ void de_copy_volume(const DeControl *c, double *out)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *out = c->volume;
}

// mixed path: FP32 bed offsets of the neighbours' centroids from the own one
// (the local datum of the mixed flux), refreshed whenever the bed changes
__global__ void __launch_bounds__(DE_BLOCK)
de_bed_offsets(int kbeg, int kend, const int4 *__restrict__ nb, const DeQ *__restrict__ q,
               DeGeoF32 *gf)
{
    const int k = kbeg + blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= kend) return;
    const int4 v = nb[k];
    const int vv[3] = {v.x, v.y, v.z};
    const double z = q[k].z;
#pragma unroll
    for (int i = 0; i < 3; i++)
        gf[k].dzc[i] = vv[i] >= 0 ? float(q[vv[i] >> 2].z - z) : 0.f;
}

// ---------------------------------------------------------------------------
// output: gauge rows and SWW frames
// ---------------------------------------------------------------------------
// One row of gauge samples: the centroid state {w, uh, vh, z} of each gauge
// triangle and the relative time. Device-controlled steps record once per
// completed step (nsteps moved since the last row); FORCE records now with the
// host's time t (host-sequenced steps). One workgroup: the row counter moves
// after every lane has written its gauges.
template <bool FORCE>
__global__ void __launch_bounds__(256)
de_sample_gauges(DeControl *c, int G, const int *__restrict__ tri, const DeQ *__restrict__ S,
                 double t, double *__restrict__ times, double *__restrict__ vals)
{
    const long long ns = c->nsteps;
    const int row = c->grows;
    const bool take = (FORCE || ns != c->gstep) && row < c->gcap;
    if (take)
        for (int g = threadIdx.x; g < G; g += blockDim.x) {
            const DeQ q = S[tri[g]];
            double *o = vals + ((size_t)row * G + g) * 4;
            o[0] = q.w;
            o[1] = q.uh;
            o[2] = q.vh;
            o[3] = q.z;
        }
    __syncthreads();
    if (take && threadIdx.x == 0) {
        times[row] = FORCE ? t : c->t;
        c->grows = row + 1;
        c->gstep = ns;
    }
}

// gauge rows: mode 0 starts recording (cap rows, the current step is not a
// new one); mode 1 marks the rows downloaded
__global__ void de_gauge_control(DeControl *c, int mode, int cap)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    if (mode == 0) {
        c->gstep = c->nsteps;
        c->gcap = cap;
    }
    c->grows = 0;
}

// Node values by centroid averaging, _average_centroid_values
// (abstract_2d_finite_volumes/quantity.c:872-914): the centroid values of
// the triangles around each node summed in the node's entry order
// (vertex_value_indices), divided by their count; orphan nodes 0. Stage,
// momenta and bed together, then the storable-depth selection of
// SWW_file.store_timestep (anuga/file/sww.py:318-356): where the node depth
// w - z is below minimum_storable_height the stage is the bed and the
// momenta 0. Written as float32 [3][nodes] (the file's precision).
__global__ void __launch_bounds__(DE_BLOCK)
de_sww_nodes(int nodes, const int *__restrict__ start, const int *__restrict__ tri,
             const DeQ *__restrict__ S, double min_storable, float *__restrict__ out)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nodes) return;
    const int b = start[j], e = start[j + 1];
    double w = 0.0, uh = 0.0, vh = 0.0, z = 0.0;
    if (e > b) {
        for (int i = b; i < e; i++) {
            const DeQ q = S[tri[i]];
            w += q.w;
            uh += q.uh;
            vh += q.vh;
            z += q.z;
        }
        const double k = (double)(e - b);
        w = w / k;
        uh = uh / k;
        vh = vh / k;
        z = z / k;
    }
    const bool storable = w - z >= min_storable;
    out[j] = (float)(storable ? w : z);
    out[nodes + j] = storable ? (float)uh : 0.0f;
    out[2 * (size_t)nodes + j] = storable ? (float)vh : 0.0f;
}

// node values of one per-triangle quantity v[k * stride] by centroid averaging,
// as float32
__global__ void __launch_bounds__(DE_BLOCK)
de_node_values(int nodes, const int *__restrict__ start, const int *__restrict__ tri,
               const double *__restrict__ v, int stride, float *__restrict__ out)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nodes) return;
    const int b = start[j], e = start[j + 1];
    double a = 0.0;
    if (e > b) {
        for (int i = b; i < e; i++) a += v[(size_t)tri[i] * stride];
        a = a / (double)(e - b);
    }
    out[j] = (float)a;
}

// centroid values in the caller's order as float32: out[q][k] for the
// quantities at offsets off[q] of a record of `stride` doubles
__global__ void __launch_bounds__(DE_BLOCK)
de_gather_f32(int N, const int *__restrict__ iperm, const double *__restrict__ v, int stride,
              int nq, int4 off, float *__restrict__ out)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= N) return;
    const double *r = v + (size_t)iperm[k] * stride;
    const int o[4] = {off.x, off.y, off.z, off.w};
    for (int q = 0; q < nq; q++) out[(size_t)q * N + k] = (float)r[o[q]];
}

// ---------------------------------------------------------------------------
// whole quantities between the internal and the caller's order
// ---------------------------------------------------------------------------
// The vertex coordinates of the n triangles of the tiles in tx, from the
// tiles' nodes: sloped friction alone reads them, so they take their 48 B per
// triangle when it is first asked for.
__global__ void __launch_bounds__(DE_BLOCK)
de_node_vertices(int n, DeTileX tx, double2 *__restrict__ vx)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= n) return;
    const double2 *nd = tx.node + tx.nstart[blockIdx.x];
    const unsigned w = tx.nodes[k];
    for (int c = 0; c < 3; c++) vx[3 * (size_t)k + c] = nd[de_field(w, c)];
}

// One centroid quantity of n triangles (internal order, caller[k] the
// caller's index of triangle k): v[k * stride], or the depth of the records
// at v (HEIGHT), to out in the caller's order, so that 8 B per triangle cross
// to the host, in the order the host keeps them. Bound by the PCIe copy that
// follows: of 4M triangles 28 us here and 1.8 ms for the whole access, which
// took 30 ms when the host downloaded the 32 B records and reordered them
// (setting a quantity: 45 -> 10.7 ms, most of it numpy's). Of small meshes out
// is pinned host memory: 1600 triangles 27.3 -> 12.9 us without the copy.
template <bool HEIGHT>
__global__ void __launch_bounds__(DE_BLOCK)
de_get_field(int n, const int *__restrict__ caller, const double *__restrict__ v, int stride,
             double *__restrict__ out)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= n) return;
    const double *r = v + (size_t)k * stride;
    out[caller[k]] = HEIGHT ? de_height(r[0], r[3]) : r[0];
}

// the same from the caller's order: v[k * stride] = in[caller[k]], and v2 too
// where given (the bed is part of both state buffers)
__global__ void __launch_bounds__(DE_BLOCK)
de_set_field(int n, const int *__restrict__ caller, const double *__restrict__ in, int stride,
             double *__restrict__ v, double *__restrict__ v2)
{
    const int k = blockIdx.x * DE_BLOCK + threadIdx.x;
    if (k >= n) return;
    const double x = in[caller[k]];
    v[(size_t)k * stride] = x;
    if (v2) v2[(size_t)k * stride] = x;
}

// ---------------------------------------------------------------------------
// fractional-step operators
// ---------------------------------------------------------------------------
// Rate_operator.__call__ (anuga/operators/rate_operators.py:149-260) on its
// triangles after a step: local rate = factor * dt * rate; with all rates
// >= 0 the stage rises by it; otherwise (`careful`) the loss is capped at the
// depth and the momenta scale with the depth that remains. The inflow
// (local rate * area) is accumulated per workgroup, in influx[blockIdx.x],
// and summed when it is asked for (de_sum_parts). Atomic adds to one address were
// the kernel's time (36k triangles: 11.5 us with one per triangle, 9.4 with one
// per wave, 4.0 with none).
// Set_stage_operator after a step (set_quantity.py:95-131, quantity
// 'stage'): the stage centroid values of the region become the given values
// (value[i], or value0 for all); momenta and bed unchanged.
__global__ void __launch_bounds__(DE_BLOCK)
de_set_stage(const DeControl *ctl, int n, const int *__restrict__ idx,
             const double *__restrict__ value, double value0, DeQ *S)
{
    if (ctl->done) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    S[idx[i]].w = value ? value[i] : value0;
}

// The sum of n parts by one workgroup, in a fixed order, to pinned host memory:
// 8 B cross instead of the parts: 21.9 -> 15.0 us a read at 4M triangles, which
// have 15,625, and 12 to 13 either way at 400.
#define DE_SUM_THREADS 1024
__global__ void __launch_bounds__(DE_SUM_THREADS)
de_sum_parts(int n, const double *__restrict__ part, double *__restrict__ sum)
{
    __shared__ double red[DE_SUM_THREADS / 64];
    double a[4] = {0.0, 0.0, 0.0, 0.0};   // four loads on their way at a time
    for (int i = threadIdx.x; i < n; i += 4 * DE_SUM_THREADS)
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (i + j * DE_SUM_THREADS < n) a[j] += part[i + j * DE_SUM_THREADS];
    double s = de_wave_sum_nz((a[0] + a[1]) + (a[2] + a[3]));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x) return;
    for (int j = 1; j < DE_SUM_THREADS / 64; j++) s += red[j];
    *sum = s;
}

__global__ void __launch_bounds__(DE_BLOCK)
de_rate(const DeControl *ctl, int n, const int *__restrict__ idx, const double *__restrict__ rate,
        double rate0, double factor, int careful, DeQ *S, const double *__restrict__ area,
        double *influx)
{
    if (ctl->done) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double gain = 0.0;
    if (i < n) {
        const int k = idx[i];
        const double r = rate ? rate[i] : rate0;
        const double dt = ctl->dt;
        DeQ q = S[k];
        double lr = factor * dt * r;
        if (!careful) {
            q.w = q.w + lr;
        } else {
            const double h = q.w - q.z;
            lr = fmax(lr, -h);
            const double lf = lr < 0.0 ? (lr + h) / (h + 1.0e-10) : 1.0;
            q.w = q.w + lr;
            q.uh = q.uh * lf;
            q.vh = q.vh * lf;
        }
        S[k] = q;
        gain = lr * area[k];
    }
    __shared__ double red[DE_BLOCK / 64];
    gain = de_wave_sum_nz(gain);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = gain;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int j = 1; j < DE_BLOCK / 64; j++) gain += red[j];
        influx[blockIdx.x] += gain;
    }
}

// ---------------------------------------------------------------------------
// Inlet_operator (anuga/structures/inlet_operator.py:75-183) on the device:
// one workgroup levels the region with the reference's numpy arithmetic
// ---------------------------------------------------------------------------
#define DE_INLET_MAX 2048
#define DE_INLET_THREADS 1024

// numpy's sum of a contiguous float64 array (pairwise_sum of
// numpy/_core/src/umath/loops_utils.h.src): fewer than 8 in order from 0.0;
// up to 128 in eight interleaved partial sums, combined as a tree, then the
// rest in order; above 128 the halves at a multiple of 8, added.
__device__ __noinline__ double de_np_leaf(const double *x, int n)
{
    if (n < 8) {
        double r = 0.0;
        for (int i = 0; i < n; i++) r += x[i];
        return r;
    }
    double r[8];
#pragma unroll
    for (int j = 0; j < 8; j++) r[j] = x[j];
    int i = 8;
    for (; i < n - (n % 8); i += 8) {
#pragma unroll
        for (int j = 0; j < 8; j++) r[j] += x[i + j];
    }
    double res = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
    for (; i < n; i++) res += x[i];
    return res;
}

template <int D>
__device__ double de_np_sum(const double *x, int n)
{
    if (n <= 128) return de_np_leaf(x, n);
    int n2 = n / 2;
    n2 -= n2 % 8;
    return de_np_sum<D - 1>(x, n2) + de_np_sum<D - 1>(x + n2, n - n2);
}
template <>
__device__ double de_np_sum<0>(const double *x, int n)
{
    return de_np_leaf(x, n);
}

// Inlet parameters: the discharge over the step is 0.5 (Q1 + Q2) (Q at the
// operator's time and one timestep later); vmode 0: momenta from the
// region's velocities, 1: from (u, v), 2: zero. stats: cumulative volume,
// total applied volume, total requested volume, applied discharge.
struct DeInlet {
    int n;
    const int *idx;       // [n] internal triangles, in the operator's order
    const double *area;   // [n]
    double total_area;    // np.sum(area)
    double Q1, Q2;
    int vmode;
    double u, v;
    double *stats;        // [4]
};

__global__ void __launch_bounds__(DE_INLET_THREADS)
de_inlet(const DeControl *ctl, DeInlet in, DeQ *S)
{
    __shared__ double st[DE_INLET_MAX], el[DE_INLET_MAX], buf[DE_INLET_MAX];
    __shared__ int order[DE_INLET_MAX];
    __shared__ double level;
    __shared__ int how, last;
    if (ctl->done) return;
    const int n = in.n, t = threadIdx.x;
    const double vp = 1.0e-6;   // anuga/config.py velocity_protection
    for (int i = t; i < n; i += DE_INLET_THREADS) {
        const DeQ q = S[in.idx[i]];
        st[i] = q.w;
        el[i] = q.z;
        buf[i] = (q.w - q.z) * in.area[i];
    }
    __syncthreads();
    const double dt = ctl->dt;
    // the step's volume (inlet_operator.py:86-96); the case is uniform
    const double Q = 0.5 * (in.Q1 + in.Q2);
    const double volume = Q * dt;
    if (t == 0) {
        const double cv = de_np_sum<6>(buf, n);   // np.sum(depths * areas)
        how = volume >= 0.0 ? 0 : (cv + volume >= 0.0 ? 1 : 2);
        level = cv;
        if (how == 0) {
            in.stats[0] += volume;     // fractional_step_volume_integral
            in.stats[2] += volume;     // total_requested_volume
            in.stats[1] += volume;     // total_applied_volume
            in.stats[3] = Q;
        } else if (how == 1) {
            in.stats[2] += volume;
            in.stats[0] += volume;
            in.stats[1] += volume;
            in.stats[3] = Q;
        } else {
            in.stats[2] += volume;
            in.stats[0] -= cv;
            in.stats[1] += -cv;
            in.stats[3] = -cv / dt;
        }
    }
    __syncthreads();
    if (how == 0) {
        // set_stages_evenly (inlet.py:192-225): stages.argsort(), ties by
        // position; then the cumulative areas and volumes in that order
        int np2 = 1;
        while (np2 < n) np2 <<= 1;
        for (int i = t; i < np2; i += DE_INLET_THREADS) {
            order[i] = i < n ? i : -1;
            if (i < n) buf[i] = in.area[i];
        }
        __syncthreads();
        for (int size = 2; size <= np2; size <<= 1) {
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                for (int i = t; i < np2; i += DE_INLET_THREADS) {
                    const int j = i ^ stride;
                    if (j > i) {
                        const int a = order[i], b = order[j];
                        // -1 (padding) sorts last
                        const bool gt = a < 0 ? b >= 0
                                      : (b >= 0 && (st[a] > st[b] || (st[a] == st[b] && a > b)));
                        const bool up = (i & size) == 0;
                        if (gt == up) {
                            order[i] = b;
                            order[j] = a;
                        }
                    }
                }
                __syncthreads();
            }
        }
        if (t == 0) {
            double sa = buf[order[0]], sv = 0.0, sa_at = sa, sv_at = 0.0;
            int index = 0;
            for (int i = 1; i < n; i++) {
                const double nsv = sv + sa * (st[order[i]] - st[order[i - 1]]);
                sa = sa + buf[order[i]];
                sv = nsv;
                if (!(sv <= volume)) break;
                index = i;
                sa_at = sa;
                sv_at = sv;
            }
            const double depth = (volume - sv_at) / sa_at;
            level = st[order[index]] + depth;
            last = index;
        }
        __syncthreads();
        for (int i = t; i <= last; i += DE_INLET_THREADS) st[order[i]] = level;
    } else if (how == 1) {
        const double depth = (level + volume) / in.total_area;
        for (int i = t; i < n; i += DE_INLET_THREADS) st[i] = el[i] + depth;
    } else {
        for (int i = t; i < n; i += DE_INLET_THREADS) st[i] = el[i] + 0.0;
    }
    __syncthreads();
    // momenta from the velocities before the change (inlet.py:122-128)
    for (int i = t; i < n; i += DE_INLET_THREADS) {
        const int k = in.idx[i];
        DeQ q = S[k];
        const double d0 = q.w - q.z, d1 = st[i] - el[i];
        if (how == 2 || in.vmode == 2) {
            q.uh = 0.0;
            q.vh = 0.0;
        } else if (in.vmode == 1) {
            q.uh = d1 * in.u;
            q.vh = d1 * in.v;
        } else {
            const double u = q.uh * d0 / (d0 * d0 + vp);
            const double v = q.vh * d0 / (d0 * d0 + vp);
            q.uh = d1 * u;
            q.vh = d1 * v;
        }
        q.w = st[i];
        S[k] = q;
    }
}

// state of a subset of triangles (internal ids) to [n][4] {w, uh, vh, z}
__global__ void __launch_bounds__(DE_BLOCK)
de_gather_state(int n, const int *__restrict__ idx, const DeQ *__restrict__ S, DeQ *__restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = S[idx[i]];
}

// w, uh, vh of a subset of triangles from [n][4] (the bed is kept)
__global__ void __launch_bounds__(DE_BLOCK)
de_scatter_state(int n, const int *__restrict__ idx, const DeQ *__restrict__ in, DeQ *S)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    DeQ q = S[idx[i]];
    const DeQ v = in[i];
    q.w = v.w;
    q.uh = v.uh;
    q.vh = v.vh;
    S[idx[i]] = q;
}
