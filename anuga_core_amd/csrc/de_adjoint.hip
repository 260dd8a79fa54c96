// Discrete adjoint of the FP64 DE1 step with a fixed timestep, on the device.
//
// One thread per triangle, as the forward. Each kernel applies vector-Jacobian
// products of de_adjoint.h to its triangle. The adjoint of a gather is a
// scatter; it is kept deterministic and free of atomics: every thread writes
// its own triangle's entries only, what belongs to a neighbour into a slot of
// its own, and the neighbour sums the slots that are meant for it in a fixed
// order in the next kernel. Gradients are therefore the same bits on every
// run. The forward quantities each product needs (flags, edge values, explicit
// updates, the stage state) come from the production kernels, recomputed step
// by step from checkpoints.
#include "de_adjoint.h"

__device__ __forceinline__ int adj_tid() { return blockIdx.x * blockDim.x + threadIdx.x; }
// the triangle of a thread: the workgroups' order of the production kernels
__device__ __forceinline__ int adj_triangle() { return xcd_block() * DE_BLOCK + threadIdx.x; }

// Adjoint of the update (friction, update, fix_negative) and of the flux of
// one stage of the step. SECOND: lam is the adjoint of the step's result, half
// of which enters this stage (the final saxpy); the adjoint of the stage's
// state, without the extrapolation's share, goes to lam1. Otherwise the first
// stage: lam1 and the second stage's extrapolation (X) are the adjoint of its
// result, and lam becomes half of itself (the saxpy's direct path) plus this
// stage's share. lamE: the adjoints of a triangle's edge values from its own
// flux, lamN those of its neighbours' from it, both in its own slots.
//
// Update, flux, saxpy and the gather of X only meet in a triangle's own
// entries, which stay in registers between them, and the update's product is
// one reverse sweep instead of two passes of 4 duals. As separate kernels over
// zeroed arrays, which 28 FP64 atomics a triangle added to, the second stage
// took 55 us at 160k triangles and the first 54; now 20 and 27. Bound by
// latency: 168 and 184 VGPRs leave 3 and 2 waves per SIMD for some 550 B a
// triangle; held to 168, the first stage spills 24 and gains nothing.
template <bool SECOND>
__global__ void __launch_bounds__(DE_BLOCK)
adj_k_stage(AdjView m, const double *__restrict__ S, const unsigned char *__restrict__ fl,
            const double *__restrict__ E, const double *__restrict__ ex,
            const double *__restrict__ X, double *lam, double *lam1, double *__restrict__ lamE,
            double *__restrict__ lamN, double *zbar, double *nbar)
{
    const int k = adj_triangle();
    if (k >= m.N) return;
    const size_t N = m.N;
    int v[3], sur[3];
    adj_neighbours(m, k, v, sur);
    const double q[4] = {S[4 * (size_t)k], S[4 * (size_t)k + 1], S[4 * (size_t)k + 2],
                         S[4 * (size_t)k + 3]};
    const unsigned f = fl[k];
    double c[4];
    adj_centroid<double>(q, f, c);
    double lz = zbar[k], lo[3], ls[3];
    for (int j = 0; j < 3; j++) {
        const double half = 0.5 * lam[j * N + k];
        lo[j] = SECOND ? half : lam1[j * N + k];
        ls[j] = SECOND ? 0.0 : half;
    }
    if constexpr (!SECOND) adj_sum_extrap(m, X, k, v, lo, lz);
    double lex[3], lc[4];
    {
        const double e[3] = {ex[k], ex[N + k], ex[2 * N + k]};
        double g[8];
        adj_advance_vjp(c, m.eta[k], e, m.dt, m.p, lo, g);
        adj_add_centroid(f, g, ls, lz);
        if (g[4] != 0.0) nbar[k] += g[4];
        for (int j = 0; j < 3; j++) lex[j] = g[5 + j];
    }
    const auto own = [&](int i, const double g[4]) {
        for (int t = 0; t < 4; t++) lamE[4 * (i * N + k) + t] = g[t];
    };
    const auto other = [&](int i, const double g[4]) {
        for (int t = 0; t < 4; t++) lamN[4 * (i * N + k) + t] = g[t];
    };
    adj_flux_vjp(m, E, c, lex, k, v, own, other, lc);
    adj_add_centroid(f, lc, ls, lz);
    zbar[k] = lz;
    for (int j = 0; j < 3; j++) (SECOND ? lam1 : lam)[j * N + k] = ls[j];
}

// Adjoint of the extrapolation: a triangle's own flux's adjoints of its edge
// values and those that its neighbours' fluxes left in the slots of the edges
// that name its edge (one, but for meshes whose triangles share two edges).
// The slots are records of 4, so that a neighbour's comes with one line: 26.6
// to 22.9 us at 160k triangles together with four limiters instead of seven
// (1684 FP64 instructions instead of 2287). 187 VGPRs, 2 waves per SIMD; held
// to 168 it spills 50 and takes 26.7.
__global__ void __launch_bounds__(DE_BLOCK)
adj_k_extrap(AdjView m, const double *__restrict__ S, const unsigned char *__restrict__ fl,
             const double *__restrict__ lamE, const double *__restrict__ lamN,
             double *__restrict__ X)
{
    const int k = adj_triangle();
    if (k >= m.N) return;
    const size_t N = m.N;
    int v[3], sur[3];
    adj_neighbours(m, k, v, sur);
    double lo[12];
    for (int i = 0; i < 3; i++) {
        for (int t = 0; t < 4; t++) lo[4 * i + t] = lamE[4 * (i * N + k) + t];
        if (v[i] < 0) continue;
        const int me = 4 * k + i, n = sur[i];
        const int4 w = reinterpret_cast<const int4 *>(m.nb)[n];
        const bool at[3] = {w.x == me, w.y == me, w.z == me};
        const int j = at[0] ? 0 : (at[1] ? 1 : 2);
        if (at[0] || at[1] || at[2])
            for (int t = 0; t < 4; t++) lo[4 * i + t] += lamN[4 * (j * N + n) + t];
        for (int l = 1; l < 3; l++)
            if (at[l] && l != j)
                for (int t = 0; t < 4; t++) lo[4 * i + t] += lamN[4 * (l * N + n) + t];
    }
    adj_store_extrap(m, S, fl, lo, k, v, sur, X);
}

// the first stage's extrapolation adjoints, stored per stencil slot, summed
// per triangle in a fixed order: the step's start
__global__ void __launch_bounds__(DE_BLOCK)
adj_k_extrap_gather(AdjView m, const double *__restrict__ X, double *lamS, double *zbar)
{
    const int t = adj_triangle();
    if (t >= m.N) return;
    adj_gather_extrap(m, X, t, lamS, zbar);
}

// stage of the gauge triangles into a record row
__global__ void adj_k_gauges(int G, const int *__restrict__ gauges, const DeQ *__restrict__ S,
                             double *__restrict__ row)
{
    const int g = adj_tid();
    if (g < G) row[g] = S[gauges[g]].w;
}

// add the loss's sensitivity to the gauges' stage into the stage adjoint
// (gauges are distinct)
__global__ void adj_k_gauge_seed(int G, const int *__restrict__ gauges,
                                 const double *__restrict__ row, double *lam)
{
    const int g = adj_tid();
    if (g < G) lam[gauges[g]] += row[g];
}
