/*
 * hs_hines.hip -- multicompartment cells on gfx950: a batch of independent
 * SpatialNeuron trees, one workgroup per tree, the tree's state held on chip
 * (registers + LDS) for all the steps of a launch.
 *
 * Per step, in the reference's arithmetic (spatialstateupdate.cu), parallel
 * where the reference's serial loops have independent iterations:
 *   1. lanes over compartments: HH channels linearised at the start of the
 *      step (_gtot, _I0); the main diagonal and right-hand side of each
 *      compartment go to LDS
 *   2. lanes over sections: Thomas elimination + back substitution with three
 *      right-hand sides (v_star, u_plus, u_minus) walking the section in LDS
 *   3. the coupling system over section end points: built node-parallel (each
 *      node adds its children's terms in the reference's order), eliminated
 *      level by level from the leaves, substituted level by level from the root
 *      -- every node sees exactly the operations of the serial loops
 *   4. lanes over compartments: v = v_star + B[parent] u_minus + B[i+1] u_plus
 * and, independent of the solve (they only need the old v), the gates advance
 * one exponential-Euler step.  The solve is FP64; the channel arithmetic is FP64
 * or FP32.
 *
 * What bounds a step: at one or two trees per compute unit the chain of one tree --
 * two rows of divisions per section and two hops per tree level, 5 + 3 us -- and at
 * eight the instructions as much as the chains (of what the VALU can issue 57% with
 * FP64 channels, 66% with FP32; 46 and 25 bytes of gates a compartment and step).
 *
 * Split: the first waves of a workgroup (one per 64 sections) solve -- 2 and 3,
 * a serial chain of divisions per section and per tree level that more lanes
 * would not shorten -- while the others advance the gates, most of the
 * arithmetic, in chunks of 64 compartments that they take from a counter; a
 * solver that is done takes chunks too.  Any wave may take any chunk, so the
 * gates live in LDS where that has room, else in global memory (L1/L2: 24 bytes in
 * and out per compartment and step).  Two barriers a step.  Waves per tree follow
 * the batch, about 16 per compute unit in all: two per tree at 2048 trees, whose
 * chains overlap with the other trees' arithmetic, up to 16 for one tree per unit
 * (24 per unit gained 10% on 2000 trees of 30 to 120 compartments and lost 5% at
 * 2048 of 100 to 400 and 40% where 64 sections take more registers).
 *
 * Layout: sections by length, compartments row by row over them (hs_h_place), so
 * that the solver's lanes touch neighbouring words, and a compartment's four values
 * together.  Trees in the order of their size, dealt out so that the ones sharing a
 * compute unit add up to about the same.
 *
 * Measured, us a step, with every wave doing all phases over its own compartments
 * held in registers, an array per value and IEEE divisions -> now: 2048 trees of 100
 * to 400 compartments FP64 32.2 -> 19.8, 301 of 20 to 700 FP32 31.9 -> 10.5, 900 of
 * 200 to 800 FP64 42.5 -> 18, 40 of 10 to 50 FP64 10.8 -> 6.0.
 *
 * Fewer instructions for the same bits: a reciprocal of a row and a quotient of
 * rates is the compiler's sequence (v_rcp, two Newton steps, quotient, residual
 * correction) without v_div_scale and v_div_fixup, which only act outside the
 * exponent range that the constants (checked when the batch is created) and the
 * potentials and conductances (checked every step, a step outside takes the IEEE
 * division) stay in;
 * a division by a constant c is x*(1/c) and one residual correction, exact because
 * 1/c rounded is within half an ulp's relative error of 1/c for these c; exp skips
 * its clamps.
 */
#include <stdarg.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <memory>
#include <vector>

#include "../../include/hs.h"
#include "hs_device.h"

#define HS_HINES_MAXC 1024
#define HS_HINES_MAXS 255
#define HS_HINES_RL 4 /* children per node */
#define HS_HINES_PF 2 /* rows that the Thomas sweep reads ahead (2048 trees: 20.9 us a step, 4: 22.3, 8: 27.7) */
/* potentials (V) whose channel rates, and dt times them, the short forms cover:
   the largest rate there is beta_m(-0.1) = 1.04e6/s, so dt <= 7e-5 s keeps every
   exponent of exp within +-75 */
#define HS_HINES_VLO (-0.1)
#define HS_HINES_VHI 0.2
#define HS_HINES_DTMAX 7e-5
/* conductance densities (S/m2) that leave the rows' pivots to their constants: gates may be
   set to anything, and a pivot of 0 or infinity takes the IEEE division */
#define HS_HINES_GMAX 1e30

template <typename R>
struct HinesDesc {
    const int32_t *tree_comp, *tree_sec;
    const int32_t *order; /* tree of each workgroup */
    /* per compartment, in the caller's order: the state, which a launch reads and writes
       once, and where the compartment is in the order of hs_h_place, from its tree's first */
    double *v;
    R *m, *n, *h;
    const int32_t *place;
    /* per compartment, in the order of hs_h_place */
    R *wm, *wn, *wh; /* the gates of a launch, where LDS has no room for them */
    const double2 *band; /* superdiagonal, subdiagonal of its row */
    const double *ab1, *cdt, *iext;
    const int32_t *ends; /* nodes at the two ends of each compartment's section: parent | own << 8 */
    /* rows: off[tree_row[t] + q] is the tree's first compartment that is the q-th of its
       section (2 HS_HINES_PF + 2 entries more than the longest section has compartments) */
    const int32_t *tree_row, *off;
    /* per section: its first and last compartment, the node above */
    const int32_t *first, *last, *mparent;
    const double *invr0, *invrn;
    /* per section by rank: compartments, b_plus at the last one, b_minus at the first */
    const int32_t *len;
    const double *bplus, *bminus;
    /* per node (tree-local node k of tree t at tree_sec[t] + t + k) */
    const int32_t *nchild, *child, *level; /* level: depth of the node */
    const int32_t *nlevels;                /* per tree */
    int32_t *spikes;                       /* per tree */
    R chan[7];
    double vth;
    int cmax, smax, rmax; /* most compartments, sections, rows of a tree */
    int narrow; /* the constants allow the short divisions */
    int row;    /* workgroups per round of the chip: one per compute unit */
};

/* n / d as the compiler expands it, without the scaling and the fix-up of operands
   at the ends of the exponent range.  For the rates of the channels and for the
   reciprocals of the rows, whose operands stay clear of them */
template <bool SHORT> __device__ __forceinline__ double hs_quot(double n, double d)
{
    if (!SHORT) return n / d;
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    const double q = n * r;
    return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

template <bool SHORT> __device__ __forceinline__ float hs_quot(float n, float d)
{
    if (!SHORT) return n / d;
    float r = __builtin_amdgcn_rcpf(d);
    r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
    float q = n * r;
    q = __builtin_fmaf(__builtin_fmaf(-d, q, n), r, q);
    return __builtin_fmaf(__builtin_fmaf(-d, q, n), r, q);
}

/* x / c, y = 1 / c rounded: |c y - 1| is at most 0.43 of the unit roundoff for
   0.01, 0.018, 0.02 and 0.08 in double, so x*y is within one ulp and the residual
   step rounds correctly (Markstein); in float the same, over every float in
   [2^-40, 2^9) */
__device__ __forceinline__ double hs_quotc(double x, double c, double y)
{
    const double q = x * y;
    return __builtin_fma(__builtin_fma(-c, q, x), y, q);
}

__device__ __forceinline__ float hs_quotc(float x, float c, float y)
{
    const float q = x * y;
    return __builtin_fmaf(__builtin_fmaf(-c, q, x), y, q);
}

/* the channel expressions with the short forms */
#pragma push_macro("HS_HD")
#undef HS_HD
#define HS_HD __device__ static inline __attribute__((always_inline))
#define HS_FAST_CONTRACT
#define HS_DIV(a, b) hs_quot<true>(a, b)
#define HS_DIVC(a, c) hs_quotc(a, c, (R)1.0 / (c))
#define R double
#define HS_SFX(name) name##_f64n
#define HS_EXP hs_exp_core
#include "hs_model_body.inc"
#undef R
#undef HS_SFX
#undef HS_EXP
#define R float
#define HS_SFX(name) name##_f32n
#define HS_EXP hs_expf_core
#include "hs_model_body.inc"
#undef R
#undef HS_SFX
#undef HS_EXP
#undef HS_DIV
#undef HS_DIVC
#undef HS_FAST_CONTRACT
#pragma pop_macro("HS_HD")

template <typename R> struct HsMc;
template <> struct HsMc<double> {
    static __device__ __forceinline__ void conduct(const double *g, const double *k, double *gt, double *i0)
    {
        hs_mc_conduct_f64(g, k, gt, i0);
    }
    template <bool SHORT> static __device__ __forceinline__ void gates(double v, double *g, double dt)
    {
        if (SHORT) hs_mc_gates_f64n(v, g, dt);
        else hs_mc_gates_f64(v, g, dt);
    }
};
template <> struct HsMc<float> {
    static __device__ __forceinline__ void conduct(const float *g, const float *k, float *gt, float *i0)
    {
        hs_mc_conduct_f32(g, k, gt, i0);
    }
    template <bool SHORT> static __device__ __forceinline__ void gates(float v, float *g, float dt)
    {
        if (SHORT) hs_mc_gates_f32n(v, g, dt);
        else hs_mc_gates_f32(v, g, dt);
    }
};

/* a compartment's row: main diagonal, then c (superdiagonal after elimination);
   right-hand side, then v_star; u_minus; u_plus.  Together, as 16-byte words: one
   address, and half the LDS accesses of an array each */
struct alignas(16) HinesRow {
    double a, v, m, p;
};

struct HinesLds {
    HinesRow *row;            /* per compartment */
    double *V;                /* the potential */
    double2 *G;               /* per node: terms for the parent's row */
    double *Bn;               /* per node: the solution */
    int *off;                 /* per row: its first compartment (HinesDesc.off) */
    int *wild, *next;         /* by step parity: a potential is outside the short range; the next chunk */
    int *met;                 /* arrivals of solver waves */
};

/* Thomas elimination and back substitution of the section of rank t
   (spatialstateupdate.cu:151-191), len compartments, rows: the longest of the wave.
   u_plus of the elimination is zero up to the last compartment, where it is b_plus
   times the row's factor: it is not carried along.  Every load is unconditional (at
   a clamped place) and ahead of its use -- the off-diagonal bands, an L2 round trip,
   HS_HINES_PF rows, the diagonal and right-hand side in LDS one row and before the
   stores that the compiler would not move them across -- so that a row costs its
   chain of one division; lanes whose section has ended only skip the arithmetic */
template <bool SHORT>
__device__ __forceinline__ void hs_thomas(const HinesLds &L, int t, int len, int rows, bool root, double bp, double bm,
                                          int nc, const double2 *__restrict__ band)
{
    const int end = nc - 1;
    int at[HS_HINES_PF + 1];
    double2 ca[HS_HINES_PF];
#pragma unroll
    for (int u = 0; u <= HS_HINES_PF; ++u) at[u] = min(L.off[u] + t, end);
#pragma unroll
    for (int u = 0; u < HS_HINES_PF; ++u) ca[u] = band[at[u]];
    double b_n = L.row[at[0]].a, v_n = L.row[at[0]].v;
    double cp = 0.0, vp = 0.0, upp = 0.0, ump = 0.0;
    for (int q0 = 0; q0 < rows; q0 += HS_HINES_PF) {
#pragma unroll
        for (int u = 0; u < HS_HINES_PF; ++u) {
            const int q = q0 + u, j = at[0];
            const double b = b_n, ai = ca[u].y, cd = ca[u].x, v0 = v_n;
            b_n = L.row[at[1]].a;
            v_n = L.row[at[1]].v;
            ca[u] = band[at[HS_HINES_PF]];
#pragma unroll
            for (int w = 0; w < HS_HINES_PF; ++w) at[w] = at[w + 1];
            at[HS_HINES_PF] = min(L.off[q + HS_HINES_PF + 1] + t, end);
            if (q < len) {
                double cj, vs, um;
                if (q == 0) {
                    /* section start: the subdiagonal is exactly 0 (its axial conductance is
                       cut), so (x - 0*prev)*m == x*m; the tree's first compartment has
                       divisions, as the reference has them */
                    if (root) {
                        cj = cd / b;
                        vs = v0 / b;
                        um = bm / b;
                        upp = bp / b;
                    } else {
                        const double m = hs_quot<SHORT>(1.0, b);
                        cj = cd * m;
                        vs = v0 * m;
                        um = bm * m;
                        upp = bp * m;
                    }
                } else {
                    const double m = hs_quot<SHORT>(1.0, b - ai * cp);
                    cj = cd * m;
                    vs = (v0 - ai * vp) * m;
                    um = (0.0 - ai * ump) * m;
                    upp = bp * m;
                }
                L.row[j].a = cp = cj;
                L.row[j].v = vp = vs;
                L.row[j].m = ump = um;
                if (q == len - 1) L.row[j].p = upp;
            }
        }
    }
    /* back: a group of rows is read while the one above it is computed */
    double c_n[HS_HINES_PF], r_n[HS_HINES_PF], m_n[HS_HINES_PF];
    int j_n[HS_HINES_PF];
    auto read = [&](int q0) {
#pragma unroll
        for (int u = 0; u < HS_HINES_PF; ++u) {
            const int j = min(L.off[max(q0 - u, 0)] + t, end);
            c_n[u] = L.row[j].a;
            r_n[u] = L.row[j].v;
            m_n[u] = L.row[j].m;
            j_n[u] = j;
        }
    };
    read(rows - 2);
    for (int q0 = rows - 2; q0 >= 0; q0 -= HS_HINES_PF) {
        double c[HS_HINES_PF], r[HS_HINES_PF], m[HS_HINES_PF];
        int j[HS_HINES_PF];
#pragma unroll
        for (int u = 0; u < HS_HINES_PF; ++u) {
            c[u] = c_n[u];
            r[u] = r_n[u];
            m[u] = m_n[u];
            j[u] = j_n[u];
        }
        read(q0 - HS_HINES_PF);
#pragma unroll
        for (int u = 0; u < HS_HINES_PF; ++u)
            if (q0 - u >= 0 && q0 - u <= len - 2) {
                L.row[j[u]].v = vp = r[u] - c[u] * vp;
                L.row[j[u]].p = upp = 0.0 - c[u] * upp;
                L.row[j[u]].m = ump = m[u] - c[u] * ump;
            }
    }
}

/* a wave's LDS accesses complete in order: what other lanes of the wave wrote
   before this point is read after it */
__device__ __forceinline__ void hs_wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

/* the coupling system (spatialstateupdate.cu:224-296) by one wave, node
   lane + 64 m on lane `lane`; constant per node: its level, up to four children,
   parent, section ends and conductances.  A child prepares its own term of the
   parent's row (factor times its off-diagonal, factor times its right-hand side),
   so that a level is one LDS hop, the subtractions and one division long.  The
   divisions are IEEE ones: what a far section sends may be as small as it gets */
template <int M> struct HinesNode {
    int level[M], kids[M], nkids[M], parent[M], f[M], l[M];
    double g0[M], gn[M];
};

template <int M>
__device__ __forceinline__ void hs_couple(const HinesLds &L, const HinesNode<M> &N, int nn, int nlev, int lane)
{
    double pd[M], b[M], pp[M], pc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int k = lane + HS_WAVE * m;
        if (M > 1 && HS_WAVE * m >= nn) continue; /* uniform */
        pd[m] = b[m] = pp[m] = pc[m] = 0.0;
        if (k >= nn) continue;
        if (k == 0) {
            const int f = N.f[m];
            pd[m] = L.row[f].m - 1;
            b[m] = -L.row[f].v;
        } else {
            const int f = N.f[m], l = N.l[m];
            pd[m] = (1 - L.row[l].p) * N.gn[m];
            pp[m] = -L.row[l].m * N.gn[m];
            b[m] = L.row[l].v * N.gn[m];
            if (k == 1) { /* the root section's start is node 0 itself */
                pc[m] = L.row[f].p;
            } else {
                pc[m] = -L.row[f].p * N.g0[m];
                L.G[k].x = (1 - L.row[f].m) * N.g0[m];
                L.G[k].y = L.row[f].v * N.g0[m];
            }
        }
    }
    hs_wave_fence();
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int k = lane + HS_WAVE * m;
        if (M > 1 && HS_WAVE * m >= nn) continue;
#pragma unroll
        for (int q = 0; q < HS_HINES_RL; ++q) {
            const int c = (N.kids[m] >> (8 * q)) & 255;
            if (k < nn && q < N.nkids[m] && c != 1) {
                pd[m] += L.G[c].x;
                b[m] += L.G[c].y;
            }
        }
    }
    hs_wave_fence();
    for (int lev = nlev - 1; lev >= 0; --lev) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int k = lane + HS_WAVE * m;
            if (M > 1 && HS_WAVE * m >= nn) continue;
            if (N.level[m] == lev) {
#pragma unroll
                for (int q = 0; q < HS_HINES_RL; ++q)
                    if (q < N.nkids[m]) {
                        const int c = (N.kids[m] >> (8 * q)) & 255;
                        pd[m] = pd[m] - L.G[c].x;
                        b[m] = b[m] - L.G[c].y;
                    }
                if (k > 0) {
                    const double sf = pc[m] / pd[m];
                    L.G[k].x = sf * pp[m];
                    L.G[k].y = sf * b[m];
                } else {
                    L.Bn[0] = b[m] / pd[m];
                }
            }
        }
        hs_wave_fence();
    }
    for (int lev = 1; lev < nlev; ++lev) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (M > 1 && HS_WAVE * m >= nn) continue;
            if (N.level[m] == lev) {
                const double x = b[m] - pp[m] * L.Bn[N.parent[m]];
                L.Bn[lane + HS_WAVE * m] = x / pd[m];
            }
        }
        hs_wave_fence();
    }
}

/* waves of a workgroup that solve */
__host__ __device__ static inline int hs_hines_solvers(int smax) { return (smax + HS_WAVE - 1) / HS_WAVE; }

/* per-compartment values of a tree: in LDS where the batch leaves room for it (INLDS),
   else in global memory (L1 / L2) */
template <typename R> struct HinesComp {
    R *m, *n, *h;
    const double *ab1, *cdt, *iext;
    const int32_t *ends;
};

/* M nodes per lane of the first solver wave.  Up to 128 registers: four waves per
   SIMD, 16 per compute unit, two per tree of a batch of 2048 */
template <typename R, int M, bool INLDS>
__global__ __launch_bounds__(1024) void hs_k_hines(const HinesDesc<R> d, int nsteps)
{
    extern __shared__ __align__(16) double lds[];
    /* every other round of workgroups has its waves' roles reversed: the waves of a
       workgroup go to neighbouring SIMDs, and one SIMD should not get the solvers of
       all trees of its compute unit */
    const int tree = d.order[blockIdx.x], lane = hs_lane();
    const int tid = (blockIdx.x / d.row) & 1 ? (int)blockDim.x - HS_WAVE - (int)(threadIdx.x & ~(HS_WAVE - 1)) + lane
                                            : (int)threadIdx.x;
    const int wave = tid / HS_WAVE;
    const int c0 = d.tree_comp[tree], nc = d.tree_comp[tree + 1] - c0;
    const int s0 = d.tree_sec[tree], ns = d.tree_sec[tree + 1] - s0;
    const int n0 = s0 + tree, nn = ns + 1; /* node offset, nodes */
    const int CM = d.cmax, SM = d.smax;
    HinesLds L;
    L.row = (HinesRow *)lds;
    L.G = (double2 *)(L.row + CM);
    L.V = (double *)(L.G + SM + 1);
    L.Bn = L.V + CM;
    L.off = (int *)(L.Bn + SM + 1);
    L.wild = L.off + d.rmax;
    L.next = L.wild + 2;
    L.met = L.next + 2;
    const int r0 = d.tree_row[tree], nr = d.tree_row[tree + 1] - r0;
    for (int q = tid; q < nr; q += blockDim.x) L.off[q] = d.off[r0 + q];
    /* the off-diagonal bands are constant: read from global memory (L1/L2
       resident after the first step) to keep the workgroup's LDS small enough
       for every tree of a large batch to be resident at once */
    const double2 *__restrict__ band = d.band + c0;
    HinesComp<R> C;
    if constexpr (INLDS) {
        double *const ab1 = (double *)(((size_t)(L.met + 2) + 7) & ~(size_t)7), *const cdt = ab1 + CM, *const iext = cdt + CM;
        C = {(R *)(iext + CM), (R *)(iext + CM) + CM, (R *)(iext + CM) + 2 * CM, ab1, cdt, iext,
             (int32_t *)((R *)(iext + CM) + 3 * CM)};
        for (int j = tid; j < nc; j += blockDim.x) {
            ab1[j] = d.ab1[c0 + j];
            cdt[j] = d.cdt[c0 + j];
            iext[j] = d.iext[c0 + j];
            const_cast<int32_t *>(C.ends)[j] = d.ends[c0 + j];
        }
    } else {
        C = {d.wm + c0, d.wn + c0, d.wh + c0, d.ab1 + c0, d.cdt + c0, d.iext + c0, d.ends + c0};
    }
    for (int j = tid; j < nc; j += blockDim.x) {
        const int p = d.place[c0 + j];
        L.V[p] = d.v[c0 + j];
        C.m[p] = d.m[c0 + j];
        C.n[p] = d.n[c0 + j];
        C.h[p] = d.h[c0 + j];
    }
    if (tid == 0) L.wild[0] = L.wild[1] = L.next[0] = L.next[1] = *L.met = 0;
    __syncthreads();

    const int nsolve = hs_hines_solvers(SM), nlev = d.nlevels[tree];
    HinesNode<M> N;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int k = lane + HS_WAVE * m;
        N.level[m] = -1;
        N.kids[m] = N.nkids[m] = N.parent[m] = N.f[m] = N.l[m] = 0;
        N.g0[m] = N.gn[m] = 0.0;
        if (wave != 0 || k >= nn) continue;
        N.level[m] = d.level[n0 + k];
        N.nkids[m] = d.nchild[n0 + k];
        for (int q = 0; q < HS_HINES_RL; ++q) N.kids[m] |= d.child[(n0 + k) * HS_HINES_RL + q] << (8 * q);
        if (k > 0) {
            const int i = k - 1;
            N.parent[m] = d.mparent[s0 + i];
            N.f[m] = d.first[s0 + i];
            N.l[m] = d.last[s0 + i];
            N.g0[m] = d.invr0[s0 + i];
            N.gn[m] = d.invrn[s0 + i];
        } else {
            N.f[m] = d.first[s0];
        }
    }
    /* a solver's section: by rank */
    const bool solver = wave < nsolve && tid < ns;
    const int len = solver ? d.len[s0 + tid] : 0, rows = __builtin_amdgcn_readfirstlane(len), spot = d.first[s0];
    const double bp = solver ? d.bplus[s0 + tid] : 0.0, bm = solver ? d.bminus[s0 + tid] : 0.0;
    R kc[7];
#pragma unroll
    for (int q = 0; q < 7; ++q) kc[q] = d.chan[q];
    const int met = (ns + HS_WAVE - 1) / HS_WAVE; /* solver waves with sections */
    int spikes = 0;
    for (int step = 0; step <= nsteps; ++step) {
        /* 4. of the step before: combine (spatialstateupdate.cu:339-349); 1. of this one:
           conductances (spatialstateupdate.cu:108-113) and the rows of the system */
        bool wild = false;
        for (int j = tid; j < nc; j += blockDim.x) {
            const R g3[3] = {C.m[j], C.n[j], C.h[j]};
            const double ab1 = C.ab1[j], cdt = C.cdt[j], iext = C.iext[j];
            double v = L.V[j];
            if (step > 0) {
                const int e = C.ends[j];
                const double was = v;
                v = L.row[j].v + L.Bn[e & 255] * L.row[j].m + L.Bn[e >> 8] * L.row[j].p;
                L.V[j] = v;
                if (j == spot && v > d.vth && !(was > d.vth)) ++spikes;
            }
            if (step < nsteps) {
                R gt, i0;
                HsMc<R>::conduct(g3, kc, &gt, &i0);
                const double I0 = (double)i0 + iext;
                L.row[j].a = ab1 - (double)gt;
                L.row[j].v = -(cdt * v) - I0;
                wild |= !(v > HS_HINES_VLO && v < HS_HINES_VHI && gt >= 0 && gt < (R)HS_HINES_GMAX);
            }
        }
        if (step == nsteps) break;
        const int par = step & 1;
        if (__ballot(wild) && lane == 0) L.wild[par] = 1;
        __syncthreads(); /* the rows are written */
        const bool fast = d.narrow && L.wild[par] == 0;
        if (tid == 0) L.wild[par ^ 1] = L.next[par ^ 1] = 0; /* last read before this barrier, next written after another */
        if (wave < nsolve) {
            if (solver) {
                if (fast) hs_thomas<true>(L, tid, len, rows, tid == spot, bp, bm, nc, band);
                else hs_thomas<false>(L, tid, len, rows, tid == spot, bp, bm, nc, band);
            }
            if (M > 1 && met > 1) {
                if (wave < met && lane == 0) {
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                    __hip_atomic_fetch_add(L.met, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
                if (wave == 0) { /* every one of these waves arrives once a step */
                    while (__hip_atomic_load(L.met, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < met * (step + 1))
                        __builtin_amdgcn_s_sleep(1);
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                }
            } else {
                hs_wave_fence();
            }
            if (wave == 0) hs_couple<M>(L, N, nn, nlev, lane);
        }
        /* the gates, by whoever is free */
        for (;;) {
            int q = 0;
            if (lane == 0) q = atomicAdd(&L.next[par], 1);
            const int j = __builtin_amdgcn_readfirstlane(q) * HS_WAVE + lane;
            if (j - lane >= nc) break;
            if (j < nc) {
                R g3[3] = {C.m[j], C.n[j], C.h[j]};
                const R v = (R)L.V[j];
                if (fast) HsMc<R>::template gates<true>(v, g3, kc[6]);
                else HsMc<R>::template gates<false>(v, g3, kc[6]);
                C.m[j] = g3[0];
                C.n[j] = g3[1];
                C.h[j] = g3[2];
            }
        }
        __syncthreads(); /* the solution and the gates are written */
    }
    __syncthreads(); /* the potentials are written */
    for (int j = tid; j < nc; j += blockDim.x) {
        const int p = d.place[c0 + j];
        d.v[c0 + j] = L.V[p];
        d.m[c0 + j] = C.m[p];
        d.n[c0 + j] = C.n[p];
        d.h[c0 + j] = C.h[p];
    }
    if (spikes) d.spikes[tree] += spikes;
}

/* ------------------------------------------------------------------------ */
/* host side                                                                 */
/* ------------------------------------------------------------------------ */
#define HS_HIP(call)                                                                                        \
    do {                                                                                                    \
        hipError_t _e = (call);                                                                             \
        if (_e != hipSuccess)                                                                               \
            return hs_rt_fail(HS_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(_e), __FILE__, \
                              __LINE__);                                                                    \
    } while (0)

struct hs_hines {
    int prec;
    double dt;
    int ntrees, ncomp, nsec, nnode, cmax, smax;
    std::vector<void *> allocs;
    HinesDesc<double> d64;
    HinesDesc<float> d32;
    long long steps_per_launch = 1000;
    int64_t steps = 0;
    std::unique_ptr<int32_t[]> place; /* where each compartment's constants are, from its tree's first */
    std::vector<int32_t> tree_comp;
    std::vector<double> area, I; /* host copies: the point current is stored as I / area */
    double last_wall = 0, last_gpu_ms = 0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
};

static int hs_h_alloc(hs_hines *H, size_t bytes, void **p)
{
    if (hipMalloc(p, bytes ? bytes : 1) != hipSuccess) {
        (void)hipGetLastError();
        return hs_rt_fail(HS_ERR_NOMEM, "hipMalloc(%zu) failed", bytes);
    }
    H->allocs.push_back(*p);
    return HS_OK;
}

template <typename T>
static int hs_h_upload(hs_hines *H, const T *host, size_t n, const T **dev)
{
    void *p = nullptr;
    int r = hs_h_alloc(H, sizeof(T) * n, &p);
    if (r != HS_OK) return r;
    if (n) HS_HIP(hipMemcpyAsync(p, host, sizeof(T) * n, hipMemcpyHostToDevice, hs_rt_stream()));
    *dev = (const T *)p;
    return HS_OK;
}

/* small tables, which go to the device together: an allocation and a copy of their
   own take 20 us each */
struct HinesPack {
    std::vector<char> host;
    std::vector<std::pair<const void **, size_t>> at;
};

template <typename T>
static int hs_h_upload(hs_hines *H, HinesPack &pack, const std::vector<T> &host, const T **dev)
{
    const size_t bytes = sizeof(T) * host.size(), o = (pack.host.size() + 255) & ~(size_t)255;
    if (bytes > 65536) return hs_h_upload(H, host.data(), host.size(), dev);
    pack.host.resize(o + std::max<size_t>(bytes, 1));
    if (bytes) memcpy(pack.host.data() + o, host.data(), bytes);
    pack.at.push_back({(const void **)dev, o});
    return HS_OK;
}

static int hs_h_upload(hs_hines *H, const HinesPack &pack)
{
    if (pack.at.empty()) return HS_OK;
    const char *dev = nullptr;
    const int r = hs_h_upload(H, pack.host.data(), pack.host.size(), &dev);
    for (const auto &x : pack.at) *x.first = dev + x.second;
    return r;
}

/* constants that keep the short divisions away from the ends of the exponent range:
   zero or of ordinary size */
static bool hs_h_ordinary(const double *x, size_t n)
{
    bool ok = true;
    for (size_t i = 0; i < n; ++i) {
        const double m = x[i] < 0 ? -x[i] : x[i];
        ok &= (m == 0.0) | ((m > 1e-40) & (m < 1e40));
    }
    return ok;
}

/* the pointer and size fields shared by the double and float descriptors */
template <typename R>
static void hs_h_copy_common(HinesDesc<R> &o, const HinesDesc<double> &d)
{
    o.tree_comp = d.tree_comp;
    o.tree_sec = d.tree_sec;
    o.order = d.order;
    o.row = d.row;
    o.v = d.v;
    o.place = d.place;
    o.band = d.band;
    o.ab1 = d.ab1;
    o.tree_row = d.tree_row;
    o.off = d.off;
    o.len = d.len;
    o.cdt = d.cdt;
    o.iext = d.iext;
    o.ends = d.ends;
    o.first = d.first;
    o.last = d.last;
    o.mparent = d.mparent;
    o.invr0 = d.invr0;
    o.invrn = d.invrn;
    o.bplus = d.bplus;
    o.bminus = d.bminus;
    o.nchild = d.nchild;
    o.child = d.child;
    o.level = d.level;
    o.nlevels = d.nlevels;
    o.spikes = d.spikes;
    o.vth = d.vth;
    o.cmax = d.cmax;
    o.smax = d.smax;
    o.rmax = d.rmax;
    o.narrow = d.narrow;
}

extern "C" void hs_hines_destroy(hs_hines *H)
{
    if (!H) return;
    (void)hipStreamSynchronize(hs_rt_stream());
    for (void *p : H->allocs) (void)hipFree(p);
    if (H->e0) (void)hipEventDestroy(H->e0);
    if (H->e1) (void)hipEventDestroy(H->e1);
    delete H;
}

/* which tree a workgroup takes: by size, largest first, every other round of `row`
   workgroups the other way round, so that the trees that share a compute unit add
   up to about the same work on each */
static std::vector<int32_t> hs_h_order(const int32_t *tree_comp, int n, int row)
{
    std::vector<int32_t> o((size_t)n);
    for (int t = 0; t < n; ++t) o[t] = t;
    std::stable_sort(o.begin(), o.end(), [&](int a, int b) {
        return tree_comp[a + 1] - tree_comp[a] > tree_comp[b + 1] - tree_comp[b];
    });
    for (int r = row; r < n; r += 2 * row) std::reverse(o.begin() + r, o.begin() + std::min(n, r + row));
    return o;
}

/* where the compartments of a tree are kept: sections by rank, longest first, the
   first compartment of each, then the second of each that has one, ...: the lanes of
   the Thomas sweep, one per section in the order of rank, then read and write
   neighbouring words.  In the order of the sections, a row was 64 cache lines and
   several LDS words to a bank */
static void hs_h_place(int ns, const int32_t *size, int nc, int32_t *place, int32_t *first, int32_t *last, int32_t *len,
                       std::vector<int32_t> *off)
{
    int live[HS_HINES_MAXC + 1], rank[HS_HINES_MAXC + 1]; /* sections with a q-th compartment; the next of a size */
    const int rows = *std::max_element(size, size + ns);
    std::fill(live, live + rows, 0);
    for (int s = 0; s < ns; ++s) ++live[size[s] - 1];
    for (int q = rows - 2; q >= 0; --q) live[q] += live[q + 1];
    const size_t o = off->size();
    off->resize(o + rows + 2 * HS_HINES_PF + 2, nc);
    int32_t *const row = off->data() + o;
    row[0] = 0;
    for (int q = 1; q < rows; ++q) row[q] = row[q - 1] + live[q - 1];
    for (int z = 1; z <= rows; ++z) rank[z] = z < rows ? live[z] : 0; /* the longer ones come first */
    for (int s = 0, at = 0; s < ns; at += size[s++]) {
        const int r = rank[size[s]]++;
        len[r] = size[s];
        for (int q = 0; q < size[s]; ++q) place[at + q] = row[q] + r;
        first[s] = r;
        last[s] = row[size[s] - 1] + r;
    }
}

/* a variable of all compartments to the device, and back */
static int hs_h_put(hs_hines *H, void *var, const void *host, size_t real)
{
    HS_HIP(hipMemcpyAsync(var, host, real * H->ncomp, hipMemcpyHostToDevice, hs_rt_stream()));
    HS_HIP(hipStreamSynchronize(hs_rt_stream()));
    return HS_OK;
}

static int hs_h_take(hs_hines *H, const void *var, void *host, size_t real)
{
    HS_HIP(hipMemcpyAsync(host, var, real * H->ncomp, hipMemcpyDeviceToHost, hs_rt_stream()));
    HS_HIP(hipStreamSynchronize(hs_rt_stream()));
    return HS_OK;
}

/* dynamic LDS of a workgroup (HinesLds) */
static size_t hs_h_lds(int CM, int SM, int RM, size_t real, bool inlds)
{
    return sizeof(double) * (5 * (size_t)CM + 3 * (SM + 1)) + sizeof(int) * ((size_t)RM + 6) +
           (inlds ? 8 + (size_t)CM * (3 * sizeof(double) + 3 * real + sizeof(int32_t)) : 0);
}

/* waves of a tree: 16 per compute unit over its trees, at least one besides the
   solvers, at most one besides them per 64 compartments; everything in LDS where all
   of a compute unit's trees still fit */
template <typename R> static int hs_h_waves(const HinesDesc<R> &d, int ntrees, bool *inlds)
{
    const int solvers = hs_hines_solvers(d.smax), most = solvers + (d.cmax + HS_WAVE - 1) / HS_WAVE;
    const int trees = (ntrees + hs_rt_cus() - 1) / hs_rt_cus();
    const int waves = std::min(std::min(most, 16), std::max(solvers + 1, 16 / trees));
    *inlds = hs_h_lds(d.cmax, d.smax, d.rmax, sizeof(R), true) * std::min(trees, 16 / waves) <= 160 * 1024;
    return waves;
}

extern "C" int hs_hines_create(int precision, double dt, int n_trees, const int32_t *tree_comp,
                               const int32_t *tree_sec, const int32_t *sec_first, const int32_t *sec_n,
                               const int32_t *sec_parent, const double *area, const double *rl1, const double *rl2,
                               const double *Cm, double Ri, const double *chan, double v_spike, hs_hines **out)
{
    int r = hs_rt_need_init();
    if (r != HS_OK) return r;
    if (!out || n_trees <= 0 || (precision != HS_F64 && precision != HS_F32) || !(dt > 0) || !tree_comp ||
        !tree_sec || !sec_first || !sec_n || !sec_parent || !area || !rl1 || !rl2 || !Cm || !chan)
        return hs_rt_fail(HS_ERR_ARG, "hs_hines_create: bad arguments");
    const int NC = tree_comp[n_trees], NS = tree_sec[n_trees];
    /* validate the morphology and derive the tables of the reference's prep */
    double iv[HS_HINES_MAXC], a0[HS_HINES_MAXC], a1[HS_HINES_MAXC], a2[HS_HINES_MAXC]; /* of one tree */
    /* in the order of hs_h_place */
    std::unique_ptr<double[]> pab1(new double[NC]), pcdt(new double[NC]);
    std::unique_ptr<double2[]> band(new double2[NC]);
    std::unique_ptr<int32_t[]> ends(new int32_t[NC]), place(new int32_t[NC]);
    bool narrow = dt <= HS_HINES_DTMAX && hs_h_ordinary(chan, 6); /* the short divisions */
    std::vector<double> invr0(NS), invrn(NS), bplus(NS), bminus(NS); /* the last two by rank */
    std::vector<int32_t> first(NS), endc(NS), mparent(NS);
    std::vector<int32_t> pfirst(NS), plast(NS), len(NS), off, tree_row(1, 0);
    std::vector<int32_t> nchild(NS + n_trees, 0), child((size_t)(NS + n_trees) * HS_HINES_RL, 0);
    std::vector<int32_t> level(NS + n_trees), nlev(n_trees);
    int cmax = 1, smax = 1, rmax = 1;
    for (int t = 0; t < n_trees; ++t) {
        const int c0 = tree_comp[t], N = tree_comp[t + 1] - c0;
        const int s0 = tree_sec[t], ns = tree_sec[t + 1] - s0;
        const int n0 = s0 + t;
        if (N <= 0 || ns <= 0 || N > HS_HINES_MAXC || ns > HS_HINES_MAXS)
            return hs_rt_fail(HS_ERR_UNSUPPORTED, "tree %d: %d compartments / %d sections (limits %d / %d)", t, N,
                              ns, HS_HINES_MAXC, HS_HINES_MAXS);
        cmax = std::max(cmax, N);
        smax = std::max(smax, ns);
        int expect = 0;
        std::vector<int> depth(ns + 1, 0);
        for (int s = 0; s < ns; ++s) {
            const int p = sec_parent[s0 + s];
            if (sec_first[s0 + s] != expect || sec_n[s0 + s] <= 0 || (s == 0) != (p < 0) || p >= s)
                return hs_rt_fail(HS_ERR_ARG, "tree %d section %d: sections must be depth-first, contiguous", t, s);
            expect += sec_n[s0 + s];
            first[s0 + s] = sec_first[s0 + s];
            endc[s0 + s] = sec_first[s0 + s] + sec_n[s0 + s];
            const int mp = p < 0 ? 0 : p + 1;
            mparent[s0 + s] = mp;
            if (nchild[n0 + mp] >= HS_HINES_RL)
                return hs_rt_fail(HS_ERR_UNSUPPORTED, "tree %d: more than %d children at a branch point", t,
                                  HS_HINES_RL);
            child[(size_t)(n0 + mp) * HS_HINES_RL + nchild[n0 + mp]++] = s + 1;
            depth[s + 1] = depth[mp] + 1;
        }
        if (expect != N) return hs_rt_fail(HS_ERR_ARG, "tree %d: sections cover %d of %d compartments", t, expect, N);
        /* nodes by depth */
        int maxd = 0;
        for (int k = 0; k <= ns; ++k) maxd = std::max(maxd, depth[k]);
        for (int k = 0; k <= ns; ++k) level[n0 + k] = depth[k];
        nlev[t] = maxd + 1;
        hs_h_place(ns, sec_n + s0, N, place.get() + c0, pfirst.data() + s0, plast.data() + s0, len.data() + s0, &off);
        tree_row.push_back((int32_t)off.size());
        rmax = std::max(rmax, tree_row[t + 1] - tree_row[t]);
        /* spatialstateupdate.cu:39-83, tree-local indices, same operation order */
        const double *ar = area + c0, *r1 = rl1 + c0, *r2 = rl2 + c0, *cm = Cm + c0;
        for (int i = 1; i < N; i++) iv[i] = 1.0 / (Ri * (1 / r2[i - 1] + 1 / r1[i]));
        for (int s = 0; s < ns; s++) iv[first[s0 + s]] = 0; /* (the first section's is compartment 0) */
        a0[0] = a2[N - 1] = 0.0;
        for (int i = 0; i < N; i++) a1[i] = (-(cm[i] / dt) - iv[i] / ar[i]);
        for (int i = 1; i < N; i++) {
            a0[i] = iv[i] / ar[i - 1];
            a2[i - 1] = iv[i] / ar[i];
            a1[i - 1] -= iv[i] / ar[i - 1];
        }
        for (int s = 0; s < ns; s++) {
            const int f = first[s0 + s], l = endc[s0 + s] - 1;
            const double i0 = r1[f] / Ri, in = r2[l] / Ri;
            invr0[s0 + s] = i0;
            invrn[s0 + s] = in;
            a1[f] -= (i0 / ar[f]);
            a1[l] -= (in / ar[l]);
            bplus[s0 + pfirst[s0 + s]] = -(in / ar[l]);
            bminus[s0 + pfirst[s0 + s]] = -(i0 / ar[f]);
            for (int i = f; i <= l; ++i) ends[c0 + place[c0 + i]] = mparent[s0 + s] | (s + 1) << 8;
        }
        for (int i = 0; i < N; i++) {
            const int p = c0 + place[c0 + i];
            pcdt[p] = cm[i] / dt;
            pab1[p] = a1[i];
            band[p] = make_double2(i < N - 1 ? a0[i + 1] : 0.0, i > 0 ? a2[i - 1] : 0.0);
        }
        narrow = narrow && hs_h_ordinary(a0, N) && hs_h_ordinary(a1, N) && hs_h_ordinary(a2, N) &&
                 hs_h_ordinary(pcdt.get() + c0, N);
    }
    hs_hines *H = new hs_hines();
    H->prec = precision;
    H->dt = dt;
    H->ntrees = n_trees;
    H->ncomp = NC;
    H->nsec = NS;
    H->nnode = NS + n_trees;
    H->cmax = cmax;
    H->smax = smax;
    HinesDesc<double> d;
    memset(&d, 0, sizeof(d));
    int rr = HS_OK;
    HinesPack pack;
#define UP(vec, field)                                    \
    if (rr == HS_OK) rr = hs_h_upload(H, pack, vec, &d.field);
    std::vector<int32_t> tc(tree_comp, tree_comp + n_trees + 1), ts(tree_sec, tree_sec + n_trees + 1);
    const int row = std::max(1, hs_rt_cus());
    std::vector<int32_t> order = hs_h_order(tree_comp, n_trees, row);
    d.row = row;
    UP(order, order)
#define UPC(arr, field)                                            \
    if (rr == HS_OK) rr = hs_h_upload(H, arr.get(), (size_t)NC, &d.field);
    UP(tc, tree_comp) UP(ts, tree_sec) UPC(band, band) UPC(pab1, ab1) UPC(pcdt, cdt) UPC(ends, ends) UPC(place, place)
    UP(tree_row, tree_row) UP(off, off) UP(len, len) UP(pfirst, first) UP(plast, last) UP(mparent, mparent) UP(invr0, invr0) UP(invrn, invrn) UP(bplus, bplus)
    UP(bminus, bminus) UP(nchild, nchild) UP(child, child) UP(level, level) UP(nlev, nlevels)
#undef UPC
#undef UP
    if (rr == HS_OK) rr = hs_h_upload(H, pack);
    d.cmax = cmax;
    d.smax = smax;
    d.rmax = rmax;
    bool inlds;
    if (precision == HS_F64) {
        (void)hs_h_waves<double>(d, n_trees, &inlds);
    } else {
        hs_h_copy_common(H->d32, d);
        (void)hs_h_waves<float>(H->d32, n_trees, &inlds);
    }
    void *pi = nullptr, *pw[3] = {nullptr, nullptr, nullptr};
    void *pv = nullptr, *pm = nullptr, *pn = nullptr, *ph = nullptr, *ps = nullptr;
    const size_t rs = precision == HS_F64 ? sizeof(double) : sizeof(float);
    if (rr == HS_OK) rr = hs_h_alloc(H, sizeof(double) * NC, &pi);
    for (int q = 0; q < 3; ++q)
        if (rr == HS_OK && !inlds) rr = hs_h_alloc(H, rs * NC, &pw[q]);
    if (rr == HS_OK) rr = hs_h_alloc(H, sizeof(double) * NC, &pv);
    if (rr == HS_OK) rr = hs_h_alloc(H, rs * NC, &pm);
    if (rr == HS_OK) rr = hs_h_alloc(H, rs * NC, &pn);
    if (rr == HS_OK) rr = hs_h_alloc(H, rs * NC, &ph);
    if (rr == HS_OK) rr = hs_h_alloc(H, sizeof(int32_t) * n_trees, &ps);
    if (rr != HS_OK) {
        hs_hines_destroy(H);
        return rr;
    }
    hipStream_t st = hs_rt_stream();
    if (hipMemsetAsync(pv, 0, sizeof(double) * NC, st) != hipSuccess ||
        hipMemsetAsync(pi, 0, sizeof(double) * NC, st) != hipSuccess ||
        hipMemsetAsync(pm, 0, rs * NC, st) != hipSuccess || hipMemsetAsync(pn, 0, rs * NC, st) != hipSuccess ||
        hipMemsetAsync(ph, 0, rs * NC, st) != hipSuccess ||
        hipMemsetAsync(ps, 0, sizeof(int32_t) * n_trees, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess) {
        hs_hines_destroy(H);
        return hs_rt_fail(HS_ERR_HIP, "hs_hines_create: initialising device arrays failed");
    }
    d.v = (double *)pv;
    d.iext = (const double *)pi;
    d.spikes = (int32_t *)ps;
    d.vth = v_spike;
    d.narrow = narrow && hs_h_ordinary(invr0.data(), NS) && hs_h_ordinary(invrn.data(), NS) &&
               hs_h_ordinary(bplus.data(), NS) && hs_h_ordinary(bminus.data(), NS);
    H->d64 = d;
    hs_h_copy_common(H->d32, d);
    H->area.assign(area, area + NC);
    H->I.assign(NC, 0.0);
    H->place = std::move(place);
    H->tree_comp.assign(tree_comp, tree_comp + n_trees + 1);
    H->d64.wm = (double *)pw[0];
    H->d64.wn = (double *)pw[1];
    H->d64.wh = (double *)pw[2];
    H->d32.wm = (float *)pw[0];
    H->d32.wn = (float *)pw[1];
    H->d32.wh = (float *)pw[2];
    H->d64.m = (double *)pm;
    H->d64.n = (double *)pn;
    H->d64.h = (double *)ph;
    H->d32.m = (float *)pm;
    H->d32.n = (float *)pn;
    H->d32.h = (float *)ph;
    for (int q = 0; q < 6; ++q) {
        H->d64.chan[q] = chan[q];
        H->d32.chan[q] = (float)chan[q];
    }
    H->d64.chan[6] = dt;
    H->d32.chan[6] = (float)dt;
    if (hipEventCreate(&H->e0) != hipSuccess || hipEventCreate(&H->e1) != hipSuccess) {
        hs_hines_destroy(H);
        return hs_rt_fail(HS_ERR_HIP, "hipEventCreate failed");
    }
    *out = H;
    return HS_OK;
}

static int hs_h_var(hs_hines *H, int var, void **p, bool *gate)
{
    *gate = var >= 1 && var <= 3;
    switch (var) {
    case 0: *p = H->d64.v; return HS_OK;
    case 1: *p = H->d64.m; return HS_OK;
    case 2: *p = H->d64.n; return HS_OK;
    case 3: *p = H->d64.h; return HS_OK;
    case 4: *p = (void *)H->d64.iext; return HS_OK;
    default: return hs_rt_fail(HS_ERR_ARG, "bad variable %d", var);
    }
}

extern "C" int hs_hines_set_state(hs_hines *H, int var, const double *values)
{
    if (!H || !values) return hs_rt_fail(HS_ERR_ARG, "null argument");
    void *p;
    bool gate;
    int r = hs_h_var(H, var, &p, &gate);
    if (r != HS_OK) return r;
    if (var == 4) {
        /* a point current enters the membrane equation as the density I / area */
        std::vector<double> ia(H->ncomp);
        for (int t = 0; t < H->ntrees; ++t)
            for (int c0 = H->tree_comp[t], i = c0; i < H->tree_comp[t + 1]; ++i) {
                H->I[i] = values[i];
                ia[c0 + H->place[i]] = values[i] / H->area[i];
            }
        return hs_h_put(H, p, ia.data(), sizeof(double));
    }
    if (gate && H->prec == HS_F32) {
        std::vector<float> f(H->ncomp);
        for (int i = 0; i < H->ncomp; ++i) f[i] = (float)values[i];
        return hs_h_put(H, p, f.data(), sizeof(float));
    }
    return hs_h_put(H, p, values, sizeof(double));
}

extern "C" int hs_hines_get_state(hs_hines *H, int var, double *values)
{
    if (!H || !values) return hs_rt_fail(HS_ERR_ARG, "null argument");
    void *p;
    bool gate;
    int r = hs_h_var(H, var, &p, &gate);
    if (r != HS_OK) return r;
    if (var == 4) {
        memcpy(values, H->I.data(), sizeof(double) * H->ncomp);
        return HS_OK;
    }
    if (gate && H->prec == HS_F32) {
        std::vector<float> f(H->ncomp);
        r = hs_h_take(H, p, f.data(), sizeof(float));
        for (int i = 0; i < H->ncomp; ++i) values[i] = f[i];
        return r;
    }
    return hs_h_take(H, p, values, sizeof(double));
}

extern "C" int hs_hines_set_option(hs_hines *H, int key, long long value)
{
    if (!H || key != 0 || value < 1 || value > (1 << 24)) return hs_rt_fail(HS_ERR_ARG, "bad option");
    H->steps_per_launch = value;
    return HS_OK;
}

template <typename R>
static hipError_t hs_h_launch(const HinesDesc<R> &d, int ntrees, int k, hipStream_t s)
{
    bool inlds;
    const int waves = hs_h_waves(d, ntrees, &inlds);
    const size_t lds = hs_h_lds(d.cmax, d.smax, d.rmax, sizeof(R), inlds);
    const int nn = d.smax + 1; /* nodes per lane of the first solver: 1, 2 or 4 */
    const void *f = inlds ? (nn <= HS_WAVE       ? (const void *)hs_k_hines<R, 1, true>
                             : nn <= 2 * HS_WAVE ? (const void *)hs_k_hines<R, 2, true>
                                                 : (const void *)hs_k_hines<R, 4, true>)
                          : (nn <= HS_WAVE       ? (const void *)hs_k_hines<R, 1, false>
                             : nn <= 2 * HS_WAVE ? (const void *)hs_k_hines<R, 2, false>
                                                 : (const void *)hs_k_hines<R, 4, false>);
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    HinesDesc<R> dd = d;
    void *args[] = {&dd, &k};
    return hipLaunchKernel(f, dim3(ntrees), dim3(waves * HS_WAVE), args, lds, s);
}

extern "C" int hs_hines_run(hs_hines *H, int64_t nsteps)
{
    if (!H || nsteps < 0) return hs_rt_fail(HS_ERR_ARG, "bad arguments");
    const int CM = H->cmax;
    const size_t lds = hs_h_lds(CM, H->smax, H->d64.rmax, sizeof(double), false);
    if (lds > 160 * 1024) return hs_rt_fail(HS_ERR_UNSUPPORTED, "tree too large for LDS (%zu bytes)", lds);
    hipStream_t st = hs_rt_stream();
    auto t0 = std::chrono::steady_clock::now();
    HS_HIP(hipEventRecord(H->e0, st));
    for (int64_t done = 0; done < nsteps;) {
        const int k = (int)std::min<int64_t>(H->steps_per_launch, nsteps - done);
        if (H->prec == HS_F64) HS_HIP(hs_h_launch<double>(H->d64, H->ntrees, k, st));
        else HS_HIP(hs_h_launch<float>(H->d32, H->ntrees, k, st));
        done += k;
    }
    HS_HIP(hipEventRecord(H->e1, st));
    HS_HIP(hipStreamSynchronize(st));
    auto t1 = std::chrono::steady_clock::now();
    float ms = 0;
    HS_HIP(hipEventElapsedTime(&ms, H->e0, H->e1));
    H->last_gpu_ms = ms;
    H->last_wall = std::chrono::duration<double>(t1 - t0).count();
    H->steps += nsteps;
    return HS_OK;
}

extern "C" int hs_hines_spike_counts(hs_hines *H, int32_t *counts)
{
    if (!H || !counts) return hs_rt_fail(HS_ERR_ARG, "null argument");
    hipStream_t st = hs_rt_stream();
    HS_HIP(hipMemcpyAsync(counts, H->d64.spikes, sizeof(int32_t) * H->ntrees, hipMemcpyDeviceToHost, st));
    HS_HIP(hipStreamSynchronize(st));
    return HS_OK;
}

extern "C" int hs_hines_stats(hs_hines *H, double *wall_s, double *gpu_ms, int64_t *steps)
{
    if (!H) return hs_rt_fail(HS_ERR_ARG, "null argument");
    if (wall_s) *wall_s = H->last_wall;
    if (gpu_ms) *gpu_ms = H->last_gpu_ms;
    if (steps) *steps = H->steps;
    return HS_OK;
}
