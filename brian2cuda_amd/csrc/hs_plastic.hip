/*
 * hs_plastic.hip -- spike-timing-dependent plasticity on scatter pathways: the
 * on_pre and on_post code of an STDP Synapses object, run after the step's
 * update and delivery launches (plain form: effects on the state; fused form
 * with one-step windows: effects into the accumulator of the step).
 *
 * Replaces, for these synapses, the effect kernel of the pre pathway
 * (brian2cuda/templates/synapses.cu:12-164 with synaptic_effects "synapse"
 * plus atomics on the target) and the post pathway's kernel over the synapses of
 * each spiking postsynaptic neuron (same template, launched for the post
 * pathway; synapses.cu:201-322 chooses full parallelism because the post code
 * only writes synapse variables).
 *
 * on_pre (step T): for each delay slot d, the spikes of step T - dmin - d; block
 * b takes slots b, b + grid, ...  A synapse sits in one bundle and a neuron spikes at
 * most once a step, so no two threads touch the same synapse; the target effect is a
 * hardware FP atomic (several synapses share a target).  A spike costs a chain of
 * dependent loads (count, spike, bundle, synapse, target), so beyond HS_STDP_FEW
 * spikes the threads find the bundles of 256 spikes at once, and then
 *   mean bundle up to HS_STDP_SHARE synapses: they take the synapses laid end to end,
 *     256 at a time; the effects on one target are added by one thread, in the order
 *     of the spikes, which it finds by comparing the round's targets (0.1 us a
 *     synapse);
 *   longer bundles: one after another, each by all threads (0.6 us a spike).
 * Measured, us a step of a network (update, on_pre, on_post; FP64) with a chain per
 * spike -> now, of it all synapses end to end and all bundles one after another:
 *   spikes  synapses each
 *     1.5      1           9.8 -> 10.0  (10.5, 10.6)
 *    15        1          19.6 -> 12.7  (12.9, 18.1)
 *    15        6          23.6 -> 20.8  (20.3, 22.0)
 *    15        8          23.6 -> 22.1  (23.3, 22.2)
 *   100        4         103.7 -> 49.5  (50.3, 82.9)
 *   100        8         103.9 -> 85.8  (88.8, 83.5)
 *    15     1000          81.4 -> 62.4  (1000, 68.1)
 *    10    10000           638 -> 430   (6510, 431)
 * on_post (step T): the target group's spikes of step T, block-strided; the
 * threads take that neuron's synapses (qsyn).  Launched after on_pre: Brian2
 * runs the pre pathway (order -1) before the post pathway (order +1) within the
 * synapses slot.
 * The trace and weight arithmetic is the shared expression set
 * (hs_model_body.inc: hs_stdp_decay, hs_stdp_on_pre, hs_stdp_on_post).
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hs_device.h"
#include "hs_internal.h"
#include "hs_model_exprs.h"

template <typename R> struct HsStdp;
template <> struct HsStdp<double> {
    static __device__ __forceinline__ double decay(long long n, double dt, double tau)
    {
        return hs_stdp_decay_f64(n, dt, tau);
    }
    static __device__ __forceinline__ double pre(double *w, double *a, double *b, double fa, double fb, const double *sk)
    {
        return hs_stdp_on_pre_f64(w, a, b, fa, fb, sk);
    }
    static __device__ __forceinline__ void post(double *w, double *a, double *b, double fa, double fb, const double *sk)
    {
        hs_stdp_on_post_f64(w, a, b, fa, fb, sk);
    }
};
template <> struct HsStdp<float> {
    static __device__ __forceinline__ float decay(long long n, double dt, double tau)
    {
        return hs_stdp_decay_f32(n, dt, tau);
    }
    static __device__ __forceinline__ float pre(float *w, float *a, float *b, float fa, float fb, const float *sk)
    {
        return hs_stdp_on_pre_f32(w, a, b, fa, fb, sk);
    }
    static __device__ __forceinline__ void post(float *w, float *a, float *b, float fa, float fb, const float *sk)
    {
        hs_stdp_on_post_f32(w, a, b, fa, fb, sk);
    }
};

#define HS_STDP_BLOCK 256
#define HS_STDP_FEW 2   /* spikes up to which the scans cost more than their chains: 1 us a step */
#define HS_STDP_SHARE 6 /* synapses per spike: the two forms meet between 6 and 8 */

/* exclusive prefix sum over the block; *total: of all threads.  scratch: one int per
   wave, free again after the next barrier of the caller */
__device__ __forceinline__ int hs_stdp_scan(int v, int *scratch, int *total)
{
    const int lane = hs_lane(), wave = threadIdx.x / HS_WAVE;
    int s = v;
#pragma unroll
    for (int o = 1; o < HS_WAVE; o <<= 1) {
        const int u = __shfl_up(s, o);
        if (lane >= o) s += u;
    }
    if (lane == HS_WAVE - 1) scratch[wave] = s;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < HS_STDP_BLOCK / HS_WAVE; ++w) {
        before += w < wave ? scratch[w] : 0;
        all += scratch[w];
    }
    *total = all;
    return before + s - v;
}

/* the last of HS_STDP_BLOCK ascending values that is at most x (the first is) */
__device__ __forceinline__ int hs_stdp_find(const int *at, int x)
{
    int lo = 0;
#pragma unroll
    for (int h = HS_STDP_BLOCK / 2; h > 0; h >>= 1)
        if (at[lo + h] <= x) lo += h;
    return lo;
}

/* the on_pre code of synapse q at step T; returns the effect on its target */
template <typename R>
__device__ __forceinline__ R hs_stdp_synapse(const DPath<R> &p, int q, long long T, const R *sk)
{
    const long long n = T - (long long)p.lastup[q];
    const R fa = HsStdp<R>::decay(n, p.dt, p.taupre);
    const R fb = HsStdp<R>::decay(n, p.dt, p.taupost);
    R w = p.wm[q], a = p.apre[q], b = p.apost[q];
    const R e = HsStdp<R>::pre(&w, &a, &b, fa, fb, sk);
    p.wm[q] = w;
    p.apre[q] = a;
    p.apost[q] = b;
    p.lastup[q] = (int32_t)T;
    return e;
}

/* synapses [q0, q1) of a bundle by the threads of the block */
template <typename R>
__device__ __forceinline__ void hs_stdp_bundle(const DPath<R> &p, int q0, int q1, long long T, const R *sk, R *tgt,
                                               unsigned long long *ev)
{
    for (int q = q0 + (int)threadIdx.x; q < q1; q += HS_STDP_BLOCK) {
        const int j = p.post[q];
        hs_atomic_add(tgt + j, hs_stdp_synapse(p, q, T, sk));
        ++*ev;
    }
}

template <typename R>
__global__ __launch_bounds__(HS_STDP_BLOCK) void hs_k_stdp_pre(const DPath<R> *paths, int np, HsCtl *ctl, int koff)
{
    __shared__ int s_list[HS_STDP_BLOCK], s_at[HS_STDP_BLOCK], s_from[HS_STDP_BLOCK], s_sum[2][HS_STDP_BLOCK / HS_WAVE];
    __shared__ __align__(16) int s_post[HS_STDP_BLOCK];
    __shared__ R s_eff[HS_STDP_BLOCK];
    const long long T = ctl->base + koff;
    const int tid = threadIdx.x;
    unsigned long long ev = 0;
    for (int pi = 0; pi < np; ++pi) {
        const DPath<R> &p = paths[pi];
        if (p.dmode != HS_DELIVER_PLASTIC) continue;
        R sk[5];
#pragma unroll
        for (int j = 0; j < 5; ++j) sk[j] = p.sk[j];
        /* plain form: the target state; fused form: the accumulator of step T,
           added to the state at the start of step T + 1 */
        R *tgt = p.acc ? p.acc + hs_mod(T, p.nacc) * p.n_tgt : p.target;
        for (int d = blockIdx.x; d < p.D; d += gridDim.x) {
            const long long ts = T - p.dmin - d; /* emission step of the bundles due now */
            if (ts < 0) continue;
            const long long slot = hs_mod(ts, p.Q);
            const int32_t *const hist = p.hist + slot * p.nsub * p.subcap;
            for (int sl0 = 0; sl0 < p.nsub; sl0 += HS_STDP_BLOCK) { /* the lists of the slot */
                int nspk, nsyn;
                if (p.nsub == 1) {
                    nspk = p.hist_cnt[slot * p.cstride];
                    if (nspk <= HS_STDP_FEW) {
                        for (int k = 0; k < nspk; ++k) {
                            const long long row = (long long)hist[k] * p.D + d;
                            hs_stdp_bundle(p, p.bstart[row], p.bstart[row + 1], T, sk, tgt, &ev);
                        }
                        continue;
                    }
                } else {
                    const int sl = sl0 + tid;
                    s_list[tid] = hs_stdp_scan(sl < p.nsub ? p.hist_cnt[(slot * p.nsub + sl) * p.cstride] : 0, s_sum[0], &nspk);
                    __syncthreads();
                }
                for (int k0 = 0; k0 < nspk; k0 += HS_STDP_BLOCK) { /* their spikes */
                    int from = 0, size = 0;
                    if (k0 + tid < nspk) {
                        const int l = p.nsub == 1 ? 0 : hs_stdp_find(s_list, k0 + tid), at = p.nsub == 1 ? 0 : s_list[l];
                        const long long i = hist[(long long)(sl0 + l) * p.subcap + (k0 + tid - at)];
                        from = p.bstart[i * p.D + d];
                        size = p.bstart[i * p.D + d + 1] - from;
                    }
                    s_at[tid] = hs_stdp_scan(size, s_sum[1], &nsyn);
                    s_from[tid] = from;
                    __syncthreads();
                    const int m = min(nspk - k0, HS_STDP_BLOCK);
                    if (nsyn > HS_STDP_SHARE * m) { /* a bundle after the other */
                        for (int k = 0; k < m; ++k)
                            hs_stdp_bundle(p, s_from[k], s_from[k] + (k + 1 < m ? s_at[k + 1] : nsyn) - s_at[k], T, sk, tgt,
                                           &ev);
                        __syncthreads();
                        continue;
                    }
                    for (int m0 = 0; m0 < nsyn; m0 += HS_STDP_BLOCK) { /* their synapses */
                        const int n = min(nsyn - m0, HS_STDP_BLOCK);
                        int j = -1;
                        if (tid < n) {
                            const int k = hs_stdp_find(s_at, m0 + tid), q = s_from[k] + (m0 + tid - s_at[k]);
                            j = p.post[q];
                            s_eff[tid] = hs_stdp_synapse(p, q, T, sk);
                            ev++;
                        }
                        s_post[tid] = j;
                        __syncthreads();
                        /* the first synapse of a target adds the effects of all of them */
                        bool first = tid < n;
                        for (int c = 0; c < n; c += 4) {
                            const int4 o = *(const int4 *)&s_post[c];
                            const int oc[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                            for (int u = 0; u < 4; ++u)
                                if (first && oc[u] == j) {
                                    if (c + u < tid) first = false;
                                    else hs_atomic_add(tgt + j, s_eff[c + u]);
                                }
                        }
                        if (m0 + HS_STDP_BLOCK < nsyn || k0 + HS_STDP_BLOCK < nspk || sl0 + HS_STDP_BLOCK < p.nsub)
                            __threadfence(); /* the next synapses may add to the same target from another wave */
                        __syncthreads();
                    }
                    __syncthreads();
                }
                __syncthreads();
            }
        }
    }
    ev = hs_wave_sum(ev);
    hs_flush_events(ev, ctl, (long long)blockIdx.x * (blockDim.x / HS_WAVE) + threadIdx.x / HS_WAVE);
}

template <typename R>
__global__ __launch_bounds__(256) void hs_k_stdp_post(const DPath<R> *paths, int np, HsCtl *ctl, int koff)
{
    const long long T = ctl->base + koff;
    for (int pi = 0; pi < np; ++pi) {
        const DPath<R> &p = paths[pi];
        if (p.dmode != HS_DELIVER_PLASTIC) continue;
        R sk[5];
#pragma unroll
        for (int j = 0; j < 5; ++j) sk[j] = p.sk[j];
        const long long slot = hs_mod(T, p.tQ);
        for (int sl = 0; sl < p.tnsub; ++sl) {
            const int cnt = p.thist_cnt[(slot * p.tnsub + sl) * HS_CNT_STRIDE];
            const int32_t *lst = p.thist + slot * p.tnsub * p.tsubcap + (long long)sl * p.tsubcap;
            for (int k = blockIdx.x; k < cnt; k += gridDim.x) {
                const int j = lst[k];
                const int q1 = p.qstart[j + 1];
                for (int e = p.qstart[j] + (int)threadIdx.x; e < q1; e += blockDim.x) {
                    const int q = p.qsyn[e];
                    const long long n = T - (long long)p.lastup[q];
                    const R fa = HsStdp<R>::decay(n, p.dt, p.taupre);
                    const R fb = HsStdp<R>::decay(n, p.dt, p.taupost);
                    R w = p.wm[q], a = p.apre[q], b = p.apost[q];
                    HsStdp<R>::post(&w, &a, &b, fa, fb, sk);
                    p.wm[q] = w;
                    p.apre[q] = a;
                    p.apost[q] = b;
                    p.lastup[q] = (int32_t)T;
                }
            }
        }
    }
}

template <typename R>
hipError_t hs_launch_stdp(const DPath<R> *paths, int np, HsCtl *ctl, int koff, int grid, hipStream_t s)
{
    hs_k_stdp_pre<R><<<grid, HS_STDP_BLOCK, 0, s>>>(paths, np, ctl, koff);
    hs_k_stdp_post<R><<<grid, 256, 0, s>>>(paths, np, ctl, koff);
    return hipGetLastError();
}

template hipError_t hs_launch_stdp<double>(const DPath<double> *, int, HsCtl *, int, int, hipStream_t);
template hipError_t hs_launch_stdp<float>(const DPath<float> *, int, HsCtl *, int, int, hipStream_t);

/* StateMonitor of a synapse variable (Brian2's default when='start'): at the
   start of step T, row T - t0 of buf takes src[idx[k]] for the n recorded
   synapses (positions in bundle order) */
template <typename R>
__global__ __launch_bounds__(256) void hs_k_synmon(const R *__restrict__ src, const int32_t *__restrict__ idx, int n,
                                                    R *__restrict__ buf, long long rows, long long t0, int every,
                                                    const HsCtl *ctl, int koff)
{
    const long long dt0 = ctl->base + koff - t0;
    if (dt0 < 0 || dt0 % every != 0) return;
    const long long row = dt0 / every;
    if (row >= rows) return;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x)
        buf[row * n + k] = src[idx[k]];
}

hipError_t hs_launch_synmon(int prec, const void *src, const int32_t *idx, int n, void *buf, long long rows,
                            long long t0, int every, const HsCtl *ctl, int koff, hipStream_t s)
{
    if (n <= 0 || every < 1) return hipSuccess;
    const int grid = (n + 255) / 256 > 1024 ? 1024 : (n + 255) / 256;
    if (prec == 64)
        hipLaunchKernelGGL(hs_k_synmon<double>, dim3(grid), dim3(256), 0, s, (const double *)src, idx, n,
                           (double *)buf, rows, t0, every, ctl, koff);
    else
        hipLaunchKernelGGL(hs_k_synmon<float>, dim3(grid), dim3(256), 0, s, (const float *)src, idx, n,
                           (float *)buf, rows, t0, every, ctl, koff);
    return hipGetLastError();
}
