/*
 * hs_resident.hip -- the resident step loop's launches: the (source, owning
 * block) layout of a network's synapses, the loop itself (hs_resident.h), and
 * what a run leaves behind for the launches after it.
 */
#include "hs_resident.h"

/*
 * Layout of the synapses by (source, owning block), one wave per source row.
 * WRITE false: entries per segment into cnt[row*nb + q].  WRITE true: the
 * entries, from the segment starts off[] (order within a segment is free: its
 * entries are summed).  Two passes over the bundle table, HBM-bound: 1e8
 * synapses in 256 blocks take about 1.5 ms with the prefix sum between them.
 */
#define HS_RES_LW 4 /* rows (waves) per block */
template <typename R, bool WRITE>
__global__ __launch_bounds__(HS_RES_LW *HS_WAVE) void hs_k_res_layout(const DPath<R> *__restrict__ paths, int np,
                                                                      const HsResArgs<R> a, int32_t *cnt,
                                                                      unsigned long long *nonempty)
{
    unsigned long long some = 0;
    __shared__ int seg[HS_RES_LW][256];
    int *h = seg[threadIdx.x / HS_WAVE];
    const int lane = hs_lane();
    const int nw = gridDim.x * HS_RES_LW;
    for (int row = blockIdx.x * HS_RES_LW + threadIdx.x / HS_WAVE; row < a.n; row += nw) {
        /* the counters belong to this wave alone; its LDS accesses complete in order */
        for (int q = lane; q < a.nb; q += HS_WAVE) h[q] = WRITE ? a.off[(long long)row * a.nb + q] : 0;
        __builtin_amdgcn_wave_barrier();
        for (int pi = 0; pi < np; ++pi) {
            const DPath<R> &p = paths[pi];
            const int32_t *bs = p.bstart + (long long)row * p.D;
            const int s0 = hs_ld(bs), s1 = hs_ld(bs + p.D);
            for (int s = s0 + lane; s < s1; s += HS_WAVE) {
                const int tg = hs_ld(p.post + s);
                const int q = tg / a.nown;
                if (!WRITE) {
                    atomicAdd(&h[q], 1);
                    continue;
                }
                int lo = 0, hi = p.D; /* the synapse's delay slot: bs[lo] <= s < bs[lo + 1] */
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (hs_ld(bs + mid) <= s) lo = mid;
                    else hi = mid;
                }
                const int at = atomicAdd(&h[q], 1);
                HsResSyn<R> x;
                x.pack = (uint32_t)(tg - q * a.nown) | (uint32_t)a.plane[p.var] << 10 | (uint32_t)(p.dmin + lo) << 16;
                x.w = p.wmode == HS_W_SCALAR ? p.wscalar : p.wmode == HS_W_SYNAPSE ? hs_ld(p.w + s) : hs_ld(p.w + row);
                if constexpr (sizeof(R) == 8) x.pad = 0;
                const_cast<HsResSyn<R> *>(a.syn)[at] = x;
            }
        }
        __builtin_amdgcn_wave_barrier();
        if (!WRITE)
            for (int q = lane; q < a.nb; q += HS_WAVE) {
                cnt[(long long)row * a.nb + q] = h[q];
                some += h[q] != 0;
            }
        __builtin_amdgcn_wave_barrier();
    }
    if (!WRITE) {
        some = hs_wave_sum(some);
        if (lane == 0 && some) hs_atomic_add(nonempty, some);
    }
}

/*
 * After the loop: the spike lists of its last dmax steps (what the next launch
 * replays, and the per-step forms read) from the blocks' lines, one step per block;
 * the last block empties the other ring slots, advances the step base and writes the
 * run's totals to host memory.
 */
template <typename R>
__global__ __launch_bounds__(256) void hs_k_res_close(const HsResArgs<R> a, const DGroup<R> *__restrict__ gp, int rows,
                                                      long long T0, uint32_t win0, HsResInfo *info)
{
    const DGroup<R> &g = *gp;
    const long long rowlen = (long long)g.nsub * g.subcap, Tend = T0 + a.ctl->ran;
    if ((int)blockIdx.x < rows) {
        __shared__ int cnt[32];
        const long long t = Tend - 1 - blockIdx.x;
        if (t < T0) return; /* the launch ran fewer steps than planned: a list of before */
        const int slot = (int)hs_mod(t, g.Q);
        if (threadIdx.x < 32) cnt[threadIdx.x] = 0;
        __syncthreads();
        const uint32_t win = win0 + (uint32_t)((t - T0) / a.W);
        const unsigned int j = (unsigned int)((t - T0) % a.W); /* step of the window */
        for (int q = threadIdx.x; q < a.nb; q += blockDim.x) {
            const unsigned long long *const ln = hs_res_lines(&a, win) + (size_t)q * a.mwords;
            const unsigned long long h = hs_ld(ln);
            const bool many = (h & 0x1fffu) == HS_RES_MANY;
            const int n = many ? (int)(h >> 13) & 0x1fff : 4 * a.hwords;
            for (int k = 0; k < n; ++k) {
                const uint32_t x = many ? (uint32_t)(hs_ld(ln + a.hwords + k / 2) >> (16 * (k & 1))) & 0xffffu
                                        : ((uint32_t)(hs_ld(ln + k / 4) >> (13 * (k & 3))) & 0x1fffu) - 1u;
                if ((x >> 9) != j) continue; /* (or no spike) */
                const int i = q * a.nown + (int)(x & 511u);
                const int sub = (i >> 8) & (g.nsub - 1);
                const int at = atomicAdd(&cnt[sub], 1);
                hs_st(g.hist + slot * rowlen + (long long)sub * g.subcap + at, (int32_t)i);
            }
        }
        __syncthreads();
        if ((int)threadIdx.x < g.nsub) hs_st(g.hist_cnt + ((long long)slot * g.nsub + threadIdx.x) * HS_CNT_STRIDE, cnt[threadIdx.x]);
        return;
    }
    for (int q = threadIdx.x; q < (g.Q - a.dmax) * g.nsub; q += blockDim.x)
        hs_st(g.hist_cnt + ((long long)hs_mod(Tend + q / g.nsub, g.Q) * g.nsub + q % g.nsub) * HS_CNT_STRIDE, 0);
    __shared__ unsigned long long part[2][4];
    unsigned long long ev = 0, sp = 0;
    for (int q = threadIdx.x; q < HS_EV_SLOTS; q += blockDim.x) {
        ev += a.ctl->ev_slot[q * HS_EV_STRIDE];
        sp += a.ctl->spk_slot[q * HS_EV_STRIDE];
    }
    ev = hs_wave_sum(ev);
    sp = hs_wave_sum(sp);
    if (hs_lane() == 0) {
        part[0][threadIdx.x / HS_WAVE] = ev;
        part[1][threadIdx.x / HS_WAVE] = sp;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a.ctl->base = Tend;
        a.ctl->no_reset_before = Tend;
        info->events = part[0][0] + part[0][1] + part[0][2] + part[0][3];
        info->spikes = part[1][0] + part[1][1] + part[1][2] + part[1][3];
        info->stalled = a.ctl->stalled;
        info->records = g.smon_n ? *g.smon_n : 0ull;
        info->base = Tend;
    }
}

/*
 * Back to the pipelined windows (mode 4) after a resident run: their accumulators
 * hold every effect due in the next window and, beyond it, those of delays < 2W
 * (the near synapses, pushed at emission).  Step base T = ctl->base; the
 * accumulators are zero on entry.
 */
template <typename R>
__global__ __launch_bounds__(256) void hs_k_res_refill(const DPath<R> *__restrict__ paths, int np, HsCtl *ctl, int W)
{
    __shared__ HsDeliverLds L;
    const long long T = ctl->base;
    const int wv = threadIdx.x / HS_WAVE, nwv = blockDim.x / HS_WAVE;
    unsigned long long ev = 0; /* counted elsewhere */
    for (int pi = 0; pi < np; ++pi) {
        const DPath<R> &p = paths[pi];
        const long long rank = (long long)blockIdx.x * nwv + wv, waves = (long long)gridDim.x * nwv;
        hs_deliver_path<R, true>(p, T, W, &L, rank, waves, &ev);
        if (p.nnear > 0) hs_deliver_path<R, true>(p, T + W, W, &L, rank, waves, &ev, 0, p.nnear);
    }
}

template <typename R>
hipError_t hs_launch_res_layout(const DPath<R> *paths, int np, const HsResArgs<R> &a, int32_t *cnt,
                                unsigned long long *nonempty, bool write, hipStream_t s)
{
    if (a.nb < 1 || a.nb > 256 || a.n < 1) return hipErrorInvalidValue;
    const int want = (a.n + HS_RES_LW - 1) / HS_RES_LW, most = 32 * hs_rt_cus();
    const int grid = want < most ? want : most;
    if (write)
        hipLaunchKernelGGL((hs_k_res_layout<R, true>), dim3(grid), dim3(HS_RES_LW * HS_WAVE), 0, s, paths, np, a, cnt,
                           nonempty);
    else
        hipLaunchKernelGGL((hs_k_res_layout<R, false>), dim3(grid), dim3(HS_RES_LW * HS_WAVE), 0, s, paths, np, a, cnt,
                           nonempty);
    return hipGetLastError();
}

#define HS_RES_ALIGN(x) (((x) + 15) & ~(size_t)15)
template <typename R>
void hs_res_offsets(HsResArgs<R> *a, int plain)
{
    size_t o = HS_RES_ALIGN(sizeof(HsResShared));
    auto take = [&](int *at, size_t bytes) {
        *at = (int)o;
        o += HS_RES_ALIGN(bytes);
    };
    const size_t nev = plain ? (size_t)a->nslots * a->cap : 0;
    take(&a->o_acc, (size_t)(plain ? 1 : a->nslots) * a->nplanes * a->nown * sizeof(R));
    take(&a->o_evw, nev * sizeof(R));
    take(&a->o_list, (size_t)a->list_cap * sizeof(uint32_t));
    take(&a->o_list2, (size_t)a->list_cap * sizeof(uint32_t));
    take(&a->o_cnt, (plain ? (size_t)a->nslots : 0) * sizeof(int));
    take(&a->o_big, (size_t)a->nb * sizeof(int));
    take(&a->o_evt, nev * sizeof(uint16_t));
    take(&a->o_stage, (size_t)a->nown * a->W * sizeof(uint16_t));
    a->lds = o > 0x7fffffff ? 0x7fffffff : (int)o;
}

template <typename R, int MS, bool PLAIN>
static hipError_t hs_resident_go(const HsResArgs<R> &a, const HsResArgs<R> *da, const DGroup<R> *g, int block,
                                 long long T0, int nsteps, uint32_t win0, hipStream_t s)
{
    const void *f = (const void *)hs_k_resident<R, MS, PLAIN>;
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, a.lds);
    if (e != hipSuccess) return e;
    void *args[] = {&da, &g, &T0, &nsteps, &win0};
    return hipLaunchCooperativeKernel(f, dim3(a.nb), dim3(block + (hs_res_helper<MS>() ? HS_RES_HELPERS : 0)), args,
                                      (unsigned int)a.lds, s);
}

__global__ void hs_k_res_first() {}

hipError_t hs_launch_res_first(hipStream_t s)
{
    void *none[] = {nullptr};
    return hipLaunchCooperativeKernel((const void *)hs_k_res_first, dim3(1), dim3(HS_WAVE), none, 0, s);
}

int hs_res_hwords(int ms) { return ms == HS_MODEL_LIF_NOISE ? 2 : 1; }

template <typename R>
hipError_t hs_launch_resident(const HsResArgs<R> &a, const HsResArgs<R> *da, const DGroup<R> *g, int ms, int plain,
                              int block, long long T0, int nsteps, uint32_t win0, hipStream_t s)
{
    if (a.nb < 1 || a.nb > 256 || a.nb > hs_rt_cus() || a.nown < 1 || a.nown > block || block > HS_RES_MAXT ||
        block % HS_WAVE || (long long)a.nb * a.nown < a.n || a.W < 1 || a.W > HS_MAX_WINDOW || a.nslots != a.dmax + 1 ||
        a.W > a.nslots || a.list_cap < 4 * a.hwords * a.nb || a.hwords != hs_res_hwords(ms) || a.lds > 160 * 1024 || nsteps < 1)
        return hipErrorInvalidValue;
#define HS_RES(M)                                                                  \
    (plain ? hs_resident_go<R, M, true>(a, da, g, block, T0, nsteps, win0, s)      \
           : hs_resident_go<R, M, false>(a, da, g, block, T0, nsteps, win0, s))
    if (ms == HS_MODEL_LIF_CUBA) return HS_RES(HS_MODEL_LIF_CUBA);
    if (ms == HS_MODEL_LIF_NOISE) return HS_RES(HS_MODEL_LIF_NOISE);
    if (ms == HS_MODEL_HH_COBA) return HS_RES(HS_MODEL_HH_COBA);
    if constexpr (sizeof(R) == 4)
        if (ms == HS_MODEL_HH_FAST) return HS_RES(HS_MODEL_HH_FAST);
#undef HS_RES
    return hipErrorInvalidValue;
}

template <typename R>
hipError_t hs_launch_res_close(const HsResArgs<R> &a, const DGroup<R> *g, long long T0, int nsteps, uint32_t win0,
                               HsResInfo *info, hipStream_t s)
{
    const int rows = a.dmax < nsteps ? a.dmax : nsteps;
    hipLaunchKernelGGL(hs_k_res_close<R>, dim3(rows + 1), dim3(256), 0, s, a, g, rows, T0, win0, info);
    return hipGetLastError();
}

template <typename R>
hipError_t hs_launch_res_refill(const DPath<R> *paths, int np, HsCtl *ctl, int W, hipStream_t s)
{
    hipLaunchKernelGGL(hs_k_res_refill<R>, dim3(hs_rt_cus()), dim3(256), 0, s, paths, np, ctl, W);
    return hipGetLastError();
}

#define HS_INSTANTIATE(R)                                                                                           \
    template void hs_res_offsets<R>(HsResArgs<R> *, int);                                                            \
    template hipError_t hs_launch_res_layout<R>(const DPath<R> *, int, const HsResArgs<R> &, int32_t *,              \
                                                unsigned long long *, bool, hipStream_t);                                                       \
    template hipError_t hs_launch_resident<R>(const HsResArgs<R> &, const HsResArgs<R> *, const DGroup<R> *, int, int, \
                                              int, long long, int, uint32_t, hipStream_t);                          \
    template hipError_t hs_launch_res_close<R>(const HsResArgs<R> &, const DGroup<R> *, long long, int, uint32_t,    \
                                               HsResInfo *, hipStream_t);                                           \
    template hipError_t hs_launch_res_refill<R>(const DPath<R> *, int, HsCtl *, int, hipStream_t);
HS_INSTANTIATE(double)
HS_INSTANTIATE(float)
