/*
 * hs_resident.h -- the resident step loop: one launch advances a network of one
 * group by many steps, every neuron staying on the compute unit that owns it.
 *
 * What it replaces: a launch (or two) per step or window, each of which reads
 * the state back from HBM, looks its spikes up in global lists and adds every
 * synaptic effect with a global FP atomic.  Those launches are bound by latency,
 * not by bytes: an empty kernel of a graph takes 1.6 us, the chain list count ->
 * spike -> bundle bounds -> target -> atomic four memory round trips more, and
 * random FP32 atomics run at 2e10 per second chip-wide.
 *
 * Split: block b owns neurons [b*nown, (b+1)*nown), one per thread, one block
 * per compute unit at most (the grid is resident: launched cooperatively).  The
 * state stays in registers, the effects still to come in LDS:
 *   fused form: a ring of dmax + 1 step slots of one sum per target variable
 *     and neuron (the effects due at step t are added at the start of t + 1)
 *   plain form: a bucket of events per step slot (the effects of a step are
 *     added to the state one after another, as cpp_standalone does, so their
 *     sum cannot be formed ahead); a bucket that overflows is delivered from the
 *     spikes themselves instead (hs_res_walk)
 * and the synapses are laid out per (source neuron, owning block), so that a
 * block reads the few entries of a spike that are its own (2 dependent loads)
 * and adds them with LDS atomics.
 *
 * Exchange: every window of w <= dmin + 1 steps (a spike of its first step is
 * due at the earliest at its last one, which the step after adds), each block
 * publishes its spikes in a line of its own and reads everybody's.  Every
 * 8-byte word carries the window's number in its upper half and is stored and
 * loaded as one relaxed agent-scope atomic, so a word is valid by itself: no
 * fence, no counter, one memory hop.  Measured on MI355X, 256 blocks: 1.45 us
 * per exchange with the lines 128 bytes apart, 2.2 us with the headers packed,
 * 3.8 us with an arrival counter; 64 blocks 1.05 us, 32 blocks 1.0 us.  While the
 * lines travel the block draws the next window's noise.
 * A block that waits longer than HS_RES_WAIT gives up and sets ctl->stalled;
 * all others then give up as well, so the launch always ends.
 *
 * A busy network costs the loop more than the per-step forms: every block looks at
 * every spike (20 ns a spike of a window, against 50 ps an event there), lines that
 * the lists do not hold are delivered one after another, and a step whose bucket
 * overflowed takes the spikes of dmax steps.  So each block keeps the balance of
 * what its windows held beyond a->most spikes; one whose balance exceeds
 * HS_RES_SLACK windows says so in its header, and since everybody reads every
 * header of every window, all blocks end after that window.  The host goes on in
 * the per-step form (hs_res_run).
 *
 * Measured, us per step of a network that has changed over, readback included; the
 * per-step form -> the loop:
 *   CUBA 4,000 neurons, one-step delay   FP64 plain 8.3 -> 2.2, FP32 fused 5.1 -> 1.9
 *   COBAHH 4,000, no delay               FP64 plain 11.3 -> 6.1
 *   Brunel 20,011, delays 5 to 50        FP64 plain 11.2 -> 2.2
 *   Brunel 100,000, 1e8 synapses         FP32 pipelined 3.68 -> 1.88
 *   64 CUBA networks, 128,000 neurons    FP32 fused 6.9 -> 4.5
 * What bounds it now is latency: of a CUBA window of 2 steps (3.8 us) the update
 * takes 0.8, the exchange 1.5, segment bounds and entries 1.0; of a 100,000-neuron
 * Brunel window of 6 steps (10.7 us) the noise takes 3.5 and beside it the exchange
 * and the synapses' two memory hops 8.6.
 */
#ifndef HS_RESIDENT_H
#define HS_RESIDENT_H

#include "hs_device.h"

#define HS_RES_WAIT 500000000LL /* ticks of the 100 MHz wall clock: 5 s */
#define HS_RES_FEW 64           /* spikes of a line that its polling thread reads by itself */
#define HS_RES_LINE 64          /* what a line left to the whole block costs, in listed spikes (1.2 us) */
#define HS_RES_SLACK 128        /* windows of a->most spikes: 1 to 4 ms */
#define HS_RES_STOP 1
#define HS_RES_LAST 2

__device__ __forceinline__ HsResSyn<float> hs_res_ld(const HsResSyn<float> *p)
{
    const unsigned long long x = hs_ld((const unsigned long long *)p);
    return {(uint32_t)x, __uint_as_float((uint32_t)(x >> 32))};
}

__device__ __forceinline__ HsResSyn<double> hs_res_ld(const HsResSyn<double> *p)
{
    typedef unsigned int v4 __attribute__((ext_vector_type(4)));
    const v4 x = hs_ld((const v4 *)p);
    return {__longlong_as_double((long long)((unsigned long long)x.y << 32 | x.x)), x.z, 0u};
}

__device__ __forceinline__ unsigned long long hs_mail_ld(const unsigned long long *p)
{
    return __hip_atomic_load((const HS_GLOBAL unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void hs_mail_st(unsigned long long *p, unsigned long long v)
{
    __hip_atomic_store((HS_GLOBAL unsigned long long *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* a descriptor pointer whose loads stay where they are written: fields that only
   a rare branch reads do not occupy registers in the loop around it */
template <typename T>
__device__ __forceinline__ const T *hs_here(const T *p)
{
    asm volatile("" : "+s"(p));
    return p;
}

/* the block's LDS: scalars first, then the arrays at the offsets of HsResArgs */
struct HsResShared {
    int nspk[2]; /* this block's spikes of the window and (being emptied) of the next */
    int n1, n2;  /* spikes to deliver: from header words, from lines with more */
    int nbig;
    int stop; /* HS_RES_STOP: waited in vain; HS_RES_LAST: a header asked for the end of the launch */
    int replayed; /* spikes of a walk that came from the lists of the launches before */
    int met; /* arrivals of helper waves (hs_res_meet) */
    int wsum[(HS_RES_MAXT + HS_RES_HELPERS) / HS_WAVE];
};

template <typename R>
struct HsResLds {
    HsResShared *S;
    R *acc;          /* fused: [nslots][nplanes][nown]; plain: target variables [nplanes][nown] */
    R *evw;          /* plain: event weights [nslots][cap] */
    uint32_t *list;  /* spikes being delivered: source | step offset << 20; n1 of them here */
    uint32_t *list2; /* and n2 here */
    int *cnt;        /* plain: events of a slot (more than cap: overflow) */
    int *big;        /* lines left for the whole block */
    uint16_t *evt;   /* plain: event targets, plane << 10 | index */
    uint16_t *stage; /* this block's spikes of the window: step offset << 9 | index */
};

extern __shared__ __align__(16) char hs_res_smem[];

template <typename R>
__device__ __forceinline__ HsResLds<R> hs_res_lds(const HsResArgs<R> *__restrict__ a)
{
    char *m = hs_res_smem;
    return {(HsResShared *)m,           (R *)(m + a->o_acc),   (R *)(m + a->o_evw),        (uint32_t *)(m + a->o_list),
            (uint32_t *)(m + a->o_list2), (int *)(m + a->o_cnt), (int *)(m + a->o_big),      (uint16_t *)(m + a->o_evt),
            (uint16_t *)(m + a->o_stage)};
}

/* which neurons a block owns: the blocks of one XCD (blockIdx mod 8) own
   neighbouring ranges, so that the segment bounds and entries of a spike that
   they read lie in the same cache lines of their L2 */
__device__ __forceinline__ int hs_res_owner(int b, int nb)
{
    const int x = b & 7;
    return x * (nb >> 3) + min(x, nb & 7) + (b >> 3);
}

/*
 * The block's own synapses of U spikes (source, emission step Tb + offset; word
 * e[q], valid if have[q]): a segment's bounds, then V of its entries in flight per
 * spike, from entry `sub` on in steps of `step`, so that a batch costs the two
 * memory hops once.  Steps are relative to Tb.
 * WALK false: an arrival at or after `from` goes to its slot's sum (fused) or
 * bucket (plain); returns the number arriving before `end`.
 * WALK true (plain): only arrivals at step `from`, added to the target variable.
 * tb0: Tb mod nslots; b: this block's owner index.
 */
template <typename R, bool PLAIN, bool WALK, int U, int V>
__device__ __forceinline__ unsigned int hs_res_add(const HsResArgs<R> *__restrict__ a, const HsResLds<R> &L,
                                                   const uint32_t (&e)[U], const bool (&have)[U], int sub, int step,
                                                   int tb0, int from, int end, int b)
{
    const int nown = a->nown, nslots = a->nslots;
    const HsResSyn<R> *const syn = a->syn;
    int s[U], s1[U];
    unsigned int ev = 0;
#pragma unroll
    for (int q = 0; q < U; ++q) {
        s[q] = s1[q] = 0;
        if (!have[q]) continue;
        const int32_t *const o = a->off + ((e[q] & 0xfffffu) * (uint32_t)a->nb + (uint32_t)b); /* below 2^25 */
        s[q] = hs_ld(o) + sub;
        s1[q] = hs_ld(o + 1);
    }
    bool more;
    do {
        HsResSyn<R> x[U][V];
#pragma unroll
        for (int q = 0; q < U; ++q)
#pragma unroll
            for (int u = 0; u < V; ++u) {
                x[q][u].pack = 0;
                x[q][u].w = (R)0;
                if (s[q] + u * step < s1[q]) x[q][u] = hs_res_ld(syn + s[q] + u * step);
            }
        more = false;
#pragma unroll
        for (int q = 0; q < U; ++q) {
#pragma unroll
            for (int u = 0; u < V; ++u) {
                const uint32_t pk = x[q][u].pack;
                const int arr = (int)(e[q] >> 20) + (int)(pk >> 16);
                if (s[q] + u * step >= s1[q] || (WALK ? arr != from : arr < from)) continue;
                const int at = (int)((pk >> 10) & 63u) * nown + (int)(pk & 1023u);
                if (WALK) {
                    atomicAdd(&L.acc[at], x[q][u].w);
                    continue;
                }
                /* tb0 < nslots, offset < nslots, delay < nslots */
                int slot = hs_wrap(tb0 + arr, nslots);
                slot = slot >= nslots ? slot - nslots : slot;
                if constexpr (PLAIN) {
                    const int pos = atomicAdd(&L.cnt[slot], 1);
                    if (pos < a->cap) {
                        L.evt[slot * a->cap + pos] = (uint16_t)(pk & 0xffffu);
                        L.evw[slot * a->cap + pos] = x[q][u].w;
                    }
                } else {
                    atomicAdd(&L.acc[slot * a->nplanes * nown + at], x[q][u].w);
                }
                ev += arr < end ? 1u : 0u;
            }
            s[q] += V * step;
            more |= s[q] < s1[q];
        }
    } while (more);
    return ev;
}

/* n1 + n2 listed spikes by threads `rank` of nthr (a multiple of the 64 lanes),
   2^lanes_log2 threads a spike, U spikes a thread in flight */
template <typename R, bool PLAIN, bool WALK, int U = 1>
__device__ __forceinline__ unsigned int hs_res_deliver(const HsResArgs<R> *__restrict__ a, const HsResLds<R> &L, int n1,
                                                       int n2, int tb0, int from, int end, int b, int rank, int nthr)
{
    const int lg = a->lanes_log2, items = (n1 + n2) << lg;
    unsigned int ev = 0;
    for (int it = rank; it < items; it += U * nthr) {
        uint32_t e[U];
        bool have[U];
#pragma unroll
        for (int q = 0; q < U; ++q) {
            const int sp = (it + q * nthr) >> lg;
            have[q] = sp < n1 + n2;
            e[q] = !have[q] ? 0u : sp < n1 ? L.list[sp] : L.list2[sp - n1];
        }
        ev += hs_res_add<R, PLAIN, WALK, U, 4>(a, L, e, have, it & ((1 << lg) - 1), 1 << lg, tb0, from, end, b);
    }
    return ev;
}

/* spikes emitted in steps [T0 - dmax, T0), from the group's spike lists of the
   launches before: those still to arrive at T0 or later (WALK: at step T0 + u) */
template <typename R, bool PLAIN, bool WALK>
__device__ __attribute__((noinline)) unsigned int hs_res_replay(const HsResArgs<R> *__restrict__ a,
                                                                const DGroup<R> *__restrict__ g, long long T0, int u,
                                                                int nsteps)
{
    const HsResLds<R> L = hs_res_lds(a);
    HsResShared *S = L.S;
    const int dmax = a->dmax, cap = a->list_cap, b = hs_res_owner(blockIdx.x, a->nb);
    const int Q = g->Q, nsub = g->nsub;
    const int q0 = (int)hs_mod(T0 - dmax, Q), tb0 = (int)hs_mod(T0 - dmax, a->nslots);
    const long long rowlen = (long long)nsub * g->subcap;
    const int rows = dmax * nsub;
    const int wid = threadIdx.x / HS_WAVE, nwv = blockDim.x / HS_WAVE;
    unsigned int ev = 0;
    /* a thread takes a row: its count, then its offset among the block's spikes of this pass */
    for (int r0 = 0; r0 < rows; r0 += blockDim.x) {
        const int r = r0 + threadIdx.x;
        const int st = r / nsub, sub = r - st * nsub; /* emission step T0 - dmax + st */
        const long long row = (long long)hs_wrap(q0 + st, Q);
        const int have = r < rows ? hs_ld(g->hist_cnt + (row * nsub + sub) * HS_CNT_STRIDE) : 0;
        int tot;
        const int ex = hs_wave_excl_scan(have, &tot);
        if (hs_lane() == 0) S->wsum[wid] = tot;
        __syncthreads();
        int before = 0, all = 0;
        for (int v = 0; v < nwv; ++v) {
            before += v < wid ? S->wsum[v] : 0;
            all += S->wsum[v];
        }
        if (WALK && threadIdx.x == 0) S->replayed += all;
        for (int c0 = 0; c0 < all; c0 += cap) { /* uniform */
            for (int k = max(0, c0 - before - ex); k < have; ++k) {
                const int at = before + ex + k - c0;
                if (at >= cap) break;
                L.list[at] = (uint32_t)hs_ld(g->hist + row * rowlen + (long long)sub * g->subcap + k) | (uint32_t)st << 20;
            }
            __syncthreads();
            ev += hs_res_deliver<R, PLAIN, WALK>(a, L, min(cap, all - c0), 0, tb0, dmax + u, dmax + nsteps, b,
                                                 threadIdx.x, blockDim.x);
            __syncthreads();
        }
        __syncthreads();
    }
    return ev;
}

/* a header word: the window's number mod 2048 | whether the block asks for the end of
   the launch (first word) | up to four spikes of 13 bits, each
   1 + (step offset << 9 | index in the block), 0: none.  A line starts with one
   header word, or two where blocks fire more per window (models with noise: their
   windows are longer); more spikes than they hold: 0x1fff and the count in the
   first, all of them in the words behind, two a word beside the window's whole
   number.  Header words are written every window, so their short number only has
   to differ from those of the windows that used the line last. */
#define HS_RES_MANY 0x1fffu
#define HS_RES_WIN(win) ((win) & 0x7ffu) /* beside bits 53 up; depth is below 2048 */
#define HS_RES_END (1ull << 52)

__device__ __forceinline__ unsigned long long hs_res_header(uint32_t win, int n, int most, const uint16_t *stage)
{
    unsigned long long h = (unsigned long long)HS_RES_WIN(win) << 53;
    if (n > most) return h | (unsigned long long)n << 13 | HS_RES_MANY;
    const unsigned long long four = *(const unsigned long long *)stage; /* one LDS read */
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (k < n) h |= (((four >> (16 * k)) & 0xffffu) + 1u) << (13 * k);
    return h;
}

template <typename R>
__device__ __forceinline__ unsigned long long *hs_res_lines(const HsResArgs<R> *__restrict__ a, uint32_t win)
{
    return a->mail + (size_t)((win % (uint32_t)a->depth) * (uint32_t)a->nb) * a->mwords;
}

/* a word of the others that is not there yet: true to go on waiting */
__device__ __forceinline__ bool hs_res_wait(HsCtl *ctl, int *spin, long long *t0)
{
    if ((++*spin & 63) != 0) return true;
    const long long now = wall_clock64();
    if (*t0 == 0) *t0 = now;
    if (now - *t0 > HS_RES_WAIT) hs_mail_st(&ctl->stalled, 1ull);
    return hs_mail_ld(&ctl->stalled) == 0;
}

/* the spikes of a line with more than its header holds, by the thread that polls
   it: two a word, four words in flight; false: not here, left to the block */
template <typename R>
__device__ __attribute__((noinline)) void hs_res_many(const HsResArgs<R> *__restrict__ a, int q, int n, uint32_t win)
{
    const HsResLds<R> L = hs_res_lds(a);
    HsResShared *S = L.S;
    int at = S->n2;
    bool room = n <= HS_RES_FEW;
    while (room) { /* n entries of list2, if it has them */
        room = at + n <= a->list_cap;
        if (!room) break;
        const int was = atomicCAS(&S->n2, at, at + n);
        if (was == at) break;
        at = was;
    }
    if (!room) {
        L.big[atomicAdd(&S->nbig, 1)] = q;
        return;
    }
    const unsigned long long *ln = hs_res_lines(a, win) + (size_t)q * a->mwords + a->hwords;
    const uint32_t base = (uint32_t)(q * a->nown);
    const int words = (n + 1) / 2;
    long long t0 = 0;
    int spin = 0;
    for (int w0 = 0; w0 < words; w0 += 4) {
        unsigned long long h[4];
        bool missing;
        do {
            missing = false;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                h[u] = w0 + u < words ? hs_mail_ld(ln + w0 + u) : (unsigned long long)win << 32;
                missing |= (uint32_t)(h[u] >> 32) != win;
            }
        } while (missing && hs_res_wait(a->ctl, &spin, &t0));
        if (missing) atomicOr(&S->stop, HS_RES_STOP);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            for (int p = 0; p < 2; ++p) {
                const int k = 2 * (w0 + u) + p;
                const uint32_t x = (uint32_t)(h[u] >> (16 * p)) & 0xffffu;
                if (k < n) L.list2[at + k] = (base + (x & 511u)) | (x >> 9) << 20;
            }
    }
}

/* the headers of window `win`, LPT lines of HW words a thread (rank, rank + nthr,
   ...), all in flight; false: waited in vain */
template <typename R, int LPT, int HW>
__device__ __forceinline__ bool hs_res_poll(const HsResArgs<R> *__restrict__ a, const unsigned long long *lines,
                                            uint32_t win, int rank, int nthr, unsigned long long (&h)[LPT][HW])
{
    const int nb = a->nb, mwords = a->mwords;
    long long t0 = 0;
    int spin = 0;
    bool missing;
    do {
        missing = false;
#pragma unroll
        for (int u = 0; u < LPT; ++u)
#pragma unroll
            for (int k = 0; k < HW; ++k) {
                const int q = rank + u * nthr;
                h[u][k] = q < nb ? hs_mail_ld(lines + (uint32_t)(q * mwords) + k) : (unsigned long long)HS_RES_WIN(win) << 53;
            }
#pragma unroll
        for (int u = 0; u < LPT; ++u)
#pragma unroll
            for (int k = 0; k < HW; ++k) missing |= (uint32_t)(h[u][k] >> 53) != HS_RES_WIN(win);
    } while (missing && hs_res_wait(a->ctl, &spin, &t0));
    return !missing;
}

/* the spikes of window `win` into the lists, lines rank, rank + nthr, ... (LPT a thread) */
template <typename R, int LPT, int HW>
__device__ __forceinline__ void hs_res_listed(const HsResArgs<R> *__restrict__ a, const HsResLds<R> &L, uint32_t win,
                                              int rank, int nthr)
{
    unsigned long long h[LPT][HW];
    if (!hs_res_poll<R, LPT, HW>(a, hs_res_lines(a, win), win, rank, nthr, h)) {
        atomicOr(&L.S->stop, HS_RES_STOP);
        return;
    }
#pragma unroll
    for (int u = 0; u < LPT; ++u) {
        unsigned long long c = h[u][0] & (HS_RES_END - 1);
        if (h[u][0] & HS_RES_END) atomicOr(&L.S->stop, HS_RES_LAST);
        if (c == 0) continue;
        const int q = rank + u * nthr;
        if (((uint32_t)c & 0x1fffu) == HS_RES_MANY) {
            hs_res_many(a, q, (int)(c >> 13) & 0x1fff, win);
            continue;
        }
        const uint32_t base = (uint32_t)(q * a->nown);
#pragma unroll
        for (int k = 0; k < HW; ++k) {
            if (k) c = h[u][k] & (HS_RES_END - 1);
            const int n = (c != 0) + ((c >> 13) != 0) + ((c >> 26) != 0) + ((c >> 39) != 0);
            if (n == 0) continue;
            const int at = atomicAdd(&L.S->n1, n);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t x = ((uint32_t)(c >> (13 * j)) & 0x1fffu) - 1u;
                if (j < n) L.list[at + j] = (base + (x & 511u)) | (x >> 9) << 20;
            }
        }
    }
}

/* the busy lines of window `win` (emission steps from Tw on; all steps relative
   to it): their words, all threads of the block on one line at a time */
template <typename R, bool PLAIN, bool WALK>
__device__ __attribute__((noinline)) unsigned int hs_res_busy(const HsResArgs<R> *__restrict__ a, uint32_t win, int nbig,
                                                              int tb0, int from, int end)
{
    const HsResLds<R> L = hs_res_lds(a);
    const int b = hs_res_owner(blockIdx.x, a->nb);
    unsigned int ev = 0;
    for (int q = 0; q < nbig; ++q) {
        const int o = L.big[q];
        const unsigned long long *ln = hs_res_lines(a, win) + (size_t)o * a->mwords;
        const int n = (int)(hs_mail_ld(ln) >> 13) & 0x1fff;
        for (int c0 = 0; c0 < n; c0 += a->list_cap) {
            const int m = min(a->list_cap, n - c0);
            for (int k = threadIdx.x; k < m; k += blockDim.x) {
                const int sp = c0 + k;
                unsigned long long w = hs_mail_ld(ln + a->hwords + sp / 2);
                long long t0 = 0;
                int spin = 0;
                while ((uint32_t)(w >> 32) != win && hs_res_wait(a->ctl, &spin, &t0)) w = hs_mail_ld(ln + a->hwords + sp / 2);
                if ((uint32_t)(w >> 32) != win) atomicOr(&L.S->stop, HS_RES_STOP);
                const uint32_t x = (uint32_t)(w >> (16 * (sp & 1))) & 0xffffu;
                L.list[k] = (uint32_t)(o * a->nown) + (x & 511u) | (x >> 9) << 20;
            }
            __syncthreads();
            if (L.S->stop & HS_RES_STOP) return ev;
            ev += hs_res_deliver<R, PLAIN, WALK>(a, L, m, 0, tb0, from, end, b, threadIdx.x, blockDim.x);
            __syncthreads();
        }
    }
    return ev;
}

/* what the polling threads left: listed spikes and busy lines, by all threads of
   the block (after a barrier); 0 and no further barrier when there is nothing.  Adds
   what it costs, in spikes, to *load */
template <typename R, bool PLAIN, bool WALK>
__device__ __forceinline__ unsigned int hs_res_rest(const HsResArgs<R> *__restrict__ a, const HsResLds<R> &L,
                                                    uint32_t win, int b, int tb0, int from, int end, int *load)
{
    HsResShared *S = L.S;
    const int nbig = S->nbig, n1 = S->n1, n2 = S->n2;
    if (!(nbig | n1 | n2)) return 0;
    *load += n1 + n2 + HS_RES_LINE * nbig;
    unsigned int ev = hs_res_deliver<R, PLAIN, WALK>(a, L, n1, n2, tb0, from, end, b, threadIdx.x, blockDim.x);
    __syncthreads();
    if (threadIdx.x == 0) S->n1 = S->n2 = S->nbig = 0; /* appended to again after another barrier */
    if (nbig) ev += hs_res_busy<R, PLAIN, WALK>(a, win, nbig, tb0, from, end);
    return ev;
}

/* plain form, a bucket that overflowed: the effects due at step T0 + u from the
   spikes of the last dmax steps themselves; nwin: windows of this launch
   delivered so far.  Returns to thread 0 what it cost, in spikes */
template <typename R>
__device__ __attribute__((noinline)) int hs_res_walk(const HsResArgs<R> *__restrict__ a, const DGroup<R> *__restrict__ g,
                                                      long long T0, uint32_t win0, int u, int nwin)
{
    const HsResLds<R> L = hs_res_lds(a);
    const int b = hs_res_owner(blockIdx.x, a->nb), W = a->W;
    if (threadIdx.x == 0) L.S->replayed = 0;
    if (u < a->dmax) (void)hs_res_replay<R, true, true>(a, g, T0, u, u + 1);
    int load = threadIdx.x == 0 ? L.S->replayed : 0;
    for (int k = max(0, (u - a->dmax) / W); k < nwin; ++k) {
        if (a->hwords == 1) hs_res_listed<R, 4, 1>(a, L, win0 + (uint32_t)k, threadIdx.x, blockDim.x);
        else hs_res_listed<R, 1, 2>(a, L, win0 + (uint32_t)k, threadIdx.x, blockDim.x);
        __syncthreads();
        if (L.S->stop & HS_RES_STOP) return load;
        (void)hs_res_rest<R, true, true>(a, L, win0 + (uint32_t)k, b, 0, u - k * W, 0, &load);
        __syncthreads();
    }
    return load;
}

/* plain form: the effects due at step T0 + u (slot: its bucket), one after
   another onto the target variables po[v] (LDS index of this thread's value, or -1);
   *load: what a bucket that overflowed costs */
template <typename R, int NV>
__device__ __forceinline__ void hs_res_apply(const HsResArgs<R> *__restrict__ a, const DGroup<R> *__restrict__ g,
                                             const HsResLds<R> &L, const int *po, R *s, long long T0, uint32_t win0,
                                             int u, int slot, int nwin, int *load)
{
    const int c = L.cnt[slot]; /* the same for every thread */
    if (c == 0) return;
#pragma unroll
    for (int v = 0; v < NV; ++v)
        if (po[v] >= 0) L.acc[po[v]] = s[v];
    __syncthreads();
    if (c <= a->cap) {
        const int e0 = slot * a->cap, nown = a->nown;
        for (int e = threadIdx.x; e < c; e += blockDim.x) {
            const int t = L.evt[e0 + e];
            atomicAdd(&L.acc[(t >> 10) * nown + (t & 1023)], L.evw[e0 + e]);
        }
    } else {
        *load += hs_res_walk(a, g, T0, win0, u, nwin);
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NV; ++v)
        if (po[v] >= 0) s[v] = L.acc[po[v]];
    if (threadIdx.x == 0) L.cnt[slot] = 0;
}

/* a barrier among the helper waves alone: the arrivals of all windows so far are
   counted; every one of these waves comes here once a window, whatever it found */
__device__ __forceinline__ void hs_res_meet(HsResShared *S, int arrivals)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (hs_lane() == 0) __hip_atomic_fetch_add(&S->met, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (__hip_atomic_load(&S->met, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < arrivals) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

/* a model that draws noise: the block has HS_RES_HELPERS threads more, which
   collect and deliver the others' spikes while the owners draw the next window's
   noise (3.6 us for 6 steps of 100,000 FP32 neurons) */
template <int MS> __host__ __device__ constexpr bool hs_res_helper()
{
    return MS == HS_MODEL_LIF_NOISE;
}

/* the n draws of steps T .. T+n-1: independent chains, two at a time, which with
   two waves on a SIMD fills its pipeline */
template <typename R, int MS>
__device__ __forceinline__ void hs_res_noise(const HsStepK<R> &c, int i, long long T, int n, R (&xi)[HS_MAX_WINDOW])
{
    constexpr int G = 2;
#pragma unroll
    for (int j0 = 0; j0 < HS_MAX_WINDOW; j0 += G) {
        if (j0 < n) {
#pragma unroll
            for (int j = j0; j < j0 + G; ++j) xi[j] = hs_noise<R, MS>(c.seed, c.stream, i, T + j);
        }
    }
}

template <typename R, int MS, bool PLAIN>
__global__ __launch_bounds__(HS_RES_MAXT + (hs_res_helper<MS>() ? HS_RES_HELPERS : 0)) void
hs_k_resident(const HsResArgs<R> *__restrict__ a, const DGroup<R> *__restrict__ g, const long long T0, const int nsteps,
              const uint32_t win0)
{
    constexpr int NV = HsNV<MS>::value;
    constexpr bool HELP = hs_res_helper<MS>(), NOISY = HELP;
    constexpr int HW = HELP ? 2 : 1; /* header words (a->hwords) */
    /* fused form: a's fields are then read once and kept, where the compiler would read
       them again in every step by scalar loads (100,000 neurons FP32 1.82 us a step and
       1.97, 64 networks 3.8 and 4.05); the plain form, short of registers, gains by
       those (CUBA 4,000 FP64 2.07 and 2.21) */
    if constexpr (!PLAIN) (void)hs_here(a);
    const HsResLds<R> L = hs_res_lds(a);
    HsResShared *const S = L.S;
    const int nb = a->nb, nown = a->nown, W = a->W, nslots = a->nslots;
    const int tid = threadIdx.x, b = hs_res_owner(blockIdx.x, nb), wid = tid / HS_WAVE;
    const int nwv = (int)blockDim.x / HS_WAVE - (HELP ? HS_RES_HELPERS / HS_WAVE : 0); /* waves that own neurons */
    const bool helper = HELP && wid >= nwv;
    if (helper) __builtin_amdgcn_s_setprio(3); /* few instructions, all of them waited for */
    const int i = b * nown + tid;
    const bool valid = tid < nown && i < a->n;

    R s[NV];
    int po[NV]; /* this thread's value in plane of variable v: an index into acc, or -1 */
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        s[v] = valid ? hs_ld(g->var[v] + i) : (R)0;
        po[v] = valid && a->plane[v] >= 0 ? a->plane[v] * nown + tid : -1;
    }
    int32_t last = valid ? hs_ld(g->last + i) : HS_NEVER_SPIKED;
    const HsStepK<R> c(*g);
    R k[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) k[q] = g->k[q];
    R xi[NOISY ? HS_MAX_WINDOW : 1];
    if constexpr (NOISY)
        if (valid) hs_res_noise<R, MS>(c, i, T0, min(W, nsteps), xi);
    if (tid == 0) S->nspk[0] = S->nspk[1] = S->n1 = S->n2 = S->nbig = S->stop = S->met = 0;
    if (PLAIN) {
        for (int q = tid; q < nslots; q += blockDim.x) L.cnt[q] = 0;
    } else {
        for (int q = tid; q < nslots * a->nplanes * nown; q += blockDim.x) L.acc[q] = (R)0;
    }
    __syncthreads();
    unsigned int ev = a->dmax ? hs_res_replay<R, PLAIN, false>(a, g, T0, 0, nsteps) : 0u;
    /* held: spikes and lines of the window before; load: those, and walks, beyond `most` a
       window (thread 0's count); ask: the block asks for the end of the launch */
    int most = a->most, held = 0, load = 0;
    uint32_t ask = 0;
    asm volatile("" : "+v"(most)); /* the scalar registers are taken */

    const int extras = (g->smon_n ? 1 : 0) | (g->rmon_cnt ? 2 : 0);
    const int slotlen = a->nplanes * nown;
    unsigned int spikes = 0;
    int slot = (int)hs_mod(T0 - 1, nslots); /* slot of the step before the next one */
    int nwin = 0, t = 0, stop; /* t: step - T0 */
    do {
        const int w = min(W, nsteps - t);
        const uint32_t win = win0 + (uint32_t)nwin;
        const int tb0 = slot + 1 == nslots ? 0 : slot + 1; /* slot of step t */
        unsigned int bits = 0; /* bit j: spike at step t + j */
#pragma unroll 1
        for (int j = 0; j < w; ++j) {
            if constexpr (PLAIN) {
                hs_res_apply<R, NV>(a, g, L, po, s, T0, win0, t + j - 1, slot, nwin, &load);
            } else {
                R eff[NV];
                R *const row = L.acc + slot * slotlen;
#pragma unroll
                for (int v = 0; v < NV; ++v) eff[v] = po[v] >= 0 ? row[po[v]] : (R)0;
#pragma unroll
                for (int v = 0; v < NV; ++v)
                    if (po[v] >= 0) {
                        s[v] = s[v] + eff[v];
                        row[po[v]] = (R)0;
                    }
            }
            slot = slot + 1 == nslots ? 0 : slot + 1;
            R xj = (R)0;
            if (NOISY) {
                xj = xi[0];
#pragma unroll
                for (int m = 0; m + 1 < HS_MAX_WINDOW; ++m) xi[NOISY ? m : 0] = xi[NOISY ? m + 1 : 0];
            }
            if (valid && hs_step_one<R, MS, !PLAIN>(*g, c, s, k, last, T0 + t + j, i, T0, xj)) bits |= 1u << j;
        }
        /* the block's spikes of the window: published first, monitors after that */
        if (__ballot(bits != 0))
            for (int j = 0; j < w; ++j) {
                const bool spk = (bits >> j) & 1u;
                const unsigned long long m = __ballot(spk);
                if (m) {
                    int at = 0;
                    if (hs_lane() == 0) at = atomicAdd(&S->nspk[nwin & 1], (int)__popcll(m));
                    at = __shfl(at, 0, HS_WAVE) + __popcll(m & hs_lanemask_lt());
                    if (spk) L.stage[at] = (uint16_t)(j << 9 | tid);
                }
            }
        __syncthreads();
        if (HELP && wid == 0) __builtin_amdgcn_s_setprio(3); /* the others already draw */
        const int nspk = S->nspk[nwin & 1];
        unsigned long long *const lines = hs_res_lines(a, win);
        if (tid == 0) {
            unsigned long long *const ln = lines + (uint32_t)(b * a->mwords);
            hs_mail_st(ln, hs_res_header(win, nspk, 4 * HW, L.stage) | (unsigned long long)ask << 32);
            if (HW == 2) hs_mail_st(ln + 1, hs_res_header(win, nspk > 4 && nspk <= 8 ? nspk - 4 : 0, 8, L.stage + 4));
            S->nspk[(nwin & 1) ^ 1] = 0; /* read by all before the last barrier, counted in after the next */
            spikes += (unsigned int)nspk;
        }
        if (nspk > 4 * HW)
            for (int q = tid; q < (nspk + 1) / 2; q += blockDim.x)
                hs_mail_st(lines + (uint32_t)(b * a->mwords) + HW + q,
                           (unsigned long long)win << 32 | L.stage[2 * q] |
                               (2 * q + 1 < nspk ? (uint32_t)L.stage[2 * q + 1] << 16 : 0u));
        if (HELP && wid == 0) __builtin_amdgcn_s_setprio(0);
        load = max(0, load + held - most);
        ask = load > HS_RES_SLACK * most ? (uint32_t)(HS_RES_END >> 32) : 0u;
        if (!helper) {
            if (extras) {
                const DGroup<R> *h = hs_here(g);
                if (extras & 2)
                    for (int j = 0; j < w; ++j) {
                        const unsigned long long in =
                            __ballot(((bits >> j) & 1u) && i >= h->rmon_start && i < h->rmon_stop);
                        const long long row = T0 + t + j - h->rmon_t0;
                        if (hs_lane() == 0 && in && row >= 0 && row < h->rmon_rows)
                            hs_atomic_add(h->rmon_cnt + row, (int32_t)__popcll(in));
                    }
                if ((extras & 1) && nspk && wid == 0) {
                    unsigned long long at = 0;
                    if (tid == 0) at = hs_atomic_fetch_add(h->smon_n, (unsigned long long)nspk);
                    at = __shfl(at, 0, HS_WAVE);
                    for (int q = tid; q < nspk; q += HS_WAVE) {
                        const int x = L.stage[q];
                        if ((long long)(at + q) < h->smon_cap) {
                            hs_st(h->smon_i + at + q, (int32_t)(b * nown + (x & 511)));
                            hs_st(h->smon_t + at + q, (int32_t)(T0 + t + (x >> 9)));
                        }
                    }
                }
            }
            if constexpr (NOISY)
                if (valid) hs_res_noise<R, MS>(c, i, T0 + t + w, min(W, nsteps - t - w), xi);
        }
        /* every arrival of this window's spikes lies ahead: at step t + w - 1 or later */
        if constexpr (HELP) {
            if (helper) {
                const int rank = tid - nwv * HS_WAVE;
                hs_res_listed<R, 1, HW>(a, L, win, rank, HS_RES_HELPERS);
                hs_res_meet(S, (HS_RES_HELPERS / HS_WAVE) * (nwin + 1));
                ev += hs_res_deliver<R, PLAIN, false, 2>(a, L, S->n1, S->n2, tb0, 0, nsteps - t, b, rank,
                                                         HS_RES_HELPERS);
            }
            __syncthreads();
            stop = S->stop; /* uniform: set before a barrier, and the headers are the same for everybody */
            if (stop & HS_RES_STOP) return;
            const int nbig = S->nbig;
            held = S->n1 + S->n2 + HS_RES_LINE * nbig; /* (thread 0 reads them before it clears them) */
            if (tid == 0) S->n1 = S->n2 = 0; /* read by all helpers before the barrier, appended to after another */
            if (nbig) { /* lines that hold more than HS_RES_FEW */
                __syncthreads();
                if (tid == 0) S->nbig = 0;
                ev += hs_res_busy<R, PLAIN, false>(a, win, nbig, tb0, 0, nsteps - t);
            }
        } else {
            if ((int)blockDim.x >= nb) hs_res_listed<R, 1, HW>(a, L, win, tid, blockDim.x);
            else hs_res_listed<R, 4, HW>(a, L, win, tid, blockDim.x);
            __syncthreads();
            stop = S->stop;
            if (stop & HS_RES_STOP) return;
            held = 0;
            ev += hs_res_rest<R, PLAIN, false>(a, L, win, b, tb0, 0, nsteps - t, &held);
        }
        if (S->stop & HS_RES_STOP) return;
        t += w;
        ++nwin;
    } while (!stop && t < nsteps);
    /* the state after the last step: its effects, then the resets of its spikers */
    if constexpr (PLAIN) {
        hs_res_apply<R, NV>(a, g, L, po, s, T0, win0, t - 1, slot, nwin, &load);
    } else {
#pragma unroll
        for (int v = 0; v < NV; ++v)
            if (po[v] >= 0) s[v] = s[v] + L.acc[slot * slotlen + po[v]];
    }
    const long long Tend = T0 + t;
    if (valid) {
        if (c.has_reset && (long long)last == Tend - 1) s[0] = c.vr;
#pragma unroll
        for (int v = 0; v < NV; ++v) hs_st(g->var[v] + i, s[v]);
        hs_st(g->last + i, last);
    }
    const unsigned long long evs = hs_wave_sum((unsigned long long)ev);
    hs_flush_events(evs, a->ctl, (long long)b * (blockDim.x / HS_WAVE) + wid);
    if (b == 0 && tid == 0) a->ctl->ran = t;
    if (tid == 0 && spikes)
        hs_atomic_add(&a->ctl->spk_slot[(b % HS_EV_SLOTS) * HS_EV_STRIDE], (unsigned long long)spikes);
}

#endif /* HS_RESIDENT_H */
