// PageRank over the pull layout (outDegree + in-edge CSR) on gfx950.
//
// Reference shape: prSumKernel_static / prSumKernel_dynamic / prKernel_Opt
// (PR/OneGraph/gpu_kernels.h:107-158, 295-318) driven by pr_opt
// (PR/OneGraph/CalculateOpt.h:13-185).  The numerics follow the normalised
// definition instead of the reference's 0.15 + 0.85*sum:
//   contrib[u] = rank[u] / outdeg[u]            (0 for dangling u)
//   dangling   = sum of rank[u] over outdeg[u] == 0
//   new[v]     = (1-d)/n + d * (sum_{u in in(v)} contrib[u] + dangling/n)
//   stop when sum_v |new[v] - rank[v]| < tol or after max_iterations.
// FP32 mode keeps ranks in FP32 and sums in-edges with Kahan compensation;
// the dangling mass and the L1 residual are reduced in FP64 in a fixed order
// (per-block partials, then one workgroup), so runs are deterministic.
//
// Every vertex is active each iteration, so the dynamic region is the
// contiguous in-edge range [ptr[vsplit], E): it is copied chunk by chunk
// straight from pinned host memory (no gather) on two copy streams while
// earlier chunks are being summed.
#include <algorithm>

#include "device.h"

namespace og {

constexpr int kPrLpv0 = 4;   // lanes per vertex for rows up to t1
constexpr int kPrRangeLpv = 8;  // the same in the dynamic region, whose rows come in every length
constexpr int kPrBatch = 8;  // in-edges per lane whose reads are in flight together

// A static row: its in-edges and its vertex, one 16-byte load.
struct PrRow {
    uint64_t b;
    uint32_t n, v;  // n = 0xFFFFFFFF: longer, read the row bounds
};

template <typename T>
struct Acc {  // running sum with Kahan compensation: value = s - c
    T s = 0, c = 0;
    __device__ __forceinline__ void add(T x) {
        const T y = x - c;
        const T t = s + y;
        c = (t - s) - y;
        s = t;
    }
    // Merges another accumulator using an error-free TwoSum of the heads.
    __device__ __forceinline__ void merge(T s2, T c2) {
        const T t = s + s2;
        const T bp = t - s;
        const T e = (s - (t - bp)) + (s2 - bp);
        s = t;
        c = c + c2 - e;
    }
    __device__ __forceinline__ T value() const { return s - c; }
};

template <typename T>
__device__ __forceinline__ T shfl_xor_t(T x, int m) {
    return __shfl_xor(x, m, kWave);
}

// Reduces the accumulators of LPV consecutive lanes (LPV a power of two <= 64).
template <typename T, int LPV>
__device__ __forceinline__ void group_merge(Acc<T> &a) {
#pragma unroll
    for (int m = 1; m < LPV; m <<= 1) {
        const T s2 = shfl_xor_t(a.s, m), c2 = shfl_xor_t(a.c, m);
        a.merge(s2, c2);
    }
}

__device__ __forceinline__ double block_sum_f64(double x, double *lds) {
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) x += __shfl_xor(x, m, kWave);
    if (lane == 0) lds[wid] = x;
    __syncthreads();
    double t = 0;
    for (int w = 0; w < (int)(blockDim.x / kWave); ++w) t += lds[w];
    __syncthreads();
    return t;
}

// Sum of the contributions of a row's in-edges sub, sub + L, sub + 2 L, ...
// (L lanes per row), kPrBatch edge reads and then their contributions in
// flight: one at a time a lane waited two memory latencies per edge.
// edge(i): the row's in-neighbour i.
template <typename T, class Edge>
__device__ __forceinline__ void pull_row(Acc<T> &a, Edge edge, uint64_t n, uint32_t sub, uint32_t L,
                                         const T *__restrict__ contrib) {
    for (uint64_t i = sub; i < n; i += (uint64_t)kPrBatch * L) {
        uint32_t u[kPrBatch];
        T x[kPrBatch];
#pragma unroll
        for (int k = 0; k < kPrBatch; ++k) u[k] = i + (uint64_t)k * L < n ? edge(i + (uint64_t)k * L) : 0u;
#pragma unroll
        for (int k = 0; k < kPrBatch; ++k) x[k] = i + (uint64_t)k * L < n ? contrib[u[k]] : (T)0;
#pragma unroll
        for (int k = 0; k < kPrBatch; ++k)
            if (i + (uint64_t)k * L < n) a.add(x[k]);
    }
}

// The iteration's inputs and outputs.
template <typename T>
struct PrArgs {
    const uint64_t *ptr;
    const uint32_t *edges;      // static region
    const T *contrib;           // rank / out-degree before the iteration
    T *next;                    // and after it
    T *rank;                    // updated in place: a row reads and writes its own vertex only
    const uint32_t *outdeg;
    PrState *st;
    double damping, inv_n;
    double *partial;            // two per workgroup of the iteration: residual, dangling mass
};

// New rank of v: stored with its contribution to the next iteration; adds
// the residual and the dangling mass.
template <typename T>
__device__ __forceinline__ void pr_apply(const PrArgs<T> &p, uint32_t v, T sum, T base, double &res, double &dang) {
    const T nv = base + (T)p.damping * sum;
    const uint32_t od = p.outdeg[v];
    res += fabs((double)nv - (double)p.rank[v]);
    p.rank[v] = nv;
    p.next[v] = od ? nv / (T)od : (T)0;
    if (!od) dang += (double)nv;
}

// (1-d)/n + d * dangling / n, formed in FP64 then rounded once.
template <typename T>
__device__ __forceinline__ T pr_base(const PrArgs<T> &p) {
    return (T)((1.0 - p.damping) * p.inv_n + p.damping * p.st->dangling * p.inv_n);
}

// A workgroup's partials, at slot i; device-scope stores, so that the
// workgroup that finishes the iteration can read them in the same launch.
__device__ __forceinline__ void pr_partial(double *partial, uint64_t i, double res, double dang, double *lds) {
    res = block_sum_f64(res, lds);
    dang = block_sum_f64(dang, lds);
    if (threadIdx.x == 0) {
        __hip_atomic_store(partial + 2 * i, res, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(partial + 2 * i + 1, dang, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Sums n workgroups' partials in a fixed order and closes the iteration.
// progress (pinned host memory): iterations so far << 1 | done.
__device__ __forceinline__ void pr_finish(const double *partial, uint32_t n, PrState *st, unsigned long long *progress,
                                          double *lds) {
    double res = 0, dang = 0;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
        res += __hip_atomic_load(partial + 2 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        dang += __hip_atomic_load(partial + 2 * i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    res = block_sum_f64(res, lds);
    dang = block_sum_f64(dang, lds);
    if (threadIdx.x == 0) {
        const uint32_t it = st->iterations + 1, done = res < st->tolerance ? 1u : 0u;
        st->dangling = dang;
        st->l1 = res;
        st->iterations = it;
        st->done = done;
        __hip_atomic_store(progress, (unsigned long long)it << 1 | done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ __launch_bounds__(1024) void k_pr_finish(const double *partial, uint32_t n, PrState *st,
                                                    unsigned long long *progress) {
    __shared__ double lds[1024 / kWave];
    if (st->done) return;
    pr_finish(partial, n, st, progress, lds);
}

// Start: uniform ranks and their contributions; the last workgroup sums the
// dangling mass.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pr_init(PrArgs<T> p, uint64_t V, double tolerance, CompactTotals ct) {
    __shared__ double lds[kBlock / kWave];
    __shared__ uint32_t s_last;
    const T r = (T)p.inv_n;
    double dang = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * kBlock + threadIdx.x; v < V; v += (uint64_t)gridDim.x * kBlock) {
        const uint32_t od = p.outdeg[v];
        p.rank[v] = r;
        p.next[v] = od ? r / (T)od : (T)0;
        if (!od) dang += (double)r;
    }
    pr_partial(p.partial, blockIdx.x, 0.0, dang, lds);
    if (threadIdx.x == 0) {
        wait_vmem();
        s_last = arrive_last(ct) ? 1u : 0u;
    }
    __syncthreads();
    if (!s_last) return;
    double d = 0;
    for (uint32_t i = threadIdx.x; i < gridDim.x; i += kBlock)
        d += __hip_atomic_load(p.partial + 2 * i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    d = block_sum_f64(d, lds);
    if (threadIdx.x == 0) *p.st = PrState{d, 0.0, tolerance, 0u, 0u};
}

// Pull over the static region in one launch: workgroups [0, nh) take a hub
// row each (first, as they run longest), the next g1 stride over the wave
// rows (t1 < in-degree <= t2), the rest over the short rows, kPrLpv0 lanes
// each.  With `progress` the workgroup that arrives last also closes the
// iteration, so that an iteration of a graph wholly in HBM is one launch
// (300 K vertices, 4.5 M edges, FP64: contribution pass, three pulls, two
// reductions, a copy and a host round trip took 122 us).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pr_pull(PrArgs<T> p, const PrRow *__restrict__ rows, uint32_t n0, uint32_t n1,
                                                    uint32_t nh, uint32_t g1, CompactTotals ct,
                                                    unsigned long long *progress) {
    __shared__ double lds[kBlock / kWave];
    __shared__ T s_s[kBlock / kWave], s_c[kBlock / kWave];
    __shared__ uint32_t s_last;
    if (p.st->done) return;
    const T base = pr_base(p);
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    double res = 0, dang = 0;
    auto row_at = [&](uint32_t i, uint64_t &n) {
        const PrRow r = rows[i];
        n = r.n != 0xFFFFFFFFu ? r.n : p.ptr[r.v + 1] - r.b;
        return r;
    };
    if (blockIdx.x < nh) {
        uint64_t n;
        const PrRow r = row_at(n0 + n1 + blockIdx.x, n);
        Acc<T> a;
        pull_row(a, [e = p.edges + r.b](uint64_t i) { return e[i]; }, n, threadIdx.x, kBlock, p.contrib);
        group_merge<T, kWave>(a);
        if (lane == 0) {
            s_s[wid] = a.s;
            s_c[wid] = a.c;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            Acc<T> t;
            t.s = s_s[0];
            t.c = s_c[0];
            for (int w = 1; w < kBlock / kWave; ++w) t.merge(s_s[w], s_c[w]);
            pr_apply<T>(p, r.v, t.value(), base, res, dang);
        }
    } else if (blockIdx.x < nh + g1) {
        for (uint32_t i = (blockIdx.x - nh) * (kBlock / kWave) + wid; i < n1; i += g1 * (kBlock / kWave)) {
            uint64_t n;
            const PrRow r = row_at(n0 + i, n);
            Acc<T> a;
            pull_row(a, [e = p.edges + r.b](uint64_t i) { return e[i]; }, n, lane, kWave, p.contrib);
            group_merge<T, kWave>(a);
            if (lane == 0) pr_apply<T>(p, r.v, a.value(), base, res, dang);
        }
    } else {
        const uint32_t g0 = gridDim.x - nh - g1;
        const uint32_t sub = threadIdx.x % kPrLpv0;
        for (uint64_t i = ((uint64_t)(blockIdx.x - nh - g1) * kBlock + threadIdx.x) / kPrLpv0; i < n0;
             i += (uint64_t)g0 * (kBlock / kPrLpv0)) {
            uint64_t n;
            const PrRow r = row_at((uint32_t)i, n);
            Acc<T> a;
            pull_row(a, [e = p.edges + r.b](uint64_t i) { return e[i]; }, n, sub, kPrLpv0, p.contrib);
            group_merge<T, kPrLpv0>(a);
            if (sub == 0) pr_apply<T>(p, r.v, a.value(), base, res, dang);
        }
    }
    pr_partial(p.partial, blockIdx.x, res, dang, lds);
    if (!progress) return;
    if (threadIdx.x == 0) {
        wait_vmem();
        s_last = arrive_last(ct) ? 1u : 0u;
    }
    __syncthreads();
    if (s_last) pr_finish(p.partial, gridDim.x, p.st, progress, lds);
}

// Pull for the contiguous vertex range [va, vb) whose in-edges sit in `stage`
// starting at edge ptr[va]: whole ids, or with lbits a stream of lbits-bit
// ones whose first starts `first` bits in; partials from slot poff on.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pr_pull_range(PrArgs<T> p, uint32_t va, uint32_t vb,
                                                          const uint32_t *__restrict__ stage, uint32_t lbits,
                                                          uint32_t first, uint64_t poff) {
    __shared__ double lds[kBlock / kWave];
    const uint32_t sub = threadIdx.x % kPrRangeLpv;
    const uint64_t e0 = p.ptr[va];
    const uint64_t v = va + ((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kPrRangeLpv;
    double res = 0, dang = 0;
    if (v < vb) {  // the lanes of a row go together
        const uint64_t b = p.ptr[v] - e0, n = p.ptr[v + 1] - e0 - b;
        Acc<T> a;
        if (lbits)
            pull_row(a, [=](uint64_t i) { return link_word(stage, b + i, lbits, first); }, n, sub, kPrRangeLpv, p.contrib);
        else
            pull_row(a, [=](uint64_t i) { return stage[b + i]; }, n, sub, kPrRangeLpv, p.contrib);
        group_merge<T, kPrRangeLpv>(a);
        if (sub == 0) pr_apply<T>(p, (uint32_t)v, a.value(), pr_base(p), res, dang);
    }
    pr_partial(p.partial, poff + blockIdx.x, res, dang, lds);
}

// --------------------------------------------------------------- host

namespace {

struct PrPlan {
    uint32_t n0 = 0, n1 = 0, nh = 0;  // static rows: up to t1, up to t2, hubs
    unsigned g0 = 0, g1 = 0;          // workgroups of the first two
    LinkRing *link = nullptr;         // the dynamic region's chunks (null: none)
    PrRow *d_rows = nullptr;
    uint64_t blocks = 0;              // workgroups of an iteration
    unsigned static_grid() const { return nh + g1 + g0; }
};

unsigned grid_of(uint64_t threads) {
    return (unsigned)std::max<uint64_t>(1, (threads + kBlock - 1) / kBlock);
}

// Workgroups of the short and the wave rows at most: enough to fill the chip
// (eight of 256 lanes per CU), few enough that the last one sums their
// partials quickly.
constexpr unsigned kPrGridCap = 2048;

}  // namespace

// Per-graph PageRank plan, cached on the device state.
static PrPlan &pr_plan(DeviceState *d, const og_graph *g) {
    if (d->pr_plan) return *(PrPlan *)d->pr_plan.get();
    std::shared_ptr<PrPlan> p = std::make_shared<PrPlan>();
    const uint64_t vs = d->plan.vsplit;
    auto bin = [&](uint64_t deg) { return deg <= d->tune.t1 ? 0 : deg <= d->tune.t2 ? 1 : 2; };
    uint64_t cnt[3] = {0, 0, 0};
    for (uint64_t v = 0; v < vs; ++v) cnt[bin(g->ptr[v + 1] - g->ptr[v])]++;
    std::vector<PrRow> rows(vs);
    uint64_t at[3] = {0, cnt[0], cnt[0] + cnt[1]};
    for (uint64_t v = 0; v < vs; ++v) {
        const uint64_t n = g->ptr[v + 1] - g->ptr[v];
        rows[at[bin(n)]++] = PrRow{g->ptr[v], (uint32_t)std::min<uint64_t>(n, 0xFFFFFFFFull), (uint32_t)v};
    }
    p->n0 = (uint32_t)cnt[0];
    p->n1 = (uint32_t)cnt[1];
    p->nh = (uint32_t)cnt[2];
    if (vs) {
        p->g0 = p->n0 ? std::min(kPrGridCap, grid_of((uint64_t)p->n0 * kPrLpv0)) : 0;
        p->g1 = p->n1 ? std::min(kPrGridCap, grid_of((uint64_t)p->n1 * kWave)) : 0;
        p->d_rows = (PrRow *)d->dalloc(vs * sizeof(PrRow));
        OG_HIP(hipMemcpy(p->d_rows, rows.data(), vs * sizeof(PrRow), hipMemcpyHostToDevice));
    }
    if (vs < d->V) {
        p->link = link_ring(d, g);
        if (!p->link)
            raise(OG_EBUDGET, "a vertex has more in-edges than a staging slot holds (%llu)",
                  (unsigned long long)d->slot_edges);
    }
    p->blocks = p->static_grid();
    if (p->link)
        for (auto &c : p->link->chunks) p->blocks += grid_of((uint64_t)(c.vb - c.va) * kPrRangeLpv);
    d->pr_plan = p;
    return *p;
}

template <typename T>
static void run_pr(og_graph *g, const og_pr_params &prm, T *out, og_pr_stats *stats) {
    DeviceState *d = g->dev;
    const uint64_t V = d->V;
    PrPlan &pp = pr_plan(d, g);
    hipStream_t s = d->s_compute;
    const unsigned igrid = (unsigned)std::min<uint64_t>(1024, grid_of(V));
    const uint64_t cap = std::max<uint64_t>(pp.blocks, igrid);
    // (each by itself: a call that ran out of memory leaves the rest to the next)
    if (!d->d_prstate) d->d_prstate = (PrState *)d->dalloc(sizeof(PrState));
    if (!d->h_prstate) d->h_prstate = (PrState *)d->palloc(sizeof(PrState));
    if (!d->h_progress) d->h_progress = (unsigned long long *)d->palloc(sizeof(unsigned long long));
    // sized for double so either precision fits
    if (!d->d_rank) d->d_rank = d->dalloc(V * 8);
    for (auto &c : d->d_contrib)
        if (!c) c = d->dalloc(V * 8);
    if (!d->d_outdeg) {
        uint32_t *od = (uint32_t *)d->dalloc(V * 4);
        OG_HIP(hipMemcpy(od, g->out_degree, V * 4, hipMemcpyHostToDevice));
        d->d_outdeg = od;
    }
    if (cap > d->pr_partial_cap) {
        d->d_partial = (double *)d->dalloc(cap * 2 * sizeof(double));
        d->d_prtot = (unsigned long long *)d->dalloc(totals_words(cap) * 8);
        // (on the stream whose kernels count in them: it does not wait for the null stream)
        OG_HIP(hipMemsetAsync(d->d_prtot, 0, totals_words(cap) * 8, s));
        d->pr_partial_cap = cap;
    }
    T *contrib[2] = {(T *)d->d_contrib[0], (T *)d->d_contrib[1]};
    PrArgs<T> a{d->d_ptr, (const uint32_t *)d->d_static, nullptr, contrib[0], (T *)d->d_rank, d->d_outdeg, d->d_prstate,
                prm.damping, 1.0 / (double)V, d->d_partial};
    TimedClass tc_init, tc_static, tc_dyn, tc_copy;
    d->events.reset();
    og_pr_stats st{};
    st.run.approach = (uint32_t)d->approach;

    OG_HIP(hipStreamSynchronize(d->s_copy));
    OG_HIP(hipStreamSynchronize(d->s_static));
    OG_HIP(hipStreamSynchronize(s));
    Stopwatch total;
    __atomic_store_n(d->h_progress, 0ull, __ATOMIC_RELEASE);
    {
        EventSpan span(d, &tc_init, s);
        hipLaunchKernelGGL(k_pr_init<T>, dim3(igrid), dim3(kBlock), 0, s, a, V, prm.tolerance,
                           CompactTotals{d->d_prtot, igrid, 0});
        OG_HIP(hipGetLastError());
    }
    const uint64_t vb_bytes = sizeof(T);
    const unsigned sgrid = pp.static_grid();
    // the iteration's arrays: contributions of the last one in, its own out
    auto turn = [&](uint32_t it) {
        a.contrib = contrib[it & 1];
        a.next = contrib[(it + 1) & 1];
    };
    auto pull_static = [&](hipStream_t on, unsigned long long *progress) {
        hipLaunchKernelGGL(k_pr_pull<T>, dim3(sgrid), dim3(kBlock), 0, on, a, pp.d_rows, pp.n0, pp.n1, pp.nh, pp.g1,
                           CompactTotals{d->d_prtot, sgrid, 0}, progress);
        OG_HIP(hipGetLastError());
    };
    uint32_t it = 0;
    if (!pp.link) {
        // One launch per iteration, enqueued a few ahead of the device:
        // iterations past the last one return at once.
        constexpr uint32_t kAhead = 4;
        {
            EventSpan span(d, &tc_static, s);
            for (uint32_t k = 0; k < prm.max_iterations; ++k) {
                if (k >= kAhead) wait_progress(d->h_progress, (unsigned long long)(k - kAhead + 1) << 1, s);
                if (__atomic_load_n(d->h_progress, __ATOMIC_ACQUIRE) & 1) break;
                turn(k);
                pull_static(s, d->h_progress);
            }
        }
        OG_HIP(hipMemcpyAsync(d->h_prstate, d->d_prstate, sizeof(PrState), hipMemcpyDeviceToHost, s));
        OG_HIP(hipStreamSynchronize(s));
        it = d->h_prstate->iterations;
    } else {
        // Chunk c of every iteration goes through slot (running number) % ring.
        // The copies run ahead of the pulls by the ring, into the next
        // iteration too (its edges are the same whatever the ranks are), so
        // the link does not wait for the end of an iteration nor, while the
        // ring fills, for the static pull; an iteration that turns out to be the
        // last has up to a ring of copies enqueued for nothing, which are not
        // counted.  Consecutive copies alternate
        // between two streams: the hand-over from a copy to the next one's
        // wait costs about 30 us, hidden behind the other stream's copy.
        LinkRing &lr = *pp.link;
        const uint64_t nc = lr.chunks.size();
        const uint64_t limit = prm.max_iterations * nc;
        uint64_t copied = 0, pulled = 0;
        auto copy_next = [&] {
            const LinkRing::Chunk &ch = lr.chunks[copied % nc];
            const uint32_t slot = (uint32_t)(copied % lr.ring);
            uint32_t *dslot = (uint32_t *)d->d_staging + slot * lr.slot;
            const hipStream_t on = copied & 1 ? d->s_static : d->s_copy;
            if (copied >= lr.ring) OG_HIP(hipStreamWaitEvent(on, lr.ev_use[slot], 0));
            if (ch.words)
                OG_HIP(hipMemcpyAsync(dslot, lr.src + ch.word, ch.words * 4, hipMemcpyHostToDevice, on));
            OG_HIP(hipEventRecord(lr.ev_h2d[slot], on));
            ++copied;
        };
        {
            EventSpan copies(d, &tc_copy, d->s_copy);  // first copy to last: the link is busy throughout
            while (it < prm.max_iterations) {
                turn(it);
                // the copies first: what the ring holds crosses the link beside the static pull
                while (copied < std::min(pulled + std::min<uint64_t>(lr.ring, nc), limit)) copy_next();
                if (sgrid) {
                    EventSpan span(d, &tc_static, s);
                    pull_static(s, nullptr);
                }
                uint64_t poff = sgrid;
                for (uint64_t c = 0; c < nc; ++c, ++pulled) {
                    const LinkRing::Chunk &ch = lr.chunks[c];
                    const uint32_t slot = (uint32_t)(pulled % lr.ring);
                    OG_HIP(hipStreamWaitEvent(s, lr.ev_h2d[slot], 0));
                    const unsigned gr = grid_of((uint64_t)(ch.vb - ch.va) * kPrRangeLpv);
                    {
                        EventSpan span(d, &tc_dyn, s);
                        hipLaunchKernelGGL(k_pr_pull_range<T>, dim3(gr), dim3(kBlock), 0, s, a, ch.va, ch.vb,
                                           (const uint32_t *)d->d_staging + slot * lr.slot, lr.lbits, ch.first, poff);
                        OG_HIP(hipGetLastError());
                    }
                    poff += gr;
                    OG_HIP(hipEventRecord(lr.ev_use[slot], s));
                    st.run.h2d_bytes += ch.words * 4;
                    st.run.chunks++;
                    // the slots that are free, the one this chunk leaves among them,
                    // up to the next iteration's last chunk
                    while (copied < std::min({pulled + 1 + lr.ring, (it + 2) * nc, limit})) copy_next();
                }
                hipLaunchKernelGGL(k_pr_finish, dim3(1), dim3(1024), 0, s, d->d_partial, (uint32_t)poff, d->d_prstate,
                                   d->h_progress);
                OG_HIP(hipGetLastError());
                ++it;
                wait_progress(d->h_progress, (unsigned long long)it << 1, s);
                if (__atomic_load_n(d->h_progress, __ATOMIC_ACQUIRE) & 1) break;
            }
        }
        OG_HIP(hipMemcpyAsync(d->h_prstate, d->d_prstate, sizeof(PrState), hipMemcpyDeviceToHost, s));
        OG_HIP(hipStreamSynchronize(s));
        OG_HIP(hipStreamSynchronize(d->s_copy));
        OG_HIP(hipStreamSynchronize(d->s_static));
    }
    st.run.total_ms = total.ms();
    if (out) copy_to_host(d, out, d->d_rank, V * sizeof(T), s);
    const uint64_t sedges = d->plan.vsplit ? g->ptr[d->plan.vsplit] : 0;
    // a row's bounds, rank (read and written), out-degree and contribution; an
    // edge and its contribution
    const uint64_t row = 16 + 2 * vb_bytes + 4 + vb_bytes;
    st.run.frontier_bytes = V * (4 + 2 * vb_bytes);
    st.run.relax_static_bytes = it * (row * d->plan.vsplit + (4 + vb_bytes) * sedges);
    st.run.static_work_edges = it * sedges;
    st.run.relax_dynamic_bytes = it * (row * (V - d->plan.vsplit) + (4 + vb_bytes) * (g->E - sedges));
    if (!pp.link) st.run.relax_dynamic_bytes = 0;
    st.run.work_edges = (uint64_t)it * g->E;
    st.iterations = it;
    st.final_l1 = d->h_prstate->l1;
    st.run.iterations = it;
    st.run.reached = V;
    st.run.traversed_edges = g->E;
    st.run.node_sum = (uint64_t)it * V;
    st.run.frontier_kernel_ms = sum_ms(tc_init);
    st.run.frontier_launches = tc_init.launches;
    st.run.relax_static_kernel_ms = sum_ms(tc_static);
    st.run.relax_static_launches = !pp.link ? it : tc_static.launches;
    st.run.relax_dynamic_kernel_ms = sum_ms(tc_dyn);
    st.run.relax_dynamic_launches = tc_dyn.launches;
    st.run.copy_ms = sum_ms(tc_copy);
    st.run.pre_ms = st.run.frontier_kernel_ms;
    st.run.static_ms = st.run.relax_static_kernel_ms;
    st.run.overload_ms = st.run.relax_dynamic_kernel_ms;
    st.run.overload_move_ms = st.run.copy_ms;
    if (stats) *stats = st;
}

}  // namespace og

using namespace og;

extern "C" og_status og_pagerank(og_graph *g, const og_pr_params *params, float *ranks_f32, double *ranks_f64,
                                 og_pr_stats *stats) {
    clear_error();
    if (!g || !params) return fail(OG_EINVAL, "graph/params is NULL");
    if (!g->dev) return fail(OG_ESTATE, "og_prepare has not been called for this graph");
    if (g->kind != OG_KIND_PULL) return fail(OG_EUNSUPPORTED, "PageRank needs a pull-layout graph");
    if (!(params->damping > 0 && params->damping < 1)) return fail(OG_EINVAL, "damping must be in (0, 1)");
    if (params->max_iterations == 0) return fail(OG_EINVAL, "max_iterations must be > 0");
    int expect = 0;
    if (!g->busy.compare_exchange_strong(expect, 1)) return fail(OG_EBUSY, "graph is running another call");
    og_status st = guard([&]() -> og_status {
        OG_HIP(hipSetDevice(g->dev->device));
        if (params->fp64)
            run_pr<double>(g, *params, ranks_f64, stats);
        else
            run_pr<float>(g, *params, ranks_f32, stats);
        return OG_OK;
    });
    g->busy.store(0);
    return st;
}
