// Frontier engine for BFS, SSSP and CC on gfx950: wave64 ballot/scan frontier
// compaction, degree-binned relax kernels over the HBM-resident static region,
// and the dynamic-region loaders: the relax reads active rows where they are, in
// pinned host memory, or the host streams them through staging slots.
//
// One iteration (reference loop: BFS/oneGraph_BFS/CalculateOpt.h:75-188):
//   1. k_frontier_compact: one pass over the next-frontier flags builds the
//      static bin lists, the hub tile list, the dynamic list (in vertex order
//      within windows) and its degree prefix, and clears the flags.  Replaces K1-K6
//      (gpu_kernels.h:243-379), the host prefix H4 (CalculateOpt.h:110-123)
//      and every per-iteration .wait(): counts stay on the device, and rounds
//      without a host-side loader are replayed from captured hipGraphs.
//   2. static relax: bin 0 (lpv0 lanes/vertex), bin 1 (wave/vertex), bin 2
//      (workgroup per `tile` edges, neighbour list staged in LDS).  Replaces
//      bfs_kernelStatic (gpu_kernels.h:211-241), sssp_kernel
//      (SSSP/oneGraph/gpu_kernels.h:177-203), cc_kernelStaticSwap
//      (CC/onegraph/gpu_kernels.h:133-157).
//   3. dynamic region: an edge-parallel relax reads the active rows over the
//      link (K8/K10/K12); in pageable memory the host gathers the active edges of
//      the dynamic list into a pinned slot (H5, GraphMeta.h:470-506) and
//      hipMemcpyAsync moves the slot while the other one is being gathered.
#include <algorithm>
#include <atomic>
#include <vector>
#include <cstdio>
#include <cstring>
#include <thread>

#include "device.h"

namespace og {

// ================================================================= kernels

__global__ void k_iota(uint32_t *a, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        a[i] = (uint32_t)i;
}

__device__ __forceinline__ void clock_stamp(RoundClock *clk, int prev, int kind) {
    if (clk && blockIdx.x == 0 && threadIdx.x == 0) {
        const unsigned long long t = wall_clock64();
        atomicAdd(&clk->acc[prev], t);
        atomicAdd(&clk->acc[kind], 0ull - t);
    }
}

// Start of a single-source run, one launch: values (unreached, or with IOTA
// each vertex its own label), next-frontier flags (the source, or every
// vertex), counters, clock and traversal state.  Four vertices per lane.
template <bool IOTA>
__global__ __launch_bounds__(kBlock) void k_run_init(uint32_t *__restrict__ val, uint8_t *__restrict__ flag, uint64_t V,
                                                     uint64_t Vpad, uint32_t src, RunBlock *__restrict__ blk,
                                                     unsigned long long *__restrict__ spread, RoundCtl c) {
    const uint64_t tid = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (blockIdx.x == 0) {
        if (threadIdx.x < 16) blk->counters[threadIdx.x] = 0;
        if (threadIdx.x < 3) blk->clk.acc[threadIdx.x] = 0;
        if (threadIdx.x == 0) blk->ctl = c;
        for (uint32_t i = threadIdx.x; i < kSpreadWords; i += kBlock) spread[i] = 0;
    }
    for (uint64_t i = tid; i < Vpad / 4; i += (uint64_t)gridDim.x * kBlock) {
        const uint64_t v = 4 * i;
        uint32_t x[4], f = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool on = IOTA ? v + j < V : v + j == src;
            x[j] = IOTA ? (uint32_t)(v + j) : on ? 1u : OG_UNREACHED;
            f |= (on ? 1u : 0u) << (8 * j);
        }
        ((uint4 *)val)[i] = make_uint4(x[0], x[1], x[2], x[3]);
        ((uint32_t *)flag)[i] = f;
    }
}

// Bin of an active vertex: 0..2 static bins, 3 dynamic, 4 no out-edges,
// 5 held back for a later round (near-far order: value >= threshold, checked
// first so that held-back vertices need no degree), 6 a dynamic vertex held
// back by the deferred order.
__device__ __forceinline__ int bin_of(bool far, bool hold, uint64_t v, uint64_t vsplit, uint64_t deg,
                                      const Tuning &tn) {
    if (far) return 5;
    if (deg == 0) return 4;
    if (v >= vsplit) return hold ? 6 : 3;
    if (deg <= tn.t1) return 0;
    if (deg <= tn.t2) return 1;
    return 2;
}

// Reserves n entries with dd edges at the end of the dynamic list; the two
// counts move together, so the list's degree prefix rises with the list.
// One word holds both when they fit (count in the low dsh bits); else a lock
// guards two words: its holder waits for nothing, so every waiter gets it.
__device__ __forceinline__ void reserve_dyn(const CompactTotals &ct, uint64_t n, uint64_t dd, uint64_t &p, uint64_t &pd) {
    unsigned long long *t = ct.t;
    if (ct.dsh) {
        const uint64_t old = atomicAdd(t + kTotDyn, (unsigned long long)(n | (dd << ct.dsh)));
        p = old & ((1ull << ct.dsh) - 1);
        pd = old >> ct.dsh;
        return;
    }
    while (atomicCAS(t + kTotWide, 0ull, 1ull) != 0) __builtin_amdgcn_s_sleep(2);
    p = atomicAdd(t + kTotWide + 1, (unsigned long long)n);
    pd = atomicAdd(t + kTotWide + 2, (unsigned long long)dd);
    wait_vmem();
    atomicExch(t + kTotWide, 0ull);
}

// Totals between compactions: zero, each slot's smallest held-back value all
// ones.
__global__ void k_totals_init(unsigned long long *t, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const bool far = i >= kTotSlot && i < kTotArrive && i % kTotLine == 3;
        t[i] = far ? ~0ull : 0ull;
    }
}

// End of a compaction, run by the first wave of the workgroup that arrived
// last: takes the totals (leaving them cleared for the next compaction),
// publishes the round's summary and advances the traversal state: statistics,
// liveness, the BFS direction and, when the near set is empty but vertices
// are held back, the near-far threshold (min held-back value + delta) for
// the next compaction.  progress (pinned host memory, or null): compactions so
// far << 1 | traversal ended.
__device__ __forceinline__ void compact_finish(const CompactTotals &ct, FrontierInfo *__restrict__ info,
                                               uint64_t *__restrict__ doff, RoundCtl *__restrict__ ctl,
                                               unsigned long long *progress, bool was_heavy) {
    const uint32_t lane = threadIdx.x;
    RoundCtl c = *ctl;
    uint64_t zf = 0, sd = 0, lh = 0, mf = ~0ull, a01 = 0, ath = 0, dyn = 0, wn = 0, wd = 0;
    if (lane < kTotSlots && lane < ct.nblk) {
        unsigned long long *sl = ct.t + kTotSlot + lane * kTotLine;
        zf = atomicExch(sl + 0, 0ull);
        sd = atomicExch(sl + 1, 0ull);
        lh = atomicExch(sl + 2, 0ull);
        mf = atomicExch(sl + 3, ~0ull);
    }
    if (lane == 0) {
        a01 = atomicExch(ct.t + kTotBins, 0ull);
        ath = atomicExch(ct.t + kTotTiles, 0ull);
        if (ct.dsh) {
            dyn = atomicExch(ct.t + kTotDyn, 0ull);
            wn = dyn & ((1ull << ct.dsh) - 1);
            wd = dyn >> ct.dsh;
        } else {
            wn = atomicExch(ct.t + kTotWide + 1, 0ull);
            wd = atomicExch(ct.t + kTotWide + 2, 0ull);
        }
    }
#pragma unroll
    for (int m = 1; m < (int)kTotSlots; m <<= 1) {
        zf += shfl_xor_u64(zf, m);
        sd += shfl_xor_u64(sd, m);
        lh += shfl_xor_u64(lh, m);
        mf = min(mf, shfl_xor_u64(mf, m));
    }
    if (lane != 0) return;
    FrontierInfo fi;
    fi.n[0] = (uint32_t)a01;
    fi.n[1] = (uint32_t)(a01 >> 32);
    fi.n[2] = (uint32_t)ath;
    fi.n[3] = (uint32_t)wn;
    fi.nzero = (uint32_t)zf;
    fi.nhub = (uint32_t)(ath >> 32);
    fi.static_deg = sd;
    fi.dyn_deg = wd;
    fi.nfar = (uint32_t)(zf >> 32);
    fi.min_far = (uint32_t)min(mf, (uint64_t)0xFFFFFFFFull);
    const uint32_t lagging = (uint32_t)lh, hd = (uint32_t)(lh >> 32);
    fi.dyn_held = hd ? 1u : 0u;
    const uint64_t snodes = (uint64_t)fi.n[0] + fi.n[1] + fi.nhub;
    const uint64_t active = snodes + fi.n[3] + fi.nzero;
    // light/heavy split: light rounds count the vertices they relax (they
    // turn heavy-pending); once a bucket's light rounds find nothing near,
    // the next compaction collects the heavy-pending vertices (their
    // distances are final within the bucket) before the threshold moves
    bool heavy_next = false;
    if (c.split) {
        if (was_heavy) {
            c.hpend = 0;
        } else if (active) {
            c.hpend += active;
        } else if (c.hpend && !hd) {
            heavy_next = true;
        }
    }
    // (after a heavy round a light compaction always follows: the held-back
    // vertices sit in the other flag array)
    fi.live = (active || fi.nfar || hd || heavy_next || was_heavy) ? 1u : 0u;
    // BFS direction (Beamer et al., SC'12): bottom-up once the frontier's
    // edges exceed 1/14 of the unexplored ones, back to top-down when
    // the frontier falls below V / 24.
    fi.pull = 0;
    fi.heavy = was_heavy ? 1u : 0u;
    if (c.dir_opt && active) {
        const uint64_t mf2 = fi.static_deg + fi.dyn_deg;
        if (!c.pull && mf2 > c.unexplored / 14) c.pull = 1;
        else if (c.pull && active < c.nverts / 24) c.pull = 0;
        c.unexplored -= min(mf2, c.unexplored);
        fi.pull = c.pull;
        c.pull_rounds += c.pull;
    }
    *info = fi;
    doff[fi.n[3]] = fi.dyn_deg;
    c.compactions++;
    c.live = fi.live;
    if (active) {
        c.rounds++;
        c.node_sum += active;
        c.static_node_sum += snodes;
        c.dyn_node_sum += fi.n[3];
        c.work_edges += fi.static_deg + fi.dyn_deg;
        c.static_work_edges += fi.static_deg;
        c.dyn_rounds += fi.n[3] ? 1 : 0;
    } else if (heavy_next || hd) {
        // the threshold stays: a heavy round's offers are all >= it, and held
        // dynamic vertices are below it
    } else if (fi.nfar && c.delta) {
        // Near set empty.  Lagged order: every vertex below the threshold
        // has relaxed except the waiting dynamic ones, which go next (a
        // static vertex they improve is below the threshold and joins
        // them).  Otherwise every held-back value is >= the threshold and
        // it moves to the smallest of them + delta.
        if (lagging) c.fbound = c.thresh;
        else c.thresh = (uint32_t)min((uint64_t)0xFFFFFFFFull, (uint64_t)fi.min_far + c.delta);
    }
    // deferred order: the dynamic list is held back (its vertices stay
    // flagged) until a compaction finds nothing else to relax; kDeferOnce
    // holds it back no more after that
    if (c.defer == kDeferOnce) c.hold = c.hold && active ? 1u : 0u;
    else c.hold = c.defer == 1 && !was_heavy && active ? 1u : 0u;
    c.mode = heavy_next ? 1u : 0u;
    c.near = 0;
    *ctl = c;
    if (progress)
        __hip_atomic_store(progress, (unsigned long long)c.compactions << 1 | (fi.live ? 0u : 1u), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

// Frontier compaction, one launch: flags -> bin lists, hub tiles, the dynamic
// list with its degree prefix and chunk table (dchunk[c]: the list entry
// holding edge c * kDynEdgesPerBlock of the dynamic edge space); the window's
// flags become 1 for held-back vertices, 0 elsewhere.
//
// A workgroup takes NW windows of kCompactBlock * 4 vertices, thread t the
// four consecutive ones from 4t of each, whose flags, values and degrees are
// one 4- or 16-byte load each (consecutive lanes on consecutive addresses)
// and whose bins stay in registers.  The block's counts reserve their place in
// each list with one atomic per list: blocks land in the lists in the order
// of these atomics (within a block in vertex order, so that neighbouring
// dynamic rows share link lines), and no pass over the other blocks' counts is
// needed.  Bin 0 grows up from list[0], bin 1 down from list[vsplit - 1], the
// dynamic list up from list[vsplit].  The workgroup that arrives last finishes
// the round (compact_finish).
//
// What bounds it: on graphs up to a few million vertices, latency: launch,
// the flag -> value -> degree chain, and three round trips of device-scope
// atomics (reservation, arrival, totals).  A dense round of a larger graph is
// bound by the flag, value and degree sweeps and the list stores.  Against the
// count pass, one-workgroup scan and write pass it replaces: 1 M vertices,
// dense round 41 -> 12 us, nearly empty 16 -> 7 us; 16.7 M vertices, the 33
// compactions of an out-of-memory SSSP 1.67 -> 1.13 ms.
template <int NW>
__global__ __launch_bounds__(kCompactBlock) void k_frontier_compact(
    uint8_t *__restrict__ flag_a, uint8_t *__restrict__ hflag, uint64_t Vpad, uint64_t vsplit,
    const uint64_t *__restrict__ ptr, const uint64_t *__restrict__ pmid, const uint32_t *__restrict__ deg,
    const uint32_t *__restrict__ hdeg, Tuning tn, const uint32_t *__restrict__ val_a, RoundCtl *ctl, CompactTotals ct,
    FrontierInfo *__restrict__ info, uint32_t *__restrict__ list, uint64_t *__restrict__ hub, uint64_t hub_cap,
    uint64_t *__restrict__ doff, uint32_t *__restrict__ dchunk, uint64_t dchunk_cap, RoundClock *clk, int clk_prev,
    unsigned long long *progress) {
    constexpr int kWaves = kCompactBlock / kWave;
    static_assert(NW * kWaves <= kWave, "one lane per (window, wave)");
    __shared__ uint64_t s_cnt[NW * kWaves], s_deg[NW * kWaves];  // per window and wave: packed counts, degrees
    __shared__ uint32_t s_tile[NW * kWaves];
    __shared__ unsigned long long s_stat[2];  // static degrees, packed statistics
    __shared__ uint32_t s_more[3];            // lagging, held, smallest held-back value
    __shared__ uint64_t s_base[4];            // reserved places: bins 0 | 1, tiles, dynamic list, its edges
    clock_stamp(clk, clk_prev, kClkFront);
    // a round enqueued after the traversal ended: no vertex is flagged, and
    // the summary and the traversal state stand
    if (ctl->halt && !ctl->live) return;
    // light/heavy split: a heavy compaction collects the heavy-pending
    // vertices (no near-far test) and sizes them by their heavy edges.  It does so at
    // once when the light round before it put nothing below the threshold: its
    // sweep would find nothing near, and the next one would collect them (six of
    // the 28 rounds of an in-memory SSSP, about 13 us each: 757 -> 700 us, out of
    // memory 16.5 -> 16.3 ms).  A deferred order keeps near vertices flagged, so
    // there only the sweep can tell.
    const bool heavy = pmid && (ctl->mode || (ctl->hpend && !ctl->near && !ctl->defer));
    const bool mark = pmid && !heavy;  // light round: relaxed vertices turn heavy-pending
    uint8_t *flag = heavy ? hflag : flag_a;
    const uint32_t *val = heavy ? nullptr : val_a;
    const uint64_t v0 = ((uint64_t)blockIdx.x * NW * kCompactBlock + threadIdx.x) * 4;  // window q: v0 + q * kWin
    constexpr uint64_t kWin = (uint64_t)kCompactBlock * 4;
    uint32_t fw[NW], any = 0;
#pragma unroll
    for (int q = 0; q < NW; ++q) fw[q] = v0 + q * kWin < Vpad ? *(const uint32_t *)(flag + v0 + q * kWin) : 0u;
#pragma unroll
    for (int q = 0; q < NW; ++q) any |= fw[q];
    if (threadIdx.x < 2) s_stat[threadIdx.x] = 0;
    if (threadIdx.x < 3) s_more[threadIdx.x] = threadIdx.x == 2 ? 0xFFFFFFFFu : 0u;
    if (!__syncthreads_or(any != 0)) {  // no flags here (most blocks in a small round)
        if (threadIdx.x < kWave) {
            const bool last = threadIdx.x == 0 && arrive_last(ct);
            if (__ballot(last)) compact_finish(ct, info, doff, ctl, progress, heavy);
        }
        return;
    }
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    uint32_t bins[NW];  // byte j: bin of vertex j of the window, 7 when not flagged
    uint64_t dg[NW][4];
    uint32_t c01[NW], c3[NW], tiles[NW];  // c01: bin 0 | bin 1 << 16
    uint64_t ddeg[NW];
    uint64_t stat = 0, sdeg = 0;          // stat: zero | hub << 16 | far << 32 | lagging << 48
    uint32_t held = 0, mf = 0xFFFFFFFFu;
    const uint32_t thresh = val ? ctl->thresh : 0xFFFFFFFFu;
    const bool hold = !heavy && ctl->hold;
    // lagged order: a dynamic vertex below the threshold but not below fbound
    // waits until the static part of its bucket has settled
    const bool lagged = val && ctl->defer == 2;
    const uint32_t fbound = lagged ? ctl->fbound : 0u;
    uint4 vv[NW];
    if (val) {
#pragma unroll
        for (int q = 0; q < NW; ++q)  // (the value array is padded to Vpad entries)
            if (fw[q]) vv[q] = *(const uint4 *)(val + v0 + q * kWin);
    }
    uint32_t farm = 0;  // bit 4q + j: held back by its value
    if (val) {
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            if (!fw[q]) continue;
            const uint32_t x[4] = {vv[q].x, vv[q].y, vv[q].z, vv[q].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (!((fw[q] >> (8 * j)) & 0xFFu)) continue;
                const bool lag = lagged && x[j] < thresh && x[j] >= fbound && v0 + q * kWin + j >= vsplit;
                const bool far = x[j] >= thresh || lag;
                stat += lag ? 1ull << 48 : 0ull;
                if (far) {
                    mf = min(mf, x[j]);
                    farm |= 1u << (4 * q + j);
                }
            }
        }
    }
    auto near_any = [&](int q) {  // a vertex of window q is flagged and not held back by its value
        uint32_t f = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) f |= ((fw[q] >> (8 * j)) & 0xFFu) && !((farm >> (4 * q + j)) & 1u) ? 1u : 0u;
        return f != 0;
    };
    const uint32_t *dt = pmid && heavy ? hdeg : deg;
    const bool whole = !pmid && hdeg;  // whole rows of a split graph
#pragma unroll
    for (int q = 0; q < NW; ++q) {
#pragma unroll
        for (int j = 0; j < 4; ++j) dg[q][j] = 0;
        if (!fw[q] || !near_any(q)) continue;
        const uint64_t v = v0 + q * kWin;
        if (deg) {
            const uint4 x = *(const uint4 *)(dt + v);
            dg[q][0] = x.x;
            dg[q][1] = x.y;
            dg[q][2] = x.z;
            dg[q][3] = x.w;
            if (whole) {
                const uint4 y = *(const uint4 *)(hdeg + v);
                dg[q][0] += y.x;
                dg[q][1] += y.y;
                dg[q][2] += y.z;
                dg[q][3] += y.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if ((fw[q] >> (8 * j)) & 0xFFu) dg[q][j] = round_deg(deg, hdeg, ptr, pmid, heavy, v + j);
        }
    }
#pragma unroll
    for (int q = 0; q < NW; ++q) {
        bins[q] = 0x07070707u;
        c01[q] = c3[q] = tiles[q] = 0;
        ddeg[q] = 0;
        if (!fw[q]) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (!((fw[q] >> (8 * j)) & 0xFFu)) continue;
            const uint64_t d = dg[q][j];
            const int b = bin_of((farm >> (4 * q + j)) & 1u, hold, v0 + q * kWin + j, vsplit, d, tn);
            bins[q] ^= (uint32_t)(7 ^ b) << (8 * j);
            switch (b) {
                case 0: c01[q] += 1; sdeg += d; break;
                case 1: c01[q] += 1u << 16; sdeg += d; break;
                case 2: tiles[q] += (uint32_t)((d + tn.tile - 1) / tn.tile); stat += 1ull << 16; sdeg += d; break;
                case 3: ++c3[q]; ddeg[q] += d; break;
                case 5: stat += 1ull << 32; break;
                case 6: ++held; break;
                default: ++stat; break;
            }
        }
    }
    // inclusive scans over the wave (a block's packed counts stay below 2^16)
    uint32_t i01[NW], i3[NW], it[NW];
    uint64_t id[NW];
#pragma unroll
    for (int q = 0; q < NW; ++q) {
        i01[q] = i3[q] = it[q] = 0;
        id[q] = 0;
        if (__ballot(fw[q] != 0)) {
            i01[q] = wave_scan_u32(c01[q]);
            if (__ballot(c3[q] != 0)) {
                i3[q] = wave_scan_u32(c3[q]);
                id[q] = wave_scan_u64(ddeg[q]);
            }
            if (__ballot(tiles[q] != 0)) it[q] = wave_scan_u32(tiles[q]);
        }
        if (lane == kWave - 1) {
            s_cnt[q * kWaves + wid] = (uint64_t)i01[q] | ((uint64_t)i3[q] << 32);
            s_deg[q * kWaves + wid] = id[q];
            s_tile[q * kWaves + wid] = it[q];
        }
    }
    if (__ballot(any != 0)) {  // statistics of the wave: one LDS atomic each
        const uint64_t ws = wave_scan_u64(sdeg), wp = wave_scan_u64(stat);
        if (lane == kWave - 1) {
            if (ws) atomicAdd(&s_stat[0], (unsigned long long)ws);
            if (wp) atomicAdd(&s_stat[1], (unsigned long long)wp);
        }
        if (held) atomicAdd(&s_more[1], held);
        if (mf != 0xFFFFFFFFu) atomicMin(&s_more[2], mf);
    }
    __syncthreads();
    // prefixes of the (window, wave) pairs and the block's totals, per wave
    const bool own = lane < NW * kWaves;
    const uint64_t xc = own ? s_cnt[lane] : 0, xd = own ? s_deg[lane] : 0;
    const uint32_t xt = own ? s_tile[lane] : 0;
    const uint64_t wc = wave_scan_u64(xc), wd = wave_scan_u64(xd);
    const uint32_t wt = wave_scan_u32(xt);
    const uint64_t tc = wave_read_u64(wc, kWave - 1), td = wave_read_u64(wd, kWave - 1);
    const uint32_t tt = (uint32_t)__builtin_amdgcn_readlane((int)wt, kWave - 1);
    bool last = false;
    if (wid == 0) {
        // one lane per total, so that their round trips overlap
        const uint64_t st = s_stat[1];
        const uint32_t n0 = (uint32_t)(tc & 0xFFFFu), n1 = (uint32_t)((tc >> 16) & 0xFFFFu), n3 = (uint32_t)(tc >> 32);
        unsigned long long *sl = ct.t + kTotSlot + (blockIdx.x % kTotSlots) * kTotLine;
        unsigned long long *to = nullptr;
        uint64_t add = 0;
        switch (lane) {
            case 0: to = ct.t + kTotBins; add = n0 | (uint64_t)n1 << 32; break;
            case 1: to = ct.t + kTotTiles; add = tt | ((st >> 16) & 0xFFFFu) << 32; break;
            case 2: to = sl + 0; add = (st & 0xFFFFu) | ((st >> 32) & 0xFFFFu) << 32; break;
            case 3: to = sl + 1; add = s_stat[0]; break;
            case 4: to = sl + 2; add = (st >> 48) | (uint64_t)s_more[1] << 32; break;
            default: break;
        }
        if (add) {
            const uint64_t old = atomicAdd(to, (unsigned long long)add);
            if (lane < 2) s_base[lane] = old;
        }
        if (lane == 5 && s_more[2] != 0xFFFFFFFFu) atomicMin(sl + 3, (unsigned long long)s_more[2]);
        if (lane == 6 && n3) {
            uint64_t p, pd;
            reserve_dyn(ct, n3, td, p, pd);
            s_base[2] = p;
            s_base[3] = pd;
        }
        wait_vmem();
        last = lane == 0 && arrive_last(ct);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NW; ++q) {
        // exclusive prefix of this wave in window q
        const uint64_t pc = wave_read_u64(wc - xc, q * kWaves + wid), pw = wave_read_u64(wd - xd, q * kWaves + wid);
        const uint32_t ptile = (uint32_t)__builtin_amdgcn_readlane((int)(wt - xt), q * kWaves + wid);
        if (!fw[q]) continue;
        const uint32_t e01 = i01[q] - c01[q];
        uint64_t p0 = (uint64_t)(uint32_t)s_base[0] + (uint32_t)(pc & 0xFFFFu) + (e01 & 0xFFFFu);
        uint64_t p1 = (uint64_t)(uint32_t)(s_base[0] >> 32) + (uint32_t)((pc >> 16) & 0xFFFFu) + (e01 >> 16);
        uint64_t p2 = (uint64_t)(uint32_t)s_base[1] + ptile + (it[q] - tiles[q]);
        uint64_t p3 = s_base[2] + (uint32_t)(pc >> 32) + (i3[q] - c3[q]);
        uint64_t pd = s_base[3] + pw + (id[q] - ddeg[q]);
        uint32_t left = 0, hw = 0;  // flags left (bins 5 and 6), heavy-pending flags to set
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t v = (uint32_t)(v0 + q * kWin + j);
            const uint32_t b = (bins[q] >> (8 * j)) & 0xFFu;
            if (b <= 4) hw |= 1u << (8 * j);
            if (b == 0) {
                list[p0++] = v;
            } else if (b == 1) {
                list[vsplit - 1 - p1++] = v;
            } else if (b == 2) {
                const uint32_t nt = (uint32_t)((dg[q][j] + tn.tile - 1) / tn.tile);
                for (uint32_t i = 0; i < nt; ++i, ++p2)
                    if (p2 < hub_cap) hub[p2] = ((uint64_t)i << 32) | v;
            } else if (b == 3) {
                const uint64_t d = dg[q][j];
                list[vsplit + p3] = v;
                doff[p3] = pd;
                // the dynamic relax's chunks of kDynEdgesPerBlock edges whose
                // first edge is one of v's: they start at entry p3
                for (uint64_t c = (pd + kDynEdgesPerBlock - 1) / kDynEdgesPerBlock;
                     c * kDynEdgesPerBlock < pd + d && c < dchunk_cap; ++c)
                    dchunk[c] = (uint32_t)p3;
                ++p3;
                pd += d;
            } else if (b == 5 || b == 6) {
                left |= 1u << (8 * j);
            }
        }
        if (left != fw[q]) *(uint32_t *)(flag + v0 + q * kWin) = left;
        // (the word belongs to this thread alone)
        if (mark && hw) *(uint32_t *)(hflag + v0 + q * kWin) |= hw;
    }
    if (wid == 0 && __ballot(last)) compact_finish(ct, info, doff, ctl, progress, heavy);
}

// Traversal state at the start: near-far width `delta` with the first
// threshold 1 + delta (the source's value is 1), or none for delta = 0;
// `defer` 1 holds the dynamic list back in rounds with static work, 2 lets
// dynamic vertices relax only once the static part of their bucket settled,
// kDeferOnce holds them back until the static region has settled once;
// dir_opt_edges > 0 turns on the BFS direction choice over that many edges;
// split: light/heavy split rounds (the graph's pmid rows; SSSP near-far).
static RoundCtl ctl_begin(uint64_t V, uint32_t delta, uint32_t defer, uint64_t dir_opt_edges, bool split) {
    RoundCtl c{};
    c.split = split ? 1u : 0u;
    c.delta = delta;
    c.defer = defer;
    c.dir_opt = dir_opt_edges ? 1u : 0u;
    c.unexplored = dir_opt_edges;
    c.nverts = V;
    c.thresh = delta ? (uint32_t)std::min<uint64_t>(0xFFFFFFFFull, 1ull + delta) : 0xFFFFFFFFu;
    c.fbound = 0;
    c.hold = defer == 1 || defer == kDeferOnce ? 1u : 0u;
    c.live = 1;
    c.halt = 1;
    return c;
}

// ---------------------------------------------------------------- relax

template <int ALGO>
__device__ __forceinline__ uint32_t offer(uint32_t du, uint32_t wt) {
    if (ALGO == ALGO_BFS) return du + 1;
    if (ALGO == ALGO_SSSP) {
        // distance + 1 saturates at 0xFFFFFFFE (0xFFFFFFFF means unreached):
        // min() is monotone, so the fixed point is min(dist + 1, 0xFFFFFFFE)
        const uint64_t s = (uint64_t)du + wt;
        return s > 0xFFFFFFFEull ? 0xFFFFFFFEu : (uint32_t)s;
    }
    return du;
}

// What a frontier vertex carries to its out-edges: its value, or for the
// multi-source BFS the mask of sources whose frontier holds it.
template <int H>
struct MaskOf {
    uint64_t m[H];
    MaskOf() = default;
    __device__ __forceinline__ MaskOf(int) {
#pragma unroll
        for (int h = 0; h < H; ++h) m[h] = 0;
    }
    __device__ __forceinline__ bool any() const {
        uint64_t x = 0;
#pragma unroll
        for (int h = 0; h < H; ++h) x |= m[h];
        return x != 0;
    }
};
template <int ALGO> struct SrcOf { using T = uint32_t; };
template <> struct SrcOf<ALGO_MSBFS> { using T = MaskOf<1>; };
template <> struct SrcOf<ALGO_MSBFS2> { using T = MaskOf<2>; };

// Whether a frontier vertex has anything to offer in this round.
template <int ALGO>
__device__ __forceinline__ bool offers(const typename SrcOf<ALGO>::T &s) {
    if constexpr (ms_masks(ALGO) != 0) return s.any();
    else return true;
}

template <int ALGO>
__device__ __forceinline__ typename SrcOf<ALGO>::T load_src(const RelaxArgs &a, uint32_t u) {
    if constexpr (ms_masks(ALGO) != 0) {
        constexpr int H = ms_masks(ALGO);
        MaskOf<H> s;
#pragma unroll
        for (int h = 0; h < H; ++h) s.m[h] = a.front[(uint64_t)u * H + h];
        if (H == 1 && a.pull) s.m[0] &= ~*a.pull;
        return s;
    }
    else return a.val[u];
}

// Relaxing an edge (u -> to, wt) is split in two so that a lane can keep the
// reads of several edges in flight before its first atomic: peek() reads the
// target's state, commit() compares the offers with what peek saw and applies
// them.  Values only decrease (masks only grow), so a stale peek can cost an
// atomic that finds nothing to do but never loses an update.
template <int ALGO>
__device__ __forceinline__ typename SrcOf<ALGO>::T peek(const RelaxArgs &a, uint32_t to) {
    if constexpr (ms_masks(ALGO) != 0) {
        constexpr int H = ms_masks(ALGO);
        MaskOf<H> s;
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const ulonglong2 x = a.vn[(uint64_t)to * H + h];
            s.m[h] = x.x | x.y;
        }
        return s;
    }
    else return a.val[to];
}

// A relax kernel's start and end: the threshold that an improvement is compared
// with, and whether any of the wave's fell below it (every writer stores the
// same).  Once per wave: read and noted beside each atomic they cost the dense
// rounds of an in-memory SSSP a tenth.
template <int ALGO>
__device__ __forceinline__ void relax_begin(const RelaxArgs &a) {
    a.near = 0;
    a.thresh = ALGO == ALGO_SSSP && a.ctl ? a.ctl->thresh : 0u;
}

template <int ALGO>
__device__ __forceinline__ void relax_end(const RelaxArgs &a) {
    if (ALGO == ALGO_SSSP && __ballot(a.near != 0) && threadIdx.x % kWave == 0) a.ctl->near = 1;
}

// Applies N offers of a lane (edge k valid when bit k of `ok` is set, its
// source's state src(k)) and returns how many improved their target (which is
// then flagged for the next frontier).
// BFS writes the same level from every writer in an iteration, so a plain
// store is race-free (a visited bitmap claimed with atomicOr, one writer per
// vertex, was measured slower on R-MAT 20: 14.7 vs 17.2 GTEPS); SSSP/CC use
// atomicMin so no smaller offer is lost (the reference's check-then-write in
// K7/K11 can lose one).  With AGAIN a lane first reads the targets that its
// peeks would improve once more, at the place where the device's atomics are
// performed: a peek may come from a copy in this XCD's L2 that keeps the value
// of the kernel's start, and atomics on one line queue at about 12 ns each.
// It pays beside the link's latency, in the dynamic region (out-of-memory SSSP
// R-MAT 16.7 M 16.75 -> 16.05 ms, CC 3 M 6.55 -> 6.32 ms), and costs a round trip
// elsewhere (SSSP in memory 0.77 -> 0.83 ms).  Multi-source: the sources of u's frontier that have neither reached `to`
// nor been offered to it are OR-ed into vn[to].y (one 64-bit atomic for all 64
// searches).  The two masks share a 16-byte load: with the offers unseen, every
// edge of a dense round into a well-connected vertex repeated its atomic (R-MAT
// 4 M vertices, 64 sources, the three dense rounds: 3.75, 2.43, 1.69 -> 1.86,
// 1.84, 1.70 ms, the last ones the link's; 128 sources 1.87, 1.82, 1.75).
template <int ALGO, int N, bool AGAIN = false, class Src>
__device__ __forceinline__ uint32_t commit(const RelaxArgs &a, Src src, const uint32_t (&to)[N], const uint32_t (&wt)[N],
                                           const typename SrcOf<ALGO>::T (&seen)[N], uint32_t ok) {
    uint32_t c = 0;
    if constexpr (ms_masks(ALGO) != 0) {
        constexpr int H = ms_masks(ALGO);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            if (!((ok >> k) & 1)) continue;
            const MaskOf<H> s = src(k);
            bool any = false;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const uint64_t m = s.m[h] & ~seen[k].m[h];
                if (!m) continue;
                atomicOr(&a.vn[(uint64_t)to[k] * H + h].y, (unsigned long long)m);
                any = true;
            }
            if (!any) continue;
            a.flag[to[k]] = 1;
            ++c;
        }
    } else if constexpr (ALGO == ALGO_BFS) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const uint32_t nd = offer<ALGO>(src(k), wt[k]);
            if (!((ok >> k) & 1) || nd >= seen[k]) continue;
            a.val[to[k]] = nd;
            a.flag[to[k]] = 1;
            ++c;
        }
    } else {
        uint32_t nd[N], x[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            nd[k] = offer<ALGO>(src(k), wt[k]);
            if (nd[k] >= seen[k]) ok &= ~(1u << k);
        }
        if (!ok) return 0;
        if constexpr (AGAIN) {
#pragma unroll
            for (int k = 0; k < N; ++k) {
                x[k] = 0;
                if ((ok >> k) & 1) x[k] = __hip_atomic_load(a.val + to[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
#pragma unroll
            for (int k = 0; k < N; ++k)
                if (nd[k] >= x[k]) ok &= ~(1u << k);
            if (!ok) return 0;
        }
        // all atomics before the first result is used
#pragma unroll
        for (int k = 0; k < N; ++k)
            if ((ok >> k) & 1) x[k] = atomicMin(a.val + to[k], nd[k]);
#pragma unroll
        for (int k = 0; k < N; ++k)
            if (((ok >> k) & 1) && nd[k] < x[k]) {
                a.flag[to[k]] = 1;
                ++c;
                a.near |= nd[k] < a.thresh ? 1u : 0u;
            }
    }
    return c;
}

// The relax kernels read their work counts from the round's FrontierInfo on
// the device and stride over them, so a launch needs no host-side count: a
// round can be enqueued (or captured in a graph) before its compaction ran.

// Bins 0 and 1: LPV lanes per frontier vertex (LPV = 64: one wave).  `bin`
// selects the list segment: item i of bin 0 at list[i], of bin 1 at
// list[vsplit - 1 - i].
// The bodies take the workgroup's index and the number of workgroups of its
// kind (bid, nb), so that one launch can run several kinds side by side.
template <int ALGO, bool W, bool PK, int LPV>
__device__ __forceinline__ uint32_t relax_group_body(const uint32_t *__restrict__ list, uint64_t vsplit, int bin,
                                                     const FrontierInfo *__restrict__ info,
                                                     const uint64_t *__restrict__ ptr, const void *__restrict__ edges,
                                                     const RelaxArgs &a, uint32_t bid, uint32_t nb) {
    if (info->pull) return 0;
    const bool heavy = info->heavy != 0;
    const uint32_t n = info->n[bin];
    const uint32_t sub = threadIdx.x % LPV;
    const uint64_t stride = (uint64_t)nb * (kBlock / LPV);
    uint32_t cnt = 0;
    for (uint64_t item = ((uint64_t)bid * kBlock + threadIdx.x) / LPV; item < n; item += stride) {
        const uint32_t u = list[bin ? vsplit - 1 - item : item];
        uint64_t b, e;
        row_range(ptr, a.pmid, heavy, u, b, e);
        const auto s = load_src<ALGO>(a, u);
        if (!offers<ALGO>(s)) continue;  // all of u's sources go bottom-up this round
        for (uint64_t i = b + sub; i < e; i += (uint64_t)kRelaxBatch * LPV) {
            uint32_t to[kRelaxBatch], wt[kRelaxBatch];
            typename SrcOf<ALGO>::T seen[kRelaxBatch];
#pragma unroll
            for (int k = 0; k < kRelaxBatch; ++k) {
                to[k] = 0;
                wt[k] = 0;
                if (i + (uint64_t)k * LPV < e) load_edge<W, PK>(edges, i + (uint64_t)k * LPV, a.wbits, to[k], wt[k]);
            }
            uint32_t ok = 0;
#pragma unroll
            for (int k = 0; k < kRelaxBatch; ++k) {
                seen[k] = 0;
                if (i + (uint64_t)k * LPV < e) {
                    seen[k] = peek<ALGO>(a, to[k]);
                    ok |= 1u << k;
                }
            }
            cnt += commit<ALGO, kRelaxBatch>(a, [&](int) { return s; }, to, wt, seen, ok);
        }
    }
    return cnt;
}

template <int ALGO, bool W, bool PK, int LPV>
__global__ __launch_bounds__(kBlock) void k_relax_group(const uint32_t *__restrict__ list, uint64_t vsplit, int bin,
                                                        const FrontierInfo *__restrict__ info,
                                                        const uint64_t *__restrict__ ptr,
                                                        const void *__restrict__ edges, RelaxArgs a,
                                                        unsigned long long *spread) {
    relax_begin<ALGO>(a);
    wave_count(spread, kUpdStatic, relax_group_body<ALGO, W, PK, LPV>(list, vsplit, bin, info, ptr, edges, a, blockIdx.x, gridDim.x));
    relax_end<ALGO>(a);
}

template <int ALGO, bool W, bool PK>
__device__ __forceinline__ uint32_t relax_hub_body(const uint64_t *__restrict__ hub, uint64_t hub_cap,
                                                   const FrontierInfo *__restrict__ info, uint32_t tile,
                                                   const uint64_t *__restrict__ ptr, const void *__restrict__ edges,
                                                   const RelaxArgs &a, uint32_t *s_edges, uint32_t bid, uint32_t nb) {
    constexpr bool WIDE = W && !PK;  // 8-byte edges
    const uint64_t ntiles = info->pull ? 0 : min((uint64_t)info->n[2], hub_cap);
    const bool heavy = info->heavy != 0;
    uint32_t c = 0;
    for (uint64_t ti = bid; ti < ntiles; ti += nb) {
        const uint64_t it = hub[ti];
        const uint32_t u = (uint32_t)it, t = (uint32_t)(it >> 32);
        uint64_t rb, re;
        row_range(ptr, a.pmid, heavy, u, rb, re);
        const uint64_t b = rb + (uint64_t)t * tile;
        const uint64_t e = min(re, b + tile);
        const uint32_t cnt = (uint32_t)(e - b);
        const auto s = load_src<ALGO>(a, u);
        if (!offers<ALGO>(s)) continue;  // block-uniform: u is the same for every thread
        for (uint32_t k = threadIdx.x; k < cnt; k += kBlock) {
            if (WIDE)
                ((uint2 *)s_edges)[k] = ((const uint2 *)edges)[b + k];
            else
                s_edges[k] = ((const uint32_t *)edges)[b + k];
        }
        __syncthreads();
        for (uint32_t k0 = threadIdx.x; k0 < cnt; k0 += kRelaxBatch * kBlock) {
            uint32_t to[kRelaxBatch], wt[kRelaxBatch];
            typename SrcOf<ALGO>::T seen[kRelaxBatch];
#pragma unroll
            for (int j = 0; j < kRelaxBatch; ++j) {
                to[j] = 0;
                wt[j] = 0;
                if (k0 + j * kBlock < cnt) load_edge<W, PK>(s_edges, k0 + j * kBlock, a.wbits, to[j], wt[j]);
            }
            uint32_t ok = 0;
#pragma unroll
            for (int j = 0; j < kRelaxBatch; ++j) {
                seen[j] = 0;
                if (k0 + j * kBlock < cnt) {
                    seen[j] = peek<ALGO>(a, to[j]);
                    ok |= 1u << j;
                }
            }
            c += commit<ALGO, kRelaxBatch>(a, [&](int) { return s; }, to, wt, seen, ok);
        }
        __syncthreads();  // the tile buffer is reused by the next tile
    }
    return c;
}

// Bin 2: one workgroup per tile of a hub's neighbour list (workgroups stride
// over the tiles); the tile is staged in LDS with coalesced loads before the
// relax pass.
template <int ALGO, bool W, bool PK>
__global__ __launch_bounds__(kBlock) void k_relax_hub(const uint64_t *__restrict__ hub, uint64_t hub_cap,
                                                      const FrontierInfo *__restrict__ info, uint32_t tile,
                                                      const uint64_t *__restrict__ ptr,
                                                      const void *__restrict__ edges, RelaxArgs a,
                                                      unsigned long long *spread) {
    extern __shared__ uint32_t s_edges[];
    relax_begin<ALGO>(a);
    wave_count(spread, kUpdStatic, relax_hub_body<ALGO, W, PK>(hub, hub_cap, info, tile, ptr, edges, a, s_edges, blockIdx.x, gridDim.x));
    relax_end<ALGO>(a);
}

// Dynamic region, edges [c0, min(c1, D)) of the concatenated active dynamic
// edge space (D = sum of the dynamic list's degrees; the list sits at
// list[vsplit, vsplit + n3)).  STAGED (DIRECT = false): they sit in a
// staging slot, edge q at q - c0.  DIRECT: edge q of vertex u is CSR edge
// x = ptr[u] + (q - doff[i]); when u's chunk of kResChunk vertices is
// resident in HBM (rdelta[u >> kResChunkShift] != kNotResident) it is read
// from `resident` at x + rdelta, else in place from the pinned host array
// through its device mapping (`stage`, at x - dbase, whole edges or with
// lbits a stream of lbits-bit words); reads served from HBM are counted in
// *hits.  (Storing the host rows in
// order of distance from a hub instead of vertex order was measured slower
// on R-MAT: the active list stays in vertex order, so neighbouring lanes then
// read scattered rows.)
// Each workgroup takes chunks of kDynEdgesPerBlock consecutive edges, loads
// the covering slice of the degree prefix into LDS and maps each edge to its
// source with a binary search there (every listed vertex has >= 1 edge, so a
// chunk covers at most kDynEdgesPerBlock vertices).  With the compaction's
// chunk table (dchunk, zero-copy rounds: chunks start at edge 0) the slice's
// first and last entries are two loads; the staged loader's slots start
// anywhere, so it finds them by binary search over the degree prefix.
// LDS of the dynamic relax body: the degree-prefix slice and its bounds
struct DynLds {
    uint64_t off[kDynEdgesPerBlock + 2];
    uint32_t i[2];
};

template <int ALGO, bool W, bool PACKED, bool DIRECT>
__device__ __forceinline__ uint32_t relax_dyn_body(const uint32_t *__restrict__ list,
                                                   const FrontierInfo *__restrict__ info,
                                                   const uint64_t *__restrict__ doff, const void *__restrict__ stage,
                                                   uint64_t c0, uint64_t c1max, const uint64_t *__restrict__ ptr,
                                                   uint64_t dbase, const void *__restrict__ resident,
                                                   const int64_t *__restrict__ rdelta, uint32_t wbits,
                                                   const RelaxArgs &a, const uint64_t *__restrict__ lpos,
                                                   uint64_t nl, uint64_t vsplit, const uint32_t *__restrict__ dchunk,
                                                   uint32_t lbits, DynLds &L, uint32_t bid, uint32_t nb, uint32_t &hits) {
    uint64_t *s_off = L.off;
    uint32_t *s_i = L.i;
    const uint32_t ndyn = info->n[3];
    const uint32_t *dlist = list + vsplit;
    const uint64_t c1 = min(c1max, info->dyn_deg);
    const bool heavy = info->heavy != 0;
    uint32_t c = 0, h = 0;
    for (uint64_t q0 = c0 + (uint64_t)bid * kDynEdgesPerBlock; q0 < c1; q0 += (uint64_t)nb * kDynEdgesPerBlock) {
        const uint64_t q1 = min(q0 + kDynEdgesPerBlock, c1);
        if (dchunk) {  // chunks aligned to the table (c0 = 0): two loads
            if (threadIdx.x < 2) {
                const uint64_t k = q0 / kDynEdgesPerBlock + threadIdx.x;
                // the entry holding q1 (or the last entry): one past the chunk's last edge at most
                s_i[threadIdx.x] = threadIdx.x == 1 && q1 >= info->dyn_deg ? ndyn - 1 : dchunk[k];
            }
        } else if (threadIdx.x < 2) {
            const uint64_t q = threadIdx.x == 0 ? q0 : q1 - 1;
            uint32_t lo = 0, hi = ndyn;  // largest i with doff[i] <= q; doff[0] = 0
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (doff[mid] <= q) lo = mid; else hi = mid;
            }
            s_i[threadIdx.x] = lo;
        }
        __syncthreads();
        const uint32_t i0 = s_i[0];
        const uint32_t nv = s_i[1] - i0 + 1;
        for (uint32_t k = threadIdx.x; k <= nv; k += kBlock) s_off[k] = doff[i0 + k];
        __syncthreads();
        // all edge (and source-state) reads of the lane first, then the
        // target peeks, then the commits: the link / HBM latencies overlap
        uint32_t to[kDynEdgesPerThread], wt[kDynEdgesPerThread];
        typename SrcOf<ALGO>::T sv[kDynEdgesPerThread], seen[kDynEdgesPerThread];
#pragma unroll
        for (int j = 0; j < kDynEdgesPerThread; ++j) {
            const uint64_t q = q0 + threadIdx.x + (uint64_t)j * kBlock;
            to[j] = 0;
            wt[j] = 0;
            sv[j] = 0;
            if (q < q1) {
                uint32_t lo = 0, hi = nv;
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (s_off[mid] <= q) lo = mid; else hi = mid;
                }
                const uint32_t u = dlist[i0 + lo];
                sv[j] = load_src<ALGO>(a, u);
                if (DIRECT) {
                    // hp: position of the edge in the host copy of the region
                    const uint64_t k = q - s_off[lo];
                    uint64_t hp;
                    uint64_t slot = u >> kResChunkShift;  // entry of the resident table
                    if (lpos) {  // split layout: light parts, then heavy parts
                        const uint64_t lp = lpos[u - vsplit];
                        const uint64_t hb = nl + (ptr[u] - dbase) - lp;
                        bool hv;
                        if (a.pmid) {  // a split round reads one part
                            hv = heavy;
                            hp = (hv ? hb : lp) + k;
                        } else {  // whole rows: the light part, then the heavy part
                            const uint64_t nlu = lpos[u - vsplit + 1] - lp;
                            hv = k >= nlu;
                            hp = hv ? hb + (k - nlu) : lp + k;
                        }
                        slot = 2 * slot + (hv ? 1 : 0);
                    } else {
                        hp = ((a.pmid && heavy) ? a.pmid[u] : ptr[u]) - dbase + k;
                    }
                    const int64_t dl = rdelta ? rdelta[slot] : kNotResident;
                    if (dl != kNotResident) {
                        load_edge<W, PACKED>(resident, (uint64_t)((int64_t)hp + dl), wbits, to[j], wt[j]);
                        ++h;
                    } else if (lbits) {
                        const uint32_t x = link_word((const uint32_t *)stage, hp, lbits);
                        to[j] = W ? x >> wbits : x;
                        wt[j] = W ? x & ((1u << wbits) - 1u) : 1u;
                    } else {
                        load_edge<W, PACKED>(stage, hp, wbits, to[j], wt[j]);
                    }
                } else {
                    load_edge<W, PACKED>(stage, q - c0, wbits, to[j], wt[j]);
                }
            }
        }
        uint32_t ok = 0;
#pragma unroll
        for (int j = 0; j < kDynEdgesPerThread; ++j) {
            seen[j] = 0;
            if (q0 + threadIdx.x + (uint64_t)j * kBlock < q1) {
                seen[j] = peek<ALGO>(a, to[j]);
                ok |= 1u << j;
            }
        }
        c += commit<ALGO, kDynEdgesPerThread, true>(a, [&](int j) { return sv[j]; }, to, wt, seen, ok);
        __syncthreads();  // s_off / s_i are reloaded for the next chunk
    }
    hits = h;
    return c;
}

template <int ALGO, bool W, bool PACKED, bool DIRECT>
__global__ __launch_bounds__(kBlock) void k_relax_dyn(const uint32_t *__restrict__ list,
                                                      const FrontierInfo *__restrict__ info,
                                                      const uint64_t *__restrict__ doff,
                                                      const void *__restrict__ stage, uint64_t c0, uint64_t c1max,
                                                      const uint64_t *__restrict__ ptr, uint64_t dbase,
                                                      const void *__restrict__ resident,
                                                      const int64_t *__restrict__ rdelta,
                                                      uint32_t wbits, RelaxArgs a, const uint64_t *__restrict__ lpos,
                                                      uint64_t nl, uint64_t vsplit, const uint32_t *__restrict__ dchunk,
                                                      uint32_t lbits, unsigned long long *spread) {
    __shared__ DynLds L;
    uint32_t h = 0;
    relax_begin<ALGO>(a);
    const uint32_t c = relax_dyn_body<ALGO, W, PACKED, DIRECT>(list, info, doff, stage, c0, c1max, ptr, dbase, resident,
                                                               rdelta, wbits, a, lpos, nl, vsplit, dchunk, lbits, L,
                                                               blockIdx.x, gridDim.x, h);
    relax_end<ALGO>(a);
    wave_count(spread, kUpdDynamic, c);
    if (DIRECT) wave_count(spread, kHbmEdges, h);
}

// One round's relax in a single launch: static bins 0 and 1, hub tiles and
// the zero-copy dynamic region side by side, so a device-driven round needs
// no second stream (the fork and join of which cost tens of microseconds per
// round in a replayed graph, most of a small round).  A workgroup takes its
// kind from blockIdx.x modulo a period of kFuseStatic + cd workgroups (2
// bin 0, 2 bin 1, 1 hub tile, cd dynamic): the kinds interleave in dispatch
// order, so the link-bound dynamic relax and the static bins progress
// together as the two streams did.  With K = gridDim.x / period, the kinds
// get 2K, 2K, K and cd * K workgroups.  A graph wholly in HBM runs it with
// cd = 0: its three static bins in one launch instead of three.
struct RoundRelax {
    const uint32_t *list;
    const FrontierInfo *info;
    const uint64_t *ptr;
    const void *sedges;         // static region
    const uint64_t *hub;
    uint64_t hub_cap;
    uint32_t tile;
    uint32_t cd;                // dynamic workgroups per period
    const uint64_t *doff;
    const void *stage;          // dynamic region in pinned host memory (device address)
    uint64_t dbase;
    const void *resident;       // resident chunks in HBM
    const int64_t *rdelta;
    const uint64_t *lpos;       // split layout of the host copy (null: rows whole)
    const uint32_t *dchunk;     // chunk table of the dynamic edge space
    uint32_t lbits;             // bits per edge of the dynamic region in host memory (0: whole edges)
    uint64_t nl, vsplit;
    unsigned long long *spread;  // work counters
    RoundClock *clk;            // null: not timed
};
constexpr uint32_t kFuseStatic = 5;

template <int ALGO, bool W, bool PK, int LPV>
__global__ __launch_bounds__(kBlock) void k_relax_round(RoundRelax r, RelaxArgs a) {
    extern __shared__ uint64_t s_fuse[];
    clock_stamp(r.clk, kClkFront, kClkRelax);
    relax_begin<ALGO>(a);
    const uint32_t P = kFuseStatic + r.cd;
    const uint32_t K = gridDim.x / P;
    const uint32_t k = blockIdx.x / P, j = blockIdx.x - k * P;
    if (j < 2) {
        wave_count(r.spread, kUpdStatic,
                 relax_group_body<ALGO, W, PK, LPV>(r.list, r.vsplit, 0, r.info, r.ptr, r.sedges, a, 2 * k + j, 2 * K));
    } else if (j < 4) {
        wave_count(r.spread, kUpdStatic,
                 relax_group_body<ALGO, W, PK, 64>(r.list, r.vsplit, 1, r.info, r.ptr, r.sedges, a, 2 * k + j - 2, 2 * K));
    } else if (j == 4) {
        wave_count(r.spread, kUpdStatic, relax_hub_body<ALGO, W, PK>(r.hub, r.hub_cap, r.info, r.tile, r.ptr, r.sedges, a,
                                                              (uint32_t *)s_fuse, k, K));
    } else {
        uint32_t h = 0;
        const uint32_t c = relax_dyn_body<ALGO, W, PK, true>(r.list, r.info, r.doff, r.stage, 0, ~0ull, r.ptr, r.dbase,
                                                             r.resident, r.rdelta, a.wbits, a, r.lpos, r.nl, r.vsplit,
                                                             r.dchunk, r.lbits, *(DynLds *)s_fuse, r.cd * k + (j - kFuseStatic),
                                                             r.cd * K, h);
        wave_count(r.spread, kUpdDynamic, c);
        wave_count(r.spread, kHbmEdges, h);
    }
    relax_end<ALGO>(a);
}

// Served BFS (the query server's 64-slot engines): bottom-up scan for the
// pulling slots P = *pull.  Every vertex that some slot of P has not reached
// scans its in-edges, ORing the frontier masks of its in-neighbours
// (restricted to those slots), and stops once every such slot is found.
// Found slots are offered through vn[v].y like a top-down relax.
__device__ __forceinline__ void srv_pull_body(const SrvPull &p, uint32_t bid, uint32_t nb) {
    const uint64_t P = *p.pull;
    if (!P) return;
    for (uint64_t v = (uint64_t)bid * kBlock + threadIdx.x; v < p.V; v += (uint64_t)nb * kBlock) {
        const uint64_t need = P & ~p.vn[v].x;
        if (!need) continue;
        uint64_t acc = 0;
        const uint64_t b = p.in_ptr[v], e = p.in_ptr[v + 1];
        for (uint64_t i = b; i < e && acc != need; i += kRelaxBatch) {
            uint32_t u[kRelaxBatch];
#pragma unroll
            for (int k = 0; k < kRelaxBatch; ++k) u[k] = i + k < e ? p.in_cols[i + k] : 0u;
#pragma unroll
            for (int k = 0; k < kRelaxBatch; ++k)
                if (i + k < e) acc |= p.front[u[k]] & need;
        }
        if (acc) {
            atomicOr(&p.vn[v].y, (unsigned long long)acc);
            p.flag[v] = 1;
        }
    }
}

// A served BFS round's relax in one launch: the top-down slots through the
// static bins (as k_relax_round with cd = 0) and, beside them, the bottom-up
// scan of the pulling slots (cp workgroups per period of kFuseStatic + cp).
// The two only read the reached and frontier masks and only OR into the offers
// and set flags, so
// they may run side by side.
template <bool W, bool PK, int LPV>
__global__ __launch_bounds__(kBlock) void k_srv_round(RoundRelax r, RelaxArgs a, SrvPull p, uint32_t cp) {
    extern __shared__ uint64_t s_fuse[];
    const uint32_t P = kFuseStatic + cp;
    const uint32_t K = gridDim.x / P;
    const uint32_t k = blockIdx.x / P, j = blockIdx.x - k * P;
    if (j < 2) {
        wave_count(r.spread, kUpdStatic, relax_group_body<ALGO_MSBFS, W, PK, LPV>(r.list, r.vsplit, 0, r.info, r.ptr, r.sedges, a,
                                                                         2 * k + j, 2 * K));
    } else if (j < 4) {
        wave_count(r.spread, kUpdStatic, relax_group_body<ALGO_MSBFS, W, PK, 64>(r.list, r.vsplit, 1, r.info, r.ptr, r.sedges, a,
                                                                        2 * k + j - 2, 2 * K));
    } else if (j == 4) {
        wave_count(r.spread, kUpdStatic, relax_hub_body<ALGO_MSBFS, W, PK>(r.hub, r.hub_cap, r.info, r.tile, r.ptr, r.sedges,
                                                                    a, (uint32_t *)s_fuse, k, K));
    } else {
        srv_pull_body(p, cp * k + (j - kFuseStatic), cp * K);
    }
}

// Bottom-up BFS round (direction-optimising BFS, Beamer et al., SC'12): the
// frontier is the current level L = rounds so far; every unvisited vertex
// scans its in-edges, kRelaxBatch parents' levels at a time, and takes level
// L + 1 at the first parent on level L.  Each vertex is written by its own
// lane only, and a fresh L + 1 never reads as L, so no atomics are needed.
__global__ __launch_bounds__(kBlock) void k_bfs_pull(const uint64_t *__restrict__ in_ptr,
                                                     const uint32_t *__restrict__ in_cols, uint64_t V,
                                                     const FrontierInfo *__restrict__ info,
                                                     const RoundCtl *__restrict__ ctl, uint32_t *val,
                                                     uint8_t *__restrict__ flag, unsigned long long *spread) {
    if (!info->pull) return;
    const uint32_t L = ctl->rounds;
    uint32_t c = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * kBlock + threadIdx.x; v < V; v += (uint64_t)gridDim.x * kBlock) {
        if (val[v] != OG_UNREACHED) continue;
        const uint64_t b = in_ptr[v], e = in_ptr[v + 1];
        for (uint64_t i = b; i < e; i += kRelaxBatch) {
            uint32_t lv[kRelaxBatch];
#pragma unroll
            for (int k = 0; k < kRelaxBatch; ++k) lv[k] = i + k < e ? val[in_cols[i + k]] : 0u;
            bool hit = false;
#pragma unroll
            for (int k = 0; k < kRelaxBatch; ++k) hit |= lv[k] == L;
            if (hit) {
                val[v] = L + 1;
                flag[v] = 1;
                ++c;
                break;
            }
        }
    }
    wave_count(spread, kUpdStatic, c);
}

// Order-independent digest of a result array: the sum (mod 2^64) of
// mix64(v << 32 | value[v]) over reached vertices.
__device__ __forceinline__ uint64_t d_mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// counters[2..4]: reached = #{v : val[v] != UNREACHED}, traversed = sum of
// their degrees, checksum = digest of val; folds the run's work counters.
// deg / hdeg: the degree table (hdeg: heavy degrees with the split, else
// null), or null for the row bounds.  With the table, each lane reads four
// values and four degrees per 16-byte load.  Few, large workgroups
// (stats_grid): each ends with three device-scope atomics on one line, which
// queue at about 12 ns each (1024 workgroups of 256: 41 us at 1 M vertices).
// ctl, when given: nothing is summed while the traversal has a frontier.
constexpr int kStatsBlock = 1024;
__global__ __launch_bounds__(kStatsBlock) void k_reach_stats(const uint32_t *__restrict__ val,
                                                             const uint64_t *__restrict__ ptr,
                                                             const uint32_t *__restrict__ deg,
                                                             const uint32_t *__restrict__ hdeg, uint64_t V,
                                                             unsigned long long *counters, unsigned long long *spread,
                                                             RoundClock *clk, const RoundCtl *ctl = nullptr) {
    if (ctl && ctl->live) return;
    __shared__ unsigned long long s_sum[3];
    if (threadIdx.x < 3) s_sum[threadIdx.x] = 0;
    clock_stamp(clk, kClkFront, kClkOther);
    __syncthreads();
    uint64_t r = 0, t = 0, h = 0;
    const uint64_t tid = (uint64_t)blockIdx.x * kStatsBlock + threadIdx.x,
                   nth = (uint64_t)gridDim.x * kStatsBlock;
    auto add = [&](uint64_t v, uint32_t x, uint64_t dv) {
        if (x != OG_UNREACHED) {
            ++r;
            t += dv;
            h += d_mix64((v << 32) | x);
        }
    };
    uint64_t v0 = 0;  // first vertex of the scalar tail
    if (deg) {
        // val and the table are 16-byte aligned allocations; the table is
        // padded to a multiple of 16 entries
        const uint64_t n4 = V / 4;
        // two chunks per lane per step, their loads issued together
        for (uint64_t q0 = tid; q0 < n4; q0 += 2 * nth) {
            uint4 x[2], dl[2], dh[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint64_t q = q0 + k * nth;
                const bool in = q < n4;
                x[k] = in ? ((const uint4 *)val)[q] : make_uint4(OG_UNREACHED, OG_UNREACHED, OG_UNREACHED, OG_UNREACHED);
                dl[k] = in ? ((const uint4 *)deg)[q] : make_uint4(0, 0, 0, 0);
                dh[k] = in && hdeg ? ((const uint4 *)hdeg)[q] : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint64_t q = q0 + k * nth;
                add(4 * q + 0, x[k].x, (uint64_t)dl[k].x + dh[k].x);
                add(4 * q + 1, x[k].y, (uint64_t)dl[k].y + dh[k].y);
                add(4 * q + 2, x[k].z, (uint64_t)dl[k].z + dh[k].z);
                add(4 * q + 3, x[k].w, (uint64_t)dl[k].w + dh[k].w);
            }
        }
        v0 = 4 * n4;
    }
    for (uint64_t v = v0 + tid; v < V; v += nth) {
        const uint32_t x = val[v];
        add(v, x, deg ? (uint64_t)deg[v] + (hdeg ? hdeg[v] : 0u) : (x != OG_UNREACHED ? ptr[v + 1] - ptr[v] : 0));
    }
    const uint64_t w[3] = {wave_scan_u64(r), wave_scan_u64(t), wave_scan_u64(h)};
    if ((threadIdx.x & (kWave - 1)) == kWave - 1)
#pragma unroll
        for (int i = 0; i < 3; ++i) atomicAdd(&s_sum[i], (unsigned long long)w[i]);
    __syncthreads();
    if (threadIdx.x < 3 && s_sum[threadIdx.x]) atomicAdd(counters + 2 + threadIdx.x, s_sum[threadIdx.x]);
    if (blockIdx.x == 0) fold_spread(spread, counters);
}

// ----------------------------------------------------------- small graphs
//
// A whole traversal in one launch of one workgroup, for graphs whose values fit
// its LDS.  Values, the frontier bitmaps and the round's queue live in LDS, so a
// round costs two barriers instead of two launches, and nothing but rows is
// read from memory; the end writes the result, the digest and the statistics,
// to pinned host memory too, so that the host waits for one flag.  What bounds
// it: the latency of row bounds and edges on a few hundred rows in flight, and one
// compute unit's load rate, hence the limits.  Measured through the binding
// (R-MAT, one launch / rounds): BFS 1000 vertices 12 K edges 45 / 152 us, 8000 /
// 108 K 104 / 167, 16384 / 228 K 170 / 166; SSSP 4000 / 52 K 117 / 353, 16384 /
// 228 K 380 / 414, 330 K 548 / 464; CC, whose first rounds relax every vertex,
// 8000 / 168 K 118 / 170 but 16384 / 58 K 289 / 272.
// SSSP relaxes every improved vertex in the next round here, whatever the
// bucket width.  On deep graphs that is mostly the faster way too (one launch /
// near-far rounds at delta 256, ms: a path of 16384 53 / 235, a grid of
// 128 x 128 1.8 / 4.9, 16000 x 12 random near neighbours on a ring 3.6 / 5.3),
// but not where shorter hops keep improving every long one (v to v + j at weight
// j * j: 4000 vertices x 40 160 / 57, 1000 x 196 21 / 15, 500 x 390 5.7 / 7.6).
constexpr uint32_t kSmallV = 1u << 14;
constexpr uint32_t kSmallVcc = 1u << 13;
constexpr uint64_t kSmallE = 3u << 16;
constexpr int kSmallBlock = 1024;
constexpr uint32_t kSmallMid = 32, kSmallLong = 512;  // rows: 8 lanes, a wave, the workgroup

struct SmallArgs {
    const uint64_t *ptr;
    const void *edges;
    uint32_t wbits, V, src;
    uint32_t *val;             // V values out
    uint32_t *host;            // and here (pinned host memory) unless null
    RunBlock *blk, *h_blk;     // statistics (h_blk: pinned, or null)
    unsigned long long *done;  // pinned flag raised to 1 at the end, or null
    bool check;                // offsets that do not run from 0 to E: no run, they are left in counters[14..15]
    uint64_t E;
};

constexpr size_t small_lds(uint64_t V) { return 4 * V + 8 * ((V + 31) / 32) + 2 * ((V + 1) / 2 * 2); }

template <int ALGO, bool W, bool PK>
__global__ __launch_bounds__(kSmallBlock) void k_small(SmallArgs a) {
    extern __shared__ uint32_t s_mem[];
    __shared__ uint32_t s_n[4];                       // rows of the round: short, wave, workgroup, without edges
    __shared__ unsigned long long s_tot[6];           // updates, edges, vertices; reached, traversed, digest
    __shared__ uint16_t s_long[kSmallE / kSmallLong];
    const unsigned long long t0 = wall_clock64();
    if (a.check) {
        const uint64_t p0 = a.ptr[0], p1 = a.ptr[a.V];
        if (threadIdx.x == 0) {
            a.blk->counters[14] = p0;
            a.blk->counters[15] = p1;
        }
        if (p0 != 0 || p1 != a.E) return;
    }
    const uint32_t V = a.V, nw = (V + 31) / 32, tid = threadIdx.x, lane = tid & (kWave - 1);
    uint32_t *val = s_mem, *cur = val + V, *nxt = cur + nw;
    uint16_t *q = (uint16_t *)(nxt + nw);  // short rows from the front, wave rows from the back
    for (uint32_t v = tid; v < V; v += kSmallBlock) val[v] = ALGO == ALGO_CC ? v : v == a.src ? 1u : OG_UNREACHED;
    for (uint32_t i = tid; i < nw; i += kSmallBlock) {
        if (ALGO == ALGO_CC) cur[i] = i + 1 < nw || V % 32 == 0 ? 0xFFFFFFFFu : (1u << (V % 32)) - 1u;
        else cur[i] = i == a.src / 32 ? 1u << (a.src % 32) : 0u;
        nxt[i] = 0;
    }
    if (tid < 6) s_tot[tid] = 0;
    uint32_t upd = 0, rounds = 0, nodes = 0, empty = 0;
    uint64_t work = 0;
    // offers N edges of a lane
    auto relax = [&](auto &to, auto &wt, uint32_t ok, uint32_t du) {
        constexpr int N = sizeof(to) / sizeof(uint32_t);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const uint32_t nd = offer<ALGO>(du, wt[k]);
            if (!((ok >> k) & 1) || nd >= val[to[k]]) continue;
            if (nd < atomicMin(&val[to[k]], nd)) {
                atomicOr(&nxt[to[k] / 32], 1u << (to[k] % 32));
                ++upd;
            }
        }
    };
    auto row = [&](uint32_t u, uint32_t sub, uint32_t L) {
        const uint64_t b = a.ptr[u], e = a.ptr[u + 1];
        const uint32_t du = val[u];
        for (uint64_t i = b + sub; i < e; i += (uint64_t)kRelaxBatch * L) {
            uint32_t to[kRelaxBatch], wt[kRelaxBatch], ok = 0;
#pragma unroll
            for (int k = 0; k < kRelaxBatch; ++k) {
                to[k] = wt[k] = 0;
                if (i + (uint64_t)k * L < e) {
                    load_edge<W, PK>(a.edges, i + (uint64_t)k * L, a.wbits, to[k], wt[k]);
                    ok |= 1u << k;
                }
            }
            relax(to, wt, ok, du);
        }
    };
    for (;;) {
        if (tid < 4) s_n[tid] = 0;
        __syncthreads();
        // the round's queues, four vertices of a lane in flight
        for (uint32_t v0 = 0; v0 < V; v0 += 4 * kSmallBlock) {
            uint64_t b[4], e[4];
            bool on[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t v = v0 + k * kSmallBlock + tid;
                on[k] = v < V && (cur[v / 32] >> (v % 32)) & 1;
                b[k] = on[k] ? a.ptr[v] : 0;
                e[k] = on[k] ? a.ptr[v + 1] : 0;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (!__ballot(on[k])) continue;
                const uint64_t d = e[k] - b[k];
                work += d;
                const int c = !on[k] ? 4 : d == 0 ? 3 : d <= kSmallMid ? 0 : d <= kSmallLong ? 1 : 2;
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const uint64_t m = __ballot(c == x);
                    if (!m) continue;
                    uint32_t at = 0;
                    if (lane == 0) at = atomicAdd(&s_n[x], (uint32_t)__popcll(m));
                    at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
                    at += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
                    if (c != x || x == 3) continue;
                    const uint16_t v = (uint16_t)(v0 + k * kSmallBlock + tid);
                    if (x == 0) q[at] = v;
                    else if (x == 1) q[V - 1 - at] = v;
                    else if (at < kSmallE / kSmallLong) s_long[at] = v;  // (always, but for offsets that fall)
                }
            }
        }
        __syncthreads();
        const uint32_t n0 = s_n[0], n1 = s_n[1], n2 = min(s_n[2], (uint32_t)(kSmallE / kSmallLong)), nz = s_n[3];
        if (!(n0 | n1 | n2 | nz)) break;
        ++rounds;
        nodes += n0 + n1 + n2 + nz;
        empty += nz;
        for (uint32_t i = tid; i < nw; i += kSmallBlock) cur[i] = 0;
        for (uint32_t i = 0; i < n2; ++i) row(s_long[i], tid, kSmallBlock);
        for (uint32_t i = tid / kWave; i < n1; i += kSmallBlock / kWave) row(q[V - 1 - i], lane, kWave);
        // short rows, two per group of lanes in flight
        constexpr uint32_t L = 8, G = kSmallBlock / L;
        for (uint32_t i = tid / L; i < n0; i += 2 * G) {
            uint32_t to[2][kSmallMid / L], wt[2][kSmallMid / L], ok[2] = {0, 0}, u[2] = {0, 0};
            uint64_t b[2], e[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const bool in = i + r * G < n0;
                u[r] = in ? q[i + r * G] : 0;
                b[r] = in ? a.ptr[u[r]] : 0;
                e[r] = in ? a.ptr[u[r] + 1] : 0;
            }
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int k = 0; k < (int)(kSmallMid / L); ++k) {
                    const uint64_t x = b[r] + tid % L + (uint64_t)k * L;
                    to[r][k] = wt[r][k] = 0;
                    if (x < e[r]) {
                        load_edge<W, PK>(a.edges, x, a.wbits, to[r][k], wt[r][k]);
                        ok[r] |= 1u << k;
                    }
                }
#pragma unroll
            for (int r = 0; r < 2; ++r) relax(to[r], wt[r], ok[r], val[u[r]]);
        }
        __syncthreads();
        uint32_t *t = cur;
        cur = nxt;
        nxt = t;
    }
    // the result and its sums
    uint64_t reached = 0, trav = 0, dig = 0;
    for (uint32_t v = tid; v < V; v += kSmallBlock) {
        const uint32_t x = val[v];
        a.val[v] = x;
        if (a.host) a.host[v] = x;
        if (x != OG_UNREACHED) {
            ++reached;
            trav += a.ptr[v + 1] - a.ptr[v];
            dig += d_mix64(((uint64_t)v << 32) | x);
        }
    }
    const uint64_t sums[5] = {wave_scan_u64(upd), wave_scan_u64(work), wave_scan_u64(reached), wave_scan_u64(trav),
                              wave_scan_u64(dig)};
    if (lane == kWave - 1)
#pragma unroll
        for (int i = 0; i < 5; ++i) atomicAdd(&s_tot[i], (unsigned long long)sums[i]);
    if (a.done) __threadfence_system();
    __syncthreads();
    if (tid != 0) return;
    auto fill = [&](RunBlock *o) {
        RoundCtl c{};
        c.rounds = rounds;
        c.compactions = rounds + 1;
        c.halt = 1;
        c.nverts = V;
        c.node_sum = nodes;
        c.static_node_sum = nodes - empty;
        c.work_edges = c.static_work_edges = s_tot[1];
        o->ctl = c;
        o->clk.acc[kClkRelax] = wall_clock64() - t0;
        o->clk.acc[kClkFront] = o->clk.acc[kClkOther] = 0;
        for (int i = 0; i < 14; ++i) o->counters[i] = 0;
        o->counters[kUpdStatic] = s_tot[0];
        o->counters[2] = s_tot[2];
        o->counters[3] = s_tot[3];
        o->counters[4] = s_tot[4];
    };
    if (a.h_blk) fill(a.h_blk);
    else fill(a.blk);
    if (a.done) {
        __threadfence_system();
        __hip_atomic_store(a.done, 1ull, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Launches k_small on s; its dynamic LDS exceeds what a kernel gets unasked.
template <int ALGO, bool W, bool PK>
static void launch_small(const SmallArgs &a, hipStream_t s) {
    static std::atomic<uint64_t> asked{0};  // devices, by bit
    int dev = 0;
    OG_HIP(hipGetDevice(&dev));
    const uint64_t bit = dev < 64 ? 1ull << dev : 0;
    if (!(asked.load(std::memory_order_acquire) & bit)) {
        OG_HIP(hipFuncSetAttribute((const void *)k_small<ALGO, W, PK>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)small_lds(kSmallV)));
        asked.fetch_or(bit, std::memory_order_release);
    }
    hipLaunchKernelGGL((k_small<ALGO, W, PK>), dim3(1), dim3(kSmallBlock), small_lds(a.V), s, a);
    OG_HIP(hipGetLastError());
}

// ------------------------------------------------------- multi-source BFS

// Workgroups of the commit sweep at most: each keeps its own partial sums.
constexpr unsigned kMsCommitGrid = 2048;
// A wave's reached vertices (< 2^20 of them each round: V < 2^32 over at least
// the grid's waves) and their degrees share a word; a graph has under 2^44 edges.
constexpr int kMsFcShift = 44;
constexpr int kMsGroups = 4;  // groups of 64 vertices per wave whose reads are in flight together
constexpr int kMsSums = 3 * kMsWidth;  // digest, reached, traversed per source

// Start of a batch, one launch: masks, flags and partial sums cleared, the
// traversal state set (levels, when kept, are cleared apart).
template <int H>
__global__ __launch_bounds__(kBlock) void k_ms_clear(ulonglong2 *__restrict__ vn, uint64_t *__restrict__ front,
                                                     uint8_t *__restrict__ flag, uint64_t V, uint64_t Vpad,
                                                     unsigned long long *__restrict__ part, uint64_t nparts,
                                                     RoundCtl *ctl, RoundCtl c) {
    const uint64_t tid = (uint64_t)blockIdx.x * kBlock + threadIdx.x, nth = (uint64_t)gridDim.x * kBlock;
    if (tid == 0) *ctl = c;
    for (uint64_t v = tid; v < H * V; v += nth) {
        vn[v] = make_ulonglong2(0, 0);
        front[v] = 0;
    }
    for (uint64_t i = tid; i < Vpad / 16; i += nth) ((uint4 *)flag)[i] = make_uint4(0, 0, 0, 0);
    for (uint64_t i = tid; i < nparts; i += nth) part[i] = 0;
}

// Seeds up to 64 H sources: bit j % 64 of mask j / 64 of source j, level 1,
// and its terms in the sums of the first workgroup.
template <int H>
__global__ void k_ms_init(const uint32_t *__restrict__ src, uint32_t n, ulonglong2 *vn, uint64_t *front, uint8_t *flag,
                          uint8_t *lvl, uint64_t V, const uint64_t *__restrict__ ptr, unsigned long long *part) {
    const uint32_t j = threadIdx.x % kMsWidth, h = threadIdx.x / kMsWidth;
    if (threadIdx.x < n) {
        const uint32_t s = src[threadIdx.x];
        const uint64_t at = (uint64_t)s * H + h;
        atomicOr(&vn[at].x, 1ull << j);
        atomicOr((unsigned long long *)(front + at), 1ull << j);
        flag[s] = 1;
        if (lvl) lvl[((uint64_t)h * V + s) * kMsWidth + j] = 1;
        part += h * kMsSums;
        part[j] = d_mix64(((uint64_t)s << 32) | 1u);
        part[kMsWidth + j] = 1;
        part[2 * kMsWidth + j] = ptr[s + 1] - ptr[s];
    }
}

// After a round: for every flagged vertex, the offered sources it had not
// seen become its new frontier mask and get the round's level (rounds with
// active vertices so far + 1, read from the device state; a level past 255
// sets ctl->overflow); vertices with nothing new leave the frontier.  A wave
// takes 64 vertices; the new sources of one vertex are handled side by side,
// lane = source: the lane adds the vertex to its source's digest, reached and
// traversed sums (so the results need no pass over the levels) and, when the
// caller wants levels, the row of 64 is stored as one line.  What bounds a
// dense round is the instructions per vertex: its digest term, the same for
// every source, is computed with lane = vertex, and its mask of new sources is
// the lanes that add it (R-MAT 4 M vertices, 64 sources, a dense round: 290 us
// with the terms per source, 172 now; one lane per vertex with a loop over
// its sources and byte stores took 640, and a digest pass at the end 757).  The sums of a
// workgroup go to its own slots of `part`.
template <bool LEVELS, int H>
__global__ __launch_bounds__(kBlock) void k_ms_commit(uint8_t *__restrict__ flag, uint64_t V, ulonglong2 *__restrict__ vn,
                                                      uint64_t *__restrict__ front, uint8_t *__restrict__ lvl,
                                                      const uint64_t *__restrict__ ptr,
                                                      const uint32_t *__restrict__ deg,
                                                      const uint32_t *__restrict__ hdeg, RoundCtl *ctl,
                                                      unsigned long long *__restrict__ part, RoundClock *clk) {
    constexpr int G = kMsGroups / H;
    __shared__ unsigned long long s_sum[H * kMsSums];
    clock_stamp(clk, kClkRelax, kClkOther);
    for (int i = threadIdx.x; i < H * kMsSums; i += kBlock) s_sum[i] = 0;
    const uint32_t lv32 = ctl->rounds + 1;
    const uint32_t level = min(lv32, 255u);
    const int lane = threadIdx.x & (kWave - 1);
    const uint64_t nwaves = (uint64_t)gridDim.x * (kBlock / kWave);
    uint64_t sum[H], fc[H];  // digest; reached << kMsFcShift | traversed
#pragma unroll
    for (int h = 0; h < H; ++h) sum[h] = fc[h] = 0;
    __syncthreads();
    for (uint64_t g0 = (uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; g0 * kWave < V;
         g0 += G * nwaves) {
        bool on[G];
        uint64_t nw[G][H], dv[G], mix[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const uint64_t v = (g0 + k * nwaves) * kWave + lane;
            on[k] = v < V && flag[v];
        }
        ulonglong2 x[G][H];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const uint64_t v = (g0 + k * nwaves) * kWave + lane;
#pragma unroll
            for (int h = 0; h < H; ++h) x[k][h] = on[k] ? vn[v * H + h] : make_ulonglong2(0, 0);
            dv[k] = on[k] ? round_deg(deg, hdeg, ptr, nullptr, false, v) : 0;
        }
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const uint64_t v = (g0 + k * nwaves) * kWave + lane;
            uint64_t any = 0;
#pragma unroll
            for (int h = 0; h < H; ++h) any |= nw[k][h] = x[k][h].y & ~x[k][h].x;
            mix[k] = d_mix64((v << 32) | level);
            dv[k] |= 1ull << kMsFcShift;
            if (!on[k]) continue;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                vn[v * H + h] = make_ulonglong2(x[k][h].x | nw[k][h], 0);
                front[v * H + h] = nw[k][h];
            }
            if (!any) flag[v] = 0;
        }
#pragma unroll
        for (int k = 0; k < G; ++k)
#pragma unroll
            for (int h = 0; h < H; ++h) {
                uint64_t todo = __ballot(nw[k][h] != 0);
                if (todo && lv32 > 255) ctl->overflow = 1;
                while (todo) {
                    const int l = __builtin_ctzll(todo);
                    todo &= todo - 1;
                    const uint64_t m = wave_read_u64(nw[k][h], l), d = wave_read_u64(dv[k], l), z = wave_read_u64(mix[k], l);
                    if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                        sum[h] += z;
                        fc[h] += d;
                        if (LEVELS)
                            lvl[((uint64_t)h * V + (g0 + k * nwaves) * kWave + l) * kMsWidth + lane] = (uint8_t)level;
                    }
                }
            }
    }
#pragma unroll
    for (int h = 0; h < H; ++h)
        if (__ballot(fc[h] != 0)) {
            unsigned long long *const o = s_sum + h * kMsSums;
            atomicAdd(&o[lane], (unsigned long long)sum[h]);
            atomicAdd(&o[kMsWidth + lane], (unsigned long long)(fc[h] >> kMsFcShift));
            atomicAdd(&o[2 * kMsWidth + lane], (unsigned long long)(fc[h] & ((1ull << kMsFcShift) - 1)));
        }
    __syncthreads();
    for (int i = threadIdx.x; i < H * kMsSums; i += kBlock)
        if (s_sum[i]) part[(uint64_t)blockIdx.x * H * kMsSums + i] += s_sum[i];
}

// The sources' sums over the commit's workgroups; folds the batch's work
// counters.
__global__ __launch_bounds__(1024) void k_ms_sum(const unsigned long long *__restrict__ part, uint32_t n,
                                                 unsigned long long *out, unsigned long long *counters,
                                                 unsigned long long *spread, RoundClock *clk) {
    __shared__ uint64_t s[1024];
    clock_stamp(clk, kClkFront, kClkOther);
    const uint32_t col = blockIdx.x * kMsWidth + threadIdx.x % kMsWidth;
    if (blockIdx.x == 0) fold_spread(spread, counters);
    uint64_t x = 0;
    const uint64_t row = (uint64_t)gridDim.x * kMsWidth;  // a workgroup of this kernel per 64 sums
    for (uint32_t b = threadIdx.x / kMsWidth; b < n; b += 1024 / kMsWidth) x += part[b * row + col];
    s[threadIdx.x] = x;
    __syncthreads();
    if (threadIdx.x < kMsWidth) {
        for (int k = 1; k < 1024 / kMsWidth; ++k) x += s[threadIdx.x + k * kMsWidth];
        out[col] = x;
    }
}

// Levels of sources j0 .. j0 + nj - 1 as u32 in the single-source convention,
// one row of V per source: a workgroup turns the 64-byte rows of 64 vertices
// through LDS, so that both sides move whole lines (a pass per source read
// every row's line for one byte of it).
__global__ __launch_bounds__(kBlock) void k_ms_extract(const uint8_t *__restrict__ lvl, uint64_t V, uint32_t j0, uint32_t nj,
                                                       uint32_t *__restrict__ out) {
    __shared__ uint32_t s_row[kWave][kMsWidth / 4 + 1];
    for (uint64_t v0 = (uint64_t)blockIdx.x * kWave; v0 < V; v0 += (uint64_t)gridDim.x * kWave) {
        const uint32_t r = threadIdx.x / 4, q = threadIdx.x % 4;
        const uint4 x = v0 + r < V ? ((const uint4 *)(lvl + (v0 + r) * kMsWidth))[q] : make_uint4(0, 0, 0, 0);
        s_row[r][4 * q + 0] = x.x;
        s_row[r][4 * q + 1] = x.y;
        s_row[r][4 * q + 2] = x.z;
        s_row[r][4 * q + 3] = x.w;
        __syncthreads();
        const uint64_t v = v0 + threadIdx.x % kWave;
        for (uint32_t j = threadIdx.x / kWave; j < nj; j += kBlock / kWave) {
            const uint32_t js = j0 + j;
            const uint32_t l = (s_row[threadIdx.x % kWave][js / 4] >> (8 * (js % 4))) & 0xFFu;
            if (v < V) out[(uint64_t)j * V + v] = l ? l : OG_UNREACHED;
        }
        __syncthreads();
    }
}

// ============================================================ host driver

static unsigned fill_grid(uint64_t n) { return (unsigned)std::min<uint64_t>(8192, std::max<uint64_t>(1, (n + 255) / 256)); }

void wait_progress(const unsigned long long *p, unsigned long long want, hipStream_t s) {
    for (uint64_t i = 1;; ++i) {
        const unsigned long long now = __atomic_load_n(p, __ATOMIC_ACQUIRE);
        if (now >= want || (now & 1)) return;
        if (i % 1024) {
            __builtin_ia32_pause();
            continue;
        }
        const hipError_t e = hipStreamQuery(s);  // about every 40 us: also how a device error ends the wait
        if (e == hipSuccess) return;
        if (e != hipErrorNotReady) OG_HIP(e);
        if (i >= (1u << 16)) std::this_thread::sleep_for(std::chrono::microseconds(20));
    }
}

static unsigned stats_grid(uint64_t V) {
    return (unsigned)std::min<uint64_t>(256, std::max<uint64_t>(1, (V + 8 * kStatsBlock - 1) / (8 * kStatsBlock)));
}

void device_state_free(DeviceState *d) {
    if (!d) return;
    if (d->s_compute) (void)hipStreamSynchronize(d->s_compute);
    if (d->s_copy) (void)hipStreamSynchronize(d->s_copy);
    if (d->s_static) (void)hipStreamSynchronize(d->s_static);
    for (hipEvent_t e : d->ev_h2d) (void)hipEventDestroy(e);
    for (hipEvent_t e : d->ev_relax) (void)hipEventDestroy(e);
    d->mem.release();
    // (a lane runs everything on one stream: s_copy and s_static alias it)
    if (d->s_copy && d->s_copy != d->s_compute) (void)hipStreamDestroy(d->s_copy);
    if (d->s_static && d->s_static != d->s_compute) (void)hipStreamDestroy(d->s_static);
    if (d->s_compute) (void)hipStreamDestroy(d->s_compute);
    for (hipEvent_t e : d->ev_chunk)
        if (e) (void)hipEventDestroy(e);
    if (d->ev_static) (void)hipEventDestroy(d->ev_static);
    if (d->ev_fork) (void)hipEventDestroy(d->ev_fork);
    delete d;
}

// Result copy-backs up to kOutMax bytes: the device writes slabs of kOutSlab
// bytes into pinned staging, one workgroup each, and raises the slab's flag; host
// threads copy slabs out while later ones cross the link.  (A copy into pageable
// memory goes through the runtime's own staging, a megabyte at a time with about
// 70 us between: 4 MB 236 us, this way 145.)  Larger results go through two
// pinned chunks that the copy engine fills in turn (64 MB: 47 GB/s, the slabs 44).
constexpr size_t kOutSlab = 32u << 10;
constexpr size_t kOutMax = 8u << 20;
constexpr size_t kOutChunk = 8u << 20;

__global__ __launch_bounds__(kBlock) void k_export(const uint32_t *__restrict__ src, uint64_t nwords,
                                                   uint32_t *__restrict__ dst, unsigned long long *flag,
                                                   unsigned long long seq) {
    constexpr uint32_t kWords = kOutSlab / 4, kPer = kWords / 4 / kBlock;
    const uint64_t w0 = (uint64_t)blockIdx.x * kWords;
    const uint32_t n = (uint32_t)min((uint64_t)kWords, nwords - w0);
    const uint4 *from = (const uint4 *)(src + w0);
    uint4 *to = (uint4 *)(dst + w0);
    uint4 x[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k)
        if (threadIdx.x + k * kBlock < n / 4) x[k] = from[threadIdx.x + k * kBlock];
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k)
        if (threadIdx.x + k * kBlock < n / 4) to[threadIdx.x + k * kBlock] = x[k];
    if (threadIdx.x < n % 4) dst[w0 + n / 4 * 4 + threadIdx.x] = src[w0 + n / 4 * 4 + threadIdx.x];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flag + blockIdx.x, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr size_t kOutAlone = 256u << 10;  // results up to here are copied out by the calling thread alone

OutStage::~OutStage() {
    pool.reset();
    if (buf) (void)hipHostFree(buf);
    if (flag) (void)hipHostFree(flag);
}

bool OutStage::reserve(size_t n, unsigned threads) {
    if (n > kOutMax) return false;
    const size_t want = n <= kOutAlone ? kOutAlone : kOutMax;
    auto pinned = [](size_t b) -> void * {
        void *p = nullptr;
        if (hipHostMalloc(&p, b, hipHostMallocDefault) == hipSuccess) return p;
        (void)hipGetLastError();
        return nullptr;
    };
    if (want > bytes) {
        char *p = (char *)pinned(want);
        if (!p) return false;
        if (buf) (void)hipHostFree(buf);
        buf = p;
        bytes = want;
    }
    if (!flag) {
        const size_t fb = kOutMax / kOutSlab * sizeof(unsigned long long);
        flag = (unsigned long long *)pinned(fb);
        if (!flag) return false;
        std::memset(flag, 0, fb);
    }
    if (n > kOutAlone && threads > 1 && !pool) pool.reset(new WorkerPool(std::min(4u, default_threads())));
    return true;
}

// The process's staging.
static std::shared_ptr<OutStage> out_stage() {
    static std::mutex mu;
    static std::weak_ptr<OutStage> shared;
    std::lock_guard<std::mutex> lk(mu);
    std::shared_ptr<OutStage> o = shared.lock();
    if (!o) shared = o = std::make_shared<OutStage>();
    return o;
}

// The staging with room for a result of n bytes, taken; or not (no lock): in
// use, or no memory.
static std::unique_lock<std::mutex> take_stage(DeviceState *d, size_t n) {
    if (!d->out) d->out = out_stage();
    std::unique_lock<std::mutex> use(d->out->use, std::try_to_lock);
    if (use.owns_lock() && !d->out->reserve(n, d->host_threads)) use.unlock();
    return use;
}

static void copy_chunks_to_host(DeviceState *d, void *dst, const void *src, size_t n, hipStream_t s) {
    for (auto &p : d->h_chunk)
        if (!p) p = d->palloc(kOutChunk);
    for (auto &e : d->ev_chunk)
        if (!e) OG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (!d->pool) d->pool.reset(new WorkerPool(d->host_threads));
    const size_t nch = (n + kOutChunk - 1) / kOutChunk;
    auto issue = [&](size_t k) {
        const size_t off = k * kOutChunk, len = std::min(kOutChunk, n - off);
        OG_HIP(hipMemcpyAsync(d->h_chunk[k & 1], (const char *)src + off, len, hipMemcpyDeviceToHost, s));
        OG_HIP(hipEventRecord(d->ev_chunk[k & 1], s));
    };
    issue(0);
    for (size_t k = 0; k < nch; ++k) {
        // chunk k + 1 reuses the buffer chunk k - 1 left: its host copy ended
        // in the previous iteration
        if (k + 1 < nch) issue(k + 1);
        OG_HIP(hipEventSynchronize(d->ev_chunk[k & 1]));
        const size_t off = k * kOutChunk, len = std::min(kOutChunk, n - off);
        const char *from = (const char *)d->h_chunk[k & 1];
        char *to = (char *)dst + off;
        const unsigned T = d->pool->size();
        d->pool->run([&](unsigned t) {
            const size_t a = len * t / T, b = len * (t + 1) / T;
            std::memcpy(to + a, from + a, b - a);
        });
    }
}

void copy_to_host(DeviceState *d, void *dst, const void *src, size_t n, hipStream_t s) {
    if (!n) return;
    if (n > kOutMax) return copy_chunks_to_host(d, dst, src, n, s);
    const std::unique_lock<std::mutex> use = take_stage(d, n);
    if (!use.owns_lock()) {
        OG_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s));
        OG_HIP(hipStreamSynchronize(s));
        return;
    }
    OutStage &o = *d->out;
    const size_t slabs = (n + kOutSlab - 1) / kOutSlab;
    const unsigned long long seq = ++o.seq;
    hipLaunchKernelGGL(k_export, dim3((unsigned)slabs), dim3(kBlock), 0, s, (const uint32_t *)src, (uint64_t)(n / 4),
                       (uint32_t *)o.buf, o.flag, seq);
    OG_HIP(hipGetLastError());
    std::atomic<size_t> next{0}, copied{0};
    std::atomic<int> failed{hipSuccess};
    // thread 0 asks the stream now and then: a device error ends every wait
    auto pause = [&](unsigned t, uint64_t spins) {
        if (spins % 2048) {
            __builtin_ia32_pause();
            return;
        }
        if (t == 0) {
            const hipError_t e = hipStreamQuery(s);
            if (e != hipSuccess && e != hipErrorNotReady) failed.store(e);
        }
        std::this_thread::yield();
    };
    // (the pool is the process's: of its threads as many as this preparation may use)
    const unsigned threads = n > kOutAlone && o.pool ? std::min(o.pool->size(), d->host_threads) : 1;
    auto work = [&](unsigned t) {
        if (t >= threads) return;
        for (size_t i = next.fetch_add(1); i < slabs; i = next.fetch_add(1)) {
            for (uint64_t spins = 1; __atomic_load_n(o.flag + i, __ATOMIC_ACQUIRE) != seq; ++spins) {
                if (failed.load(std::memory_order_relaxed)) return;
                pause(t, spins);
            }
            const size_t off = i * kOutSlab;
            std::memcpy((char *)dst + off, o.buf + off, std::min(kOutSlab, n - off));
            copied.fetch_add(1);
        }
        if (t == 0)
            for (uint64_t spins = 1; copied.load() < slabs && !failed.load(); ++spins) pause(t, spins);
    };
    if (threads > 1) o.pool->run(work);
    else work(0);
    if (failed.load()) {  // slabs are missing, also if the stream recovers
        (void)hipStreamSynchronize(s);
        OG_HIP((hipError_t)failed.load());
    }
}

// Largest number of hub tiles any frontier can produce for the current tuning.
static uint64_t hub_capacity(const og_graph *g, uint64_t vsplit, const Tuning &tn) {
    uint64_t cap = 0;
    for (uint64_t v = 0; v < vsplit; ++v) {
        uint64_t deg = g->ptr[v + 1] - g->ptr[v];
        if (deg > tn.t2) cap += (deg + tn.tile - 1) / tn.tile;
    }
    return cap;
}

void frontier_alloc(DeviceState *d, const og_graph *g, Frontier &f, MemPool &m) {
    const uint64_t V = d->V;
    f.flag = (uint8_t *)m.dalloc(d->Vpad);
    if (d->d_pmid) {
        f.hflag = (uint8_t *)m.dalloc(d->Vpad);
        OG_HIP(hipMemset(f.hflag, 0, d->Vpad));
    }
    f.list = (uint32_t *)m.dalloc(V * sizeof(uint32_t));
    f.doff = (uint64_t *)m.dalloc((V + 1) * sizeof(uint64_t));
    // chunk table of the dynamic relax: the dynamic edge space of a round is
    // at most the dynamic region's edges
    const uint64_t dyn_edges = d->plan.vsplit < V ? g->E - g->ptr[d->plan.vsplit] : 0;
    f.dchunk_cap = dyn_edges / kDynEdgesPerBlock + 2;
    f.dchunk = (uint32_t *)m.dalloc(f.dchunk_cap * sizeof(uint32_t));
    f.nw = (uint32_t)compact_nw(V);
    f.nblk = (uint32_t)((d->Vpad + verts_per_block(f.nw) - 1) / verts_per_block(f.nw));
    f.V = V;
    f.tot = (unsigned long long *)m.dalloc(totals_words(f.nblk) * 8);
    // dynamic list: its count and its edges in one word when they fit
    const uint32_t nb = bits_of(V - d->plan.vsplit), eb = bits_of(dyn_edges);
    f.dsh = nb + eb <= 64 && nb < 64 && !(d->flags & OG_PLAN_TEST_WIDE_LISTS) ? std::max(nb, 1u) : 0;
    hipLaunchKernelGGL(k_totals_init, dim3(fill_grid(totals_words(f.nblk))), dim3(256), 0, d->s_compute, f.tot,
                       totals_words(f.nblk));
    OG_HIP(hipGetLastError());
    OG_HIP(hipStreamSynchronize(d->s_compute));
    f.info = (FrontierInfo *)m.dalloc(sizeof(FrontierInfo));
    f.blk = (RunBlock *)m.dalloc(sizeof(RunBlock));
    f.ctl = &f.blk->ctl;
    f.clk = &f.blk->clk;
    f.counters = f.blk->counters;
    f.spread = (unsigned long long *)m.dalloc(kSpreadWords * 8);
    OG_HIP(hipMemset(f.spread, 0, kSpreadWords * 8));
    f.h_info = (FrontierInfo *)m.palloc(sizeof(FrontierInfo));
    f.h_blk = (RunBlock *)m.palloc(sizeof(RunBlock));
    f.h_progress = (unsigned long long *)m.palloc(sizeof(unsigned long long));
    const uint64_t cap = std::max<uint64_t>(hub_capacity(g, d->plan.vsplit, d->tune), 1);
    f.hub = (uint64_t *)m.dalloc(cap * sizeof(uint64_t));
    f.hub_cap = cap;
    OG_HIP(hipMemset(f.flag, 0, d->Vpad));
    RoundCtl c{};
    c.thresh = 0xFFFFFFFFu;
    OG_HIP(hipMemcpy(f.ctl, &c, sizeof c, hipMemcpyHostToDevice));
}

void frontier_compact(DeviceState *d, Frontier &f, hipStream_t s, const uint32_t *val, bool to_host,
                      const uint64_t *pmid, RoundClock *clk, int prev, unsigned long long *progress) {
    // the degree table (a split round needs its light and heavy parts)
    const uint32_t *deg = d->d_deg && (!pmid || d->deg_split) ? d->d_deg : nullptr;
    const uint32_t *hdeg = deg ? d->deg_heavy() : nullptr;
    if (f.nw == 1)
        hipLaunchKernelGGL(k_frontier_compact<1>, dim3(f.nblk), dim3(kCompactBlock), 0, s, f.flag, f.hflag, d->Vpad,
                           d->plan.vsplit, d->d_ptr, pmid, deg, hdeg, d->tune, val, f.ctl, f.totals(), f.info, f.list,
                           f.hub, f.hub_cap, f.doff, f.dchunk, f.dchunk_cap, clk, prev, progress);
    else
        hipLaunchKernelGGL(k_frontier_compact<4>, dim3(f.nblk), dim3(kCompactBlock), 0, s, f.flag, f.hflag, d->Vpad,
                           d->plan.vsplit, d->d_ptr, pmid, deg, hdeg, d->tune, val, f.ctl, f.totals(), f.info, f.list,
                           f.hub, f.hub_cap, f.doff, f.dchunk, f.dchunk_cap, clk, prev, progress);
    OG_HIP(hipGetLastError());
    if (to_host) OG_HIP(hipMemcpyAsync(f.h_info, f.info, sizeof(FrontierInfo), hipMemcpyDeviceToHost, s));
}

// Bits needed by the largest edge weight (at least 1).
static uint32_t weight_bits(const og_graph *g) {
    std::atomic<uint32_t> maxw{0};
    parallel_for(g->E, 1 << 22, 0, [&](uint64_t b, uint64_t e, unsigned) {
        uint32_t m = 0;
        for (uint64_t i = b; i < e; ++i) m = std::max(m, g->wedges[2 * i + 1]);
        uint32_t cur = maxw.load();
        while (m > cur && !maxw.compare_exchange_weak(cur, m)) {
        }
    });
    uint32_t wb = 1;
    while (wb < 32 && (maxw.load() >> wb)) ++wb;
    return wb;
}

// Rows [v0, v1) of a weighted graph as packed words (to << wb | w) at
// dst[ptr[v] - ptr[v0] ...]; with the light/heavy split (sw > 0) each row
// lists its edges of weight < sw first, then the others, each part in CSR
// order.
static void pack_rows(const og_graph *g, uint64_t v0, uint64_t v1, uint32_t wb, uint32_t sw, uint32_t *dst) {
    const uint64_t e0 = g->ptr[v0];
    parallel_for(v1 - v0, 1 << 12, 0, [&](uint64_t b, uint64_t e, unsigned) {
        for (uint64_t v = v0 + b; v < v0 + e; ++v) {
            const uint32_t *src = g->wedges + 2 * g->ptr[v];
            const uint64_t n = g->ptr[v + 1] - g->ptr[v];
            uint32_t *out = dst + (g->ptr[v] - e0);
            if (!sw) {
                for (uint64_t i = 0; i < n; ++i) out[i] = (src[2 * i] << wb) | src[2 * i + 1];
                continue;
            }
            uint64_t k = 0;
            for (uint64_t i = 0; i < n; ++i)
                if (src[2 * i + 1] < sw) out[k++] = (src[2 * i] << wb) | src[2 * i + 1];
            for (uint64_t i = 0; i < n; ++i)
                if (src[2 * i + 1] >= sw) out[k++] = (src[2 * i] << wb) | src[2 * i + 1];
        }
    });
}

// Dynamic rows [v0, V) in the split layout: the light part of v at
// dst + lpos[v - v0], its heavy part at dst + nl + (ptr[v] - ptr[v0]) -
// lpos[v - v0] (nl = lpos[V - v0], all light parts first).
static void pack_split_rows(const og_graph *g, uint64_t v0, uint32_t wb, uint32_t sw, const uint64_t *lpos,
                            uint32_t *dst) {
    const uint64_t e0 = g->ptr[v0], nl = lpos[g->V - v0];
    parallel_for(g->V - v0, 1 << 12, 0, [&](uint64_t b, uint64_t e, unsigned) {
        for (uint64_t v = v0 + b; v < v0 + e; ++v) {
            const uint32_t *src = g->wedges + 2 * g->ptr[v];
            const uint64_t n = g->ptr[v + 1] - g->ptr[v], lp = lpos[v - v0];
            uint32_t *lo = dst + lp, *hi = dst + nl + (g->ptr[v] - e0) - lp;
            for (uint64_t i = 0; i < n; ++i) {
                const uint32_t w = (src[2 * i] << wb) | src[2 * i + 1];
                if (src[2 * i + 1] < sw) *lo++ = w;
                else *hi++ = w;
            }
        }
    });
}

// Uploads the packed rows [0, vend) into dst (device): host threads pack
// row-aligned chunks of about 64 MiB into two pinned bounce buffers while
// the previous chunk is in flight on s_compute.
static void upload_packed(DeviceState *d, const og_graph *g, uint64_t vend, uint32_t *dst) {
    const uint64_t n = g->ptr[vend];
    if (!n) return;
    struct Bounce {
        hipStream_t s;
        uint32_t *b[2] = {nullptr, nullptr};
        hipEvent_t ev[2] = {nullptr, nullptr};
        ~Bounce() {
            (void)hipStreamSynchronize(s);
            for (uint32_t *p : b)
                if (p) (void)hipHostFree(p);
            for (hipEvent_t e : ev)
                if (e) (void)hipEventDestroy(e);
        }
    } bb{d->s_compute};
    uint64_t maxrow = 0;
    for (uint64_t v = 0; v < vend; ++v) maxrow = std::max(maxrow, g->ptr[v + 1] - g->ptr[v]);
    const uint64_t C = std::max<uint64_t>(std::min<uint64_t>(n, 16ull << 20), maxrow);
    for (auto &p : bb.b) OG_HIP(hipHostMalloc((void **)&p, C * 4, 0));
    for (auto &e : bb.ev) OG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    for (uint64_t v0 = 0, k = 0; v0 < vend; ++k) {
        uint64_t v1 = v0;
        while (v1 < vend && g->ptr[v1 + 1] - g->ptr[v0] <= C) ++v1;
        const int s = (int)(k & 1);
        if (k >= 2) OG_HIP(hipEventSynchronize(bb.ev[s]));
        const uint64_t m = g->ptr[v1] - g->ptr[v0];
        pack_rows(g, v0, v1, d->wbits, d->split_weight, bb.b[s]);
        OG_HIP(hipMemcpyAsync(dst + g->ptr[v0], bb.b[s], m * 4, hipMemcpyHostToDevice, d->s_compute));
        OG_HIP(hipEventRecord(bb.ev[s], d->s_compute));
        v0 = v1;
    }
    OG_HIP(hipStreamSynchronize(d->s_compute));
}

// Zero-copy loading reads dynamic rows in place, so the staging share of the
// edge budget (cap edges) holds part of the dynamic region in HBM: blocks of
// kResChunk consecutive vertices, chosen by the link lines their rows would
// cost per edge.  A row of b bytes at an arbitrary 4-byte offset touches
// (b + kLinkLine - 4) / kLinkLine lines of kLinkLine bytes on average, each
// fetched whole, so blocks of short rows are taken first (ties: lower ids).
// With the light/heavy split each chunk has two blocks, its light parts and
// its heavy parts, ranked by the same measure and chosen separately.
// (Ranking every light block first, for the light rounds' repeated reads,
// measured slower on R-MAT: the short heavy rows it leaves on the host cost
// the heavy round more.)  The chunk table (8 bytes per block) is charged to
// the same share.
static void stage_resident(DeviceState *d, const og_graph *g, uint64_t vsplit, uint64_t cap,
                           const std::vector<uint64_t> &lpos) {
    const uint64_t V = g->V, eb = d->eb;
    const bool split = !lpos.empty();  // two blocks per chunk: light parts, heavy parts
    const uint64_t nb = split ? 2 : 1;  // blocks per chunk
    const uint64_t c0 = vsplit >> kResChunkShift, c1 = (V + kResChunk - 1) >> kResChunkShift;
    const uint64_t table_edges = (nb * c1 * sizeof(int64_t) + eb - 1) / eb;
    if (vsplit >= V || cap <= table_edges) return;
    cap -= table_edges;
    const uint64_t nch = c1 - c0;
    auto first = [&](uint64_t i) { return std::max<uint64_t>((c0 + i) << kResChunkShift, vsplit); };
    auto last = [&](uint64_t i) { return std::min<uint64_t>((c0 + i + 1) << kResChunkShift, V); };
    // block k = nb * i + part of chunk i (part 0: light or whole rows, 1: heavy)
    const uint64_t nblk = nb * nch;
    std::vector<uint64_t> bedges(nblk);
    std::vector<double> score(nblk);
    auto lines_of = [&](uint64_t n) { return n ? (double)(n * eb + kLinkLine - 4) / kLinkLine : 0.0; };
    parallel_for(nch, 1 << 12, 0, [&](uint64_t b, uint64_t e, unsigned) {
        for (uint64_t i = b; i < e; ++i) {
            double lines[2] = {0, 0};
            uint64_t n[2] = {0, 0};
            for (uint64_t v = first(i); v < last(i); ++v) {
                const uint64_t deg = g->ptr[v + 1] - g->ptr[v];
                const uint64_t nl = split ? lpos[v - vsplit + 1] - lpos[v - vsplit] : deg;
                lines[0] += lines_of(nl);
                n[0] += nl;
                lines[1] += lines_of(deg - nl);
                n[1] += deg - nl;
            }
            for (uint64_t k = 0; k < nb; ++k) {
                bedges[nb * i + k] = n[k];
                score[nb * i + k] = n[k] ? lines[k] / (double)n[k] : 0.0;
            }
        }
    });
    std::vector<uint32_t> order(nblk);  // nblk <= 2^28
    for (uint64_t i = 0; i < nblk; ++i) order[i] = (uint32_t)i;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) { return score[x] > score[y]; });
    std::vector<uint8_t> take(nblk, 0);
    uint64_t used = 0;
    for (uint32_t k : order) {
        if (!bedges[k] || used + bedges[k] > cap) continue;
        take[k] = 1;
        used += bedges[k];
    }
    if (!used) return;
    // The resident buffer holds the chosen blocks in block order (a chunk's
    // light block before its heavy block); runs of host positions that follow
    // each other are gathered in one piece.  Positions are in the host copy
    // of the dynamic region (with the split: light parts, then heavy parts).
    struct Run {
        uint64_t src, dst, n;
    };
    std::vector<Run> runs;
    auto add_run = [&](uint64_t src, uint64_t dst, uint64_t n) {
        if (!n) return;
        if (!runs.empty() && runs.back().src + runs.back().n == src && runs.back().dst + runs.back().n == dst)
            runs.back().n += n;
        else
            runs.push_back({src, dst, n});
    };
    const uint64_t dbase = d->dyn_base, nl = split ? lpos[V - vsplit] : 0;
    std::vector<int64_t> delta(nb * c1, kNotResident);
    uint64_t pos = 0;
    for (uint64_t k = 0; k < nblk; ++k) {
        if (!take[k]) continue;
        const uint64_t i = k / nb, v0 = first(i);
        uint64_t h0;  // host position of the block's first edge
        if (!split) h0 = g->ptr[v0] - dbase;
        else if (k % nb == 0) h0 = lpos[v0 - vsplit];
        else h0 = nl + (g->ptr[v0] - dbase) - lpos[v0 - vsplit];
        delta[nb * c0 + k] = (int64_t)pos - (int64_t)h0;
        add_run(h0, pos, bedges[k]);
        pos += bedges[k];
    }
    MemPool tmp;
    uint8_t *hb = (uint8_t *)tmp.palloc(used * eb);
    const uint8_t *src = (const uint8_t *)d->h_dyn;
    parallel_for(runs.size(), 64, 0, [&](uint64_t b, uint64_t e, unsigned) {
        for (uint64_t r = b; r < e; ++r) memcpy(hb + runs[r].dst * eb, src + runs[r].src * eb, runs[r].n * eb);
    });
    d->dyn_resident = used;
    d->d_staging = d->dalloc(used * eb);
    d->d_rdelta = (int64_t *)d->dalloc(delta.size() * sizeof(int64_t));
    OG_HIP(hipMemcpyAsync(d->d_staging, hb, used * eb, hipMemcpyHostToDevice, d->s_compute));
    OG_HIP(hipMemcpyAsync(d->d_rdelta, delta.data(), delta.size() * sizeof(int64_t), hipMemcpyHostToDevice,
                          d->s_compute));
    OG_HIP(hipStreamSynchronize(d->s_compute));
}

// Slots of the chunk ring: two to kRing of them, as many as have kRingSlotBytes,
// which take the staging share between them.  At least that large, a copy takes
// longer than its hand-over (4 MiB: 73 us on the link); a share above 32 MiB
// makes them larger, since what the ring holds is what crosses the link
// while the static rows are summed.
constexpr uint64_t kRingSlotBytes = 4ull << 20;
constexpr uint32_t kRing = 8;

LinkRing *link_ring(DeviceState *d, const og_graph *g) {
    if (d->link_ring) return d->link_ring->ring ? d->link_ring.get() : nullptr;
    auto r = std::make_shared<LinkRing>();
    d->link_ring = r;
    const uint64_t vs = d->plan.vsplit, base = d->dyn_base;
    for (uint64_t v = vs; v < d->V; ++v) r->maxrow = std::max(r->maxrow, g->ptr[v + 1] - g->ptr[v]);
    if (r->maxrow > d->slot_edges) return nullptr;
    const uint64_t total = (uint64_t)d->nslots * d->slot_edges * d->eb / 4;  // words of the staging share
    // the link format's rows start anywhere in a word and are read eight bytes
    // at a time, so it takes slots of a few words more
    r->lbits = d->lbits && (r->maxrow * d->lbits + 31) / 32 + 2 <= total / 2 ? d->lbits : 0;
    const uint64_t bits = r->lbits ? r->lbits : 8 * d->eb;
    auto words_of = [&](uint64_t n) { return (n * bits + 31) / 32 + (r->lbits ? 2 : 0); };
    uint32_t ring = (uint32_t)std::min<uint64_t>(kRing, std::max<uint64_t>(2, total * 4 / kRingSlotBytes));
    while (ring > 2 && total / ring < words_of(r->maxrow)) --ring;
    r->slot = total / ring;
    r->src = r->lbits ? d->h_link : (const uint32_t *)d->h_dyn;
    for (uint64_t va = vs; va < d->V;) {
        uint64_t lo = va + 1, hi = d->V;
        while (lo < hi) {  // largest vb whose rows fit
            const uint64_t mid = (lo + hi + 1) / 2;
            if (words_of(g->ptr[mid] - g->ptr[va]) <= r->slot) lo = mid; else hi = mid - 1;
        }
        const uint64_t b0 = (g->ptr[va] - base) * bits, b1 = (g->ptr[lo] - base) * bits;
        const uint64_t w0 = b0 / 32, w1 = (b1 + 31) / 32 + (r->lbits && b1 > b0 ? 1 : 0);
        r->chunks.push_back({(uint32_t)va, (uint32_t)lo, w0, b1 > b0 ? w1 - w0 : 0, (uint32_t)(b0 % 32)});
        va = lo;
    }
    r->ev_h2d.assign(ring, nullptr);
    r->ev_use.assign(ring, nullptr);
    for (auto &e : r->ev_h2d) OG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    for (auto &e : r->ev_use) OG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    r->ring = ring;
    return r.get();
}

// Bits per edge of the link format (DeviceState::lbits): those of V - 1, for
// packed weighted words the weight's more; 0 where they are too many, or
// where nothing would read it: traversals that gather chunks take whole edges, and a
// weighted graph that is not packed keeps its 8-byte ones.
static uint32_t link_bits(const DeviceState *d, const og_graph *g) {
    if (!d->in_place && g->kind != OG_KIND_PULL) return 0;
    if (g->kind == OG_KIND_WEIGHTED && !d->packed) return 0;
    const uint32_t bits = std::max(bits_of(g->V - 1), 1u) + (d->packed ? d->wbits : 0);
    return bits <= kLinkBitsMax ? bits : 0;
}

// Packs the host layout's words `src` into a pinned stream of `bits`-bit words.
// With V of a few million a quarter to a third of the bytes go (ER 3 M
// x 32, 22 bits: PageRank 66 -> 46 ms, CC 7.9 -> 6.6 ms; preparing the
// packed copy takes 12 ms more).  Without pinned memory for it the edges stay
// as they are.
static void pack_link(DeviceState *d, uint32_t bits, const uint32_t *src, uint64_t n) {
    if (!bits || !n) return;
    const uint64_t words = (n * bits + 31) / 32 + 2;
    uint32_t *dst = (uint32_t *)d->mem.try_palloc(words * 4);
    if (!dst) return;
    dst[words - 1] = dst[words - 2] = 0;
    // groups of 32 edges fill `bits` whole words
    parallel_for((n + 31) / 32, 1 << 15, 0, [&](uint64_t b, uint64_t e, unsigned) {
        for (uint64_t k = b; k < e; ++k) {
            const uint64_t i1 = std::min(n, 32 * (k + 1));
            uint32_t *out = dst + k * bits;
            uint64_t acc = 0;
            uint32_t have = 0;
            for (uint64_t i = 32 * k; i < i1; ++i) {
                acc |= (uint64_t)src[i] << have;
                have += bits;
                if (have >= 32) {
                    *out++ = (uint32_t)acc;
                    acc >>= 32;
                    have -= 32;
                }
            }
            if (have) *out = (uint32_t)acc;
        }
    });
    void *hd = nullptr;
    OG_HIP(hipHostGetDevicePointer(&hd, dst, 0));
    d->lbits = bits;
    d->h_link = dst;
    d->hd_link = hd;
}

// The compaction's degree table (DeviceState::d_deg): 4 bytes per vertex
// and range in place of two 8-byte row bounds.  Not built when a degree
// exceeds 32 bits (the passes then read the row bounds).
static void upload_degrees(DeviceState *d, const og_graph *g) {
    const uint64_t V = g->V, Vp = d->Vpad;
    const bool split = d->split_weight != 0;
    std::atomic<bool> wide{false};
    std::vector<uint32_t> dg((split ? 2 : 1) * Vp, 0);
    parallel_for(V, 1 << 16, 0, [&](uint64_t b, uint64_t e, unsigned) {
        bool w = false;
        for (uint64_t v = b; v < e; ++v) {
            const uint64_t b0 = g->ptr[v], e0 = g->ptr[v + 1];
            const uint64_t m = split ? d->h_pmid[v] : e0;
            w |= (e0 - b0) >> 32 != 0;
            dg[v] = (uint32_t)(m - b0);
            if (split) dg[Vp + v] = (uint32_t)(e0 - m);
        }
        if (w) wide = true;
    });
    if (wide) return;
    d->d_deg = (uint32_t *)d->dalloc(dg.size() * sizeof(uint32_t));
    OG_HIP(hipMemcpyAsync(d->d_deg, dg.data(), dg.size() * sizeof(uint32_t), hipMemcpyHostToDevice, d->s_compute));
    OG_HIP(hipStreamSynchronize(d->s_compute));
    d->deg_split = split;
}

static void prepare_impl(og_graph *g, og_approach approach, const og_plan_params *params, og_plan_info *info) {
    if (!hip_available()) raise(OG_EHIP, "no HIP device is visible");
    if (approach != OG_ASCETIC && approach != OG_SUBWAY && approach != OG_USM)
        raise(OG_EINVAL, "unknown approach %d", (int)approach);
    og_plan_params p{};
    if (params) p = *params;
    if (g->dev) {
        device_state_free(g->dev);
        g->dev = nullptr;
    }
    std::unique_ptr<DeviceState, void (*)(DeviceState *)> d(new DeviceState, device_state_free);
    OG_HIP(hipGetDevice(&d->device));
    OG_HIP(hipDeviceGetAttribute(&d->clock_khz, hipDeviceAttributeWallClockRate, d->device));
    d->approach = approach;
    d->V = g->V;
    d->E = g->E;
    d->Vpad = (g->V + 15) / 16 * 16;
    d->eb = g->edge_bytes();
    d->flags = p.flags;
    d->host_threads = p.host_threads ? p.host_threads : default_threads();
    // Compact weighted format: when ids and weights fit one 32-bit word, the
    // static region, the staging slots and the link all carry 4 bytes per
    // edge instead of 8, so the same byte budget holds twice the edges.  The
    // planner sizes its regions in these device bytes.  USM reads the CSR as
    // it lies in host memory and keeps the 8-byte form.
    if (g->kind == OG_KIND_WEIGHTED && approach != OG_USM && !(p.flags & OG_PLAN_NO_PACK) && g->E) {
        const uint32_t wb = weight_bits(g);
        if (wb < 32 && g->V - 1 < (1ull << (32 - wb))) {
            d->packed = true;
            d->wbits = wb;
            d->eb = 4;
        }
    }
    d->deb = d->eb;
    const uint64_t V = g->V, E = g->E, eb = d->eb;
    // Light/heavy split: rows of the packed device / link copies list light
    // edges first; pmid[v] is where row v's heavy edges start.
    if (p.split_weight) {
        if (!d->packed)
            raise(OG_EUNSUPPORTED, "the light/heavy split needs packed weighted edges (Ascetic or Subway, ids and "
                                   "weights in one 32-bit word, no OG_PLAN_NO_PACK)");
        d->split_weight = p.split_weight;
        d->h_pmid.resize(V);
        parallel_for(V, 1 << 14, 0, [&](uint64_t b, uint64_t e, unsigned) {
            for (uint64_t v = b; v < e; ++v) {
                uint64_t k = g->ptr[v];
                for (uint64_t i = g->ptr[v]; i < g->ptr[v + 1]; ++i) k += g->wedges[2 * i + 1] < p.split_weight;
                d->h_pmid[v] = k;
            }
        });
    }

    // ---- plan
    og_plan_info &pl = d->plan;
    if (approach == OG_ASCETIC) {
        og_status st = og_plan_compute(V, E, g->ptr, (uint32_t)eb, &p, &pl);
        if (st != OG_OK) raise(st, "%s", og_last_error());
    } else if (approach == OG_SUBWAY) {
        // Subway keeps no static region; the whole budget is the transfer
        // buffer (reference: 0.9 * (12 GiB - 32 V) / 4, BFS/sbw_BFS/main.cpp:334).
        uint64_t total = p.edge_budget_bytes ? p.edge_budget_bytes / eb
                                             : (uint64_t)(0.9 * (double)((12ull << 30) - 32ull * V) / (double)eb);
        std::memset(&pl, 0, sizeof pl);
        pl.total_budget_edges = total;
        pl.static_edges = 0;
        pl.staging_edges = total;
        pl.overload_edges = E;
        pl.static_vertices = 0;
        pl.vsplit = 0;
        pl.advisek_used = 0.0f;
    } else {
        std::memset(&pl, 0, sizeof pl);
        pl.total_budget_edges = E;
        pl.static_edges = E;
        pl.static_vertices = V;
        pl.vsplit = V;
        pl.advisek_used = 1.0f;
    }
    pl.approach = (uint32_t)approach;

    OG_HIP(hipStreamCreateWithFlags(&d->s_compute, hipStreamNonBlocking));
    OG_HIP(hipStreamCreateWithFlags(&d->s_copy, hipStreamNonBlocking));
    OG_HIP(hipStreamCreateWithFlags(&d->s_static, hipStreamNonBlocking));
    OG_HIP(hipEventCreateWithFlags(&d->ev_static, hipEventDisableTiming));
    OG_HIP(hipEventCreateWithFlags(&d->ev_fork, hipEventDisableTiming));

    // ---- graph placement
    if (approach == OG_USM) {
        // Graph arrays stay in pinned host memory and the kernels read them
        // through the device mapping: what SYCL malloc_shared gives on a GPU
        // without XNACK page migration.
        if (!g->pinned_ptr || !(eb == 8 ? g->pinned_wedges : g->pinned_cols))
            raise(OG_EUNSUPPORTED, "USM approach needs the graph in pinned host memory");
        void *dp = nullptr, *de = nullptr;
        OG_HIP(hipHostGetDevicePointer(&dp, g->ptr, 0));
        OG_HIP(hipHostGetDevicePointer(&de, (void *)g->edge_data(), 0));
        d->d_ptr = (uint64_t *)dp;
        d->d_static = de;
        d->static_used = E;
        d->managed = true;
    } else {
        d->d_ptr = (uint64_t *)d->dalloc((V + 1) * sizeof(uint64_t));
        OG_HIP(hipMemcpyAsync(d->d_ptr, g->ptr, (V + 1) * sizeof(uint64_t), hipMemcpyHostToDevice, d->s_compute));
        if (d->split_weight) {
            d->d_pmid = (uint64_t *)d->dalloc(std::max<uint64_t>(V, 1) * sizeof(uint64_t));
            OG_HIP(hipMemcpyAsync(d->d_pmid, d->h_pmid.data(), V * sizeof(uint64_t), hipMemcpyHostToDevice,
                                  d->s_compute));
        }
        upload_degrees(d.get(), g);
        if (pl.static_edges) {
            d->d_static = d->dalloc(pl.static_edges * eb);
            d->static_used = g->ptr[pl.vsplit];
            if (d->packed)
                upload_packed(d.get(), g, pl.vsplit, (uint32_t *)d->d_static);
            else if (d->static_used)
                OG_HIP(hipMemcpyAsync(d->d_static, g->edge_data(), d->static_used * eb, hipMemcpyHostToDevice,
                                      d->s_compute));
        }
        if (pl.vsplit < V) {
            // PageRank streams its dynamic region through the slots (vertex-
            // aligned chunks), so a pull-layout graph always gets them
            //
            // Traversals read the dynamic rows where they are, in pinned host
            // memory, also when the copy loader was asked for: an active row
            // crosses the link once at the link's speed and no round waits
            // for the host, where gathering took the host's threads (16 GB/s)
            // and two round trips per round (BFS R-MAT 1 M, a quarter of the
            // edges on the device: gathered and copied 5.0 ms, rows moved
            // whole through a ring of slots 2.9, in place 1.1).  Gathered
            // chunks stay for graphs in pageable memory and for the A/B flags.
            const bool zc = g->kind != OG_KIND_PULL &&
                            ((p.flags & OG_PLAN_ZERO_COPY) ||
                             (!(p.flags & (OG_PLAN_NO_OVERLAP | OG_PLAN_NO_FUSE)) &&
                              (d->packed || (eb == 8 ? g->pinned_wedges : g->pinned_cols))));
            d->in_place = zc;
            // Staging slots: gather, copy and relax of consecutive chunks
            // overlap.  Chunks of ~kSlotTargetBytes: smaller ones cost more
            // in per-chunk gather dispatch and launches than they save in
            // pipeline fill.  Never smaller than the largest dynamic row,
            // which the vertex-aligned PageRank chunks need whole.
            uint64_t maxdyn = 0;
            for (uint64_t v = pl.vsplit; v < V; ++v) maxdyn = std::max(maxdyn, g->ptr[v + 1] - g->ptr[v]);
            uint32_t ns = (uint32_t)std::min<uint64_t>(kMaxSlots, std::max<uint64_t>(2, pl.staging_edges * eb /
                                                                                          kSlotTargetBytes));
            while (ns > 2 && pl.staging_edges / ns < maxdyn) --ns;
            d->nslots = ns;
            d->slot_edges = pl.staging_edges / ns;
            if (d->slot_edges == 0 && (!zc || !(p.flags & OG_PLAN_ZERO_COPY)))
                raise(OG_EBUDGET, "edge budget leaves %llu staging edges for %llu dynamic-region edges",
                      (unsigned long long)pl.staging_edges, (unsigned long long)(E - g->ptr[pl.vsplit]));
            if (!zc) {
                d->d_staging = d->dalloc((uint64_t)ns * d->slot_edges * eb);
                d->h_stage.resize(ns);
                d->ev_h2d.assign(ns, nullptr);
                d->ev_relax.assign(ns, nullptr);
                d->slot_h2d_pending.assign(ns, 0);
                d->slot_relax_pending.assign(ns, 0);
                for (uint32_t s = 0; s < ns; ++s) {
                    d->h_stage[s] = d->palloc(d->slot_edges * eb);
                    OG_HIP(hipEventCreateWithFlags(&d->ev_h2d[s], hipEventDisableTiming));
                    OG_HIP(hipEventCreateWithFlags(&d->ev_relax[s], hipEventDisableTiming));
                }
                d->h_dlist = (uint32_t *)d->palloc(V * sizeof(uint32_t));
                d->h_doff = (uint64_t *)d->palloc((V + 1) * sizeof(uint64_t));
                d->pool.reset(new WorkerPool(d->host_threads));
            }
            // Host source of the dynamic region in the device format: the
            // CSR itself, or (packed) a pinned packed copy built once here.
            d->dyn_base = g->ptr[pl.vsplit];
            const uint64_t nd = E - d->dyn_base;
            // zero-copy reads with the light/heavy split: all light parts
            // first, so that a light round's reads of neighbouring rows share
            // the link's 128-byte lines (staged chunks keep rows whole)
            std::vector<uint64_t> lpos;
            if (zc && d->split_weight) {
                lpos.resize(V - pl.vsplit + 1);
                lpos[0] = 0;
                for (uint64_t v = pl.vsplit; v < V; ++v)
                    lpos[v - pl.vsplit + 1] = lpos[v - pl.vsplit] + (d->h_pmid[v] - g->ptr[v]);
                d->split_nl = lpos.back();
                d->d_lpos = (uint64_t *)d->dalloc(lpos.size() * sizeof(uint64_t));
                OG_HIP(hipMemcpyAsync(d->d_lpos, lpos.data(), lpos.size() * sizeof(uint64_t), hipMemcpyHostToDevice,
                                      d->s_compute));
                OG_HIP(hipStreamSynchronize(d->s_compute));
            }
            // With the link format in place of it, the packed copy is only a
            // step on the way and need not be pinned.
            const uint32_t bits = link_bits(d.get(), g);
            std::unique_ptr<uint32_t[]> step;
            if (d->packed) {
                uint32_t *pk;
                if (zc && bits && nd) {
                    step.reset(new uint32_t[nd]);
                    pk = step.get();
                } else {
                    pk = (uint32_t *)d->palloc(std::max<uint64_t>(nd, 1) * 4);
                }
                if (!lpos.empty()) pack_split_rows(g, pl.vsplit, d->wbits, d->split_weight, lpos.data(), pk);
                else pack_rows(g, pl.vsplit, V, d->wbits, d->split_weight, pk);
                d->h_dyn = pk;
            } else {
                d->h_dyn = (const uint8_t *)g->edge_data() + d->dyn_base * eb;
            }
            d->slot_dyn = d->slot_edges;
            if (zc) {
                if (!d->packed && !(eb == 8 ? g->pinned_wedges : g->pinned_cols))
                    raise(OG_EUNSUPPORTED, "zero-copy loading needs the graph in pinned host memory");
                // Reading in place needs no transit slots, so the staging
                // share of the budget keeps part of the dynamic region
                // resident in HBM instead.
                stage_resident(d.get(), g, pl.vsplit, pl.staging_edges, lpos);
            }
            pack_link(d.get(), bits, (const uint32_t *)d->h_dyn, nd);
            if (step) {
                if (d->lbits) {
                    d->h_dyn = nullptr;
                } else {  // no link format after all
                    d->h_dyn = std::memcpy(d->palloc(nd * 4), step.get(), nd * 4);
                }
            }
            if (zc && d->h_dyn) {
                // map the allocation's base, then offset to the dynamic region
                const void *hbase = d->packed ? d->h_dyn : g->edge_data();
                void *hd = nullptr;
                OG_HIP(hipHostGetDevicePointer(&hd, (void *)hbase, 0));
                d->hd_dyn = (const uint8_t *)hd + ((const uint8_t *)d->h_dyn - (const uint8_t *)hbase);
            }
        }
    }

    // ---- in-edge CSR for direction-optimising BFS (counting sort by target)
    if (p.flags & OG_PLAN_DIRECTION_OPT) {
        if (approach != OG_ASCETIC || pl.vsplit < V)
            raise(OG_EUNSUPPORTED, "direction-optimising BFS needs the whole graph in HBM (Ascetic, vsplit = V)");
        if (g->kind == OG_KIND_PULL) raise(OG_EUNSUPPORTED, "pull-layout graphs serve PageRank only");
        const bool wt = g->kind == OG_KIND_WEIGHTED;
        auto col = [&](uint64_t i) { return wt ? g->wedges[2 * i] : g->cols[i]; };
        std::vector<uint64_t> iptr(V + 1, 0);
        std::vector<std::atomic<uint64_t>> cnt(V);
        parallel_for(V, 1 << 16, 0, [&](uint64_t b, uint64_t e, unsigned) {
            for (uint64_t v = b; v < e; ++v) cnt[v].store(0, std::memory_order_relaxed);
        });
        parallel_for(E, 1 << 20, 0, [&](uint64_t b, uint64_t e, unsigned) {
            for (uint64_t i = b; i < e; ++i) cnt[col(i)].fetch_add(1, std::memory_order_relaxed);
        });
        for (uint64_t v = 0; v < V; ++v) iptr[v + 1] = iptr[v] + cnt[v].load(std::memory_order_relaxed);
        parallel_for(V, 1 << 16, 0, [&](uint64_t b, uint64_t e, unsigned) {
            for (uint64_t v = b; v < e; ++v) cnt[v].store(iptr[v], std::memory_order_relaxed);
        });
        std::vector<uint32_t> icol(std::max<uint64_t>(E, 1));
        parallel_for(V, 1 << 12, 0, [&](uint64_t b, uint64_t e, unsigned) {
            for (uint64_t u = b; u < e; ++u)
                for (uint64_t i = g->ptr[u]; i < g->ptr[u + 1]; ++i)
                    icol[cnt[col(i)].fetch_add(1, std::memory_order_relaxed)] = (uint32_t)u;
        });
        d->d_in_ptr = (uint64_t *)d->dalloc((V + 1) * sizeof(uint64_t));
        d->d_in_cols = (uint32_t *)d->dalloc(std::max<uint64_t>(E, 1) * sizeof(uint32_t));
        OG_HIP(hipMemcpy(d->d_in_ptr, iptr.data(), (V + 1) * sizeof(uint64_t), hipMemcpyHostToDevice));
        OG_HIP(hipMemcpy(d->d_in_cols, icol.data(), std::max<uint64_t>(E, 1) * sizeof(uint32_t),
                         hipMemcpyHostToDevice));
    }

    // ---- vertex state
    d->d_val = (uint32_t *)d->dalloc(d->Vpad * sizeof(uint32_t));
    OG_HIP(hipStreamSynchronize(d->s_compute));
    frontier_alloc(d.get(), g, d->fr, d->mem);
    (void)take_stage(d.get(), V * sizeof(uint32_t));
    pl.device_bytes = d->device_bytes();
    if (info) *info = pl;
    g->dev = d.release();
}

// ------------------------------------------------------- frontier driver

enum { kClsFront = 0, kClsStat = 1, kClsDyn = 2, kClsCopy = 3 };

struct RunTimers {
    TimedClass front, stat, dyn, copy;
    int clocked = -1;  // the relax class that the device's clock timed (with front), -1: none
    TimedClass &at(int c) { return c == kClsFront ? front : c == kClsStat ? stat : c == kClsDyn ? dyn : copy; }
};

// A captured batch of device-driven rounds, replayed with one hipGraphLaunch.
// Its timing marks are external event-record nodes, read after each replay.
struct RoundGraph {
    struct Mark {
        int cls;
        hipEvent_t a, b;
    };
    uint64_t key = ~0ull;
    hipGraphExec_t exec = nullptr;
    std::vector<hipEvent_t> events;
    std::vector<Mark> marks;
    ~RoundGraph() {
        if (exec) (void)hipGraphExecDestroy(exec);
        for (hipEvent_t e : events) (void)hipEventDestroy(e);
    }
};

// Timing marks of enqueued work.  EagerSpan: an EventSpan of the run per
// launch sequence.  GraphSpan: a pair of event-record nodes in the graph
// being captured.  NoSpan: none (work that the device's clock times).
struct EagerSpan {
    DeviceState *d;
    RunTimers &tm;
    template <class F>
    void operator()(int cls, hipStream_t s, F &&fn) const {
        EventSpan span(d, &tm.at(cls), s);
        fn();
    }
};

struct GraphSpan {
    RoundGraph *rg;
    template <class F>
    void operator()(int cls, hipStream_t s, F &&fn) const {
        hipEvent_t a = nullptr, b = nullptr;
        OG_HIP(hipEventCreate(&a));
        rg->events.push_back(a);
        OG_HIP(hipEventRecordWithFlags(a, s, hipEventRecordExternal));
        OG_HIP(hipEventCreate(&b));
        rg->events.push_back(b);
        fn();
        OG_HIP(hipEventRecordWithFlags(b, s, hipEventRecordExternal));
        rg->marks.push_back({cls, a, b});
    }
};

struct NoSpan {
    template <class F>
    void operator()(int, hipStream_t, F &&fn) const {
        fn();
    }
};

// Captured batches of rounds of one preparation, by key (algorithm, layout,
// rounds per batch); the oldest is dropped beyond kGraphCache.
constexpr size_t kGraphCache = 8;
struct RoundGraphCache {
    std::vector<std::unique_ptr<RoundGraph>> g;
};

// The cached graph for `key`, captured on the compute stream by body(rg)
// when the cache does not hold it.
template <class Body>
static RoundGraph *round_graph_for(DeviceState *d, uint64_t key, Body body) {
    if (!d->round_graph)
        d->round_graph = std::shared_ptr<void>(new RoundGraphCache,
                                               [](void *p) { delete static_cast<RoundGraphCache *>(p); });
    auto &cache = static_cast<RoundGraphCache *>(d->round_graph.get())->g;
    for (auto &c : cache)
        if (c->key == key) return c.get();
    std::unique_ptr<RoundGraph> rg(new RoundGraph);
    hipStream_t s = d->s_compute;
    OG_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    hipGraph_t graph = nullptr;
    try {
        body(rg.get());
    } catch (...) {
        (void)hipStreamEndCapture(s, &graph);
        if (graph) (void)hipGraphDestroy(graph);
        throw;
    }
    OG_HIP(hipStreamEndCapture(s, &graph));
    const hipError_t e = hipGraphInstantiate(&rg->exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    OG_HIP(e);
    rg->key = key;
    if (cache.size() >= kGraphCache) cache.erase(cache.begin());
    cache.push_back(std::move(rg));
    return cache.back().get();
}

// Host gather of dynamic edges [c0, c1) into a pinned slot (reference
// fillEdgeArrByMultiThread, GraphMeta.h:470-506, with the copy offsets taken
// from the device-built degree prefix instead of a serial host scan).  The
// source is the dynamic region in its transfer format (d->h_dyn, whose first
// element is edge d->dyn_base of the CSR).
static void gather(DeviceState *d, const og_graph *g, uint32_t ndyn, uint64_t c0, uint64_t c1, uint8_t *dst,
                   bool heavy) {
    const uint64_t eb = d->deb;
    const uint8_t *src = (const uint8_t *)d->h_dyn;
    const uint64_t base = d->dyn_base;
    const uint64_t n = c1 - c0;
    const unsigned T = d->pool->size();
    const unsigned use = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(T, n / 16384));
    const uint64_t L = (n + use - 1) / use;
    auto part = [&](unsigned t) {
        if (t >= use) return;
        const uint64_t p0 = c0 + (uint64_t)t * L;
        const uint64_t p1 = std::min(c1, p0 + L);
        if (p0 >= p1) return;
        uint64_t i = (uint64_t)(std::upper_bound(d->h_doff, d->h_doff + ndyn + 1, p0) - d->h_doff) - 1;
        uint64_t p = p0;
        while (p < p1) {
            const uint32_t v = d->h_dlist[i];
            const uint64_t vb = d->h_doff[i], ve = d->h_doff[i + 1];
            const uint64_t stop = std::min(ve, p1);
            const uint64_t rb = heavy ? d->h_pmid[v] : g->ptr[v];  // row start of the round's range
            std::memcpy(dst + (p - c0) * eb, src + (rb - base + (p - vb)) * eb, (stop - p) * eb);
            p = stop;
            ++i;
        }
    };
    if (use == 1) part(0);  // (waking the pool takes longer than this copy)
    else d->pool->run(part);
}

template <int ALGO>
static RelaxArgs relax_args(DeviceState *d) {
    const DeviceState::MsState &m = d->d_ms;
    return RelaxArgs{d->d_val, d->fr.flag, m.vn, m.front, d->wbits, nullptr, d->run_pmid,
                     d->run_pmid ? d->fr.ctl : nullptr};
}

// Grids of device-count launches: the kernels stride over whatever count
// the round's compaction produced, so without a host-side count a fixed
// grid that fills the chip (256 CUs) is launched.
constexpr unsigned kGroupGridCap = 2048;  // workgroups of k_relax_group
constexpr unsigned kHubGridCap = 1024;    // workgroups of k_relax_hub
constexpr unsigned kDynGridCap = 8192;    // workgroups of k_relax_dyn (zero-copy reads want many in flight)

static unsigned capped(uint64_t blocks, unsigned cap) {
    return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(blocks, cap));
}

template <int ALGO, bool W, bool PK>
static void launch_static_relax_fmt(DeviceState *d, Frontier &f, const FrontierInfo *hfi, const RelaxArgs &a,
                                    hipStream_t s) {
    const void *edges = d->d_static;
    unsigned long long *upd = f.spread;
    const uint32_t lpv0 = d->tune.lpv0;
    if (!hfi || hfi->n[0]) {
        const dim3 gr(hfi ? capped(((uint64_t)hfi->n[0] * lpv0 + kBlock - 1) / kBlock, kGroupGridCap) : kGroupGridCap);
        switch (lpv0) {
#define OG_LPV(L)                                                                                                 \
    case L:                                                                                                       \
        hipLaunchKernelGGL((k_relax_group<ALGO, W, PK, L>), gr, dim3(kBlock), 0, s, f.list, d->plan.vsplit, 0, f.info, d->d_ptr, \
                           edges, a, upd);                                                                        \
        break;
            OG_LPV(1) OG_LPV(2) OG_LPV(4) OG_LPV(8) OG_LPV(16) OG_LPV(32)
            default: OG_LPV(64)
#undef OG_LPV
        }
    }
    if (!hfi || hfi->n[1])
        hipLaunchKernelGGL((k_relax_group<ALGO, W, PK, 64>),
                           dim3(hfi ? capped(((uint64_t)hfi->n[1] * 64 + kBlock - 1) / kBlock, kGroupGridCap)
                                    : kGroupGridCap),
                           dim3(kBlock), 0, s, f.list, d->plan.vsplit, 1, f.info, d->d_ptr, edges, a, upd);
    if (!hfi || hfi->n[2])
        hipLaunchKernelGGL((k_relax_hub<ALGO, W, PK>), dim3(hfi ? capped(hfi->n[2], kHubGridCap) : kHubGridCap),
                           dim3(kBlock), d->tune.tile * d->eb, s, f.hub, f.hub_cap, f.info, d->tune.tile, d->d_ptr,
                           edges, a, upd);
    OG_HIP(hipGetLastError());
}

template <int ALGO, bool W>
void launch_static_relax(DeviceState *d, Frontier &f, const FrontierInfo *hfi, const RelaxArgs &a, hipStream_t s) {
    if (W && d->packed) launch_static_relax_fmt<ALGO, W, true>(d, f, hfi, a, s);
    else launch_static_relax_fmt<ALGO, W, false>(d, f, hfi, a, s);
}
template void launch_static_relax<ALGO_MSBFS, false>(DeviceState *, Frontier &, const FrontierInfo *, const RelaxArgs &, hipStream_t);
template void launch_static_relax<ALGO_MSBFS, true>(DeviceState *, Frontier &, const FrontierInfo *, const RelaxArgs &, hipStream_t);

// Static-region relax of a round on s_static, so that it overlaps the
// dynamic region (link bound): forked from the compute stream after the
// compaction; returns true when the caller must join ev_static before the
// next compaction.  All relax updates are monotone (atomicMin / same-level
// stores / atomicOr), so the two regions may interleave.  NO_OVERLAP runs it
// (and a plan without a dynamic region) runs it on the compute stream
// instead.  hfi: the round's summary when the host has
// it (sizes the grids, skips empty bins), else null.
template <int ALGO, bool W, class Span>
static bool launch_static(DeviceState *d, const FrontierInfo *hfi, const Span &span) {
    if (hfi && !(hfi->n[0] | hfi->n[1] | hfi->n[2])) return false;
    if ((d->flags & OG_PLAN_NO_OVERLAP) || d->plan.vsplit >= d->V) {  // nothing to overlap with
        span(kClsStat, d->s_compute,
             [&] { launch_static_relax<ALGO, W>(d, d->fr, hfi, relax_args<ALGO>(d), d->s_compute); });
        return false;
    }
    OG_HIP(hipEventRecord(d->ev_fork, d->s_compute));
    OG_HIP(hipStreamWaitEvent(d->s_static, d->ev_fork, 0));
    span(kClsStat, d->s_static, [&] { launch_static_relax<ALGO, W>(d, d->fr, hfi, relax_args<ALGO>(d), d->s_static); });
    OG_HIP(hipEventRecord(d->ev_static, d->s_static));
    return true;
}

template <int ALGO, bool W, bool PACKED, bool DIRECT>
static void launch_dyn(DeviceState *d, unsigned grid, const void *src, uint64_t c0, uint64_t c1) {
    hipLaunchKernelGGL((k_relax_dyn<ALGO, W, PACKED, DIRECT>), dim3(grid), dim3(kBlock), 0, d->s_compute, d->fr.list,
                       d->fr.info, d->fr.doff, src, c0, c1, d->d_ptr, d->dyn_base, (const void *)d->d_staging,
                       DIRECT ? (const int64_t *)d->d_rdelta : nullptr, d->wbits, relax_args<ALGO>(d),
                       DIRECT ? (const uint64_t *)d->d_lpos : nullptr, d->split_nl, d->plan.vsplit,
                       DIRECT && c0 == 0 ? (const uint32_t *)d->fr.dchunk : nullptr, DIRECT ? d->lbits : 0u, d->fr.spread);
}

// The fused round relax (k_relax_round) of a device-driven round on the
// compute stream: the static grids of the separate launches (kGroupGridCap
// twice, kHubGridCap) and, with_dyn (zero-copy), the dynamic grid rounded up
// to a multiple of kHubGridCap.
template <int ALGO, bool W, bool PK, int LPV>
static void launch_round_lpv(DeviceState *d, const RoundRelax &r, unsigned grid, size_t lds) {
    hipLaunchKernelGGL((k_relax_round<ALGO, W, PK, LPV>), dim3(grid), dim3(kBlock), lds, d->s_compute, r,
                       relax_args<ALGO>(d));
}

template <int ALGO, bool W, bool PK>
static void launch_round_fmt(DeviceState *d, bool with_dyn) {
    static_assert(2 * kHubGridCap == kGroupGridCap, "period layout: 2 + 2 + 1 static workgroups per K");
    const unsigned dyn = d->tune.dyn_grid ? d->tune.dyn_grid : kDynGridCap;
    RoundRelax r{};
    r.list = d->fr.list;
    r.info = d->fr.info;
    r.ptr = d->d_ptr;
    r.sedges = d->d_static;
    r.hub = d->fr.hub;
    r.hub_cap = d->fr.hub_cap;
    r.tile = d->tune.tile;
    r.cd = with_dyn ? (dyn + kHubGridCap - 1) / kHubGridCap : 0;
    r.doff = d->fr.doff;
    r.stage = d->lbits ? d->hd_link : d->hd_dyn;
    r.lbits = d->lbits;
    r.dbase = d->dyn_base;
    r.resident = d->d_staging;
    r.rdelta = d->d_rdelta;
    r.lpos = d->d_lpos;
    r.dchunk = d->fr.dchunk;
    r.nl = d->split_nl;
    r.vsplit = d->plan.vsplit;
    r.spread = d->fr.spread;
    r.clk = d->fr.clk;
    const unsigned grid = (kFuseStatic + r.cd) * kHubGridCap;
    const size_t lds = std::max<size_t>(with_dyn ? sizeof(DynLds) : 0, (size_t)d->tune.tile * d->eb);
    switch (d->tune.lpv0) {
        case 1: launch_round_lpv<ALGO, W, PK, 1>(d, r, grid, lds); break;
        case 2: launch_round_lpv<ALGO, W, PK, 2>(d, r, grid, lds); break;
        case 4: launch_round_lpv<ALGO, W, PK, 4>(d, r, grid, lds); break;
        case 8: launch_round_lpv<ALGO, W, PK, 8>(d, r, grid, lds); break;
        case 16: launch_round_lpv<ALGO, W, PK, 16>(d, r, grid, lds); break;
        case 32: launch_round_lpv<ALGO, W, PK, 32>(d, r, grid, lds); break;
        default: launch_round_lpv<ALGO, W, PK, 64>(d, r, grid, lds); break;
    }
    OG_HIP(hipGetLastError());
}

template <int ALGO, bool W>
static void launch_round_relax(DeviceState *d, bool with_dyn) {
    if (W && d->packed) launch_round_fmt<ALGO, W, true>(d, with_dyn);
    else launch_round_fmt<ALGO, W, false>(d, with_dyn);
}

template <bool W, bool PK>
static void launch_srv_round_fmt(DeviceState *d, Frontier &f, const RelaxArgs &a, hipStream_t s, const SrvPull *pull) {
    RoundRelax r{};
    r.list = f.list;
    r.info = f.info;
    r.ptr = d->d_ptr;
    r.sedges = d->d_static;
    r.hub = f.hub;
    r.hub_cap = f.hub_cap;
    r.tile = d->tune.tile;
    r.vsplit = d->plan.vsplit;
    r.spread = f.spread;
    SrvPull p{};
    if (pull) p = *pull;
    const uint32_t cp = pull ? kDynGridCap / kHubGridCap : 0;  // the separate pull's 8192 workgroups
    const unsigned grid = (kFuseStatic + cp) * kHubGridCap;
    const size_t lds = (size_t)d->tune.tile * d->eb;
    switch (d->tune.lpv0) {
#define OG_SRV(L)                                                                                                  \
    case L:                                                                                                        \
        hipLaunchKernelGGL((k_srv_round<W, PK, L>), dim3(grid), dim3(kBlock), lds, s, r, a, p, cp);               \
        break;
        OG_SRV(1) OG_SRV(2) OG_SRV(4) OG_SRV(8) OG_SRV(16) OG_SRV(32)
        default: OG_SRV(64)
#undef OG_SRV
    }
    OG_HIP(hipGetLastError());
}

void launch_srv_round(DeviceState *d, Frontier &f, const RelaxArgs &a, hipStream_t s, const SrvPull *pull,
                      bool weighted) {
    if (weighted && d->packed) launch_srv_round_fmt<true, true>(d, f, a, s, pull);
    else if (weighted) launch_srv_round_fmt<true, false>(d, f, a, s, pull);
    else launch_srv_round_fmt<false, false>(d, f, a, s, pull);
}

// Dynamic relax of edges [c0, min(c1, D)); `known` = c1 - c0 when the host
// knows the edge count (exact grid), else 0 (fixed grid).
template <int ALGO, bool W>
static void launch_dyn_any(DeviceState *d, const void *src, uint64_t c0, uint64_t c1, uint64_t known, bool direct) {
    const unsigned cap = d->tune.dyn_grid ? d->tune.dyn_grid : kDynGridCap;
    const unsigned grid = known ? capped((known + kDynEdgesPerBlock - 1) / kDynEdgesPerBlock, cap) : cap;
    if (d->packed) {
        if (direct) launch_dyn<ALGO, W, true, true>(d, grid, src, c0, c1);
        else launch_dyn<ALGO, W, true, false>(d, grid, src, c0, c1);
    } else {
        if (direct) launch_dyn<ALGO, W, false, true>(d, grid, src, c0, c1);
        else launch_dyn<ALGO, W, false, false>(d, grid, src, c0, c1);
    }
    OG_HIP(hipGetLastError());
}

// Staged dynamic region of a round whose summary the host holds: the host
// gathers the active edges into pinned slots and the copy stream moves them
// while the other slot is relaxed.
template <int ALGO, bool W>
static void run_dynamic(DeviceState *d, const og_graph *g, const FrontierInfo &fi, RunTimers &tm, og_run_stats &st,
                        double &gather_ms) {
    const uint32_t ndyn = fi.n[3];
    const uint64_t D = fi.dyn_deg;
    if (!ndyn || !D) return;
    const uint32_t *d_dlist = d->fr.list + d->plan.vsplit;
    const uint64_t eb = d->deb;
    OG_HIP(hipMemcpyAsync(d->h_dlist, d_dlist, (size_t)ndyn * 4, hipMemcpyDeviceToHost, d->s_copy));
    OG_HIP(hipMemcpyAsync(d->h_doff, d->fr.doff, ((size_t)ndyn + 1) * 8, hipMemcpyDeviceToHost, d->s_copy));
    OG_HIP(hipStreamSynchronize(d->s_copy));
    const uint64_t C = d->slot_dyn;
    const bool serial = (d->flags & OG_PLAN_NO_OVERLAP) != 0;
    for (uint64_t c0 = 0, c = 0; c0 < D; c0 += C, ++c) {
        const uint64_t c1 = std::min(D, c0 + C);
        const int slot = (int)(c % d->nslots);
        if (d->slot_h2d_pending[slot]) OG_HIP(hipEventSynchronize(d->ev_h2d[slot]));
        Stopwatch sw;
        gather(d, g, ndyn, c0, c1, (uint8_t *)d->h_stage[slot], d->run_pmid && fi.heavy);
        gather_ms += sw.ms();
        uint8_t *dslot = (uint8_t *)d->d_staging + (uint64_t)slot * d->slot_edges * d->eb;
        if (d->slot_relax_pending[slot]) OG_HIP(hipStreamWaitEvent(d->s_copy, d->ev_relax[slot], 0));
        {
            EventSpan span(d, &tm.copy, d->s_copy);
            OG_HIP(hipMemcpyAsync(dslot, d->h_stage[slot], (c1 - c0) * eb, hipMemcpyHostToDevice, d->s_copy));
        }
        OG_HIP(hipEventRecord(d->ev_h2d[slot], d->s_copy));
        d->slot_h2d_pending[slot] = true;
        OG_HIP(hipStreamWaitEvent(d->s_compute, d->ev_h2d[slot], 0));
        {
            EventSpan span(d, &tm.dyn, d->s_compute);
            launch_dyn_any<ALGO, W>(d, (const void *)dslot, c0, c1, c1 - c0, false);
        }
        OG_HIP(hipEventRecord(d->ev_relax[slot], d->s_compute));
        d->slot_relax_pending[slot] = true;
        if (serial) OG_HIP(hipStreamSynchronize(d->s_compute));
        st.h2d_bytes += (c1 - c0) * eb;
        st.chunks++;
    }
}

// Algorithmic bytes per relaxed edge: column (+ weight) and the target state.
template <int ALGO, bool W>
constexpr uint64_t edge_bytes_alg() {
    return ms_masks(ALGO) ? 4ull + 8ull * ms_masks(ALGO) : (ALGO == ALGO_SSSP ? 12ull : 8ull);
}

constexpr int kRoundBatch = 4;     // device-driven rounds enqueued per host check
constexpr uint64_t kRoundsAhead = 2;  // rounds enqueued before the device has reached them (OG_PLAN_NO_GRAPH)
constexpr int kRoundBatchMax = 64;  // largest first batch (sized from the previous run)

// Iterates compaction -> static relax || dynamic relax -> after() until no
// vertex is active or held back.  Accumulates into st / tm.
//
// Without a host-side loader (whole graph in HBM, zero-copy dynamic region,
// USM) the rounds are device-driven: every kernel reads its counts from the
// round's FrontierInfo and the near-far threshold advances on the device, so
// rounds are enqueued a batch at a time and the host reads the traversal
// state once per batch (rounds enqueued past the end find no flags and do no
// work).  The first batch holds as many rounds as the previous run of the
// algorithm on this preparation took, rounded up to a multiple of
// kRoundBatch (a repeated traversal then needs one launch and no host round
// trip: each costs about 50 us); later batches kRoundBatch.  The staged loader needs
// the host in every round (gather, copies), so it synchronises on each
// round's summary.
// quiet_after: after() enqueues nothing (the compaction follows the relax).
// begin(ctl): enqueues the start of the run with that traversal state.
// variant: tells runs apart whose after() captures other work.
template <int ALGO, bool W, class Begin, class After>
static void frontier_loop(og_graph *g, DeviceState *d, og_run_stats &st, RunTimers &tm, double &gather_ms,
                          double &overload_wall, Begin begin, After after, bool quiet_after, bool variant = false) {
    hipStream_t s = d->s_compute;
    const uint64_t V = d->V;
    // SSSP near-far order: only vertices below the threshold relax in a
    // round; when none is left it moves to (smallest held-back value + delta).
    const uint32_t delta = ALGO == ALGO_SSSP ? d->tune.delta : 0;
    const uint32_t *nf_val = delta ? d->d_val : nullptr;
    const bool has_dyn = d->plan.vsplit < d->V;
    const bool staged = has_dyn && !d->in_place;
    // deferring dynamic vertices reorders relaxations across levels, which
    // only the atomicMin relaxes (SSSP, CC) tolerate.  CC starts with every
    // vertex active: at 0 its dynamic vertices wait until the static region has
    // settled once, so that most of them carry their final label when their rows
    // cross the link (ER 3 M x 32, a quarter of the edges on the device: the
    // rows are read once instead of about twice, 10.5 -> 7.9 ms); 2 is both
    // regions every round.
    uint32_t defer = (ALGO == ALGO_SSSP || ALGO == ALGO_CC) && has_dyn ? d->tune.defer : 0;
    if (ALGO == ALGO_CC) {
        if (defer == 2) defer = 0;
        else if (defer == 0 && has_dyn && d->plan.vsplit) defer = kDeferOnce;
    }
    const bool dir_opt = ALGO == ALGO_BFS && d->d_in_ptr != nullptr;
    // light/heavy split: near-far SSSP on a graph prepared with it
    const bool split = ALGO == ALGO_SSSP && delta && d->d_pmid;
    d->run_pmid = split ? d->d_pmid : nullptr;
    const uint64_t *pm = d->run_pmid;
    begin(ctl_begin(V, delta, defer, dir_opt ? std::max<uint64_t>(d->E, 1) : 0, split));
    RunBlock *const h = d->fr.h_blk;
    if (!staged) {
        // one batch: kRoundBatch x (static || dynamic relax, after, compaction),
        // then the traversal state to the host
        // With both regions the static and dynamic relax of a round run as
        // one launch (k_relax_round); with OG_PLAN_NO_FUSE on two streams,
        // the dynamic relax enqueued before the static fork (a replay submits
        // the graph's kernels in capture order, and the link-bound relax
        // should not wait for the static launches).
        // A graph wholly in HBM runs its three static bins as one fused launch.
        const bool overlap = has_dyn && !(d->flags & OG_PLAN_NO_OVERLAP);
        const bool fuse = overlap && !(d->flags & OG_PLAN_NO_FUSE);
        const bool fuse_static = !has_dyn && !(d->flags & OG_PLAN_NO_FUSE);
        // One launch per round and region is timed by the device's clock, the
        // two-stream and separate launches by events.
        const bool clocked = fuse || fuse_static;
        RoundClock *const clk = clocked ? d->fr.clk : nullptr;
        const EagerSpan eager{d, tm};
        unsigned long long *const progress = clocked && (d->flags & OG_PLAN_NO_GRAPH) ? d->fr.h_progress : nullptr;
        auto first = [&] { frontier_compact(d, d->fr, s, nf_val, false, pm, clk, kClkOther, progress); };
        if (progress) __atomic_store_n(progress, 0ull, __ATOMIC_RELEASE);
        if (clocked) first();
        else eager(kClsFront, s, first);
        auto batch = [&](const auto &span, int rounds) {
            for (int r = 0; r < rounds; ++r) {
                bool joined = false;
                if (fuse) {
                    span(kClsDyn, s, [&] { launch_round_relax<ALGO, W>(d, true); });
                } else if (fuse_static) {
                    span(kClsStat, s, [&] { launch_round_relax<ALGO, W>(d, false); });
                } else if (overlap) {
                    OG_HIP(hipEventRecord(d->ev_fork, s));
                    span(kClsDyn, s, [&] { launch_dyn_any<ALGO, W>(d, d->lbits ? d->hd_link : d->hd_dyn, 0, ~0ull, 0, true); });
                    OG_HIP(hipStreamWaitEvent(d->s_static, d->ev_fork, 0));
                    span(kClsStat, d->s_static,
                         [&] { launch_static_relax<ALGO, W>(d, d->fr, nullptr, relax_args<ALGO>(d), d->s_static); });
                    OG_HIP(hipEventRecord(d->ev_static, d->s_static));
                    joined = true;
                } else {
                    joined = launch_static<ALGO, W>(d, nullptr, span);
                    if (has_dyn) span(kClsDyn, s, [&] { launch_dyn_any<ALGO, W>(d, d->lbits ? d->hd_link : d->hd_dyn, 0, ~0ull, 0, true); });
                }
                if (dir_opt)
                    span(kClsStat, s, [&] {
                        hipLaunchKernelGGL(k_bfs_pull, dim3(capped((d->V + kBlock - 1) / kBlock, kGroupGridCap)),
                                           dim3(kBlock), 0, s, d->d_in_ptr, d->d_in_cols, d->V, d->fr.info,
                                           d->fr.ctl, d->d_val, d->fr.flag, d->fr.spread);
                        OG_HIP(hipGetLastError());
                    });
                if (joined) OG_HIP(hipStreamWaitEvent(s, d->ev_static, 0));
                after(clk);
                span(kClsFront, s,
                     [&] {
                         frontier_compact(d, d->fr, s, nf_val, false, pm, clk, quiet_after ? kClkRelax : kClkOther,
                                          progress);
                     });
            }
            if (!progress) OG_HIP(hipMemcpyAsync(h, d->fr.blk, sizeof(RunBlock), hipMemcpyDeviceToHost, s));
        };
        const NoSpan untimed;
        auto enqueue = [&](const auto &span, int rounds) {
            if (clocked) batch(untimed, rounds);
            else batch(span, rounds);
        };
        uint64_t enqueued = 0;
        if (!(d->flags & OG_PLAN_NO_GRAPH)) {
            // first batch: exactly the pairs the previous run took (a 6-round
            // BFS replayed 8 rounds when this was rounded up to a multiple of
            // kRoundBatch, two empty relax + compaction pairs per run)
            const uint32_t guess = std::min<uint32_t>(d->last_pairs[ALGO], kRoundBatchMax);
            int rounds = guess ? (int)guess : kRoundBatch;
            for (;;) {
                const uint64_t key = (uint64_t)ALGO | (uint64_t)W << 4 | (uint64_t)(delta != 0) << 5 |
                                     (uint64_t)has_dyn << 6 | (uint64_t)dir_opt << 7 | (uint64_t)split << 16 |
                                     (uint64_t)variant << 17 | (uint64_t)rounds << 8;
                RoundGraph *rg = round_graph_for(d, key, [&](RoundGraph *n) {
                    enqueue(GraphSpan{n}, rounds);
                });
                enqueued += rounds;
                rounds = kRoundBatch;
                OG_HIP(hipGraphLaunch(rg->exec, s));
                OG_HIP(hipStreamSynchronize(s));
                for (const auto &m : rg->marks) {
                    float ms = 0;
                    if (hipEventElapsedTime(&ms, m.a, m.b) == hipSuccess) {
                        tm.at(m.cls).ms += ms;
                        tm.at(m.cls).launches++;
                    } else {
                        (void)hipGetLastError();
                    }
                }
                if (!h->ctl.live) break;
            }
            // relax + compaction pairs of this run, for the next run's first batch
            d->last_pairs[ALGO] = h->ctl.compactions ? h->ctl.compactions - 1 : 0;
        } else if (progress) {
            // rounds are enqueued kRoundsAhead ahead of the device, which
            // tells how far it is: no host round trip between rounds, and that
            // many empty ones (about 8 us each) at the end
            for (;; ++enqueued) {
                if (enqueued >= kRoundsAhead) wait_progress(progress, (enqueued + 1 - kRoundsAhead) << 1, s);
                if (__atomic_load_n(progress, __ATOMIC_ACQUIRE) & 1) break;
                enqueue(untimed, 1);
            }
        } else {
            for (;;) {
                enqueue(eager, kRoundBatch);
                enqueued += kRoundBatch;
                OG_HIP(hipStreamSynchronize(s));
                if (!h->ctl.live) break;
            }
        }
        if (clocked) {  // their times come with the run block, once the run's last kernel has left the compaction
            (fuse ? tm.dyn : tm.stat).launches += enqueued * (dir_opt ? 2 : 1);
            tm.front.launches += enqueued + 1;
            tm.clocked = fuse ? kClsDyn : kClsStat;
        }
    } else {
        {
            EventSpan span(d, &tm.front, s);
            frontier_compact(d, d->fr, s, nf_val, true, pm);
        }
        OG_HIP(hipStreamSynchronize(s));
        for (;;) {
            const FrontierInfo fi = *d->fr.h_info;
            if (!fi.live) break;
            const uint64_t active = (uint64_t)fi.n[0] + fi.n[1] + fi.nhub + fi.n[3] + fi.nzero;
            if (active) {  // else only the near-far threshold moved
                if (fi.n[2] > d->fr.hub_cap)
                    raise(OG_EHIP, "hub tile list overflow (%u > %llu)", fi.n[2], (unsigned long long)d->fr.hub_cap);
                const bool joined = launch_static<ALGO, W>(d, &fi, EagerSpan{d, tm});
                if (fi.n[3]) {
                    Stopwatch ow;
                    run_dynamic<ALGO, W>(d, g, fi, tm, st, gather_ms);
                    overload_wall += ow.ms();
                }
                if (joined) OG_HIP(hipStreamWaitEvent(s, d->ev_static, 0));
                after(nullptr);
            }
            {
                EventSpan span(d, &tm.front, s);
                frontier_compact(d, d->fr, s, nf_val, true, pm);
            }
            OG_HIP(hipStreamSynchronize(s));
        }
    }
}

// Adds a traversal's statistics, whose run block is on the host.
template <int ALGO, bool W>
static void collect_loop(DeviceState *d, og_run_stats &st) {
    const RoundCtl c = d->fr.h_blk->ctl;
    const bool has_dyn = d->plan.vsplit < d->V;
    if (c.overflow) raise(OG_EUNSUPPORTED, "multi-source BFS deeper than 254 levels");
    st.iterations += c.rounds;
    st.node_sum += c.node_sum;
    st.static_node_sum += c.static_node_sum;
    st.work_edges += c.work_edges;
    st.static_work_edges += c.static_work_edges;
    // per edge: the edge in the device format (d->eb bytes) + the target state
    const uint64_t per_edge = edge_bytes_alg<ALGO, W>() - (W ? 8ull : 4ull) + d->eb;
    const uint64_t dyn_edges = c.work_edges - c.static_work_edges;
    st.relax_static_bytes += 24ull * c.static_node_sum + per_edge * c.static_work_edges;
    st.relax_dynamic_bytes += 24ull * c.dyn_node_sum + per_edge * dyn_edges;
    st.frontier_bytes += 2ull * d->Vpad * c.compactions + 4ull * c.node_sum;
    if (has_dyn && d->in_place) {  // every active dynamic edge read in place (HBM-resident ones taken off later)
        st.h2d_bytes += dyn_edges;
        st.chunks += c.dyn_rounds;
    }
}

static void finish_stats(og_run_stats &st, RunTimers &tm, double gather_ms, double overload_wall, const DeviceState *d,
                         uint64_t upd_bytes) {
    const RunBlock &h = *d->fr.h_blk;
    const unsigned long long *ctr = h.counters;
    if (tm.clocked >= 0) {
        tm.at(tm.clocked).ms += (double)(int64_t)h.clk.acc[kClkRelax] / d->clock_khz;
        tm.front.ms += (double)(int64_t)h.clk.acc[kClkFront] / d->clock_khz;
    }
    st.updates = ctr[0] + ctr[1];
    // zero-copy: h2d_bytes counts edges so far; those served from the
    // HBM-resident blocks did not cross the link
    if (d->in_place) {
        const uint64_t crossed = st.h2d_bytes - std::min<uint64_t>(st.h2d_bytes, ctr[5]);
        st.h2d_bytes = d->lbits ? (crossed * d->lbits + 7) / 8 : crossed * d->deb;
    }
    st.relax_static_bytes += upd_bytes * ctr[0];
    st.relax_dynamic_bytes += upd_bytes * ctr[1];
    st.frontier_kernel_ms = sum_ms(tm.front);
    st.frontier_launches = tm.front.launches;
    st.relax_static_kernel_ms = sum_ms(tm.stat);
    st.relax_static_launches = tm.stat.launches;
    st.relax_dynamic_kernel_ms = sum_ms(tm.dyn);
    st.relax_dynamic_launches = tm.dyn.launches;
    st.copy_ms = sum_ms(tm.copy);
    st.pre_ms = st.frontier_kernel_ms;
    st.static_ms = st.relax_static_kernel_ms;
    st.overload_ms = overload_wall;
    st.overload_move_ms = st.copy_ms;
    st.gather_ms = gather_ms;
}

// Whether a run is one launch of k_small: a small graph wholly in HBM (the A/B
// flags keep the rounds).
template <int ALGO>
static bool one_launch(const DeviceState *d) {
    return !d->managed && d->plan.vsplit >= d->V && d->V <= (ALGO == ALGO_CC ? kSmallVcc : kSmallV) &&
           d->E <= kSmallE && !(d->flags & (OG_PLAN_NO_FUSE | OG_PLAN_NO_OVERLAP));
}

template <int ALGO, bool W>
static void run_frontier(og_graph *g, uint32_t src, uint32_t *out, og_run_stats *stats, DeviceState *dv = nullptr) {
    DeviceState *d = dv ? dv : g->dev;
    const uint64_t V = d->V;
    og_run_stats st{};
    st.approach = (uint32_t)d->approach;
    RunTimers tm;
    d->events.reset();
    double gather_ms = 0, overload_wall = 0;
    hipStream_t s = d->s_compute;

    OG_HIP(hipStreamSynchronize(d->s_copy));
    OG_HIP(hipStreamSynchronize(d->s_static));
    OG_HIP(hipStreamSynchronize(s));
    Stopwatch total;
    if (one_launch<ALGO>(d)) {
        std::unique_lock<std::mutex> use;
        if (out) use = take_stage(d, V * 4);
        const bool direct = use.owns_lock();
        __atomic_store_n(d->fr.h_progress, 0ull, __ATOMIC_RELEASE);
        const SmallArgs a{d->d_ptr, d->d_static, d->wbits, (uint32_t)V, src, d->d_val,
                          direct ? (uint32_t *)d->out->buf : nullptr, d->fr.blk, d->fr.h_blk, d->fr.h_progress, false, 0};
        if (W && d->packed) launch_small<ALGO, W, true>(a, s);
        else launch_small<ALGO, W, false>(a, s);
        wait_progress(d->fr.h_progress, 1, s);
        if (!__atomic_load_n(d->fr.h_progress, __ATOMIC_ACQUIRE)) OG_HIP(hipStreamSynchronize(s));
        st.total_ms = total.ms();
        if (direct) std::memcpy(out, d->out->buf, V * 4);
        else if (out) copy_to_host(d, out, d->d_val, V * 4, s);
        tm.stat.launches = 1;
        tm.clocked = kClsStat;
        collect_loop<ALGO, W>(d, st);
        st.reached = d->fr.h_blk->counters[2];
        st.traversed_edges = d->fr.h_blk->counters[3];
        st.checksum = d->fr.h_blk->counters[4];
        finish_stats(st, tm, gather_ms, overload_wall, d, 8);
        if (stats) *stats = st;
        return;
    }
    auto begin = [&](const RoundCtl &c) {
        hipLaunchKernelGGL((k_run_init<ALGO == ALGO_CC>), dim3(fill_grid(d->Vpad / 4)), dim3(kBlock), 0, s, d->d_val,
                           d->fr.flag, V, d->Vpad, src, d->fr.blk, d->fr.spread, c);
        OG_HIP(hipGetLastError());
    };
    frontier_loop<ALGO, W>(g, d, st, tm, gather_ms, overload_wall, begin, [](RoundClock *) {}, true);
    st.total_ms = total.ms();

    hipLaunchKernelGGL(k_reach_stats, dim3(stats_grid(V)), dim3(kStatsBlock), 0, s, d->d_val, d->d_ptr, d->d_deg,
                       d->deg_heavy(), V, d->fr.counters, d->fr.spread, tm.clocked >= 0 ? d->fr.clk : nullptr);
    OG_HIP(hipGetLastError());
    OG_HIP(hipMemcpyAsync(d->fr.h_blk, d->fr.blk, sizeof(RunBlock), hipMemcpyDeviceToHost, s));
    if (out) copy_to_host(d, out, d->d_val, V * sizeof(uint32_t), s);
    OG_HIP(hipStreamSynchronize(s));
    collect_loop<ALGO, W>(d, st);
    st.reached = d->fr.h_blk->counters[2];
    st.traversed_edges = d->fr.h_blk->counters[3];
    st.checksum = d->fr.h_blk->counters[4];
    finish_stats(st, tm, gather_ms, overload_wall, d, 8);
    if (stats) *stats = st;
}

// Multi-source BFS: sources in batches of 64, two batches walking the graph
// together while more than 64 sources are left; per vertex and batch, u64 masks
// of the sources that reached it, that were offered to it this round (side by
// side) and whose frontier holds it; levels as u8 per (vertex, source) when the
// caller wants them.
constexpr uint64_t kExtractBytes = 256ull << 20;  // device buffer of levels on their way to the host, at most

// Workgroups of the commit sweep.
static unsigned ms_commit_grid(uint64_t V) {
    return (unsigned)std::min<uint64_t>(kMsCommitGrid, std::max<uint64_t>(1, (V + kBlock - 1) / kBlock));
}

// The state for a walk of H masks per vertex.  Narrower arrays leave before
// wider ones take their place, with the captured rounds that hold their addresses.
static DeviceState::MsState &ms_state(DeviceState *d, uint32_t H, bool levels) {
    DeviceState::MsState &m = d->d_ms;
    const uint64_t V = d->V;
    if (m.masks < H) {
        if (m.vn) d->round_graph.reset();
        m.masks = 0;
        d->mem.dfree(m.vn);
        d->mem.dfree(m.front);
        d->mem.dfree(m.src);
        d->mem.dfree(m.part);
        d->mem.dfree(m.sum);
        m.vn = (ulonglong2 *)d->dalloc(H * V * 16);
        m.front = (uint64_t *)d->dalloc(H * V * 8);
        m.src = (uint32_t *)d->dalloc(H * kMsWidth * 4);
        m.part = (unsigned long long *)d->dalloc((uint64_t)ms_commit_grid(V) * H * kMsSums * 8);
        m.sum = (unsigned long long *)d->dalloc(H * kMsSums * 8);
        m.masks = H;
    }
    if (levels && m.lvl_masks < H) {
        if (m.lvl) d->round_graph.reset();
        m.lvl_masks = 0;
        d->mem.dfree(m.lvl);
        m.lvl = (uint8_t *)d->dalloc(H * V * kMsWidth);
        m.lvl_masks = H;
    }
    return m;
}

// One traversal from nb <= 64 H sources.
template <int H, bool W>
static void ms_batch(og_graph *g, DeviceState *d, const uint32_t *sources, uint32_t nb, uint32_t *levels,
                     uint64_t *checksums, uint64_t *reached, og_run_stats &st, RunTimers &tm, double &gather_ms,
                     double &overload_wall, const Stopwatch &total, double &device_ms) {
    constexpr int ALGO = H == 1 ? ALGO_MSBFS : ALGO_MSBFS2;
    const uint64_t V = d->V;
    hipStream_t s = d->s_compute;
    DeviceState::MsState &m = ms_state(d, H, levels != nullptr);
    const unsigned cgrid = ms_commit_grid(V);
    if (levels && !d->d_extract) {  // fewer sources at a time where memory is short
        uint32_t cap = (uint32_t)std::min<uint64_t>(kMsWidth, std::max<uint64_t>(1, kExtractBytes / (V * 4)));
        void *p = nullptr;
        while (cap > 1 && !(p = d->mem.try_dalloc((uint64_t)cap * V * 4))) cap /= 2;
        d->d_extract = (uint32_t *)(p ? p : d->dalloc((uint64_t)cap * V * 4));
        d->extract_cap = cap;
    }
    uint8_t *const lvl = levels ? m.lvl : nullptr;
    std::vector<unsigned long long> hsum(H * kMsSums);
    if (lvl) OG_HIP(hipMemsetAsync(lvl, 0, H * V * kMsWidth, s));
    OG_HIP(hipMemcpyAsync(m.src, sources, nb * 4, hipMemcpyHostToDevice, s));
    auto begin = [&](const RoundCtl &c) {
        hipLaunchKernelGGL(k_ms_clear<H>, dim3(fill_grid(V)), dim3(kBlock), 0, s, m.vn, m.front, d->fr.flag, V, d->Vpad,
                           m.part, (uint64_t)cgrid * H * kMsSums, d->fr.ctl, c);
        hipLaunchKernelGGL(k_ms_init<H>, dim3(1), dim3(H * kMsWidth), 0, s, m.src, nb, m.vn, m.front, d->fr.flag, lvl, V,
                           d->d_ptr, m.part);
        OG_HIP(hipGetLastError());
    };
    auto commit = [&](RoundClock *clk) {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(cgrid), dim3(kBlock), 0, s, d->fr.flag, V, m.vn, m.front, lvl, d->d_ptr,
                               d->d_deg, d->deg_heavy(), d->fr.ctl, m.part, clk);
        };
        if (lvl) launch(k_ms_commit<true, H>);
        else launch(k_ms_commit<false, H>);
        OG_HIP(hipGetLastError());
    };
    frontier_loop<ALGO, W>(g, d, st, tm, gather_ms, overload_wall, begin, commit, false, lvl != nullptr);
    hipLaunchKernelGGL(k_ms_sum, dim3(3 * H), dim3(1024), 0, s, m.part, cgrid, m.sum, d->fr.counters, d->fr.spread,
                       tm.clocked >= 0 ? d->fr.clk : nullptr);
    OG_HIP(hipGetLastError());
    OG_HIP(hipMemcpyAsync(d->fr.h_blk, d->fr.blk, sizeof(RunBlock), hipMemcpyDeviceToHost, s));
    OG_HIP(hipMemcpyAsync(hsum.data(), m.sum, H * kMsSums * 8, hipMemcpyDeviceToHost, s));
    OG_HIP(hipStreamSynchronize(s));
    device_ms = total.ms();
    collect_loop<ALGO, W>(d, st);
    for (uint32_t j = 0; j < nb; ++j) {
        const unsigned long long *const x = hsum.data() + j / kMsWidth * kMsSums + j % kMsWidth;
        if (checksums) checksums[j] = x[0];
        if (reached) reached[j] = x[kMsWidth];
        st.reached += x[kMsWidth];
        st.traversed_edges += x[2 * kMsWidth];
        st.checksum += x[0];
    }
    if (!levels) return;
    for (uint32_t j = 0; j < nb;) {  // groups of sources of one mask
        const uint32_t h = j / kMsWidth, j0 = j % kMsWidth;
        const uint32_t nj = std::min({d->extract_cap, nb - j, (uint32_t)kMsWidth - j0});
        hipLaunchKernelGGL(k_ms_extract, dim3((unsigned)std::min<uint64_t>(8192, (V + kWave - 1) / kWave)), dim3(kBlock),
                           0, s, lvl + (uint64_t)h * V * kMsWidth, V, j0, nj, d->d_extract);
        OG_HIP(hipGetLastError());
        copy_to_host(d, levels + (uint64_t)j * V, d->d_extract, (uint64_t)nj * V * 4, s);
        j += nj;
    }
}

// Whether two batches of sources walk the graph together.  A dense round costs
// the reading of the edges (over the link, or random reads of the targets'
// masks, whose line two batches share), so a walk with two masks per vertex
// takes little more than one with one: R-MAT 4 M vertices 67 M edges, 128
// sources, 0.4 of the edges in HBM: 12.0 -> 6.8 ms, in HBM 6.1 -> 4.4; 4096
// vertices 0.48 -> 0.26; 72 sources 11.0 -> 6.4, 5.4 -> 4.0, 0.46 -> 0.25.  It was faster at
// every size and for as few as 8 sources in the second batch; the line is the
// memory that the wider masks (and levels) take, an eighth of what is free.
static bool ms_wide(const DeviceState *d, uint32_t left, bool levels) {
    if (left <= kMsWidth) return false;
    const DeviceState::MsState &m = d->d_ms;
    const uint64_t more = (24 * (2 - m.masks) + (levels ? kMsWidth * (2 - m.lvl_masks) : 0)) * d->V;
    if (!more) return true;
    size_t free = 0, all = 0;
    OG_HIP(hipMemGetInfo(&free, &all));
    return more <= free / 8;
}

template <bool W>
static void run_msbfs(og_graph *g, const uint32_t *sources, uint32_t n, uint32_t *levels, uint64_t *checksums,
                      uint64_t *reached, og_run_stats *stats) {
    DeviceState *d = g->dev;
    hipStream_t s = d->s_compute;
    og_run_stats st{};
    st.approach = (uint32_t)d->approach;
    RunTimers tm;
    d->events.reset();
    double gather_ms = 0, overload_wall = 0, device_ms = 0;
    OG_HIP(hipStreamSynchronize(d->s_copy));
    OG_HIP(hipStreamSynchronize(d->s_static));
    OG_HIP(hipStreamSynchronize(s));
    Stopwatch total;
    OG_HIP(hipMemsetAsync(d->fr.blk, 0, sizeof(RunBlock), s));
    OG_HIP(hipMemsetAsync(d->fr.spread, 0, kSpreadWords * 8, s));
    for (uint32_t b0 = 0, nb = 0; b0 < n; b0 += nb) {
        const bool wide = ms_wide(d, n - b0, levels != nullptr);
        nb = std::min<uint32_t>(wide ? 2 * kMsWidth : kMsWidth, n - b0);
        auto run = [&](auto batch) {
            batch(g, d, sources + b0, nb, levels ? levels + (uint64_t)b0 * d->V : nullptr,
                  checksums ? checksums + b0 : nullptr, reached ? reached + b0 : nullptr, st, tm, gather_ms,
                  overload_wall, total, device_ms);
        };
        if (wide) run(ms_batch<2, W>);
        else run(ms_batch<1, W>);
    }
    st.total_ms = device_ms;
    if (!n) *d->fr.h_blk = RunBlock{};
    finish_stats(st, tm, gather_ms, overload_wall, d, 9);
    if (stats) *stats = st;
}

DeviceState *lane_state_create(og_graph *g, uint32_t delta) {
    const DeviceState *d = g->dev;
    if (d->plan.vsplit < d->V || d->managed) raise(OG_EUNSUPPORTED, "a lane needs the whole graph in device memory");
    std::unique_ptr<DeviceState, void (*)(DeviceState *)> l(new DeviceState, device_state_free);
    // the graph as prepared (read only: every array below belongs to g->dev)
    l->approach = d->approach;
    l->device = d->device;
    l->clock_khz = d->clock_khz;
    l->V = d->V;
    l->E = d->E;
    l->Vpad = d->Vpad;
    l->eb = d->eb;
    l->deb = d->deb;
    l->plan = d->plan;
    l->tune = d->tune;
    if (delta) l->tune.delta = delta;
    l->host_threads = d->host_threads;
    l->flags = d->flags;
    l->d_ptr = d->d_ptr;
    l->d_pmid = d->d_pmid;
    l->d_deg = d->d_deg;
    l->deg_split = d->deg_split;
    l->split_weight = d->split_weight;
    l->d_static = d->d_static;
    l->static_used = d->static_used;
    l->packed = d->packed;
    l->wbits = d->wbits;
    l->d_in_ptr = d->d_in_ptr;
    l->d_in_cols = d->d_in_cols;
    // the lane's own run state, on one stream: a graph wholly in HBM has no
    // dynamic region to copy or overlap, and every stream of a process takes
    // a hardware queue (or shares one) while the server runs
    OG_HIP(hipSetDevice(d->device));
    OG_HIP(hipStreamCreateWithFlags(&l->s_compute, hipStreamNonBlocking));
    l->s_copy = l->s_static = l->s_compute;
    OG_HIP(hipEventCreateWithFlags(&l->ev_static, hipEventDisableTiming));
    OG_HIP(hipEventCreateWithFlags(&l->ev_fork, hipEventDisableTiming));
    l->d_val = (uint32_t *)l->dalloc(l->Vpad * sizeof(uint32_t));
    frontier_alloc(l.get(), g, l->fr, l->mem);
    OG_HIP(hipDeviceSynchronize());
    return l.release();
}

uint64_t lane_state_bytes(const og_graph *g) {
    const DeviceState *d = g->dev;
    const uint64_t V = d->V, Vpad = d->Vpad;
    const uint64_t nblk = (Vpad + verts_per_block(compact_nw(V)) - 1) / verts_per_block(compact_nw(V));
    const uint64_t hub = std::max<uint64_t>(hub_capacity(g, d->plan.vsplit, d->tune), 1);
    // what lane_state_create and frontier_alloc request: values, flags (and
    // the heavy-round flags with the split), bin lists, degree prefix, the
    // (empty) dynamic chunk table, compaction totals, round summary, run
    // block, work counters and hub tiles
    return 4 * Vpad + Vpad * (d->d_pmid ? 2 : 1) + 4 * V + 8 * (V + 1) + 4 * 2 + 8 * totals_words(nblk) +
           sizeof(FrontierInfo) + sizeof(RunBlock) + 8 * kSpreadWords + 8 * hub;
}

void lane_run_sssp(og_graph *g, DeviceState *lane, uint32_t src, uint32_t *out, og_run_stats *st) {
    run_frontier<ALGO_SSSP, true>(g, src, out, st, lane);
}

static og_status run_algo(og_graph *g, int algo, uint32_t src, uint32_t *out, og_run_stats *stats) {
    clear_error();
    if (!g) return fail(OG_EINVAL, "graph is NULL");
    if (!g->dev) return fail(OG_ESTATE, "og_prepare has not been called for this graph");
    if (algo != ALGO_CC && src >= g->V) return fail(OG_EINVAL, "source %u >= V=%llu", src, (unsigned long long)g->V);
    if (g->kind == OG_KIND_PULL) return fail(OG_EUNSUPPORTED, "pull-layout graphs serve PageRank only");
    if (algo == ALGO_SSSP && g->kind != OG_KIND_WEIGHTED) return fail(OG_EUNSUPPORTED, "SSSP needs a weighted graph");
    int expect = 0;
    if (!g->busy.compare_exchange_strong(expect, 1)) return fail(OG_EBUSY, "graph is running another call");
    og_status st = guard([&]() -> og_status {
        OG_HIP(hipSetDevice(g->dev->device));
        const bool w = g->kind == OG_KIND_WEIGHTED;
        if (algo == ALGO_BFS) {
            if (w) run_frontier<ALGO_BFS, true>(g, src, out, stats);
            else run_frontier<ALGO_BFS, false>(g, src, out, stats);
        } else if (algo == ALGO_SSSP) {
            run_frontier<ALGO_SSSP, true>(g, src, out, stats);
        } else {
            if (w) run_frontier<ALGO_CC, true>(g, 0, out, stats);
            else run_frontier<ALGO_CC, false>(g, 0, out, stats);
        }
        return OG_OK;
    });
    g->busy.store(0);
    return st;
}

}  // namespace og

using namespace og;

extern "C" og_status og_prepare(og_graph *g, og_approach approach, const og_plan_params *params, og_plan_info *info) {
    clear_error();
    if (!g) return fail(OG_EINVAL, "graph is NULL");
    int expect = 0;
    if (!g->busy.compare_exchange_strong(expect, 1)) return fail(OG_EBUSY, "graph is running another call");
    og_status st = guard([&]() -> og_status {
        prepare_impl(g, approach, params, info);
        return OG_OK;
    });
    g->busy.store(0);
    return st;
}

extern "C" og_status og_release(og_graph *g) {
    clear_error();
    if (!g) return fail(OG_EINVAL, "graph is NULL");
    int expect = 0;
    if (!g->busy.compare_exchange_strong(expect, 1)) return fail(OG_EBUSY, "graph is running another call");
    device_state_free(g->dev);
    g->dev = nullptr;
    g->busy.store(0);
    return OG_OK;
}

extern "C" og_status og_bfs(og_graph *g, uint32_t source, uint32_t *levels, og_run_stats *stats) {
    return run_algo(g, ALGO_BFS, source, levels, stats);
}

extern "C" og_status og_sssp(og_graph *g, uint32_t source, uint32_t *dist, og_run_stats *stats) {
    return run_algo(g, ALGO_SSSP, source, dist, stats);
}

extern "C" og_status og_cc(og_graph *g, uint32_t *labels, og_run_stats *stats) {
    return run_algo(g, ALGO_CC, 0, labels, stats);
}

extern "C" og_status og_msbfs(og_graph *g, const uint32_t *sources, uint32_t num_sources, uint32_t *levels,
                              uint64_t *checksums, uint64_t *reached, og_run_stats *stats) {
    clear_error();
    if (!g || (!sources && num_sources)) return fail(OG_EINVAL, "graph/sources is NULL");
    if (!g->dev) return fail(OG_ESTATE, "og_prepare has not been called for this graph");
    if (g->kind == OG_KIND_PULL) return fail(OG_EUNSUPPORTED, "pull-layout graphs serve PageRank only");
    for (uint32_t i = 0; i < num_sources; ++i)
        if (sources[i] >= g->V) return fail(OG_EINVAL, "source %u >= V", sources[i]);
    int expect = 0;
    if (!g->busy.compare_exchange_strong(expect, 1)) return fail(OG_EBUSY, "graph is running another call");
    og_status st = guard([&]() -> og_status {
        OG_HIP(hipSetDevice(g->dev->device));
        if (g->kind == OG_KIND_WEIGHTED) run_msbfs<true>(g, sources, num_sources, levels, checksums, reached, stats);
        else run_msbfs<false>(g, sources, num_sources, levels, checksums, reached, stats);
        return OG_OK;
    });
    g->busy.store(0);
    return st;
}

// ------------------------------------------------------------ link probe

namespace og {

__global__ __launch_bounds__(kBlock) void k_probe_contig(const uint32_t *__restrict__ p, uint64_t n, uint32_t *out) {
    uint32_t acc = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock) acc ^= p[i];
    if (acc == 0x9E3779B9u) out[0] = acc;  // keeps the reads alive
}

// Rows r = [off[r], off[r+1]) of the concatenated space start at base[r] in p;
// lane q finds its row by binary search (as k_relax_dyn does).
__global__ __launch_bounds__(kBlock) void k_probe_rows(const uint32_t *__restrict__ p,
                                                       const uint64_t *__restrict__ off,
                                                       const uint64_t *__restrict__ base, uint32_t nrows, uint64_t m,
                                                       uint32_t *out) {
    uint32_t acc = 0;
    for (uint64_t q = (uint64_t)blockIdx.x * kBlock + threadIdx.x; q < m; q += (uint64_t)gridDim.x * kBlock) {
        uint32_t lo = 0, hi = nrows;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (off[mid] <= q) lo = mid; else hi = mid;
        }
        acc ^= p[base[lo] + (q - off[lo])];
    }
    if (acc == 0x9E3779B9u) out[0] = acc;
}

}  // namespace og

namespace og {

// Random 4-byte gathers from a table of n words: each lane draws its indices
// with SplitMix64 from its own counter and keeps kGatherIlp loads in flight.
constexpr int kGatherIlp = 8;
__global__ __launch_bounds__(kBlock) void k_probe_gather(const uint32_t *__restrict__ t, uint64_t n, uint64_t per,
                                                         uint64_t seed, uint32_t *out) {
    const uint64_t tid = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    uint32_t acc = 0;
    for (uint64_t i = 0; i < per; i += kGatherIlp) {
        uint32_t x[kGatherIlp];
#pragma unroll
        for (int k = 0; k < kGatherIlp; ++k) x[k] = t[d_mix64(seed + tid * per + i + k) % n];
#pragma unroll
        for (int k = 0; k < kGatherIlp; ++k) acc ^= x[k];
    }
    if (acc == 0x9E3779B9u) out[0] = acc;  // keeps the reads alive
}

}  // namespace og

// Random-gather probe (no reference counterpart: a measurement helper for the
// relax kernels, whose per-edge target reads are random 4-byte accesses).
extern "C" og_status og_probe_hbm_gather(uint64_t table_bytes, double *gather_gbs, double *mgathers_per_s) {
    clear_error();
    if (table_bytes < (1u << 16) || table_bytes > (64ull << 30)) return fail(OG_EINVAL, "table must be 64 KiB .. 64 GiB");
    return guard([&]() -> og_status {
        if (!hip_available()) raise(OG_EHIP, "no HIP device is visible");
        MemPool m;
        const uint64_t n = table_bytes / 4;
        uint32_t *t = (uint32_t *)m.dalloc(n * 4);
        uint32_t *dout = (uint32_t *)m.dalloc(4);
        hipLaunchKernelGGL(k_iota, dim3(fill_grid(n)), dim3(256), 0, 0, t, n);
        const unsigned grid = 8192;
        const uint64_t per = 8 * kGatherIlp;  // gathers per lane
        const double total = (double)grid * kBlock * per;
        hipEvent_t a, b;
        OG_HIP(hipEventCreate(&a));
        OG_HIP(hipEventCreate(&b));
        hipLaunchKernelGGL(k_probe_gather, dim3(grid), dim3(kBlock), 0, 0, t, n, per, 1ull, dout);
        OG_HIP(hipDeviceSynchronize());
        OG_HIP(hipEventRecord(a, 0));
        for (int r = 0; r < 3; ++r)
            hipLaunchKernelGGL(k_probe_gather, dim3(grid), dim3(kBlock), 0, 0, t, n, per, 2ull + r, dout);
        OG_HIP(hipEventRecord(b, 0));
        OG_HIP(hipEventSynchronize(b));
        OG_HIP(hipGetLastError());
        float ms = 0;
        OG_HIP(hipEventElapsedTime(&ms, a, b));
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
        const double per_s = 3.0 * total / (ms * 1e-3);
        if (gather_gbs) *gather_gbs = per_s * 4 / 1e9;
        if (mgathers_per_s) *mgathers_per_s = per_s / 1e6;
        return OG_OK;
    });
}

extern "C" og_status og_probe_host_link(uint64_t bytes, double *contig_gbs, double *scattered_gbs,
                                        double *memcpy_gbs) {
    clear_error();
    if (bytes < (1u << 20) || bytes > (64ull << 30)) return fail(OG_EINVAL, "probe size must be 1 MiB .. 64 GiB");
    return guard([&]() -> og_status {
        if (!hip_available()) raise(OG_EHIP, "no HIP device is visible");
        MemPool m;
        const uint64_t n = bytes / 4;
        uint32_t *h = (uint32_t *)m.palloc(n * 4);
        parallel_for(n, 1 << 20, 0, [&](uint64_t b, uint64_t e, unsigned) {
            for (uint64_t i = b; i < e; ++i) h[i] = (uint32_t)i;
        });
        void *hd = nullptr;
        OG_HIP(hipHostGetDevicePointer(&hd, h, 0));
        // rows of 1..19 words with gaps of 0..39 words (SplitMix64 draws)
        std::vector<uint64_t> off{0}, base;
        uint64_t pos = 0, key = rng_key(7);
        for (uint64_t r = 0;; ++r) {
            const uint64_t x = rng_draw(key, r);
            const uint64_t len = 1 + x % 19, gap = (x >> 32) % 40;
            if (pos + gap + len > n) break;
            pos += gap;
            base.push_back(pos);
            pos += len;
            off.push_back(off.back() + len);
        }
        const uint32_t nrows = (uint32_t)base.size();
        const uint64_t mwords = off.back();
        uint64_t *doff = (uint64_t *)m.dalloc(off.size() * 8), *dbase = (uint64_t *)m.dalloc(base.size() * 8 + 8);
        uint32_t *dout = (uint32_t *)m.dalloc(4), *ddst = (uint32_t *)m.dalloc(n * 4);
        OG_HIP(hipMemcpy(doff, off.data(), off.size() * 8, hipMemcpyHostToDevice));
        OG_HIP(hipMemcpy(dbase, base.data(), base.size() * 8, hipMemcpyHostToDevice));
        hipEvent_t a, b;
        OG_HIP(hipEventCreate(&a));
        OG_HIP(hipEventCreate(&b));
        auto timed = [&](double useful, auto fn) {
            fn();
            OG_HIP(hipDeviceSynchronize());
            OG_HIP(hipEventRecord(a, 0));
            for (int r = 0; r < 3; ++r) fn();
            OG_HIP(hipEventRecord(b, 0));
            OG_HIP(hipEventSynchronize(b));
            float ms = 0;
            OG_HIP(hipEventElapsedTime(&ms, a, b));
            return 3.0 * useful / (ms * 1e-3) / 1e9;
        };
        const double c = timed((double)n * 4, [&] {
            hipLaunchKernelGGL(k_probe_contig, dim3(4096), dim3(kBlock), 0, 0, (const uint32_t *)hd, n, dout);
        });
        const double sc = timed((double)mwords * 4, [&] {
            hipLaunchKernelGGL(k_probe_rows, dim3(4096), dim3(kBlock), 0, 0, (const uint32_t *)hd, doff, dbase, nrows,
                               mwords, dout);
        });
        const double mc = timed((double)n * 4, [&] { OG_HIP(hipMemcpyAsync(ddst, h, n * 4, hipMemcpyHostToDevice, 0)); });
        OG_HIP(hipGetLastError());
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
        if (contig_gbs) *contig_gbs = c;
        if (scattered_gbs) *scattered_gbs = sc;
        if (memcpy_gbs) *memcpy_gbs = mc;
        return OG_OK;
    });
}

// Host digest of a result array, equal to the one the device computes:
// sum (mod 2^64) of mix64(v << 32 | value[v]) over v with value != UNREACHED.
extern "C" og_status og_levels_checksum(const uint32_t *values, uint64_t num_vertices, uint64_t *checksum) {
    if (!values || !checksum) return fail(OG_EINVAL, "null argument");
    uint64_t h = 0;
    for (uint64_t v = 0; v < num_vertices; ++v)
        if (values[v] != OG_UNREACHED) h += mix64((v << 32) | values[v]);
    *checksum = h;
    return OG_OK;
}

// ------------------------------------------------------------------ tuning

namespace og {

static og_status check_tuning(const og_tuning *t) {
    const uint32_t l = t->lpv0;
    if (!(l == 1 || l == 2 || l == 4 || l == 8 || l == 16 || l == 32 || l == 64))
        return fail(OG_EINVAL, "lpv0 must be a power of two in [1, 64]");
    if (t->t1 < 1 || t->t2 < t->t1) return fail(OG_EINVAL, "need 1 <= t1 <= t2");
    if (t->tile < 64 || t->tile > 4096) return fail(OG_EINVAL, "tile must be in [64, 4096]");
    if (t->defer > 2) return fail(OG_EINVAL, "defer must be 0, 1 or 2");
    if (t->dyn_grid > 65535) return fail(OG_EINVAL, "dyn_grid must be at most 65535");
    return OG_OK;
}

static void apply_tuning(og_graph *g, const og_tuning *t) {
    DeviceState *d = g->dev;
    d->tune.t1 = t->t1;
    d->tune.lpv0 = t->lpv0;
    d->tune.t2 = t->t2;
    d->tune.tile = t->tile;
    d->tune.delta = t->delta;
    d->tune.defer = t->defer;
    d->tune.dyn_grid = t->dyn_grid;
    const uint64_t cap = hub_capacity(g, d->plan.vsplit, d->tune);
    if (cap > d->fr.hub_cap) {
        d->fr.hub = (uint64_t *)d->dalloc(cap * sizeof(uint64_t));
        d->fr.hub_cap = cap;
    }
    d->pr_plan.reset();      // PageRank bins follow t1 / t2
    d->round_graph.reset();  // captured rounds hold the tuning and the hub list
}

static og_tuning tuning_of(const DeviceState *d) {
    return og_tuning{d->tune.t1, d->tune.lpv0, d->tune.t2, d->tune.tile, d->tune.delta, d->tune.defer,
                     d->tune.dyn_grid};
}

// The multi-source tuning batch: 64 sources drawn uniformly (SplitMix64
// seeded with `seed`) among the vertices with out-edges.
static std::vector<uint32_t> tune_sources(const og_graph *g, uint32_t seed) {
    std::vector<uint32_t> cand;
    for (uint64_t v = 0; v < g->V; ++v)
        if (g->ptr[v + 1] > g->ptr[v]) cand.push_back((uint32_t)v);
    std::vector<uint32_t> out;
    if (cand.empty()) return out;
    const uint64_t key = rng_key(seed);
    for (uint32_t i = 0; i < (uint32_t)kMsWidth; ++i) out.push_back(cand[rng_draw(key, i) % cand.size()]);
    return out;
}

static double time_algo(og_graph *g, uint32_t algo, uint32_t src, uint32_t runs) {
    std::vector<double> ts;
    const bool w = g->kind == OG_KIND_WEIGHTED;
    const std::vector<uint32_t> batch = algo == OG_TUNE_MSBFS ? tune_sources(g, src) : std::vector<uint32_t>();
    for (uint32_t r = 0; r < runs; ++r) {
        og_run_stats st;
        if (algo == OG_TUNE_MSBFS) {
            if (w) run_msbfs<true>(g, batch.data(), (uint32_t)batch.size(), nullptr, nullptr, nullptr, &st);
            else run_msbfs<false>(g, batch.data(), (uint32_t)batch.size(), nullptr, nullptr, nullptr, &st);
        } else if (algo == OG_TUNE_BFS) {
            if (w) run_frontier<ALGO_BFS, true>(g, src, nullptr, &st);
            else run_frontier<ALGO_BFS, false>(g, src, nullptr, &st);
        } else if (algo == OG_TUNE_SSSP) {
            run_frontier<ALGO_SSSP, true>(g, src, nullptr, &st);
        } else {
            if (w) run_frontier<ALGO_CC, true>(g, 0, nullptr, &st);
            else run_frontier<ALGO_CC, false>(g, 0, nullptr, &st);
        }
        ts.push_back(st.total_ms);
    }
    std::sort(ts.begin(), ts.end());
    return ts[ts.size() / 2];
}

}  // namespace og

extern "C" og_status og_get_tuning(const og_graph *g, og_tuning *t) {
    clear_error();
    if (!g || !t) return fail(OG_EINVAL, "null argument");
    if (!g->dev) return fail(OG_ESTATE, "og_prepare has not been called for this graph");
    *t = tuning_of(g->dev);
    return OG_OK;
}

extern "C" og_status og_set_tuning(og_graph *g, const og_tuning *t) {
    clear_error();
    if (!g || !t) return fail(OG_EINVAL, "null argument");
    if (!g->dev) return fail(OG_ESTATE, "og_prepare has not been called for this graph");
    og_status st = check_tuning(t);
    if (st != OG_OK) return st;
    int expect = 0;
    if (!g->busy.compare_exchange_strong(expect, 1)) return fail(OG_EBUSY, "graph is running another call");
    st = guard([&]() -> og_status {
        apply_tuning(g, t);
        return OG_OK;
    });
    g->busy.store(0);
    return st;
}

extern "C" og_status og_autotune(og_graph *g, uint32_t algo, uint32_t source, uint32_t runs, og_tuning *best,
                                 double *best_ms) {
    clear_error();
    if (!g) return fail(OG_EINVAL, "graph is NULL");
    if (!g->dev) return fail(OG_ESTATE, "og_prepare has not been called for this graph");
    if (algo > OG_TUNE_MSBFS)
        return fail(OG_EINVAL, "algo must be OG_TUNE_BFS, OG_TUNE_SSSP, OG_TUNE_CC or OG_TUNE_MSBFS");
    if (g->kind == OG_KIND_PULL) return fail(OG_EUNSUPPORTED, "pull-layout graphs serve PageRank only");
    if (algo == OG_TUNE_SSSP && g->kind != OG_KIND_WEIGHTED) return fail(OG_EUNSUPPORTED, "SSSP needs weights");
    if ((algo == OG_TUNE_BFS || algo == OG_TUNE_SSSP) && source >= g->V) return fail(OG_EINVAL, "source out of range");
    if (runs == 0) runs = 1;
    int expect = 0;
    if (!g->busy.compare_exchange_strong(expect, 1)) return fail(OG_EBUSY, "graph is running another call");
    og_status st = guard([&]() -> og_status {
        OG_HIP(hipSetDevice(g->dev->device));
        og_tuning cur = tuning_of(g->dev);
        (void)time_algo(g, algo, source, 1);  // warm-up
        double cur_ms = time_algo(g, algo, source, runs);
        auto trial = [&](og_tuning cand) {
            if (check_tuning(&cand) != OG_OK) return;
            apply_tuning(g, &cand);
            const double ms = time_algo(g, algo, source, runs);
            if (ms < cur_ms) {
                cur_ms = ms;
                cur = cand;
            }
            apply_tuning(g, &cur);
        };
        const bool has_dyn = g->dev->plan.vsplit < g->V;
        // a run in one launch has no shape to tune: the candidates would differ
        // by noise, and other calls on the preparation would get the choice
        const bool fixed = algo == OG_TUNE_BFS    ? one_launch<ALGO_BFS>(g->dev)
                           : algo == OG_TUNE_SSSP ? one_launch<ALGO_SSSP>(g->dev)
                           : algo == OG_TUNE_CC   ? one_launch<ALGO_CC>(g->dev)
                                                  : false;
        for (int pass = 0; pass < 2 && !fixed; ++pass) {
            if ((algo == OG_TUNE_SSSP || algo == OG_TUNE_CC) && has_dyn)
                for (uint32_t df : {0u, 1u, 2u}) {
                    og_tuning c = cur;
                    c.defer = df;
                    trial(c);
                }
            if (algo == OG_TUNE_SSSP)
                for (uint32_t dl : {0u, 8u, 16u, 32u, 64u, 128u, 256u, 512u}) {
                    og_tuning c = cur;
                    c.delta = dl;
                    trial(c);
                }
            for (uint32_t t1 : {4u, 8u, 16u, 32u, 64u})
                for (uint32_t l : {2u, 4u, 8u, 16u}) {
                    og_tuning c = cur;
                    c.t1 = t1;
                    c.lpv0 = l;
                    if (c.t2 < t1) c.t2 = t1;
                    trial(c);
                }
            for (uint32_t t2 : {512u, 1024u, 2048u, 4096u, 16384u, 65536u}) {
                og_tuning c = cur;
                c.t2 = std::max(t2, c.t1);
                trial(c);
            }
            for (uint32_t tile : {512u, 1024u, 2048u, 4096u}) {
                og_tuning c = cur;
                c.tile = tile;
                trial(c);
            }
            if (has_dyn)
                for (uint32_t dg : {512u, 1024u, 2048u, 4096u, 8192u}) {
                    og_tuning c = cur;
                    c.dyn_grid = dg;
                    trial(c);
                }
        }
        apply_tuning(g, &cur);
        if (best) *best = cur;
        if (best_ms) *best_ms = cur_ms;
        return OG_OK;
    });
    g->busy.store(0);
    return st;
}

// ==================================================== allocation-free BFS
//
// og_bfs_device_noalloc: og_bfs over a CSR that already sits in device
// memory, for callers that cannot allocate (hipMalloc / hipFree / an
// allocating library call) at run time.  Every buffer beyond the caller's
// inputs and output -- next-frontier flags, bin lists, hub tiles, compaction
// totals, the round's summary and control block, counters -- lives in the
// file-scope device array `scratch` below, sized for V <= kNoAllocMaxV and
// E <= kNoAllocMaxE.  Rounds are enqueued directly (no captured hipGraph, no
// events) after one kernel that sets everything up, so the call allocates
// nothing; graphs of k_small's size take its one launch.
// Each GPU holds its own copy of `scratch` until the process ends; calls
// that overlap on one GPU share it and race.

namespace og {

constexpr uint64_t kNoAllocMaxV = 1ull << 21;  // vertices
constexpr uint64_t kNoAllocMaxE = 1ull << 26;  // edges
constexpr uint64_t kNoAlign = 256;
constexpr uint64_t na_up(uint64_t x) { return (x + kNoAlign - 1) / kNoAlign * kNoAlign; }
// Hub tiles of any graph within the limits under the default tuning: a vertex
// of degree d > t2 takes ceil(d / tile) <= d / tile + 1 tiles, and at most
// E / (t2 + 1) vertices exceed t2.
constexpr uint64_t kNoAllocHubCap = kNoAllocMaxE / 2048 + kNoAllocMaxE / 4097 + 1;
static_assert(compact_nw(kNoAllocMaxV) == 1, "the allocation-free BFS runs the one-window compaction");
constexpr uint64_t kNoAllocMaxBlk = (kNoAllocMaxV + verts_per_block(1) - 1) / verts_per_block(1);
constexpr uint64_t kNaFlag = 0;
constexpr uint64_t kNaList = kNaFlag + na_up(kNoAllocMaxV);
constexpr uint64_t kNaHub = kNaList + na_up(4 * kNoAllocMaxV);
constexpr uint64_t kNaDoff = kNaHub + na_up(8 * kNoAllocHubCap);
constexpr uint64_t kNaTot = kNaDoff + na_up(8 * 16);
constexpr uint64_t kNaInfo = kNaTot + na_up(8 * totals_words(kNoAllocMaxBlk));
constexpr uint64_t kNaBlk = kNaInfo + na_up(sizeof(FrontierInfo));
constexpr uint64_t kNaSpread = kNaBlk + na_up(sizeof(RunBlock));
constexpr uint64_t kNoAllocScratchBytes = kNaSpread + na_up(8 * kSpreadWords);

// The scratch memory of og_bfs_device_noalloc.  In host code `scratch` is a
// stand-in for the symbol, not a device address: kernels get the address
// that hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kNoAllocMaxDevices = 64;
static std::mutex g_na_mu;
static void *g_na_ptr[kNoAllocMaxDevices];  // device address of `scratch`, per device

// Device address of `scratch` on the current device, looked up once per
// device with that device current.
static uint8_t *noalloc_scratch(int dev) {
    if (dev < 0 || dev >= kNoAllocMaxDevices) raise(OG_EUNSUPPORTED, "device %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_na_mu);
    if (!g_na_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            raise(OG_EHIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        }
        g_na_ptr[dev] = p;
    }
    return (uint8_t *)g_na_ptr[dev];
}

// Start of an allocation-free run, one launch: levels, flags, totals, counters
// and traversal state.  Row offsets that do not run from 0 to E end the run
// before it begins and leave the levels alone; counters[14..15] keep them.
__global__ __launch_bounds__(kBlock) void k_noalloc_init(const uint64_t *__restrict__ ptr, uint64_t V, uint64_t E,
                                                         uint32_t src, uint32_t *__restrict__ levels,
                                                         uint8_t *__restrict__ flag, uint64_t Vpad,
                                                         unsigned long long *__restrict__ tot, uint64_t ntot,
                                                         unsigned long long *__restrict__ spread, RunBlock *blk,
                                                         FrontierInfo *info, RoundCtl c) {
    const uint64_t tid = (uint64_t)blockIdx.x * kBlock + threadIdx.x, nth = (uint64_t)gridDim.x * kBlock;
    const uint64_t p0 = ptr[0], p1 = ptr[V];
    const bool good = p0 == 0 && p1 == E;
    if (tid == 0) {
        c.live = good ? 1u : 0u;
        blk->ctl = c;
        for (int i = 0; i < 16; ++i) blk->counters[i] = i == 14 ? p0 : i == 15 ? p1 : 0;
        *info = FrontierInfo{};
    }
    for (uint64_t i = tid; i < ntot; i += nth) tot[i] = i >= kTotSlot && i < kTotArrive && i % kTotLine == 3 ? ~0ull : 0ull;
    for (uint64_t i = tid; i < kSpreadWords; i += nth) spread[i] = 0;
    if (!good) return;
    for (uint64_t v = tid; v < V; v += nth) levels[v] = v == src ? 1u : OG_UNREACHED;
    for (uint64_t v = tid; v < Vpad; v += nth) flag[v] = v == src ? 1 : 0;
}

static void noalloc_bfs(const uint64_t *d_ptr, const uint32_t *d_cols, uint64_t V, uint64_t E, uint32_t src,
                        uint32_t *d_levels, hipStream_t s, og_run_stats *stats) {
    int dev = 0;
    OG_HIP(hipGetDevice(&dev));
    uint8_t *base = noalloc_scratch(dev);
    RunBlock *blk = (RunBlock *)(base + kNaBlk);
    RunBlock h{};
    auto check_ends = [&] {
        if (h.counters[14] != 0 || h.counters[15] != E)
            raise(OG_EINVAL, "row offsets must run from 0 to E=%llu over V+1 entries (got %llu .. %llu)",
                  (unsigned long long)E, h.counters[14], h.counters[15]);
    };
    auto fetch = [&] {
        OG_HIP(hipGetLastError());
        OG_HIP(hipMemcpyAsync(&h, blk, sizeof h, hipMemcpyDeviceToHost, s));
        OG_HIP(hipStreamSynchronize(s));
    };
    Stopwatch total;
    if (V <= kSmallV && E <= kSmallE) {
        launch_small<ALGO_BFS, false, false>(
            SmallArgs{d_ptr, d_cols, 0, (uint32_t)V, src, d_levels, nullptr, blk, nullptr, nullptr, true, E}, s);
        fetch();
        check_ends();
    } else {
        const uint64_t Vpad = (V + 15) / 16 * 16;
        const uint32_t nblk = (uint32_t)((Vpad + verts_per_block(1) - 1) / verts_per_block(1));
        uint8_t *flag = base + kNaFlag;
        uint32_t *list = (uint32_t *)(base + kNaList);
        uint64_t *hub = (uint64_t *)(base + kNaHub);
        uint64_t *doff = (uint64_t *)(base + kNaDoff);
        const CompactTotals ct{(unsigned long long *)(base + kNaTot), nblk, 1};  // (no dynamic list)
        FrontierInfo *info = (FrontierInfo *)(base + kNaInfo);
        unsigned long long *spread = (unsigned long long *)(base + kNaSpread);
        const Tuning tn;  // default bins: the hub bound above assumes its t2 and tile
        static_assert(Tuning{}.t2 == 4096 && Tuning{}.tile == 2048, "hub capacity bound follows the default tuning");
        hipLaunchKernelGGL(k_noalloc_init, dim3(fill_grid(V)), dim3(kBlock), 0, s, d_ptr, V, E, src, d_levels, flag, Vpad,
                           ct.t, totals_words(nblk), spread, blk, info, ctl_begin(V, 0, 0, 0, false));
        auto compact = [&] {
            hipLaunchKernelGGL(k_frontier_compact<1>, dim3(nblk), dim3(kCompactBlock), 0, s, flag, (uint8_t *)nullptr,
                               Vpad, V, d_ptr, (const uint64_t *)nullptr, (const uint32_t *)nullptr,
                               (const uint32_t *)nullptr, tn, (const uint32_t *)nullptr, &blk->ctl, ct, info, list, hub,
                               kNoAllocHubCap, doff, (uint32_t *)nullptr, (uint64_t)0, (RoundClock *)nullptr,
                               (int)kClkOther, (unsigned long long *)nullptr);
        };
        RoundRelax r{};
        r.list = list;
        r.info = info;
        r.ptr = d_ptr;
        r.sedges = d_cols;
        r.hub = hub;
        r.hub_cap = kNoAllocHubCap;
        r.tile = tn.tile;
        r.cd = 0;  // the whole graph is static: three bins in one launch
        r.vsplit = V;
        r.spread = spread;
        const RelaxArgs a{d_levels, flag, nullptr, nullptr, 0, nullptr, nullptr, nullptr};
        static_assert(Tuning{}.lpv0 == 8, "the relax below is instantiated for 8 lanes per bin-0 vertex");
        compact();
        // the first batch covers most traversals of skewed graphs: an empty
        // round costs about 8 us, a host round trip 25
        for (int rounds = 2 * kRoundBatch;; rounds = kRoundBatch) {
            for (int k = 0; k < rounds; ++k) {
                hipLaunchKernelGGL((k_relax_round<ALGO_BFS, false, false, 8>), dim3(kFuseStatic * kHubGridCap),
                                   dim3(kBlock), (size_t)tn.tile * 4, s, r, a);
                compact();
            }
            hipLaunchKernelGGL(k_reach_stats, dim3(stats_grid(V)), dim3(kStatsBlock), 0, s, d_levels, d_ptr,
                               (const uint32_t *)nullptr, (const uint32_t *)nullptr, V, blk->counters, spread,
                               (RoundClock *)nullptr, (const RoundCtl *)&blk->ctl);
            fetch();
            check_ends();
            if (!h.ctl.live) break;
        }
    }
    if (stats) {
        og_run_stats st{};
        st.approach = OG_ASCETIC;
        st.iterations = h.ctl.rounds;
        st.node_sum = h.ctl.node_sum;
        st.static_node_sum = h.ctl.static_node_sum;
        st.work_edges = h.ctl.work_edges;
        st.static_work_edges = h.ctl.static_work_edges;
        st.updates = h.counters[0];
        st.reached = h.counters[2];
        st.traversed_edges = h.counters[3];
        st.checksum = h.counters[4];
        st.total_ms = total.ms();
        *stats = st;
    }
}

}  // namespace og

extern "C" og_status og_bfs_device_noalloc(const uint64_t *row_ptr, const uint32_t *cols, uint64_t num_vertices,
                                           uint64_t num_edges, uint32_t source, uint32_t *levels, void *stream,
                                           og_run_stats *stats) {
    clear_error();
    if (!row_ptr || !levels || (num_edges && !cols)) return fail(OG_EINVAL, "null device pointer");
    if (num_vertices == 0 || source >= num_vertices)
        return fail(OG_EINVAL, "source %u out of range for V=%llu", source, (unsigned long long)num_vertices);
    if (num_vertices > kNoAllocMaxV || num_edges > kNoAllocMaxE)
        return fail(OG_EINVAL,
                    "og_bfs_device_noalloc handles V <= %llu and E <= %llu (its scratch is fixed at %llu bytes); "
                    "got V=%llu E=%llu",
                    (unsigned long long)kNoAllocMaxV, (unsigned long long)kNoAllocMaxE,
                    (unsigned long long)kNoAllocScratchBytes, (unsigned long long)num_vertices,
                    (unsigned long long)num_edges);
    return guard([&]() -> og_status {
        if (!hip_available()) raise(OG_EHIP, "no HIP device is visible");
        noalloc_bfs(row_ptr, cols, num_vertices, num_edges, source, levels, (hipStream_t)stream, stats);
        return OG_OK;
    });
}
