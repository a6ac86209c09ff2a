// Device-side state and helpers shared by engine.hip and pagerank.hip.
// gfx950 only: 64-lane wavefronts, 160 KiB LDS per CU.
#pragma once

#include <hip/hip_runtime.h>

#include <chrono>
#include <memory>
#include <mutex>
#include <vector>

#include "og_internal.h"

#define OG_HIP(x)                                                                          \
    do {                                                                                   \
        hipError_t e_ = (x);                                                               \
        if (e_ != hipSuccess)                                                              \
            ::og::raise(e_ == hipErrorOutOfMemory ? OG_ENOMEM_DEVICE : OG_EHIP, "%s: %s", \
                        #x, hipGetErrorString(e_));                                        \
    } while (0)

namespace og {

constexpr int kWave = 64;
constexpr int kBlock = 256;             // threads per block of the frontier kernels
// Frontier compaction: a workgroup of kCompactBlock threads takes NW windows
// of four vertices per thread.  Graphs up to kSmallFrontierV vertices use one
// (their rounds are latency bound); larger ones four (a quarter of the
// workgroups that reserve list places one after another).
constexpr int kCompactBlock = 1024;
constexpr uint64_t kSmallFrontierV = 1ull << 22;
constexpr int compact_nw(uint64_t V) { return V <= kSmallFrontierV ? 1 : 4; }
constexpr uint64_t verts_per_block(int nw) { return 4ull * kCompactBlock * nw; }
constexpr int kDynEdgesPerThread = 8;   // dynamic relax: edges per lane
constexpr int kDynEdgesPerBlock = kBlock * kDynEdgesPerThread;
constexpr int kMaxSlots = 16;           // staging slots of the dynamic-region pipeline
// Zero-copy loading keeps part of the dynamic region in HBM in whole chunks of
// kResChunk consecutive vertices; the link moves pinned host memory in lines
// of kLinkLine bytes, each fetched whole.
constexpr uint32_t kResChunkShift = 5;
constexpr uint32_t kResChunk = 1u << kResChunkShift;
constexpr int64_t kNotResident = INT64_MIN;
constexpr uint32_t kLinkLine = 128;
constexpr uint64_t kSlotTargetBytes = 256ull << 20;  // preferred slot (chunk) size

enum Algo { ALGO_BFS = 0, ALGO_SSSP = 1, ALGO_CC = 2, ALGO_MSBFS = 3, ALGO_MSBFS2 = 4 };

constexpr int kMsWidth = 64;            // sources per mask of the multi-source BFS (bits of a u64)
// Masks of a multi-source traversal (ALGO_MSBFS2: two batches of 64 sources
// that walk the graph together); 0: one value per vertex instead.
constexpr int ms_masks(int algo) { return algo == ALGO_MSBFS ? 1 : algo == ALGO_MSBFS2 ? 2 : 0; }

// Per-vertex state the relax kernels touch.
struct RoundCtl;
struct RelaxArgs {
    uint32_t *val;        // BFS level / SSSP distance / CC label
    uint8_t *flag;        // next-frontier flags
    ulonglong2 *vn;       // multi-source: x sources that reached v, y sources offered to v this round
    const uint64_t *front;// multi-source: sources whose frontier holds v
    uint32_t wbits;       // packed weighted edges: bits of the weight field
    const uint64_t *pull; // multi-source, optional: sources relaxed bottom-up this round
                          // (left out of the top-down relax)
    const uint64_t *pmid; // light/heavy split, optional: end of each row's light edges
    RoundCtl *ctl;        // with the split: notes that the round put a value below its threshold
    // of a lane, filled and noted by the kernels (relax_begin, relax_end)
    mutable uint32_t thresh = 0, near = 0;
};

// Edge range of u in a round: the whole row, or with the light/heavy split
// its light part [ptr[u], pmid[u]) or, in a heavy round, [pmid[u], ptr[u+1]).
__device__ __forceinline__ void row_range(const uint64_t *__restrict__ ptr, const uint64_t *__restrict__ pmid,
                                          bool heavy, uint64_t u, uint64_t &b, uint64_t &e) {
    if (!pmid) {
        b = ptr[u];
        e = ptr[u + 1];
    } else if (heavy) {
        b = pmid[u];
        e = ptr[u + 1];
    } else {
        b = ptr[u];
        e = pmid[u];
    }
}

// Degree of u's row in the round's range.  With a degree table (4 bytes per
// vertex: deg the whole-row degrees, or with the split deg the light and
// hdeg the heavy degrees) one or two loads replace the two 8-byte row
// bounds; a round over whole rows of a split graph adds the two parts.
__device__ __forceinline__ uint64_t round_deg(const uint32_t *__restrict__ deg, const uint32_t *__restrict__ hdeg,
                                              const uint64_t *__restrict__ ptr, const uint64_t *__restrict__ pmid,
                                              bool heavy, uint64_t u) {
    if (deg) {
        if (pmid) return heavy ? hdeg[u] : deg[u];
        return (uint64_t)deg[u] + (hdeg ? hdeg[u] : 0u);
    }
    uint64_t b, e;
    row_range(ptr, pmid, heavy, u, b, e);
    return e - b;
}

// Degree-bin thresholds and shapes for the static relax (autotunable).
struct Tuning {
    uint32_t t1 = 32;      // bin 0: 1 <= deg <= t1, lpv0 lanes per vertex
    uint32_t lpv0 = 8;     // 1, 2, 4, 8, 16, 32 or 64
    uint32_t t2 = 4096;    // bin 1: t1 < deg <= t2, one wave per vertex
    uint32_t tile = 2048;  // bin 2: deg > t2, tiles of `tile` edges, one workgroup each
    uint32_t delta = 0;    // SSSP near-far bucket width (0: every improved vertex every round)
    uint32_t defer = 0;    // SSSP / CC: 1 = hold dynamic vertices back while static ones are active;
                           // SSSP with delta > 0: 2 = dynamic vertices relax only after the
                           // static part of their near-far bucket has settled
    uint32_t dyn_grid = 0; // workgroups of the dynamic-region relax (0: kDynGridCap)
};

// Frontier summary produced on the device each iteration and read by the host.
struct FrontierInfo {
    uint32_t n[4];          // bin0 vertices, bin1 vertices, bin2 tiles, dynamic vertices
    uint32_t nzero;         // active vertices with no out-edge
    uint32_t nhub;          // bin2 vertices
    uint64_t static_deg;    // sum of degrees over static active vertices
    uint64_t dyn_deg;       // sum of degrees over dynamic active vertices
    uint32_t nfar;          // active vertices held back (value >= threshold)
    uint32_t min_far;       // smallest value among them
    uint32_t live;          // 1 while active or held-back vertices remain
    uint32_t dyn_held;      // 1: dynamic vertices were held back this round
    uint32_t pull;          // 1: BFS round runs bottom-up (the lists are not read)
    uint32_t heavy;         // 1: light/heavy split, this round relaxes heavy edges
};

// Device-resident driver state of one traversal.  The end of each
// compaction advances it, so rounds can be enqueued without a host round
// trip: the near-far threshold moves on the device and the statistics the
// host used to add up per round accumulate here.
struct RoundCtl {
    uint32_t thresh;             // near-far threshold of the next compaction (0xFFFFFFFF: off)
    uint32_t delta;              // near-far bucket width (0: off)
    uint32_t defer;              // 1: hold the dynamic list back while static vertices are active;
                                 // 2: dynamic vertices are near only below fbound
    uint32_t fbound;             // defer 2: dynamic vertices with value < fbound are near
    uint32_t split;              // light/heavy split in use (rows: light edges, then heavy)
    uint32_t mode;               // split: 1 = the next compaction collects the heavy-pending vertices
    uint64_t hpend;              // split: vertices light-relaxed since the last heavy round
    uint32_t rounds;             // compactions that found active vertices
    uint32_t compactions;        // all compactions
    uint32_t live;               // last compaction's FrontierInfo::live
    uint32_t overflow;           // multi-source: a level past 255 was needed
    uint32_t dir_opt;            // BFS: choose top-down / bottom-up per round
    uint32_t pull;               // direction of the current round (1: bottom-up)
    uint32_t pull_rounds;        // rounds run bottom-up
    uint64_t unexplored;         // BFS: edges of vertices not yet in any frontier
    uint64_t nverts;             // V (the bottom-up -> top-down switch compares the frontier with V / 24)
    uint64_t node_sum;           // active vertices, summed over rounds
    uint64_t static_node_sum;    // ... of them in the static bins
    uint64_t dyn_node_sum;       // ... of them in the dynamic list
    uint64_t work_edges;         // degree sums over active vertices
    uint64_t static_work_edges;  // ... over the static bins
    uint64_t dyn_rounds;         // rounds with a dynamic list
    uint32_t halt;               // 1 (device-driven runs): once a compaction finds nothing live, the
                                 // compactions of rounds enqueued past the end skip their sweep
    uint32_t hold;               // defer 1: the next compaction holds the dynamic vertices back
    uint32_t near;               // split: the round's relax put a value below thresh (set by the relax kernels)
};

// Time of a device-driven run by kind of work, from the device's constant
// 100 MHz clock.  A kernel that begins work of one kind after another kind
// adds its start time to the old kind and subtracts it from its own, two
// atomics that nothing waits for, so that each kind sums up to end - begin.
// (Event nodes in the stream or the captured graph stalled each kernel for
// about 10 us: two of them per round.)
enum ClockKind { kClkRelax = 0, kClkFront = 1, kClkOther = 2 };
struct RoundClock {
    unsigned long long acc[3];
};

// What a run leaves on the device beside its values; one copy brings it over.
struct RunBlock {
    RoundCtl ctl;
    RoundClock clk;
    unsigned long long counters[16];  // [0] updates static, [1] updates dynamic, [2..] scratch
};

constexpr uint32_t kDeferOnce = 3;      // RoundCtl::defer: hold the dynamic vertices back until the static region
                                        // has settled once

// Totals of one compaction, in 128-byte lines so that the device-scope
// atomics of different totals do not queue behind each other: list
// reservations (bins 0|1, hub tiles|hub vertices, the dynamic list's
// vertices|edges, their wide form), arrivals, and kTotSlots slots of the
// sums that nothing is reserved with (vertices without edges | held back,
// static degrees, lagging | held dynamic vertices, smallest held-back value),
// block b adding to slot b % kTotSlots.
constexpr uint32_t kTotLine = 16;                  // u64 per line
constexpr uint32_t kTotBins = 0 * kTotLine;
constexpr uint32_t kTotTiles = 1 * kTotLine;
constexpr uint32_t kTotDyn = 2 * kTotLine;
constexpr uint32_t kTotWide = 3 * kTotLine;        // lock, vertices, edges
constexpr uint32_t kTotRoot = 4 * kTotLine;        // arrived groups
constexpr uint32_t kTotSlot = 8 * kTotLine;
constexpr uint32_t kTotSlots = 32;
constexpr uint32_t kTotArrive = kTotSlot + kTotSlots * kTotLine;  // arrivals per group of kTotGroup blocks
constexpr uint32_t kTotGroup = 32;
constexpr uint64_t totals_words(uint64_t nblk) {
    return kTotArrive + (nblk + kTotGroup - 1) / kTotGroup * kTotLine;
}
struct CompactTotals {
    unsigned long long *t;
    uint32_t nblk;
    uint32_t dsh;  // dynamic list: vertices in the low dsh bits of one word, edges above; 0: the wide form
};
constexpr uint32_t bits_of(uint64_t x) { return x ? 64u - (uint32_t)__builtin_clzll(x) : 0u; }

// Buffers of one frontier traversal: next-frontier flags, the compacted bin
// lists, the dynamic degree prefix and the compaction's totals.  A graph's
// single-source runs use DeviceState::fr; each serving engine owns its own so
// that engines can iterate concurrently on different streams.
struct Frontier {
    uint8_t *flag = nullptr;         // Vpad next-frontier flags
    uint8_t *hflag = nullptr;        // Vpad light/heavy split: heavy-pending flags
    uint32_t *list = nullptr;        // V: bin 0 up from 0, bin 1 down from vsplit - 1, dynamic list up from vsplit
    uint64_t *hub = nullptr;         // hub tiles (tile << 32 | vertex)
    uint64_t hub_cap = 0;
    uint64_t *doff = nullptr;        // V + 1 degree prefix of the dynamic list
    uint32_t *dchunk = nullptr;      // list entry holding edge c * kDynEdgesPerBlock of the dynamic edge space
    uint64_t dchunk_cap = 0;
    unsigned long long *tot = nullptr;  // compaction totals (cleared between compactions)
    uint32_t nblk = 0;
    uint32_t dsh = 0;
    CompactTotals totals() const { return CompactTotals{tot, nblk, dsh}; }
    uint32_t nw = 4;                 // windows per workgroup of the compaction (compact_nw)
    uint64_t V = 0;
    FrontierInfo *info = nullptr;
    FrontierInfo *h_info = nullptr;  // pinned
    RunBlock *blk = nullptr;
    RunBlock *h_blk = nullptr;       // pinned
    RoundCtl *ctl = nullptr;         // parts of blk
    unsigned long long *counters = nullptr;
    RoundClock *clk = nullptr;
    unsigned long long *h_progress = nullptr;  // pinned, written by the device: compactions << 1 | ended
    unsigned long long *spread = nullptr;  // kSpreadWords: the relax kernels' counters on their way to blk
};

// Timing of one class of launches: pairs of events on the launching stream.
struct TimedClass {
    std::vector<std::pair<hipEvent_t, hipEvent_t>> marks;
    uint64_t launches = 0;
    double ms = 0;  // already resolved (marks of captured graphs, read after each replay)
};

class EventPool {
  public:
    ~EventPool() {
        for (auto e : all_) (void)hipEventDestroy(e);
    }
    hipEvent_t get() {
        if (next_ == all_.size()) {
            hipEvent_t e;
            OG_HIP(hipEventCreate(&e));
            all_.push_back(e);
        }
        return all_[next_++];
    }
    void reset() { next_ = 0; }

  private:
    std::vector<hipEvent_t> all_;
    size_t next_ = 0;
};

// Owner of device and pinned host allocations; frees them all at once.
struct MemPool {
    struct Block {
        void *p;
        size_t bytes;
    };
    std::vector<Block> dev;
    std::vector<void *> pin;
    uint64_t device_bytes = 0;
    MemPool() = default;
    MemPool(const MemPool &) = delete;
    MemPool &operator=(const MemPool &) = delete;
    ~MemPool() { release(); }
    // null when there is no memory (the error in *err)
    void *try_dalloc(size_t bytes, hipError_t *err = nullptr) {
        void *p = nullptr;
        if (bytes == 0) bytes = 256;
        const hipError_t e = hipMalloc(&p, bytes);
        if (err) *err = e;
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        dev.push_back({p, bytes});
        device_bytes += bytes;
        return p;
    }
    void *dalloc(size_t bytes) {
        hipError_t e = hipSuccess;
        void *p = try_dalloc(bytes, &e);
        if (!p) raise(OG_ENOMEM_DEVICE, "hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(e));
        return p;
    }
    // Gives one device allocation back before the others (null: nothing).
    template <class T>
    void dfree(T *&p) {
        for (size_t i = 0; p && i < dev.size(); ++i)
            if (dev[i].p == p) {
                device_bytes -= dev[i].bytes;
                dev.erase(dev.begin() + i);
                (void)hipFree(p);
                break;
            }
        p = nullptr;
    }
    // null when there is no memory
    void *try_palloc(size_t bytes) {
        void *p = nullptr;
        if (hipHostMalloc(&p, bytes ? bytes : 8, hipHostMallocDefault) != hipSuccess || !p) {
            (void)hipGetLastError();
            return nullptr;
        }
        pin.push_back(p);
        return p;
    }
    void *palloc(size_t bytes) {
        void *p = try_palloc(bytes);
        if (!p) raise(OG_ENOMEM_HOST, "pinned host allocation of %zu bytes failed", bytes);
        return p;
    }
    void release() {
        for (const Block &b : dev) (void)hipFree(b.p);
        for (void *p : pin) (void)hipHostFree(p);
        dev.clear();
        pin.clear();
        device_bytes = 0;
    }
};

// The dynamic region as chunks of whole rows that cross the link in vertex
// order, straight from the host copy (no gather), through a ring of `ring`
// slots of `slot` words in the staging share (PageRank's iterations).
struct LinkRing {
    struct Chunk {
        uint32_t va, vb;       // vertices
        uint64_t word, words;  // of the host source
        uint32_t first;        // bits before the first edge
    };
    std::vector<Chunk> chunks;
    uint32_t ring = 0;
    uint32_t lbits = 0;        // bits per edge on the link, 0: whole edges
    uint64_t slot = 0;
    uint64_t maxrow = 0;       // edges of the longest row
    const uint32_t *src = nullptr;
    std::vector<hipEvent_t> ev_h2d, ev_use;  // copy into / use of the slot finished
    ~LinkRing() {
        for (hipEvent_t e : ev_h2d) (void)hipEventDestroy(e);
        for (hipEvent_t e : ev_use) (void)hipEventDestroy(e);
    }
};

// What result copy-backs go through (copy_to_host): pinned staging, a word per
// slab that the device writes once the slab is there, and threads that copy
// slabs out.  Shared by every preparation of the process and given back with the
// last of them: a new graph's first result would otherwise wait for the threads
// to start and for the link's page tables to learn 4 MB of new staging (about
// 0.75 ms).  One copy uses it at a time; another that finds it taken goes
// through the runtime.
struct OutStage {
    std::mutex use;        // held by the copy that uses the rest
    char *buf = nullptr;
    size_t bytes = 0;
    unsigned long long *flag = nullptr;
    unsigned long long seq = 0;
    std::unique_ptr<WorkerPool> pool;
    // Makes ready for a result of n bytes that up to `threads` threads copy out
    // (`use` held); false when that is too large or there is no memory for it.
    bool reserve(size_t n, unsigned threads);
    ~OutStage();
};

// PageRank's scalars on the device: what an iteration leaves for the next.
struct PrState {
    double dangling;      // rank mass of the vertices without out-edges
    double l1;            // residual of the last iteration
    double tolerance;
    uint32_t iterations;
    uint32_t done;        // the residual fell below the tolerance: later iterations do nothing
};

struct DeviceState {
    og_approach approach = OG_ASCETIC;
    int device = 0;
    int clock_khz = 100000;          // rate of the device's constant clock
    uint64_t V = 0, E = 0, Vpad = 0;
    uint32_t eb = 4;                 // bytes per edge on the device (static region, staging) and the link
    og_plan_info plan{};
    Tuning tune;
    unsigned host_threads = 0;
    uint32_t flags = 0;

    // graph on the device
    uint64_t *d_ptr = nullptr;       // V + 1 (device copy; USM: managed)
    uint64_t *d_pmid = nullptr;      // light/heavy split: V, end of the light edges of each row
    uint32_t *d_deg = nullptr;       // degree table of the compaction: Vpad whole-row degrees, or with
                                     // the split Vpad light then Vpad heavy degrees (null: row bounds)
    bool deg_split = false;          // d_deg holds light and heavy degrees
    const uint32_t *deg_heavy() const { return d_deg && deg_split ? d_deg + Vpad : nullptr; }
    std::vector<uint64_t> h_pmid;    // host copy (the staged gather)
    uint32_t split_weight = 0;       // light: weight < split_weight (0: no split)
    const uint64_t *run_pmid = nullptr;  // d_pmid while a run uses the split (SSSP near-far), else null
    void *d_static = nullptr;        // static-region edges (USM: managed, whole graph)
    uint64_t static_used = 0;        // edges of the static vertices, = ptr[vsplit]
    void *d_staging = nullptr;       // nslots * slot_edges edges (zero-copy: the resident chunks)
    uint64_t slot_edges = 0;
    bool managed = false;
    // Weighted edges on the device and the link: one 4-byte word
    // (to << wbits | w) when packed, else the CSR's 8-byte {to, w}.
    bool packed = false;
    uint32_t wbits = 0;
    uint32_t deb = 4;                // bytes per dynamic-region edge on the link (= eb)
    bool in_place = false;           // traversals read the dynamic region in pinned host memory
    uint64_t dyn_base = 0;           // first edge of the dynamic region (= ptr[vsplit])
    const void *h_dyn = nullptr;     // host source of dynamic edges (packed copy, null once the link format has
                                     // taken its place, or the CSR)
    const void *hd_dyn = nullptr;    // the same, as a device address (zero-copy mode)
    uint64_t slot_dyn = 0;           // dynamic edges per staging slot in the transfer format
    // zero-copy with the light/heavy split: the host copy of the dynamic
    // region holds every row's light part in vertex order, then every heavy
    // part (light part of v at lpos[v - vsplit], heavy part at
    // split_nl + (ptr[v] - dyn_base) - lpos[v - vsplit]); lpos has
    // V - vsplit + 1 entries
    uint64_t *d_lpos = nullptr;
    uint64_t split_nl = 0;           // light edges of the dynamic region
    // Link format: when an edge word (id, or id << wbits | weight) fits lbits
    // <= kLinkBitsMax bits, the dynamic region crosses the link as a stream of
    // lbits-bit words (edge i of the host layout at bit i * lbits): zero-copy
    // reads and PageRank's chunks.  0: the 4- or 8-byte edges.
    uint32_t lbits = 0;
    const uint32_t *h_link = nullptr;   // pinned
    const void *hd_link = nullptr;      // the same, as a device address
    std::shared_ptr<LinkRing> link_ring;  // built on first use
    uint64_t dyn_resident = 0;       // zero-copy: dynamic edges held in d_staging (whole chunks)
    int64_t *d_rdelta = nullptr;     // zero-copy: per chunk of kResChunk vertices (index v >> kResChunkShift),
                                     // d_staging index - host-array position, or kNotResident; two per
                                     // chunk (light block, heavy block) with d_lpos
    uint64_t *m_ptr = nullptr;       // USM managed copies
    void *m_edges = nullptr;

    // per-vertex state
    uint32_t *d_val = nullptr;       // Vpad
    Frontier fr;                     // frontier buffers of single-source / batch runs

    // pinned host mirrors of the dynamic list
    uint32_t *h_dlist = nullptr;     // V
    uint64_t *h_doff = nullptr;      // V + 1
    std::vector<void *> h_stage;     // pinned gather buffer per staging slot

    hipStream_t s_compute = nullptr, s_copy = nullptr;
    hipStream_t s_static = nullptr;  // static-region relax, overlapping the dynamic region
    hipEvent_t ev_fork = nullptr;    // compaction of the round finished (static relax may start)
    hipEvent_t ev_static = nullptr;  // static relax of the round finished
    uint32_t nslots = 0;             // staging slots (a pipeline of small chunks)
    std::vector<hipEvent_t> ev_h2d;    // copy into slot finished
    std::vector<hipEvent_t> ev_relax;  // relax reading slot finished
    std::vector<char> slot_h2d_pending, slot_relax_pending;
    EventPool events;
    std::unique_ptr<WorkerPool> pool;

    // Multi-source BFS state, allocated on first use (ms_state) for walks of
    // `masks` masks per vertex; what is there for two serves walks of one.
    struct MsState {
        ulonglong2 *vn = nullptr;            // masks x V: sources that reached v, sources offered to v this round
        uint64_t *front = nullptr;           // masks x V: sources whose frontier holds v
        unsigned long long *part = nullptr;  // per commit workgroup: digest, reached, traversed of the sources
        uint32_t *src = nullptr;             // the batch's sources
        unsigned long long *sum = nullptr;   // per mask 3 x 64: digest, reached, traversed per source
        uint8_t *lvl = nullptr;              // lvl_masks x V x 64 levels, vertex-major (0 = unreached); only when levels are asked for
        uint32_t masks = 0, lvl_masks = 0;
    } d_ms;
    uint32_t *d_extract = nullptr;   // u32 levels of extract_cap sources on their way to the host
    uint32_t extract_cap = 0;
    // direction-optimising BFS: in-edge CSR (OG_PLAN_DIRECTION_OPT)
    uint64_t *d_in_ptr = nullptr;    // V + 1
    uint32_t *d_in_cols = nullptr;   // E in-neighbours

    // PageRank state (allocated on first use)
    void *d_rank = nullptr;
    void *d_contrib[2] = {nullptr, nullptr};  // read / written in turn
    uint32_t *d_outdeg = nullptr;
    double *d_partial = nullptr;     // per-block residual and dangling partials
    unsigned long long *d_prtot = nullptr;  // arrivals of the pull's workgroups
    uint64_t pr_partial_cap = 0;     // workgroups that d_partial and d_prtot are sized for
    PrState *d_prstate = nullptr;
    PrState *h_prstate = nullptr;    // pinned
    unsigned long long *h_progress = nullptr;  // pinned, written by the device: iterations << 1 | done
    std::shared_ptr<void> pr_plan;   // PageRank rows and chunk ranges (pagerank.hip)
    std::shared_ptr<void> round_graph;  // captured batches of device-driven rounds (engine.hip)
    std::shared_ptr<OutStage> out;        // result copy-backs up to kOutMax bytes
    // and the two chunks of larger ones
    void *h_chunk[2] = {nullptr, nullptr};
    hipEvent_t ev_chunk[2] = {nullptr, nullptr};
    uint32_t last_pairs[8] = {};        // relax + compaction pairs of the last device-driven run, per algorithm

    MemPool mem;                     // device + pinned allocations of this preparation

    void *dalloc(size_t bytes) { return mem.dalloc(bytes); }
    void *palloc(size_t bytes) { return mem.palloc(bytes); }
    uint64_t device_bytes() const { return mem.device_bytes; }
};

// ------------------------------------------------------------ wave helpers

// Waits until the wave's memory operations, atomics among them, are done.
// With device-scope atomics on both sides (performed at one place for the
// whole device) this orders a workgroup's reservations before its arrival
// without a release fence, which on gfx950 writes the whole L2 of the XCD
// back.
__device__ __forceinline__ void wait_vmem() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// True in the workgroup that arrives last (called by one thread of each).
// Arrivals are counted in two levels, kTotGroup workgroups per first-level
// counter: same-address atomics take about 12 ns each.
__device__ __forceinline__ bool arrive_last(const CompactTotals &ct) {
    const uint32_t g = blockIdx.x / kTotGroup, ng = (ct.nblk + kTotGroup - 1) / kTotGroup;
    unsigned long long *at = ct.t + kTotArrive + (uint64_t)g * kTotLine;
    if (atomicAdd(at, 1ull) + 1 != min(kTotGroup, ct.nblk - g * kTotGroup)) return false;
    atomicExch(at, 0ull);
    if (ng > 1) {
        if (atomicAdd(ct.t + kTotRoot, 1ull) + 1 != ng) return false;
        atomicExch(ct.t + kTotRoot, 0ull);
    }
    return true;
}

__device__ __forceinline__ uint64_t shfl_up_u64(uint64_t x, int d) {
    uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    lo = __shfl_up(lo, d, kWave);
    hi = __shfl_up(hi, d, kWave);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t x, int m) {
    uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    lo = __shfl_xor(lo, m, kWave);
    hi = __shfl_xor(hi, m, kWave);
    return ((uint64_t)hi << 32) | lo;
}

// Inclusive scan over the wave with DPP moves (rows of 16 lanes, then the
// rows' last lanes broadcast): no LDS round trips.
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t x) {
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, false);  // row_shr:1
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, false);  // row_shr:2
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, false);  // row_shr:4
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, false);  // row_shr:8
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false);  // row_bcast:15 to rows 1, 3
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false);  // row_bcast:31 to rows 2, 3
    return x;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ uint64_t dpp_add_u64(uint64_t x) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, CTRL, ROWS, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), CTRL, ROWS, 0xF, false);
    return x + (((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ uint64_t wave_scan_u64(uint64_t x) {
    x = dpp_add_u64<0x111, 0xF>(x);
    x = dpp_add_u64<0x112, 0xF>(x);
    x = dpp_add_u64<0x114, 0xF>(x);
    x = dpp_add_u64<0x118, 0xF>(x);
    x = dpp_add_u64<0x142, 0xA>(x);
    x = dpp_add_u64<0x143, 0xC>(x);
    return x;
}

// Lane l's value (l the same for the whole wave).
__device__ __forceinline__ uint64_t wave_read_u64(uint64_t x, int l) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), l);
    return ((uint64_t)hi << 32) | lo;
}

// N independent exclusive scans over the block in one pass (one LDS round):
// ex[i] = sum of x[i] over lower threads, tot[i] = block sum.  `lds` must
// hold N * blockDim.x / 64 entries.  Contains __syncthreads.
template <int N>
__device__ __forceinline__ void block_scan_n(const uint64_t (&x)[N], uint64_t (&ex)[N], uint64_t (&tot)[N],
                                             uint64_t *lds) {
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    const int nw = blockDim.x / kWave;
    uint64_t inc[N];
#pragma unroll
    for (int i = 0; i < N; ++i) inc[i] = x[i];
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint64_t y = shfl_up_u64(inc[i], o);
            if (lane >= o) inc[i] += y;
        }
    }
    if (lane == kWave - 1)
#pragma unroll
        for (int i = 0; i < N; ++i) lds[i * nw + wid] = inc[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        uint64_t before = 0, t = 0;
        for (int w = 0; w < nw; ++w) {
            const uint64_t s = lds[i * nw + w];
            before += (w < wid) ? s : 0;
            t += s;
        }
        ex[i] = before + inc[i] - x[i];
        tot[i] = t;
    }
    __syncthreads();
}

// Work counters of a run's relax kernels, spread over kSpread lines of 16
// words: every wave of a launch adds to one, and on a single line those
// atomics queued at about 12 ns each (20480 waves of a round: 230 us, which is
// what a dense round took whatever it relaxed).  The run's last kernel folds
// them (fold_spread).
constexpr uint32_t kSpread = 128;
constexpr uint32_t kSpreadWords = kSpread * 16;
enum SpreadWord { kUpdStatic = 0, kUpdDynamic = 1, kHbmEdges = 5 };  // word of a line = index in RunBlock::counters

// Adds the wave's per-lane counts with one atomic per wave.
__device__ __forceinline__ void wave_count(unsigned long long *spread, int word, uint32_t v) {
    const uint32_t s = wave_scan_u32(v);
    const uint32_t line = (blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave) % kSpread;
    if ((threadIdx.x & (kWave - 1)) == kWave - 1 && s) atomicAdd(spread + line * 16 + word, (unsigned long long)s);
}

// counters[w] += the lines' words w, which restart at zero (one workgroup of
// at least kSpread threads).
__device__ __forceinline__ void fold_spread(unsigned long long *spread, unsigned long long *counters) {
    if (threadIdx.x >= kSpread) return;
    const int words[3] = {kUpdStatic, kUpdDynamic, kHbmEdges};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const uint64_t s = wave_scan_u64(atomicExch(spread + threadIdx.x * 16 + words[i], 0ull));
        if ((threadIdx.x & (kWave - 1)) == kWave - 1 && s) atomicAdd(counters + words[i], (unsigned long long)s);
    }
}

constexpr int kRelaxBatch = 4;  // edges per lane whose reads are issued together

// Edge i of an edge array: 4-byte column (unweighted), the packed 4-byte
// weighted word (to << wbits | w), or the CSR's 8-byte AoS {to, w}.
template <bool W, bool PK>
__device__ __forceinline__ void load_edge(const void *__restrict__ edges, uint64_t i, uint32_t wbits, uint32_t &to,
                                          uint32_t &wt) {
    if (W && PK) {
        const uint32_t x = ((const uint32_t *)edges)[i];
        to = x >> wbits;
        wt = x & ((1u << wbits) - 1u);
    } else if (W) {
        const uint2 e = ((const uint2 *)edges)[i];
        to = e.x;
        wt = e.y;
    } else {
        to = ((const uint32_t *)edges)[i];
        wt = 1;
    }
}

// Narrowest saving worth a second copy of the dynamic region in host memory:
// an eighth of the link's bytes.
constexpr uint32_t kLinkBitsMax = 28;

// Word i of a stream of `bits`-bit words that starts `first` bits into p: one
// 8-byte load (the stream is padded by a word), so that a wave's lanes touch
// each link line once.
__device__ __forceinline__ uint32_t link_word(const uint32_t *__restrict__ p, uint64_t i, uint32_t bits, uint32_t first = 0) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2), aligned(4)));
    const uint64_t at = i * bits + first;
    const u32x2 x = *(const u32x2 *)(p + (at >> 5));
    const uint64_t w = ((uint64_t)x.y << 32 | x.x) >> (at & 31);
    return (uint32_t)w & (uint32_t)((1ull << bits) - 1);
}

// ------------------------------------------------------------- host timing

struct Stopwatch {
    std::chrono::steady_clock::time_point t0 = std::chrono::steady_clock::now();
    double ms() const {
        return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    }
};

// Records a start/stop event pair around a launch sequence on `s`.
struct EventSpan {
    DeviceState *d;
    TimedClass *cls;
    hipStream_t s;
    hipEvent_t a;
    EventSpan(DeviceState *d_, TimedClass *c, hipStream_t s_) : d(d_), cls(c), s(s_) {
        a = d->events.get();
        OG_HIP(hipEventRecord(a, s));
    }
    ~EventSpan() noexcept(false) {
        hipEvent_t b = d->events.get();
        OG_HIP(hipEventRecord(b, s));
        cls->marks.push_back({a, b});
        cls->launches++;
    }
};

inline double sum_ms(const TimedClass &c) {
    double t = c.ms;
    for (auto &m : c.marks) {
        float ms = 0;
        OG_HIP(hipEventElapsedTime(&ms, m.first, m.second));
        t += ms;
    }
    return t;
}

// Waits until the device has raised the pinned word *p (which it writes with
// system scope while it runs: count << 1 | ended) to at least `want` or to an
// ended one, or the stream has drained.
void wait_progress(const unsigned long long *p, unsigned long long want, hipStream_t s);

// The preparation's chunk ring, or null when a row does not fit a slot.
LinkRing *link_ring(DeviceState *d, const og_graph *g);

// Copies n bytes (a multiple of 4) of device memory at src (16-byte aligned) to
// host memory at dst, pageable or not, on stream s and returns when they are
// there.
void copy_to_host(DeviceState *d, void *dst, const void *src, size_t n, hipStream_t s);

// Allocates a frontier (device buffers + pinned summaries) sized for the
// graph and the current tuning; freed with the DeviceState.
void frontier_alloc(DeviceState *d, const og_graph *g, Frontier &f, MemPool &m);

// A single-source lane over a prepared, wholly device-resident graph: it
// shares the graph's device arrays (row pointers, edges, degree table, light
// / heavy split, in-edges) and owns values, frontier buffers, streams and
// captured rounds, so several lanes run single-source traversals side by
// side on their own streams.  `delta` (0: the graph's tuning) is the lane's
// near-far width.  Freed with device_state_free, which releases only what
// the lane allocated.
DeviceState *lane_state_create(og_graph *g, uint32_t delta);
// Device bytes lane_state_create allocates for graph g (values, flags, bin
// lists, degree prefix, block counts, hub tiles).
uint64_t lane_state_bytes(const og_graph *g);
// og_sssp from src on a lane; out (V values) may be null.
void lane_run_sssp(og_graph *g, DeviceState *lane, uint32_t src, uint32_t *out, og_run_stats *st);

// One compaction: flags -> bin lists / hub tiles / dynamic list with
// its degree prefix, flags cleared; f.info and f.ctl updated on the device.
// With `val` non-null, vertices whose value is >= f.ctl->thresh stay flagged
// and are only counted (near-far order).  With to_host, the summary is also
// copied to f.h_info (stream-ordered, not synchronised).
// pmid (light/heavy split, a run with RoundCtl::split): rows are ranged by
// the round's mode.  clk (optional): the run's clock, which leaves `prev`.
void frontier_compact(DeviceState *d, Frontier &f, hipStream_t s, const uint32_t *val = nullptr,
                      bool to_host = true, const uint64_t *pmid = nullptr, RoundClock *clk = nullptr,
                      int prev = kClkOther, unsigned long long *progress = nullptr);


// Launches the static-region relax of the bins for op ALGO.  The kernels
// read their counts from f.info; `hfi` (the host copy of it, or null when the
// host does not know it) only sizes the grids and skips empty bins.
template <int ALGO, bool W>
void launch_static_relax(DeviceState *d, Frontier &f, const FrontierInfo *hfi, const RelaxArgs &a, hipStream_t s);
// Served BFS: the bottom-up scan's arrays (graphs with their in-edges).
struct SrvPull {
    const uint64_t *in_ptr;
    const uint32_t *in_cols;
    uint64_t V;
    ulonglong2 *vn;
    const uint64_t *front;
    uint8_t *flag;
    const unsigned long long *pull;  // bit j: slot j scans bottom-up this round
};
// One launch relaxing a served round: top-down slots through the static
// bins and, with `pull`, the bottom-up scan beside them.
void launch_srv_round(DeviceState *d, Frontier &f, const RelaxArgs &a, hipStream_t s, const SrvPull *pull,
                      bool weighted);

}  // namespace og
