// Synchronous label propagation on gfx950: one kernel family serves both the size-constrained
// clustering of the coarsening phase (labels = clusters, bound B; reference:
// lib/partition/coarsening/clustering/size_constraint_label_propagation.cpp:134-194) and the
// LP refinement of the uncoarsening phase (labels = blocks, bound U; reference:
// lib/partition/uncoarsening/refinement/label_propagation_refinement/
// label_propagation_refinement.cpp:21-155).
//
// A round is S sub-rounds; a node belongs to sub-round hash3(seed ^ kSubSalt, 0, v) % S. One
// sub-round is three or four launches (or a part of refine_tail, which runs the rounds of a small
// refinement frontier in one workgroup), all order-independent, so the result is bit-identical to
// the CPU mirror of the same schedule whatever the thread interleaving:
//   propose  every node of the sub-round picks its best eligible neighbouring label from the
//            label / weight snapshot; proposers append a mover record and add their weight and
//            priority key to the target's inc / top (integer atomics: order-free);
//   filter   (refinement, while a block is overloaded) departures from overloaded blocks;
//   admit    a proposal is admitted if all proposals into its target fit, or if it is the
//            target's top-priority proposal and fits alone;
//   apply    admitted moves update labels and label weights; scratch is reset.
// Nodes are binned by degree (per sub-round lists built once per call):
//   deg <= 8/16/32/64   8 or 16 lanes per node, 1 to 4 edges per lane, summed by DPP moves;
//   deg <= 512          one wave per node, LDS hash table (open addressing, LDS atomics);
//                       one launch of a sub-round serves all of these lists;
//   larger              one workgroup per node, hash table in a pre-cleared global region.

#include <algorithm>
#include <cstring>

#include <rocprim/device/device_scan.hpp>

#include "common.hpp"
#include "lp.hpp"

namespace kahip {

namespace {

constexpr int kWaveCap = 1024;    // LDS hash slots per wave (degree <= 512 => load <= 1/2)
static_assert(kWaveCap == 1024, "wave_vb loads up to kWaveCap / 2 edges per wave");
constexpr int kWaveDense = 2048;  // dense LDS counters per wave (refinement, k <= 2048)
constexpr int kWaveDenseSmall = 512;  // the frontier kernel's counters for k <= 512 (less LDS)
constexpr int kBlock = 256;
constexpr int kFrontierGrid = 2048;  // workgroups of a refinement list kernel (grid-stride)
// nodes per lane group in flight in group_vb: BinConfig::group_items (1, 2 or 4)
constexpr int kHubChunk = 4096;   // hub edges per workgroup
constexpr int kHubCap = 8192;     // LDS hash slots per hub chunk (load <= 1/2)
constexpr int kHubThreads = 1024;      // clustering hub chunks (4 edges per thread)
constexpr int kMidThreads = 256;       // hubs of kMidChunk edges or fewer (4 edges per thread)
constexpr int kMidChunk = 1024;
constexpr int kHubDenseThreads = 512;  // refinement hub chunks (8 edges per thread)
constexpr int kLongRow = 1024;    // refinement: moved rows beyond are marked by all workgroups
constexpr int kHubDense = 4096;   // dense LDS counters per hub (refinement, k <= 4096)
constexpr long long kAllHubCounters = 1LL << 28;  // counters (ints) for incremental hubs
constexpr int kHubDenseSlots = 12288;  // dynamic LDS counters (48 KB): min(8, slots / k) copies
constexpr int kFinThreads = 1024;  // hub_bucket_merge workgroup
constexpr int kFinCap = 16384;     // LDS hash slots of hub_bucket_merge (128 KB)
constexpr int kFinLds = 8192;      // buckets up to this many entries merge in LDS
constexpr int kMaxBuckets = 2048;  // buckets per hub: min(kBucketsPerChunk x chunks, kMaxBuckets)
constexpr int kBucketsPerChunk = 4;  // ~1000 entries per (hub, bucket)
constexpr int kTinyThreads = 256;    // tiny bucket merge: <= kTinyMax entries in 16 KB of LDS
constexpr int kTinyCap = 2048;
constexpr int kTinyMax = 1024;
constexpr int kTinyTasks = 2048;     // sub-rounds of more merge tasks start with it
constexpr int kSmallThreads = 512;   // small bucket merge: <= kSmallMax entries in 32 KB of LDS
constexpr int kSmallCap = 4096;
constexpr int kSmallMax = 2048;
constexpr int kSmallGrid = 1024;     // its workgroups over a queue (four per CU)
// Sub-rounds of at most kHubJoin chunks and mid-size hubs (two workgroups of kHubThreads per CU)
// take the mid-size hubs along in the chunk kernel's launch.
constexpr int kHubJoin = 512;
constexpr int kHubStage = 256;       // merge tasks of hubs of at most this many chunks sum the
                                     // chunks' entry counts themselves and keep the offsets in LDS
static_assert(kHubStage <= kTinyThreads, "a thread per chunk");

struct Cand {
    int conn;
    uint32_t tie;
    int lab;
    int size;
};
static_assert(sizeof(Cand) == sizeof(int4), "bucket results are stored as int4");

// The arguments of clustering blockIdx.y of a launch over several (uniform).
__device__ inline void select_copy(LpArgs& a) {
    const int y = blockIdx.y;
    if (y == 0) return;
    const long long o = y * a.copy_stride;
    a.label += o;
    a.size += o;
    a.inc += o;
    a.top += o;
    a.prop_t += o;
    a.prop_gain += o;
    a.prop_ok += o;
    a.tie_seed = y == 1 ? a.copy_tie1 : a.copy_tie2;
}

// Bucket of a label among P buckets of a hub (independent of the LDS slot hash).
__device__ inline int bucket_of(int lab, int P) {
    return (int)(mix32((uint32_t)lab ^ 0x5bd1e995u) % (uint32_t)P);
}

__device__ inline int bound_of(const LpArgs& a, int lab) {
    return a.lbound ? a.lbound[lab] : a.bound;
}

__device__ inline bool better(int ac, uint32_t at, int al, int bc, uint32_t bt, int bl) {
    return ac > bc || (ac == bc && (at > bt || (at == bt && al < bl)));
}

// Candidate (conn, lab) of node v (weight nw) against the best so far: the label's size (and
// bound) is read only when the candidate would beat c, so a thread reads the sizes of its running
// maxima only. The result, the maximum of better() over the eligible labels, is the same as with
// every size read: c only ever holds eligible labels, and the best eligible one beats whatever c
// holds when it comes up.
__device__ inline void consider(const LpArgs& a, int v, int nw, int conn, int lab, Cand& c) {
    const uint32_t t = hash3(a.tie_seed, (uint32_t)v, (uint32_t)lab);
    if (!better(conn, t, lab, c.conn, c.tie, c.lab)) return;
    const int sz = a.size[lab];
    if ((long long)sz + nw >= (long long)bound_of(a, lab)) return;
    c = Cand{conn, t, lab, sz};
}

template <int W>
__device__ inline void reduce_cand(Cand& c) {
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1) {
        int oc = __shfl_xor(c.conn, o, W);
        uint32_t ot = (uint32_t)__shfl_xor((int)c.tie, o, W);
        int ol = __shfl_xor(c.lab, o, W);
        int os = __shfl_xor(c.size, o, W);
        if (better(oc, ot, ol, c.conn, c.tie, c.lab)) {
            c.conn = oc;
            c.tie = ot;
            c.lab = ol;
            c.size = os;
        }
    }
}

// ---- lane groups of 8 and 16 (DPP: full-rate VALU moves, no LDS crossbar)
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppXor3 = 0x1B;  // quad_perm
constexpr int kDppRor = 0x120;                                    // row_ror: + 1 .. 15
constexpr int kDppMirror = 0x140, kDppHalfMirror = 0x141;         // lane xor 15, xor 7
template <int CTRL>
__device__ inline int dpp(int x) {
    return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, true);
}

// Maximum / minimum over the 8 or 16 lanes of a group, in every lane. After two steps the lanes
// of a quad agree, so the mirrors pair the quads and then the halves.
template <int W, class F>
__device__ inline int group_fold(int x, F f) {
    static_assert(W == 8 || W == 16, "lane groups of 8 or 16");
    x = f(x, dpp<kDppXor1>(x));
    x = f(x, dpp<kDppXor2>(x));
    x = f(x, dpp<kDppHalfMirror>(x));
    if constexpr (W == 16) x = f(x, dpp<kDppMirror>(x));
    return x;
}
template <int W>
__device__ inline int group_max(int x) {
    return group_fold<W>(x, [](int a, int b) { return max(a, b); });
}
template <int W>
__device__ inline uint32_t group_umax(uint32_t x) {
    return (uint32_t)group_fold<W>(
        (int)x, [](int a, int b) { return (int)max((uint32_t)a, (uint32_t)b); });
}
template <int W>
__device__ inline int group_min(int x) {
    return group_fold<W>(x, [](int a, int b) { return min(a, b); });
}

// conn[j] += the weights of the entries that CTRL brings from another lane and whose label is
// lab[j].
template <int CTRL, int E>
__device__ inline void add_equal(const int (&lab)[E], const int (&l)[E], const int (&w)[E],
                                 int (&conn)[E]) {
#pragma unroll
    for (int k = 0; k < E; ++k) {
        const int lr = dpp<CTRL>(l[k]), wr = dpp<CTRL>(w[k]);
#pragma unroll
        for (int j = 0; j < E; ++j) conn[j] += lr == lab[j] ? wr : 0;
    }
}
template <int R, int E>
__device__ inline void add_rotations(const int (&lab)[E], const int (&w)[E], int (&conn)[E]) {
    if constexpr (R < 16) {
        add_equal<kDppRor + R>(lab, lab, w, conn);
        add_rotations<R + 1>(lab, w, conn);
    }
}

// conn[j] = summed weight of the entries of the lane group (E per lane) with the label of the
// lane's entry j; absent entries have label -1 and weight 0. Every other lane is visited once: 8
// lanes by lane xor 1..7 (xor 4..7 through one half mirror), 16 lanes by rotations.
template <int W, int E>
__device__ inline void group_sums(const int (&lab)[E], const int (&w)[E], int (&conn)[E]) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
        conn[j] = w[j];
#pragma unroll
        for (int k = 0; k < E; ++k)
            if (k != j) conn[j] += lab[k] == lab[j] ? w[k] : 0;
    }
    if constexpr (W == 16) {
        add_rotations<1>(lab, w, conn);
    } else {
        int hl[E], hw[E];
#pragma unroll
        for (int k = 0; k < E; ++k) {
            hl[k] = dpp<kDppHalfMirror>(lab[k]);
            hw[k] = dpp<kDppHalfMirror>(w[k]);
#pragma unroll
            for (int j = 0; j < E; ++j) conn[j] += hl[k] == lab[j] ? hw[k] : 0;
        }
        add_equal<kDppXor1>(lab, lab, w, conn);
        add_equal<kDppXor2>(lab, lab, w, conn);
        add_equal<kDppXor3>(lab, lab, w, conn);
        add_equal<kDppXor1>(lab, hl, hw, conn);
        add_equal<kDppXor2>(lab, hl, hw, conn);
        add_equal<kDppXor3>(lab, hl, hw, conn);
    }
}

// Best candidate of a lane group: entry j of a lane brings (conn[j], lab[j], size[j]) if conn[j]
// >= 0 (entries of one label bring the same candidate). The maximum of better() is taken field by
// field, one fold each, instead of by exchanging whole candidates. conn = -1 if there is none.
template <int W, int E>
__device__ inline Cand group_best(uint32_t tie_seed, int v, const int (&conn)[E],
                                  const int (&lab)[E], const int (&size)[E]) {
    Cand c{-1, 0u, 0x7fffffff, 0};
#pragma unroll
    for (int j = 0; j < E; ++j) c.conn = max(c.conn, conn[j]);
    c.conn = group_max<W>(c.conn);
    uint32_t tie[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        tie[j] = 0u;
        if (conn[j] == c.conn) tie[j] = hash3(tie_seed, (uint32_t)v, (uint32_t)lab[j]);
        c.tie = max(c.tie, tie[j]);
    }
    c.tie = group_umax<W>(c.tie);
#pragma unroll
    for (int j = 0; j < E; ++j)
        if (conn[j] == c.conn && tie[j] == c.tie) c.lab = min(c.lab, lab[j]);
    c.lab = group_min<W>(c.lab);
#pragma unroll
    for (int j = 0; j < E; ++j)
        if (lab[j] == c.lab) c.size = max(c.size, size[j]);
    c.size = group_max<W>(c.size);
    return c;
}

template <int W>
__device__ inline int reduce_max(int x) {
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o, W));
    return x;
}

// A proposal's contribution to the admission scratch: weight and priority into the target label
// (inc / top) or, for a departure from an overloaded block, out of the own block (out / dtop).
struct Contrib {
    int label;  // -1: none
    int w;
    unsigned long long key;
    bool departure;
};

// Adds the threads' traversed edges to the counters: one atomic per workgroup of kBlock threads
// (all of them call this), at its end. Atomics on one line take turns in the L2: one per node
// or per 64 nodes was most of the time of a large launch.
__device__ inline void count_traversed(const LpArgs& a, unsigned long long edges) {
    __shared__ unsigned long long red[kBlock / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) edges += __shfl_xor(edges, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = edges;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long sum = 0;
        for (int i = 0; i < kBlock / 64; ++i) sum += red[i];
        if (sum) atomicAdd(&a.trav[blockIdx.x & 63], sum);
    }
}

// The proposal rule of one proposing node (called by one lane): writes the proposal slot of the
// node's list position (the admission kernels then read the slots of a list in order instead of
// gathering them by node) and returns the scratch contribution, which the caller adds with
// atomics.
template <LpMode M>
__device__ inline Contrib propose(const LpArgs& a, int pos, int v, int own, int w,
                                  int conn_own, const Cand& c) {
    Contrib r{-1, 0, 0ull, false};
    if (c.conn < 0) return r;  // no eligible candidate
    const int size_own = a.size[own];
    bool go;
    bool overloaded = false;
    if (M == LpMode::Cluster) {
        go = c.conn > conn_own || (c.conn == conn_own && c.size >= size_own);
    } else {
        overloaded = size_own > bound_of(a, own);
        go = c.conn > conn_own || overloaded ||
             (c.conn == conn_own && (long long)c.size + 2LL * w <= (long long)size_own);
    }
    if (!go) return r;
    const int gain = c.conn - conn_own;
    const unsigned long long key = prio_key(gain, v);
    a.prop_t[pos] = c.lab;
    a.prop_gain[pos] = gain;
    a.prop_ok[pos] = 1;
    const bool dep = M == LpMode::Refine && overloaded;
    return Contrib{dep ? own : c.lab, w, key, dep};
}

__device__ inline void add_contrib(const LpArgs& a, const Contrib& r) {
    if (r.label < 0) return;
    if (r.departure) {
        atomicAdd(&a.out[r.label], r.w);
        atomicMax(&a.dtop[r.label], r.key);
    } else {
        atomicAdd(&a.inc[r.label], r.w);
        atomicMax(&a.top[r.label], r.key);
    }
}

template <LpMode M>
__device__ inline void decide(const LpArgs& a, int pos, int v, int own, int w, int conn_own,
                              const Cand& c) {
    add_contrib(a, propose<M>(a, pos, v, own, w, conn_own, c));
}

// Decision scan of a wave's LDS label table: the best eligible label among the slots lane,
// lane + 64, ... below cap (keys K, summed weights V; empty slots -1) and the weight towards the
// own label. A pass takes SLOTS slots per lane: it reads their keys and values, then issues the
// label-weight (and per-label bound) gathers of all of them, then evaluates, so a lane waits for
// one gather latency per pass instead of one per slot. Candidates compare by the total order of
// better(), so the result does not depend on the scan order. `other` receives the lane's largest
// weight towards another label, eligible or not. (The workgroup-per-hub kernels keep the
// slot-by-slot scan: there the batched form measured slower.)
template <int SLOTS>
__device__ __attribute__((always_inline)) inline void scan_wave_table(
    const LpArgs& a, const int* K, const int* V, int cap, int lane, int v, int own, int nw,
    int& conn_own, Cand& c, int& other) {
    for (int base = lane; base < cap; base += SLOTS * 64) {
        int lk[SLOTS], lv[SLOTS], ls[SLOTS], lb[SLOTS];
#pragma unroll
        for (int j = 0; j < SLOTS; ++j) {
            const int i = base + j * 64;
            lk[j] = i < cap ? K[i] : -1;
            lv[j] = lk[j] >= 0 ? V[i] : 0;
        }
#pragma unroll
        for (int j = 0; j < SLOTS; ++j) ls[j] = lk[j] >= 0 && lk[j] != own ? a.size[lk[j]] : 0;
        if (a.lbound) {  // uniform (a select between the two would put a.bound in scratch)
#pragma unroll
            for (int j = 0; j < SLOTS; ++j)
                lb[j] = lk[j] >= 0 && lk[j] != own ? a.lbound[lk[j]] : 0;
        } else {
#pragma unroll
            for (int j = 0; j < SLOTS; ++j) lb[j] = a.bound;
        }
#pragma unroll
        for (int j = 0; j < SLOTS; ++j) {
            const int lab = lk[j];
            if (lab < 0) continue;
            if (lab == own) {
                conn_own = lv[j];
                continue;
            }
            other = max(other, lv[j]);
            if ((long long)ls[j] + nw >= (long long)lb[j] || lv[j] < c.conn) continue;
            const uint32_t t = hash3(a.tie_seed, (uint32_t)v, (uint32_t)lab);
            if (better(lv[j], t, lab, c.conn, c.tie, c.lab)) c = Cand{lv[j], t, lab, ls[j]};
        }
    }
}

// ---------------------------------------------------------------- W lanes per node, E edges per lane
// Nodes of up to W x E edges: 8 lanes x 1 or 2, 16 lanes x 2 or 4. Bound by vector instructions
// (RGG 2^22, 12 to 20 edges a node: the time of a launch is its instruction count over the SIMDs'
// rate), so the labels are summed by comparing every entry with every other one by DPP moves, four
// instructions a pair of lanes, without finding a leader per label (entries of one label bring the
// same candidate); several entries per lane share the rest of the work among fewer lanes.
// Measured per launch at RGG 2^22 against one entry per lane, leaders and whole candidates
// exchanged through the LDS crossbar: degree 9..16 102 -> 68 us, 17..32 105 -> 52 us.
// A virtual block holds IT x (kBlock / W) nodes: every lane group serves IT nodes at once, whose
// dependent loads (list, offsets, targets, labels, label weights) are issued together, so each
// wave has that many chains in flight.
// One virtual block (IT x kBlock / W nodes of the list); every thread of the workgroup calls it
// (it synchronises the workgroup). `edges` adds up the traversed edges (refinement and SETTLE).
// SETTLE: also flags the nodes that are not settled (kSettleRound).
template <LpMode M, int W, int E, int IT, bool SETTLE = false>
__device__ __attribute__((always_inline)) inline void group_vb(const LpArgs& a,
                                                               const int* __restrict__ list,
                                                               int base, int count, int vb,
                                                               unsigned long long& edges) {
    constexpr int NB = kBlock / W;  // nodes per item and workgroup
    const int gl = threadIdx.x & (W - 1);
    int v[IT], own[IT], beg[IT], deg[IT], lab[IT][E], w[IT][E];
    bool valid[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const long long gi = ((long long)vb * IT + i) * NB + threadIdx.x / W;
        valid[i] = gi < count;
        v[i] = valid[i] ? list[gi] : 0;
    }
    // every lane of the group takes part in the exchanges below: no early exit
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        own[i] = valid[i] ? a.label[v[i]] : -1;
        beg[i] = valid[i] ? a.xadj[v[i]] : 0;
        deg[i] = valid[i] ? a.xadj[v[i] + 1] - beg[i] : 0;
    }
#pragma unroll
    for (int i = 0; i < IT; ++i)
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const int e = gl + j * W;
            lab[i][j] = -1;
            w[i][j] = 0;
            if (e >= deg[i]) continue;
            if constexpr (W * E > 8) {  // rows of 9..64 entries: streamed (non-temporal)
                lab[i][j] = __builtin_nontemporal_load(a.adjncy + beg[i] + e);
                w[i][j] = __builtin_nontemporal_load(a.adjwgt + beg[i] + e);
            } else {
                lab[i][j] = a.adjncy[beg[i] + e];
                w[i][j] = a.adjwgt[beg[i] + e];
            }
        }
#pragma unroll
    for (int i = 0; i < IT; ++i)
#pragma unroll
        for (int j = 0; j < E; ++j)
            if (lab[i][j] >= 0) lab[i][j] = a.label[lab[i][j]];
    int nw[IT], sz[IT][E], lb[IT][E];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        nw[i] = valid[i] ? a.vwgt[v[i]] : 0;
#pragma unroll
        for (int j = 0; j < E; ++j)
            sz[i][j] = lab[i][j] >= 0 && lab[i][j] != own[i] ? a.size[lab[i][j]] : 0;
    }
    if (a.lbound) {  // uniform
#pragma unroll
        for (int i = 0; i < IT; ++i)
#pragma unroll
            for (int j = 0; j < E; ++j)
                lb[i][j] = lab[i][j] >= 0 && lab[i][j] != own[i] ? a.lbound[lab[i][j]] : 0;
    } else {
#pragma unroll
        for (int i = 0; i < IT; ++i)
#pragma unroll
            for (int j = 0; j < E; ++j) lb[i][j] = a.bound;
    }
    Contrib r[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        int conn[E], conn_own = 0, other = -1;
        group_sums<W>(lab[i], w[i], conn);
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const int l = lab[i][j];
            conn_own = max(conn_own, (l >= 0) & (l == own[i]) ? conn[j] : 0);
            // candidates: other labels with room for the node (a select without branches: hipcc
            // 7.2 lost the -1 of a lane in the branching form)
            const bool room = (long long)sz[i][j] + nw[i] < (long long)lb[i][j];
            if (SETTLE) other = max(other, (l >= 0) & (l != own[i]) ? conn[j] : -1);
            conn[j] = (l >= 0) & (l != own[i]) & room ? conn[j] : -1;
        }
        conn_own = group_max<W>(conn_own);
        if (SETTLE) {
            other = group_max<W>(other);
            if (valid[i] && gl == 0) a.next_active[v[i]] = other >= conn_own;
        }
        const Cand c = group_best<W>(a.tie_seed, v[i], conn, lab[i], sz[i]);
        const int pos = base + (int)(((long long)vb * IT + i) * NB) + threadIdx.x / W;
        r[i] = (valid[i] && gl == 0) ? propose<M>(a, pos, v[i], own[i], nw[i], conn_own, c)
                                     : Contrib{-1, 0, 0ull, false};
    }
    // The block's proposals are combined per (target, kind) in an LDS hash before the atomics:
    // many low-degree nodes propose the same (hub) label, and one atomic per distinct target
    // keeps them from serialising on it.
    constexpr int HC = 2 * IT * NB;  // slots (load <= 1/2)
    // probed with a mask: a size that is not a power of two leaves slots unreachable and the
    // probe loop below would never end
    static_assert((HC & (HC - 1)) == 0, "IT x kBlock / W must be a power of two");
    __shared__ int h_tag[HC];        // (label << 1) | departure, -1: empty
    __shared__ int h_w[HC];
    __shared__ unsigned long long h_key[HC];
    for (int i = threadIdx.x; i < HC; i += kBlock) {
        h_tag[i] = -1;
        h_w[i] = 0;
        h_key[i] = 0ull;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        if (r[i].label < 0) continue;
        const int tag = (r[i].label << 1) | (r[i].departure ? 1 : 0);
        const int h = probe_claim(h_tag, HC, tag);  // at most IT x NB tags in HC slots
        if (h < 0) {
            *a.err = kErrProbe;
            continue;
        }
        atomicAdd(&h_w[h], r[i].w);
        atomicMax(&h_key[h], r[i].key);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < HC; i += kBlock) {
        const int tag = h_tag[i];
        if (tag >= 0) add_contrib(a, Contrib{tag >> 1, h_w[i], h_key[i], (tag & 1) != 0});
    }
    if (M == LpMode::Refine || SETTLE) {
#pragma unroll
        for (int i = 0; i < IT; ++i)
            if (valid[i] && gl == 0) edges += (unsigned long long)deg[i];
    }
    __syncthreads();  // the LDS of this virtual block is read before the next one writes it
}

// ---------------------------------------------------------------- one wave per node
// Labels are aggregated in LDS: a hash table (open addressing, LDS atomics) in general, or a
// dense counter per label when the labels are the k blocks of the refinement and k is small.
// The node's table belongs to its wave, whose LDS operations are in order: no barriers.
constexpr int kWaveEdges = kWaveCap / 2 / 64;  // edges per lane at the largest degree
// EPL: edges per lane, 64 x EPL >= degree.
template <LpMode M, bool DENSE, int EPL, bool SETTLE>
__device__ __attribute__((always_inline)) inline void wave_node(const LpArgs& a, int pos, int v,
                                                                int beg, int deg, int num_labels,
                                                                int lane, int* K, int* V) {
    const int own = a.label[v];
    int cap = 64;
    if (DENSE) {
        cap = num_labels;
    } else {
        while (cap < 2 * deg) cap <<= 1;  // deg <= kWaveCap / 2 => cap <= kWaveCap
    }
    // All of a lane's edges are loaded first so that their label gathers are in flight together;
    // the LDS insertions follow.
    int labs[EPL], ws[EPL];
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        const int e = beg + lane + 64 * j;
        // a row read once per sub-round: streamed (non-temporal)
        labs[j] = e < beg + deg ? __builtin_nontemporal_load(a.adjncy + e) : -1;
        ws[j] = e < beg + deg ? __builtin_nontemporal_load(a.adjwgt + e) : 0;
    }
    for (int i = lane; i < cap; i += 64) {
        if (!DENSE) K[i] = -1;
        V[i] = 0;
    }
#pragma unroll
    for (int j = 0; j < EPL; ++j)
        if (labs[j] >= 0) labs[j] = a.label[labs[j]];
    wave_lds_order();
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        const int lab = labs[j];
        if (lab < 0) continue;
        const int w = ws[j];
        if (DENSE) {
            atomicAdd(&V[lab], w);
            continue;
        }
        const int h = probe_claim(K, cap, lab);  // cap >= 2 x degree
        if (h < 0) {
            *a.err = kErrProbe;
            continue;
        }
        atomicAdd(&V[h], w);
    }
    wave_lds_order();
    const int nw = a.vwgt[v];
    int conn_own = 0, other = -1;
    Cand c{-1, 0u, 0x7fffffff, 0};
    if (!DENSE) {
        scan_wave_table<EPL < 8 ? 2 * EPL : 8>(a, K, V, cap, lane, v, own, nw, conn_own, c, other);
    } else {
        for (int i = lane; i < cap; i += 64) {
            const int lab = V[i] ? i : -1;
            if (lab < 0) continue;
            const int conn = V[i];
            if (lab == own) {
                conn_own = conn;
                continue;
            }
            const int sz = a.size[lab];
            if ((long long)sz + nw >= (long long)bound_of(a, lab)) continue;
            const uint32_t t = hash3(a.tie_seed, (uint32_t)v, (uint32_t)lab);
            if (better(conn, t, lab, c.conn, c.tie, c.lab)) c = Cand{conn, t, lab, sz};
        }
    }
    conn_own = reduce_max<64>(conn_own);
    reduce_cand<64>(c);
    if (SETTLE) {
        other = reduce_max<64>(other);
        if (lane == 0) a.next_active[v] = other >= conn_own;
    }
    if (lane == 0) decide<M>(a, pos, v, own, nw, conn_own, c);
    wave_lds_order();  // the table is read before the wave's next node clears it
}

// One virtual block: kBlock / 64 nodes of the list, a wave each. DCAP: dense counters per wave
// (num_labels <= DCAP). Rows of up to LpArgs::wave_small edges take the variant with half the
// registers and predicated loads.
template <LpMode M, bool DENSE, int DCAP = kWaveDense, bool SETTLE = false>
__device__ __attribute__((always_inline)) inline void wave_vb(const LpArgs& a,
                                                              const int* __restrict__ list,
                                                              int base, int count, int num_labels,
                                                              int vb, unsigned long long& edges) {
    __shared__ int skey[kBlock / 64][DENSE ? 1 : kWaveCap];
    __shared__ int sval[kBlock / 64][DENSE ? DCAP : kWaveCap];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int gi = vb * (kBlock / 64) + wave;
    if (gi >= count) return;
    const int v = list[gi];
    const int beg = a.xadj[v], deg = a.xadj[v + 1] - beg;
    if (deg <= a.wave_small)
        wave_node<M, DENSE, kWaveEdges / 2, SETTLE>(a, base + gi, v, beg, deg, num_labels, lane,
                                            skey[wave], sval[wave]);
    else
        wave_node<M, DENSE, kWaveEdges, SETTLE>(a, base + gi, v, beg, deg, num_labels, lane,
                                                skey[wave], sval[wave]);
    if ((M == LpMode::Refine || SETTLE) && lane == 0) edges += (unsigned long long)deg;
}

// Clustering: the proposals of a sub-round's lists in one launch, the longest rows first, one
// workgroup per virtual block. A launch per list left the chip idle at the end of each, six times
// a sub-round. WAVES = false, for sub-rounds of lane groups only, needs no table (6 KB of LDS
// instead of 38).
// Measured, kahip_partition: R-MAT 2^17 k = 8 23.9 -> 20.8 ms, 2^13 k = 6 10.2 -> 9.0 ms,
// kahip_lp_cluster of R-MAT 2^20 18.5 -> 17.2 ms, of 2^15 3.3 -> 2.0 ms; meshes of 2^22 nodes,
// whose lists fill the chip, the same.
struct ClusterLists {
    const int* list[kNumBins - 1];
    int base[kNumBins - 1];  // list positions of their first entries
    int count[kNumBins - 1];
    const int* dcount;  // lengths on the device (a compacted sub-round), else nullptr
};
// Turnover of a sub-round without an admission launch (kTurnNodes): the workgroups past the lists'
// copy the label weights to the array that the application updates and clear the next sub-round's
// admission scratch, kTurnItems labels a thread.
constexpr int kTurnItems = 4;
template <int IT, bool WAVES, bool SETTLE>
__global__ __launch_bounds__(kBlock) void propose_lists(LpArgs a, ClusterLists F, Turnover T) {
    select_copy(a);
    constexpr LpMode C = LpMode::Cluster;
    constexpr int N = kNumBins - 1;
    constexpr int NPB[N] = {IT * (kBlock / 8), IT * (kBlock / 8), IT * (kBlock / 16),
                            IT * (kBlock / 16), kBlock / 64};
    int cnt[N], nvb[N], total = 0;
#pragma unroll
    for (int b = 0; b < N; ++b) {
        cnt[b] = SETTLE && F.dcount ? F.dcount[b] : F.count[b];
        nvb[b] = (cnt[b] + NPB[b] - 1) / NPB[b];
        total += nvb[b];
    }
    if (!SETTLE && (int)blockIdx.x >= total) {  // uniform
        const int i0 = ((int)blockIdx.x - total) * kBlock * kTurnItems + threadIdx.x;
#pragma unroll
        for (int j = 0; j < kTurnItems; ++j) {
            const int i = i0 + j * kBlock;
            if (i >= T.n) break;
            T.size[i] = a.size[i];
            T.inc[i] = 0;
            T.top[i] = 0ull;
        }
        return;
    }
    unsigned long long edges = 0;
    for (int t = blockIdx.x; t < total; t += gridDim.x) {  // one pass over whole lists
        int vb = t, b = N - 1;  // uniform per workgroup
#pragma unroll
        for (int k = N - 1; k > 0; --k)
            if (b == k && vb >= nvb[k]) {
                vb -= nvb[k];
                b = k - 1;
            }
        switch (b) {
            case 0: group_vb<C, 8, 1, IT, SETTLE>(a, F.list[0], F.base[0], cnt[0], vb, edges); break;
            case 1: group_vb<C, 8, 2, IT, SETTLE>(a, F.list[1], F.base[1], cnt[1], vb, edges); break;
            case 2: group_vb<C, 16, 2, IT, SETTLE>(a, F.list[2], F.base[2], cnt[2], vb, edges); break;
            case 3: group_vb<C, 16, 4, IT, SETTLE>(a, F.list[3], F.base[3], cnt[3], vb, edges); break;
            default:
                if constexpr (WAVES)
                    wave_vb<C, false, kWaveDense, SETTLE>(a, F.list[4], F.base[4], cnt[4], 0, vb,
                                                          edges);
        }
    }
    if (SETTLE && F.dcount) count_traversed(a, edges);  // (whole lists: known to the host)
}

// ---------------------------------------------------------------- clustering: settled nodes
// A node whose weight towards its own cluster exceeds that towards every other one does not
// propose, whatever the clusters' sizes and the tie-breaking, until it is moved or a neighbour
// moves into another cluster than the node's own. On a mesh that is most of the nodes after two
// rounds (RGG 2^18: 87 % after two, 92 % after three, 97 % after ten), so from round kSettleRound
// on a proposing kernel also flags the nodes that are not settled, an application flags the moved
// nodes and those neighbours, and from the round after it a sub-round first compacts its lists to
// the flagged nodes (right before it, as the earlier sub-rounds' moves unsettle nodes of this one).
// Earlier, most nodes move and flag all of their neighbours: measured, RGG 2^22, k = 2, coarsening
// from round 1 9.3, from 2 8.9, from 3 9.0 ms, without 10.1 ms. For graphs of more than kSettleEdges
// edges only: below, a sub-round is bound by its launches, and the compaction is one more (RGG of
// 60 001 nodes: 0.80 -> 1.12 ms). That still holds some way above the line: clustering and
// contraction of an RGG, k = 4, without flags and with them, 200 003 nodes 0.94 and 1.34, 400 003
// nodes 2.05 and 2.18, 1 000 003 nodes 2.98 and 2.83, 4 194 304 nodes 9.0 and 7.2 ms. Not for graphs
// with hubs: on R-MAT graphs 14 to 18 % of the nodes settle and hardly fewer edges are read. Not for
// a single sub-round: whole rounds of simultaneous moves leave 72 to 100 % of the edges with nodes
// that are not settled (dense communities alone gained, 0.75 to 0.93 of the time).
// And the graph has to settle: the flags cost the marking of every mover's row, so the first
// sub-round with flags is asked how much it has left, and if that is more than kSettleShare of its
// lists' edges, nothing is skipped. Left with 4 (8) sub-rounds, and clustering and contraction with
// all flags over those without any: RGG 0.32 to 0.35 (0.20), 4 194 304 nodes 0.80 (0.82); rings with
// rewired edges 0.36 (0.20), 400 000 nodes 0.89 (0.99); dense communities 0.00 to 0.06, 0.62 to 0.93
// (0.67 to 0.86); grid 2000 x 2000 0.47 (0.36), 0.96 (0.95); 160^3 0.59 (0.45), 1.05 (1.08); random
// and regular graphs of degree 8 to 500 0.70 to 1.00, 1.10 to 2.0 (1.12 to 2.1); RGG of average
// degree 247 0.85 (0.65), 1.24 (1.39); communities of 300 that the cluster bound splits 0.96, 2.1
// (2.9). With the answer no, 1.00 to 1.2.
constexpr int kSettleRound = 2;
constexpr long long kSettleEdges = 1LL << 21;
constexpr double kSettleShare = 0.5;

// Refinement: the proposals of all degree lists of a sub-round in one launch. The lists are the
// round's compacted frontier (lengths on the device); the workgroups stride over the virtual
// blocks of the five lists in order (8 or 16 lanes per node, then a wave per node), so a
// sub-round costs one launch instead of five. Same per-node code as the per-list kernels.
// Refinement hubs with kept per-block counters (every hub of the level has them when their
// counters fit): one wave per active hub decides from its k counters (as hub_dense_decide does
// with keep = 1; no row is read).
__device__ __attribute__((always_inline)) inline void hubcnt_vb(const LpArgs& a,
                                                                const int* __restrict__ list,
                                                                int base, int count,
                                                                int num_labels, int vb) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int gi = vb * (kBlock / 64) + wave;
    if (gi >= count) return;  // uniform per wave; no workgroup barrier below
    const int v = list[gi];
    const int* cnt = a.hub_cnt + a.hub_slot[v];
    const int own = a.label[v];
    const int nw = a.vwgt[v];
    int conn_own = 0;
    Cand c{-1, 0u, 0x7fffffff, 0};
    for (int b = lane; b < num_labels; b += 64) {
        const int conn = cnt[b];
        if (conn == 0) continue;
        if (b == own) {
            conn_own = conn;
            continue;
        }
        const int sz = a.size[b];
        if ((long long)sz + nw >= (long long)bound_of(a, b)) continue;
        const uint32_t t = hash3(a.tie_seed, (uint32_t)v, (uint32_t)b);
        if (better(conn, t, b, c.conn, c.tie, c.lab)) c = Cand{conn, t, b, sz};
    }
    conn_own = reduce_max<64>(conn_own);
    reduce_cand<64>(c);
    if (lane == 0) decide<LpMode::Refine>(a, base + gi, v, own, nw, conn_own, c);
}

struct FrontierLists {
    const int* list[kNumBins];
    int base[kNumBins];           // list positions of their first entries
    const int* dcount[kNumBins];  // dcount[kNumBins - 1] == nullptr: hubs decide elsewhere
};
template <int IT, bool DENSE, int DCAP = kWaveDense>
__global__ __launch_bounds__(kBlock) void propose_frontier(LpArgs a, FrontierLists F,
                                                           int num_labels) {
    constexpr int NPB[kNumBins] = {IT * (kBlock / 8), IT * (kBlock / 8), IT * (kBlock / 16),
                                   IT * (kBlock / 16), kBlock / 64, kBlock / 64};
    int cnt[kNumBins], nvb[kNumBins], total = 0;
#pragma unroll
    for (int b = 0; b < kNumBins; ++b) {
        cnt[b] = F.dcount[b] ? *F.dcount[b] : 0;
        nvb[b] = (cnt[b] + NPB[b] - 1) / NPB[b];
        total += nvb[b];
    }
    unsigned long long edges = 0;
    for (int t = blockIdx.x; t < total; t += gridDim.x) {
        int vb = t, b = 0;  // uniform per workgroup
#pragma unroll
        for (int k = 0; k < kNumBins - 1; ++k)
            if (b == k && vb >= nvb[k]) {
                vb -= nvb[k];
                b = k + 1;
            }
        switch (b) {
            case 0: group_vb<LpMode::Refine, 8, 1, IT>(a, F.list[0], F.base[0], cnt[0], vb, edges); break;
            case 1: group_vb<LpMode::Refine, 8, 2, IT>(a, F.list[1], F.base[1], cnt[1], vb, edges); break;
            case 2: group_vb<LpMode::Refine, 16, 2, IT>(a, F.list[2], F.base[2], cnt[2], vb, edges); break;
            case 3: group_vb<LpMode::Refine, 16, 4, IT>(a, F.list[3], F.base[3], cnt[3], vb, edges); break;
            case 4:
                wave_vb<LpMode::Refine, DENSE, DCAP>(a, F.list[4], F.base[4], cnt[4], num_labels, vb,
                                                      edges);
                break;
            default: hubcnt_vb(a, F.list[5], F.base[5], cnt[5], num_labels, vb);
        }
    }
    count_traversed(a, edges);
}

// Workgroup-wide reduction of (conn_own, best candidate); the result is valid in thread 0.
template <int THREADS>
__device__ inline void block_reduce(int& conn_own, Cand& c) {
    __shared__ Cand red[THREADS / 64];
    __shared__ int red_own[THREADS / 64];
    conn_own = reduce_max<64>(conn_own);
    reduce_cand<64>(c);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[wave] = c;
        red_own[wave] = conn_own;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < THREADS / 64; ++i) {
            conn_own = max(conn_own, red_own[i]);
            if (better(red[i].conn, red[i].tie, red[i].lab, c.conn, c.tie, c.lab)) c = red[i];
        }
    }
}

// ---------------------------------------------------------------- hubs, refinement: dense LDS
// Per-wave copies of the per-block counters (the k blocks are few, so a single shared array
// would serialise on LDS atomics), summed before the decision.
// Chunked variant for refinement hubs of more than kHubChunk edges: one workgroup per chunk sums
// its edges into per-wave LDS counters and adds the non-zero block sums to the hub's global
// counters (dense_off[hub] + b); hub_dense_decide then decides. Single-chunk hubs decide here.
// Hubs with global counters (dense_off >= 0) add their chunk sums there and are decided by
// hub_dense_decide. build: only those hubs, regardless of the frontier (the initial counters of
// the incremental scheme); incremental: those hubs are skipped (the moves keep their counters up
// to date).
__global__ __launch_bounds__(kHubDenseThreads) void propose_hub_dense_chunk(
    LpArgs a, const int4* __restrict__ cmap, int num_labels, const int* __restrict__ dense_off,
    int* __restrict__ dcnt, int build, int incremental) {
    extern __shared__ int cnt[];  // copies x num_labels counters (dynamic: small k, more blocks)
    const int4 cm = cmap[blockIdx.x];  // {hub index, chunk of the hub, chunks of the hub, node}
    const int gi = cm.x;
    const int v = cm.w;
    const bool counted = dense_off[gi] >= 0;  // the hub keeps global counters
    if (build ? !counted : (a.active[v] == 0 || (incremental && counted)))
        return;  // uniform per block
    const int c_idx = cm.y;
    const int beg = a.xadj[v];
    const int end = a.xadj[v + 1];
    const int e0 = beg + c_idx * kHubChunk;
    const int e1 = min(end, e0 + kHubChunk);
    const int copies = min(kHubDenseThreads / 64, kHubDenseSlots / num_labels);
    int* mine = cnt + ((threadIdx.x >> 6) % copies) * num_labels;
    for (int i = threadIdx.x; i < copies * num_labels; i += kHubDenseThreads) cnt[i] = 0;
    __syncthreads();
    constexpr int EPT = kHubChunk / kHubDenseThreads;
    int labs[EPT], ws[EPT];
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
        const int e = e0 + threadIdx.x + kHubDenseThreads * j;
        // the hub's row is read once per sub-round: streamed (non-temporal), so the caches stay
        // with the label gathers
        labs[j] = e < e1 ? __builtin_nontemporal_load(a.adjncy + e) : -1;
        ws[j] = e < e1 ? __builtin_nontemporal_load(a.adjwgt + e) : 0;
    }
#pragma unroll
    for (int j = 0; j < EPT; ++j)
        if (labs[j] >= 0) labs[j] = a.label[labs[j]];
#pragma unroll
    for (int j = 0; j < EPT; ++j)
        if (labs[j] >= 0) atomicAdd(&mine[labs[j]], ws[j]);
    __syncthreads();
    // traversed edges: the edges this chunk read (hubs deciding from kept counters read none)
    if (threadIdx.x == 0) atomicAdd(&a.trav[blockIdx.x & 63], (unsigned long long)(e1 - e0));
    if (counted) {
        int* out = dcnt + dense_off[gi];
        for (int b = threadIdx.x; b < num_labels; b += kHubDenseThreads) {
            int conn = 0;
            for (int j = 0; j < copies; ++j) conn += cnt[j * num_labels + b];
            if (conn) atomicAdd(&out[b], conn);
        }
        return;
    }
    const int own = a.label[v];
    const int nw = a.vwgt[v];
    int conn_own = 0;
    Cand c{-1, 0u, 0x7fffffff, 0};
    for (int b = threadIdx.x; b < num_labels; b += kHubDenseThreads) {
        int conn = 0;
        for (int j = 0; j < copies; ++j) conn += cnt[j * num_labels + b];
        if (conn == 0) continue;
        if (b == own) {
            conn_own = conn;
            continue;
        }
        const int sz = a.size[b];
        if ((long long)sz + nw >= (long long)bound_of(a, b)) continue;
        const uint32_t t = hash3(a.tie_seed, (uint32_t)v, (uint32_t)b);
        if (better(conn, t, b, c.conn, c.tie, c.lab)) c = Cand{conn, t, b, sz};
    }
    block_reduce<kHubDenseThreads>(conn_own, c);
    if (threadIdx.x == 0) decide<LpMode::Refine>(a, a.base + gi, v, own, nw, conn_own, c);
}

// One workgroup per multi-chunk refinement hub: decides from the summed counters and clears them
// (keep: the incremental counters stay).
__global__ __launch_bounds__(256) void hub_dense_decide(
    LpArgs a, const int* __restrict__ list, const int* __restrict__ multi, int n_multi,
    int num_labels, const int* __restrict__ dense_off, int* __restrict__ dcnt, int keep) {
    const int mi = blockIdx.x;
    if (mi >= n_multi) return;
    const int gi = multi[mi];
    const int v = list[gi];
    if (a.active[v] == 0) return;  // uniform per block
    int* cnt = dcnt + dense_off[gi];
    const int own = a.label[v];
    const int nw = a.vwgt[v];
    int conn_own = 0;
    Cand c{-1, 0u, 0x7fffffff, 0};
    for (int b = threadIdx.x; b < num_labels; b += 256) {
        const int conn = cnt[b];
        if (conn == 0) continue;
        if (!keep) cnt[b] = 0;
        if (b == own) {
            conn_own = conn;
            continue;
        }
        const int sz = a.size[b];
        if ((long long)sz + nw >= (long long)bound_of(a, b)) continue;
        const uint32_t t = hash3(a.tie_seed, (uint32_t)v, (uint32_t)b);
        if (better(conn, t, b, c.conn, c.tie, c.lab)) c = Cand{conn, t, b, sz};
    }
    block_reduce<256>(conn_own, c);
    // no traversed edges here: the chunks that read the hub's edges counted them
    if (threadIdx.x == 0) decide<LpMode::Refine>(a, a.base + gi, v, own, nw, conn_own, c);
}

// ---------------------------------------------------------------- hubs: chunked LDS hash
// One workgroup per chunk of CHUNK edges of a hub. The chunk's labels are aggregated in an LDS
// hash table; a hub of one chunk decides right away, otherwise the chunk's (label, partial sum)
// entries are written out grouped by bucket(label), one bucket per later workgroup. The mid-size
// instance (kMidThreads, kMidChunk) serves hubs of one chunk only, in small workgroups that
// share a CU eight at a time.
template <LpMode M, int THREADS, int CHUNK>
__global__ __launch_bounds__(THREADS) void propose_hub_chunk(
    LpArgs a, const int4* __restrict__ cmap, int2* __restrict__ partials,
    const long long* __restrict__ offm_base, int* __restrict__ offm,
    const int* __restrict__ ct_base, int* __restrict__ cntT) {
    constexpr int CAP = 2 * CHUNK;
    constexpr bool MULTI = CHUNK == kHubChunk;  // hubs of several chunks come here
    static_assert(!MULTI || THREADS == kHubThreads, "the multi-chunk path assumes kHubThreads");
    __shared__ int K[CAP];
    __shared__ int V[CAP];
    const int chunk = blockIdx.x;
    const int4 cm = cmap[chunk];  // {hub index, chunk of the hub, chunks of the hub, node}
    const int gi = cm.x;
    const int v = cm.w;
    if (M == LpMode::Refine && a.active[v] == 0) return;  // uniform per block
    const int nchunks = cm.z;
    const int c_idx = cm.y;
    const int beg = a.xadj[v];
    const int end = a.xadj[v + 1];
    const int e0 = beg + c_idx * CHUNK;
    const int e1 = min(end, e0 + CHUNK);
    // a hub of one chunk uses a table of the next power of two >= 2 x its degree
    int cap = CAP;
    if (nchunks == 1)
        while (cap > 256 && cap >= 4 * (e1 - e0)) cap >>= 1;
    for (int i = threadIdx.x; i < cap; i += THREADS) {
        K[i] = -1;
        V[i] = 0;
    }
    __syncthreads();
    // load every edge of the thread first (independent label gathers in flight), then insert
    constexpr int EPT = CHUNK / THREADS;
    int labs[EPT], ws[EPT];
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
        const int e = e0 + threadIdx.x + THREADS * j;
        // the hub's row is read once per sub-round: streamed (non-temporal), so the caches stay
        // with the label gathers
        labs[j] = e < e1 ? __builtin_nontemporal_load(a.adjncy + e) : -1;
        ws[j] = e < e1 ? __builtin_nontemporal_load(a.adjwgt + e) : 0;
    }
#pragma unroll
    for (int j = 0; j < EPT; ++j)
        if (labs[j] >= 0) labs[j] = a.label[labs[j]];
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
        const int lab = labs[j];
        if (lab < 0) continue;
        const int h = probe_claim(K, cap, lab);  // cap >= 2 x the chunk's edges
        if (h < 0) {
            *a.err = kErrProbe;
            continue;
        }
        atomicAdd(&V[h], ws[j]);
    }
    __syncthreads();
    if constexpr (MULTI) if (nchunks > 1) {
        // The chunk's (label, partial sum) entries, grouped by bucket(label): P buckets per hub,
        // bucket b of chunk c at [offm[c*(P+1)+b], offm[c*(P+1)+b+1]) of the chunk's region.
        __shared__ int bcur[kMaxBuckets + 1];
        __shared__ int wsum[kHubThreads / 64];
        const int P = min(kBucketsPerChunk * nchunks, kMaxBuckets);
        for (int i = threadIdx.x; i <= P; i += kHubThreads) bcur[i] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < kHubCap; i += kHubThreads)
            if (K[i] >= 0) atomicAdd(&bcur[bucket_of(K[i], P)], 1);
        __syncthreads();
        // exclusive scan of bcur[0..P): each thread owns a run of buckets
        const int per = (P + kHubThreads - 1) / kHubThreads;
        const int b0 = threadIdx.x * per, b1 = min(P, b0 + per);
        int run = 0;
        for (int b = b0; b < b1; ++b) run += bcur[b];
        int incl = run;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if ((int)(threadIdx.x & 63) >= o) incl += y;
        }
        if ((threadIdx.x & 63) == 63) wsum[threadIdx.x >> 6] = incl;
        __syncthreads();
        int wbase = 0;
        for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) wbase += wsum[w];
        int acc = wbase + incl - run;
        for (int b = b0; b < b1; ++b) {
            const int cnt = bcur[b];
            bcur[b] = acc;
            acc += cnt;
        }
        __syncthreads();
        int* offs = offm + offm_base[gi] + (long long)c_idx * (P + 1);
        int* cnt_t = cntT + ct_base[gi] + c_idx;  // bucket-major: [b * nchunks + c_idx]
        for (int b = threadIdx.x; b < P; b += kHubThreads) {
            offs[b] = bcur[b];
            if (b + 1 < P) cnt_t[(long long)b * nchunks] = bcur[b + 1] - bcur[b];
        }
        if (threadIdx.x == 0) {
            int tot = 0;
            for (int w = 0; w < kHubThreads / 64; ++w) tot += wsum[w];
            offs[P] = tot;
            cnt_t[(long long)(P - 1) * nchunks] = tot - bcur[P - 1];
        }
        __syncthreads();
        int2* out = partials + (long long)chunk * kHubChunk;
        for (int i = threadIdx.x; i < kHubCap; i += kHubThreads) {
            const int lab = K[i];
            if (lab < 0) continue;
            out[atomicAdd(&bcur[bucket_of(lab, P)], 1)] = make_int2(lab, V[i]);
        }
        return;
    }
    const int own = a.label[v];
    const int nw = a.vwgt[v];
    int conn_own = 0;
    Cand c{-1, 0u, 0x7fffffff, 0};
    for (int i = threadIdx.x; i < cap; i += THREADS) {
        const int lab = K[i];
        if (lab < 0) continue;
        const int conn = V[i];
        if (lab == own) {
            conn_own = conn;
            continue;
        }
        consider(a, v, nw, conn, lab, c);
    }
    block_reduce<THREADS>(conn_own, c);
    if (threadIdx.x == 0) {
        decide<M>(a, a.base + gi, v, own, nw, conn_own, c);
        if (M == LpMode::Refine) atomicAdd(&a.trav[blockIdx.x & 63], (unsigned long long)(end - beg));
    }
}

// Merge of one (multi-chunk hub, bucket) task: the bucket's entries of all chunks of the hub are
// summed in an LDS hash (or in the hub's global table, filtering by bucket); the bucket's best
// candidate and, for the bucket of the own label, conn(own) are left in bres / bown. LEVEL 1 (512
// threads, 32 KB of LDS, four per CU) takes every task of the sub-round; those of more than
// kSmallMax entries use the global table, or are queued for LEVEL 2 (1024 threads, 128 KB, up to
// kFinLds entries, grid-stride over the queue) where a hub's buckets have reached kMaxBuckets, so
// that tasks are larger than ~1000 entries by size and not by bad luck.
// One launch where there were four (a scan of the counts over all tasks, and a launch per level):
// measured in kahip_partition, together with the mid-size hubs' place in the chunk launch: R-MAT
// 2^17, k = 8 20.8 -> 19.0 ms (coarsening 9.1 -> 7.3), R-MAT 2^20, k = 16 coarsening 24.4 -> 22.8 ms.
// Sub-rounds of more than kTinyTasks tasks fill the chip many times over, a launch more is nothing
// there and a task's latency (chunk counts, table, reduction) is the bound: LEVEL 0 (256 threads,
// 16 KB, eight per CU) takes every task and queues those of more than kTinyMax entries for LEVEL 1.
// Eight waves per SIMD need at most 96 SGPRs (by launch_bounds; 106 without). Measured, merges of a
// clustering: R-MAT 2^24 (38 600 tasks a sub-round) 42.4 -> 27.8 ms, 2^22 (6 650) 7.1 -> 5.2, 2^21
// (3 950) 2.26 -> 1.85, 2^18 with 64 samples a node (2 390) 2.73 -> 2.62; LEVEL 0 below the limit:
// 2^20 (730) 2.13 -> 2.61, 2^17 (40) 0.64 -> 0.77 ms.
template <LpMode M, int LEVEL>
__global__ __launch_bounds__(LEVEL == 0 ? kTinyThreads : (LEVEL == 1 ? kSmallThreads : kFinThreads),
                             LEVEL == 2 ? 4 : 8)
void hub_bucket_merge(
    LpArgs a, int n_tasks, const int4* __restrict__ tmap, const int2* __restrict__ tsub,
    const int* __restrict__ cntT, const int* __restrict__ posT,
    const int* __restrict__ chunk_prefix, const long long* __restrict__ offm_base,
    const int* __restrict__ offm, const int2* __restrict__ partials,
    const long long* __restrict__ tab_off, int* __restrict__ gkey, int* __restrict__ gval,
    Cand* __restrict__ bres, int* __restrict__ bown, uint8_t* __restrict__ fb,
    const int* __restrict__ in_q, const int* __restrict__ in_n, int* __restrict__ out_q,
    int* __restrict__ out_n) {
    constexpr int THREADS = LEVEL == 0 ? kTinyThreads : (LEVEL == 1 ? kSmallThreads : kFinThreads);
    constexpr int CAP = LEVEL == 0 ? kTinyCap : (LEVEL == 1 ? kSmallCap : kFinCap);
    constexpr int MAXE = LEVEL == 0 ? kTinyMax : (LEVEL == 1 ? kSmallMax : kFinLds);
    static_assert(2 * MAXE <= CAP, "merge tables fill at most half");
    __shared__ int K[CAP];
    __shared__ int V[CAP];
    __shared__ int spre[kHubStage + 1];  // task offsets of the chunks' bucket segments
    __shared__ int sstart[kHubStage];    // the segments' starts in their chunks' partials
    __shared__ int wsum[kHubStage / 64];
    const int n_iter = LEVEL > 0 && in_q ? *in_n : n_tasks;
    for (int it = blockIdx.x; it < n_iter; it += gridDim.x) {
        const int task = LEVEL > 0 && in_q ? in_q[it] : it;
        const int4 tm = tmap[task];  // {first count index, one past the last, hub index, node}
        const int2 ts = tsub[task];  // {multi-chunk hub index, bucket | buckets << 16}
        const int mi = ts.x;
        const int gi = tm.z;
        const int v = tm.w;
        if (M == LpMode::Refine && a.active[v] == 0) {  // uniform per block
            __syncthreads();
            continue;
        }
        const int P = ts.y >> 16;
        const int b = ts.y & 0xffff;
        const int nch = tm.y - tm.x;
        const int* offs = offm + offm_base[gi] + b;
        const bool staged = nch <= kHubStage;  // uniform
        int r0 = 0, total;
        if (staged) {
            const int c = threadIdx.x;
            const int cnt = c < nch ? cntT[tm.x + c] : 0;
            if (c < nch) sstart[c] = offs[(long long)c * (P + 1)];
            int incl = cnt;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(incl, o, 64);
                if ((c & 63) >= o) incl += y;
            }
            if (c < kHubStage && (c & 63) == 63) wsum[c >> 6] = incl;
            __syncthreads();
            if (c < nch) {
                for (int w = 0; w < c >> 6; ++w) incl += wsum[w];
                spre[c + 1] = incl;
            }
            if (c == 0) spre[0] = 0;
            __syncthreads();
            total = spre[nch];
        } else {  // the sub-round's scan of the counts
            r0 = posT[tm.x];
            total = posT[tm.y] - r0;
        }
        if (LEVEL < 2 && total > MAXE && out_q) {
            if (threadIdx.x == 0) out_q[atomicAdd(out_n, 1)] = task;
            __syncthreads();
            continue;
        }
        const bool in_lds = total <= MAXE;
        const int deg = a.xadj[v + 1] - a.xadj[v];
        // The task's entries are read where the hub's chunks wrote them: chunk c holds entries
        // [pre(c), pre(c + 1)) of the task, pre the prefix of their counts, in its partials at
        // offm[offm_base[gi] + c (P + 1) + b]; the chunk of entry i is the largest c with
        // pre(c) <= i (empty segments are skipped).
        const long long c0 = chunk_prefix[gi];
        long long cap = CAP;
        int* TK = K;
        int* TV = V;
        if (in_lds) {
            cap = 64;
            while (cap < 2 * total) cap <<= 1;
            for (int i = threadIdx.x; i < cap; i += THREADS) {
                K[i] = -1;
                V[i] = 0;
            }
        } else {
            cap = 64;
            while (cap < 2LL * deg) cap <<= 1;
            TK = gkey + tab_off[gi];
            TV = gval + tab_off[gi];
            if (threadIdx.x == 0) fb[mi] = 1;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < total; i += THREADS) {
            int lo = 0, hi = nch - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                const int pm = staged ? spre[mid] : posT[tm.x + mid] - r0;
                if (pm <= i) lo = mid; else hi = mid - 1;
            }
            const int pre = staged ? spre[lo] : posT[tm.x + lo] - r0;
            const int start = staged ? sstart[lo] : offs[(long long)lo * (P + 1)];
            const int2 kv = partials[(c0 + lo) * kHubChunk + start + (i - pre)];
            // LDS: cap >= 2 x the bucket's entries; global: cap >= 2 x the hub's degree
            const long long h = probe_claim(TK, cap, kv.x);
            if (h < 0) {
                *a.err = kErrProbe;
                continue;
            }
            atomicAdd(&TV[h], kv.y);
        }
        // Only the global table needs the device-scope fence (it waits for the atomics and
        // invalidates the vector L1); it is costly, so the LDS path, the common one, skips it.
        if (!in_lds) __threadfence();  // uniform per block
        __syncthreads();
        const int own = a.label[v];
        const int nw = a.vwgt[v];
        int conn_own = 0;
        Cand c{-1, 0u, 0x7fffffff, 0};
        for (long long i = threadIdx.x; i < cap; i += THREADS) {
            const int lab = TK[i];
            if (lab < 0) continue;
            if (!in_lds && bucket_of(lab, P) != b) continue;
            const int conn = TV[i];
            if (lab == own) {
                conn_own = conn;
                continue;
            }
            consider(a, v, nw, conn, lab, c);
        }
        block_reduce<THREADS>(conn_own, c);
        if (threadIdx.x == 0) {
            bres[task] = c;
            bown[task] = conn_own;
        }
        __syncthreads();
    }
}

// One workgroup per multi-chunk hub: the best of its bucket winners decides; a global table used
// by an oversized bucket is cleared here.
template <LpMode M>
__global__ __launch_bounds__(256) void hub_decide(
    LpArgs a, const int* __restrict__ list, const int* __restrict__ multi, int n_multi,
    const int* __restrict__ task_prefix, const long long* __restrict__ tab_off,
    int* __restrict__ gkey, int* __restrict__ gval, const Cand* __restrict__ bres,
    const int* __restrict__ bown, uint8_t* __restrict__ fb) {
    const int mi = blockIdx.x;
    if (mi >= n_multi) return;
    const int gi = multi[mi];
    const int v = list[gi];
    if (M == LpMode::Refine && a.active[v] == 0) return;  // uniform per block
    const int t0 = task_prefix[mi], t1 = task_prefix[mi + 1];
    int conn_own = 0;
    Cand c{-1, 0u, 0x7fffffff, 0};
    for (int t = t0 + threadIdx.x; t < t1; t += 256) {
        conn_own = max(conn_own, bown[t]);
        const Cand o = bres[t];
        if (better(o.conn, o.tie, o.lab, c.conn, c.tie, c.lab)) c = o;
    }
    const int deg = a.xadj[v + 1] - a.xadj[v];
    block_reduce<256>(conn_own, c);
    if (threadIdx.x == 0) {
        decide<M>(a, a.base + gi, v, a.label[v], a.vwgt[v], conn_own, c);
        if (M == LpMode::Refine) atomicAdd(&a.trav[blockIdx.x & 63], (unsigned long long)deg);
    }
    if (fb[mi]) {  // uniform per block
        long long cap = 64;
        while (cap < 2LL * deg) cap <<= 1;
        int* TK = gkey + tab_off[gi];
        int* TV = gval + tab_off[gi];
        for (long long i = threadIdx.x; i < cap; i += 256) {
            TK[i] = -1;
            TV[i] = 0;
        }
        __syncthreads();
        if (threadIdx.x == 0) fb[mi] = 0;
    }
}

// ---------------------------------------------------------------- filter / admit / apply
// The filter / admit / apply kernels run over the node list of the sub-round; positions without a
// proposal (prop_t < 0) return at once, without reading their node: they stream the proposal
// slots. Measured, clustering of RGG 2^22, sub-rounds of 1 M nodes: with the slots by node id a
// late admission gathered a line per node, admit_moves 12 -> 8.5 us on average (the call
// 19.4 -> 18.5 ms).
__device__ inline void filter_one(const LpArgs& a, int pos, int v, int t) {
    const int own = a.label[v];
    const int so = a.size[own];
    const int ub = bound_of(a, own);
    if (so <= ub) return;  // not a departure from an overloaded block
    const int w = a.vwgt[v];
    const unsigned long long key = prio_key(a.prop_gain[pos], v);
    const bool pass = (long long)so - (long long)a.out[own] >= (long long)ub ||
                      a.dtop[own] == key;
    if (pass) {
        atomicAdd(&a.inc[t], w);
        atomicMax(&a.top[t], key);
    } else {
        a.prop_ok[pos] = 0;
    }
}

__device__ inline bool admit_one(const LpArgs& a, int pos, int v, int t) {
    if (!a.prop_ok[pos]) return false;
    const int w = a.vwgt[v];
    const long long st = a.size[t];
    const long long bt = bound_of(a, t);
    const bool ok = st + (long long)a.inc[t] < bt ||
                    (a.top[t] == prio_key(a.prop_gain[pos], v) && st + w < bt);
    if (!ok) a.prop_ok[pos] = 0;
    return ok;
}

// Applies the proposal of list position pos (node v to label t) if it is admitted and clears its
// scratch; true if v moved (from label *from).
template <LpMode M>
__device__ inline bool apply_one(const LpArgs& a, int pos, int v, int t, int* from) {
    const int own = a.label[v];
    a.inc[t] = 0;
    a.top[t] = 0ull;
    if (M == LpMode::Refine) {
        a.out[own] = 0;
        a.dtop[own] = 0ull;
    }
    a.prop_t[pos] = -1;
    if (!a.prop_ok[pos]) return false;
    const int w = a.vwgt[v];
    atomicSub(&a.size[own], w);
    atomicAdd(&a.size[t], w);
    a.label[v] = t;
    *from = own;
    return true;
}

__global__ void admit_moves(LpArgs a, const int* __restrict__ list, int count) {
    select_copy(a);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const int t = a.prop_t[a.base + i];
    if (t >= 0) admit_one(a, a.base + i, list[i], t);
}

// The clustering's application, at most kApplyGrid workgroups over the list. Few and large
// workgroups: each adds its moves to the round's one counter, and those atomics take turns
// (4096 workgroups of 256 took 48 us however few nodes moved). Measured, sub-rounds of 1 M nodes
// (RGG 2^22): 50 -> 20 us on average over the rounds, 5 us when few move.
constexpr int kApplyThreads = 1024;
constexpr int kApplyGrid = 512;
__global__ __launch_bounds__(kApplyThreads) void apply_moves(LpArgs a,
                                                             const int* __restrict__ list,
                                                             int count) {
    select_copy(a);
    __shared__ int block_moves;
    if (threadIdx.x == 0) block_moves = 0;
    __syncthreads();
    int mine = 0;
    for (unsigned i = blockIdx.x * kApplyThreads + threadIdx.x; i < (unsigned)count;
         i += gridDim.x * kApplyThreads) {
        const int t = a.prop_t[a.base + i];
        int from;
        if (t >= 0) mine += apply_one<LpMode::Cluster>(a, a.base + i, list[i], t, &from);
    }
    if (mine) atomicAdd(&block_moves, mine);
    __syncthreads();
    if (threadIdx.x == 0 && block_moves) atomicAdd(a.moves, block_moves);
}

// Admission and application in one launch: the weights that admission reads (a.size, a.inc, a.top)
// stay as they are, the moves go to the next sub-round's label weights (`size`, a copy of a.size),
// and the scratch is cleared by the next sub-round's proposals (Turnover). For graphs of up to
// kTurnNodes nodes, whose sub-rounds are bound by their launches: copying and clearing 20 bytes a
// label takes as long as the launch beyond (R-MAT 2^20: the same either way). Measured: RGG 2^22,
// k = 2 13.55 -> 13.17 ms (its coarse levels), R-MAT 2^17, k = 8 18.7 -> 18.3 ms, kahip_lp_cluster of
// R-MAT 2^15 1.97 -> 1.88 ms.
constexpr int kTurnNodes = 1 << 18;
__global__ __launch_bounds__(kApplyThreads) void admit_apply(LpArgs a, int* __restrict__ size,
                                                             const int* __restrict__ list,
                                                             int count) {
    __shared__ int block_moves;
    if (threadIdx.x == 0) block_moves = 0;
    __syncthreads();
    int mine = 0;
    for (unsigned i = blockIdx.x * kApplyThreads + threadIdx.x; i < (unsigned)count;
         i += gridDim.x * kApplyThreads) {
        const int pos = a.base + i;
        const int t = a.prop_t[pos];
        if (t < 0) continue;
        const int v = list[i], w = a.vwgt[v], own = a.label[v];
        const long long st = a.size[t], bt = bound_of(a, t);
        a.prop_t[pos] = -1;
        if (st + (long long)a.inc[t] < bt ||
            (a.top[t] == prio_key(a.prop_gain[pos], v) && st + w < bt)) {
            atomicSub(&size[own], w);
            atomicAdd(&size[t], w);
            a.label[v] = t;
            ++mine;
        }
    }
    if (mine) atomicAdd(&block_moves, mine);
    __syncthreads();
    if (threadIdx.x == 0 && block_moves) atomicAdd(a.moves, block_moves);
}

// The refinement's filter / admit / apply run over the sub-round's compacted frontier of every
// list, the hub list included (lengths on the device; every proposer is active, and nodes off
// the frontier have no proposal, on which the three steps do nothing). Thread i of the
// grid-stride loop takes element i of the lists' concatenation.
struct SubLists {
    const int* list[kNumBins];
    int base[kNumBins];           // list positions of their first entries
    const int* dcount[kNumBins];  // device-side length
};
__device__ inline int sub_lengths(const SubLists& L, int* cnt) {
    int total = 0;
#pragma unroll
    for (int b = 0; b < kNumBins; ++b) {
        cnt[b] = *L.dcount[b];
        total += cnt[b];
    }
    return total;
}
// Entry i of the lists' concatenation: its list position, the list in *list (with the entry at
// list[*index]).
__device__ inline int sub_entry(const SubLists& L, const int* cnt, int i, const int** list,
                                int* index) {
    // unrolled select (no dynamically indexed register array)
    const int* lp = L.list[0];
    int base = L.base[0];
    bool found = false;
#pragma unroll
    for (int b = 0; b < kNumBins; ++b) {
        const bool here = !found && i < cnt[b];
        if (here) {
            lp = L.list[b];
            base = L.base[b];
        }
        found |= here;
        if (!found) i -= cnt[b];
    }
    *list = lp;
    *index = i;
    return base + i;
}

__global__ __launch_bounds__(256) void filter_departures_sub(LpArgs a, SubLists L) {
    int cnt[kNumBins];
    const int total = sub_lengths(L, cnt);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int* list;
        int index;
        const int pos = sub_entry(L, cnt, i, &list, &index);
        const int t = a.prop_t[pos];
        if (t >= 0) filter_one(a, pos, list[index], t);
    }
}

// (also lists the admitted moves of long rows, a.big)
__global__ __launch_bounds__(256) void admit_moves_sub(LpArgs a, SubLists L) {
    int cnt[kNumBins];
    const int total = sub_lengths(L, cnt);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int* list;
        int index;
        const int pos = sub_entry(L, cnt, i, &list, &index);
        const int t = a.prop_t[pos];
        if (t < 0) continue;
        const int v = list[index];
        if (!admit_one(a, pos, v, t) || !a.big) continue;
        const int beg = a.xadj[v], deg = a.xadj[v + 1] - beg;
        if (deg > kLongRow) a.big[atomicAdd(a.n_big, 1)] = make_int4(beg, deg, a.label[v], t);
    }
}

// Application, then the rows of the moved nodes: their neighbours enter the next frontier, and
// hub neighbours with kept counters have them moved along. The rows of a step's movers are one
// range of edges over the workgroup's threads, kApplyEdges apiece in flight (an edge is a chain
// of three gathers: neighbour, hub slot, counter): with a lane per row, a row of 64 entries was
// 64 such chains one after the other. Measured, R-MAT 2^20, k = 16: 58 -> 37 us on average, R-MAT
// 2^17 16 -> 10 us.
// Clustering: flags the moved nodes and those neighbours that a move may unsettle (a neighbour in
// the target cluster stays settled, unless the edge's weight is negative). A neighbour moved by
// the same launch is flagged by its own move, so it does not matter which of its labels is read.
// Rows of more than kLongRow edges (one pass of the workgroup) are listed by the admission and
// spread over all workgroups in pieces: a moved hub's row, up to 100 passes one after the other, was
// the launch's time. Measured, R-MAT 2^20, k = 16: 26 -> 12 us on average, 2^17 10.7 -> 9.0 us.
// (Summing the counter updates per workgroup in LDS first: 30 us; they do not wait for each other.)
constexpr int kApplyEdges = 4;
static_assert(kLongRow == kApplyEdges * kBlock, "a piece of a long row is a pass of the workgroup");
template <LpMode M>
__global__ __launch_bounds__(kBlock) void apply_moves_sub(LpArgs a, SubLists L) {
    __shared__ int block_moves;
    __shared__ unsigned long long claimed;  // {movers, their edges} of the step
    __shared__ int row_at[kBlock];          // first edge of mover k in the step's range
    __shared__ int row_beg[kBlock], row_from[kBlock], row_to[kBlock];
    if (threadIdx.x == 0) block_moves = 0;
    int cnt[kNumBins];
    const int total = sub_lengths(L, cnt);
    unsigned long long edges = 0;
    // neighbours u at entries e (-1: none) of rows moved between the labels
    const auto mark = [&](const int (&e)[kApplyEdges], const int (&u)[kApplyEdges],
                          const int (&from)[kApplyEdges], const int (&to)[kApplyEdges]) {
        int slot[kApplyEdges];
#pragma unroll
        for (int j = 0; j < kApplyEdges; ++j) {
            slot[j] = -1;
            if (e[j] >= 0) {
                a.next_active[u[j]] = 1;
                if (a.hub_cnt) slot[j] = a.hub_slot[u[j]];
            }
        }
#pragma unroll
        for (int j = 0; j < kApplyEdges; ++j)
            if (slot[j] >= 0) {
                const int w = a.adjwgt[e[j]];
                atomicSub(&a.hub_cnt[slot[j] + from[j]], w);
                atomicAdd(&a.hub_cnt[slot[j] + to[j]], w);
            }
    };
    for (int base = blockIdx.x * kBlock; base < total; base += gridDim.x * kBlock) {  // uniform
        if (threadIdx.x == 0) claimed = 0ull;
        __syncthreads();
        const int i = base + threadIdx.x;
        const int* list;
        int index;
        const int pos = i < total ? sub_entry(L, cnt, i, &list, &index) : 0;
        const int t = i < total ? a.prop_t[pos] : -1;
        if (t >= 0) {
            const int v = list[index];
            int from;
            if (apply_one<M>(a, pos, v, t, &from)) {
                if (M == LpMode::Cluster) a.next_active[v] = 1;
                const int beg = a.xadj[v], row = a.xadj[v + 1] - beg;
                const bool lng = M == LpMode::Refine && row > kLongRow;
                if (lng) edges += (unsigned long long)row;
                const int deg = lng ? 0 : row;  // a long row is marked below
                // index and first edge from one atomic: the movers' edges ascend with k
                const unsigned long long at =
                    atomicAdd(&claimed, (1ull << 32) | (unsigned long long)deg);
                const int k = (int)(at >> 32);
                row_at[k] = (int)(unsigned)at;
                row_beg[k] = beg;
                row_from[k] = from;
                row_to[k] = t;
            }
        }
        __syncthreads();
        const int movers = (int)(claimed >> 32);
        const unsigned range = (unsigned)claimed;
        if (threadIdx.x == 0) {
            block_moves += movers;
            edges += (unsigned long long)range;
        }
        for (unsigned e0 = threadIdx.x; e0 < range; e0 += kApplyEdges * kBlock) {
            int u[kApplyEdges], k[kApplyEdges], e[kApplyEdges];
#pragma unroll
            for (int j = 0; j < kApplyEdges; ++j) {
                const unsigned x = e0 + j * kBlock;
                k[j] = 0;
                e[j] = -1;
                u[j] = 0;
                if (x < range) {
                    int lo = 0, hi = movers - 1;  // last mover with row_at <= x
                    while (lo < hi) {
                        const int mid = (lo + hi + 1) >> 1;
                        if ((unsigned)row_at[mid] <= x) lo = mid; else hi = mid - 1;
                    }
                    k[j] = lo;
                    e[j] = row_beg[lo] + (int)(x - (unsigned)row_at[lo]);
                    u[j] = a.adjncy[e[j]];
                }
            }
            if constexpr (M == LpMode::Cluster) {
                int lab[kApplyEdges];
#pragma unroll
                for (int j = 0; j < kApplyEdges; ++j) lab[j] = e[j] >= 0 ? a.label[u[j]] : 0;
#pragma unroll
                for (int j = 0; j < kApplyEdges; ++j)
                    if (e[j] >= 0 && (lab[j] != row_to[k[j]] || a.adjwgt[e[j]] < 0))
                        a.next_active[u[j]] = 1;
                continue;
            }
            int from[kApplyEdges], to[kApplyEdges];
#pragma unroll
            for (int j = 0; j < kApplyEdges; ++j) {
                from[j] = row_from[k[j]];
                to[j] = row_to[k[j]];
            }
            mark(e, u, from, to);
        }
        __syncthreads();  // the step's rows are done before the movers are reset
    }
    if (M == LpMode::Refine && a.big) {
        __shared__ int piece[kBlock];  // first piece past row i of the batch
        __shared__ int wave_pieces[kBlock / 64];
        const int n_big = *a.n_big;
        for (int b0 = 0; b0 < n_big; b0 += kBlock) {  // uniform
            const int i = b0 + (int)threadIdx.x;
            int incl = i < n_big ? (a.big[i].y + kLongRow - 1) / kLongRow : 0;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(incl, o, 64);
                if ((int)(threadIdx.x & 63) >= o) incl += y;
            }
            if ((threadIdx.x & 63) == 63) wave_pieces[threadIdx.x >> 6] = incl;
            __syncthreads();
            for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) incl += wave_pieces[w];
            piece[threadIdx.x] = incl;
            __syncthreads();
            const int pieces = piece[kBlock - 1];
            for (int p = blockIdx.x; p < pieces; p += gridDim.x) {
                int lo = 0, hi = kBlock - 1;  // first row that ends past p
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (piece[mid] > p) hi = mid; else lo = mid + 1;
                }
                const int4 r = a.big[b0 + lo];
                const int e0 = (p - (lo ? piece[lo - 1] : 0)) * kLongRow + (int)threadIdx.x;
                int e[kApplyEdges], u[kApplyEdges], from[kApplyEdges], to[kApplyEdges];
#pragma unroll
                for (int j = 0; j < kApplyEdges; ++j) {
                    e[j] = e0 + j * kBlock < r.y ? r.x + e0 + j * kBlock : -1;
                    u[j] = e[j] >= 0 ? a.adjncy[e[j]] : 0;
                    from[j] = r.z;
                    to[j] = r.w;
                }
                mark(e, u, from, to);
            }
            __syncthreads();  // `piece` is rewritten by the next batch
        }
    }
    if (M == LpMode::Refine) count_traversed(a, edges);
    if (threadIdx.x == 0 && block_moves) atomicAdd(a.moves, block_moves);
}

__global__ void set_hub_slots(const int* __restrict__ list, const int* __restrict__ multi,
                              int n_multi, const int* __restrict__ dense_off,
                              int* __restrict__ hub_slot) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_multi) return;
    const int i = multi[t];
    hub_slot[list[i]] = dense_off[i];
}

// ---------------------------------------------------------------- refinement: small frontiers
// After a few rounds the frontier of a refinement is a few hundred nodes (RGG 2^20, k = 2: 1 M
// nodes in round 0, then 600, 88, 24, none), and a round over the grid is bound by its launches
// (~3 us each, 14 a round) whatever the frontier. refine_tail runs the remaining rounds in one
// workgroup: the frontier, the proposals, the label weights and the admission scratch live in
// LDS, so a sub-round costs a few workgroup barriers, and the rounds end with the frontier. One
// workgroup and not a grid with device-wide barriers: a barrier across the XCDs' L2s costs about
// as much as a launch. The limits keep it to frontiers for which one CU is faster than the grid:
// a pass of 64 nodes of <= 16 edges takes about 2 us, so kTailNodes / 4 nodes of a sub-round
// stay at the cost of its launches; with fewer than four sub-rounds the frontier's limits are that
// much lower (tail_nodes, tail_edges: one sub-round, 2040 nodes of 16 edges, k = 500: kahip_lp_refine
// 3.40 ms with the limits of four, 1.02 with these, 1.32 before refine_tail). Larger frontiers (or
// labels beyond the LDS, or hubs among the nodes) are left to the grid. Graphs within the limits start
// here without node lists. Measured, calls of kahip_partition: RGG 2^10 k = 2 5.1 -> 2.2 ms (refinement 3.0 -> 0.3), RGG
// 2^22 k = 2 32.3 -> 26.1 ms, R-MAT 2^17 k = 8 39.1 -> 36.8 ms (its coarse levels settle early).
constexpr int kTailThreads = 1024;
constexpr int kTailNodes = 2048;     // frontier nodes, at most
constexpr int kTailEdges = 1 << 15;  // edges of the frontier's rows, at most
constexpr int kTailLabels = 512;     // labels (blocks) held in LDS
constexpr int kTailHash = 2 * kTailNodes;
constexpr int kTailWaves = kTailThreads / 64;
constexpr int kTailDegree = 512;     // largest degree (8 edges per lane of a wave)
constexpr int kTailGroup = 16;       // lanes per node of degree <= 16
inline int tail_nodes(int S) { return std::min(kTailNodes, S * (kTailNodes / 4)); }
inline int tail_edges(int S) { return std::min(kTailEdges, S * (kTailEdges / 4)); }

// Runs rounds a.round.. while the frontier is small; *state receives the round to go on with
// (`rounds`: all done), whose frontier is then flagged in a.next_active, or compacted already if
// no round ran.
__global__ __launch_bounds__(kTailThreads) void refine_tail(LpArgs a, TailArgs t) {
    __shared__ int lsize[kTailLabels], linc[kTailLabels], lout[kTailLabels];
    __shared__ unsigned long long ltop[kTailLabels], ldtop[kTailLabels];
    __shared__ int conn_of[kTailWaves][kTailLabels];
    __shared__ int raw[kTailNodes];   // the round's frontier, in any order
    __shared__ int item[kTailNodes];  // ... grouped by (sub-round, degree class)
    __shared__ int pt[kTailNodes], pg[kTailNodes];  // proposal of item i: target (-1 none), gain
    __shared__ int mv[kTailNodes];    // items moved in the sub-round
    __shared__ int hash[kTailHash];   // next frontier
    __shared__ int seg[2 * kMaxSub + 1], cur[2 * kMaxSub];
    __shared__ int pre[kMaxSub * kNumBins + 1];
    // (nfront is written by wave 0 or counted below, after the barrier)
    __shared__ int nfront, nnext, nedges, nmv, nmoves, over, spill, bad;
    __shared__ unsigned long long trav;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int grp = tid / kTailGroup, gl = tid & (kTailGroup - 1);
    const int k = t.num_labels;
    if (tid == 0) {
        nedges = over = bad = 0;
        trav = 0ull;
        if (!t.clists) nfront = 0;
    }
    if (t.clists && wave == 0) {  // list offsets in the frontier: nseg <= 48 lists, a lane each
        static_assert(kMaxSub * kNumBins < 64, "one lane per list");
        const int cnt = lane < t.nseg ? t.ccount[lane] : 0;
        int incl = cnt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        if (lane <= t.nseg) pre[lane] = incl - cnt;
        if (lane == 63) nfront = incl;
    }
    __syncthreads();
    for (int i = tid; i < t.nseg; i += kTailThreads)
        if (t.cnext) t.cnext[i] = 0;
    // the grid's filter launches are needed only while a block is overloaded: admitted moves
    // never overload one
    for (int b = tid; b < k; b += kTailThreads)
        if (a.size[b] > bound_of(a, b)) over = 1;
    if (t.clists) {
        if (nfront <= t.max_nodes)
            for (int i = tid; i < nfront; i += kTailThreads) {
                int lo = 0, hi = t.nseg - 1;  // last list starting at or before i
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (pre[mid] <= i) lo = mid; else hi = mid - 1;
                }
                raw[i] = t.clists[t.offsets[lo] + (i - pre[lo])];
            }
    } else {  // round 0 of a graph of at most t.max_nodes nodes (host)
        for (int v = tid; v < t.n; v += kTailThreads)
            if (a.xadj[v + 1] > a.xadj[v]) raw[atomicAdd(&nfront, 1)] = v;
    }
    __syncthreads();
    int r = t.round;
    bool fits = nfront <= t.max_nodes && k <= kTailLabels && !t.hubs;  // uniform
    if (fits) {
        for (int i = tid; i < nfront; i += kTailThreads) {
            const int d = a.xadj[raw[i] + 1] - a.xadj[raw[i]];
            atomicAdd(&nedges, min(d, kTailEdges));
            if (d > kTailDegree) bad = 1;
        }
        __syncthreads();
        fits = nedges <= t.max_edges && !bad;
    }
    if (fits && nfront > 0 && r < t.rounds) {
        for (int b = tid; b < k; b += kTailThreads) {
            lsize[b] = a.size[b];
            linc[b] = lout[b] = 0;
            ltop[b] = ldtop[b] = 0ull;
            for (int w = 0; w < kTailWaves; ++w) conn_of[w][b] = 0;
        }
        for (int i = tid; i < kTailHash; i += kTailThreads) hash[i] = -1;
        while (true) {  // one round; every branch below is uniform
            if (tid < 2 * kMaxSub) cur[tid] = 0;
            if (tid == 0) nmoves = nnext = nedges = spill = 0;
            __syncthreads();
            const int nf = nfront;
            // items by (sub-round, class): class 0 has up to kTailGroup edges
            int myc[kTailNodes / kTailThreads], myr[kTailNodes / kTailThreads];
#pragma unroll
            for (int j = 0; j < kTailNodes / kTailThreads; ++j) {
                const int i = tid + j * kTailThreads;
                myc[j] = -1;
                if (i < nf) {
                    const int v = raw[i];
                    const int d = a.xadj[v + 1] - a.xadj[v];
                    myc[j] = 2 * subround_of(t.seed, v, t.S) + (d > kTailGroup ? 1 : 0);
                    myr[j] = atomicAdd(&cur[myc[j]], 1);
                    atomicAdd(&trav, (unsigned long long)d);
                }
            }
            __syncthreads();
            if (wave == 0) {
                const int cnt = lane < 2 * kMaxSub ? cur[lane] : 0;
                int incl = cnt;
#pragma unroll
                for (int o = 1; o < 2 * kMaxSub; o <<= 1) {
                    const int y = __shfl_up(incl, o, 64);
                    if (lane >= o) incl += y;
                }
                if (lane <= 2 * kMaxSub) seg[lane] = lane < 2 * kMaxSub ? incl - cnt : nf;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kTailNodes / kTailThreads; ++j)
                if (myc[j] >= 0) {
                    const int at = seg[myc[j]] + myr[j];
                    item[at] = raw[tid + j * kTailThreads];
                    pt[at] = -1;
                }
            __syncthreads();
            const uint32_t tie_seed = tie_seed_of(t.seed, r);
            for (int sr = 0; sr < t.S; ++sr) {
                const int s0 = seg[2 * sr], s1 = seg[2 * sr + 1], s2 = seg[2 * sr + 2];
                if (s0 == s2) continue;
                if (tid == 0) nmv = 0;
                // the proposal of item i (one lane calls it)
                auto put = [&](int i, int v, int own, int w, int conn_own, const Cand& c) {
                    if (c.conn < 0) return;
                    const int so = lsize[own];
                    const bool ovl = so > bound_of(a, own);
                    if (!(c.conn > conn_own || ovl ||
                          (c.conn == conn_own && (long long)c.size + 2LL * w <= (long long)so)))
                        return;
                    pt[i] = c.lab;
                    pg[i] = c.conn - conn_own;
                    const unsigned long long key = prio_key(c.conn - conn_own, v);
                    atomicAdd(ovl ? &lout[own] : &linc[c.lab], w);
                    atomicMax(ovl ? &ldtop[own] : &ltop[c.lab], key);
                };
                // kTailGroup lanes per node of up to kTailGroup edges
                for (int base = s0; base < s1; base += kTailThreads / kTailGroup) {
                    const int i = base + grp;
                    const bool valid = i < s1;
                    const int v = valid ? item[i] : 0;
                    const int own = valid ? a.label[v] : -1;
                    const int beg = valid ? a.xadj[v] : 0;
                    const int deg = valid ? a.xadj[v + 1] - beg : 0;
                    int lab[1] = {gl < deg ? a.adjncy[beg + gl] : -1};
                    const int w[1] = {gl < deg ? a.adjwgt[beg + gl] : 0};
                    if (lab[0] >= 0) lab[0] = a.label[lab[0]];
                    const int nw = valid ? a.vwgt[v] : 0;
                    int conn[1], size[1] = {lab[0] >= 0 ? lsize[lab[0]] : 0};
                    group_sums<kTailGroup>(lab, w, conn);
                    const int conn_own =
                        group_max<kTailGroup>(lab[0] >= 0 && lab[0] == own ? conn[0] : 0);
                    const int lb = a.lbound ? (lab[0] >= 0 ? a.lbound[lab[0]] : 0) : a.bound;
                    const bool room = (long long)size[0] + nw < (long long)lb;
                    conn[0] = (lab[0] >= 0) & (lab[0] != own) & room ? conn[0] : -1;
                    const Cand c = group_best<kTailGroup>(tie_seed, v, conn, lab, size);
                    if (valid && gl == 0) put(i, v, own, nw, conn_own, c);
                }
                // one wave per larger node: a counter per label, summed with LDS atomics; every
                // lane then tries the labels of its own edges (a label's candidate is the same
                // whichever lane brings it)
                for (int i = s1 + wave; i < s2; i += kTailWaves) {
                    int* const V = conn_of[wave];
                    const int v = item[i];
                    const int own = a.label[v];
                    const int beg = a.xadj[v], end = a.xadj[v + 1];
                    constexpr int EPL = kTailDegree / 64;
                    int labs[EPL], ws[EPL];
#pragma unroll
                    for (int j = 0; j < EPL; ++j) {
                        const int e = beg + lane + 64 * j;
                        labs[j] = e < end ? a.adjncy[e] : -1;
                        ws[j] = e < end ? a.adjwgt[e] : 0;
                    }
#pragma unroll
                    for (int j = 0; j < EPL; ++j)
                        if (labs[j] >= 0) labs[j] = a.label[labs[j]];
#pragma unroll
                    for (int j = 0; j < EPL; ++j)
                        if (labs[j] >= 0) atomicAdd(&V[labs[j]], ws[j]);
                    wave_lds_order();
                    const int nw = a.vwgt[v];
                    int conn_own = 0;
                    Cand c{-1, 0u, 0x7fffffff, 0};
#pragma unroll
                    for (int j = 0; j < EPL; ++j) {
                        const int lab = labs[j];
                        if (lab < 0) continue;
                        const int conn = V[lab];
                        if (lab == own) {
                            conn_own = conn;
                            continue;
                        }
                        if ((long long)lsize[lab] + nw >= (long long)bound_of(a, lab)) continue;
                        const uint32_t tie = hash3(tie_seed, (uint32_t)v, (uint32_t)lab);
                        if (better(conn, tie, lab, c.conn, c.tie, c.lab))
                            c = Cand{conn, tie, lab, lsize[lab]};
                    }
                    conn_own = reduce_max<64>(conn_own);
                    reduce_cand<64>(c);
                    wave_lds_order();
#pragma unroll
                    for (int j = 0; j < EPL; ++j)
                        if (labs[j] >= 0) V[labs[j]] = 0;
                    if (lane == 0) put(i, v, own, nw, conn_own, c);
                }
                __syncthreads();
                // filter, admit and apply as on the grid, a thread per item
                constexpr int IPT = kTailNodes / kTailThreads;
                int own[IPT], w[IPT];
                bool ok[IPT];
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const int i = s0 + tid + j * kTailThreads;
                    ok[j] = i < s2 && pt[i] >= 0;
                    own[j] = ok[j] ? a.label[item[i]] : 0;
                    w[j] = ok[j] ? a.vwgt[item[i]] : 0;
                }
                if (over) {
#pragma unroll
                    for (int j = 0; j < IPT; ++j) {
                        const int i = s0 + tid + j * kTailThreads;
                        if (!ok[j]) continue;
                        const int so = lsize[own[j]], ub = bound_of(a, own[j]);
                        if (so <= ub) continue;
                        const unsigned long long key = prio_key(pg[i], item[i]);
                        if ((long long)so - (long long)lout[own[j]] >= (long long)ub ||
                            ldtop[own[j]] == key) {
                            atomicAdd(&linc[pt[i]], w[j]);
                            atomicMax(&ltop[pt[i]], key);
                        } else {
                            ok[j] = false;
                        }
                    }
                    __syncthreads();
                }
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const int i = s0 + tid + j * kTailThreads;
                    if (!ok[j]) continue;
                    const int to = pt[i];
                    const long long st = lsize[to], bt = bound_of(a, to);
                    ok[j] = st + (long long)linc[to] < bt ||
                            (ltop[to] == prio_key(pg[i], item[i]) && st + w[j] < bt);
                }
                __syncthreads();
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const int i = s0 + tid + j * kTailThreads;
                    if (i >= s2 || pt[i] < 0) continue;
                    const int to = pt[i], v = item[i], from = a.label[v];
                    linc[to] = 0;
                    ltop[to] = 0ull;
                    lout[from] = 0;
                    ldtop[from] = 0ull;
                    if (!ok[j]) continue;
                    atomicSub(&lsize[from], w[j]);
                    atomicAdd(&lsize[to], w[j]);
                    a.label[v] = to;
                    mv[atomicAdd(&nmv, 1)] = v;
                }
                __syncthreads();
                // the moved nodes' neighbours form the next frontier: flagged for the grid and
                // collected in the hash (a full hash only stops the collecting)
                const int nm = nmv;
                for (int m = wave; m < nm; m += kTailWaves) {
                    const int v = mv[m];
                    const int beg = a.xadj[v], end = a.xadj[v + 1];
                    if (lane == 0) atomicAdd(&trav, (unsigned long long)(end - beg));
                    for (int e = beg + lane; e < end; e += 64) {
                        const int u = a.adjncy[e];
                        a.next_active[u] = 1;
                        bool fresh = false;
                        if (!spill && probe_claim(hash, kTailHash, u, fresh) < 0) spill = 1;
                        if (fresh && atomicAdd(&nnext, 1) >= t.max_nodes) spill = 1;
                    }
                }
                if (tid == 0) nmoves += nm;
                __syncthreads();
            }
            if (tid == 0) {
                t.moves[r] = nmoves;
                nfront = 0;
            }
            ++r;
            __syncthreads();
            if (spill) break;
            for (int i = tid; i < kTailHash; i += kTailThreads) {
                const int u = hash[i];
                if (u < 0) continue;
                raw[atomicAdd(&nfront, 1)] = u;  // nnext <= t.max_nodes
                const int d = a.xadj[u + 1] - a.xadj[u];
                atomicAdd(&nedges, min(d, kTailEdges));
                if (d > kTailDegree) bad = 1;
            }
            __syncthreads();
            if (nfront == 0 || nedges > t.max_edges || bad || r == t.rounds) break;
            for (int i = tid; i < kTailHash; i += kTailThreads) {
                if (hash[i] >= 0) a.next_active[hash[i]] = 0;
                hash[i] = -1;
            }
            __syncthreads();
        }
        for (int b = tid; b < k; b += kTailThreads) a.size[b] = lsize[b];
        if (tid == 0 && trav) atomicAdd(&a.trav[0], trav);
    }
    __syncthreads();
    if (tid == 0) {
        const int next = nfront == 0 && !(r > t.round && spill) ? t.rounds : r;
        t.state[1] = next;
        t.state[2] = over;
        __threadfence_system();
        __hip_atomic_store(&t.state[0], t.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---------------------------------------------------------------- binning
__device__ inline int bin_of(const BinConfig& cfg, int deg) {
#pragma unroll
    for (int b = 0; b < kNumBins - 1; ++b)
        if (deg <= cfg.hi[b]) return b;
    return kNumBins - 1;
}

// The two binning kernels take a contiguous span of nodes per workgroup, at most kBinGrid of them:
// each adds its counts to (and claims its list parts from) the same few global counters, and
// those atomics take turns. With a workgroup per 256 nodes they were all of the time; kBinGrid
// workgroups fill the chip. Measured at n = 2^22: bin_count 265 -> 17 us,
// bin_scatter 250 -> 18 us.
constexpr int kBinThreads = 512;
constexpr int kBinGrid = 512;
constexpr int kBinItems = 4;  // nodes per thread in flight
constexpr int kBinLists = kMaxSub * kNumBins;

// List of node v (-1: in none).
__device__ inline int list_of(const BinConfig& cfg, const uint8_t* __restrict__ include,
                              uint32_t seed, int S, int v, int deg) {
    if (deg <= 0 || (include && !include[v])) return -1;
    return subround_of(seed, v, S) * kNumBins + bin_of(cfg, deg);
}

// counts[l] / edges[l]: nodes and edges of list l = sub-round * kNumBins + bin.
// blocks[workgroup][l]: the workgroup's nodes per list.
__global__ __launch_bounds__(kBinThreads) void bin_count(
    int n, int span, const int* __restrict__ xadj, uint32_t seed, int S, BinConfig cfg,
    const uint8_t* __restrict__ include, int* __restrict__ counts,
    unsigned long long* __restrict__ edges, int* __restrict__ blocks) {
    __shared__ unsigned long long local[kBinLists];  // {edges, nodes}: both below 2^31
    for (int i = threadIdx.x; i < kBinLists; i += kBinThreads) local[i] = 0ull;
    __syncthreads();
    const unsigned lo = blockIdx.x * span, hi = lo + min(span, (int)(n - lo));
    for (unsigned v0 = lo + threadIdx.x; v0 < hi; v0 += kBinItems * kBinThreads) {
        int deg[kBinItems];
#pragma unroll
        for (int j = 0; j < kBinItems; ++j) {
            const unsigned v = v0 + j * kBinThreads;
            deg[j] = v < hi ? xadj[v + 1] - xadj[v] : 0;
        }
#pragma unroll
        for (int j = 0; j < kBinItems; ++j) {
            const int v = (int)(v0 + j * kBinThreads);
            const int l = list_of(cfg, include, seed, S, v, deg[j]);
            if (l >= 0) atomicAdd(&local[l], ((unsigned long long)deg[j] << 32) | 1ull);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kBinLists; i += kBinThreads) {
        const int c = (int)(unsigned)local[i];
        blocks[blockIdx.x * kBinLists + i] = c;
        if (c) {
            atomicAdd(&counts[i], c);
            atomicAdd(&edges[i], local[i] >> 32);
        }
    }
}

__global__ __launch_bounds__(kBinThreads) void bin_scatter(
    int n, int span, const int* __restrict__ xadj, uint32_t seed, int S, BinConfig cfg,
    const uint8_t* __restrict__ include, const int* __restrict__ counts,
    const int* __restrict__ blocks, int* __restrict__ offsets, int* __restrict__ cursor,
    int* __restrict__ lists) {
    static_assert(kBinLists < 64, "one lane per list");
    __shared__ int next[kBinLists];  // the workgroup's next free entry per list
    __shared__ int off[64];
    if (threadIdx.x < 64) {  // list offsets: the lists in order (workgroup 0 keeps them)
        const int lane = threadIdx.x;
        const int cnt = lane < kBinLists ? counts[lane] : 0;
        int incl = cnt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        off[lane] = incl - cnt;
        if (blockIdx.x == 0 && lane < kBinLists) offsets[lane] = incl - cnt;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kBinLists; i += kBinThreads) {
        const int c = blocks[blockIdx.x * kBinLists + i];
        next[i] = c ? off[i] + atomicAdd(&cursor[i], c) : 0;
    }
    __syncthreads();
    const unsigned lo = blockIdx.x * span, hi = lo + min(span, (int)(n - lo));
    for (unsigned v0 = lo + threadIdx.x; v0 < hi; v0 += kBinItems * kBinThreads) {
        int deg[kBinItems];
#pragma unroll
        for (int j = 0; j < kBinItems; ++j) {
            const unsigned v = v0 + j * kBinThreads;
            deg[j] = v < hi ? xadj[v + 1] - xadj[v] : 0;
        }
#pragma unroll
        for (int j = 0; j < kBinItems; ++j) {
            const int v = (int)(v0 + j * kBinThreads);
            const int l = list_of(cfg, include, seed, S, v, deg[j]);
            if (l >= 0) lists[atomicAdd(&next[l], 1)] = v;
        }
    }
}

// Frontier of a refinement round, or the nodes that a sub-round looks at: the active nodes of the
// lists in entries [first, first + total), compacted per list into clists (same offsets as lists);
// ccount[l] receives list l's length. The order inside a list is free: the synchronous schedule
// does not depend on it. clear: the flags are consumed, so that the array serves as the next
// round's (unless a kernel of this round still reads them). also: further flags (or nullptr), kept.
constexpr int kCompactItems = 8;  // list entries per thread of compact_active
__global__ __launch_bounds__(256) void compact_active(const int* __restrict__ lists,
                                                      const int* __restrict__ offsets, int nseg,
                                                      int first, int total,
                                                      uint8_t* __restrict__ active,
                                                      int clear,
                                                      const uint8_t* __restrict__ also,
                                                      int* __restrict__ ccount,
                                                      int* __restrict__ clists) {
    __shared__ int off[kMaxSub * kNumBins];
    __shared__ int local[kMaxSub * kNumBins];
    __shared__ int base[kMaxSub * kNumBins];
    for (int i = threadIdx.x; i < nseg; i += blockDim.x) {
        off[i] = offsets[i];
        local[i] = 0;
    }
    __syncthreads();
    // kCompactItems entries per thread, 256 apart (coalesced), their flag gathers in flight
    // together; one global count update per list and workgroup
    const int i0 = first + blockIdx.x * 256 * kCompactItems + threadIdx.x;
    int v[kCompactItems], l[kCompactItems], r[kCompactItems];
#pragma unroll
    for (int j = 0; j < kCompactItems; ++j) {
        const int i = i0 + 256 * j;
        v[j] = i < first + total ? lists[i] : -1;
    }
#pragma unroll
    for (int j = 0; j < kCompactItems; ++j) {
        const int i = i0 + 256 * j;
        l[j] = -1;
        // every list, the hub list included (its frontier feeds the counter-based hub decisions)
        if (v[j] >= 0 && (active[v[j]] || (also && also[v[j]]))) {
            int lo = 0, hi = nseg - 1;  // last list with off <= i
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (off[mid] <= i) lo = mid; else hi = mid - 1;
            }
            l[j] = lo;
            r[j] = atomicAdd(&local[lo], 1);
            if (clear) active[v[j]] = 0;
        }
    }
    __syncthreads();
    for (int j = threadIdx.x; j < nseg; j += blockDim.x)
        base[j] = local[j] ? atomicAdd(&ccount[j], local[j]) : 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kCompactItems; ++j)
        if (l[j] >= 0) clists[off[l[j]] + base[l[j]] + r[j]] = v[j];
}

// Block descriptors of the hub kernels, built once per level: chunk c of the sub-round's hub
// list -> {hub index, chunk of the hub, chunks of the hub, node}.
__global__ void build_chunk_map(const int* __restrict__ list, int count,
                                const int* __restrict__ chunk_prefix, int4* __restrict__ cmap) {
    const int gi = blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= count) return;
    const int c0 = chunk_prefix[gi], c1 = chunk_prefix[gi + 1];
    const int v = list[gi];
    for (int c = c0; c < c1; ++c) cmap[c] = make_int4(gi, c - c0, c1 - c0, v);
}

// Hub gi of the mid-size kernel -> mmap[midpos[gi]] = {hub index, 0, 1, node}.
__global__ void build_mid_map(const int* __restrict__ list, int count,
                              const int* __restrict__ midpos, int4* __restrict__ mmap) {
    const int gi = blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= count) return;
    const int m = midpos[gi];
    if (m >= 0) mmap[m] = make_int4(gi, 0, 1, list[gi]);
}

// (hub, bucket) task t of a sub-round -> {multi-chunk hub index, bucket, buckets, hub index}.
// tmap[t] = {index of the bucket's first count in the bucket-major table, index one past its
// last, hub index, node}; tsub[t] = {multi-chunk hub index, bucket | buckets << 16}.
__global__ void build_task_map(const int* __restrict__ list, const int* __restrict__ multi,
                               int n_multi, const int* __restrict__ task_prefix,
                               const int* __restrict__ chunk_prefix,
                               const int* __restrict__ ct_base, int4* __restrict__ tmap,
                               int2* __restrict__ tsub) {
    const int mi = blockIdx.x * blockDim.x + threadIdx.x;
    if (mi >= n_multi) return;
    const int t0 = task_prefix[mi], t1 = task_prefix[mi + 1];
    const int gi = multi[mi];
    const int nch = chunk_prefix[gi + 1] - chunk_prefix[gi];
    const int cb = ct_base[gi];
    const int v = list[gi];
    for (int t = t0; t < t1; ++t) {
        const int b = t - t0;
        tmap[t] = make_int4(cb + b * nch, cb + (b + 1) * nch, gi, v);
        tsub[t] = make_int2(mi, b | ((t1 - t0) << 16));
    }
}

__global__ void hub_degrees(const int* __restrict__ list, int count, const int* __restrict__ xadj,
                            int* __restrict__ deg) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) deg[i] = xadj[list[i] + 1] - xadj[list[i]];
}

__global__ void fill_i32(int* p, long long n, int value) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

__global__ void copy_i32(int* __restrict__ to, const int* __restrict__ from, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) to[i] = from[i];
}

__global__ void fill_u64(unsigned long long* p, long long n, unsigned long long value) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

__global__ void fill_i64(long long* p, long long n, long long value) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

__global__ void fill_u8(uint8_t* p, long long n, uint8_t value) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

// Admission scratch of a clustering (labels = nodes) or refinement, the binning's counters and the
// error flag (if err).
__global__ void init_scratch(long long n, int* __restrict__ prop_t, long long nl,
                             int* __restrict__ inc, unsigned long long* __restrict__ top,
                             int* __restrict__ out, unsigned long long* __restrict__ dtop, int nbin,
                             int* __restrict__ bin, int* __restrict__ err) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nbin) bin[i] = 0;
    if (i == 0 && err) *err = 0;
    if (i < n) prop_t[i] = -1;
    if (i < nl) {
        inc[i] = 0;
        top[i] = 0ull;
        if (out) {
            out[i] = 0;
            dtop[i] = 0ull;
        }
    }
}

// Frontier flags (value, or those of start at map[i]) and list lengths of a refinement.
__global__ void init_frontier(int n, uint8_t* __restrict__ act, uint8_t value,
                              const int* __restrict__ map, const uint8_t* __restrict__ start,
                              uint8_t* __restrict__ nxt, int m, int* __restrict__ ccount) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        act[i] = start ? start[map[i]] : value;
        nxt[i] = 0;
    }
    if (i < m) ccount[i] = 0;
}

// From a start set, the first round compacts each sub-round's lists, one launch more each, and
// looks at the start set and at the neighbours of the nodes moved so far. It pays from about 2^19
// nodes on. Measured, refinement of RGG 2^22 k = 64: 1.73 -> 1.32 ms, 2^21 1.30 -> 1.15, 2^20 0.89
// -> 0.84, 2^19 0.716 -> 0.711; 2^18 0.675 -> 0.692, 2^16 0.457 -> 0.492 ms.
constexpr int kStartNodes = 1 << 19;
// Nodes that may have a neighbour in another block: those with one among their first
// kBorderEdges, and those of longer rows (one thread per row: a long one would keep the launch).
constexpr int kBorderEdges = 64;
__global__ __launch_bounds__(256) void border_nodes(int n, const int* __restrict__ xadj,
                                                    const int* __restrict__ adjncy,
                                                    const int* __restrict__ part,
                                                    uint8_t* __restrict__ border) {
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= n) return;
    const int own = part[v], beg = xadj[v], end = xadj[v + 1];
    uint8_t b = end - beg > kBorderEdges;
    for (int e = beg; e < end && !b; ++e) b = part[adjncy[e]] != own;
    border[v] = b;
}

// (blockIdx.y: copies, one after the other)
__global__ void init_labels(int n, int* __restrict__ label, int* __restrict__ size,
                            const int* __restrict__ vwgt) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    const long long o = (long long)blockIdx.y * n;
    if (v < n) {
        label[o + v] = v;
        size[o + v] = vwgt[v];
    }
}

__global__ void block_weights_kernel(int n, const int* __restrict__ part,
                                     const int* __restrict__ vwgt, int k, int* __restrict__ W) {
    extern __shared__ int lw[];
    for (int i = threadIdx.x; i < k; i += blockDim.x) lw[i] = 0;
    __syncthreads();
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x)
        atomicAdd(&lw[part[v]], vwgt[v]);
    __syncthreads();
    for (int i = threadIdx.x; i < k; i += blockDim.x)
        if (lw[i]) atomicAdd(&W[i], lw[i]);
}

__global__ void block_weights_global(int n, const int* __restrict__ part,
                                     const int* __restrict__ vwgt, int* __restrict__ W) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < n) atomicAdd(&W[part[v]], vwgt[v]);
}

inline int grid_for(long long work, int block) { return (int)((work + block - 1) / block); }

void launch_frontier(int items, bool dense, const LpArgs& a, const FrontierLists& F, int nl,
                     int listed, hipStream_t s) {
    // virtual blocks of at least 4 nodes: a listed count bounds the grid
    const dim3 grid(std::min(grid_for(listed, kBlock / 64), kFrontierGrid));
    // dense counters of k <= kWaveDenseSmall labels fit a quarter of the LDS
    const bool small = dense && nl <= kWaveDenseSmall;
    switch (items * 4 + (dense ? 1 : 0) + (small ? 2 : 0)) {
        case 4: hipLaunchKernelGGL((propose_frontier<1, false>), grid, dim3(kBlock), 0, s, a, F, nl); break;
        case 5: hipLaunchKernelGGL((propose_frontier<1, true>), grid, dim3(kBlock), 0, s, a, F, nl); break;
        case 7: hipLaunchKernelGGL((propose_frontier<1, true, kWaveDenseSmall>), grid, dim3(kBlock), 0, s, a, F, nl); break;
        case 16: hipLaunchKernelGGL((propose_frontier<4, false>), grid, dim3(kBlock), 0, s, a, F, nl); break;
        case 17: hipLaunchKernelGGL((propose_frontier<4, true>), grid, dim3(kBlock), 0, s, a, F, nl); break;
        case 19: hipLaunchKernelGGL((propose_frontier<4, true, kWaveDenseSmall>), grid, dim3(kBlock), 0, s, a, F, nl); break;
        case 9: hipLaunchKernelGGL((propose_frontier<2, true>), grid, dim3(kBlock), 0, s, a, F, nl); break;
        case 11: hipLaunchKernelGGL((propose_frontier<2, true, kWaveDenseSmall>), grid, dim3(kBlock), 0, s, a, F, nl); break;
        default: hipLaunchKernelGGL((propose_frontier<2, false>), grid, dim3(kBlock), 0, s, a, F, nl);
    }
}

}  // namespace

// ================================================================= host side

void fill_async(int* p, long long n, int value, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(fill_i32, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, value);
}
void fill_async(unsigned long long* p, long long n, unsigned long long value, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(fill_u64, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, value);
}
void fill_async(uint8_t* p, long long n, uint8_t value, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(fill_u8, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, value);
}
void fill_async(long long* p, long long n, long long value, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(fill_i64, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, value);
}

void LpWorkspace::prepare(LpMode mode, const DGraph& g, int num_labels, int S, uint32_t seed,
                          const BinConfig& bins, hipStream_t s, const uint8_t* include,
                          int copies) {
    KH_REQUIRE(copies == 1 || (mode == LpMode::Cluster && S == 1 && copies <= kMaxCopies),
               "copies are one-sub-round clusterings");
    KH_REQUIRE(S >= 1 && S <= kMaxSub, "sub-rounds must be in [1, 8]");
    KH_REQUIRE(bins.hi[kNumBins - 2] <= 512, "the wave bin holds degrees <= 512");
    KH_REQUIRE(bins.group_items == 1 || bins.group_items == 2 || bins.group_items == 4,
               "group_items must be 1, 2 or 4");
    KH_REQUIRE(bins.wave_small == 64 || bins.wave_small == 128 || bins.wave_small == 256,
               "wave_small must be 64, 128 or 256");
    bins_ = bins;
    KH_REQUIRE(g.n < (1 << 30) && num_labels < (1 << 30), "labels must be below 2^30");
    subrounds_ = S;
    num_labels_ = num_labels;
    ctl_.reserve(kCtlInts);
    clear_err_ = !keep_err_;  // (run() clears the other counters)
    keep_err_ = false;
    if (mode == LpMode::Refine) {
        active_.reserve(g.n);
        next_active_.reserve(g.n);
    }
    // a graph that refine_tail takes from round 0 needs no lists
    small_ = mode == LpMode::Refine && !include && g.n <= tail_nodes(S) &&
             g.m2 <= tail_edges(S) && num_labels <= kTailLabels;
    if (!small_) build_lists(mode, g, seed, s, include, copies);
    else if (clear_err_) fill_async(ctl_.p + kCtlErr, 1, 0, s);
    clear_err_ = false;  // (run() may build the lists later on)
}

void LpWorkspace::build_lists(LpMode mode, const DGraph& g, uint32_t seed, hipStream_t s,
                              const uint8_t* include, int copies) {
    const int S = subrounds_;
    const long long num_labels = num_labels_, scratch_n = (long long)copies * g.n;
    const long long scratch_l = copies * num_labels;
    const BinConfig& bins = bins_;
    dense_wave_ = mode == LpMode::Refine && num_labels <= kWaveDense;
    dense_hub_ = mode == LpMode::Refine && num_labels <= kHubDense;
    const int L = kMaxSub * kNumBins;
    lists_.reserve(g.n);
    if (mode == LpMode::Refine) {
        clists_.reserve(g.n);
        ccount_.reserve(2 * L);
    }
    offsets_.reserve(L);
    // {edges per list (64 bit), counts per list, cursors}
    constexpr int kBinInts = 4 * kMaxSub * kNumBins;
    bin_.reserve(kBinInts);
    unsigned long long* edges = reinterpret_cast<unsigned long long*>(bin_.p);
    counts_ = bin_.p + 2 * L;
    int* cursor = counts_ + L;
    prop_t_.reserve(scratch_n);
    prop_gain_.reserve(scratch_n);
    prop_ok_.reserve(scratch_n);
    inc_.reserve(scratch_l);
    top_.reserve(scratch_l);
    if (mode == LpMode::Refine) {
        out_.reserve(num_labels);
        dtop_.reserve(num_labels);
    }

    // a span of nodes per binning workgroup: one pass of its threads up to kBinGrid workgroups
    const int span = std::max(grid_for(grid_for(g.n, kBinGrid), kBinThreads), 1) * kBinThreads;
    const int bin_grid = grid_for(g.n, span);
    bin_blocks_.reserve((long long)bin_grid * kBinLists);
    const bool refine = mode == LpMode::Refine;
    const long long init_n = std::max<long long>({scratch_n, scratch_l, kBinInts});
    hipLaunchKernelGGL(init_scratch, dim3(grid_for(init_n, 256)), dim3(256), 0, s, scratch_n,
                       prop_t_.p, scratch_l, inc_.p, top_.p, refine ? out_.p : nullptr,
                       refine ? dtop_.p : nullptr, kBinInts, bin_.p,
                       clear_err_ ? ctl_.p + kCtlErr : nullptr);
    if (g.n > 0)
        hipLaunchKernelGGL(bin_count, dim3(bin_grid), dim3(kBinThreads), 0, s, g.n, span, g.xadj,
                           seed, S, bins, include, counts_, edges, bin_blocks_.p);
    mail_.post(s, {bin_.p, 2 * L + L});
    if (g.n > 0)
        hipLaunchKernelGGL(bin_scatter, dim3(bin_grid), dim3(kBinThreads), 0, s, g.n, span, g.xadj,
                           seed, S, bins, include, counts_, bin_blocks_.p, offsets_.p, cursor,
                           lists_.p);
    KH_CHECK(hipGetLastError());
    const int* got = mail_.wait(s);  // (the scatter runs meanwhile)
    std::memcpy(host_edges, got, sizeof(long long) * L);
    std::memcpy(host_counts, got + 2 * L, sizeof(int) * L);
    int acc = 0;
    for (int i = 0; i < L; ++i) {
        host_offsets[i] = acc;
        acc += host_counts[i];
    }

    // hubs (last bin): chunk prefix per sub-round list, global tables for multi-chunk hubs
    int hubs = 0;
    for (int sr = 0; sr < S; ++sr) {
        hub_base_[sr] = hubs;
        hub_n_[sr] = host_counts[sr * kNumBins + kNumBins - 1];
        hubs += hub_n_[sr];
    }
    hub_total_ = 0;
    dense_total_ = 0;
    for (int sr = 0; sr < S; ++sr) {
        hub_chunks_[sr] = hub_multi_n_[sr] = mid_n_[sr] = 0;
        mid_edges_[sr] = 0;
    }
    if (hubs == 0) {
        KH_CHECK(hipGetLastError());
        return;
    }
    hub_deg_.reserve(hubs);
    for (int sr = 0; sr < S; ++sr) {
        const int l = sr * kNumBins + kNumBins - 1;
        if (hub_n_[sr] == 0) continue;
        hipLaunchKernelGGL(hub_degrees, dim3(grid_for(hub_n_[sr], 256)), dim3(256), 0, s,
                           lists_.p + host_offsets[l], hub_n_[sr], g.xadj,
                           hub_deg_.p + hub_base_[sr]);
    }
    std::vector<int> deg(hubs);
    KH_CHECK(hipMemcpyAsync(deg.data(), hub_deg_.p, sizeof(int) * hubs, hipMemcpyDeviceToHost, s));
    KH_CHECK(hipStreamSynchronize(s));
    if (dense_hub_) {
        // chunked dense refinement: chunk prefix per sub-round and global counters for the hubs
        // that keep them (every hub when hubs x labels counters fit in kAllHubCounters, else the
        // hubs of more than one chunk)
        std::vector<int> prefix, multi, doff(hubs, -1);
        long long dtotal = 0;
        dense_all_ = (long long)hubs * num_labels <= kAllHubCounters;
        for (int sr = 0; sr < S; ++sr) {
            chunk_base_[sr] = (int)prefix.size();
            multi_base_[sr] = (int)multi.size();
            int c = 0;
            for (int i = 0; i < hub_n_[sr]; ++i) {
                const int nch = (deg[hub_base_[sr] + i] + kHubChunk - 1) / kHubChunk;
                prefix.push_back(c);
                c += nch;
                if (nch > 1 || dense_all_) {
                    doff[hub_base_[sr] + i] = (int)dtotal;
                    dtotal += num_labels;
                    multi.push_back(i);
                }
            }
            prefix.push_back(c);
            hub_chunks_[sr] = c;
            hub_multi_n_[sr] = (int)multi.size() - multi_base_[sr];
        }
        KH_REQUIRE(dtotal < (1LL << 31), "too many refinement hub counters");
        dense_total_ = dtotal;
        chunk_prefix_.reserve((long long)prefix.size());
        multi_.reserve(std::max<long long>((long long)multi.size(), 1));
        dense_off_.reserve(hubs);
        dense_cnt_.reserve(std::max<long long>(dtotal, 1));
        fill_async(dense_cnt_.p, std::max<long long>(dtotal, 1), 0, s);
        hub_slot_.reserve(g.n);
        fill_async(hub_slot_.p, g.n, -1, s);
        KH_CHECK(hipMemcpyAsync(chunk_prefix_.p, prefix.data(), sizeof(int) * prefix.size(),
                                hipMemcpyHostToDevice, s));
        if (!multi.empty())
            KH_CHECK(hipMemcpyAsync(multi_.p, multi.data(), sizeof(int) * multi.size(),
                                    hipMemcpyHostToDevice, s));
        KH_CHECK(hipMemcpyAsync(dense_off_.p, doff.data(), sizeof(int) * hubs,
                                hipMemcpyHostToDevice, s));
        build_chunk_maps(s);
        for (int sr = 0; sr < S; ++sr)
            if (hub_multi_n_[sr] > 0)
                hipLaunchKernelGGL(set_hub_slots, dim3(grid_for(hub_multi_n_[sr], 256)),
                                   dim3(256), 0, s,
                                   lists_.p + host_offsets[sr * kNumBins + kNumBins - 1],
                                   multi_.p + multi_base_[sr], hub_multi_n_[sr],
                                   dense_off_.p + hub_base_[sr], hub_slot_.p);
        KH_CHECK(hipStreamSynchronize(s));  // the host vectors must outlive the copies
        KH_CHECK(hipGetLastError());
        return;
    }
    std::vector<int> prefix, multi, tasks, midpos(hubs, -1);
    std::vector<long long> toff(hubs, 0), tcap(hubs, 0), obase(hubs, 0);
    std::vector<int> ctb(hubs, 0);
    int mids = 0;
    long long offm_total = 0, ct_total = 0, ct_sr_start = 0;
    int max_tasks = 0, max_multi = 0;
    for (int sr = 0; sr < S; ++sr) {
        chunk_base_[sr] = (int)prefix.size();
        multi_base_[sr] = (int)multi.size();
        task_base_[sr] = (int)tasks.size();
        int c = 0, t = 0;
        mid_base_[sr] = mids;
        mid_edges_[sr] = 0;
        hub_wide_[sr] = hub_capped_[sr] = false;
        long long units = 0;  // chunks and mid-size hubs
        for (int i = 0; i < hub_n_[sr]; ++i)
            units += (deg[hub_base_[sr] + i] + kHubChunk - 1) / kHubChunk;
        const bool join = units <= kHubJoin;
        for (int i = 0; i < hub_n_[sr]; ++i) {
            const int d = deg[hub_base_[sr] + i];
            prefix.push_back(c);
            if (d <= kMidChunk && !join) {  // the mid-size kernel, no chunk of the big one
                midpos[hub_base_[sr] + i] = mids++ - mid_base_[sr];
                mid_edges_[sr] += d;
                continue;
            }
            const int nch = (d + kHubChunk - 1) / kHubChunk;
            c += nch;
            if (nch > 1) {
                const int P = std::min(kBucketsPerChunk * nch, kMaxBuckets);
                hub_wide_[sr] |= nch > kHubStage;
                hub_capped_[sr] |= P < kBucketsPerChunk * nch;
                long long cap = 64;
                while (cap < 2LL * d) cap <<= 1;
                toff[hub_base_[sr] + i] = hub_total_;
                tcap[hub_base_[sr] + i] = cap;
                hub_total_ += cap;
                obase[hub_base_[sr] + i] = offm_total;
                offm_total += (long long)nch * (P + 1);
                ctb[hub_base_[sr] + i] = (int)ct_total;
                ct_total += (long long)nch * P;
                multi.push_back(i);
                tasks.push_back(t);
                t += P;
            }
        }
        prefix.push_back(c);
        tasks.push_back(t);
        ct_sr_base_[sr] = (int)ct_sr_start;
        ct_sr_size_[sr] = (int)(ct_total - ct_sr_start);
        ct_total += 1;  // zero sentinel after the sub-round's counts
        ct_sr_start = ct_total;
        hub_chunks_[sr] = c;
        mid_n_[sr] = mids - mid_base_[sr];
        hub_multi_n_[sr] = (int)multi.size() - multi_base_[sr];
        hub_tasks_[sr] = t;
        max_tasks = std::max(max_tasks, t);
        max_multi = std::max(max_multi, hub_multi_n_[sr]);
    }
    chunk_prefix_.reserve((long long)prefix.size());
    tab_off_.reserve(hubs);
    tab_cap_.reserve(hubs);
    offm_base_.reserve(hubs);
    task_prefix_.reserve((long long)tasks.size());
    multi_.reserve((long long)multi.size());
    offm_.reserve(offm_total);
    KH_REQUIRE(ct_total < (1LL << 31), "hub bucket table exceeds 2^31 entries");
    ct_base_.reserve(hubs);
    cnt_t_.reserve(ct_total);
    pos_t_.reserve(ct_total);
    if (std::any_of(hub_wide_, hub_wide_ + S, [](bool w) { return w; }))
        fill_async(cnt_t_.p, ct_total, 0, s);  // sentinels stay zero
    KH_CHECK(hipMemcpyAsync(ct_base_.p, ctb.data(), sizeof(int) * hubs, hipMemcpyHostToDevice,
                            s));
    {
        size_t bytes = 0, need = 0;
        for (int sr = 0; sr < S; ++sr) {
            if (!hub_wide_[sr]) continue;
            KH_CHECK(rocprim::exclusive_scan(nullptr, bytes, cnt_t_.p, pos_t_.p, 0,
                                             (size_t)ct_sr_size_[sr] + 1, rocprim::plus<int>(), s));
            need = std::max(need, bytes);
        }
        scan_tmp_.reserve((long long)need + 1);
        scan_tmp_bytes_ = need;
    }
    bres_.reserve(max_tasks);
    bown_.reserve(max_tasks);
    big_tasks_.reserve(max_tasks);
    if (max_tasks > kTinyTasks) mid_tasks_.reserve(max_tasks);
    fb_.reserve(max_multi);
    fill_async(fb_.p, max_multi, (uint8_t)0, s);
    KH_CHECK(hipMemcpyAsync(chunk_prefix_.p, prefix.data(), sizeof(int) * prefix.size(),
                            hipMemcpyHostToDevice, s));
    KH_CHECK(hipMemcpyAsync(tab_off_.p, toff.data(), sizeof(long long) * hubs,
                            hipMemcpyHostToDevice, s));
    KH_CHECK(hipMemcpyAsync(tab_cap_.p, tcap.data(), sizeof(long long) * hubs,
                            hipMemcpyHostToDevice, s));
    KH_CHECK(hipMemcpyAsync(offm_base_.p, obase.data(), sizeof(long long) * hubs,
                            hipMemcpyHostToDevice, s));
    KH_CHECK(hipMemcpyAsync(task_prefix_.p, tasks.data(), sizeof(int) * tasks.size(),
                            hipMemcpyHostToDevice, s));
    if (!multi.empty())
        KH_CHECK(hipMemcpyAsync(multi_.p, multi.data(), sizeof(int) * multi.size(),
                                hipMemcpyHostToDevice, s));
    build_chunk_maps(s);
    mmap_.reserve(std::max(mids, 1));
    midpos_.reserve(hubs);
    KH_CHECK(hipMemcpyAsync(midpos_.p, midpos.data(), sizeof(int) * hubs, hipMemcpyHostToDevice,
                            s));
    for (int sr = 0; sr < S; ++sr) {
        KH_REQUIRE(mid_base_[sr] + mid_n_[sr] <= std::max(mids, 1), "mid hub map overflow");
        if (mid_n_[sr] > 0)
            hipLaunchKernelGGL(build_mid_map, dim3(grid_for(hub_n_[sr], 256)), dim3(256), 0, s,
                               lists_.p + host_offsets[sr * kNumBins + kNumBins - 1], hub_n_[sr],
                               midpos_.p + hub_base_[sr], mmap_.p + mid_base_[sr]);
    }
    {
        long long all_tasks = 0;  // one descriptor per (hub, bucket) task of every sub-round
        for (int sr = 0; sr < S; ++sr) all_tasks += hub_tasks_[sr];
        tmap_.reserve(std::max<long long>(all_tasks, 1));
        tsub_.reserve(std::max<long long>(all_tasks, 1));
        long long tb = 0;
        for (int sr = 0; sr < S; ++sr) {
            KH_REQUIRE(tb + hub_tasks_[sr] <= all_tasks, "task map overflow");
            if (hub_multi_n_[sr] > 0)
                hipLaunchKernelGGL(build_task_map, dim3(grid_for(hub_multi_n_[sr], 256)), dim3(256),
                                   0, s, lists_.p + host_offsets[sr * kNumBins + kNumBins - 1],
                                   multi_.p + multi_base_[sr], hub_multi_n_[sr],
                                   task_prefix_.p + task_base_[sr],
                                   chunk_prefix_.p + chunk_base_[sr], ct_base_.p + hub_base_[sr],
                                   tmap_.p + tb, tsub_.p + tb);
            tmap_base_[sr] = (int)tb;
            tb += hub_tasks_[sr];
        }
    }
    if (hub_total_ > 0) {
        hub_key_.reserve(hub_total_);
        hub_val_.reserve(hub_total_);
        fill_async(hub_key_.p, hub_total_, -1, s);
        fill_async(hub_val_.p, hub_total_, 0, s);
    }
    int max_chunks = 0;
    for (int sr = 0; sr < S; ++sr) max_chunks = std::max(max_chunks, hub_chunks_[sr]);
    partials_.reserve((long long)max_chunks * kHubChunk);
    KH_CHECK(hipStreamSynchronize(s));  // the host vectors above must outlive the copies
    KH_CHECK(hipGetLastError());
}

void LpWorkspace::build_chunk_maps(hipStream_t s) {
    long long total = 0;
    for (int sr = 0; sr < subrounds_; ++sr) total += hub_chunks_[sr];
    cmap_.reserve(std::max<long long>(total, 1));
    long long cb = 0;
    for (int sr = 0; sr < subrounds_; ++sr) {
        KH_REQUIRE(cb + hub_chunks_[sr] <= total, "chunk map overflow");
        cmap_base_[sr] = (int)cb;
        if (hub_n_[sr] > 0)
            hipLaunchKernelGGL(build_chunk_map, dim3(grid_for(hub_n_[sr], 256)), dim3(256), 0, s,
                               lists_.p + host_offsets[sr * kNumBins + kNumBins - 1], hub_n_[sr],
                               chunk_prefix_.p + chunk_base_[sr], cmap_.p + cb);
        cb += hub_chunks_[sr];
    }
}

void LpWorkspace::run(LpMode mode, const DGraph& g, int* label, int* size, int bound, int rounds,
                      uint32_t seed, hipStream_t s, Profiler* prof, const char* phase,
                      const int* lbound, const int* map, const uint8_t* start) {
    KH_REQUIRE(rounds >= 0 && rounds <= kMaxRounds, "LP rounds must be in [0, 64]");
    const int S = subrounds_;
    const bool cl = mode == LpMode::Cluster;
    KH_REQUIRE(cl || !(dense_wave_ || dense_hub_) || num_labels_ > 0, "prepare() not called");
    whole_rounds_ = rounds;
    settled_rec_ = -1;
    fill_async(ctl_.p, kCtlErr, 0, s);  // the error flag is cleared by prepare()
    fetched_ = false;
    if (rounds == 0) return;
    LpArgs a{};
    a.xadj = g.xadj;
    a.adjncy = g.adjncy;
    a.adjwgt = g.adjwgt;
    a.vwgt = g.vwgt;
    a.label = label;
    a.size = size;
    a.bound = bound;
    a.lbound = lbound;
    a.wave_small = bins_.wave_small;
    a.trav = reinterpret_cast<unsigned long long*>(ctl_.p);
    a.err = ctl_.p + kCtlErr;
    uint8_t* act = active_.p;
    uint8_t* nxt = next_active_.p;
    int r = 0;
    bool filter = !cl;  // an overloaded block may exist
    if (small_) {
        // the whole refinement in one workgroup; the lists are built only if it stops early
        hipLaunchKernelGGL(init_frontier, dim3(std::max(grid_for(g.n, 256), 1)), dim3(256), 0, s,
                           g.n, act, (uint8_t)0, nullptr, nullptr, nxt, 0, nullptr);
        a.next_active = nxt;
        TailArgs t{};
        t.n = g.n;
        t.rounds = rounds;
        t.seed = seed;
        r = run_tail(a, t, s, &filter);
        if (r >= rounds) return;
        start = nullptr;  // (r > 0: the tail starts from every node)
        build_lists(mode, g, seed, s, nullptr, 1);
        std::swap(act, nxt);  // round r's frontier (r > 0)
    }
    a.inc = inc_.p;
    a.top = top_.p;
    a.out = out_.p;
    a.dtop = dtop_.p;
    a.prop_t = prop_t_.p;
    a.prop_gain = prop_gain_.p;
    a.prop_ok = prop_ok_.p;
    // Refinement hubs of more than one chunk keep per-block connection counters across the
    // rounds: one scan builds them, every applied move updates its hub neighbours' counters, and
    // the hubs then decide from the counters instead of rescanning their edges each round.
    const bool incremental = !cl && dense_hub_ && dense_total_ > 0;
    a.hub_slot = incremental ? hub_slot_.p : nullptr;
    a.hub_cnt = incremental ? dense_cnt_.p : nullptr;
    const std::string base = std::string(phase ? phase : (cl ? "lp_cluster" : "lp_refine"));
    if (incremental) {
        ProfScope ps(prof, base + "_hub_counters", 0.0, 0, s);
        fill_async(dense_cnt_.p, dense_total_, 0, s);
        const int copies = std::min(kHubDenseThreads / 64, kHubDenseSlots / num_labels_);
        const size_t lds = sizeof(int) * (size_t)copies * num_labels_;
        for (int sr = 0; sr < S; ++sr) {
            if (hub_multi_n_[sr] == 0) continue;
            hipLaunchKernelGGL(propose_hub_dense_chunk, dim3(hub_chunks_[sr]), dim3(kHubDenseThreads), lds, s, a, cmap_.p + cmap_base_[sr], num_labels_, dense_off_.p + hub_base_[sr], dense_cnt_.p, 1, 0);
        }
    }
    const int nl = num_labels_;
    // every refinement hub decides from kept counters: those decisions join the frontier launch
    const bool fused_hubs = incremental && dense_all_;
    const int nseg = S * kNumBins;
    const int listed = host_offsets[nseg - 1] + host_counts[nseg - 1];
    int hubs = 0;
    for (int sr = 0; sr < S; ++sr) hubs += host_counts[sr * kNumBins + kNumBins - 1];
    // the compaction consumes the frontier flags unless hub kernels of the round read them
    const bool keep_flags = hubs > 0 && !fused_hubs;
    if (!cl) {
        if (listed == 0) return;
        const int nf = r == 0 ? g.n : 0;  // else flagged by the tail
        hipLaunchKernelGGL(init_frontier, dim3(grid_for(std::max(nf, 2 * nseg), 256)), dim3(256),
                           0, s, nf, act, (uint8_t)(keep_flags ? 1 : 0), map, start, nxt, 2 * nseg, ccount_.p);
    }
    bool settle = cl && hubs == 0 && S > 1 && rounds > kSettleRound + 1 && g.m2 > kSettleEdges;
    if (settle) {
        whole_rounds_ = kSettleRound + 1;
        active_.reserve(g.n);
        clists_.reserve(g.n);
        ccount_.reserve(rounds * nseg);  // list lengths per round
        fill_async(ccount_.p, rounds * nseg, 0, s);
        act = active_.p;
    }
    // admission and application in one launch; the label weights change places each sub-round
    // (run_copies() runs single rounds one after the other on one preparation's scratch)
    const bool turn = cl && !settle && rounds > 1 && g.n <= kTurnNodes;
    int* turn_size = nullptr;
    int* turn_inc = nullptr;
    unsigned long long* turn_top = nullptr;
    if (turn) {
        turn_size = size2_.reserve(g.n);
        turn_inc = inc2_.reserve(g.n);
        turn_top = top2_.reserve(g.n);
    }
    int* cnow = ccount_.p;  // list lengths of the frontier, cleared by the tail before last
    int* cnext = cnow + nseg;
    if (!cl && hubs > 0) a.big = big_.reserve(g.m2 / kLongRow + 1);
    while (r < rounds) {
        // refinement: round 0 works on the whole lists (or, sub-round by sub-round, on the nodes
        // that may have a candidate by then, if a start set is given), later rounds on the
        // compacted frontier
        const bool from_start = r == 0 && start;
        const int* flists = from_start ? clists_.p : lists_.p;
        const int* fcount = from_start ? cnow : counts_;
        if (!cl && r > 0) {
            ProfScope ps(prof, base + "_frontier", 0.0, 0, s);
            std::swap(cnow, cnext);
            hipLaunchKernelGGL(compact_active, dim3(grid_for(listed, 256 * kCompactItems)), dim3(256), 0, s,
                               lists_.p, offsets_.p, nseg, 0, listed, act, keep_flags ? 0 : 1, nullptr, cnow, clists_.p);
            a.next_active = nxt;
            TailArgs t{};
            t.clists = clists_.p;
            t.offsets = offsets_.p;
            t.ccount = cnow;
            t.cnext = cnext;
            t.nseg = nseg;
            t.n = g.n;
            t.round = r;
            t.rounds = rounds;
            t.seed = seed;
            t.hubs = hubs;
            const int next = run_tail(a, t, s, &filter);
            if (next != r) {
                r = next;
                std::swap(act, nxt);
                continue;
            }
            flists = clists_.p;
            fcount = cnow;
        }
        a.tie_seed = tie_seed_of(seed, r);
        a.moves = ctl_.p + kCtlMoves + r;
        a.active = cl ? nullptr : act;
        a.next_active = cl ? nullptr : nxt;
        int sr0 = 0;  // sub-rounds run with flags
        if (settle && r >= kSettleRound) {
            ProfScope ps(prof, base + "_settled", 0.0, 0, s);
            a.next_active = act;
            bool asked = r > kSettleRound;
            for (; sr0 < S && settle; ++sr0) {
                int* dcount = ccount_.p + r * nseg + sr0 * kNumBins;
                if (!settled_subround(a, sr0, r == kSettleRound ? nullptr : dcount, s, prof, base) || asked) continue;
                asked = true;
                settle = few_unsettled(act, sr0, dcount, s);
            }
            if (settle) {
                ++r;
                continue;
            }
            whole_rounds_ = rounds;
            a.next_active = nullptr;
        }
        for (int sr = sr0; sr < S; ++sr) {
            int sub_total = 0;
            if (!cl) {
                if (from_start) {
                    // right before the sub-round: a node outside the start set has a candidate
                    // once a neighbour has moved in an earlier sub-round of this round
                    const int l0 = sr * kNumBins;
                    int total = 0;
                    for (int b = 0; b < kNumBins; ++b) total += host_counts[l0 + b];
                    if (total == 0) continue;
                    hipLaunchKernelGGL(compact_active, dim3(grid_for(total, 256 * kCompactItems)), dim3(256), 0, s,
                                       lists_.p, offsets_.p + l0, kNumBins, host_offsets[l0], total, act, 1, nxt, cnow + l0, clists_.p);
                }
                if (a.big) a.n_big = ctl_.p + kCtlLong + (r * S + sr);
                // refinement: the five degree lists' proposals in one launch over the frontier,
                // and the hubs' decisions from their kept counters when every hub has them
                FrontierLists F{};
                int listed_sr = 0;
                for (int b = 0; b < kNumBins; ++b) {
                    const int l = sr * kNumBins + b;
                    const bool take = b < kNumBins - 1 || fused_hubs;
                    F.list[b] = flists + host_offsets[l];
                    F.base[b] = host_offsets[l];
                    F.dcount[b] = take ? fcount + l : nullptr;
                    listed_sr += take ? host_counts[l] : 0;
                }
                if (listed_sr > 0)
                    launch_frontier(bins_.group_items, dense_wave_, a, F, nl, listed_sr, s);
            } else {
                long long ledges = 0, lnodes = 0;
                for (int b = 0; b < kNumBins - 1; ++b) {
                    ledges += host_edges[sr * kNumBins + b];
                    lnodes += host_counts[sr * kNumBins + b];
                }
                // algorithmic bytes: 12 B per traversed edge (target, weight, label gather) and
                // 16 B per node (two offsets, weight, own label); label weights are O(moved).
                ProfScope ps(prof, base + "_propose_lists", 12.0 * (double)ledges + 16.0 * (double)lnodes, ledges, s);
                for (int b = 0; b < kNumBins; ++b) sub_total += host_counts[sr * kNumBins + b];
                if (sub_total == 0) continue;
                const Turnover T{turn ? g.n : 0, turn_size, turn_inc, turn_top};
                launch_lists(a, sr, 1, nullptr, false, T, s);
            }
            const int cnt = host_counts[sr * kNumBins + kNumBins - 1];
            if (!cl)
                for (int b = 0; b < kNumBins; ++b) sub_total += host_counts[sr * kNumBins + b];
            if (cnt > 0 && !fused_hubs) propose_hubs(mode, a, r, sr, incremental, s, prof, base);
            if (sub_total == 0) continue;
            const int gm = grid_for(sub_total, 256);
            const int* sub_list = lists_.p + host_offsets[sr * kNumBins];  // bins are contiguous
            ProfScope ps(prof, base + "_admit_apply", 0.0, 0, s);
            if (turn) {
                a.base = host_offsets[sr * kNumBins];
                hipLaunchKernelGGL(admit_apply, dim3(std::min(grid_for(sub_total, kApplyThreads), kApplyGrid)), dim3(kApplyThreads), 0, s, a, turn_size, sub_list, sub_total);
                std::swap(a.size, turn_size);
                std::swap(a.inc, turn_inc);
                std::swap(a.top, turn_top);
            } else if (cl) {
                a.base = host_offsets[sr * kNumBins];
                hipLaunchKernelGGL(admit_moves, dim3(gm), dim3(256), 0, s, a, sub_list, sub_total);
                hipLaunchKernelGGL(apply_moves, dim3(std::min(grid_for(sub_total, kApplyThreads), kApplyGrid)), dim3(kApplyThreads), 0, s, a, sub_list, sub_total);
            } else {
                SubLists L{};
                for (int b = 0; b < kNumBins; ++b) {
                    const int l = sr * kNumBins + b;
                    // every list's compacted frontier; hubs whose kernels work on the whole list
                    // have their proposals at its positions
                    const bool whole = b == kNumBins - 1 && !fused_hubs;
                    L.list[b] = (whole ? lists_.p : flists) + host_offsets[l];
                    L.dcount[b] = (whole ? counts_ : fcount) + l;
                    L.base[b] = host_offsets[l];
                }
                const int gs = std::min(gm, 1024);
                if (filter) hipLaunchKernelGGL(filter_departures_sub, dim3(gs), dim3(256), 0, s, a, L);
                hipLaunchKernelGGL(admit_moves_sub, dim3(gs), dim3(256), 0, s, a, L);
                hipLaunchKernelGGL(apply_moves_sub<LpMode::Refine>, dim3(gs), dim3(kBlock), 0, s, a, L);
            }
        }
        if (!cl) {
            std::swap(act, nxt);
            if (keep_flags) fill_async(nxt, g.n, (uint8_t)0, s);
        }
        ++r;
    }
    if (a.size != size)  // an odd number of turnovers
        hipLaunchKernelGGL(copy_i32, dim3(grid_for(g.n, 256)), dim3(256), 0, s, size, a.size, g.n);
    KH_CHECK(hipGetLastError());
}

// The proposals of sub-round sr's hub list.
void LpWorkspace::propose_hubs(LpMode mode, LpArgs a, int r, int sr, bool incremental, hipStream_t s,
                               Profiler* prof, const std::string& base) {
    const bool cl = mode == LpMode::Cluster;
    const int S = subrounds_, nl = num_labels_;
    const int l = sr * kNumBins + kNumBins - 1;
    const int* lst = lists_.p + host_offsets[l];
    a.base = host_offsets[l];
    // (the list's mid-size hubs are timed in a scope of their own)
    const long long ledges = host_edges[l] - mid_edges_[sr];
    const int lnodes = host_counts[l] - mid_n_[sr];
    const double bytes = cl ? 12.0 * (double)ledges + 16.0 * lnodes : 0.0;
    ProfScope ps(prof, base + "_propose_hub", bytes, cl ? ledges : 0, s);
    if (!cl && dense_hub_) {
        const int4* cm = cmap_.p + cmap_base_[sr];
        const int* dof = dense_off_.p + hub_base_[sr];
        const int copies = std::min(kHubDenseThreads / 64, kHubDenseSlots / nl);
        const size_t lds = sizeof(int) * (size_t)copies * nl;
        if (!(incremental && dense_all_))  // otherwise every hub decides from counters
            hipLaunchKernelGGL(propose_hub_dense_chunk, dim3(hub_chunks_[sr]), dim3(kHubDenseThreads), lds, s, a, cm, nl, dof, dense_cnt_.p, 0, incremental ? 1 : 0);
        ps.close();
        if (hub_multi_n_[sr] > 0) {
            ProfScope pf(prof, base + "_propose_hub_merge", 0.0, hub_multi_n_[sr], s);
            hipLaunchKernelGGL(hub_dense_decide, dim3(hub_multi_n_[sr]), dim3(256), 0, s, a, lst, multi_.p + multi_base_[sr], hub_multi_n_[sr], nl, dof, dense_cnt_.p, incremental ? 1 : 0);
        }
        return;
    }
    const int4* cm = cmap_.p + cmap_base_[sr];
    const long long* to = tab_off_.p + hub_base_[sr];
    const long long* ob = offm_base_.p + hub_base_[sr];
    const int* ctb = ct_base_.p + hub_base_[sr];
    if (hub_chunks_[sr] > 0) {
        if (cl) hipLaunchKernelGGL((propose_hub_chunk<LpMode::Cluster, kHubThreads, kHubChunk>), dim3(hub_chunks_[sr]), dim3(kHubThreads), 0, s, a, cm, partials_.p, ob, offm_.p, ctb, cnt_t_.p);
        else hipLaunchKernelGGL((propose_hub_chunk<LpMode::Refine, kHubThreads, kHubChunk>), dim3(hub_chunks_[sr]), dim3(kHubThreads), 0, s, a, cm, partials_.p, ob, offm_.p, ctb, cnt_t_.p);
    }
    ps.close();  // the hub scope times the chunked kernel alone
    if (mid_n_[sr] > 0) {
        const double mb = cl ? 12.0 * (double)mid_edges_[sr] + 16.0 * mid_n_[sr] : 0.0;
        ProfScope pm(prof, base + "_propose_hub_mid", mb, cl ? mid_edges_[sr] : 0, s);
        const int4* mm = mmap_.p + mid_base_[sr];
        if (cl) hipLaunchKernelGGL((propose_hub_chunk<LpMode::Cluster, kMidThreads, kMidChunk>), dim3(mid_n_[sr]), dim3(kMidThreads), 0, s, a, mm, partials_.p, ob, offm_.p, ctb, cnt_t_.p);
        else hipLaunchKernelGGL((propose_hub_chunk<LpMode::Refine, kMidThreads, kMidChunk>), dim3(mid_n_[sr]), dim3(kMidThreads), 0, s, a, mm, partials_.p, ob, offm_.p, ctb, cnt_t_.p);
    }
    if (hub_multi_n_[sr] > 0) {
        ProfScope pf(prof, base + "_propose_hub_merge", 0.0, hub_tasks_[sr], s);
        const int* ml = multi_.p + multi_base_[sr];
        const int* tp = task_prefix_.p + task_base_[sr];
        const int4* tm = tmap_.p + tmap_base_[sr];
        const int2* tsb = tsub_.p + tmap_base_[sr];
        const int nm = hub_multi_n_[sr];
        Cand* br = reinterpret_cast<Cand*>(bres_.p);
        const int nt = hub_tasks_[sr];
        if (hub_wide_[sr]) {
            // bucket-major positions, relative to this sub-round's block of counts
            size_t sb = scan_tmp_bytes_;
            KH_CHECK(rocprim::exclusive_scan(scan_tmp_.p, sb, cnt_t_.p + ct_sr_base_[sr], pos_t_.p + ct_sr_base_[sr], 0, (size_t)ct_sr_size_[sr] + 1, rocprim::plus<int>(), s));
        }
        const int* cp = chunk_prefix_.p + chunk_base_[sr];
        const bool tiny = nt > kTinyTasks;
        int* mid = tiny ? mid_tasks_.p : nullptr;
        int* queue = hub_capped_[sr] ? big_tasks_.p : nullptr;
        int* n_mid = ctl_.p + kCtlMid + (r * S + sr);
        int* queued = ctl_.p + kCtlBig + (r * S + sr);
        const auto merge = [&](auto kernel, int grid, int threads, const int* in_q, const int* in_n, int* out_q, int* out_n) {
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, s, a, nt, tm, tsb, cnt_t_.p, pos_t_.p, cp, ob, offm_.p, partials_.p, to, hub_key_.p, hub_val_.p, br, bown_.p, fb_.p, in_q, in_n, out_q, out_n);
        };
        const auto merges = [&](auto k0, auto k1, auto k2) {
            if (tiny) merge(k0, nt, kTinyThreads, nullptr, nullptr, mid, n_mid);
            merge(k1, tiny ? kSmallGrid : nt, kSmallThreads, mid, n_mid, queue, queued);
            if (queue) merge(k2, std::min(nt, 256), kFinThreads, queue, queued, nullptr, nullptr);
        };
        const auto decide = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(nm), dim3(256), 0, s, a, lst, ml, nm, tp, to, hub_key_.p, hub_val_.p, br, bown_.p, fb_.p);
        };
        if (cl) {
            merges(hub_bucket_merge<LpMode::Cluster, 0>, hub_bucket_merge<LpMode::Cluster, 1>, hub_bucket_merge<LpMode::Cluster, 2>);
            decide(hub_decide<LpMode::Cluster>);
        } else {
            merges(hub_bucket_merge<LpMode::Refine, 0>, hub_bucket_merge<LpMode::Refine, 1>, hub_bucket_merge<LpMode::Refine, 2>);
            decide(hub_decide<LpMode::Refine>);
        }
    }
}

void LpWorkspace::run_copies(const DGraph& g, int* label, int* size, int bound,
                             const uint32_t* seeds, int copies, hipStream_t s) {
    if (g.n == 0) return;
    hipLaunchKernelGGL(init_labels, dim3(grid_for(g.n, 256), copies), dim3(256), 0, s, g.n, label,
                       size, g.vwgt);
    if (host_counts[kNumBins - 1] > 0) {  // the hub kernels take one clustering at a time
        for (int i = 0; i < copies; ++i)
            run(LpMode::Cluster, g, label + (long long)i * g.n, size + (long long)i * g.n, bound, 1,
                seeds[i], s, nullptr, "rating_sweep");
        return;
    }
    fetched_ = false;
    LpArgs a{};
    a.xadj = g.xadj;
    a.adjncy = g.adjncy;
    a.adjwgt = g.adjwgt;
    a.vwgt = g.vwgt;
    a.label = label;
    a.size = size;
    a.bound = bound;
    a.wave_small = bins_.wave_small;
    a.inc = inc_.p;
    a.top = top_.p;
    a.prop_t = prop_t_.p;
    a.prop_gain = prop_gain_.p;
    a.prop_ok = prop_ok_.p;
    a.moves = ctl_.p + kCtlMoves;
    a.err = ctl_.p + kCtlErr;
    a.copy_stride = g.n;
    static_assert(kMaxCopies == 3, "one tie seed per copy");
    a.tie_seed = tie_seed_of(seeds[0], 0);
    if (copies > 1) a.copy_tie1 = tie_seed_of(seeds[1], 0);
    if (copies > 2) a.copy_tie2 = tie_seed_of(seeds[2], 0);
    int total = 0;
    for (int b = 0; b < kNumBins - 1; ++b) total += host_counts[b];
    if (total == 0) return;
    launch_lists(a, 0, copies, nullptr, false, Turnover{}, s);
    const dim3 grid(grid_for(total, 256), copies);
    hipLaunchKernelGGL(admit_moves, grid, dim3(256), 0, s, a, lists_.p, total);
    hipLaunchKernelGGL(apply_moves, dim3(std::min(grid_for(total, kApplyThreads), kApplyGrid), copies),
                       dim3(kApplyThreads), 0, s, a, lists_.p, total);
    KH_CHECK(hipGetLastError());
}

// The clustering proposals of sub-round sr's lists (not the hub list); dcount: compacted to these
// lengths; settle: also flag the nodes that are not settled.
void LpWorkspace::launch_lists(const LpArgs& a, int sr, int copies, const int* dcount, bool settle,
                               const Turnover& T, hipStream_t s) {
    ClusterLists F{};
    F.dcount = dcount;
    const int items = bins_.group_items;
    int blocks = 0;
    for (int b = 0; b < kNumBins - 1; ++b) {
        const int l = sr * kNumBins + b;
        F.list[b] = (dcount ? clists_.p : lists_.p) + host_offsets[l];
        F.base[b] = host_offsets[l];
        F.count[b] = host_counts[l];
        const int per = b < 2 ? items * (kBlock / 8) : b < 4 ? items * (kBlock / 16) : kBlock / 64;
        blocks += grid_for(host_counts[l], per);
    }
    blocks += grid_for(T.n, kBlock * kTurnItems);
    if (blocks == 0) return;
    const dim3 grid(dcount ? std::min(blocks, kFrontierGrid) : blocks, copies);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, s, a, F, T);
    };
    const bool waves = F.count[kNumBins - 2] > 0;
    switch (items * 4 + (waves ? 1 : 0) + (settle ? 2 : 0)) {
        case 4: launch(propose_lists<1, false, false>); break;
        case 5: launch(propose_lists<1, true, false>); break;
        case 6: launch(propose_lists<1, false, true>); break;
        case 7: launch(propose_lists<1, true, true>); break;
        case 16: launch(propose_lists<4, false, false>); break;
        case 17: launch(propose_lists<4, true, false>); break;
        case 18: launch(propose_lists<4, false, true>); break;
        case 19: launch(propose_lists<4, true, true>); break;
        case 9: launch(propose_lists<2, true, false>); break;
        case 10: launch(propose_lists<2, false, true>); break;
        case 11: launch(propose_lists<2, true, true>); break;
        default: launch(propose_lists<2, false, false>);
    }
}

// Sub-round sr of a clustering from round kSettleRound on: over the whole lists (dcount nullptr)
// or over their nodes that are not settled (dcount: their lengths, zero on entry). False if it has
// no nodes.
bool LpWorkspace::settled_subround(const LpArgs& a, int sr, int* dcount, hipStream_t s,
                                   Profiler* prof, const std::string& base) {
    const int l0 = sr * kNumBins;
    int total = 0;
    long long edges = 0;  // of the whole lists
    for (int b = 0; b < kNumBins; ++b) {
        total += host_counts[l0 + b];
        edges += host_edges[l0 + b];
    }
    if (total == 0) return false;
    if (dcount)
        hipLaunchKernelGGL(compact_active, dim3(grid_for(total, 256 * kCompactItems)), dim3(256), 0,
                           s, lists_.p, offsets_.p + l0, kNumBins, host_offsets[l0], total,
                           a.next_active, 1, nullptr, dcount, clists_.p);
    {
        ProfScope ps(prof, base + "_propose_settled", dcount ? 0.0 : 12.0 * (double)edges + 16.0 * total,
                     dcount ? 0 : edges, s);
        if (dcount && settled_rec_ < 0) settled_rec_ = ps.idx;  // (booked by book_edges())
        launch_lists(a, sr, 1, dcount, true, Turnover{}, s);
    }
    SubLists L{};
    for (int b = 0; b < kNumBins; ++b) {
        L.list[b] = (dcount ? clists_.p : lists_.p) + host_offsets[l0 + b];
        L.base[b] = host_offsets[l0 + b];
        L.dcount[b] = (dcount ? dcount : counts_ + l0) + b;
    }
    const int gs = std::min(grid_for(total, 256), 1024);
    hipLaunchKernelGGL(admit_moves_sub, dim3(gs), dim3(256), 0, s, a, L);
    hipLaunchKernelGGL(apply_moves_sub<LpMode::Cluster>, dim3(gs), dim3(kBlock), 0, s, a, L);
    return true;
}

// Whether the nodes of sub-round sr that are not settled hold few of its lists' edges. count:
// kNumBins counters, zero on entry.
bool LpWorkspace::few_unsettled(uint8_t* flags, int sr, int* count, hipStream_t s) {
    const int l0 = sr * kNumBins;
    int total = 0;
    for (int b = 0; b < kNumBins; ++b) total += host_counts[l0 + b];
    hipLaunchKernelGGL(compact_active, dim3(grid_for(total, 256 * kCompactItems)), dim3(256), 0, s,
                       lists_.p, offsets_.p + l0, kNumBins, host_offsets[l0], total, flags, 0,
                       nullptr, count, clists_.p);
    mail_.post(s, {count, kNumBins});
    const int* left = mail_.wait(s);
    double edges = 0.0, read = 0.0;
    for (int b = 0; b < kNumBins; ++b) {
        const int l = l0 + b;
        edges += (double)host_edges[l];
        if (host_counts[l] > 0) read += (double)host_edges[l] * left[b] / host_counts[l];
    }
    return read <= kSettleShare * edges;
}

// Launches refine_tail and waits for its answer: the round to go on with, and whether a block is
// overloaded.
int LpWorkspace::run_tail(const LpArgs& a, TailArgs& t, hipStream_t s, bool* overloaded) {
    t.num_labels = num_labels_;
    t.S = subrounds_;
    t.max_nodes = tail_nodes(subrounds_);
    t.max_edges = tail_edges(subrounds_);
    t.moves = ctl_.p + kCtlMoves;
    t.state = mail_.box();
    t.seq = mail_.next();
    hipLaunchKernelGGL(refine_tail, dim3(1), dim3(kTailThreads), 0, s, a, t);
    KH_CHECK(hipGetLastError());
    const int* answer = mail_.wait(s);
    *overloaded = answer[1] != 0;
    return answer[0];
}

void LpWorkspace::fetch(hipStream_t s) {
    if (fetched_) return;
    mail_.post(s, {ctl_.p, kCtlBig}, {ctl_.p + kCtlErr, 1});
    std::memcpy(host_ctl_, mail_.wait(s), sizeof(host_ctl_));
    fetched_ = true;
}

void LpWorkspace::read_moves(int rounds, int* out, hipStream_t s) {
    fetch(s);
    std::memcpy(out, host_ctl_ + kCtlMoves, sizeof(int) * std::max(rounds, 0));
}

void LpWorkspace::check(hipStream_t s) {
    keep_err_ = false;
    fetch(s);
    KH_REQUIRE(host_ctl_[kCtlBig] == 0,
               "label propagation: a hash table probe found no free slot (kernel table "
               "sizing invariant violated); the result is invalid");
}

long long LpWorkspace::traversed(hipStream_t s) {
    fetch(s);
    unsigned long long h[64];
    std::memcpy(h, host_ctl_, sizeof(h));
    long long t = 0;
    for (int i = 0; i < 64; ++i) t += (long long)h[i];
    return t;
}

long long LpWorkspace::book_edges(hipStream_t s, Profiler* prof) {
    const long long compacted = traversed(s);
    if (prof && settled_rec_ >= 0) {
        prof->recs[settled_rec_].edges = compacted;
        prof->recs[settled_rec_].bytes = 12.0 * (double)compacted;
    }
    long long edges = 0;
    for (int l = 0; l < subrounds_ * kNumBins; ++l) edges += host_edges[l];
    return edges * whole_rounds_ + compacted;
}

void LpWorkspace::border(const DGraph& g, const int* part, uint8_t* flags, hipStream_t s) {
    if (g.n > 0)
        hipLaunchKernelGGL(border_nodes, dim3(grid_for(g.n, 256)), dim3(256), 0, s, g.n, g.xadj,
                           g.adjncy, part, flags);
    KH_CHECK(hipGetLastError());
}

bool LpWorkspace::takes_start() const {
    if (small_) return false;
    int listed = 0;
    for (int l = 0; l < subrounds_ * kNumBins; ++l) {
        if (l % kNumBins == kNumBins - 1 && host_counts[l] > 0) return false;
        listed += host_counts[l];
    }
    return listed > kStartNodes;
}

void LpWorkspace::init_cluster_labels(const DGraph& g, int* label, int* size, hipStream_t s) {
    if (g.n > 0)
        hipLaunchKernelGGL(init_labels, dim3(grid_for(g.n, 256)), dim3(256), 0, s, g.n, label,
                           size, g.vwgt);
}

void compute_block_weights(const DGraph& g, const int* part, int k, int* W, hipStream_t s) {
    KH_REQUIRE(k >= 1, "k must be >= 1");
    fill_async(W, k, 0, s);
    if (g.n == 0) return;
    if (k > 8192) {  // per-workgroup LDS histograms only up to 32 KiB
        hipLaunchKernelGGL(block_weights_global, dim3(grid_for(g.n, 256)), dim3(256), 0, s, g.n,
                           part, g.vwgt, W);
        return;
    }
    const int grid = std::min(grid_for(g.n, 256), 2048);
    hipLaunchKernelGGL(block_weights_kernel, dim3(grid), dim3(256), sizeof(int) * k, s, g.n,
                       part, g.vwgt, k, W);
}

}  // namespace kahip
