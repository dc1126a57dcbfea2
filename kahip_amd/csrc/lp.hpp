// Host interface of the synchronous LP kernels (clustering and refinement).
#pragma once

#include "common.hpp"
#include "devbuf.hpp"
#include "mail.hpp"

namespace kahip {

constexpr int kMaxSub = 8;
constexpr int kMaxRounds = 64;
constexpr int kMaxCopies = 3;  // clusterings of run_copies()

// Kernel arguments shared by the propose / filter / admit / apply launches of one sub-round.
struct LpArgs {
    const int* xadj;
    const int* adjncy;
    const int* adjwgt;
    const int* vwgt;
    int* label;        // label of each node (cluster id or block id)
    int* size;         // weight of each label
    int bound;         // admission bound: size + w < bound
    const int* lbound; // per-label bounds (a disjoint union of graphs), nullptr: `bound` for all
    int wave_small;    // one-wave nodes up to this degree: half the edges per lane
    uint32_t tie_seed;
    const uint8_t* active;  // refinement frontier (nullptr for clustering)
    uint8_t* next_active;  // clustering: nodes that are not settled
    int* inc;                  // per label: summed weight of proposals into it
    unsigned long long* top;   // per label: top proposal priority into it
    int* out;                  // per label: summed weight of departures (refinement)
    unsigned long long* dtop;  // per label: top departure priority (refinement)
    int base;                  // list position of the launch's first list entry
    int* prop_t;               // per list position: proposed label, -1 outside propose..apply
    int* prop_gain;
    uint8_t* prop_ok;
    int* moves;
    unsigned long long* trav;  // refinement: traversed directed edges, 64 spread counters
    // Refinement with incremental hub counters (nullptr otherwise): hub_slot[v] is the offset of
    // node v's per-block connection counters in hub_cnt, or -1; moves update the counters of
    // their hub neighbours.
    const int* hub_slot;
    int* hub_cnt;
    // Refinement of a graph with hubs (nullptr otherwise): admitted moves of rows of more than
    // kLongRow edges, {first edge, edges, old label, new label}, and their number (zero on entry).
    int4* big;
    int* n_big;
    int* err;  // device error flag (kErrProbe), cleared by prepare(), read by check()
    // Independent clusterings of one graph in one launch (gridDim.y of them): clustering y has its
    // arrays y * copy_stride further on and the tie seed tie_seed, copy_tie1, copy_tie2 (not an
    // array: indexing a kernel argument by y would put all of them in scratch memory).
    long long copy_stride;
    uint32_t copy_tie1, copy_tie2;
};

// Arguments of refine_tail beyond LpArgs.
struct TailArgs {
    const int* clists;   // round `round`'s frontier, compacted per list; nullptr: every node
    const int* offsets;  // list offsets
    const int* ccount;   // list lengths
    int* cnext;          // cleared for the next compaction (nseg entries)
    int nseg, n, num_labels, S, round, rounds;
    uint32_t seed;
    int max_nodes, max_edges;  // of a frontier that it takes
    int hubs;            // nodes of more than the wave bin's degree exist: never run here
    int* moves;          // per round
    int* state;          // mail: {number, next round, overloaded block exists}
    int seq;
};

// Arrays of the next clustering sub-round that a proposal launch makes ready.
struct Turnover {
    int n = 0;  // labels; 0: none
    int* size = nullptr;
    int* inc = nullptr;
    unsigned long long* top = nullptr;
};

class LpWorkspace {
public:
    // Bins the nodes of g into per-(sub-round, degree bin) lists and sizes the scratch for
    // num_labels labels. One small host readback.
    // Nodes with include[v] == 0 (include may be null) are left out: they never propose.
    // copies > 1: for run_copies().
    void prepare(LpMode mode, const DGraph& g, int num_labels, int subrounds, uint32_t seed,
                 const BinConfig& bins, hipStream_t s, const uint8_t* include = nullptr,
                 int copies = 1);
    // One round of `copies` clusterings from single nodes that differ in the seed (and so in the
    // tie-breaking; the sub-rounds are prepare()'s, one): label receives copies x n labels, size
    // (scratch) their weights.
    void run_copies(const DGraph& g, int* label, int* size, int bound, const uint32_t* seeds,
                    int copies, hipStream_t s);
    // Runs `rounds` synchronous rounds. label/size are device arrays (node -> label,
    // label -> weight). Refinement starts from an all-active frontier.
    // lbound (optional): the bound of each label, replacing `bound`.
    // start (optional): the first round starts from the nodes v with start[map[v]] set; the others
    // must have no neighbour in another block, so that they have no candidate until a neighbour
    // moves, and enter the round's later sub-rounds when one does. Same result as from all nodes.
    void run(LpMode mode, const DGraph& g, int* label, int* size, int bound, int rounds,
             uint32_t seed, hipStream_t s, Profiler* prof, const char* phase,
             const int* lbound = nullptr, const int* map = nullptr,
             const uint8_t* start = nullptr);
    // flags[v] = 1 if v may have a neighbour in another block, else 0
    static void border(const DGraph& g, const int* part, uint8_t* flags, hipStream_t s);
    // Whether `start` is of use on the graph of the last prepare(): it is large, has no hubs and is
    // not refined by one workgroup from its first round on.
    bool takes_start() const;
    // label[v] = v, size[v] = vwgt[v]
    static void init_cluster_labels(const DGraph& g, int* label, int* size, hipStream_t s);
    // Moves per round of the last run (waits for it).
    void read_moves(int rounds, int* out, hipStream_t s);
    // Directed edges read by the last refinement run (waits for it): the rows scanned
    // by the proposal kernels (hubs deciding from their kept counters read none) and the rows of
    // moved nodes scanned to mark their neighbours and update hub counters. Clustering: the rows
    // of the rounds that skip settled nodes.
    long long traversed(hipStream_t s);
    // Directed edges read by the proposals of the last clustering run (waits for it); books those
    // of the rounds that skip settled nodes on their first profile record.
    long long book_edges(hipStream_t s, Profiler* prof);
    // Rounds of the last clustering run that looked at every listed node.
    int whole_rounds() const { return whole_rounds_; }
    // Throws if a kernel of a run() since the last prepare() set the device error flag (waits for
    // the last run).
    void check(hipStream_t s);
    // Leaves that to the next check(): the next prepare() keeps the flag.
    void check_later() { keep_err_ = true; }

    int host_counts[kMaxSub * kNumBins] = {};
    long long host_edges[kMaxSub * kNumBins] = {};
    int host_offsets[kMaxSub * kNumBins] = {};

private:
    void build_lists(LpMode mode, const DGraph& g, uint32_t seed, hipStream_t s,
                     const uint8_t* include, int copies);
    void launch_lists(const LpArgs& a, int sr, int copies, const int* dcount, bool settle,
                      const Turnover& T, hipStream_t s);
    bool settled_subround(const LpArgs& a, int sr, int* dcount, hipStream_t s, Profiler* prof,
                          const std::string& base);
    bool few_unsettled(uint8_t* flags, int sr, int* count, hipStream_t s);
    void propose_hubs(LpMode mode, LpArgs a, int r, int sr, bool incremental, hipStream_t s,
                      Profiler* prof, const std::string& base);
    int run_tail(const LpArgs& a, TailArgs& t, hipStream_t s, bool* overloaded);
    void fetch(hipStream_t s);  // host_ctl_ of the last run
    Mail mail_;
    // Counters of a run: {traversed edges in 64 spread 64-bit counters, moves per round, lengths
    // of the hub merges' big and mid-size task queues and of the long moved rows per sub-round,
    // error flag}
    static constexpr int kCtlMoves = 128, kCtlBig = kCtlMoves + kMaxRounds,
                         kCtlMid = kCtlBig + kMaxSub * kMaxRounds,
                         kCtlLong = kCtlMid + kMaxSub * kMaxRounds,
                         kCtlErr = kCtlLong + kMaxSub * kMaxRounds, kCtlInts = kCtlErr + 1;
    DevBuf<int> ctl_;
    int host_ctl_[kCtlBig + 1] = {};  // the traversed edges, the moves, the error flag
    bool fetched_ = false;
    int whole_rounds_ = 0;
    int settled_rec_ = -1;  // profile record of the first proposals over compacted lists
    bool keep_err_ = false, clear_err_ = false;
    bool small_ = false;  // refinement that starts in refine_tail, without lists
    void build_chunk_maps(hipStream_t s);  // cmap_ of every sub-round (after chunk_prefix_)
    int subrounds_ = 1;
    int num_labels_ = 0;
    BinConfig bins_;  // degree bins and tile shapes of the last prepare()
    bool dense_wave_ = false, dense_hub_ = false;
    // per sub-round hub bookkeeping (hub list = last degree bin)
    int hub_n_[kMaxSub] = {};
    int hub_chunks_[kMaxSub] = {};
    int hub_multi_n_[kMaxSub] = {};
    int hub_base_[kMaxSub] = {};    // offset into tab_off_/tab_cap_ (list order)
    int chunk_base_[kMaxSub] = {};  // offset into chunk_prefix_
    int cmap_base_[kMaxSub] = {};   // offset into cmap_ (chunks of the earlier sub-rounds)
    int tmap_base_[kMaxSub] = {};   // offset into tmap_ (tasks of the earlier sub-rounds)
    int mid_n_[kMaxSub] = {};       // hubs of the mid-size kernel per sub-round
    int mid_base_[kMaxSub] = {};    // offset into mmap_
    long long mid_edges_[kMaxSub] = {};  // edges of those hubs
    int multi_base_[kMaxSub] = {};  // offset into multi_
    int task_base_[kMaxSub] = {};   // offset into task_prefix_
    int hub_tasks_[kMaxSub] = {};   // (hub, bucket) tasks per sub-round
    int ct_sr_base_[kMaxSub] = {};  // bucket-major count block of each sub-round
    int ct_sr_size_[kMaxSub] = {};
    bool hub_wide_[kMaxSub] = {};    // a hub of more than kHubStage chunks: the counts are scanned
    bool hub_capped_[kMaxSub] = {};  // a hub at kMaxBuckets: large tasks go to the big merge
    size_t scan_tmp_bytes_ = 0;
    DevBuf<int> hub_deg_, chunk_prefix_, multi_;
    DevBuf<long long> tab_off_, tab_cap_;
    DevBuf<int2> partials_;
    DevBuf<int> ct_base_, cnt_t_, pos_t_;
    DevBuf<char> scan_tmp_;
    DevBuf<long long> offm_base_;
    DevBuf<int> offm_, task_prefix_, bown_, big_tasks_, mid_tasks_;
    DevBuf<int4> bres_, big_;
    DevBuf<int4> cmap_, tmap_, mmap_;  // hub-chunk, (hub, bucket) task, mid-size hub descriptors
    DevBuf<int> midpos_;
    DevBuf<int2> tsub_;  // (hub, bucket) task: {multi-chunk hub index, bucket | buckets << 16}
    DevBuf<uint8_t> fb_;
    DevBuf<int> lists_, bin_, bin_blocks_, offsets_;
    int* counts_ = nullptr;  // in bin_: list lengths
    DevBuf<int> clists_, ccount_;  // frontier (or nodes not settled) per list, compacted
    DevBuf<int> prop_t_, prop_gain_;
    DevBuf<uint8_t> prop_ok_;
    DevBuf<int> inc_, out_;
    DevBuf<unsigned long long> top_, dtop_;
    DevBuf<int> size2_, inc2_;  // of every other sub-round of a clustering with turnover
    DevBuf<unsigned long long> top2_;
    DevBuf<uint8_t> active_, next_active_;
    DevBuf<int> hub_key_, hub_val_;
    DevBuf<int> dense_off_, dense_cnt_;  // chunked dense refinement hubs: per-hub counters
    DevBuf<int> hub_slot_;
    long long dense_total_ = 0;
    bool dense_all_ = false;
    long long hub_total_ = 0;
};

void fill_async(int* p, long long n, int value, hipStream_t s);
void fill_async(unsigned long long* p, long long n, unsigned long long value, hipStream_t s);
void fill_async(uint8_t* p, long long n, uint8_t value, hipStream_t s);
void fill_async(long long* p, long long n, long long value, hipStream_t s);

// W[b] = sum of vwgt over nodes in block b (k <= 65536).
void compute_block_weights(const DGraph& g, const int* part, int k, int* W, hipStream_t s);

}  // namespace kahip
