// CPU initial partitioning of the coarsest graph: recursive multilevel bisection, after the
// reference's scheme (initial_partitioning.cpp:39-134 repeats
// initial_partition_bipartition.cpp:22-60, which runs graph_partitioner.cpp:110-238: bisect the
// block range [lb, ub] at floor((lb+ub)/2), extract both sides, recurse). Each bisection is
// multilevel: size-constrained LP coarsening (cluster bound ceil(max side / 12), as
// initial_partition_bipartition.cpp:39-43), BFS-grown starts (bipartition_tries of them, as
// bipartition.cpp:24-75) refined by 2-way FM, and FM at every uncoarsening level.
//
// The implementation is this library's own: sequential code, one independent RNG stream per
// (repetition, block range), so results do not depend on the number of threads used. Nodes of
// degree 0 do not affect the cut; they are left out of the bisections and packed into the
// lightest blocks at the end (heaviest first).

#include "initial_partition.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <exception>
#include <functional>
#include <future>
#include <numeric>
#include <queue>
#include <system_error>
#include <thread>

namespace kahip {

long long HostGraph::total_weight() const {
    long long s = 0;
    for (int v = 0; v < n; ++v) s += vwgt[v];
    return s;
}

long long host_edge_cut(const HostGraph& g, const std::vector<int>& part) {
    long long c = 0;
    for (int v = 0; v < g.n; ++v)
        for (int e = g.xadj[v]; e < g.xadj[v + 1]; ++e)
            if (part[v] != part[g.adjncy[e]]) c += g.adjwgt[e];
    return c / 2;
}

namespace {

struct Rng {
    uint64_t s;
    explicit Rng(uint64_t seed) : s(seed) {}
    uint64_t next() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ULL);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
        return z ^ (z >> 31);
    }
    uint32_t below(uint32_t n) { return n ? (uint32_t)(next() % n) : 0; }
    bool coin() { return next() & 1; }
};

uint64_t stream_seed(uint64_t seed, uint64_t a, uint64_t b) {
    Rng r(seed ^ (a * 0xD1B54A32D192ED03ULL) ^ (b * 0x8CB92BA72F3D8DD7ULL));
    r.next();
    return r.next();
}

// ------------------------------------------------------------------ graphs of the bisections
// Target and weight of an edge side by side: every loop below reads both.
struct Edge {
    int to, w;
};
struct Graph {
    int n = 0;
    std::vector<int> xadj, vwgt;
    std::vector<Edge> edges;
    long long total_weight() const {
        long long t = 0;
        for (int v = 0; v < n; ++v) t += vwgt[v];
        return t;
    }
};

// Graphs of more nodes than this miss the near caches when they are walked in random order; the
// walks then fetch the rows and labels of the nodes ahead (RGG 2^22, k = 64: clustering in the
// bisections 1.7 -> 1.1 s of thread time).
constexpr int kPrefetchNodes = 4096;

// ------------------------------------------------------------------ coarsening for bisection
// Sequential size-constrained LP in a random order (the reference's IP uses the same clustering
// with factor 12 inside the bisection hierarchy). Returns the number of clusters; label is
// renumbered to 0..nc-1 in first-appearance order.
int lp_cluster(const Graph& g, long long bound, int iters, Rng& rng, std::vector<int>& label_out) {
    const int n = g.n;
    label_out.resize(n);
    // int32 sizes and connection sums: the library keeps total node and edge weight below 2^31
    int max_row = 0;
    for (int v = 0; v < n; ++v) max_row = std::max(max_row, g.xadj[v + 1] - g.xadj[v]);
    std::vector<int> size_v(g.vwgt), order_v(n), acc_v(n, 0), touched_v(max_row + 1);
    int* const label = label_out.data();
    int* const size = size_v.data();
    int* const order = order_v.data();
    int* const acc = acc_v.data();
    int* const touched = touched_v.data();
    const int* const xadj = g.xadj.data();
    const int* const vwgt = g.vwgt.data();
    const Edge* const edges = g.edges.data();
    for (int v = 0; v < n; ++v) {
        label[v] = v;
        order[v] = v;
    }
    for (int i = n - 1; i > 0; --i) std::swap(order[i], order[rng.below(i + 1)]);
    const bool far = n > kPrefetchNodes;
    constexpr int kFar = 24, kMid = 12, kNear = 6, kRow = 16;
    for (int it = 0; it < iters; ++it) {
        int moved = 0;
        for (int i = 0; i < n; ++i) {
            if (far) {
                if (i + kFar < n) {
                    __builtin_prefetch(xadj + order[i + kFar]);
                    __builtin_prefetch(label + order[i + kFar]);
                }
                if (i + kMid < n) __builtin_prefetch(edges + xadj[order[i + kMid]]);
                if (i + kNear < n) {
                    const int u = order[i + kNear];
                    const int e1 = std::min(xadj[u + 1], xadj[u] + kRow);
                    for (int e = xadj[u]; e < e1; ++e) __builtin_prefetch(label + edges[e].to);
                }
            }
            const int v = order[i];
            const int own = label[v];
            int cnt = 0;
            for (int e = xadj[v], e1 = xadj[v + 1]; e < e1; ++e) {
                const int c = label[edges[e].to];
                const int old = acc[c];
                touched[cnt] = c;
                cnt += old == 0;
                acc[c] = old + edges[e].w;
            }
            int best = own;
            int bv = acc[own];
            for (int t = 0; t < cnt; ++t) {
                const int c = touched[t];
                const int ac = acc[c];
                // the connection test first: it rejects most candidates without reading size[c]
                if (c == own || ac < bv) continue;
                if ((long long)size[c] + vwgt[v] >= bound) continue;
                if (ac > bv || rng.coin()) {
                    best = c;
                    bv = ac;
                }
            }
            for (int t = 0; t < cnt; ++t) acc[touched[t]] = 0;
            if (best != own) {
                size[own] -= vwgt[v];
                size[best] += vwgt[v];
                label[v] = best;
                ++moved;
            }
        }
        if (moved == 0) break;
    }
    std::fill(acc, acc + n, -1);  // now: new id of a label
    int nc = 0;
    for (int v = 0; v < n; ++v) {
        int& r = acc[label[v]];
        if (r < 0) r = nc++;
        label[v] = r;
    }
    return nc;
}

Graph contract(const Graph& g, const std::vector<int>& label_v, int nc) {
    Graph c;
    c.n = nc;
    c.vwgt.assign(nc, 0);
    c.xadj.assign(nc + 1, 0);
    const int* const label = label_v.data();
    std::vector<int> start(nc + 1, 0), members(g.n);
    for (int v = 0; v < g.n; ++v) {
        c.vwgt[label[v]] += g.vwgt[v];
        start[label[v] + 1]++;
    }
    for (int p = 0; p < nc; ++p) start[p + 1] += start[p];
    std::vector<int> pos(start.begin(), start.end() - 1);
    for (int v = 0; v < g.n; ++v) members[pos[label[v]]++] = v;
    std::vector<int> acc_v(nc, 0), touched;
    int* const acc = acc_v.data();
    const int* const xadj = g.xadj.data();
    const Edge* const edges = g.edges.data();
    c.edges.reserve(g.edges.size() / 2);
    const bool far = g.n > kPrefetchNodes;
    constexpr int kMid = 12, kNear = 6, kRow = 16;
    for (int p = 0; p < nc; ++p) {
        for (int i = start[p]; i < start[p + 1]; ++i) {
            if (far) {
                if (i + kMid < g.n) __builtin_prefetch(edges + xadj[members[i + kMid]]);
                if (i + kNear < g.n) {
                    const int u = members[i + kNear];
                    const int e1 = std::min(xadj[u + 1], xadj[u] + kRow);
                    for (int e = xadj[u]; e < e1; ++e) __builtin_prefetch(label + edges[e].to);
                }
            }
            const int v = members[i];
            for (int e = xadj[v], e1 = xadj[v + 1]; e < e1; ++e) {
                const int q = label[edges[e].to];
                if (q == p) continue;
                if (acc[q] == 0) touched.push_back(q);
                acc[q] += edges[e].w;
            }
        }
        for (int q : touched) {
            c.edges.push_back({q, acc[q]});
            acc[q] = 0;
        }
        touched.clear();
        c.xadj[p + 1] = (int)c.edges.size();
    }
    return c;
}

// ------------------------------------------------------------------ 2-way FM
struct Bisection {
    std::vector<char> side;
    long long w[2] = {0, 0};
    long long cut = 0;
    bool counted = true;  // false: cut is not known yet, the first FM pass counts it
};

inline long long overload(const long long w[2], const long long maxw[2]) {
    return std::max(0LL, w[0] - maxw[0]) + std::max(0LL, w[1] - maxw[1]);
}

// What a move reads and writes of a neighbour.
struct FmNode {
    long long gain;
    int pos;  // index in its side's heap, -1: not in it
    char side, locked;
};

// Addressable 4-ary max-heap of the FM queue of one side: one entry per node, ordered by (gain,
// random tiebreak, node), a total order, so the order of the pops does not depend on the shape of
// the heap. Entries carry their keys: a sift reads four neighbouring entries instead of keys
// scattered over the nodes. A gain change draws a new tiebreak and moves the entry in place.
struct FmEntry {
    long long gain;
    uint64_t key;  // tie << 32 | node
    int node() const { return (int)(uint32_t)key; }
    unsigned __int128 order() const {  // one comparison without branches
        return ((unsigned __int128)((uint64_t)gain ^ (1ull << 63)) << 64) | key;
    }
    bool operator<(const FmEntry& o) const {
        return order() < o.order();
    }
};
struct FmHeap {
    FmEntry* h = nullptr;
    int size = 0;
    FmNode* node = nullptr;
    void put(int i, const FmEntry& e) {
        h[i] = e;
        node[e.node()].pos = i;
    }
    void up(int i, const FmEntry& e) {
        while (i > 0) {
            const int p = (i - 1) >> 2;
            if (!(h[p] < e)) break;
            put(i, h[p]);
            i = p;
        }
        put(i, e);
    }
    void down(int i, const FmEntry& e) {
        while (true) {
            const int c0 = 4 * i + 1;
            if (c0 >= size) break;
            const int c1 = std::min(c0 + 4, size);
            int c = c0;
            if (c1 - c0 == 4) {
                const int x = c0 + (h[c0] < h[c0 + 1]), y = c0 + 2 + (h[c0 + 2] < h[c0 + 3]);
                c = h[x] < h[y] ? y : x;
            } else {
                for (int j = c0 + 1; j < c1; ++j)
                    if (h[c] < h[j]) c = j;
            }
            if (!(e < h[c])) break;
            put(i, h[c]);
            i = c;
        }
        put(i, e);
    }
    void append(const FmEntry& e) { h[size++] = e; }  // before heapify()
    void heapify() {
        for (int i = 0; i < size; ++i) node[h[i].node()].pos = i;
        for (int i = (size - 2) >> 2; i >= 0 && size > 1; --i) down(i, FmEntry(h[i]));
    }
    void insert(const FmEntry& e) { up(size++, e); }
    void update(int i, const FmEntry& e) {
        if (i > 0 && h[(i - 1) >> 2] < e) up(i, e);
        else down(i, e);
    }
    void pop() {
        node[h[0].node()].pos = -1;
        const FmEntry last = h[--size];
        if (size > 0) down(0, last);
    }
};

// Buffers of fm_pass, kept per thread across calls (the tries call it thousands of times on
// graphs of a few hundred nodes, where allocation would dominate).
struct FmScratch {
    std::vector<FmNode> node;
    std::vector<FmEntry> heap[2];
    std::vector<int> moved;
};

// One FM pass with rollback to the best prefix. State order: lower overload first, then lower
// cut. Returns true when the state improved. Queues: boundary nodes of each side by gain; a node
// enters its queue when it first has a moved neighbour or at the start if it is on the boundary.
bool fm_pass(const Graph& g, Bisection& b, const long long maxw[2], int stall_limit,
             int stall_pct, Rng& rng) {
    static thread_local FmScratch sc;
    const int n = g.n;
    if ((int)sc.node.size() < n) {
        sc.node.resize(n);
        sc.heap[0].resize(n);
        sc.heap[1].resize(n);
        sc.moved.resize(n);
    }
    FmNode* const node = sc.node.data();
    int* const moved = sc.moved.data();
    FmHeap pq[2];
    pq[0].h = sc.heap[0].data();
    pq[1].h = sc.heap[1].data();
    pq[0].node = pq[1].node = node;
    const int* const xadj = g.xadj.data();
    const int* const vwgt = g.vwgt.data();
    const Edge* const edges = g.edges.data();
    char* const side = b.side.data();
    int nb = 0;
    long long ext2 = 0;  // twice the cut
    for (int v = 0; v < n; ++v) {
        const char sv = side[v];
        long long ext = 0, all = 0;
        bool bnd = false;
        for (int e = xadj[v], e1 = xadj[v + 1]; e < e1; ++e) {
            const bool other = side[edges[e].to] != sv;
            const long long w = edges[e].w;
            all += w;
            ext += other ? w : 0;
            bnd |= other;
        }
        ext2 += ext;
        node[v] = FmNode{2 * ext - all, -1, sv, 0};
        if (bnd) {
            pq[(int)sv].append({2 * ext - all, ((uint64_t)(uint32_t)rng.next() << 32) | (uint32_t)v});
            ++nb;
        }
    }
    if (!b.counted) b.cut = ext2 / 2;
    b.counted = true;
    pq[0].heapify();
    pq[1].heapify();
    if (stall_pct > 0) stall_limit = std::max(15, (int)((long long)stall_pct * nb / 100));
    long long cut = b.cut, w[2] = {b.w[0], b.w[1]};
    long long best_cut = cut, best_over = overload(w, maxw);
    int n_moved = 0, best_len = 0;
    int since_best = 0;
    while (true) {
        // a move from s to 1-s is allowed if the target stays within its bound or the source
        // is overloaded
        auto ok = [&](int s) {
            if (pq[s].size == 0) return false;
            const int t = 1 - s;
            return w[t] + vwgt[pq[s].h[0].node()] <= maxw[t] || w[s] > maxw[s];
        };
        const bool a0 = ok(0), a1 = ok(1);
        int s;
        if (a0 && a1) {
            const long long g0 = pq[0].h[0].gain, g1 = pq[1].h[0].gain;
            s = g0 > g1 || (g0 == g1 && w[0] >= w[1]) ? 0 : 1;
        } else if (a0) {
            s = 0;
        } else if (a1) {
            s = 1;
        } else {
            break;
        }
        const int v = pq[s].h[0].node();
        const long long gv = pq[s].h[0].gain;
        pq[s].pop();
        node[v].side = (char)(1 - s);
        node[v].locked = 1;
        w[s] -= vwgt[v];
        w[1 - s] += vwgt[v];
        cut -= gv;
        moved[n_moved++] = v;
        for (int e = xadj[v], e1 = xadj[v + 1]; e < e1; ++e) {
            const int u = edges[e].to;
            FmNode& nu = node[u];
            if (nu.locked) continue;
            // v left u's side (if u on s) or joined u's side (if u on 1-s)
            const long long d = 2LL * edges[e].w;
            nu.gain += nu.side == s ? d : -d;
            const FmEntry en{nu.gain, ((uint64_t)(uint32_t)rng.next() << 32) | (uint32_t)u};
            FmHeap& q = pq[(int)nu.side];
            if (nu.pos < 0) q.insert(en);
            else q.update(nu.pos, en);
        }
        const long long ov = overload(w, maxw);
        if (ov < best_over || (ov == best_over && cut < best_cut)) {
            best_over = ov;
            best_cut = cut;
            best_len = n_moved;
            since_best = 0;
        } else if (++since_best > stall_limit) {
            break;
        }
    }
    // keep the best prefix
    for (int i = n_moved; i > best_len; --i) {
        const int v = moved[i - 1];
        const int s = node[v].side;
        w[s] -= vwgt[v];
        w[1 - s] += vwgt[v];
    }
    for (int i = 0; i < best_len; ++i) side[moved[i]] = node[moved[i]].side;
    const long long old_over = overload(b.w, maxw);
    const bool improved = best_over < old_over || (best_over == old_over && best_cut < b.cut);
    b.w[0] = w[0];
    b.w[1] = w[1];
    b.cut = best_cut;
    return improved;
}

void fm_refine(const Graph& g, Bisection& b, const long long maxw[2], int stall, int pct,
               Rng& rng) {
    for (int pass = 0; pass < 8; ++pass)
        if (!fm_pass(g, b, maxw, stall, pct, rng)) break;
}

// BFS growing of side 0 from random starts until it reaches target0 (the cut is left to the
// first FM pass).
void grow(const Graph& g, long long total, long long target0, Rng& rng, Bisection& b,
          std::vector<char>& seen_v, std::vector<int>& queue_v) {
    b.side.assign(g.n, 1);
    seen_v.assign(g.n, 0);
    queue_v.resize(g.n);
    char* const seen = seen_v.data();
    int* const queue = queue_v.data();
    const int* const xadj = g.xadj.data();
    const Edge* const edges = g.edges.data();
    long long w0 = 0;
    int head = 0, tail = 0;
    int remaining = g.n;
    while (w0 < target0 && remaining > 0) {
        if (head == tail) {
            int s = (int)rng.below((uint32_t)g.n);
            while (seen[s]) s = (s + 1) % g.n;
            seen[s] = 1;
            queue[tail++] = s;
        }
        const int v = queue[head++];
        --remaining;
        b.side[v] = 0;
        w0 += g.vwgt[v];
        for (int e = xadj[v], e1 = xadj[v + 1]; e < e1; ++e) {
            const int u = edges[e].to;
            if (!seen[u]) {
                seen[u] = 1;
                queue[tail++] = u;
            }
        }
    }
    b.w[0] = w0;
    b.w[1] = total - w0;
    b.counted = false;
}

bool better_bis(const Bisection& a, const Bisection& b, const long long maxw[2]) {
    const long long oa = overload(a.w, maxw), ob = overload(b.w, maxw);
    return oa < ob || (oa == ob && a.cut < b.cut);
}

// Multilevel bisection of g. side[v] = 0 for the first part.
std::vector<char> ml_bisect(const Graph& g, long long target0, const long long maxw[2],
                            const IpParams& p, Rng& rng) {
    std::vector<Graph> levels;
    std::vector<std::vector<int>> maps;
    const Graph* cur = &g;
    const long long cbound = std::max(1LL, (std::min(maxw[0], maxw[1]) + p.coarsen_factor - 1) /
                                               p.coarsen_factor);
    while (cur->n > p.stop_nodes) {
        std::vector<int> label;
        const int nc = lp_cluster(*cur, cbound, 3, rng, label);
        if ((double)cur->n / (double)nc < 1.1) break;
        Graph c = contract(*cur, label, nc);
        maps.push_back(std::move(label));
        levels.push_back(std::move(c));
        cur = &levels.back();
    }
    Bisection best, b;
    bool have = false;
    std::vector<char> seen;
    std::vector<int> queue;
    const long long total = cur->total_weight();
    for (int t = 0; t < p.bisection_tries; ++t) {
        grow(*cur, total, target0, rng, b, seen, queue);
        fm_refine(*cur, b, maxw, p.fm_stall, p.fm_pct_coarsest, rng);
        if (!have || better_bis(b, best, maxw)) {
            std::swap(best, b);
            have = true;
        }
    }
    for (int l = (int)levels.size() - 1; l >= 0; --l) {
        const Graph& fine = l == 0 ? g : levels[l - 1];
        const std::vector<int>& map = maps[l];
        b.side.resize(fine.n);
        for (int v = 0; v < fine.n; ++v) b.side[v] = best.side[map[v]];
        b.w[0] = best.w[0];
        b.w[1] = best.w[1];
        b.cut = best.cut;
        fm_refine(fine, b, maxw, p.fm_stall, p.fm_pct_levels, rng);
        std::swap(best, b);
    }
    return std::move(best.side);
}

// Both sides of g as graphs of their own; ids[s][i] = node of g.
void extract(const Graph& g, const std::vector<char>& side, Graph out[2], std::vector<int> ids[2]) {
    std::vector<int> local(g.n);
    int cnt[2] = {0, 0};
    for (int v = 0; v < g.n; ++v) local[v] = cnt[(int)side[v]]++;
    for (int s = 0; s < 2; ++s) {
        out[s].n = cnt[s];
        out[s].xadj.resize(cnt[s] + 1);
        out[s].xadj[0] = 0;
        out[s].vwgt.resize(cnt[s]);
        out[s].edges.reserve(g.edges.size() / 2);
        ids[s].resize(cnt[s]);
    }
    for (int v = 0; v < g.n; ++v) {
        const int s = side[v];
        Graph& o = out[s];
        const int i = local[v];
        ids[s][i] = v;
        o.vwgt[i] = g.vwgt[v];
        for (int e = g.xadj[v]; e < g.xadj[v + 1]; ++e) {
            const int u = g.edges[e].to;
            if (side[u] == s) o.edges.push_back({local[u], g.edges[e].w});
        }
        o.xadj[i + 1] = (int)o.edges.size();
    }
}

struct RecCtx {
    const IpParams* p;
    uint64_t rep_seed;
    std::atomic<int>* idle;  // threads not in use, shared by the repetitions
};
constexpr int kSpawnNodes = 1000;  // halves of fewer nodes are not worth a thread

// Takes a thread if one is idle.
bool take_thread(std::atomic<int>& idle) {
    int have = idle.load();
    while (have > 0)
        if (idle.compare_exchange_weak(have, have - 1)) return true;
    return false;
}

// Partitions g into blocks lb..ub; part receives block ids for g's nodes.
void recurse(const Graph& g, int lb, int ub, RecCtx& ctx, std::vector<int>& part) {
    part.assign(g.n, lb);
    const int kk = ub - lb + 1;
    if (kk <= 1 || g.n == 0) return;
    const int mid = (lb + ub) / 2;
    const int k1 = mid - lb + 1, k2 = ub - mid;
    const long long W = g.total_weight();
    const long long target0 = (long long)std::llround((double)W * k1 / kk);
    // Each side may hold up to (number of its final blocks) x U: the imbalance budget is taken
    // against the global ideal block weight at every level, so every sub-problem stays feasible
    // and final blocks respect U whenever each bisection respects its bounds.
    long long maxw[2] = {(long long)k1 * ctx.p->block_bound, (long long)k2 * ctx.p->block_bound};
    maxw[0] = std::max(maxw[0], target0);
    maxw[1] = std::max(maxw[1], W - target0);
    Rng rng(stream_seed(ctx.rep_seed, (uint64_t)lb, (uint64_t)ub));
    std::vector<char> side;
    if (g.n == 1) {
        side.assign(1, 0);
    } else {
        side = ml_bisect(g, target0, maxw, *ctx.p, rng);
    }
    std::vector<int> ids[2];
    Graph half[2];
    extract(g, side, half, ids);
    std::vector<int> p0, p1;
    std::future<void> fut;
    if (k1 > 1 && k2 > 1 && g.n > kSpawnNodes && take_thread(*ctx.idle)) {
        try {
            fut = std::async(std::launch::async, [&] {
                struct Back {  // the thread is idle again, also after an exception
                    std::atomic<int>* idle;
                    ~Back() { ++*idle; }
                } back{ctx.idle};
                recurse(half[0], lb, mid, ctx, p0);
            });
        } catch (const std::system_error&) {  // the system has no thread to give: go on without
        }
    }
    if (!fut.valid()) recurse(half[0], lb, mid, ctx, p0);
    recurse(half[1], mid + 1, ub, ctx, p1);
    if (fut.valid()) fut.get();
    for (size_t i = 0; i < ids[0].size(); ++i) part[ids[0][i]] = p0[i];
    for (size_t i = 0; i < ids[1].size(); ++i) part[ids[1][i]] = p1[i];
}

// Moves nodes out of blocks heavier than `bound` until none is (or no move is possible): nodes
// of overloaded blocks are ranked by the cut increase of their best move into a block with room
// (neighbouring blocks, else the lightest block) and moved greedily; rankings are recomputed
// when a target fills up. Isolated nodes cost nothing and go first.
void rebalance(const HostGraph& g, int k, long long bound, std::vector<int>& part) {
    std::vector<long long> W(k, 0);
    for (int v = 0; v < g.n; ++v) W[part[v]] += g.vwgt[v];
    std::vector<long long> conn(k, 0);
    std::vector<int> touched;
    for (int pass = 0; pass < 64; ++pass) {
        bool any_over = false;
        for (int b = 0; b < k; ++b) any_over |= W[b] > bound;
        if (!any_over) return;
        const int lightest = (int)(std::min_element(W.begin(), W.end()) - W.begin());
        struct Move {
            long long loss;
            int v, to;
        };
        std::vector<Move> moves;
        for (int v = 0; v < g.n; ++v) {
            const int own = part[v];
            if (W[own] <= bound) continue;
            for (int e = g.xadj[v]; e < g.xadj[v + 1]; ++e) {
                const int b = part[g.adjncy[e]];
                if (conn[b] == 0) touched.push_back(b);
                conn[b] += g.adjwgt[e];
            }
            int t = -1;
            long long tc = -1;
            for (int b : touched)
                if (b != own && W[b] + g.vwgt[v] <= bound && conn[b] > tc) {
                    t = b;
                    tc = conn[b];
                }
            if (t < 0 && lightest != own && W[lightest] + g.vwgt[v] <= bound) {
                t = lightest;
                tc = conn[lightest];
            }
            const long long own_conn = conn[own];
            for (int b : touched) conn[b] = 0;
            touched.clear();
            if (t >= 0) moves.push_back({own_conn - tc, v, t});
        }
        if (moves.empty()) return;
        std::sort(moves.begin(), moves.end(), [](const Move& a, const Move& b) {
            return a.loss < b.loss || (a.loss == b.loss && a.v < b.v);
        });
        bool moved = false;
        for (const Move& m : moves) {
            const int own = part[m.v];
            if (W[own] <= bound) continue;
            if (W[m.to] + g.vwgt[m.v] > bound) continue;  // target filled up: next pass re-ranks
            W[own] -= g.vwgt[m.v];
            W[m.to] += g.vwgt[m.v];
            part[m.v] = m.to;
            moved = true;
        }
        if (!moved) return;
    }
}

}  // namespace

void initial_partition(const HostGraph& g, const IpParams& p, std::vector<int>& part) {
    const int k = std::max(1, p.k);
    part.assign(g.n, 0);
    if (k == 1 || g.n == 0) return;
    // split off isolated nodes
    std::vector<int> ids, iso_ids, local(g.n, -1);
    for (int v = 0; v < g.n; ++v) {
        if (g.xadj[v + 1] > g.xadj[v]) {
            local[v] = (int)ids.size();
            ids.push_back(v);
        } else {
            iso_ids.push_back(v);
        }
    }
    Graph core;
    core.n = (int)ids.size();
    core.xadj.assign(core.n + 1, 0);
    core.vwgt.resize(core.n);
    core.edges.reserve(g.adjncy.size());
    for (int i = 0; i < core.n; ++i) {
        const int v = ids[i];
        core.vwgt[i] = g.vwgt[v];
        for (int e = g.xadj[v]; e < g.xadj[v + 1]; ++e)
            if (local[g.adjncy[e]] >= 0) core.edges.push_back({local[g.adjncy[e]], g.adjwgt[e]});
        core.xadj[i + 1] = (int)core.edges.size();
    }
    unsigned hw = std::thread::hardware_concurrency();
    int threads = p.threads > 0 ? p.threads : (int)std::min(16u, hw ? hw : 1u);
    const int reps = std::max(1, p.repetitions);

    std::vector<std::vector<int>> results(reps);
    std::vector<long long> cuts(reps, 0);
    std::atomic<int> idle{std::max(0, threads - reps)};
    auto run_rep = [&](int r) {
        RecCtx ctx;
        ctx.p = &p;
        ctx.rep_seed = stream_seed(p.seed, 0x1e5u, (uint64_t)r);
        ctx.idle = &idle;
        std::vector<int> cp;
        recurse(core, 0, k - 1, ctx, cp);
        results[r] = std::move(cp);
        const std::vector<int>& part_r = results[r];
        long long cut = 0;
        for (int v = 0; v < core.n; ++v)
            for (int e = core.xadj[v]; e < core.xadj[v + 1]; ++e)
                if (part_r[v] != part_r[core.edges[e].to]) cut += core.edges[e].w;
        cuts[r] = cut;
    };
    if (threads <= 1) {  // the caller parallelises (e.g. over the graphs of a batch)
        for (int r = 0; r < reps; ++r) run_rep(r);
    } else {
        // an exception (e.g. bad_alloc) is rethrown here, not left to end the process
        std::vector<std::exception_ptr> err(reps);
        std::vector<std::thread> pool;
        const auto rep = [&](int r) {
            try {
                run_rep(r);
            } catch (...) {
                err[r] = std::current_exception();
            }
            ++idle;
        };
        pool.reserve(reps);
        for (int r = 0; r < reps; ++r) {
            try {
                pool.emplace_back(rep, r);
            } catch (const std::system_error&) {  // no thread to be had: on this one
                rep(r);
            }
        }
        for (auto& t : pool) t.join();
        for (auto& e : err)
            if (e) std::rethrow_exception(e);
    }
    int best = 0;
    for (int r = 1; r < reps; ++r)
        if (cuts[r] < cuts[best]) best = r;
    std::vector<long long> bw(k, 0);
    for (size_t i = 0; i < ids.size(); ++i) {
        part[ids[i]] = results[best][i];
        bw[results[best][i]] += g.vwgt[ids[i]];
    }
    // isolated nodes: heaviest first into the lightest block (lowest id on ties)
    std::stable_sort(iso_ids.begin(), iso_ids.end(),
                     [&](int a, int b) { return g.vwgt[a] > g.vwgt[b]; });
    using E = std::pair<long long, int>;
    std::priority_queue<E, std::vector<E>, std::greater<E>> heap;
    for (int b = 0; b < k; ++b) heap.emplace(bw[b], b);
    for (int v : iso_ids) {
        auto [w, b] = heap.top();
        heap.pop();
        part[v] = b;
        heap.emplace(w + g.vwgt[v], b);
    }
    if (p.block_bound > 0) rebalance(g, k, p.block_bound, part);
}

}  // namespace kahip
