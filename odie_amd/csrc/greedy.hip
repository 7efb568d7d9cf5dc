// B2 exact greedy support selection (odie/selection.py:129-207) for gfx950.
//
// The rule: repeatedly take the free cell (all four closure nodes already present) with the
// smallest id; otherwise the cell with the best score/cost over costs 1..min(4, cap-used),
// compared by cross-multiplication in fp64 and ties to the lower id; each taken cell adds
// its missing nodes and lowers the cost of the cells that share them.
//
// Layout and work split:
//  * a tournament tree per cost category 1..4 with fan 64 (one wave per node): level 0 nodes
//    hold, for 64 consecutive cells, the best cell of that category (largest sign-cleared
//    fp64 score key, then lowest id; -1 if none), higher levels the best of 64 nodes below;
//  * the levels whose nodes fit in 64 KiB live in LDS for the whole launch (loaded at entry,
//    written back at exit); lower levels stay in the caller's tree buffer;
//  * one workgroup runs the sequential choices; per choice it re-scans only the tree nodes
//    on the paths of the cells whose category changed (one wave per node, in parallel).
// Free cells never need the tree: a free cell adds no node and so changes no other cell's
// cost, hence every cell freed by a choice is taken right after it, in ascending id, exactly
// where the reference's "free first" rule takes them.  Category 0 is therefore not stored,
// and iteration counts, choices and trace order are those of the reference rule.
//
// Bulk start (odie_selection_relax, odie_selection_bulk).  Taking a cell only lowers the cost of
// others, so a cell's score/cost only ever rises.  Hence the cells the rule has taken when no
// cell with score/cost >= t is left are the closure of "take any cell with score/cost >= t",
// in whatever order, and they can be found in parallel, without the order:
//  * level of a node = the largest t at which it is taken = the largest level of its cells;
//    level of a cell = max over c of min(score/c, the (4-c)-th largest level of its nodes)
//    (c = 1..4 nodes still missing; 0 missing: the smallest node level alone).  The levels are the
//    least fixed point, reached from score/4 by relaxation in any order (relax_kernel);
//  * the number of nodes taken at t is the number of node levels >= t.  A radix select finds the
//    lowest t that keeps it within cap - 4 nodes, so that the rule's "cost <= cap - used" never
//    bound a choice on the way; the state at t is written and the sequential kernel goes on from
//    there (a few dozen choices instead of all of them).
// The comparisons of the rule are of rounded products, so t must be clear of every score/c: a
// score/c within 2^-47 of t (or a score that is negative, NaN or above 2^1000) leaves the initial
// state as it is, and the sequential kernel does everything.
// What bounds it: the relaxation's chains (a row of cells each freed by the last), walked inside a
// tile in LDS and across tiles by launches.  738^2 cells, cap 87936 (75,473 cells taken): 765 ms
// one choice at a time (about 10 us each, latency of one workgroup), 1.4-2.1 ms with the bulk start
// (12 relaxations 0.54 ms, the select and the writing 0.12 ms, the last choices 0.1-0.8 ms, the rest
// the host's two waits).
#include <algorithm>

#include "common.h"
#include "../../include/odie_amd.h"

namespace odie {
namespace {

constexpr int kFan = 64;
constexpr int kCats = 4;                // cost categories 1..4
constexpr int kGreedyBlock = 512;
constexpr int kGreedyWaves = kGreedyBlock / 64;
constexpr int kMaxLevels = 8;
constexpr int kLdsTreeInts = 12288;     // 48 KiB of tree ids in LDS
constexpr int kMaxTasks = 64;

struct TreeShape {
    int levels;
    int first_lds;                      // levels >= first_lds are kept in LDS during a launch
    int64_t size[kMaxLevels];           // nodes per level
    int64_t offset[kMaxLevels];         // first int of a level in the tree buffer (4 per node)
    int lds_ints;                       // ints of the LDS-resident levels
};

TreeShape tree_shape(int64_t n) {
    TreeShape t{};
    int64_t children = n, offset = 0;
    int levels = 0;
    do {
        const int64_t parents = (children + kFan - 1) / kFan;
        t.size[levels] = parents;
        t.offset[levels] = offset;
        offset += parents * kCats;
        children = parents;
        ++levels;
    } while (children > 1 && levels < kMaxLevels);
    t.levels = levels;
    t.first_lds = levels - 1;
    int64_t ints = t.size[levels - 1] * kCats;
    while (t.first_lds > 0 && ints + t.size[t.first_lds - 1] * kCats <= kLdsTreeInts) {
        --t.first_lds;
        ints += t.size[t.first_lds] * kCats;
    }
    t.lds_ints = static_cast<int>(ints);
    return t;
}

int64_t tree_ints(const TreeShape& t) { return t.offset[t.levels - 1] + t.size[t.levels - 1] * kCats; }

__device__ inline uint64_t score_key(const double* scores, int id) {
    return static_cast<uint64_t>(__double_as_longlong(scores[id])) & 0x7fffffffffffffffull;
}

__device__ inline bool better(int a, uint64_t ka, int b, uint64_t kb) {
    if (a < 0) return false;
    if (b < 0) return true;
    return ka > kb || (ka == kb && a < b);
}

// Best (id, key) over the wave: lane values in, result in every lane.
__device__ inline int wave_best(int id, uint64_t key) {
    for (int step = 32; step; step >>= 1) {
        const int other = __shfl_xor(id, step);
        const uint64_t other_key = __shfl_xor(key, step);
        if (better(other, other_key, id, key)) {
            id = other;
            key = other_key;
        }
    }
    return id;
}

// Offset of closure corner k (0..3) from its cell: 0, 1, R, R+1 (odie/selection.py:158).
__device__ inline int corner_delta(int k, int resolution) { return (k & 1) + (k >> 1) * resolution; }

struct GreedyArgs {
    const double* scores;
    int* missing;
    uint8_t* chosen;
    uint8_t* nodes;
    int* tree;
    int64_t* stats;
    int* trace;
    int n;
    int points;
    int resolution;
    int cap;
    int normalized;
    int chunk;
    TreeShape shape;
};

__device__ inline int& tree_at(const GreedyArgs& a, int* lds_tree, int level, int64_t node, int cat) {
    if (level >= a.shape.first_lds)
        return lds_tree[a.shape.offset[level] - a.shape.offset[a.shape.first_lds] + node * kCats + (cat - 1)];
    return a.tree[a.shape.offset[level] + node * kCats + (cat - 1)];
}

// Best cell of category `cat` under level-`level` node `node`, computed by one wave from the
// level below (cells for level 0).
__device__ inline int rescan(const GreedyArgs& a, int* lds_tree, int level, int64_t node, int cat) {
    const int lane = threadIdx.x % 64;
    const int64_t child = node * kFan + lane;
    int id = -1;
    if (level == 0) {
        if (child < a.n && !a.chosen[child] && a.missing[child] == cat) id = static_cast<int>(child);
    } else if (child < a.shape.size[level - 1]) {
        id = tree_at(a, lds_tree, level - 1, child, cat);
    }
    const uint64_t key = id >= 0 ? score_key(a.scores, id) : 0;
    return wave_best(id, key);
}

__global__ __launch_bounds__(kGreedyBlock) void init_kernel(GreedyArgs a) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kGreedyBlock + threadIdx.x;
    if (i < a.n) {
        a.missing[i] = 4;
        a.chosen[i] = 0;
    }
    if (i < a.points) a.nodes[i] = 0;
    if (i < 4) a.stats[i] = 0;
}

// One wave per (node, category) of one level; level 0 reads the cells.
__global__ __launch_bounds__(256) void build_kernel(GreedyArgs a, int level) {
    const int64_t task = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) / 64;
    const int64_t node = task / kCats;
    const int cat = static_cast<int>(task % kCats) + 1;
    if (node >= a.shape.size[level]) return;  // the whole wave takes the same branch
    const int lane = threadIdx.x % 64;
    const int64_t child = node * kFan + lane;
    int id = -1;
    if (level == 0) {
        if (child < a.n && !a.chosen[child] && a.missing[child] == cat) id = static_cast<int>(child);
    } else if (child < a.shape.size[level - 1]) {
        id = a.tree[a.shape.offset[level - 1] + child * kCats + (cat - 1)];
    }
    const uint64_t key = id >= 0 ? score_key(a.scores, id) : 0;
    id = wave_best(id, key);
    if (lane == 0) a.tree[a.shape.offset[level] + node * kCats + (cat - 1)] = id;
}

__global__ __launch_bounds__(kGreedyBlock) void greedy_kernel(GreedyArgs a) {
    extern __shared__ int lds_tree[];
    __shared__ int cell, cost, stop, nadded, added[4], naffected, affected[16], old_cat[16], new_cat[16];
    __shared__ int nfree, freed[16], ntasks, tasks_node[kMaxTasks], tasks_cat[kMaxTasks];
    __shared__ int changed[kMaxTasks];
    __shared__ int halted, invalid;
    __shared__ long long used, iterations;
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int64_t lds_base = a.shape.offset[a.shape.first_lds];
    for (int j = tid; j < a.shape.lds_ints; j += kGreedyBlock) lds_tree[j] = a.tree[lds_base + j];
    if (tid == 0) {
        used = a.stats[0];
        iterations = a.stats[1];
        halted = a.stats[2] != 0 || a.stats[3] != 0;
        stop = 0;
        invalid = 0;
    }
    __syncthreads();
    const int top = a.shape.levels - 1;
    // `stop` is read only right after a barrier, before thread 0 can write it again
    for (int step = 0; step < a.chunk && !halted; ++step) {
        // A. choose the best costly cell: the root winners of costs 1..min(4, cap-used),
        // score/cost compared by cross-multiplication, ties to the lower id
        if (tid == 0) {
            const int64_t remaining = static_cast<int64_t>(a.cap) - used;
            int best = -1, best_cost = 0;
            double best_score = 0.0;
            for (int c = 1; c <= 4 && c <= remaining; ++c) {
                const int candidate = tree_at(a, lds_tree, top, 0, c);
                if (candidate < 0) continue;
                const double score = a.scores[candidate];
                if (best >= 0) {
                    const double left = a.normalized ? score * static_cast<double>(best_cost) : score;
                    const double right = a.normalized ? best_score * static_cast<double>(c) : best_score;
                    if (!(left > right || (left == right && candidate < best))) continue;
                }
                best = candidate;
                best_cost = c;
                best_score = score;
            }
            cell = best;
            cost = best_cost;
            stop = best < 0;
        }
        __syncthreads();
        if (stop) break;
        // B. take it: mark its closure nodes, count the new ones
        if (wave == 0) {
            int node = 0;
            bool fresh = false;
            if (lane < 4) {
                node = static_cast<int>((static_cast<int64_t>(cell) + corner_delta(lane, a.resolution)) % a.points);
                fresh = a.nodes[node] == 0;
            }
            const uint64_t fresh_mask = __ballot(lane < 4 && fresh);
            if (lane < 4 && fresh) {
                a.nodes[node] = 1;
                added[__popcll(fresh_mask & ((uint64_t{1} << lane) - 1))] = node;
            }
            if (lane == 0) {
                nadded = __popcll(fresh_mask);
                a.chosen[cell] = 1;
                if (a.trace) a.trace[iterations] = cell;
                iterations += 1;
                used += nadded;
                invalid = nadded != cost;
                if (invalid) a.stats[3] = 1;
            }
        }
        __syncthreads();
        if (invalid) break;
        // C. cells sharing the new nodes lose one missing node per shared corner
        if (wave == 0) {
            int inc = -1;
            if (lane < 4 * nadded) {
                const int node = added[lane / 4];
                inc = static_cast<int>((static_cast<int64_t>(node) - corner_delta(lane % 4, a.resolution) + a.points) % a.points);
                if (inc >= a.n || a.chosen[inc]) inc = -1;
            }
            // distinct cells among the 16 lanes; the first lane of each counts the duplicates
            int dup = 0;
            bool first = inc >= 0;
            for (int j = 0; j < 16; ++j) {
                const int other = __shfl(inc, j);
                if (inc >= 0 && other == inc) {
                    ++dup;
                    if (j < lane) first = false;
                }
            }
            const uint64_t firsts = __ballot(first);
            int old = 0, now = 0;
            if (first) {
                old = a.missing[inc];
                now = old - dup;
                a.missing[inc] = now;
                const int slot = __popcll(firsts & ((uint64_t{1} << lane) - 1));
                affected[slot] = inc;
                old_cat[slot] = old;
                new_cat[slot] = now;
            }
            // cells freed by this choice are taken now, in ascending id
            const bool frees = first && now == 0;
            const uint64_t free_mask = __ballot(frees);
            int rank = 0;
            for (int j = 0; j < 16; ++j) {
                const int other = __shfl(inc, j);
                if (((free_mask >> j) & 1) && other < inc) ++rank;
            }
            if (frees) {
                freed[rank] = inc;
                a.chosen[inc] = 1;
            }
            if (lane == 0) {
                naffected = __popcll(firsts);
                nfree = __popcll(free_mask);
            }
        }
        __syncthreads();
        if (tid == 0) {
            for (int j = 0; j < nfree; ++j) {
                if (a.trace) a.trace[iterations] = freed[j];
                iterations += 1;
            }
            // D. tree tasks at level 0: the taken cell leaves category `cost`; every affected
            // cell leaves its old category and joins its new one (none if freed).
            int count = 0;
            auto add_task = [&](int node, int cat) {
                if (cat < 1 || cat > 4) return;
                for (int j = 0; j < count; ++j)
                    if (tasks_node[j] == node && tasks_cat[j] == cat) return;
                tasks_node[count] = node;
                tasks_cat[count] = cat;
                ++count;
            };
            add_task(cell / kFan, cost);
            for (int j = 0; j < naffected; ++j) {
                add_task(affected[j] / kFan, old_cat[j]);
                add_task(affected[j] / kFan, new_cat[j]);
            }
            ntasks = count;
        }
        __syncthreads();
        for (int level = 0; level <= top; ++level) {
            for (int t = wave; t < ntasks; t += kGreedyWaves) {
                const int node = tasks_node[t], cat = tasks_cat[t];
                const int best = rescan(a, lds_tree, level, node, cat);
                if (lane == 0) {
                    int& slot = tree_at(a, lds_tree, level, node, cat);
                    changed[t] = slot != best;
                    slot = best;
                }
            }
            __syncthreads();
            if (tid == 0) {
                int count = 0;
                for (int t = 0; t < ntasks; ++t) {
                    if (!changed[t]) continue;
                    const int node = tasks_node[t] / kFan, cat = tasks_cat[t];
                    bool seen = false;
                    for (int j = 0; j < count; ++j) seen |= tasks_node[j] == node && tasks_cat[j] == cat;
                    if (!seen) {
                        tasks_node[count] = node;
                        tasks_cat[count] = cat;
                        ++count;
                    }
                }
                ntasks = level < top ? count : 0;
            }
            __syncthreads();
            if (ntasks == 0) break;
        }
    }
    __syncthreads();
    for (int j = tid; j < a.shape.lds_ints; j += kGreedyBlock) a.tree[lds_base + j] = lds_tree[j];
    if (tid == 0) {
        a.stats[0] = used;
        a.stats[1] = iterations;
        if (stop && !invalid) a.stats[2] = 1;
    }
}

// ---------------------------------------------------------------------------------------
// Bulk start
// ---------------------------------------------------------------------------------------
constexpr int kTileX = 64, kTileY = 32;                 // cells of a relaxation tile
constexpr int kTilePitch = kTileX + 1;
constexpr int kTileNodes = kTilePitch * (kTileY + 1);   // 17 KB of LDS: two workgroups per CU
constexpr int kRelaxBlock = 1024;
constexpr int kRelaxRounds = 96;                        // about a tile's perimeter; unfinished tiles go on next launch
constexpr int kDigitBits = 11, kDigitBins = 1 << kDigitBits, kDigitPasses = 6;   // 66 >= 63 bits of a level
constexpr double kLargestScore = 0x1p1000, kSmallestLevel = 0x1p-900;

// Workspace: the node levels, the digit histograms, the select's state before every pass.
struct BulkState {
    uint64_t prefix[kDigitPasses + 1];      // digits of the threshold found before pass p
    int64_t remaining[kDigitPasses + 1];    // rank of the threshold among the keys of that prefix
    uint64_t above;                         // smallest level above the threshold
    uint64_t bad;                           // 1: no bulk start
};

struct BulkArgs {
    const double* scores;
    uint64_t* level;       // [points], bits of non-negative doubles (ordered as the doubles are)
    uint32_t* histogram;   // [kDigitPasses][kDigitBins]
    BulkState* state;
    int64_t* flag;         // relaxation: set to 1 when this launch raised a level
    int* missing;
    uint8_t* chosen;
    uint8_t* nodes;
    int64_t* stats;
    int n;
    int points;
    int resolution;
    int normalized;
    int rank;              // 0-based rank, from the largest, of the first level that is left out
};

struct BulkLayout { size_t histogram, state, total; };

BulkLayout bulk_layout(int64_t points) {
    const auto align = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
    BulkLayout l{};
    l.histogram = align(static_cast<size_t>(points) * 8);
    l.state = l.histogram + align(sizeof(uint32_t) * kDigitPasses * kDigitBins);
    l.total = l.state + align(sizeof(BulkState));
    return l;
}

__device__ inline double level_value(uint64_t bits) { return __longlong_as_double(static_cast<long long>(bits)); }
__device__ inline uint64_t level_bits(double value) { return static_cast<uint64_t>(__double_as_longlong(value)); }

// Level of a cell of score s (>= 0) from its nodes' levels.
__device__ inline double cell_level(double s, double a, double b, double c, double d, bool normalized) {
    const double hi0 = fmax(a, b), lo0 = fmin(a, b), hi1 = fmax(c, d), lo1 = fmin(c, d);
    const double smallest = fmin(lo0, lo1);
    if (!normalized) return fmax(s, smallest);
    const double largest = fmax(hi0, hi1), x = fmin(hi0, hi1), y = fmax(lo0, lo1);
    const double second = fmax(x, y), third = fmin(x, y);
    double t = fmax(s * 0.25, smallest);
    t = fmax(t, fmin(s / 3.0, largest));
    t = fmax(t, fmin(s * 0.5, second));
    return fmax(t, fmin(s, third));
}

__device__ inline int64_t wrap_node(int64_t id, int points) { return id >= points ? id - points : id; }

__global__ __launch_bounds__(256) void bulk_reset_kernel(BulkArgs a) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i < a.points) a.level[i] = 0;
    if (i < kDigitPasses * kDigitBins) a.histogram[i] = 0;
    if (i == 0) {
        a.state->above = ~uint64_t{0};
        a.state->bad = 0;
    }
}

__global__ __launch_bounds__(kRelaxBlock) void relax_kernel(BulkArgs a) {
    __shared__ uint64_t node[kTileNodes];
    const int r = a.resolution;
    const int x0 = blockIdx.x * kTileX, y0 = blockIdx.y * kTileY;
    const int nx = min(kTileX, r - x0) + 1, ny = min(kTileY, r - y0) + 1;   // nodes of the tile
    for (int j = threadIdx.x; j < kTileNodes; j += kRelaxBlock) {
        const int dx = j % kTilePitch, dy = j / kTilePitch;
        if (dx < nx && dy < ny)
            node[j] = a.level[wrap_node(static_cast<int64_t>(y0 + dy) * r + x0 + dx, a.points)];
    }
    constexpr int kRows = kRelaxBlock / kTileX, kCells = kTileY / kRows;
    const int dx = threadIdx.x % kTileX, row = threadIdx.x / kTileX;
    double score[kCells];
    bool refused = false;
#pragma unroll
    for (int j = 0; j < kCells; ++j) {
        const int dy = row + j * kRows;
        const bool real = dx < nx - 1 && dy < ny - 1;
        const double s = real ? a.scores[static_cast<int64_t>(y0 + dy) * r + x0 + dx] : 0.0;
        refused |= !(s >= 0.0 && s <= kLargestScore);
        score[j] = real && !refused ? fabs(s) : -1.0;
    }
    if (refused) a.state->bad = 1;
    __syncthreads();
    for (int round = 0; round < kRelaxRounds; ++round) {
        bool raised = false;
#pragma unroll
        for (int j = 0; j < kCells; ++j) {
            if (score[j] < 0.0) continue;
            uint64_t* corner = node + (row + j * kRows) * kTilePitch + dx;
            uint64_t at[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                at[k] = __hip_atomic_load(corner + (k & 1) + (k >> 1) * kTilePitch, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_WORKGROUP);
            const uint64_t t = level_bits(cell_level(score[j], level_value(at[0]), level_value(at[1]),
                                                     level_value(at[2]), level_value(at[3]), a.normalized));
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (t > at[k]) {
                    atomicMax(reinterpret_cast<unsigned long long*>(corner + (k & 1) + (k >> 1) * kTilePitch), t);
                    raised = true;
                }
        }
        if (!__syncthreads_or(raised)) break;
    }
    __syncthreads();
    bool wrote = false;
    for (int j = threadIdx.x; j < kTileNodes; j += kRelaxBlock) {
        const int ex = j % kTilePitch, ey = j / kTilePitch;
        if (ex >= nx || ey >= ny) continue;
        uint64_t* out = a.level + wrap_node(static_cast<int64_t>(y0 + ey) * r + x0 + ex, a.points);
        if (node[j] > *out) {
            atomicMax(reinterpret_cast<unsigned long long*>(out), node[j]);
            wrote = true;
        }
    }
    if (__syncthreads_or(wrote) && threadIdx.x == 0) *a.flag = 1;
}

// The select's state before pass `pass`, from the histogram of the pass before: the digit whose
// bin, counted from the largest, holds the rank.  Every block works it out (256 threads, eight
// bins each); block 0 stores it for the pass after next.
__device__ inline void next_digit(const BulkArgs& a, int pass, uint64_t& prefix, int64_t& remaining) {
    __shared__ int64_t sums[256];
    __shared__ uint64_t found_prefix;
    __shared__ int64_t found_remaining;
    if (pass == 0) {
        prefix = 0;
        remaining = a.rank;
    } else {
        constexpr int kPer = kDigitBins / 256;
        const uint32_t* bins = a.histogram + (pass - 1) * kDigitBins;
        const int64_t rank = a.state->remaining[pass - 1];
        const uint64_t before = a.state->prefix[pass - 1];
        const int shift = kDigitBits * (kDigitPasses - pass);
        // thread t takes the bins kDigitBins-1-kPer*t downwards
        int64_t mine = 0;
        for (int j = 0; j < kPer; ++j) mine += bins[kDigitBins - 1 - kPer * threadIdx.x - j];
        sums[threadIdx.x] = mine;
        __syncthreads();
        for (int step = 1; step < 256; step <<= 1) {
            const int64_t add = static_cast<int>(threadIdx.x) >= step ? sums[threadIdx.x - step] : 0;
            __syncthreads();
            sums[threadIdx.x] += add;
            __syncthreads();
        }
        int64_t at = sums[threadIdx.x] - mine;
        if (rank >= at && rank < at + mine)
            for (int j = 0; j < kPer; ++j) {
                const int bin = kDigitBins - 1 - kPer * threadIdx.x - j;
                const int64_t count = bins[bin];
                if (rank < at + count) {
                    found_prefix = before | (static_cast<uint64_t>(bin) << shift);
                    found_remaining = rank - at;
                    break;
                }
                at += count;
            }
        __syncthreads();
        prefix = found_prefix;
        remaining = found_remaining;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.state->prefix[pass] = prefix;
        a.state->remaining[pass] = remaining;
    }
}

__global__ __launch_bounds__(256) void level_histogram_kernel(BulkArgs a, int pass) {
    __shared__ uint32_t bins[kDigitBins];
    for (int j = threadIdx.x; j < kDigitBins; j += 256) bins[j] = 0;
    uint64_t prefix;
    int64_t remaining;
    next_digit(a, pass, prefix, remaining);
    __syncthreads();
    const int shift = kDigitBits * (kDigitPasses - 1 - pass);
    const int above = shift + kDigitBits;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < a.points; i += gridDim.x * 256ll) {
        const uint64_t key = a.level[i];
        if (above >= 64 || (key >> above) == (prefix >> above)) atomicAdd(bins + ((key >> shift) & (kDigitBins - 1)), 1u);
    }
    __syncthreads();
    for (int j = threadIdx.x; j < kDigitBins; j += 256)
        if (bins[j]) atomicAdd(a.histogram + pass * kDigitBins + j, bins[j]);
}

// The smallest level above the threshold (the first level left out).
__global__ __launch_bounds__(256) void level_above_kernel(BulkArgs a) {
    __shared__ unsigned long long least;
    if (threadIdx.x == 0) least = ~0ull;
    uint64_t left_out;
    int64_t remaining;
    next_digit(a, kDigitPasses, left_out, remaining);
    __syncthreads();
    unsigned long long mine = ~0ull;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < a.points; i += gridDim.x * 256ll)
        if (a.level[i] > left_out && a.level[i] < mine) mine = a.level[i];
    if (mine != ~0ull) atomicMin(&least, mine);
    __syncthreads();
    if (threadIdx.x == 0 && least != ~0ull) atomicMin(reinterpret_cast<unsigned long long*>(&a.state->above), least);
}

// t between the threshold's two levels, or a negative value when there is no room for it.
__device__ inline double bulk_level(const BulkState& state) {
    if (state.above == ~uint64_t{0}) return -1.0;
    const double low = level_value(state.prefix[kDigitPasses]), high = level_value(state.above);
    if (!(high >= kSmallestLevel) || !(high - low > high * 0x1p-40)) return -1.0;
    return low + (high - low) * 0.5;
}

__global__ __launch_bounds__(256) void bulk_check_kernel(BulkArgs a) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const double t = bulk_level(*a.state);
    bool close = t < 0.0;
    if (i < a.n && !close) {
        const double s = a.scores[i];
        for (int c = 1; c <= (a.normalized ? 4 : 1); ++c) close |= fabs(s - t * c) <= s * 0x1p-47;
    }
    if (close) a.state->bad = 1;
}

// Blocks of 1024, so that the two counters take few atomics (52 us in blocks of 256, 19 us so).
__global__ __launch_bounds__(1024) void bulk_apply_kernel(BulkArgs a) {
    if (a.state->bad) return;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 1024 + threadIdx.x;
    const double t = bulk_level(*a.state);
    bool node = false, taken = false;
    if (i < a.points) {
        node = level_value(a.level[i]) >= t;
        a.nodes[i] = node;
    }
    if (i < a.n) {
        double at[4];
        int lacking = 0;
        for (int k = 0; k < 4; ++k) {
            at[k] = level_value(a.level[wrap_node(i + corner_delta(k, a.resolution), a.points)]);
            lacking += at[k] < t;
        }
        taken = cell_level(fabs(a.scores[i]), at[0], at[1], at[2], at[3], a.normalized) >= t;
        a.chosen[i] = taken;
        a.missing[i] = lacking;
    }
    const int nodes = __syncthreads_count(node), cells = __syncthreads_count(taken);
    if (threadIdx.x == 0) {
        if (nodes) atomicAdd(reinterpret_cast<unsigned long long*>(a.stats), static_cast<unsigned long long>(nodes));
        if (cells) atomicAdd(reinterpret_cast<unsigned long long*>(a.stats + 1), static_cast<unsigned long long>(cells));
    }
}

int check_common(const char* what, const double* scores, int n, int points, int* missing, uint8_t* chosen,
                 uint8_t* nodes, int* tree, int64_t* stats) {
    const std::string w(what);
    if (n < 1) return fail(w + ": n must be positive");
    if (points < n || points % 8) return fail(w + ": points must be an 8-aligned count >= n");
    if (!scores || !missing || !chosen || !nodes || !tree || !stats) return fail(w + ": null pointer");
    return 0;
}

}  // namespace
}  // namespace odie

using namespace odie;

ODIE_API int64_t odie_selection_tree_ints(int n) {
    if (n < 1) return -1;
    return tree_ints(tree_shape(n));
}

// Same signature as selection_init (odie/native/selection_cuda.cu:208-220), and the same failure
// value: the runtime's error code (hipErrorInvalidValue for a refused argument), the message in
// odie_error().  host_offsets /
// host_sizes / levels describe the caller's fan-32 tree allocation; this selector lays out its
// own fan-64 tree, which needs no more ints than that allocation (checked when given).
ODIE_API int selection_init(const double* scores, int n, int points, int* missing, uint8_t* chosen, uint8_t* nodes,
                            int* tree, int64_t* stats, const int* host_offsets, const int* host_sizes, int levels,
                            uint64_t stream) {
    if (check_common("selection_init", scores, n, points, missing, chosen, nodes, tree, stats)) return hipErrorInvalidValue;
    const TreeShape shape = tree_shape(n);
    if (host_offsets && host_sizes && levels > 0) {
        const int64_t available = static_cast<int64_t>(host_offsets[levels - 1]) + 5LL * host_sizes[levels - 1];
        if (available < tree_ints(shape)) return fail_code("selection_init: tree buffer too small");
    }
    GreedyArgs a{};
    a.scores = scores;
    a.missing = missing;
    a.chosen = chosen;
    a.nodes = nodes;
    a.tree = tree;
    a.stats = stats;
    a.n = n;
    a.points = points;
    a.shape = shape;
    const hipStream_t s = as_stream(stream);
    const int64_t count = points > n ? points : n;
    init_kernel<<<static_cast<uint32_t>((count + kGreedyBlock - 1) / kGreedyBlock), kGreedyBlock, 0, s>>>(a);
    for (int level = 0; level < shape.levels; ++level) {
        const int64_t waves = shape.size[level] * kCats;
        build_kernel<<<static_cast<uint32_t>((waves + 3) / 4), 256, 0, s>>>(a, level);
    }
    return launch_code("selection_init");
}

// Same signature as selection_chunk (odie/native/selection_cuda.cu:222-230); offsets, sizes and
// levels (the caller's fan-32 layout) are not needed.  Runs up to `chunk` choices (a choice's
// freed cells are taken with it); stats = {used nodes, iterations, done, invariant error}.
ODIE_API int selection_chunk(const double* scores, int n, int points, int resolution, int cap, bool normalized,
                             int* missing, uint8_t* chosen, uint8_t* nodes, int* tree, const int* offsets,
                             const int* sizes, int levels, int chunk, int64_t* stats, int* trace, uint64_t stream) {
    (void)offsets;
    (void)sizes;
    (void)levels;
    if (check_common("selection_chunk", scores, n, points, missing, chosen, nodes, tree, stats)) return hipErrorInvalidValue;
    if (resolution < 2 || static_cast<int64_t>(resolution) * resolution != n)
        return fail_code("selection_chunk: n must be resolution^2");
    if (cap < 0 || cap % 8 || cap > points) return fail_code("selection_chunk: cap must be 8-aligned within points");
    if (chunk < 1) return fail_code("selection_chunk: chunk must be positive");
    GreedyArgs a{};
    a.scores = scores;
    a.missing = missing;
    a.chosen = chosen;
    a.nodes = nodes;
    a.tree = tree;
    a.stats = stats;
    a.trace = trace;
    a.n = n;
    a.points = points;
    a.resolution = resolution;
    a.cap = cap;
    a.normalized = normalized ? 1 : 0;
    a.chunk = chunk;
    a.shape = tree_shape(n);
    greedy_kernel<<<1, kGreedyBlock, static_cast<size_t>(a.shape.lds_ints) * 4, as_stream(stream)>>>(a);
    return launch_code("selection_chunk");
}

ODIE_API int64_t odie_selection_bulk_workspace(int points) {
    if (points < 8 || points % 8) return -1;
    return static_cast<int64_t>(bulk_layout(points).total);
}

ODIE_API int odie_selection_relax(const double* scores, int n, int points, int resolution, int normalized,
                                  void* workspace, int64_t workspace_bytes, int first, int64_t* flags, int launches,
                                  uint64_t stream) {
    if (n < 4 || points < n || points % 8) return fail("odie_selection_relax: points must be an 8-aligned count >= n");
    if (resolution < 2 || static_cast<int64_t>(resolution) * resolution != n)
        return fail("odie_selection_relax: n must be resolution^2");
    if (!scores || !workspace || !flags) return fail("odie_selection_relax: null pointer");
    if (launches < 1) return fail("odie_selection_relax: launches must be positive");
    const BulkLayout l = bulk_layout(points);
    if (workspace_bytes < static_cast<int64_t>(l.total) || reinterpret_cast<uintptr_t>(workspace) % 16)
        return fail("odie_selection_relax: workspace must be aligned and hold odie_selection_bulk_workspace(points) bytes");
    char* space = static_cast<char*>(workspace);
    BulkArgs a{};
    a.scores = scores;
    a.level = reinterpret_cast<uint64_t*>(space);
    a.histogram = reinterpret_cast<uint32_t*>(space + l.histogram);
    a.state = reinterpret_cast<BulkState*>(space + l.state);
    a.n = n;
    a.points = points;
    a.resolution = resolution;
    a.normalized = normalized ? 1 : 0;
    const hipStream_t s = as_stream(stream);
    if (first) {
        const int64_t words = std::max<int64_t>(points, kDigitPasses * kDigitBins);
        bulk_reset_kernel<<<static_cast<uint32_t>((words + 255) / 256), 256, 0, s>>>(a);
    }
    const dim3 tiles((resolution + kTileX - 1) / kTileX, (resolution + kTileY - 1) / kTileY);
    for (int launch = 0; launch < launches; ++launch) {
        a.flag = flags + launch;
        relax_kernel<<<tiles, kRelaxBlock, 0, s>>>(a);
    }
    return check_launch("odie_selection_relax");
}

ODIE_API int odie_selection_bulk(const double* scores, int n, int points, int resolution, int cap, int normalized,
                                 int* missing, uint8_t* chosen, uint8_t* nodes, int* tree, int64_t* stats,
                                 void* workspace, int64_t workspace_bytes, uint64_t stream) {
    if (check_common("odie_selection_bulk", scores, n, points, missing, chosen, nodes, tree, stats)) return -1;
    if (resolution < 2 || static_cast<int64_t>(resolution) * resolution != n)
        return fail("odie_selection_bulk: n must be resolution^2");
    if (cap < 8 || cap % 8 || cap > points) return fail("odie_selection_bulk: cap must be 8-aligned within 8..points");
    const BulkLayout l = bulk_layout(points);
    if (!workspace || workspace_bytes < static_cast<int64_t>(l.total) || reinterpret_cast<uintptr_t>(workspace) % 16)
        return fail("odie_selection_bulk: workspace must be aligned and hold odie_selection_bulk_workspace(points) bytes");
    char* space = static_cast<char*>(workspace);
    BulkArgs a{};
    a.scores = scores;
    a.level = reinterpret_cast<uint64_t*>(space);
    a.histogram = reinterpret_cast<uint32_t*>(space + l.histogram);
    a.state = reinterpret_cast<BulkState*>(space + l.state);
    a.missing = missing;
    a.chosen = chosen;
    a.nodes = nodes;
    a.stats = stats;
    a.n = n;
    a.points = points;
    a.resolution = resolution;
    a.normalized = normalized ? 1 : 0;
    a.rank = cap - 4;   // at most cap - 4 levels lie above the one of this rank
    const hipStream_t s = as_stream(stream);
    const uint32_t blocks = static_cast<uint32_t>((points + 255) / 256);
    const uint32_t scan_blocks = std::min<uint32_t>(blocks, 2 * kCus);
    for (int pass = 0; pass < kDigitPasses; ++pass) level_histogram_kernel<<<scan_blocks, 256, 0, s>>>(a, pass);
    level_above_kernel<<<scan_blocks, 256, 0, s>>>(a);
    bulk_check_kernel<<<blocks, 256, 0, s>>>(a);
    bulk_apply_kernel<<<static_cast<uint32_t>((points + 1023) / 1024), 1024, 0, s>>>(a);
    GreedyArgs g{};
    g.scores = scores;
    g.missing = missing;
    g.chosen = chosen;
    g.nodes = nodes;
    g.tree = tree;
    g.stats = stats;
    g.n = n;
    g.points = points;
    g.shape = tree_shape(n);
    for (int level = 0; level < g.shape.levels; ++level) {
        const int64_t waves = g.shape.size[level] * kCats;
        build_kernel<<<static_cast<uint32_t>((waves + 3) / 4), 256, 0, s>>>(g, level);
    }
    return check_launch("odie_selection_bulk");
}
