// kc_count.hip -- exact k-clique counting kernels for gfx950 and kc_count().
//
// Reference kernels replaced (one wave of 64 lanes per task here, one
// 128-thread block per task there):
//   node orientation  kckernel_node_block_warp_binary_count   kclique/kckernels_orientation.cuh:319-475
//   edge orientation  kckernel_edge_block_warp_binary_count_o2 kclique/kckernels_orientation.cuh:479-650
//   node pivoting     kckernel_node_block_warp_binary_pivot_count kclique/kckernels_pivoting.cuh:2-346
//   edge pivoting     kckernel_edge_block_warp_binary_pivot_count kclique/kckernels.cuh:2263-2630
// plus the task selection of kclique/kclique.cuh:1318-1406 (degree-window
// buckets) -> size classes built by one device pass.
//
// Per task (a vertex u, or an oriented edge u->v) the wave
//   1. stages the task vertex list in LDS: N+(u), or T = N+(u) & N+(v)
//      (block_count_and_set_tri, include/TriCountPrim.cuh:2071-2103);
//   2. builds the induced subgraph as 64-bit bitmap rows in LDS: lanes stream
//      the concatenated out-lists of the task vertices (coalesced reads) and
//      binary-search each entry in the staged list (the reference searches the
//      other way, warp_sorted_count_and_encode, TriCountPrim.cuh:1768-1900);
//   3. counts:
//      orientation: P-lane partitions run independent DFS over the rows, a
//        child candidate set is the AND of two rows, the last level adds a
//        popcount (kckernels_orientation.cuh:381-463);
//      pivoting: one SCT tree per wave (per block of waves above 256
//        vertices); the pivot is the smallest index among the candidates j
//        maximising |X & row_j|; leaves add C(pivots, k - held) from an exact
//        uint64 table with overflow bits.  Branches on non-pivot vertices are
//        taken first and the pivot branch last as a tail call, so the stack
//        never holds more than k - held + 2 levels (the reference keeps
//        maxDeg levels in HBM).  Subtrees are re-encoded into one-, two- or
//        four-word rows held in registers once their candidate sets shrink,
//        and the last levels close in form (edges; triangles by lane walks;
//        3- and 4-cliques from the complement, by MFMA where a set is dense
//        enough).
// Sizes: tasks are binned by their exact list size (64, 128, 256 vertices in
// registers, 512, 1024 in LDS, larger in an HBM slice), each class cut into
// slices drained largest first.
//
// Also here: the serving loop's resident launches (k_pivot_open and its host
// side, OpenEngine), which take tasks from queues the host extends while they
// run.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "kc_device.h"

namespace kc {

constexpr int NCLASS = 6;
constexpr uint32_t CLASS_ROWS[NCLASS] = {64, 128, 256, 512, 1024, 0xFFFFFFFFu};
constexpr uint32_t INF32 = 0xFFFFFFFFu;
constexpr int ACC = 8;  // per-class accumulator slots
// A launch's tasks are dealt over NQUEUE queues, its accumulators kept in
// NSTRIPE copies, each in its own 64 bytes.  Atomics of the whole device on
// one address complete one every ~10 ns: with one queue head and one set of
// accumulators that, and not the work, bound launches of many small tasks
// (970,000 node tasks of 96 small graphs, one grab per four: 3.0 ms).
constexpr uint32_t NQUEUE = 32, QSTRIDE = 16;  // heads, u32 from one to the next
constexpr uint32_t NSTRIPE = 32;
constexpr uint32_t PIVOT_TOP2 = 256;  // largest pivoting task of the four-word register kernel

// one query of a launch: the oriented graph it runs on and its k
struct QDesc {
    const uint32_t *rowptr, *col, *src, *key;
    uint32_t k, gran, sample, offset;  // tasks with id % sample == offset run
    uint32_t psize;                    // lanes per partition of this query
};
static_assert(sizeof(QDesc) % 8 == 0, "QDesc is read as 64-bit words");

// the graph and k of the task a wave is working on
struct Cur {
    const uint32_t *rowptr, *col, *src, *key;  // key: the orientation's (null: not at hand)
    uint32_t k, gran, psize;
};

struct CountArgs {
    const QDesc *qd;
    const uint64_t *tasks;  // (query << 32) | vertex-or-edge id
    uint32_t ntasks;
    const uint32_t *ntasks_p;  // where the device has the number of tasks, when the host does not know it (or null)
    uint32_t nparts;        // partitions per wave the orientation DFS stacks are laid out for
    uint32_t chunk_log;     // log2 of the tasks per queue grab
    uint32_t rmax;          // row capacity of the workspace
    uint32_t wmax;          // words per row capacity
    uint32_t levels;        // stack levels
    const uint64_t *binom;
    const uint8_t *binom_ovf;
    uint32_t bstride;       // binom[n * bstride + r]
    uint32_t *qhead;        // NQUEUE heads: chunks taken
    uint32_t direct;        // 1: one block per chunk, block i takes chunk i (no queue)
    uint32_t single;        // 1: one query, its count is summed in acc[0] and acc[6] (below)
    uint64_t *acc;          // [0] count [1] bytes [2] tasks [3] tree nodes [4] max task ticks [5] sum task ticks [6] count
    uint32_t acc_mask;      // copies of acc - 1 (a wave adds to copy blockIdx & acc_mask)
    uint64_t *qcount;       // per query two sums: of the low and of the high 32 bits of what the waves add
    uint32_t *qovf;         // per query
    uint64_t *gscr;
    uint64_t gscr_words;
    uint64_t *local;        // per-vertex counts of the (single) query, or null
    uint32_t chain;         // wide kernel: pivot-chain levels walked before the entries
    const uint64_t *bits;   // per edge (u, v), N+(v) among N+(u): word o of edge e at o * bits_m + e (or null)
    uint64_t bits_m;
};

// ---- workspace layout (u64 units) -----------------------------------------
// Per-vertex counting (LOCAL) adds, for pivoting, the held and pivot sets of
// the current node and of every stack level, and for both traversals a u64
// accumulator per task vertex (lacc) and the DFS path of each partition.
struct Layout {
    uint64_t misc, list, offs, starts, keys, rows, stk, x, scal, lacc, path, total;
};
constexpr uint32_t PAIR_ROWS = 64;  // largest class whose bitmaps can be built pair by pair

__host__ __device__ inline Layout make_layout(uint32_t rmax, uint32_t wmax, uint32_t levels, uint32_t nparts,
                                              bool pivot, bool local = false)
{
    Layout L;
    L.misc = 0;
    L.list = L.misc + 8;
    L.starts = L.list + (rmax + 1) / 2;  // list and starts are dead once the rows are built
    L.offs = L.starts + (rmax + 1) / 2;
    L.keys = L.offs + (rmax + 2) / 2;
    L.rows = L.keys + (rmax <= PAIR_ROWS ? (rmax + 1) / 2 : 0);
    L.stk = L.rows + (uint64_t)rmax * wmax;
    const uint64_t sets = local ? 4 : 2;  // per level: candidates, branches (+ held, pivots)
    if (pivot) {
        L.x = L.stk + (uint64_t)levels * sets * wmax;
        L.scal = L.x + (local ? 3 : 1) * (uint64_t)wmax;  // X (+ current held, pivots)
        L.lacc = L.scal + (uint64_t)levels * 2;
        L.path = L.lacc + (local ? rmax : 0);
        L.total = L.path;
    } else {
        L.x = L.scal = L.stk + (uint64_t)nparts * levels * 2 * wmax;
        L.lacc = L.x;
        L.path = L.lacc + (local ? rmax : 0);
        L.total = L.path + (local ? ((uint64_t)nparts * levels + 1) / 2 : 0);
    }
    return L;
}

// ---- wave helpers ------------------------------------------------------------
__device__ inline int lane_id() { return threadIdx.x & 63; }

// A value every lane holds alike, moved to scalar registers: the compiler then
// treats what is derived from it as uniform (scalar ALU, scalar branches)
// instead of masking the wave lane by lane.
__device__ inline uint32_t uni32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

__device__ inline uint64_t uni64(uint64_t v)
{
    return ((uint64_t)uni32((uint32_t)(v >> 32)) << 32) | uni32((uint32_t)v);
}

__device__ inline uint64_t lanemask_lt()
{
    int l = lane_id();
    return l == 0 ? 0ull : (~0ull >> (64 - l));
}

__device__ inline uint32_t wave_incl_scan32(uint32_t x)
{
    int lane = lane_id();
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t y = __shfl_up(x, (unsigned)d, 64);
        if (lane >= d) x += y;
    }
    return x;
}

__device__ inline uint32_t wave_min32(uint32_t x)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x = min(x, (uint32_t)__shfl_xor(x, d, 64));
    return x;
}

__device__ inline uint64_t wave_max64(uint64_t x)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        uint64_t y = __shfl_xor(x, d, 64);
        x = y > x ? y : x;
    }
    return x;
}

// Barrier for the state of one traversal: the whole block when a block is
// one wave, only the wave when the waves of a block run separate subtrees.
template <bool WIDE>
__device__ inline void sync_tree()
{
    if (WIDE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// checked sum over the wave; *ovf set on carry-out
__device__ inline uint64_t wave_sum64_checked(uint64_t x, uint32_t &ovf)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        uint64_t y = __shfl_xor(x, d, 64);
        uint64_t s = x + y;
        if (s < x) ovf = 1;
        x = s;
    }
    return x;
}

// reductions inside a partition of P lanes (P a power of two, aligned)
__device__ inline uint32_t part_min32(uint32_t x, uint32_t P)
{
    for (uint32_t d = P >> 1; d >= 1; d >>= 1) x = min(x, (uint32_t)__shfl_xor(x, (int)d, 64));
    return x;
}

__device__ inline uint32_t part_sum32(uint32_t x, uint32_t P)
{
    for (uint32_t d = P >> 1; d >= 1; d >>= 1) x += __shfl_xor(x, (int)d, 64);
    return x;
}

__device__ inline void add_checked(uint64_t &acc, uint64_t v, uint32_t &ovf)
{
    uint64_t s = acc + v;
    if (s < acc) ovf = 1;
    acc = s;
}

// first index in sorted a[0..n) with a[i] >= x
template <class P>
__device__ inline uint32_t lower_bound_u32(const P *a, uint32_t n, uint32_t x)
{
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        uint32_t mid = (lo + hi) >> 1;
        if (a[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// ---- step 2: bitmap rows of the induced subgraph on list[0..R) -------------
// bit j of row i <=> list[j] in N+(list[i]); FULL also sets bit i of row j.
// Two ways, the cheaper one a task:
//   entries: stream the members' out-lists (coalesced) and search each entry
//     in the staged list (LDS), ceil(sum d+/64) rounds of ~8 instructions per
//     halving of R;
//   pairs: search each pair's later vertex in the earlier one's out-list
//     (global, two searches in flight per lane), ceil(R(R-1)/256) rounds, each
//     priced 60 + 40 per halving of the longest list (25 and 80 a halving
//     measured the same and 3 to 10% slower).  The orientation's key tells
//     which of the two holds the edge.
// Power-law graphs have out-lists much longer than the part of them inside a
// task (Chung-Lu n=1.2M, edge tasks of at most 64 vertices: 26 members, 1,530
// entries, 330 pairs): wave time of those tasks 58 -> 33 s at k=5, 68 -> 39 at
// k=7, and n=500k at k=7 6.0 -> 5.3 ms.  Above 64 vertices the gathers lose
// (65..128 at k=5: 32 -> 63 s).  keys = null: entries only.  Tasks whose rows
// come from the adjacency words (rows_from_bits) need neither.
template <bool FULL>
__device__ __attribute__((always_inline)) void build_rows(const Cur &g, uint32_t *list, uint32_t *offs,
                                                         uint32_t *starts, uint32_t *keys, uint64_t *rows, uint32_t R,
                                                         uint32_t W, uint64_t &bytes)
{
    const int lane = lane_id();
    for (uint32_t i = lane; i < R * W; i += 64) rows[i] = 0;
    uint32_t carry = 0, longest = 0;
    for (uint32_t base = 0; base < R; base += 64) {
        uint32_t i = base + lane, d = 0;
        if (i < R) {
            uint32_t w = list[i];
            uint32_t s = g.rowptr[w];
            d = g.rowptr[w + 1] - s;
            starts[i] = s;
            if (keys && g.key) keys[i] = g.key[w];
        }
        uint32_t inc = wave_incl_scan32(d);
        if (i < R) offs[i] = carry + inc - d;
        carry += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
        longest = max(longest, d);
    }
    if (lane == 0) offs[R] = carry;
    __syncthreads();
    const uint32_t total = uni32(carry);
    bytes += 8ull * R + 4ull * total;
    auto set = [&](uint32_t i, uint32_t j) {
        atomicOr((unsigned long long *)&rows[(uint64_t)i * W + (j >> 6)], 1ull << (j & 63));
        if (FULL) atomicOr((unsigned long long *)&rows[(uint64_t)j * W + (i >> 6)], 1ull << (i & 63));
    };
    longest = (uint32_t)__builtin_amdgcn_readfirstlane((int)__ockl_wfred_max_u32(longest));
    const uint32_t npair = R * (R - 1) / 2, depth = 32u - (uint32_t)__clz(longest | 1u);
    const uint32_t by_pair = ((npair + 127) / 128) * (60 + 40 * depth);
    const uint32_t by_entry = ((total + 63) / 64) * (16 + 8 * (32u - (uint32_t)__clz(R)));
    if (keys && g.key && by_pair < by_entry) {
        // pair f = (i, i + 1 + c mod R) with f = c R + i: every pair once, lanes side by side
        uint32_t i = lane, c = 0;
        auto wrap = [&]() {
            while (i >= R) {
                i -= R;
                ++c;
            }
        };
        wrap();
        for (uint32_t f = lane; f < npair; f += 128) {
            uint32_t lo[2], hi[2], x[2], n[2], pos[2] = {0, 0};
            const uint32_t *l[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                uint32_t j = i + 1 + c;
                j = j >= R ? j - R : j;
                const uint32_t ki = keys[i], kj = keys[j], vi = list[i], vj = list[j];
                const bool first = ki < kj || (ki == kj && vi < vj);
                lo[e] = first ? i : j;
                hi[e] = first ? j : i;
                x[e] = first ? vj : vi;
                const bool in = f + 64 * e < npair;
                n[e] = in ? offs[lo[e] + 1] - offs[lo[e]] : 0;
                l[e] = g.col + starts[lo[e]];
                if (f + 64 * (e + 1) < npair) {  // (i stays a member past the end)
                    i += 64;
                    wrap();
                }
            }
            for (uint32_t step = 1u << (depth - 1); step; step >>= 1)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t to = pos[e] + step;
                    if (to <= n[e] && l[e][to - 1] < x[e]) pos[e] = to;
                }
#pragma unroll
            for (int e = 0; e < 2; ++e)
                if (pos[e] < n[e] && l[e][pos[e]] == x[e]) set(lo[e], hi[e]);
        }
    } else {
        const uint32_t lo_v = list[0], hi_v = list[R - 1];
        uint32_t lo = 0;  // row of entry f: the last i with offs[i] <= f (f only grows)
        for (uint32_t f = lane; f < total; f += 64) {
            while (offs[lo + 1] <= f) ++lo;
            uint32_t x = g.col[starts[lo] + (f - offs[lo])];
            if (x < lo_v || x > hi_v) continue;
            uint32_t j = lower_bound_u32(list, R, x);
            if (j < R && list[j] == x) set(lo, j);
        }
    }
    __syncthreads();
}

// ---- step 3a: orientation DFS ---------------------------------------------
// Number of r-vertex cliques of the DAG rows (r >= 2).  Partitions of P lanes
// take first-level rows from a per-task LDS counter (*next_row) and run an
// independent DFS each; a lane only ever touches its own words (w = lip,
// lip + P, ...), so the DFS needs no barrier.  Returns the lane's share.
// LOCAL also adds, per found clique, 1 to each member in lacc (the task
// vertices; the root is credited with the task's count by the caller):
// partitions share lacc, so those adds are LDS atomics.
template <bool LOCAL>
__device__ uint64_t orient_count(const CountArgs &a, uint32_t P, const uint64_t *rows, uint64_t *stk,
                                 uint32_t *next_row, uint32_t R, uint32_t W, uint32_t r, uint64_t &nodes, uint32_t &ovf,
                                 uint64_t *lacc, uint32_t *path)
{
    const int lane = lane_id();
    uint64_t cnt = 0;
    if (r == 2) {
        for (uint32_t i = lane; i < R * W; i += 64) {
            const uint64_t x = rows[i];
            cnt += (uint64_t)__popcll(x);
            if (LOCAL && x) {
                const uint32_t row = i / W, wbase = (i % W) * 64;
                atomicAdd((unsigned long long *)&lacc[row], (unsigned long long)__popcll(x));
                for (uint64_t b = x; b; b &= b - 1)
                    atomicAdd((unsigned long long *)&lacc[wbase + (uint32_t)__builtin_ctzll(b)], 1ull);
            }
        }
        return cnt;
    }
    // P lanes per partition (the task's query); the stacks hold a.nparts partitions
    const uint32_t NP = 64 / P < a.nparts ? 64 / P : a.nparts;
    const uint32_t part = lane / P, lip = lane % P;
    if (part >= NP) return 0;
    const uint32_t wmax = a.wmax;
    uint64_t *base = stk + (uint64_t)part * a.levels * 2 * wmax;
    uint32_t *mypath = LOCAL ? path + (uint64_t)part * a.levels : nullptr;
    const uint32_t rem0 = r - 1;  // vertices still to pick below a first-level row
    uint64_t my_nodes = 0;
    for (;;) {
        uint32_t j = 0;
        if (lip == 0) j = atomicAdd(next_row, 1u);
        j = __shfl(j, (int)(part * P), 64);
        if (j >= R) break;
        // level 0: C = I = row j
        uint32_t c0 = 0;
        for (uint32_t w = lip; w < W; w += P) {
            uint64_t v = rows[(uint64_t)j * W + w];
            base[w] = v;
            base[wmax + w] = v;
            c0 += (uint32_t)__popcll(v);
        }
        c0 = part_sum32(c0, P);
        if (c0 < rem0) continue;
        int t = 0;
        for (;;) {
            uint64_t *C = base + (uint64_t)t * 2 * wmax, *I = C + wmax;
            uint32_t b = INF32;
            for (uint32_t w = lip; w < W; w += P) {
                uint64_t x = I[w];
                if (x) {
                    b = w * 64 + (uint32_t)__builtin_ctzll(x);
                    break;
                }
            }
            b = part_min32(b, P);
            if (b == INF32) {
                if (t == 0) break;
                --t;
                continue;
            }
            const uint32_t bw = b >> 6;
            if (bw % P == lip) I[bw] &= ~(1ull << (b & 63));
            if (LOCAL && lip == 0) mypath[t] = b;
            uint64_t *Cn = C + 2 * wmax;
            const uint64_t *rb = rows + (uint64_t)b * W;
            uint32_t c = 0;
            for (uint32_t w = lip; w < W; w += P) {
                uint64_t x = C[w] & rb[w];
                Cn[w] = x;
                Cn[wmax + w] = x;
                c += (uint32_t)__popcll(x);
            }
            c = part_sum32(c, P);
            ++my_nodes;
            const uint32_t remc = rem0 - 1 - (uint32_t)t;  // picks left below b
            if (remc == 1) {
                if (lip == 0) add_checked(cnt, c, ovf);
                if (LOCAL && c) {
                    // clique = root + j + path[0..t] + one vertex of Cn
                    for (uint32_t w = lip; w < W; w += P)
                        for (uint64_t x = Cn[w]; x; x &= x - 1)
                            atomicAdd((unsigned long long *)&lacc[w * 64 + (uint32_t)__builtin_ctzll(x)], 1ull);
                    if (lip == 0) {
                        atomicAdd((unsigned long long *)&lacc[j], (unsigned long long)c);
                        for (int l = 0; l <= t; ++l)
                            atomicAdd((unsigned long long *)&lacc[mypath[l]], (unsigned long long)c);
                    }
                }
            } else if (c >= remc) {
                ++t;
            }
        }
    }
    if (lip == 0) nodes += my_nodes;
    return cnt;
}

__device__ inline uint64_t rdlane64(uint64_t v, uint32_t src)
{
    uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)src);
    uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), (int)src);
    return ((uint64_t)hi << 32) | lo;
}

// ---- closed forms over one- and two-word candidate sets ----------------------
// |E|, triangles and 4-cliques of G[X] from its complement H (the non-edges
// inside X), by inclusion-exclusion over the edge sets F of H that span at
// most four vertices, sum_F (-1)^|F| C(n - |V(F)|, 4 - |V(F)|):
//   c4 = C(n,4) - m C(n-2,2) + C(m,2) + (n-4) P3 - (n-3) K3 - P4 - S3 + C4 + paw - dia + K4
// where, all as subgraphs of H: m edges, P3 = sum_x C(d_x,2) two-edge paths
// (C(m,2) - P3 is the number of two-edge matchings), K3 triangles,
// P4 = sum_{xy in E} (d_x-1)(d_y-1) - 3 K3 three-edge paths, S3 = sum_x C(d_x,3)
// three-edge stars, C4 = 1/2 sum_{x<y} C(c_xy,2) four-cycles (c_xy = common
// neighbours), paw = sum_x t_x (d_x-2) triangles with a pendant edge, dia =
// sum_{xy in E} C(c_xy,2) four-cycles with a chord, K4 four-cliques; and
// Goodman's c3 = C(n,3) - 1/2 sum_x d_x (n-1-d_x) - K3.
// With, per vertex x,
//   q = sum_u c_ux^2,  qE = sum_{u in Hx} c_ux^2,  t2 = sum_{u in Hx} c_ux = 2 t_x,
//   sd = sum_u c_ux = sum_{u in Hx} d_u
// (8 C4 = sum (q - d^2) - (sd - d), 2 P4 + 6 K3 = sum (d-1)(sd-d), 4 dia = sum
// qE - t2) the terms beyond the counts of edges come to
//   24 c4 = n(n-1)(n-2)(n-3) - 12 m (n-2)(n-3) + 12 m (m-1) + 24 K4
//           + sum_x t2 (12d - 4n + 6) - sd (12d - 9) + 3q - 6qE + d(d-1)(12n - 31 - 4d)
//   6 c3  = n(n-1)(n-2) - sum_x 3d(n-1-d) + t2
// (all modulo 2^32: 24 c4 <= 128^4 fits).  A K4 of H has every vertex in at
// least three H-triangles, so the K4 walk (over the H-edges u < v, counting
// the H-edges inside Hu & Hv above v) only visits such vertices.
//
// The c_ux are the matrix H H^T, which the matrix cores make 32 x 32 entries
// at a time (v_mfma_i32_32x32x32_i8, the bits of H as bytes 0 and 1).  A lane
// (j, b) = (lane & 31, lane >> 5) gets, of column j, the rows 8g + 4b + i (g, i
// < 4) in entry 4g + i.  The order of the summed index is free as long as
// both operands agree, so byte i of operand word g holds bit 8g + 4b + i: the
// operand words of a column are then also the 0/1 masks of its four entries.
// Entries are at most 127, so four pack into a word for the dot products.
// The walk this replaces took ~17 vector instructions per vertex u of X
// (~45 over two words); here a 32 x 32 block takes 4 x 10 and 8 matrix
// passes per 32 of the summed index.
struct CliqueCounts {
    uint32_t e, c3, c4;
};

// How the tree walk below a task closes its nodes, by the kernel around it:
//   MFMA      register kernels: sets of 33..128 vertices go through the matrix cores
//   LEAN      such sets by a uniform walk (no operand registers)
//   WIDE_SCT  the block-wide kernel: as LEAN, its one-word walk a function of its
//         own, the binomials of a closing node computed: two waves per SIMD do not
//         hide the trip to the table, and its registers are full.  With the matrix
//         cores and pivot_count as a function it spilled 736 bytes a lane and saved
//         registers at every call (R-MAT scale 22: edge tasks of 257..512 vertices
//         at k=5 2.16 s, 1.69 s now, node tasks above 512 0.84 -> 0.73 s; 1/1024 of
//         the edge tasks at k=8, both classes, 1.51 + 1.92 -> 1.22 + 1.58 s)
//   WIDE_DEEP  the same for deep trees: with the matrix cores, all its register walks
//         functions of their own (it spills 55 registers around the calls)
//   OPEN_SCT  the serving loop's resident kernel: as LEAN, without the step from 64-
//         to 32-vertex words inside a walk, whose two stacks do not fit its 64
//         registers together
enum Kind { MFMA, LEAN, WIDE_SCT, OPEN_SCT, WIDE_DEEP };
__host__ __device__ constexpr bool wide_kind(Kind k) { return k == WIDE_SCT || k == WIDE_DEEP; }

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// the lane's bit of a uniform mask
__device__ inline bool in_mask(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

__device__ inline uint32_t wave_sum32(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)__ockl_wfred_add_u32(x));
}

// lower lanes' values (both halves), upper lanes' values (both halves)
__device__ inline void halves(uint32_t x, uint32_t &lo, uint32_t &hi)
{
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    lo = r[0];
    hi = r[1];
}

// operand words of 32 bits of a row: byte i of word g = bit 8g + 4b + i
__device__ inline v4i spread_bits(uint32_t x)
{
    const uint32_t y = x >> ((lane_id() >> 5) * 4);
    v4i r;
#pragma unroll
    for (int g = 0; g < 4; ++g) r[g] = (int)(__umul24((y >> (8 * g)) & 15u, 0x204081u) & 0x01010101u);
    return r;
}

// The lane's share of the sums above over blocks of 32 vertices: H[I][K] is
// word K of the complement row of vertex 32 I + (lane & 31) (zero outside X).
// s4 += the sum's terms of 24 c4, s3 += those of 6 c3, sd += degrees; T3[J] =
// the block's vertices in three or more triangles of H.  live: blocks with a
// member (the others are branched over, which also keeps the blocks' entries
// from being in registers together).
template <int NB>
__device__ inline void complement_sums(const uint32_t (&H)[NB][NB], uint32_t live, uint32_t n, uint32_t &s4, uint32_t &s3,
                                       uint32_t &sd, uint32_t (&T3)[NB])
{
    const bool once = lane_id() < 32;
    v4i E[NB][NB];
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int K = 0; K < NB; ++K) E[I][K] = spread_bits(H[I][K]);
#pragma unroll
    for (int J = 0; J < NB; ++J) {
        T3[J] = 0;
        if (NB > 1 && !((live >> J) & 1u)) continue;
        uint32_t d = 0, q = 0, qE = 0, t2 = 0, sm = 0;
#pragma unroll
        for (int K = 0; K < NB; ++K) d += (uint32_t)__popc(H[J][K]);
#pragma unroll
        for (int I = 0; I < NB; ++I) {
            if (NB > 1 && !((live >> I) & 1u)) continue;
            v16i c = {0};
#pragma unroll
            for (int K = 0; K < NB; ++K) c = __builtin_amdgcn_mfma_i32_32x32x32_i8(E[I][K], E[J][K], c, 0, 0, 0);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint32_t cp = (uint32_t)c[4 * g] | ((uint32_t)c[4 * g + 1] << 8) | ((uint32_t)c[4 * g + 2] << 16) |
                                    ((uint32_t)c[4 * g + 3] << 24);
                const uint32_t hb = (uint32_t)E[J][I][g];
                const uint32_t cm = cp & ((hb << 8) - hb);
                t2 = __builtin_amdgcn_udot4(cp, hb, t2, false);
                sm = __builtin_amdgcn_udot4(cp, 0x01010101u, sm, false);
                q = __builtin_amdgcn_udot4(cp, cp, q, false);
                qE = __builtin_amdgcn_udot4(cm, cm, qE, false);
            }
        }
        s3 += t2 + (once ? 3u * d * (n - 1 - d) : 0u);
        sd += once ? d : 0u;
        s4 += t2 * (12 * d - 4 * n + 6) - sm * (12 * d - 9) + 3 * q - 6 * qE +
              (once ? d * (d - 1) * (12 * n - 31 - 4 * d) : 0u);
        uint32_t lo, hi;
        halves(t2, lo, hi);
        T3[J] = (uint32_t)__ballot(lo + hi >= 6);
    }
}

// the counts from the wave's sums
__device__ inline CliqueCounts complement_counts(uint32_t n, uint32_t m, uint32_t s3, uint32_t s4)
{
    CliqueCounts r;
    r.e = n * (n - 1) / 2 - m;
    r.c3 = (n * (n - 1) * (n - 2) - s3) / 6;
    r.c4 = (n * (n - 1) * (n - 2) * (n - 3) - 12 * m * (n - 2) * (n - 3) + 12 * m * (m - 1) + s4) / 24;
    return r;
}

// One-word sets.  U = uint64_t: lane l holds vertex l.  U = uint32_t: lanes l
// and l + 32 both hold vertex l.  mask64: the lanes of a set's members.
__device__ inline uint64_t mask64(uint64_t X) { return X; }
__device__ inline uint64_t mask64(uint32_t X) { return ((uint64_t)X << 32) | X; }
__device__ inline uint32_t bits_of(uint64_t x) { return (uint32_t)__popcll(x); }
__device__ inline uint32_t bits_of(uint32_t x) { return (uint32_t)__popc(x); }
__device__ inline uint32_t low_bit(uint64_t x) { return (uint32_t)__builtin_ctzll(x); }
__device__ inline uint32_t low_bit(uint32_t x) { return (uint32_t)__builtin_ctz(x); }
__device__ inline uint64_t rdlane(uint64_t v, uint32_t src) { return rdlane64(v, src); }
__device__ inline uint32_t rdlane(uint32_t v, uint32_t src)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)src);
}
// bits above b (b < bits of U)
template <class U>
__device__ inline U above(uint32_t b)
{
    return (~(U)0 << b) << 1;
}

// c2, c3 and (with_c4) c4 of G[X], n = |X| >= 1 (row: the lane's vertex's row)
// MM: 64-vertex sets go through the matrix cores too (48 more registers)
template <bool MM, class U>
__device__ __attribute__((always_inline)) CliqueCounts close_word(U X, U row, uint32_t n, bool with_c4)
{
    constexpr int BITS = 8 * sizeof(U);
    const uint32_t v = (uint32_t)lane_id() & (BITS - 1);
    const U Hl = in_mask(mask64(X)) ? (U)(X & ~row & ~((U)1 << v)) : (U)0;
    if (__ballot(Hl != 0) == 0) return complement_counts(n, 0, 0, 0);  // X is a clique
    uint32_t s4 = 0, s3 = 0, sd = 0;
    U T3 = 0;
    if constexpr (BITS == 32) {
        uint32_t H[1][1], t3[1];
        H[0][0] = Hl;
        complement_sums<1>(H, 1, n, s4, s3, sd, t3);
        T3 = t3[0];
    } else if constexpr (MM) {
        uint32_t H[2][2], t3[2];
        halves((uint32_t)Hl, H[0][0], H[1][0]);
        halves((uint32_t)(Hl >> 32), H[0][1], H[1][1]);
        complement_sums<2>(H, ((uint32_t)X ? 1u : 0u) | ((uint32_t)(X >> 32) ? 2u : 0u), n, s4, s3, sd, t3);
        T3 = ((uint64_t)t3[1] << 32) | t3[0];
    } else {
        // a uniform walk over u in X hands c_ux = |Hu & Hx| to every lane x
        const uint32_t d = bits_of(Hl);
        uint32_t q = 0, qE = 0, t2 = 0, sm = 0;
        for (U b = X; b; b &= b - 1) {
            const U Hu = rdlane(Hl, low_bit(b));
            const uint32_t c = bits_of((U)(Hl & Hu)), cm = in_mask(Hu) ? c : 0u;
            sm += c;
            t2 += cm;
            q += __umul24(c, c);
            qE += __umul24(cm, cm);
        }
        s4 = t2 * (12 * d - 4 * n + 6) - sm * (12 * d - 9) + 3 * q - 6 * qE + d * (d - 1) * (12 * n - 31 - 4 * d);
        s3 = in_mask(X) ? t2 + 3 * d * (n - 1 - d) : 0u;
        sd = d;
        T3 = __ballot(t2 >= 6);
    }
    if (with_c4 && bits_of(T3) >= 4) {  // K4 of H among the vertices in >= 3 H-triangles
        uint32_t k4 = 0;
        for (U ub = T3; ub; ub &= ub - 1) {
            const uint32_t u = low_bit(ub);
            const U Hu = T3 & rdlane(Hl, u) & above<U>(u);
            if (bits_of(Hu) < 3) continue;
            for (U vb = Hu; vb; vb &= vb - 1) {
                const uint32_t w = low_bit(vb);
                const U S = Hu & rdlane(Hl, w) & above<U>(w);
                if (bits_of(S) >= 2) k4 += in_mask(mask64(S)) ? bits_of((U)(S & Hl & above<U>(v))) : 0u;
            }
        }
        s4 += BITS == 32 ? 12 * k4 : 24 * k4;  // (32 vertices: both halves of the wave counted)
    }
    // n <= 64: s3 <= 6 C(64,3) < 2^20 and the degrees sum to less than 2^12
    const uint32_t sum = wave_sum32(s3 + (sd << 20));
    return complement_counts(n, (sum >> 20) / 2, sum & 0xFFFFFu, with_c4 ? wave_sum32(s4) : 0u);
}

__device__ inline uint64_t mul_chk(uint64_t x, uint64_t y, uint32_t &ovf)
{
    uint64_t r;
    if (__builtin_mul_overflow(x, y, &r)) ovf = 1;
    return r;
}

__device__ inline uint64_t binom_chk(const CountArgs &a, uint32_t n, uint32_t r, uint32_t &ovf)
{
    if (r > n) return 0;
    const uint64_t idx = (uint64_t)n * a.bstride + r;
    if (a.binom_ovf[idx]) ovf = 1;
    return a.binom[idx];
}

// k-cliques of a subtree at h = k-3: C(p,3) + C(p,2)|X| + p|E(X)| + t(X)
__device__ inline uint64_t close_k3(const CountArgs &a, uint32_t p, uint32_t cx, uint64_t e, uint64_t tri,
                                    uint32_t &ovf)
{
    uint64_t r = 0;
    add_checked(r, binom_chk(a, p, 3, ovf), ovf);
    add_checked(r, mul_chk(binom_chk(a, p, 2, ovf), cx, ovf), ovf);
    add_checked(r, mul_chk(p, e, ovf), ovf);
    add_checked(r, tri, ovf);
    return r;
}

// The k-cliques of a subtree with `need` vertices to find and no 5-clique
// wanted inside X: sum_{j <= min(need, 4)} C(p, need-j) c_j(X), c_0 = 1, c_1 = |X|.
// Lane j adds term j to its own sum (the wave's share of a count is spread
// over the lanes until the task ends).  The five binomials are one load,
// issued before the counts are made: term by term they were five dependent
// trips to memory, which a closing node waited for longer than it computed.
// With COMPUTED they are worked out for need <= 4 (p < 2^16: p^4 fits 64 bits).
template <bool COMPUTED>
struct CloseTerm {
    uint64_t b = 0;
    uint32_t o = 0;
    __device__ CloseTerm(const CountArgs &a, uint32_t need, uint32_t p)
    {
        const uint32_t j = (uint32_t)lane_id();
        if (COMPUTED && need <= 4) {
            const uint32_t r = need - j;  // (j > need: no term)
            const uint64_t q = p, p2 = p ? q * (q - 1) : 0ull, p3 = p > 1 ? p2 * (q - 2) : 0ull;
            b = r == 0 ? 1ull : r == 1 ? q : r == 2 ? p2 / 2 : r == 3 ? p3 / 6 : r == 4 && p > 2 ? p3 * (q - 3) / 24 : 0ull;
        } else if (j <= 4 && j <= need) {
            const uint64_t idx = (uint64_t)p * a.bstride + (need - j);
            b = a.binom[idx];
            o = a.binom_ovf[idx];
        }
    }
    __device__ void add(uint64_t &acc, uint32_t &ovf, uint32_t cx, const CliqueCounts &c) const
    {
        const uint32_t j = (uint32_t)lane_id();
        const uint32_t m = j == 0 ? 1u : j == 1 ? cx : j == 2 ? c.e : j == 3 ? c.c3 : j == 4 ? c.c4 : 0u;
        const uint64_t lo = (b & 0xFFFFFFFFull) * m, hi = (b >> 32) * m + (lo >> 32);
        if (m && (o || (hi >> 32))) ovf = 1;
        add_checked(acc, (hi << 32) | (lo & 0xFFFFFFFFull), ovf);
    }
};

// the wave's total of per-lane shares, in every lane; ovf (uniform) with it
__device__ inline uint64_t wave_total(uint64_t x, uint32_t lane_ovf, uint32_t &ovf)
{
    const uint64_t t = uni64(wave_sum64_checked(x, lane_ovf));
    if (__ballot(lane_ovf != 0)) ovf = 1;
    return t;
}

// SCT of a subproblem of at most 64 (U = uint64_t) or 32 (uint32_t) vertices
// held one row per lane: X0 is the candidate set, h0/p0 the held and pivot
// counts above it.  Every set is one uniform word, a score is one AND +
// popcount.  The open level is in scalar registers (tC candidates, tB branches
// left, the pivot, h, p); levels below it are put away across the lanes (lane
// i = level i) when a node opens a new level over one that has branches left,
// so the chain of pivot branches moves nothing.
// Returns the lanes' shares of the count.  A node closes in form at h >= k-4
// (close_word), and, at any h, once at most four candidates are left, which cannot hold a 5-clique.  Candidates
// adjacent to all others lie in every maximal clique of X: they become pivots
// together instead of one node each.  A 64-vertex subtree whose candidates
// are at most 32 is re-encoded as a 32-vertex one (not with OPEN_SCT).
template <Kind KIND, class U>
__device__ uint64_t sct_word(const CountArgs &a, uint32_t k, U row, U X0, uint32_t h0, uint32_t p0, uint64_t &nodes,
                             uint32_t &ovf)
{
    constexpr uint32_t BITS = 8 * sizeof(U);
    constexpr bool MM = KIND == MFMA || KIND == WIDE_DEEP;
    const uint32_t lane = (uint32_t)lane_id(), v = lane & (BITS - 1);
    k = uni32(k);
    U X = BITS == 64 ? (U)uni64(X0) : (U)uni32((uint32_t)X0);
    U tC = 0, tB = 0, stkC = 0, stkB = 0;
    uint32_t tM = 0, stkM = 0;  // h | p << 8 | pivot << 24 (p < 2^16, pivot < 256)
    bool open = false;
    int t = -1;
    uint32_t h = uni32(h0), p = uni32(p0);
    uint64_t acc = 0, my_nodes = 0;
    for (;;) {
        ++my_nodes;
        uint32_t cx = bits_of(X);
        const uint32_t need = k - h;  // (h <= k)
        if (p + cx >= need) {
            if (BITS == 64 && KIND != OPEN_SCT && cx <= 32 && need >= 3 && cx > 0) {
                if constexpr (BITS == 64 && KIND != OPEN_SCT) {
                    uint32_t row1 = 0, X1 = (uint32_t)X;
                    if ((X >> 32) == 0) {
                        uint32_t up;
                        halves((uint32_t)row, row1, up);
                    } else {
                        // the members' rows to the lanes 0..cx-1 (the other rows to lane 63), then
                        // new row j = ballot of bit x_j over them (the bitmap is symmetric)
                        const int to = (int)((in_mask(X) ? (uint32_t)__popcll(X & lanemask_lt()) : 63u) << 2);
                        uint32_t lo = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)(uint32_t)row);
                        uint32_t hi = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)(uint32_t)(row >> 32));
                        if (lane >= cx) lo = hi = 0;
                        uint32_t j = 0;
                        for (uint32_t bits = (uint32_t)X; bits; bits &= bits - 1, ++j) {
                            const uint32_t col = (uint32_t)__ballot((lo & (bits & -bits)) != 0);
                            row1 = (lane & 31) == j ? col : row1;
                        }
                        for (uint32_t bits = (uint32_t)(X >> 32); bits; bits &= bits - 1, ++j) {
                            const uint32_t col = (uint32_t)__ballot((hi & (bits & -bits)) != 0);
                            row1 = (lane & 31) == j ? col : row1;
                        }
                        X1 = cx >= 32 ? ~0u : (1u << cx) - 1;
                    }
                    add_checked(acc, sct_word<KIND, uint32_t>(a, k, row1, X1, h, p, nodes, ovf), ovf);
                    --my_nodes;  // counted again as the subtree's root
                }
            } else {
                bool close = need < 5 || cx == 0;
                if (!close) {
                    const uint32_t sc = bits_of((U)(X & row));
                    const U all = (U)__ballot(in_mask(mask64(X)) && sc + 1 == cx);  // adjacent to every other candidate
                    const uint32_t na = bits_of(all);
                    X &= ~all;
                    p += na;
                    cx -= na;
                    close = cx <= 4;
                    if (!close) {
                        // (score + 1, BITS-1 - index): the max names the smallest index of the largest score
                        uint32_t key = in_mask(mask64(X)) ? ((sc - na + 1) << 8) | (BITS - 1 - v) : 0u;
                        key = (uint32_t)__builtin_amdgcn_readfirstlane((int)__ockl_wfred_max_u32(key));
                        if ((key >> 8) + p >= need) {  // (key >> 8) = max score + 1 bounds the clique inside X
                            const uint32_t pv = BITS - 1 - (key & 0xFFu);
                            if (open) {
                                ++t;
                                stkC = lane == (uint32_t)t ? tC : stkC;
                                stkB = lane == (uint32_t)t ? tB : stkB;
                                stkM = lane == (uint32_t)t ? tM : stkM;
                            }
                            open = true;
                            tC = X;
                            tB = X & ~rdlane(row, pv) & ~((U)1 << pv);
                            tM = h | (p << 8) | (pv << 24);
                        }
                    }
                }
                if (close) {
                    const CloseTerm<wide_kind(KIND)> term(a, need, p);
                    CliqueCounts c{0, 0, 0};
                    if (cx >= 2 && need >= 3) {
                        c = close_word<MM>(X, row, cx, need > 3);
                    } else if (cx >= 2 && need == 2) {
                        const uint32_t sc = in_mask(mask64(X)) ? bits_of((U)(X & row)) : 0u;
                        c.e = wave_sum32(sc) / (BITS == 32 ? 4 : 2);
                    }
                    term.add(acc, ovf, cx, c);
                }
            }
        }
        // next branch of the open level: non-pivot vertices first, the pivot last
        if (!open) {
            if (t < 0) break;
            tC = rdlane(stkC, (uint32_t)t);
            tB = rdlane(stkB, (uint32_t)t);
            tM = (uint32_t)__builtin_amdgcn_readlane((int)stkM, t);
            --t;
            open = true;
        }
        h = tM & 0xFF;
        p = (tM >> 8) & 0xFFFF;
        if (tB) {
            const uint32_t b = low_bit(tB);
            X = tC & rdlane(row, b);
            tC &= ~((U)1 << b);
            tB &= tB - 1;
            ++h;
        } else {  // the pivot branch replaces its level
            X = tC & rdlane(row, tM >> 24);
            ++p;
            open = false;
        }
    }
    if (lane == 0) nodes += my_nodes;
    return acc;
}

// SCT of a one-word subproblem (row = the lane's row, 0 beyond the subproblem)
template <Kind KIND>
__device__ inline uint64_t sct64(const CountArgs &a, uint32_t k, uint64_t row, uint64_t X0, uint32_t h0, uint32_t p0,
                                 uint64_t &nodes, uint32_t &ovf)
{
    return sct_word<KIND, uint64_t>(a, k, row, X0, h0, p0, nodes, ovf);
}
template <Kind KIND>
__device__ __attribute__((noinline)) uint64_t sct64_wide(const CountArgs &a, uint32_t k, uint64_t row, uint64_t X0,
                                                         uint32_t h0, uint32_t p0, uint64_t &nodes, uint32_t &ovf)
{
    return sct64<KIND>(a, k, row, X0, h0, p0, nodes, ovf);
}

// A set of task vertices as S uniform words.
template <int S>
struct Words {
    uint64_t w[S];
};

// word o of the row of vertex v (uniform), from the lanes that hold the rows
template <int S>
__device__ __forceinline__ uint64_t row_word(const uint64_t (&row)[S][S], uint32_t v, int o)
{
    if (S == 1) return rdlane64(row[0][0], v);
    return v < 64 ? rdlane64(row[0][o], v) : rdlane64(row[S - 1][o], v & 63);
}

// The SCT of a task of at most 64 * S vertices with per-vertex credits: lane l
// holds the rows and credits of vertices l, l + 64, ..; the sets X (candidates),
// H (held) and P (pivots) of a node are uniform words, kept with every open
// level as in sct_word (a level stays open only while a vertex of its branches
// is held, so there are at most k - 3 of them).  A subtree
// with t = k - h vertices to find and no 4-clique wanted inside X (t <= 3, or at
// most three candidates) closes with
//     in all      sum_j C(p, t-j) c_j(X)            (every held vertex)
//     a pivot     sum_j C(p-1, t-1-j) c_j(X)
//     x in X      sum_j C(p, t-j) c_{j-1}(X & row_x)
// j <= 3, the triangles through x counted by a uniform walk of X; the eight
// binomials are one load.  No credit can wrap unless the count does.
// Returns the count of the subtree (every lane).
template <int S>
__device__ uint64_t sct_local(const CountArgs &a, uint32_t k, const uint64_t (&row)[S][S], uint32_t R, uint32_t h0,
                              uint64_t (&credit)[S], uint64_t &nodes, uint32_t &ovf)
{
    static_assert(KC_MAX_K <= 64, "a level per lane");
    const uint32_t lane = (uint32_t)lane_id();
    k = uni32(k);
    Words<S> X, H, P, tC, tB, tH, tP, stkC, stkB, stkH, stkP;
#pragma unroll
    for (int o = 0; o < S; ++o) {
        const uint32_t r = R > 64u * o ? R - 64u * o : 0u;
        X.w[o] = uni64(r >= 64 ? ~0ull : (1ull << r) - 1);
        H.w[o] = P.w[o] = tC.w[o] = tB.w[o] = tH.w[o] = tP.w[o] = 0;
        stkC.w[o] = stkB.w[o] = stkH.w[o] = stkP.w[o] = 0;
    }
    uint32_t tM = 0, stkM = 0;  // h | p << 8 | pivot << 24 (p < 2^16, pivot < 256)
    bool open = false;
    int t = -1;
    uint32_t h = uni32(h0), p = 0;
    uint64_t acc = 0, my_nodes = 0;
    for (;;) {
        ++my_nodes;
        uint32_t cx = 0;
#pragma unroll
        for (int o = 0; o < S; ++o) cx += (uint32_t)__popcll(X.w[o]);
        const uint32_t need = k - h;
        if (p + cx >= need) {
            uint32_t sc[S];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                sc[s] = 0;
#pragma unroll
                for (int o = 0; o < S; ++o) sc[s] += (uint32_t)__popcll(X.w[o] & row[s][o]);
            }
            bool close = need <= 3;
            if (!close) {
                uint32_t na = 0;
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const uint64_t all = __ballot(in_mask(X.w[s]) && sc[s] + 1 == cx);  // adjacent to every other candidate
                    na += (uint32_t)__popcll(all);
                    X.w[s] &= ~all;
                    P.w[s] |= all;
                }
                p += na;
                cx -= na;
#pragma unroll
                for (int s = 0; s < S; ++s) sc[s] -= na;  // (members of X: each is adjacent to all of them)
                close = cx <= 3;
            }
            if (close) {
                uint64_t b = 0;
                uint32_t o8 = 0;
                const int up = lane < 4 ? 0 : 1, r = (int)need - up - (int)(lane & 3);
                if (lane < 8 && r >= 0 && (up == 0 || p > 0)) {
                    const uint64_t at = (uint64_t)(p - up) * a.bstride + (uint32_t)r;
                    b = a.binom[at];
                    o8 = a.binom_ovf[at];
                }
                uint32_t e = 0, tri = 0, t2[S];
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    t2[s] = 0;
                    e += in_mask(X.w[s]) ? sc[s] : 0u;
                }
                e = cx >= 2 && need >= 2 ? wave_sum32(e) / 2 : 0u;
                if (cx >= 3 && need >= 3) {
                    uint64_t g[S][S];
#pragma unroll
                    for (int s = 0; s < S; ++s)
#pragma unroll
                        for (int o = 0; o < S; ++o) g[s][o] = in_mask(X.w[s]) ? (X.w[o] & row[s][o]) : 0ull;
#pragma unroll
                    for (int q = 0; q < S; ++q)
                        for (uint64_t bits = X.w[q]; bits; bits &= bits - 1) {
                            const uint32_t u = (uint32_t)__builtin_ctzll(bits);
                            uint64_t gu[S];
#pragma unroll
                            for (int o = 0; o < S; ++o) gu[o] = rdlane64(g[q][o], u);
#pragma unroll
                            for (int s = 0; s < S; ++s) {
                                uint32_t c = 0;
#pragma unroll
                                for (int o = 0; o < S; ++o) c += (uint32_t)__popcll(g[s][o] & gu[o]);
                                t2[s] += in_mask(gu[s]) ? c : 0u;
                            }
                        }
#pragma unroll
                    for (int s = 0; s < S; ++s) tri += t2[s];
                    tri = wave_sum32(tri) / 6;
                }
                const uint64_t B0 = rdlane64(b, 0), B1 = rdlane64(b, 1), B2 = rdlane64(b, 2), B3 = rdlane64(b, 3);
                uint64_t all = 0;
                add_checked(all, B0, ovf);
                add_checked(all, mul_chk(B1, cx, ovf), ovf);
                add_checked(all, mul_chk(B2, e, ovf), ovf);
                add_checked(all, mul_chk(B3, tri, ovf), ovf);
                const uint32_t oc = lane == 0 ? 1u : lane == 1 ? cx : lane == 2 ? e : lane == 3 ? tri : 0u;
                if (__ballot(o8 && oc)) ovf = 1;
                add_checked(acc, all, ovf);
                const uint64_t piv = rdlane64(b, 4) + rdlane64(b, 5) * cx + rdlane64(b, 6) * e + rdlane64(b, 7) * tri;
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const uint64_t own = B1 + B2 * sc[s] + B3 * (t2[s] / 2);
                    credit[s] += in_mask(X.w[s]) ? own : in_mask(H.w[s]) ? all : in_mask(P.w[s]) ? piv : 0ull;
                }
                // (B1, B2 and B3 are 0 where need has no room for them)
            } else {
                uint32_t key = 0;
#pragma unroll
                for (int s = 0; s < S; ++s)
                    key = in_mask(X.w[s]) ? max(key, ((sc[s] + 1) << 8) | (64u * S - 1 - 64u * s - lane)) : key;
                key = (uint32_t)__builtin_amdgcn_readfirstlane((int)__ockl_wfred_max_u32(key));
                if ((key >> 8) + p >= need) {
                    const uint32_t pv = 64u * S - 1 - (key & 0xFFu);
                    if (open) {
                        ++t;
                        const bool here = lane == (uint32_t)t;
#pragma unroll
                        for (int o = 0; o < S; ++o) {
                            stkC.w[o] = here ? tC.w[o] : stkC.w[o];
                            stkB.w[o] = here ? tB.w[o] : stkB.w[o];
                            stkH.w[o] = here ? tH.w[o] : stkH.w[o];
                            stkP.w[o] = here ? tP.w[o] : stkP.w[o];
                        }
                        stkM = here ? tM : stkM;
                    }
                    open = true;
#pragma unroll
                    for (int o = 0; o < S; ++o) {
                        tC.w[o] = X.w[o];
                        tB.w[o] = X.w[o] & ~row_word<S>(row, pv, o) & ~((pv >> 6) == (uint32_t)o ? 1ull << (pv & 63) : 0ull);
                        tH.w[o] = H.w[o];
                        tP.w[o] = P.w[o];
                    }
                    tM = h | (p << 8) | (pv << 24);
                }
            }
        }
        // next branch of the open level: non-pivot vertices first, the pivot last
        if (!open) {
            if (t < 0) break;
#pragma unroll
            for (int o = 0; o < S; ++o) {
                tC.w[o] = rdlane64(stkC.w[o], (uint32_t)t);
                tB.w[o] = rdlane64(stkB.w[o], (uint32_t)t);
                tH.w[o] = rdlane64(stkH.w[o], (uint32_t)t);
                tP.w[o] = rdlane64(stkP.w[o], (uint32_t)t);
            }
            tM = (uint32_t)__builtin_amdgcn_readlane((int)stkM, t);
            --t;
            open = true;
        }
        h = tM & 0xFF;
        p = (tM >> 8) & 0xFFFF;
        H = tH;
        P = tP;
        uint64_t left = tB.w[0];
        if (S > 1) left |= tB.w[S - 1];
        const bool held = left != 0;
        uint32_t v = tM >> 24;
        if (held) v = tB.w[0] ? (uint32_t)__builtin_ctzll(tB.w[0]) : 64u + (uint32_t)__builtin_ctzll(tB.w[S - 1]);
#pragma unroll
        for (int o = 0; o < S; ++o) {
            const uint64_t bit = (v >> 6) == (uint32_t)o ? 1ull << (v & 63) : 0ull;
            X.w[o] = tC.w[o] & row_word<S>(row, v, o);
            H.w[o] |= held ? bit : 0ull;
            P.w[o] |= held ? 0ull : bit;
            if (held) {
                tC.w[o] &= ~bit;
                tB.w[o] &= ~bit;
            }
        }
        h += held ? 1u : 0u;
        p += held ? 0u : 1u;
        open = held;  // the pivot branch replaces its level
    }
    if (lane == 0) nodes += my_nodes;
    return acc;
}

// ---- step 3b: pivoting (SCT) ----------------------------------------------
struct Scal {
    uint32_t held, piv, pivot, pad;
};

// A subtree rooted at a node with h held vertices, p pivot vertices and
// candidate set X represents every clique R_h + S + Q with S a clique of G[X]
// and Q a subset of the pivots, so its k-cliques number
//     sum_j C(p, k-h-j) * c_j(X),   c_j = j-cliques of G[X].
// With c_0 = 1, c_1 = |X| and c_2 = |E(X)| = (1/2) sum_{j in X} |X & row_j|
// (the pivot scores) the subtree is closed-form once h >= k-2:
//     h = k:   1        h = k-1:   p + |X|        h = k-2:  C(p,2) + p|X| + |E(X)|
// so the SCT is only expanded while h < k-2.  h = k-3 closes with c_3 =
// triangles of G[X] (lane walks; with per-vertex credits for LOCAL), and the
// register kernels close h = k-4 with c_3 and c_4 of near-cliques from the
// complement.  A node is also dropped when
// h + p + max_j|X & row_j| + 1 < k (the largest clique inside X has at most
// maxIntersection + 1 vertices, cf. kclique/kckernels.cuh:2573-2584).
//
// LOCAL also credits every task vertex in lacc with the k-cliques of the
// subtree that contain it (the root with the task's count, by the caller).
// A subtree (H, P, X) with t = k - h holds the cliques H + S + Q, S a subset
// of P and Q a clique of G[X] with |S| + |Q| = t, so
//     held vertex  sum_j C(p, t-j) c_j(X)      pivot vertex  sum_j C(p-1, t-1-j) c_j(X)
//     x in X       sum_j C(p, t-j) c_{j-1}(X & row_x)
// which at a leaf (X empty) is the reference's hold/pivot split
// (kclique/kclique_local.cuh, kckernels_local.cuh).  The sets H and P of the
// node live beside X, and each stack level keeps its own copies.  Vertex sets
// H, P and X are disjoint and lane w owns the 64 vertices of word w, so the
// adds need no atomics; no add can wrap unless the task count does.
__device__ inline uint64_t binom_at(const CountArgs &a, int64_t n, int64_t r)
{
    return (r < 0 || n < 0 || r > n) ? 0ull : a.binom[(uint64_t)n * a.bstride + (uint64_t)r];
}

// The SCT from the root candidate set (all R task vertices, held h0, no
// pivots), or -- with init_x false -- from the candidate set already in X
// with h0 held and p0 pivot vertices (a subtree handed to one wave of a block).
template <int S>
__device__ uint32_t tri_lanes(const uint64_t *rows, uint32_t W, const uint64_t (&X)[S], uint32_t cx, uint32_t e2,
                              uint32_t *idx);
// (WIDE_SCT: four words close h = k-4 near-cliques too; the wide kernel has the
// registers for it, the one-wave four-word kernel keeps its budget)
template <int S, Kind KIND>
__device__ __attribute__((always_inline)) uint64_t pivot_reg(const CountArgs &a, uint32_t k, const uint64_t *rows, uint32_t R, uint32_t h0,
                              uint32_t *idx, uint64_t &nodes, uint32_t &ovf, uint32_t p0, uint64_t *crows, uint32_t wv = 0,
                              uint32_t nw = 1);

// the register walks of the deep block-wide kernel, functions of their own
template <int S>
__device__ __attribute__((noinline)) uint64_t pivot_deep(const CountArgs &a, uint32_t k, const uint64_t *rows, uint32_t R,
                                                         uint32_t h0, uint32_t *idx, uint64_t &nodes, uint32_t &ovf,
                                                         uint32_t p0, uint64_t *crows)
{
    return pivot_reg<S, WIDE_DEEP>(a, k, rows, R, h0, idx, nodes, ovf, p0, crows);
}

// triangles of G[X] with X in LDS (W words): the lane walks with the words in registers
// (inline, except the sixteen-word walk; build_rows_block likewise: what the wide
// kernel has inline is fixed here, it decides what it spills)
template <int S>
__device__ __attribute__((always_inline)) uint32_t tri_lds(const uint64_t *rows, uint32_t W, const uint64_t *X, uint32_t cx, uint32_t e2,
                            uint32_t *idx)
{
    uint64_t Xr[S];
#pragma unroll
    for (int w = 0; w < S; ++w) Xr[w] = (uint32_t)w < W ? uni64(X[w]) : 0ull;
    return tri_lanes<S>(rows, W, Xr, cx, e2, idx);
}

__device__ __attribute__((noinline)) uint32_t tri_lds16(const uint64_t *rows, uint32_t W, const uint64_t *X, uint32_t cx,
                                                        uint32_t e2, uint32_t *idx)
{
    return tri_lds<16>(rows, W, X, cx, e2, idx);
}

// (inline always: as a function of its own it saved and restored its registers for
// every entry of the wide kernel)
template <bool LOCAL, bool WIDE = false, Kind KIND = WIDE_SCT>
__device__ __attribute__((always_inline)) uint64_t pivot_count(const CountArgs &a, uint32_t P, uint32_t k, const uint64_t *rows, uint64_t *stk,
                                uint64_t *X, Scal *scal, uint32_t *cand, uint32_t R, uint32_t W, uint32_t h0,
                                uint64_t &nodes, uint32_t &ovf, uint64_t *lacc, uint32_t p0 = 0, bool init_x = true,
                                uint64_t *crows2 = nullptr, uint64_t *crows4 = nullptr)
{
    const int lane = lane_id();
    const uint64_t lt = lanemask_lt();
    const uint32_t wmax = a.wmax;
    const uint32_t NPp = 64 / P, part = lane / P, lip = lane % P;  // P lanes score one candidate
    const uint32_t lvl = LOCAL ? 4 * wmax : 2 * wmax;  // stack words per level
    uint64_t *Hc = X + wmax, *Pc = X + 2 * wmax;     // LOCAL: held / pivot sets of the node
    uint64_t acc = 0;
    // root candidate set = all R list vertices
    if (init_x)
        for (uint32_t w = lane; w < W; w += 64) {
            uint32_t lo = w * 64;
            X[w] = (R - lo >= 64) ? ~0ull : ((1ull << (R - lo)) - 1);
            if (LOCAL) Hc[w] = Pc[w] = 0;
        }
    sync_tree<WIDE>();
    int t = -1;
    bool pending = true;
    uint32_t h = h0, p = p0;
    uint64_t my_nodes = 0;
    // LOCAL: add vh to each held and vp to each pivot vertex of the node
    auto credit_hp = [&](uint64_t vh, uint64_t vp) {
        if (!LOCAL || (!vh && !vp)) return;
        for (uint32_t w = lane; w < W; w += 64) {
            if (vh)
                for (uint64_t x = Hc[w]; x; x &= x - 1) lacc[w * 64 + (uint32_t)__builtin_ctzll(x)] += vh;
            if (vp)
                for (uint64_t x = Pc[w]; x; x &= x - 1) lacc[w * 64 + (uint32_t)__builtin_ctzll(x)] += vp;
        }
    };
    for (;;) {
        if (pending) {
            pending = false;
            ++my_nodes;
            // candidate list of X (uniform word loop: the ballot of a word is the word)
            uint32_t cx = 0;
            for (uint32_t w = 0; w < W; ++w) {
                const uint64_t xw = X[w];
                if ((xw >> lane) & 1ull) cand[cx + (uint32_t)__popcll(xw & lt)] = w * 64 + (uint32_t)lane;
                cx += (uint32_t)__popcll(xw);
            }
            sync_tree<WIDE>();
            if (cx == 0) {
                if (k >= h && k - h <= p) {
                    uint64_t idx = (uint64_t)p * a.bstride + (k - h);
                    if (a.binom_ovf[idx]) ovf = 1;
                    add_checked(acc, a.binom[idx], ovf);
                    if (LOCAL) credit_hp(a.binom[idx], binom_at(a, (int64_t)p - 1, (int64_t)(k - h) - 1));
                }
            } else if (h >= k) {
                add_checked(acc, 1, ovf);
                if (LOCAL) credit_hp(1, 0);
            } else if (h + 1 == k) {
                add_checked(acc, (uint64_t)p + cx, ovf);
                if (LOCAL) {
                    credit_hp((uint64_t)p + cx, 1);
                    for (uint32_t c = lane; c < cx; c += 64) lacc[cand[c]] += 1;
                }
            } else if (!LOCAL && cx <= 64 && h + 3 <= k && h + p + cx >= k) {
                // at most 64 candidates left: re-encode the subtree one word per
                // row (row j of the subproblem = ballot of bit cand[j] over the
                // rows of the candidates) and finish it in sct64
                const uint32_t mine = lane < cx ? cand[lane] : 0u;
                uint64_t row1 = 0;
                for (uint32_t j = 0; j < cx; ++j) {
                    const uint32_t xj = cand[j];
                    const uint64_t wv = lane < cx ? rows[(uint64_t)mine * W + (xj >> 6)] : 0ull;
                    const uint64_t col = __ballot((wv >> (xj & 63)) & 1ull);
                    row1 = (lane == j) ? col : row1;
                }
                uint32_t lo = 0;
                const uint64_t part = sct64_wide<KIND>(a, k, row1, cx >= 64 ? ~0ull : ((1ull << cx) - 1), h, p, nodes, lo);
                add_checked(acc, wave_total(part, lo, ovf), ovf);
                --my_nodes;  // counted again as the subtree's root
            } else if (!LOCAL && crows4 && cx > 128 && cx <= 256 && h + 3 <= k && h + p + cx >= k) {
                // 129..256 candidates: re-encode three or four words per row the
                // same way and finish the subtree in the four-word register SCT
                // (which closes an h = k-4 near-clique at its root)
                const uint32_t Wc = (cx + 63) / 64;
                uint32_t mt[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) mt[t] = 64u * t + lane < cx ? cand[64u * t + lane] : 0u;
                for (uint32_t j = 0; j < cx; ++j) {
                    const uint32_t xj = cand[j];
                    uint64_t mine = 0;
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const uint64_t wv = 64u * t + lane < cx ? rows[(uint64_t)mt[t] * W + (xj >> 6)] : 0ull;
                        const uint64_t col = __ballot((wv >> (xj & 63)) & 1ull);
                        mine = lane == (uint32_t)t ? col : mine;
                    }
                    if (lane < Wc) crows4[(uint64_t)Wc * j + lane] = mine;
                }
                sync_tree<WIDE>();
                uint32_t lo = 0;
                const uint64_t part = KIND == WIDE_DEEP ? pivot_deep<4>(a, k, crows4, cx, h, cand, nodes, lo, p, crows2)
                                                       : pivot_reg<4, WIDE_SCT>(a, k, crows4, cx, h, cand, nodes, lo, p, crows2);
                add_checked(acc, wave_total(part, lo, ovf), ovf);
                --my_nodes;
            } else if (!LOCAL && crows2 && cx <= 128 && h + 3 <= k && h + p + cx >= k) {
                // 65..128 candidates: re-encode two words per row (word t of new
                // row j = ballot of bit cand[j] over the rows of candidates
                // 64t + lane) and finish the subtree in the two-word register SCT
                const uint32_t m0 = cand[lane], m1 = lane + 64 < cx ? cand[lane + 64] : 0u;
                for (uint32_t j = 0; j < cx; ++j) {
                    const uint32_t xj = cand[j];
                    const uint64_t w0 = rows[(uint64_t)m0 * W + (xj >> 6)];
                    const uint64_t w1 = lane + 64 < cx ? rows[(uint64_t)m1 * W + (xj >> 6)] : 0ull;
                    const uint64_t c0 = __ballot((w0 >> (xj & 63)) & 1ull), c1 = __ballot((w1 >> (xj & 63)) & 1ull);
                    if (lane < 2) crows2[2 * j + lane] = lane ? c1 : c0;
                }
                sync_tree<WIDE>();
                uint32_t lo = 0;
                const uint64_t part = KIND == WIDE_DEEP ? pivot_deep<2>(a, k, crows2, cx, h, cand, nodes, lo, p, nullptr)
                                                       : pivot_reg<2, WIDE_SCT>(a, k, crows2, cx, h, cand, nodes, lo, p, nullptr);
                add_checked(acc, wave_total(part, lo, ovf), ovf);
                --my_nodes;
            } else if (h + p + cx >= k) {
                // scores |X & row_j| for j in X: P lanes per candidate
                uint32_t best_s = 0, best_j = INF32;
                uint64_t sum_s = 0;
                for (uint32_t c = part; c < cx; c += NPp) {
                    const uint32_t j = cand[c];
                    const uint64_t *rj = rows + (uint64_t)j * W;
                    uint32_t sc = 0;
                    for (uint32_t w = lip; w < W; w += P) sc += (uint32_t)__popcll(X[w] & rj[w]);
                    sc = part_sum32(sc, P);
                    sum_s += sc;
                    if (best_j == INF32 || sc > best_s) {
                        best_s = sc;
                        best_j = j;
                    }
                    // h = k-2: x in X lies in C(p,1) + |X & row_x| of the subtree's cliques
                    if (LOCAL && h + 2 == k && lip == 0) lacc[j] += (uint64_t)p + sc;
                }
                uint64_t key = (lip == 0 && best_j != INF32) ? (((uint64_t)best_s << 32) | (INF32 - best_j)) : 0ull;
                key = wave_max64(key);
                uint32_t dummy = 0;
                const uint64_t tot_s = wave_sum64_checked(lip == 0 ? sum_s : 0ull, dummy);
                const uint32_t max_s = (uint32_t)(key >> 32);
                if (h + 2 == k) {
                    const uint64_t before = acc;
                    add_checked(acc, (uint64_t)p * (p - (p ? 1 : 0)) / 2, ovf);
                    add_checked(acc, (uint64_t)p * cx, ovf);
                    add_checked(acc, tot_s / 2, ovf);
                    if (LOCAL) credit_hp(acc - before, (p ? (uint64_t)p - 1 : 0) + cx);
                } else if (LOCAL && h + 3 == k) {
                    // h = k-3 with per-vertex credits: x in X lies in
                    // C(p,2) + p deg_X(x) + t_X(x) of the subtree's cliques (t_X(x) =
                    // edges of G[X] inside N(x), walked by the lane that owns x),
                    // a pivot in C(p-1,2) + (p-1)|X| + |E(X)|, a held vertex in all
                    sync_tree<WIDE>();  // (lacc of the score pass)
                    const uint64_t pp = p, cp2 = pp * (pp - (pp ? 1 : 0)) / 2;
                    uint64_t t3 = 0;
                    for (uint32_t c = lane; c < cx; c += 64) {
                        const uint32_t x = cand[c];
                        const uint64_t *rx = rows + (uint64_t)x * W;
                        uint64_t deg = 0, t2 = 0;
                        for (uint32_t w = 0; w < W; ++w) {
                            const uint64_t yw = X[w] & rx[w];
                            deg += (uint64_t)__popcll(yw);
                            for (uint64_t bits = yw; bits; bits &= bits - 1) {
                                const uint64_t *ry = rows + (uint64_t)(w * 64 + (uint32_t)__builtin_ctzll(bits)) * W;
                                for (uint32_t v = 0; v < W; ++v) t2 += (uint64_t)__popcll(X[v] & rx[v] & ry[v]);
                            }
                        }
                        lacc[x] += cp2 + pp * deg + t2 / 2;
                        t3 += t2 / 2;
                    }
                    uint32_t dummy = 0;
                    const uint64_t tri = wave_sum64_checked(t3, dummy) / 3;
                    const uint64_t e = tot_s / 2;
                    const uint64_t before = acc;
                    add_checked(acc, close_k3(a, p, cx, e, tri, ovf), ovf);
                    const uint64_t q = pp ? pp - 1 : 0;
                    credit_hp(acc - before, p ? q * (q - (q ? 1 : 0)) / 2 + q * cx + e : 0);
                    sync_tree<WIDE>();
                } else if (!LOCAL && h + 3 == k && W <= 16) {
                    // h = k-3: closed form with the triangles of G[X] (lane walks)
                    const uint32_t e2 = (uint32_t)tot_s;
                    const uint32_t tri = W <= 4 ? tri_lds<4>(rows, W, X, cx, e2, cand)
                                         : W <= 8 ? tri_lds<8>(rows, W, X, cx, e2, cand)
                                                  : tri_lds16(rows, W, X, cx, e2, cand);
                    add_checked(acc, close_k3(a, p, cx, tot_s / 2, tri, ovf), ovf);
                } else if (h + p + max_s + 1 >= k) {
                    const uint32_t pv = INF32 - (uint32_t)(key & 0xFFFFFFFFull);
                    ++t;
                    uint64_t *Cc = stk + (uint64_t)t * lvl, *B = Cc + wmax;
                    const uint64_t *rp = rows + (uint64_t)pv * W;
                    for (uint32_t w = lane; w < W; w += 64) {
                        uint64_t x = X[w];
                        Cc[w] = x;
                        B[w] = x & ~rp[w];
                        if (LOCAL) {  // level layout: Cc, B, held, pivots (wmax words each)
                            Cc[2 * wmax + w] = Hc[w];
                            Cc[3 * wmax + w] = Pc[w];
                        }
                    }
                    if (lane == 0) scal[t] = Scal{h, p, pv, 0};
                    sync_tree<WIDE>();
                }
            }
        }
        if (t < 0) break;
        // next branch of level t: non-pivot vertices first, the pivot last
        uint64_t *Cc = stk + (uint64_t)t * lvl, *B = Cc + wmax;
        const Scal sc = scal[t];
        uint32_t b = INF32;
        for (uint32_t w = lane; w < W; w += 64) {
            uint64_t x = B[w];
            if (w == (sc.pivot >> 6)) x &= ~(1ull << (sc.pivot & 63));
            if (x) {
                b = w * 64 + (uint32_t)__builtin_ctzll(x);
                break;
            }
        }
        b = wave_min32(b);
        const bool last = (b == INF32);
        if (last) b = sc.pivot;
        const uint64_t *rb = rows + (uint64_t)b * W;
        for (uint32_t w = lane; w < W; w += 64) {
            uint64_t c = Cc[w];
            X[w] = c & rb[w];
            if (LOCAL) {
                const uint64_t bit = (w == (b >> 6)) ? (1ull << (b & 63)) : 0ull;
                Hc[w] = Cc[2 * wmax + w] | (b != sc.pivot ? bit : 0ull);
                Pc[w] = Cc[3 * wmax + w] | (b == sc.pivot ? bit : 0ull);
            }
            if (w == (b >> 6)) {
                Cc[w] = c & ~(1ull << (b & 63));
                B[w] &= ~(1ull << (b & 63));
            }
        }
        sync_tree<WIDE>();
        h = sc.held + (b != sc.pivot ? 1u : 0u);
        p = sc.piv + (b == sc.pivot ? 1u : 0u);
        if (last) --t;  // the pivot branch replaces its level
        if (h <= k) pending = true;
    }
    if (lane == 0) nodes += my_nodes;
    return acc;
}

// ---- step 3c: pivoting with the bitmap in registers (R <= 64*S) -------------
// Lane l holds rows l, l+64, ..., l+64(S-1) of the bitmap (in VGPRs for the
// one- and two-word kernels; the four-word level reads them from LDS), so a
// pivot score is S*S AND+popcount on the lane's own rows; the rows a branch
// needs whole are broadcast-read from the LDS copy left by the build.  The SCT
// state is uniform: candidate set X and the level variables live in scalar
// registers, and the stack is spread across the lanes (lane t keeps level t in
// VGPRs, read back with v_readlane).  Arg-max and sums are wave reductions.

// word w of row b from the LDS copy (uniform address: a broadcast read)
__device__ inline uint64_t lds_row_word(const uint64_t *rows, uint32_t W, uint32_t b, int w)
{
    if ((uint32_t)w >= W) return 0ull;
    const uint64_t v = rows[(uint64_t)b * W + w];
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// Compaction: once a node's candidate set X has at most 64 vertices, its
// subtree is re-encoded as a 64-vertex subproblem (vertex j = the j-th member
// of X) and finished by sct64.  Lane i loads the full row of the i-th member
// from the LDS copy; new row j is the ballot over lanes of bit x_j of those
// rows (the bitmap is symmetric).  Cost ~ 6 instructions per member.
template <int S, Kind KIND>
__device__ uint64_t compact_and_count(const CountArgs &a, uint32_t k, const uint64_t *rows, uint32_t W,
                                      const uint64_t (&X)[S], uint32_t *idx, uint32_t h, uint32_t p,
                                      uint64_t &nodes, uint32_t &ovf)
{
    const uint32_t lane = (uint32_t)lane_id();
    const uint64_t lt = lanemask_lt();
    uint32_t before = 0, cx = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if ((X[s] >> lane) & 1ull) idx[before + (uint32_t)__popcll(X[s] & lt)] = 64u * s + lane;
        before += (uint32_t)__popcll(X[s]);
    }
    cx = before;
    sync_tree<true>();
    uint64_t o[S];
    const uint32_t mine = lane < cx ? idx[lane] : 0u;
#pragma unroll
    for (int w = 0; w < S; ++w) o[w] = (lane < cx && (uint32_t)w < W) ? rows[(uint64_t)mine * W + w] : 0ull;
    sync_tree<true>();  // idx is reused by the next compaction
    uint64_t row1 = 0;
    uint32_t j = 0;
#pragma unroll
    for (int w = 0; w < S; ++w) {
        for (uint64_t bits = X[w]; bits; bits &= bits - 1, ++j) {
            const uint32_t bj = (uint32_t)__builtin_ctzll(bits);
            const uint64_t col = __ballot((o[w] >> bj) & 1ull);
            row1 = (lane == j) ? col : row1;
        }
    }
    const uint64_t X1 = cx >= 64 ? ~0ull : ((1ull << cx) - 1);
    if constexpr (wide_kind(KIND)) return sct64_wide<KIND>(a, k, row1, X1, h, p, nodes, ovf);
    else return sct64<KIND>(a, k, row1, X1, h, p, nodes, ovf);
}

// Triangles of G[X] for X of up to 64*S vertices (rows of stride W in LDS) by
// lane-parallel forward walks.  Lane l takes the members l, 127-l, 128+l,
// 255-l, ... of X (in index order; the pairs balance the walks) and, for each
// member x, walks its forward neighbours F = N(x) & X above x lowest first:
// popping j leaves in F exactly the forward neighbours above j, so
// |F & N(j)| counts the triangles x < j < y once.  When more than half the
// pairs of X are edges the walk runs in the complement H instead (F = the
// non-neighbours above x) and Goodman's identity
//     t(G) = C(n,3) - 1/2 sum_x d_x (n-1-d_x) - t(H)
// gives the count; either way a lane walks min(density, 1-density) * n
// neighbours per member.  e2 = 2|E(X)|.  idx takes the member list.
template <int S>
__device__ uint32_t tri_lanes(const uint64_t *rows, uint32_t W, const uint64_t (&X)[S], uint32_t cx, uint32_t e2,
                              uint32_t *idx)
{
    const uint32_t lane = (uint32_t)lane_id();
    const uint64_t lt = lanemask_lt();
    uint32_t before = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if ((X[s] >> lane) & 1ull) idx[before + (uint32_t)__popcll(X[s] & lt)] = 64u * s + lane;
        before += (uint32_t)__popcll(X[s]);
    }
    sync_tree<true>();
    const bool comp = e2 > cx * (cx - 1) / 2;  // |E| > C(n,2)/2
    const uint64_t flip = comp ? ~0ull : 0ull;
    constexpr int NR = S > 2 ? S : 2;  // member slots per lane
    uint32_t val = 0, cnt = 0;
    int r = -1;
    uint64_t F[S];
#pragma unroll
    for (int w = 0; w < S; ++w) F[w] = 0;
    for (;;) {
        bool empty = true;
#pragma unroll
        for (int w = 0; w < S; ++w) empty = empty && F[w] == 0;
        while (empty && r < NR - 1) {  // the lane's next member
            ++r;
            const uint32_t m = (r & 1) ? (128u * (uint32_t)(r >> 1) + 127u - lane) : (128u * (uint32_t)(r >> 1) + lane);
            if (m >= cx) continue;
            const uint32_t x = idx[m], xw = x >> 6, xb = x & 63;
            uint32_t dg = 0;
#pragma unroll
            for (int w = 0; w < S; ++w) {
                const uint64_t rw = (uint32_t)w < W ? rows[(uint64_t)x * W + w] : 0ull;
                dg += (uint32_t)__popcll(X[w] & rw);
                const uint64_t above = (uint32_t)w > xw ? ~0ull : ((uint32_t)w < xw || xb == 63) ? 0ull : (~0ull << (xb + 1));
                F[w] = X[w] & (rw ^ flip) & above;
                empty = empty && F[w] == 0;
            }
            if (comp) val += dg * (cx - 1 - dg);
        }
        if (!__ballot(!empty)) break;
        if (!empty) {
            uint32_t j = 0;
            bool found = false;
#pragma unroll
            for (int w = 0; w < S; ++w) {
                if (!found && F[w]) {
                    j = 64u * w + (uint32_t)__builtin_ctzll(F[w]);
                    F[w] &= F[w] - 1;
                    found = true;
                }
            }
#pragma unroll
            for (int w = 0; w < S; ++w)
                if ((uint32_t)w < W) cnt += (uint32_t)__popcll(F[w] & (rows[(uint64_t)j * W + w] ^ flip));
        }
    }
    val += 2 * cnt;
    const uint32_t tot = (uint32_t)__builtin_amdgcn_readfirstlane((int)__ockl_wfred_add_u32(val));
    sync_tree<true>();  // idx is reused
    return comp ? cx * (cx - 1) * (cx - 2) / 6 - tot / 2 : tot / 2;
}

// The counts of close_word for X of up to 64*S vertices (rows of stride W in
// LDS): lane l takes the vertices l + 64s, s < S, with their complement rows in
// S words each.  With MM two words go through the matrix cores like one; else
// (over four words the operands would not fit the registers) a uniform walk
// over u in X keeps the four running sums of each vertex, summed over the
// lanes in 64 bits (C(256,4) * 24 does not fit 32).  Used at h = k-4 when X
// is a near-clique (the K4 walk, over the vertices in three or more complement
// triangles, stays short).
template <int S, bool MM>
__device__ CliqueCounts k34_complement_rows(const uint64_t *rows, uint32_t W, const uint64_t (&X)[S], uint32_t cx)
{
    const uint32_t lane = (uint32_t)lane_id();
    const int64_t n = cx;
    uint64_t Hl[S][S];
    int64_t d[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const uint32_t v = lane + 64u * s;
        const bool mem = (X[s] >> lane) & 1ull;
        d[s] = 0;
#pragma unroll
        for (int w = 0; w < S; ++w) {
            const uint64_t rw = (mem && (uint32_t)w < W) ? rows[(uint64_t)v * W + w] : ~0ull;
            Hl[s][w] = X[w] & ~rw & (w == s ? ~(1ull << lane) : ~0ull);
            d[s] += __popcll(Hl[s][w]);
        }
    }
    uint64_t T3[S];
    uint32_t s4 = 0, s3 = 0, s2 = 0;  // (MM)
    uint32_t q[S], qE[S], t2[S], sd[S];
    if constexpr (S == 2 && MM) {
        uint32_t H[4][4], t3[4], live = 0;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                halves((uint32_t)Hl[s][w], H[2 * s][2 * w], H[2 * s + 1][2 * w]);
                halves((uint32_t)(Hl[s][w] >> 32), H[2 * s][2 * w + 1], H[2 * s + 1][2 * w + 1]);
            }
#pragma unroll
        for (int J = 0; J < 4; ++J) live |= (uint32_t)(X[J >> 1] >> (32 * (J & 1))) ? 1u << J : 0u;
        complement_sums<4>(H, live, cx, s4, s3, s2, t3);
        T3[0] = ((uint64_t)t3[1] << 32) | t3[0];
        T3[1] = ((uint64_t)t3[3] << 32) | t3[2];
    } else {
#pragma unroll
        for (int s = 0; s < S; ++s) q[s] = qE[s] = t2[s] = sd[s] = 0;
#pragma unroll
        for (int wu = 0; wu < S; ++wu) {
            for (uint64_t bits = X[wu]; bits; bits &= bits - 1) {
                const uint32_t u = 64u * wu + (uint32_t)__builtin_ctzll(bits);
                uint64_t Hu[S];
                uint32_t du = 0;
#pragma unroll
                for (int w = 0; w < S; ++w) {
                    Hu[w] = X[w] & ~lds_row_word(rows, W, u, w) & (w == wu ? ~(1ull << (u & 63)) : ~0ull);
                    du += (uint32_t)__popcll(Hu[w]);
                }
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    uint32_t c = 0;
#pragma unroll
                    for (int w = 0; w < S; ++w) c += (uint32_t)__popcll(Hl[s][w] & Hu[w]);
                    const uint32_t c2 = c * c, in = (uint32_t)(Hu[s] >> lane) & 1u;
                    q[s] += c2;
                    qE[s] += in * c2;
                    t2[s] += in * c;
                    sd[s] += in * du;
                }
            }
        }
#pragma unroll
        for (int s = 0; s < S; ++s) T3[s] = __ballot(t2[s] >= 6);
    }
    // K4 of H among the vertices in >= 3 H-triangles (bit l of word s = vertex l + 64s)
    uint32_t nt3 = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) nt3 += (uint32_t)__popcll(T3[s]);
    int64_t k4acc[S];
#pragma unroll
    for (int s = 0; s < S; ++s) k4acc[s] = 0;
    if (nt3 >= 4) {
#pragma unroll
        for (int wu = 0; wu < S; ++wu) {
            for (uint64_t ub = T3[wu]; ub; ub &= ub - 1) {
                const uint32_t u = 64u * wu + (uint32_t)__builtin_ctzll(ub);
                uint64_t Hu[S];
#pragma unroll
                for (int w = 0; w < S; ++w) {
                    const uint64_t above = w > wu ? ~0ull : w < wu ? 0ull : ((u & 63) == 63 ? 0ull : (~0ull << ((u & 63) + 1)));
                    Hu[w] = T3[w] & ~lds_row_word(rows, W, u, w) & above;
                }
#pragma unroll
                for (int wv = 0; wv < S; ++wv) {
                    for (uint64_t vb = Hu[wv]; vb; vb &= vb - 1) {
                        const uint32_t v = 64u * wv + (uint32_t)__builtin_ctzll(vb);
                        uint64_t Sv[S];
                        uint32_t ns = 0;
#pragma unroll
                        for (int w = 0; w < S; ++w) {
                            const uint64_t above = w > wv ? ~0ull : w < wv ? 0ull : ((v & 63) == 63 ? 0ull : (~0ull << ((v & 63) + 1)));
                            Sv[w] = Hu[w] & ~lds_row_word(rows, W, v, w) & above;
                            ns += (uint32_t)__popcll(Sv[w]);
                        }
                        if (ns < 2) continue;
#pragma unroll
                        for (int s = 0; s < S; ++s) {
                            if (!((Sv[s] >> lane) & 1ull)) continue;
                            uint32_t z = 0;
#pragma unroll
                            for (int w = 0; w < S; ++w) {
                                const uint64_t above = w > s ? ~0ull : w < s ? 0ull : (lane == 63 ? 0ull : (~0ull << (lane + 1)));
                                z += (uint32_t)__popcll(Sv[w] & Hl[s][w] & above);
                            }
                            k4acc[s] += z;
                        }
                    }
                }
            }
        }
    }
    if constexpr (S == 2 && MM) {
        s4 += 24 * (uint32_t)(k4acc[0] + k4acc[1]);
        return complement_counts(cx, wave_sum32(s2) / 2, wave_sum32(s3), wave_sum32(s4));
    }
    int64_t c4l = 0, c3l = 0, sdl = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int64_t dd = d[s], t = t2[s] / 2, iq = q[s], iqE = qE[s], isd = sd[s], it2 = t2[s];
        c4l += 12 * (n - 4) * dd * (dd - 1) - 8 * (n - 3) * t - 12 * (dd - 1) * (isd - dd) + 24 * t -
               4 * dd * (dd - 1) * (dd - 2) + 3 * ((iq - dd * dd) - (isd - dd)) + 24 * t * (dd - 2) - 6 * (iqE - it2) +
               24 * k4acc[s];
        c3l += -3 * dd * (n - 1 - dd) - 2 * t;
        sdl += dd;
    }
    uint32_t dummy = 0;
    const int64_t s_d = (int64_t)uni64(wave_sum64_checked((uint64_t)sdl, dummy));
    const int64_t s_4 = (int64_t)uni64(wave_sum64_checked((uint64_t)c4l, dummy));
    const int64_t s_3 = (int64_t)uni64(wave_sum64_checked((uint64_t)c3l, dummy));
    const int64_t m = s_d / 2;
    const int64_t c4_24 = n * (n - 1) * (n - 2) * (n - 3) - 12 * m * (n - 2) * (n - 3) + 12 * m * (m - 1) + s_4;
    const int64_t c3_6 = n * (n - 1) * (n - 2) + s_3;
    CliqueCounts r;
    r.e = (uint32_t)(n * (n - 1) / 2 - m);
    r.c3 = (uint32_t)(c3_6 / 6);
    r.c4 = (uint32_t)(c4_24 / 24);
    return r;
}

// Compaction to two words: once a node of the four-word kernel has 65..128
// candidates, its subtree is re-encoded as a subproblem of at most 128
// vertices (vertex j = the j-th member of X) with two-word rows in crows and
// finished by the two-word register SCT, whose scores and closed forms cost a
// quarter of the four-word ones.  Lanes l and l+64 load the full rows of
// members l and l+64; word t of new row j is the ballot over lanes of bit x_j
// of the rows of members 64t + lane (the bitmap is symmetric).
template <int S, Kind KIND>
__device__ uint64_t compact2_and_count(const CountArgs &a, uint32_t k, const uint64_t *rows, uint32_t W,
                                       const uint64_t (&X)[S], uint32_t *idx, uint64_t *crows, uint32_t h, uint32_t p,
                                       uint64_t &nodes, uint32_t &ovf, uint32_t wv, uint32_t nw)
{
    const uint32_t lane = (uint32_t)lane_id();
    const uint64_t lt = lanemask_lt();
    uint32_t cx = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if ((X[s] >> lane) & 1ull) idx[cx + (uint32_t)__popcll(X[s] & lt)] = 64u * s + lane;
        cx += (uint32_t)__popcll(X[s]);
    }
    sync_tree<true>();
    const bool hi_ok = lane + 64 < cx;
    const uint32_t m0 = idx[lane], m1 = hi_ok ? idx[lane + 64] : 0u;  // cx > 64: every lane has a first member
    uint64_t o0[S], o1[S];
#pragma unroll
    for (int w = 0; w < S; ++w) {
        o0[w] = (uint32_t)w < W ? rows[(uint64_t)m0 * W + w] : 0ull;
        o1[w] = (hi_ok && (uint32_t)w < W) ? rows[(uint64_t)m1 * W + w] : 0ull;
    }
    sync_tree<true>();  // idx is reused by the two-word kernel
    uint32_t j = 0;
#pragma unroll
    for (int w = 0; w < S; ++w) {
        for (uint64_t bits = X[w]; bits; bits &= bits - 1, ++j) {
            const uint32_t bj = (uint32_t)__builtin_ctzll(bits);
            const uint64_t c0 = __ballot((o0[w] >> bj) & 1ull), c1 = __ballot((o1[w] >> bj) & 1ull);
            if (lane < 2) crows[2 * j + lane] = lane ? c1 : c0;
        }
    }
    sync_tree<true>();
    if constexpr (KIND == WIDE_DEEP) return pivot_deep<2>(a, k, crows, cx, h, idx, nodes, ovf, p, nullptr);
    else return pivot_reg<2, KIND>(a, k, crows, cx, h, idx, nodes, ovf, p, nullptr, wv, nw);
}

// nw > 1: this wave is number wv of nw that walk the same subtree, each with
// its own idx and crows: all of them walk the root's pivot chain (the nodes
// with h0 held), each takes every nw-th branch off it, and what a chain node
// itself adds is wave 0's.
template <int S, Kind KIND>
__device__ __attribute__((always_inline)) uint64_t pivot_reg(const CountArgs &a, uint32_t k, const uint64_t *rows, uint32_t R, uint32_t h0,
                              uint32_t *idx, uint64_t &nodes, uint32_t &ovf, uint32_t p0, uint64_t *crows, uint32_t wv,
                              uint32_t nw)
{
    const uint32_t lane = (uint32_t)lane_id();
    k = uni32(k);
    R = uni32(R);
    h0 = uni32(h0);
    p0 = uni32(p0);
    const uint32_t W = (R + 63) / 64;
    if (S == 1) {
        const uint64_t r1 = lane < R ? rows[lane] : 0ull;
        return sct64<LEAN>(a, k, r1, R >= 64 ? ~0ull : ((1ull << R) - 1), h0, p0, nodes, ovf);
    }
    // rows of the lane in VGPRs for the two-word kernel; the four-word level
    // (a small share of the work once subtrees of <= 128 candidates are
    // compacted) reads them from LDS, which keeps its register budget at the
    // two-word kernel's
    constexpr bool REG = S <= 2;
    constexpr int SR = REG ? S : 1;
    uint64_t row[SR][SR];
#pragma unroll
    for (int s = 0; s < SR; ++s) {
        const uint32_t j = lane + 64u * s;
#pragma unroll
        for (int w = 0; w < SR; ++w) row[s][w] = (REG && j < R && (uint32_t)w < W) ? rows[(uint64_t)j * W + w] : 0ull;
    }
    auto row_word = [&](int s, int w) -> uint64_t {
        if constexpr (REG) {
            return row[s][w];
        } else {
            const uint32_t j = lane + 64u * s;
            return (j < R && (uint32_t)w < W) ? rows[(uint64_t)j * W + w] : 0ull;
        }
    };
    uint64_t X[S], stkC[S], stkB[S];
    uint32_t stkM = 0;
#pragma unroll
    for (int w = 0; w < S; ++w) {
        const uint32_t lo = 64u * w;
        X[w] = R <= lo ? 0ull : (R - lo >= 64 ? ~0ull : ((1ull << (R - lo)) - 1));
        stkC[w] = stkB[w] = 0;
    }
    int t = -1;
    bool pending = true;
    uint32_t h = h0, p = p0, turn = wv;  // branches off the chain until the next of this wave's
    uint64_t acc = 0, my_nodes = 0;
    for (;;) {
        if (pending) {
            pending = false;
            const bool chain = h == h0, solo = !chain || wv == 0;
            uint32_t cx = 0;
#pragma unroll
            for (int w = 0; w < S; ++w) cx += (uint32_t)__popcll(X[w]);
            if (S == 4 && cx > 64 && cx <= 128 && h + 3 <= k && h + p + cx >= k) {
                // a subtree of at most 128 candidates: two words per row from here on
                add_checked(acc, compact2_and_count<S, KIND>(a, k, rows, W, X, idx, crows, h, p, nodes, ovf, chain ? wv : 0u,
                                                          chain ? nw : 1u),
                            ovf);
            } else if (cx <= 64 && cx > 0 && h + 3 <= k && h + p + cx >= k) {
                // a subtree of at most 64 candidates: one word per row from here on
                if (solo) add_checked(acc, compact_and_count<S, KIND>(a, k, rows, W, X, idx, h, p, nodes, ovf), ovf);
            } else if (my_nodes += solo, h + p + cx >= k) {
                // scores |X & row_j| of the lane's member rows; key packs
                // (score + 1, 0xFFFF - j), so the wave max names the smallest j of
                // the largest score
                const uint32_t need = k - h;  // (h <= k)
                uint32_t key = 0, lsum = 0;
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    uint32_t v = 0;
#pragma unroll
                    for (int w = 0; w < S; ++w) v += (uint32_t)__popcll(X[w] & row_word(s, w));
                    if ((X[s] >> lane) & 1ull) {
                        lsum += v;
                        const uint32_t kk = ((v + 1) << 16) | (0xFFFFu - (64u * s + lane));
                        key = kk > key ? kk : key;
                    }
                }
                uint32_t e2 = 0;  // twice the edges of G[X]
                if (need <= 4) e2 = wave_sum32(lsum);
                const bool near = (S == 2 || (S == 4 && wide_kind(KIND))) && need == 4 && 4 * (uint64_t)e2 >= 3ull * cx * (cx - 1);
                if (near || need <= 3 || cx == 0) {
                    if (!solo) break;  // (a chain node that closes ends the chain: the wave's branches are done)
                    // closed forms: h >= k-3, and h = k-4 over a near-clique (complement
                    // density <= 1/4)
                    const CloseTerm<wide_kind(KIND)> term(a, need, p);
                    CliqueCounts c{0, 0, 0};
                    if (near && cx) c = k34_complement_rows<S, KIND == MFMA || KIND == WIDE_DEEP>(rows, W, X, cx);
                    else if (need >= 2) c.e = e2 / 2;
                    if (need == 3 && cx) c.c3 = tri_lanes<S>(rows, W, X, cx, e2, idx);
                    term.add(acc, ovf, cx, c);
                } else if ((((key = (uint32_t)__builtin_amdgcn_readfirstlane((int)__ockl_wfred_max_u32(key))) >> 16) +
                            h + p) >= k) {  // (key >> 16) = max score + 1 bounds the clique inside X
                    const uint32_t pv = 0xFFFFu - (key & 0xFFFFu);
                    ++t;
#pragma unroll
                    for (int w = 0; w < S; ++w) {
                        const uint64_t bw = X[w] & ~lds_row_word(rows, W, pv, w);
                        stkC[w] = (lane == (uint32_t)t) ? X[w] : stkC[w];
                        stkB[w] = (lane == (uint32_t)t) ? bw : stkB[w];
                    }
                    const uint32_t M = h | (p << 8) | (pv << 24);
                    stkM = (lane == (uint32_t)t) ? M : stkM;
                }
            }
        }
        if (t < 0) break;
        // next branch of level t: non-pivot vertices first, the pivot last
        uint64_t Cc[S], B[S];
#pragma unroll
        for (int w = 0; w < S; ++w) {
            Cc[w] = rdlane64(stkC[w], (uint32_t)t);
            B[w] = rdlane64(stkB[w], (uint32_t)t);
        }
        const uint32_t M = (uint32_t)__builtin_amdgcn_readlane((int)stkM, t);
        const uint32_t hh = M & 0xFF, pp = (M >> 8) & 0xFFFF, pv = M >> 24;
        uint32_t b = INF32;
#pragma unroll
        for (int w = S - 1; w >= 0; --w) {
            uint64_t x = B[w];
            if ((uint32_t)w == (pv >> 6)) x &= ~(1ull << (pv & 63));
            if (x) b = 64u * w + (uint32_t)__builtin_ctzll(x);
        }
        const bool last = (b == INF32);
        if (last) b = pv;
        const uint32_t bs = b >> 6, bl = b & 63;
#pragma unroll
        for (int w = 0; w < S; ++w) X[w] = Cc[w] & lds_row_word(rows, W, b, w);
        h = hh + (b != pv ? 1u : 0u);
        p = pp + (b == pv ? 1u : 0u);
        bool mine = true;
        if (nw > 1 && hh == h0 && !last) {
            mine = turn == 0;
            turn = mine ? nw - 1 : turn - 1;
        }
        if (last) {
            --t;  // the pivot branch replaces its level
        } else {
#pragma unroll
            for (int w = 0; w < S; ++w) {
                if ((uint32_t)w == bs) {
                    Cc[w] &= ~(1ull << bl);
                    B[w] &= ~(1ull << bl);
                }
                stkC[w] = (lane == (uint32_t)t) ? Cc[w] : stkC[w];
                stkB[w] = (lane == (uint32_t)t) ? B[w] : stkB[w];
            }
        }
        if (h <= k) pending = mine;
    }
    if (lane == 0) nodes += my_nodes;
    return acc;
}

// ---- step 1: stage a task's vertex list in list[] ------------------------------
// node task: N+(u); edge task: T = N+(u) & N+(v), walking the shorter list and
// binary-searching the longer one, compacted with a ballot (ascending order).
__device__ __attribute__((always_inline)) uint32_t stage_task(const Cur &g, uint32_t task, uint32_t *list,
                                                              uint64_t &bytes)
{
    const int lane = lane_id();
    if (!g.gran) {
        const uint32_t b = g.rowptr[task], e = g.rowptr[task + 1];
        const uint32_t R = e - b;
        bytes += 8 + 4ull * R;
        for (uint32_t i = lane; i < R; i += 64) list[i] = g.col[b + i];
        return R;
    }
    const uint32_t u = g.src[task], v = g.col[task];
    const uint32_t ub = g.rowptr[u], ue = g.rowptr[u + 1], vb = g.rowptr[v], ve = g.rowptr[v + 1];
    const uint32_t du = ue - ub, dv = ve - vb;
    bytes += 24 + 4ull * (du + dv);
    const uint32_t *sa = g.col + (du <= dv ? ub : vb), *sb = g.col + (du <= dv ? vb : ub);
    const uint32_t la = min(du, dv), lb = max(du, dv);
    uint32_t cnt = 0;
    for (uint32_t i0 = 0; i0 < la; i0 += 64) {
        const uint32_t i = i0 + lane;
        bool hit = false;
        uint32_t x = 0;
        if (i < la) {
            x = sa[i];
            const uint32_t j = lower_bound_u32(sb, lb, x);
            hit = j < lb && sb[j] == x;
        }
        const uint64_t bal = __ballot(hit);
        if (hit) list[cnt + (uint32_t)__popcll(bal & lanemask_lt())] = x;
        cnt += (uint32_t)__popcll(bal);
    }
    return cnt;
}

// Steps 1 and 2 from the words of a.bits, for d+(u) <= BITS_ROW.  An edge task
// (u, v) reads T, as places in N+(u), in the word of (u, v); a node task takes
// all places.  The words of (u, w), w in T, hold every edge inside T, and one
// pass over T's places turns them into rows of the task: place j's bit of every
// member is one ballot, the in-neighbours of j, and a bit of each member's own
// out-neighbours (all that is wanted without FULL, as in build_rows).  IDS: list[]
// ends with the vertices.  Returns |T|; touches a wave's own LDS only.
// About 6 S instructions a member, where streaming the members' out-lists and
// searching the staged list took ~100 per 64 entries of them, for every edge
// task of u anew: without the tree walk, the launches of edge tasks of Chung-Lu
// n=1.2M at k=5 took 14.7 ms, with it 16.2, and from the words 4.3.
constexpr uint32_t BITS_ROW = 256;

template <int S, bool IDS, bool FULL = true>
__device__ __attribute__((always_inline)) uint32_t rows_from_bits(const CountArgs &a, const Cur &g, uint32_t task,
                                                                  uint32_t *list, uint64_t *rows, uint64_t &bytes)
{
    const uint32_t lane = (uint32_t)lane_id();
    const uint32_t u = g.gran ? uni32(g.src[task]) : task;
    const uint32_t ub = uni32(g.rowptr[u]), du = uni32(g.rowptr[u + 1]) - ub;
    uint64_t T[4], t0 = 0;
    if (lane * 64 < du) {
        const uint32_t left = du - lane * 64;
        t0 = g.gran ? a.bits[lane * a.bits_m + task] : left >= 64 ? ~0ull : (1ull << left) - 1;
    }
    uint32_t R = 0;
    if (g.gran) {
        const uint32_t v = uni32(g.col[task]);
        bytes += 24 + 4ull * (du + uni32(g.rowptr[v + 1]) - uni32(g.rowptr[v]));
    } else {
        bytes += 8 + 4ull * du;
    }
#pragma unroll
    for (int o = 0; o < 4; ++o) {
        T[o] = rdlane64(t0, o);
        if (in_mask(T[o])) list[R + (uint32_t)__popcll(T[o] & lanemask_lt())] = 64u * o + lane;
        R += (uint32_t)__popcll(T[o]);
    }
    sync_tree<true>();
    uint32_t r[S][8], id[S], d = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const uint32_t i = lane + 64u * s;
        const uint64_t at = (uint64_t)ub + (i < R ? list[i] : 0u);
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            const uint64_t x = i < R && 64u * o < du ? a.bits[o * a.bits_m + at] : 0ull;
            r[s][2 * o] = (uint32_t)x;
            r[s][2 * o + 1] = (uint32_t)(x >> 32);
        }
        id[s] = g.col[at];
        d += i < R ? g.rowptr[id[s] + 1] - g.rowptr[id[s]] : 0u;
    }
    bytes += 8ull * R + 4ull * wave_sum32(d);
    const uint32_t W = (R + 63) / 64;
    for (uint32_t i = lane; i < R * W; i += 64) rows[i] = 0;
    if (IDS) {
        sync_tree<true>();
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (lane + 64u * s < R) list[lane + 64u * s] = id[s];
    }
    sync_tree<true>();
    uint32_t jj = 0, out[S], inl[S], inh[S];
#pragma unroll
    for (int s = 0; s < S; ++s) out[s] = inl[s] = inh[s] = 0;
    uint32_t *half = reinterpret_cast<uint32_t *>(rows);
#pragma unroll
    for (int h = 0; h < 8; ++h) {
        for (uint32_t b = (uint32_t)(T[h >> 1] >> (32 * (h & 1))); b; b &= b - 1) {
            const uint32_t sh = (uint32_t)__builtin_ctz(b);
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const uint32_t bit = (r[s][h] >> sh) & 1u;
                out[s] |= bit << (jj & 31);
                if (!FULL) continue;
                const uint64_t in = __ballot(bit != 0);
                inl[s] = lane == (jj & 63) ? (uint32_t)in : inl[s];
                inh[s] = lane == (jj & 63) ? (uint32_t)(in >> 32) : inh[s];
            }
            ++jj;
            if ((jj & 31) == 0 || jj == R) {  // 32 columns: into the members' rows
                const uint32_t q = (jj - 1) >> 5;
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    if (lane + 64u * s < R) half[(lane + 64u * s) * 2 * W + q] |= out[s];
                    out[s] = 0;
                }
                sync_tree<true>();
                if (FULL && ((jj & 63) == 0 || jj == R)) {  // 64 members' in-neighbours: into their rows
                    const uint32_t j = (q >> 1) * 64 + lane;
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        if (j < R && (uint32_t)s < W) rows[(uint64_t)j * W + s] |= ((uint64_t)inh[s] << 32) | inl[s];
                        inl[s] = inh[s] = 0;
                    }
                    sync_tree<true>();
                }
            }
        }
    }
    return R;
}

// true if the task's rows come from a.bits
__device__ inline bool has_bits(const CountArgs &a, const Cur &g, uint32_t task)
{
    if (!a.bits || (g.gran && g.k == 3)) return false;
    const uint32_t u = g.gran ? uni32(g.src[task]) : task;
    return uni32(g.rowptr[u + 1]) - uni32(g.rowptr[u]) <= BITS_ROW;
}

// Per-wave bookkeeping shared by the kernels: the graph of the current task,
// the running count of the current query (flushed to qcount[] when the query
// changes and at the end), and the launch statistics.
struct WaveAcc {
    uint32_t q = INF32;
    uint64_t run = 0;      // this lane's share of the query's count
    uint32_t run_ovf = 0;  // this lane saw an overflow
    uint64_t bytes = 0, ntask = 0, nodes = 0, tmax = 0, tsum = 0;
};

// add a value every lane holds alike to the wave's running count
__device__ inline void run_add(WaveAcc &w, uint64_t v) { add_checked(w.run, lane_id() == 0 ? v : 0ull, w.run_ovf); }

__device__ __attribute__((always_inline)) void flush_query(const CountArgs &a, WaveAcc &w)
{
    if (w.q == INF32) return;
    // low and high half into sums of their own, in one instruction: neither can
    // wrap, so nothing has to come back, and the host joins them and sees an
    // overflow of the whole
    const int lane = lane_id();
    uint32_t ovf = 0;
    const uint64_t run = wave_total(w.run, w.run_ovf, ovf);
    if (lane < 2 && run) {
        uint64_t *at = a.single ? a.acc + (uint64_t)(blockIdx.x & a.acc_mask) * ACC + 6 * lane : a.qcount + 2ull * w.q + lane;
        atomicAdd((unsigned long long *)at, (unsigned long long)(lane ? run >> 32 : run & 0xFFFFFFFFull));
    }
    if (lane == 0 && ovf) atomicOr(&a.qovf[w.q], 1u);
    w.run = 0;
    w.run_ovf = 0;
}

__device__ __attribute__((always_inline)) Cur select_task(const CountArgs &a, uint64_t code, WaveAcc &w,
                                                          uint32_t &task)
{
    const uint32_t q = (uint32_t)(code >> 32);
    task = (uint32_t)code;
    if (q != w.q) {
        flush_query(a, w);
        w.q = q;
    }
    const QDesc d = a.qd[q];
    return Cur{d.rowptr, d.col, d.src, d.key, d.k, d.gran, d.psize};
}

__device__ __attribute__((always_inline)) void finish_wave(const CountArgs &a, WaveAcc &w)
{
    if (w.ntask == 0 && w.q == INF32) return;  // (a wide block's other waves have a query, no tasks)
    flush_query(a, w);
    uint32_t nd_wrap = 0;
    const uint64_t nd = wave_sum64_checked(w.nodes, nd_wrap);  // tree nodes are per-lane shares
    unsigned long long *acc = reinterpret_cast<unsigned long long *>(a.acc + (uint64_t)(blockIdx.x & a.acc_mask) * ACC);
    const int lane = lane_id();
    const uint64_t v = lane == 1 ? w.bytes : lane == 2 ? w.ntask : lane == 3 ? nd : lane == 5 ? w.tsum : 0ull;
    if (v) atomicAdd(&acc[lane], (unsigned long long)v);
    if (lane == 4) atomicMax(&acc[4], (unsigned long long)w.tmax);
}

__device__ inline uint32_t ld_head(uint32_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// The next chunk of tasks of a wave (every lane active).  Chunk c lies in
// queue c % NQUEUE and a wave takes from the heads of the queues in turn, so
// the queues go through the tasks side by side and a launch still starts its
// first (largest) tasks first; a wave that meets an empty queue finds the next
// that is not by one load per lane.  No chunk belongs to a block before the
// block runs: the launches of the size classes share the device, and the large
// tasks of blocks that had to wait for a slot started last (Chung-Lu n=1.2M,
// k=5..8: 330 -> 357 ms).
// One head -> NQUEUE heads: 970,000 node tasks of 96 small graphs at k = 4..7
// 3.8 -> 2.4 ms a call.
// Few tasks (host: at most DIRECT_ROUNDS per block slot) need no queue: the
// launch has one block per chunk and the device starts the blocks in order.
// 8,192 waves that look at the heads once and leave take 80 us: 9,208 node
// tasks of a 10,000-vertex graph 559 us with one head, 77 with NQUEUE, 23 so.
struct TaskQueue {
    uint32_t queue, left = 1;
    __device__ explicit TaskQueue(uint32_t block) : queue(block % NQUEUE) {}
};

// chunks of queue q
__device__ inline uint32_t queue_len(const CountArgs &a, uint32_t q)
{
    const uint32_t nchunk = (uint32_t)(((uint64_t)a.ntasks + (1u << a.chunk_log) - 1) >> a.chunk_log);
    return (nchunk + NQUEUE - 1 - q) / NQUEUE;
}

// the first task of the wave's next chunk, INF32 when there is none (moved to
// a scalar register: the callers' loops must be uniform)
__device__ __attribute__((always_inline)) uint32_t next_tasks(const CountArgs &a, TaskQueue &tq)
{
    const uint32_t lane = (uint32_t)lane_id();
    uint32_t c = INF32;
    if (a.direct) {
        const bool mine = tq.left && ((uint64_t)blockIdx.x << a.chunk_log) < a.ntasks;
        tq.left = 0;
        return mine ? uni32(blockIdx.x << a.chunk_log) : INF32;
    }
    // with fewer chunks than blocks (the host sizes a one-bin launch by the tasks
    // before binning) the blocks past their number leave the heads alone
    if (((uint64_t)blockIdx.x << a.chunk_log) >= a.ntasks) return INF32;
    for (;;) {
        uint32_t i = 0;
        if (lane == 0) i = atomicAdd(&a.qhead[tq.queue * QSTRIDE], 1u);
        i = uni32(i);
        if (i < queue_len(a, tq.queue)) {
            c = i * NQUEUE + tq.queue;
            tq.queue = (tq.queue + 1) % NQUEUE;
            break;
        }
        const uint32_t q = (tq.queue + lane) % NQUEUE;
        const bool open = lane < NQUEUE && ld_head(&a.qhead[q * QSTRIDE]) < queue_len(a, q);
        const uint64_t any = __ballot(open);
        if (!any) break;
        tq.queue = uni32((tq.queue + (uint32_t)__builtin_ctzll(any)) % NQUEUE);
    }
    return c == INF32 ? INF32 : uni32(c << a.chunk_log);
}

// register-bitmap pivoting kernel for tasks of at most 64*S vertices
// waves per SIMD the register budget is held to: 4 (<= 128 VGPRs), 8 for S = 1, 6 for S = 2 LEAN
template <int S, Kind KIND>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(S == 1 ? 8 : S == 2 && KIND == LEAN ? 6 : 4)))
void k_pivot_reg(CountArgs a)
{
    extern __shared__ uint64_t lds[];
    const int lane = lane_id();
    const Layout L = make_layout(a.rmax, a.wmax, 0, 0, true);
    uint32_t *list = reinterpret_cast<uint32_t *>(lds + L.list);
    uint32_t *offs = reinterpret_cast<uint32_t *>(lds + L.offs);
    uint32_t *starts = reinterpret_cast<uint32_t *>(lds + L.starts);
    uint32_t *keys = reinterpret_cast<uint32_t *>(lds + L.keys);
    uint64_t *rows = lds + L.rows;
    // (S = 4) the two-word rows of a compacted subtree, 128 x 2 words, over
    // list and starts (256 u32 each, dead once the bitmap is built)
    uint64_t *crows = lds + L.list;
    // the launch statistics are kept in LDS (lane 0; as acc, [6] the task's
    // start): they are touched once a task and would hold registers through it
    uint64_t *st = lds + L.misc;
    if (lane < 8) st[lane] = 0;
    WaveAcc w;
    if (a.ntasks_p) a.ntasks = uni32(*a.ntasks_p);
    TaskQueue tq(blockIdx.x);
    for (;;) {
        const uint32_t start = uni32(next_tasks(a, tq));
        if (start == INF32) break;
        const uint32_t stop = start + min(a.ntasks - start, 1u << a.chunk_log);
        for (uint32_t ti = start; ti < stop; ++ti) {
            if (lane == 0) st[6] = wall_clock64();
            uint32_t task;
            const Cur g = select_task(a, a.tasks[ti], w, task);
            uint64_t bytes = 0;
            const bool made = has_bits(a, g, task);
            const uint32_t R = made ? rows_from_bits<S, false>(a, g, task, list, rows, bytes)
                                    : stage_task(g, task, list, bytes);
            if (lane == 0) ++st[2];
            if (g.gran && g.k == 3) {  // an edge task at k=3 adds |T| (no bitmap needed)
                run_add(w, R);
                if (lane == 0) st[1] += bytes;
                __syncthreads();
                continue;
            }
            __syncthreads();
            if (!made) build_rows<true>(g, list, offs, starts, S == 1 ? keys : nullptr, rows, R, (R + 63) / 64, bytes);
            if (lane == 0) st[1] += bytes;
            uint64_t nodes = 0;
            add_checked(w.run, pivot_reg<S, KIND>(a, g.k, rows, R, g.gran ? 2u : 1u, offs, nodes, w.run_ovf, 0u, crows),
                        w.run_ovf);
            __syncthreads();
            if (lane == 0) {
                const uint64_t dt = wall_clock64() - st[6];
                st[3] += nodes;
                st[4] = dt > st[4] ? dt : st[4];
                st[5] += dt;
            }
        }
    }
    __syncthreads();
    w.bytes = st[1];
    w.ntask = st[2];
    w.nodes = lane == 0 ? st[3] : 0;
    w.tmax = st[4];
    w.tsum = st[5];
    finish_wave(a, w);
}

// ---- open queues: the serving loop's resident launches ------------------------
// The server keeps resident launches of k_pivot_open while queries arrive,
// each draining one FIFO queue of tasks.  A query is a segment (base, slot,
// task count) of the queue's task index space.  The host admits a query with
// plain stores to pinned host memory (the slot's descriptor, the segment,
// then the queue's task total with release), so admission needs no HIP call
// and no free CU while the launch runs.  A wave takes the next task index
// with one fetch-add on a device word; an index beyond what the device knows
// is published is held until it is (at most every POLL_TICKS one wave reads
// the host's total and raises the device's copy).  The host ends a launch by
// publishing a stop segment of one index per wave, so no index is ever
// handed back; a wave also ends by itself when it has held an index for
// safety_ticks (the host is gone).  A task's size is computed by the wave
// that stages it, and tasks below the clique part still to find add 0.  A
// wave keeps the running count of its slot and flushes it, with the number
// of tasks it finished, when the slot changes and before it waits; the flush
// that completes the slot's task count resets the slot's sums and writes the
// result to the slot's mailbox in host memory.
constexpr uint32_t OPEN_STOP = 0xFFFFFFFFu;  // slot of a stop segment

struct OpenArgs {
    CountArgs c;              // binom, qcount / qovf per slot
    uint64_t *counter;        // next task index
    uint64_t *known;          // task indices the device knows are published
    uint64_t *last_poll;      // wall clock of the last read of the host's total
    uint64_t *qdone;          // per slot: tasks finished
    const uint64_t *htotal;   // host: task indices published
    const uint64_t *hnseg;    // host: segments published
    const uint64_t *hseg;     // host: per segment base, then (slot << 32) | task count
    const OpenSlot *hslot;    // host: per slot descriptor
    OpenMail *mail;           // host: per slot result
    uint64_t safety_ticks;    // wall-clock ticks (100 MHz) a wave waits for its index at most
};

constexpr uint64_t POLL_TICKS = 200;  // 2 us

__device__ inline uint64_t ld_agent(uint64_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline uint64_t ld_host(const uint64_t *p)
{
    return __hip_atomic_load(const_cast<uint64_t *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// lane 0: read the host's task total, at most once per POLL_TICKS over the launch
__device__ inline void open_refresh(const OpenArgs &oa)
{
    const uint64_t now = wall_clock64();
    uint64_t last = ld_agent(oa.last_poll);
    if (now - last < POLL_TICKS) return;
    if (!__hip_atomic_compare_exchange_strong(oa.last_poll, &last, now, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT))
        return;
    const uint64_t h = ld_host(oa.htotal);
    if (h > ld_agent(oa.known)) __hip_atomic_fetch_max(oa.known, h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The segment a wave last resolved an index in (indices a wave takes only grow;
// desc = 0: none yet, no segment is empty).  It is in LDS, touched by lane 0
// alone: it is needed once a task and would hold registers through the tree
// walk.  With it there, statistics that nobody read, and the walk's step from 64- to
// 32-vertex words, the kernel spilled 176 bytes a lane, none now: 220 queries on
// Barabasi-Albert graphs of 3,000 to 100,000 vertices at k=4..8 5.3 -> 3.75 s, the
// 110th answer after 1080 -> 839 ms (spills of 88 bytes still made it 890).
struct SegCache {
    uint64_t seg, base, desc;
};

// lane 0: the segment holding published index i (segments are in base
// order; binary search in host memory from the cached one)
__device__ inline void open_resolve(const OpenArgs &oa, SegCache &sc, uint64_t i)
{
    if (i >= sc.base && i - sc.base < (uint32_t)sc.desc) return;
    uint64_t lo = sc.seg, hi = ld_host(oa.hnseg);  // base[lo] <= i < total
    while (hi - lo > 1) {
        const uint64_t mid = (lo + hi) >> 1;
        if (ld_host(oa.hseg + 2 * mid) <= i) lo = mid;
        else hi = mid;
    }
    sc.seg = lo;
    sc.base = ld_host(oa.hseg + 2 * lo);
    sc.desc = ld_host(oa.hseg + 2 * lo + 1);
}

// flush the running count of the current slot and the tasks finished for it;
// the flush that completes the slot publishes its result and resets its sums
__device__ __attribute__((always_inline)) void open_flush(const OpenArgs &oa, WaveAcc &w, uint32_t &pend,
                                                         uint64_t total, uint32_t seq)
{
    if (w.q == INF32) return;
    const CountArgs &a = oa.c;
    uint32_t run_ovf = 0;
    const uint64_t run = wave_total(w.run, w.run_ovf, run_ovf);
    if (lane_id() == 0 && pend) {
        const uint32_t q = w.q;
        const unsigned long long old = atomicAdd((unsigned long long *)&a.qcount[q], (unsigned long long)run);
        if (old + run < old || run_ovf) atomicOr(&a.qovf[q], 1u);
        const uint64_t before = __hip_atomic_fetch_add(&oa.qdone[q], (uint64_t)pend, __ATOMIC_ACQ_REL,
                                                       __HIP_MEMORY_SCOPE_AGENT);
        if (before + pend == total) {
            const uint64_t cnt = ld_agent(&a.qcount[q]);
            const uint32_t ovf = __hip_atomic_load(&a.qovf[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&a.qcount[q], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&a.qovf[q], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&oa.qdone[q], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&oa.mail[q].count, cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(&oa.mail[q].ovf, ovf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(&oa.mail[q].seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    w.run = 0;
    w.run_ovf = 0;
    pend = 0;
    w.q = INF32;  // the slot may hold another query by the time this wave sees it again
}

// the SCT of a task of at most 64 vertices, in words of 32 where it has no more
__device__ __attribute__((always_inline)) uint64_t open_tree(const CountArgs &a, uint32_t k, const uint64_t *rows, uint32_t R,
                                                            uint32_t h0, uint64_t &nodes, uint32_t &ovf)
{
    const uint32_t lane = (uint32_t)lane_id(), half = lane & 31;
    if (R <= 32)
        return sct_word<OPEN_SCT, uint32_t>(a, k, half < R ? (uint32_t)rows[half] : 0u, R == 32 ? ~0u : (1u << R) - 1, h0, 0u,
                                            nodes, ovf);
    return sct64<OPEN_SCT>(a, k, lane < R ? rows[lane] : 0ull, R == 64 ? ~0ull : (1ull << R) - 1, h0, 0u, nodes, ovf);
}

// one-word rows: every task of the graphs the resident launches take fits
// 64 vertices, so the kernel keeps the one-word kernel's register budget
// (eight waves per SIMD)
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8))) void k_pivot_open(OpenArgs oa)
{
    extern __shared__ uint64_t lds[];
    const CountArgs &a = oa.c;
    const int lane = lane_id();
    const Layout L = make_layout(a.rmax, a.wmax, 0, 0, true);
    uint32_t *list = reinterpret_cast<uint32_t *>(lds + L.list);
    uint32_t *offs = reinterpret_cast<uint32_t *>(lds + L.offs);
    uint32_t *starts = reinterpret_cast<uint32_t *>(lds + L.starts);
    uint64_t *rows = lds + L.rows;
    WaveAcc w;
    SegCache &sc = *reinterpret_cast<SegCache *>(lds + L.misc);
    if (lane == 0) sc = SegCache{0, 0, 0};
    uint32_t pend = 0, seq = 0;
    uint64_t total = 0;
    Cur g{};
    for (;;) {
        // lane 0 takes an index and waits until it is published
        uint64_t idx = 0;
        uint32_t ready = 0;
        if (lane == 0) {
            idx = __hip_atomic_fetch_add(oa.counter, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            open_refresh(oa);
            ready = idx < ld_agent(oa.known);
        }
        ready = uni32(__shfl(ready, 0, 64));
        if (!ready) {
            open_flush(oa, w, pend, total, seq);  // nothing held back while the wave waits
            if (lane == 0) {
                // back off while nothing is published: 1, 2, 4 .. 16 sleeps of
                // about 3.4 us between polls, so idle waves do not crowd the
                // device words (and the memory channel) the busy ones use
                const uint64_t t0 = wall_clock64();
                uint32_t naps = 1;
                while (!ready && wall_clock64() - t0 < oa.safety_ticks) {
                    for (uint32_t z = 0; z < naps; ++z) __builtin_amdgcn_s_sleep(127);
                    naps = naps < 16 ? 2 * naps : 16;
                    open_refresh(oa);
                    ready = idx < ld_agent(oa.known);
                }
            }
            ready = uni32(__shfl(ready, 0, 64));
            if (!ready) break;  // the host is gone: give up the index
        }
        uint32_t slot = 0, task = 0;
        if (lane == 0) {
            open_resolve(oa, sc, idx);
            slot = (uint32_t)(sc.desc >> 32);
            task = (uint32_t)(idx - sc.base);
        }
        slot = uni32(__shfl(slot, 0, 64));
        task = uni32(__shfl(task, 0, 64));
        if (slot == OPEN_STOP) break;
        if (slot != w.q) {
            open_flush(oa, w, pend, total, seq);
            w.q = slot;
            // the slot's descriptor, from host memory (lanes 0..5 read one word each)
            const uint64_t *hs = reinterpret_cast<const uint64_t *>(oa.hslot + slot);
            const uint64_t word = lane < (int)(sizeof(OpenSlot) / 8) ? ld_host(hs + lane) : 0ull;
            OpenSlot d;
            uint64_t *dw = reinterpret_cast<uint64_t *>(&d);
#pragma unroll
            for (int i = 0; i < (int)(sizeof(OpenSlot) / 8); ++i) dw[i] = uni64(rdlane64(word, (uint32_t)i));
            g = Cur{d.rowptr, d.col, d.src, nullptr, d.k, d.gran, 1u};
            total = d.total;
            seq = d.seq;
        }
        ++pend;
        uint64_t bytes = 0, nodes = 0;  // (statistics nobody asks for here)
        const uint32_t R = stage_task(g, task, list, bytes);
        const uint32_t need = g.gran ? g.k - 2 : g.k - 1;
        if (R >= need) {
            if (g.gran && g.k == 3) {
                run_add(w, R);
            } else {
                __syncthreads();
                build_rows<true>(g, list, offs, starts, nullptr, rows, R, (R + 63) / 64, bytes);
                add_checked(w.run,
                            open_tree(a, g.k, rows, R, g.gran ? 2u : 1u, nodes, w.run_ovf),
                            w.run_ovf);
            }
        }
        __syncthreads();
    }
    open_flush(oa, w, pend, total, seq);
}

// ---- the generic kernel: LDS (or HBM) bitmap, orientation or pivoting ------
// LOCAL: per-vertex counts of one query into a.local (the -m lkc path): each
// task zeroes its vertex accumulators, the traversal fills them, and at the
// end one HBM atomic per credited task vertex plus one per root vertex (the
// root lies in every clique of its task) publishes them.
template <bool LOCAL>
__device__ __attribute__((always_inline)) void publish_local(const CountArgs &a, const Cur &g, uint32_t task,
                                                             const uint32_t *list, const uint64_t *lacc, uint32_t R,
                                                             uint64_t task_count)
{
    if (!LOCAL) return;
    const int lane = lane_id();
    for (uint32_t i = lane; i < R; i += 64)
        if (lacc[i]) atomicAdd((unsigned long long *)&a.local[list[i]], (unsigned long long)lacc[i]);
    if (lane == 0 && task_count) {
        const uint32_t u = g.gran ? g.src[task] : task;
        atomicAdd((unsigned long long *)&a.local[u], (unsigned long long)task_count);
        if (g.gran) atomicAdd((unsigned long long *)&a.local[g.col[task]], (unsigned long long)task_count);
    }
}

constexpr uint32_t LOCAL_CACHE_LOG = 8, LOCAL_CACHE = 1u << LOCAL_CACHE_LOG;  // per wave: sum, vertex, owner lane

// Per-vertex counts of pivoting tasks of at most 64 * S vertices, one wave a task,
// the credits in registers.  The generic kernel kept X, the held and pivot sets,
// every level's copies and the credits in LDS behind block barriers.
// The credits of a task go to a direct-mapped table of sums per wave in LDS, and
// to HBM when another vertex takes the entry: the vertices of neighbouring tasks
// are largely the same, and the few high in the order are in most of them, so
// that their atomics would queue at one address.
// Chung-Lu n=300,000, m=1.96M, k=6, edge tasks: generic kernel 9.1 ms, credits
// straight to HBM 5.5, through tables of 128 / 256 / 512 entries 3.75 / 3.35 /
// 3.9 (512 cost resident waves); without the atomics at all it took 2.9.
// Two words (S = 2) against the generic kernel: node tasks of the same graph,
// 2,055 of them above 64 vertices, 28.1 -> 8.0 ms for the launch.
template <int S>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(S == 1 ? 6 : 4))) void k_local_reg(CountArgs a)
{
    extern __shared__ uint64_t lds[];
    const int lane = lane_id();
    const Layout L = make_layout(a.rmax, a.wmax, 0, 0, true);
    uint32_t *list = reinterpret_cast<uint32_t *>(lds + L.list);
    uint32_t *offs = reinterpret_cast<uint32_t *>(lds + L.offs);
    uint32_t *starts = reinterpret_cast<uint32_t *>(lds + L.starts);
    uint32_t *keys = reinterpret_cast<uint32_t *>(lds + L.keys);
    uint64_t *rows = lds + L.rows;
    uint64_t *csum = lds + L.total;
    uint32_t *ckey = reinterpret_cast<uint32_t *>(csum + LOCAL_CACHE);
    uint8_t *cown = reinterpret_cast<uint8_t *>(ckey + LOCAL_CACHE);
    for (uint32_t i = lane; i < LOCAL_CACHE; i += 64) {
        csum[i] = 0;
        ckey[i] = INF32;
    }
    WaveAcc w;
    if (a.ntasks_p) a.ntasks = uni32(*a.ntasks_p);
    TaskQueue tq(blockIdx.x);
    for (;;) {
        const uint32_t start = uni32(next_tasks(a, tq));
        if (start == INF32) break;
        const uint32_t stop = start + min(a.ntasks - start, 1u << a.chunk_log);
        for (uint32_t ti = start; ti < stop; ++ti) {
            const uint64_t t0 = wall_clock64();
            uint32_t task;
            const Cur g = select_task(a, a.tasks[ti], w, task);
            ++w.ntask;
            const bool made = has_bits(a, g, task);
            const uint32_t R = made ? rows_from_bits<S, true>(a, g, task, list, rows, w.bytes)
                                    : stage_task(g, task, list, w.bytes);
            uint64_t credit[S] = {}, count = 0;
            __syncthreads();
            if (g.gran && g.k == 3) {  // an edge task at k=3 adds |T| (no bitmap needed)
                count = R;
#pragma unroll
                for (int s = 0; s < S; ++s) credit[s] = 1;
            } else {
                if (!made) build_rows<true>(g, list, offs, starts, S == 1 ? keys : nullptr, rows, R, S, w.bytes);
                uint64_t row[S][S];
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int o = 0; o < S; ++o)
                        row[s][o] = (uint32_t)lane + 64u * s < R ? rows[((uint32_t)lane + 64u * s) * S + o] : 0ull;
                count = sct_local<S>(a, g.k, row, R, g.gran ? 2u : 1u, credit, w.nodes, w.run_ovf);
            }
            run_add(w, count);
            // a sum per lane: the vertices of the task, then its root vertices (those
            // by themselves when the task leaves no lane free)
            const uint32_t roots = g.gran ? 2u : 1u, last = R - min(R, 64u * (S - 1));
            const uint32_t rt = (uint32_t)lane - (last + roots <= 64 ? last : 0u);
            const uint32_t root = rt == 0 ? (g.gran ? g.src[task] : task) : rt == 1 && g.gran ? g.col[task] : INF32;
            if (last + roots > 64 && root != INF32 && count)
                atomicAdd((unsigned long long *)&a.local[root], (unsigned long long)count);
#pragma unroll
            for (int s = 0; s < S; ++s) {
                uint32_t v = (uint32_t)lane + 64u * s < R ? list[lane + 64 * s] : INF32;
                uint64_t c = credit[s];
                if (s == S - 1 && last + roots <= 64 && (uint32_t)lane >= last && root != INF32) {
                    v = root;
                    c = count;
                }
                const bool has = v != INF32 && c;
                const uint32_t slot = (v * 0x9E3779B1u) >> (32 - LOCAL_CACHE_LOG);
                if (has) cown[slot] = (uint8_t)lane;
                __syncthreads();
                if (has) {
                    uint32_t ov = v;
                    uint64_t oc = c;
                    if (cown[slot] == (uint8_t)lane) {
                        const uint32_t kv = ckey[slot];
                        const uint64_t kc = csum[slot];
                        csum[slot] = kv == v ? kc + c : c;
                        ckey[slot] = v;
                        ov = kv == v ? INF32 : kv;
                        oc = kc;
                    }
                    if (ov != INF32) atomicAdd((unsigned long long *)&a.local[ov], (unsigned long long)oc);
                }
                __syncthreads();
            }
            const uint64_t dt = wall_clock64() - t0;
            w.tmax = dt > w.tmax ? dt : w.tmax;
            w.tsum += dt;
        }
    }
    for (uint32_t i = lane; i < LOCAL_CACHE; i += 64)
        if (ckey[i] != INF32) atomicAdd((unsigned long long *)&a.local[ckey[i]], (unsigned long long)csum[i]);
    finish_wave(a, w);
}

// SMALL: the orientation's tasks of at most 128 vertices in LDS, whose rows may come
// from the adjacency words (Chung-Lu n=200,000, k=5, edge tasks 0.95 -> 0.71 ms a
// call, n=300,000, k=4 1.27 -> 0.61) or pair by pair.  The registers of both ways
// cost the larger tasks, whose DFS is the time: R-MAT scale 18, node tasks at k=5
// in degeneracy order 218 ms with them in every instance, 205 so.
template <bool PIVOT, bool GLOBAL, bool LOCAL, bool SMALL>
__global__ __launch_bounds__(64) void k_count(CountArgs a)
{
    extern __shared__ uint64_t lds[];
    const int lane = lane_id();
    uint64_t *ws = GLOBAL ? a.gscr + (uint64_t)blockIdx.x * a.gscr_words : lds;
    const Layout L = make_layout(a.rmax, a.wmax, a.levels, a.nparts, PIVOT, LOCAL);
    uint32_t *misc = reinterpret_cast<uint32_t *>(ws + L.misc);
    uint32_t *list = reinterpret_cast<uint32_t *>(ws + L.list);
    uint32_t *offs = reinterpret_cast<uint32_t *>(ws + L.offs);
    uint32_t *starts = reinterpret_cast<uint32_t *>(ws + L.starts);
    uint32_t *keys = SMALL && a.rmax <= PAIR_ROWS ? reinterpret_cast<uint32_t *>(ws + L.keys) : nullptr;
    uint64_t *rows = ws + L.rows;
    uint64_t *stk = ws + L.stk;
    uint64_t *X = ws + L.x;
    Scal *scal = reinterpret_cast<Scal *>(ws + L.scal);
    uint64_t *lacc = ws + L.lacc;
    uint32_t *path = reinterpret_cast<uint32_t *>(ws + L.path);
    WaveAcc w;
    if (a.ntasks_p) a.ntasks = uni32(*a.ntasks_p);
    TaskQueue tq(blockIdx.x);
    for (;;) {
        const uint32_t start = uni32(next_tasks(a, tq));
        if (start == INF32) break;
        const uint32_t stop = start + min(a.ntasks - start, 1u << a.chunk_log);
        for (uint32_t ti = start; ti < stop; ++ti) {
            const uint64_t t0 = wall_clock64();
            uint32_t task;
            const Cur g = select_task(a, a.tasks[ti], w, task);
            const uint32_t k = g.k;
            ++w.ntask;
            const bool made = SMALL && has_bits(a, g, task);
            const uint32_t R = !made          ? stage_task(g, task, list, w.bytes)
                               : a.rmax <= 64 ? rows_from_bits<1, LOCAL, false>(a, g, task, list, rows, w.bytes)
                                              : rows_from_bits<2, LOCAL, false>(a, g, task, list, rows, w.bytes);
            if (LOCAL)
                for (uint32_t i = lane; i < R; i += 64) lacc[i] = 0;
            if (g.gran && k == 3) {  // an edge task at k=3 adds |T| (no bitmap needed)
                run_add(w, R);
                if (LOCAL) {
                    for (uint32_t i = lane; i < R; i += 64) lacc[i] = 1;
                    __syncthreads();
                    publish_local<LOCAL>(a, g, task, list, lacc, R, R);
                    __syncthreads();
                }
                continue;
            }
            if (lane == 0) misc[0] = 0;
            __syncthreads();
            const uint32_t W = (R + 63) / 64;
            uint64_t task_count;
            if (!PIVOT) {
                // (k-1)-cliques of the DAG on N+(u) / (k-2)-cliques of the DAG on T
                if (!made) build_rows<false>(g, list, offs, starts, keys, rows, R, W, w.bytes);
                uint32_t povf = 0;
                uint64_t part = orient_count<LOCAL>(a, g.psize, rows, stk, misc, R, W, g.gran ? k - 2 : k - 1,
                                                    w.nodes, povf, lacc, path);
                task_count = LOCAL ? wave_sum64_checked(part, povf) : 0ull;
                w.run_ovf |= povf;
                add_checked(w.run, part, w.run_ovf);
            } else {
                // SCT rooted at the node (held 1) or the edge (held 2)
                build_rows<true>(g, list, offs, starts, keys, rows, R, W, w.bytes);
                task_count = pivot_count<LOCAL>(a, g.psize, k, rows, stk, X, scal, offs, R, W, g.gran ? 2u : 1u,
                                                w.nodes, w.run_ovf, lacc);
                run_add(w, task_count);
            }
            __syncthreads();
            publish_local<LOCAL>(a, g, task, list, lacc, R, task_count);
            if (LOCAL) __syncthreads();
            const uint64_t dt = wall_clock64() - t0;
            w.tmax = dt > w.tmax ? dt : w.tmax;
            w.tsum += dt;
        }
    }
    finish_wave(a, w);
}

// ---- the wide kernel: one block of NW waves per large task -----------------
// Tasks of 257..1024 vertices (LDS) and above (HBM slice) hold a bitmap of up
// to 128 KB, so a one-wave block leaves most of a CU idle.  Here the NW waves
// of a block share one task: they build its bitmap together, then wave 0
// walks the SCT's pivot chain from the root (node j = the j-th pivot child:
// h0 held, j pivots) down to a node of at most 64 candidates or to the chain
// cap, and every non-pivot branch b hanging off chain node j -- candidates
// (X_j minus the non-pivot branches of j before b) & N(b), h0+1 held, j
// pivots -- plus the chain's last node become entries that the waves take
// from an LDS counter and finish with their own stacks
// (pivot_count<false, true>).  The chain is the part of the tree that one
// wave would otherwise walk alone: the cap is 32 levels when the chain lives
// in LDS and the whole chain (up to 1024 levels) in the HBM slice.  Blocks
// have up to 8 waves (512 threads), which leaves the register SCT that
// pivot_count hands subtrees of <= 256 candidates to its full register
// budget; each wave has its own LDS areas for those subtrees' rows.
struct WideLayout {
    uint64_t ctl, list, offs, starts, chain, rows, wave, per_wave, total;
};

__host__ __device__ inline WideLayout make_wide_layout(uint32_t rmax, uint32_t wmax, uint32_t levels, uint32_t nw,
                                                       uint32_t chain)
{
    WideLayout L;
    L.ctl = 0;
    L.list = L.ctl + 8;
    L.offs = L.list + (rmax + 1) / 2;
    L.starts = L.offs + (rmax + 2) / 2;
    L.chain = L.starts + (rmax + 1) / 2;         // per chain level: candidates, non-pivot branches
    L.rows = L.chain + (uint64_t)chain * 2 * wmax;
    L.wave = L.rows + (uint64_t)rmax * wmax;
    // + the rows of compacted subtrees: 128 x 2 and 256 x 4 words
    L.per_wave = (uint64_t)levels * 2 * wmax + wmax + (uint64_t)levels * 2 + (rmax + 1) / 2 + 256 + 1024;
    L.total = L.wave + L.per_wave * nw;
    return L;
}

// bitmap rows of the task by every thread of the block (build_rows with the
// row offsets scanned by wave 0)
__device__ __attribute__((noinline)) void build_rows_block(const Cur &g, const uint32_t *list, uint32_t *offs, uint32_t *starts, uint64_t *rows,
                                 uint32_t R, uint32_t W, uint64_t &bytes)
{
    const uint32_t tid = threadIdx.x, nt = blockDim.x, lane = tid & 63;
    for (uint32_t i = tid; i < R * W; i += nt) rows[i] = 0;
    if (tid < 64) {
        uint32_t carry = 0;
        for (uint32_t base = 0; base < R; base += 64) {
            const uint32_t i = base + lane;
            uint32_t d = 0;
            if (i < R) {
                const uint32_t w = list[i];
                const uint32_t st = g.rowptr[w];
                d = g.rowptr[w + 1] - st;
                starts[i] = st;
            }
            const uint32_t inc = wave_incl_scan32(d);
            if (i < R) offs[i] = carry + inc - d;
            carry += __shfl(inc, 63, 64);
        }
        if (lane == 0) offs[R] = carry;
        bytes += 8ull * R + 4ull * carry;
    }
    __syncthreads();
    const uint32_t total = offs[R];
    const uint32_t lo_v = list[0], hi_v = list[R - 1];
    uint32_t lo = 0;  // row of entry f (f only grows)
    for (uint32_t f = tid; f < total; f += nt) {
        while (offs[lo + 1] <= f) ++lo;
        const uint32_t x = g.col[starts[lo] + (f - offs[lo])];
        if (x < lo_v || x > hi_v) continue;
        const uint32_t j = lower_bound_u32(list, R, x);
        if (j < R && list[j] == x) {
            atomicOr((unsigned long long *)&rows[(uint64_t)lo * W + (j >> 6)], 1ull << (j & 63));
            atomicOr((unsigned long long *)&rows[(uint64_t)j * W + (lo >> 6)], 1ull << (lo & 63));
        }
    }
    __syncthreads();
}

// Tasks of 129..256 vertices, one block of NW waves each: the waves build the
// bitmap together, share it in LDS and split the SCT by the branches off its
// root chain (pivot_reg).  For launches that are over with their longest task
// (at most BLOCK_TASKS_PER_CU tasks per CU, what the one-wave kernel holds at
// once): 2,825 node tasks of an R-MAT graph at k=5, 3.6 -> 3.2 ms with two
// waves, 3.5 with four (each walks the chain again).  With many tasks the
// second walk of the chain only costs (37,889 edge tasks of Chung-Lu n=1.2M
// at k=5..8: 242 -> 254 ms in all with two waves, 280 with four).
constexpr uint32_t BLOCK_WAVES = 2, BLOCK_TASKS_PER_CU = 14;

struct BlockLayout {
    uint64_t st, ctl, list, starts, offs, rows, wave, per_wave, total;
};

__host__ __device__ inline BlockLayout make_block_layout(uint32_t nw)
{
    BlockLayout L;
    L.st = 0;
    L.ctl = 8;
    L.list = L.ctl + 2;
    L.starts = L.list + 128;
    L.offs = L.starts + 128;
    L.rows = L.offs + 129;
    L.wave = L.rows + 256 * 4;
    L.per_wave = 128 + 256;  // member list (256 u32), two-word rows of a compacted subtree (128 x 2)
    L.total = L.wave + L.per_wave * nw;
    return L;
}

template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void k_pivot_block(CountArgs a)
{
    extern __shared__ uint64_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = uni32(tid >> 6);
    const BlockLayout L = make_block_layout(NW);
    uint64_t *st = lds + L.st;  // launch statistics (as acc, [6] the task's start)
    uint32_t *ctl = reinterpret_cast<uint32_t *>(lds + L.ctl);
    uint32_t *list = reinterpret_cast<uint32_t *>(lds + L.list);
    uint32_t *starts = reinterpret_cast<uint32_t *>(lds + L.starts);
    uint32_t *offs = reinterpret_cast<uint32_t *>(lds + L.offs);
    uint64_t *rows = lds + L.rows;
    uint32_t *idx = reinterpret_cast<uint32_t *>(lds + L.wave + wv * L.per_wave);
    uint64_t *crows = lds + L.wave + wv * L.per_wave + 128;
    if (tid < 8) st[tid] = 0;
    WaveAcc w;
    TaskQueue tq(blockIdx.x);
    for (;;) {
        if (wv == 0) {
            const uint32_t start = next_tasks(a, tq);
            if (lane == 0) ctl[0] = start;
        }
        __syncthreads();
        const uint32_t ti = uni32(ctl[0]);
        if (ti == INF32) break;
        uint32_t task;
        const Cur g = select_task(a, a.tasks[ti], w, task);
        uint64_t bytes = 0;
        if (wv == 0) {
            if (lane == 0) st[6] = wall_clock64();
            const bool made = has_bits(a, g, task);
            const uint32_t r = made ? rows_from_bits<4, false>(a, g, task, list, rows, bytes)
                                    : stage_task(g, task, list, bytes);
            if (lane == 0) {
                ctl[1] = r;
                ctl[2] = made ? 1u : 0u;
            }
        }
        __syncthreads();
        const uint32_t R = uni32(ctl[1]);
        if (g.gran && g.k == 3) {  // an edge task at k=3 adds |T| (no bitmap needed)
            if (wv == 0) run_add(w, R);
        } else {
            if (!uni32(ctl[2])) build_rows_block(g, list, offs, starts, rows, R, (R + 63) / 64, bytes);
            uint64_t nodes = 0;
            add_checked(w.run, pivot_reg<4, MFMA>(a, g.k, rows, R, g.gran ? 2u : 1u, idx, nodes, w.run_ovf, 0u, crows, wv, NW),
                        w.run_ovf);
            if (lane == 0) atomicAdd((unsigned long long *)&st[3], (unsigned long long)nodes);
        }
        __syncthreads();
        if (tid == 0) {
            st[1] += bytes;
            ++st[2];
            if (!(g.gran && g.k == 3)) {
                const uint64_t dt = wall_clock64() - st[6];
                st[4] = dt > st[4] ? dt : st[4];
                st[5] += dt * NW;
            }
        }
    }
    if (wv == 0) {
        w.bytes = st[1];
        w.ntask = st[2];
        w.nodes = lane == 0 ? st[3] : 0;
        w.tmax = st[4];
        w.tsum = st[5];
    }
    finish_wave(a, w);
}

template <bool GLOBAL, Kind KIND>
__global__ __launch_bounds__(512) void k_pivot_wide(CountArgs a)
{
    extern __shared__ uint64_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, NW = blockDim.x >> 6;
    uint64_t *ws = GLOBAL ? a.gscr + (uint64_t)blockIdx.x * a.gscr_words : lds;
    const WideLayout L = make_wide_layout(a.rmax, a.wmax, a.levels, NW, a.chain);
    uint32_t *ctl = reinterpret_cast<uint32_t *>(ws + L.ctl);  // task, R, next branch, branches, pivot
    uint32_t *list = reinterpret_cast<uint32_t *>(ws + L.list);
    uint32_t *offs = reinterpret_cast<uint32_t *>(ws + L.offs);  // row offsets, then the entries (j << 16 | b)
    uint32_t *starts = reinterpret_cast<uint32_t *>(ws + L.starts);
    uint64_t *rows = ws + L.rows;
    uint64_t *stk = ws + L.wave + (uint64_t)wv * L.per_wave;
    uint64_t *X = stk + (uint64_t)a.levels * 2 * a.wmax;
    Scal *scal = reinterpret_cast<Scal *>(X + a.wmax);
    uint32_t *cand = reinterpret_cast<uint32_t *>(X + a.wmax + (uint64_t)a.levels * 2);
    uint64_t *crows2 = X + a.wmax + (uint64_t)a.levels * 2 + (a.rmax + 1) / 2;  // 128 x 2 words
    uint64_t *crows4 = crows2 + 256;                                           // 256 x 4 words
    WaveAcc w;
    TaskQueue tq(blockIdx.x);
    uint64_t no_bytes = 0;
    for (;;) {
        if (wv == 0) {  // (one task per grab)
            const uint32_t start = next_tasks(a, tq);
            if (lane == 0) ctl[0] = start;
        }
        __syncthreads();
        const uint32_t ti = ctl[0];
        if (ti == INF32) break;
        const uint64_t t0 = wall_clock64();
        uint32_t task;
        const Cur g = select_task(a, a.tasks[ti], w, task);
        const uint32_t k = g.k, h0 = g.gran ? 2u : 1u;
        if (wv == 0) {
            const uint32_t r = stage_task(g, task, list, w.bytes);
            if (lane == 0) ctl[1] = r;
            ++w.ntask;
        }
        __syncthreads();
        const uint32_t R = ctl[1], W = (R + 63) / 64;
        if (g.gran && k == 3) {  // an edge task at k=3 adds |T| (no bitmap needed)
            if (wv == 0) run_add(w, R);
            __syncthreads();
            continue;
        }
        build_rows_block(g, list, offs, starts, rows, R, W, wv == 0 ? w.bytes : no_bytes);
        // the pivot chain, by wave 0: closed forms at the root, or the entries
        uint64_t *chX = ws + L.chain, *chB = chX + a.wmax;  // level j at chX + 2 j wmax
        if (wv == 0) {
            uint32_t ne = 0, endj = INF32;
            for (uint32_t x = lane; x < W; x += 64) {
                const uint32_t lo = x * 64;
                chX[x] = (R - lo >= 64) ? ~0ull : ((1ull << (R - lo)) - 1);
            }
            sync_tree<true>();
            for (uint32_t j = 0;; ++j) {
                const uint64_t *Xj = chX + (uint64_t)j * 2 * a.wmax;
                uint64_t *Bj = chB + (uint64_t)j * 2 * a.wmax;
                const uint32_t p = j;
                uint32_t cx = 0;
                for (uint32_t x = 0; x < W; ++x) {
                    const uint64_t xw = Xj[x];
                    if ((xw >> lane) & 1ull) cand[cx + (uint32_t)__popcll(xw & lanemask_lt())] = x * 64 + lane;
                    cx += (uint32_t)__popcll(xw);
                }
                sync_tree<true>();
                if (cx == 0) {
                    if (k >= h0 && k - h0 <= p) {
                        const uint64_t idx = (uint64_t)p * a.bstride + (k - h0);
                        if (a.binom_ovf[idx]) w.run_ovf = 1;
                        run_add(w, a.binom[idx]);
                    }
                    break;
                }
                if (h0 + p + cx < k) break;
                if (cx <= 64 || j + 1 == a.chain) {  // the rest of the chain is one entry
                    endj = j;
                    break;
                }
                uint32_t best_s = 0, best_j = INF32;
                uint64_t sum_s = 0;
                for (uint32_t c = lane; c < cx; c += 64) {
                    const uint32_t v = cand[c];
                    const uint64_t *rv = rows + (uint64_t)v * W;
                    uint32_t sc = 0;
                    for (uint32_t x = 0; x < W; ++x) sc += (uint32_t)__popcll(Xj[x] & rv[x]);
                    sum_s += sc;
                    if (best_j == INF32 || sc > best_s) {
                        best_s = sc;
                        best_j = v;
                    }
                }
                uint64_t key = best_j != INF32 ? (((uint64_t)best_s << 32) | (INF32 - best_j)) : 0ull;
                key = wave_max64(key);
                uint32_t dummy = 0;
                const uint64_t tot_s = wave_sum64_checked(sum_s, dummy);
                const uint32_t max_s = (uint32_t)(key >> 32), pv = INF32 - (uint32_t)(key & 0xFFFFFFFFull);
                if (j == 0 && h0 + 2 == k) {  // k-cliques of T with the root's h0 held: |E(T)|
                    run_add(w, tot_s / 2);
                    break;
                }
                if (h0 + p + max_s + 1 < k) break;
                const uint64_t *rp = rows + (uint64_t)pv * W;
                uint64_t *Xn = chX + (uint64_t)(j + 1) * 2 * a.wmax;
                for (uint32_t x = 0; x < W; ++x) {
                    uint64_t bw = Xj[x] & ~rp[x];
                    if (x == (pv >> 6)) bw &= ~(1ull << (pv & 63));
                    if (lane == 0) {
                        Bj[x] = bw;
                        Xn[x] = Xj[x] & ~bw & rp[x];
                    }
                    if ((bw >> lane) & 1ull) offs[ne + (uint32_t)__popcll(bw & lanemask_lt())] = (j << 16) | (x * 64 + lane);
                    ne += (uint32_t)__popcll(bw);
                }
                sync_tree<true>();
            }
            if (lane == 0) {
                if (endj != INF32) offs[ne++] = (endj << 16) | 0xFFFFu;
                ctl[2] = 0;
                ctl[3] = ne;
            }
        }
        __syncthreads();
        const uint32_t ne = ctl[3];
        for (;;) {
            uint32_t i = 0;
            if (lane == 0) i = atomicAdd(&ctl[2], 1u);
            i = uni32(i);
            if (i >= ne) break;
            const uint32_t e = offs[i], j = e >> 16, b = e & 0xFFFFu;
            const uint64_t *Xj = chX + (uint64_t)j * 2 * a.wmax, *Bj = chB + (uint64_t)j * 2 * a.wmax;
            const bool end = (b == 0xFFFFu);
            const uint64_t *rb = rows + (uint64_t)(end ? 0 : b) * W;
            for (uint32_t x = lane; x < W; x += 64) {
                if (end) {
                    X[x] = Xj[x];
                } else {
                    // the non-pivot branches of node j taken before b
                    const uint64_t taken = x < (b >> 6) ? Bj[x] : x == (b >> 6) ? (Bj[x] & ((1ull << (b & 63)) - 1)) : 0ull;
                    X[x] = Xj[x] & ~taken & rb[x];
                }
            }
            const uint32_t h = end ? h0 : h0 + 1;
            run_add(w, pivot_count<false, true, KIND>(a, g.psize, k, rows, stk, X, scal, cand, R, W, h, w.nodes, w.run_ovf,
                                                nullptr, j, false, crows2, crows4));
        }
        __syncthreads();
        if (wv == 0) {
            const uint64_t dt = wall_clock64() - t0;
            w.tmax = dt > w.tmax ? dt : w.tmax;
            w.tsum += dt;
        }
    }
    finish_wave(a, w);
}

// ---- task sizes and classes over the concatenated task space of a launch ----
// Query q owns global task ids [qoff[q], qoff[q+1]): its vertices (node
// granularity) or its oriented edges (edge granularity).
__device__ inline uint32_t query_of(const uint64_t *qoff, uint32_t nq, uint64_t g)
{
    uint32_t lo = 0, hi = nq - 1;  // last q with qoff[q] <= g
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (qoff[mid] <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// size of an edge task: |T| = |N+(u) & N+(v)| (merge)
__global__ __launch_bounds__(256) void k_task_size(const QDesc *qd, const uint64_t *qoff, uint32_t nq, uint64_t total,
                                                    uint32_t *size)
{
    for (uint64_t gi = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; gi < total;
         gi += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t q = query_of(qoff, nq, gi);
        const QDesc d = qd[q];
        const uint32_t t = (uint32_t)(gi - qoff[q]);
        if (!d.gran) continue;  // (a node task's size is its row length)
        const uint32_t u = d.src[t], v = d.col[t];
        uint32_t i = d.rowptr[u], ie = d.rowptr[u + 1], j = d.rowptr[v], je = d.rowptr[v + 1];
        uint32_t c = 0;
        while (i < ie && j < je) {
            const uint32_t x = d.col[i], y = d.col[j];
            c += (x == y);
            i += (x <= y);
            j += (y <= x);
        }
        size[gi] = c;
    }
}

// size class of a task; for pivoting, tasks above top2 (<= 256) go to the
// block-wide kernel instead of the four-word register kernel
__device__ inline int class_of(uint32_t s, uint32_t top2)
{
    return s <= 64 ? 0 : s <= 128 ? 1 : s <= top2 ? 2 : s <= 512 ? 3 : s <= 1024 ? 4 : 5;
}

// Sizes |T| = |N+(u) & N+(v)| of every edge task of one graph, with sum
// what a count at k = 3 adds for them (triangles, tasks and bytes by size
// class), and with bits the adjacency words that rows_from_bits reads.
// A wave takes 64 consecutive edges; the edges of one u share a hash of N+(u)
// in LDS (at most half full), and four lists N+(v) at a time are streamed
// against it by 16 lanes each, two loads in flight, the hits counted by ballot.
// The merge of both lists by one lane an edge, and at k = 3 staging every task
// once more to add its size, were bound by uncoalesced loads and divergence
// (R-MAT scale 18, 3.8 M edges: sizes 4.3 -> 1.1 ms, a call at k = 3 4.1 -> 1.3
// ms).  Rows above HASH_ROW are searched in place.
constexpr uint32_t HASH_SLOTS = 1024, HASH_ROW = 512;

struct EdgeArgs {
    const uint32_t *rowptr, *col, *src;
    uint32_t m, sample, offset, top2, sum;
    uint32_t *size;
    uint64_t *acc;  // the algorithm's first bin (copies as in CountArgs)
    uint64_t *bits;  // as CountArgs::bits, written (or null)
};

template <bool BITS>
__global__ __launch_bounds__(256) void k_edge_sizes(EdgeArgs a)
{
    __shared__ uint32_t tables[4][HASH_SLOTS];
    __shared__ uint8_t places[BITS ? 4 : 1][BITS ? HASH_SLOTS : 1];  // of the table's vertices in N+(u)
    __shared__ unsigned long long words[BITS ? 4 : 1][4][BITS_ROW / 64];
    if (BITS && threadIdx.x < 4 * 4 * (BITS_ROW / 64)) (&words[0][0][0])[threadIdx.x] = 0;
    __shared__ unsigned long long sums[NCLASS][3];
    if (threadIdx.x < NCLASS * 3) (&sums[0][0])[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t lane = (uint32_t)lane_id(), wv = uni32(threadIdx.x >> 6), grp = lane >> 4, sub = lane & 15;
    uint32_t *tab = tables[wv];
    const uint32_t nwave = gridDim.x * 4;
    for (uint64_t e0 = (uint64_t)(blockIdx.x * 4 + wv) * 64; e0 < a.m; e0 += (uint64_t)nwave * 64) {
        const uint32_t cnt = (uint32_t)min((uint64_t)64, a.m - e0);
        uint32_t u = INF32, vb = 0, dv = 0, du = 0, mine = 0;
        if (lane < cnt) {
            u = a.src[e0 + lane];
            const uint32_t v = a.col[e0 + lane];
            vb = a.rowptr[v];
            dv = a.rowptr[v + 1] - vb;
        }
        for (uint32_t pos = 0; pos < cnt;) {
            const uint32_t uu = (uint32_t)__builtin_amdgcn_readlane((int)u, (int)pos);
            const uint32_t nseg = (uint32_t)__popcll(__ballot(u == uu));  // (side by side: edges are sorted by u)
            const uint32_t ub = a.rowptr[uu], d = a.rowptr[uu + 1] - ub;
            const uint32_t *row = a.col + ub;
            if (u == uu) du = d;
            if (BITS && !a.size && (d < 2 || d > BITS_ROW)) {  // (node tasks want the words alone)
                pos += nseg;
                continue;
            }
            uint32_t bits = 6;
            while (bits < 10 && (1u << bits) < 4 * d) ++bits;
            const uint32_t mask = (1u << bits) - 1;
            const bool hashed = d <= HASH_ROW, bits_on = BITS && d <= BITS_ROW;
            auto slot_of = [&](uint32_t x) { return (x * 2654435761u) >> (32 - bits); };
            if (hashed) {
                for (uint32_t i = lane; i <= mask; i += 64) tab[i] = INF32;
                sync_tree<true>();
                for (uint32_t i = lane; i < d; i += 64) {
                    const uint32_t x = row[i];
                    uint32_t s = slot_of(x);
                    while (atomicCAS(&tab[s], INF32, x) != INF32) s = (s + 1) & mask;
                    if (bits_on) places[wv][s] = (uint8_t)i;
                }
                sync_tree<true>();
            }
            auto found = [&](uint32_t x) {  // (and the bit of the group's list)
                if (!hashed) {
                    const uint32_t i = lower_bound_u32(row, d, x);
                    return i < d && row[i] == x;
                }
                uint32_t s = slot_of(x), t = tab[s];
                while (t != x && t != INF32) {
                    s = (s + 1) & mask;
                    t = tab[s];
                }
                if (bits_on && t == x) {
                    const uint32_t at = places[wv][s];
                    atomicOr(&words[wv][grp][at >> 6], 1ull << (at & 63));
                }
                return t == x;
            };
            for (uint32_t q = 0; q < nseg; q += 4) {
                const int from = (int)((pos + q + grp) & 63);
                const uint32_t b = __shfl(vb, from, 64), l0 = __shfl(dv, from, 64), len = q + grp < nseg ? l0 : 0;
                uint32_t hits = 0;
                for (uint32_t j = sub; __ballot(j < len); j += 32) {
                    const bool in0 = j < len, in1 = j + 16 < len;
                    const uint32_t x0 = in0 ? a.col[b + j] : INF32, x1 = in1 ? a.col[b + j + 16] : INF32;
                    const uint64_t h0 = __ballot(in0 && found(x0)), h1 = __ballot(in1 && found(x1));
                    hits += (uint32_t)__popc((uint32_t)(h0 >> (16 * grp)) & 0xFFFFu) +
                            (uint32_t)__popc((uint32_t)(h1 >> (16 * grp)) & 0xFFFFu);
                }
                const uint32_t mq = lane - (pos + q), h = __shfl(hits, (int)((mq & 3) * 16), 64);
                if (mq < 4 && q + mq < nseg) mine = h;
                if (bits_on) {
                    sync_tree<true>();
                    if (sub * 64 < d && q + grp < nseg) {
                        a.bits[(uint64_t)sub * a.m + e0 + pos + q + grp] = words[wv][grp][sub];
                        words[wv][grp][sub] = 0;
                    }
                    sync_tree<true>();
                }
            }
            if (hashed) sync_tree<true>();  // the table is cleared next
            pos += nseg;
        }
        if (lane < cnt) {
            const uint32_t e = (uint32_t)e0 + lane;
            if (!BITS || a.size) a.size[e] = mine;
            if (!BITS && a.sum && mine && (a.sample <= 1 || e % a.sample == a.offset)) {
                const int c = class_of(mine, a.top2);
                atomicAdd(&sums[c][0], (unsigned long long)mine);
                atomicAdd(&sums[c][1], 24ull + 4ull * ((uint64_t)du + dv));
                atomicAdd(&sums[c][2], 1ull);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < NCLASS * 3) {
        const uint32_t c = threadIdx.x / 3, i = threadIdx.x % 3;
        const unsigned long long v = sums[c][i];
        unsigned long long *acc = reinterpret_cast<unsigned long long *>(
            a.acc + ((uint64_t)c * NSTRIPE + blockIdx.x % NSTRIPE) * ACC);
        if (i != 0) {
            if (v) atomicAdd(&acc[i], v);
        } else if (v) {  // a count: its low and high half (flush_query)
            atomicAdd(&acc[0], v & 0xFFFFFFFFull);
            atomicAdd(&acc[6], v >> 32);
        }
    }
}

// Bin tasks by (algorithm, size class, size slice); a task smaller than the
// clique part still to find (k-1 for a node, k-2 for an edge) is dropped.
// Each class from 65 to 1024 vertices is cut into NSUB slices of its size
// range, largest first, and a class's slices are contiguous in the task
// array, so a class launch drains its largest tasks first and the long ones
// do not start last.  k_bin_count counts per slice and takes the max size of
// the unbounded class and of the launch (bin_max[15]), k_bin_offsets places the
// slices, k_bin_scatter writes (query << 32 | task).
// A block adds up its tiles (or one tile) in LDS and touches the device's
// counters once per slice it met: with an atomic per wave and slice, the few
// counters -- one of them takes most tasks -- bound both passes (0.8 ms each
// over 7.8 M edge tasks; 970,000 node tasks of 96 graphs: two passes of 176 us
// -> one of 29 us).
constexpr int NSUB = 16;
constexpr int NSLICE = 2 * NCLASS * NSUB;
constexpr int BIN_T = 256;
// tasks per thread: 16 keep the device's counters quiet where tasks are many,
// 2 fill the device where they are few
constexpr int BIN_I = 16, BIN_I_FEW = 2;

__device__ inline int slice_of(uint32_t s, int c, uint32_t top2)
{
    if (c == 0 || c == NCLASS - 1) return 0;  // (the many small tasks: one slice keeps classification cheap)
    const uint32_t lo = c == 3 ? top2 : CLASS_ROWS[c - 1], hi = c == 2 ? top2 : CLASS_ROWS[c];
    const uint32_t sl = (hi - s) * NSUB / (hi - lo);
    return sl < NSUB ? (int)sl : NSUB - 1;
}

struct BinArgs {
    const QDesc *qd;
    const uint8_t *qalgo;
    const uint64_t *qoff;
    uint32_t nq;
    uint32_t pivot_top2;
    uint64_t total;
    const uint32_t *size;   // edge tasks' sizes (a node task's is its row length)
    uint32_t *sub_cnt;      // [NSLICE] tasks of each slice
    uint32_t *bin_max;      // [16] largest task of the unbounded bins, [15] of the launch
    uint32_t *sub_pos;      // [NSLICE] tasks of each slice written so far
    uint32_t *sub_off;      // [NSLICE] first task of each slice
    uint64_t *out;
    uint64_t *binom;        // C(n, r), then a byte per entry: over 64 bits (null: not needed)
    uint32_t brows, bstride;
};

// the query of the tasks a thread goes through in ascending order
struct BinCursor {
    uint32_t q;
    uint64_t begin, end;  // its global tasks
    QDesc d;
    uint32_t algo;
    __device__ BinCursor(const BinArgs &b, uint64_t gi) { load(b, b.nq == 1 ? 0 : query_of(b.qoff, b.nq, gi)); }
    __device__ void load(const BinArgs &b, uint32_t qq)
    {
        q = qq;
        begin = b.qoff[q];
        end = b.qoff[q + 1];
        d = b.qd[q];
        algo = b.qalgo[q] ? 1 : 0;
    }
    __device__ void seek(const BinArgs &b, uint64_t gi)  // gi < total
    {
        while (gi >= end) load(b, q + 1);
    }
};

// the slice of global task gi < total of size s, -1 when the task does not run
__device__ inline int bin_of(const BinArgs &b, const BinCursor &c, uint64_t gi, uint32_t s)
{
    const QDesc &d = c.d;
    if (s < (d.gran ? d.k - 2 : d.k - 1) || (d.sample > 1 && (uint32_t)(gi - c.begin) % d.sample != d.offset)) return -1;
    const uint32_t top2 = c.algo ? b.pivot_top2 : CLASS_ROWS[2];
    const int cl = class_of(s, top2);
    return (int)(c.algo * NCLASS + cl) * NSUB + slice_of(s, cl, top2);
}

__device__ inline uint32_t task_size(const BinArgs &b, const BinCursor &c, uint64_t gi)
{
    const uint32_t t = (uint32_t)(gi - c.begin);
    return c.d.gran ? b.size[gi] : c.d.rowptr[t + 1] - c.d.rowptr[t];
}

// the sizes of a thread's I tasks of a tile (task i at base + i * BIN_T), all
// loads in flight together where the tile lies in one query
template <int I>
__device__ inline void tile_sizes(const BinArgs &b, BinCursor c, uint64_t base, uint32_t (&s)[I])
{
#pragma unroll
    for (int i = 0; i < I; ++i) {
        const uint64_t gi = base + (uint64_t)i * BIN_T;
        s[i] = 0;
        if (gi >= b.total) continue;
        if (gi >= c.end) c.seek(b, gi);
        s[i] = task_size(b, c, gi);
    }
}

template <int I>
__global__ __launch_bounds__(BIN_T) void k_bin_count(BinArgs b)
{
    __shared__ uint32_t cnt[NSLICE], mx[3];
    for (int i = threadIdx.x; i < NSLICE; i += BIN_T) cnt[i] = 0;
    if (threadIdx.x < 3) mx[threadIdx.x] = 0;
    __syncthreads();
    uint32_t m[3] = {0, 0, 0};  // largest task; of the unbounded orientation and pivoting bins
    for (uint64_t base = (uint64_t)blockIdx.x * BIN_T * I; base < b.total; base += (uint64_t)gridDim.x * BIN_T * I) {
        BinCursor c(b, base);
        uint32_t s[I];
        tile_sizes(b, c, base + threadIdx.x, s);
#pragma unroll
        for (int i = 0; i < I; ++i) {
            const uint64_t gi = base + (uint64_t)i * BIN_T + threadIdx.x;
            if (gi >= b.total) continue;
            c.seek(b, gi);
            const int fb = bin_of(b, c, gi, s[i]);
            if (fb < 0) continue;
            atomicAdd(&cnt[fb], 1u);
            m[0] = max(m[0], s[i]);
            if (fb / NSUB == NCLASS - 1) m[1] = max(m[1], s[i]);
            if (fb / NSUB == 2 * NCLASS - 1) m[2] = max(m[2], s[i]);
        }
    }
    for (int i = 0; i < 3; ++i)
        if (m[i]) atomicMax(&mx[i], m[i]);
    __syncthreads();
    for (int i = threadIdx.x; i < NSLICE; i += BIN_T)
        if (cnt[i]) atomicAdd(&b.sub_cnt[i], cnt[i]);
    if (threadIdx.x < 3 && mx[threadIdx.x])
        atomicMax(&b.bin_max[threadIdx.x == 0 ? 15 : threadIdx.x * NCLASS - 1], mx[threadIdx.x]);
}

// exact C(n, r) for n <= nmax, r < bstride <= 64, one row a step, by one wave
// (lane r); the byte after the table is 1 where the value exceeds 2^64-1
__device__ inline void binom_rows(const BinArgs &b, uint32_t nmax)
{
    const uint32_t r = (uint32_t)lane_id();
    uint8_t *ovf = reinterpret_cast<uint8_t *>(b.binom + (uint64_t)(b.brows) * b.bstride);
    uint64_t v = r == 0 ? 1 : 0;
    uint32_t o = 0;
    for (uint32_t n = 0;; ++n) {
        if (r < b.bstride) {
            b.binom[(uint64_t)n * b.bstride + r] = v;
            ovf[(uint64_t)n * b.bstride + r] = (uint8_t)o;
        }
        if (n == nmax) break;
        // (the lane below's values: a wave shift in the ALU, not a trip through LDS, a row)
        auto below = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x138, 0xf, 0xf, false); };
        const uint64_t w = ((uint64_t)below((uint32_t)(v >> 32)) << 32) | below((uint32_t)v);
        const uint32_t ow = below(o);
        if (r > 0) {
            const uint64_t sum = v + w;
            o |= ow | (sum < v ? 1u : 0u);
            v = sum;
        }
    }
}

// block 0: where each slice's tasks go; block 1: the binomial table, for
// every task size of the launch
__global__ __launch_bounds__(64) void k_bin_offsets(BinArgs b)
{
    if (blockIdx.x == 1) {
        if (b.binom) binom_rows(b, min(b.brows - 1, b.bin_max[15] + 1));
        return;
    }
    uint32_t carry = 0;
    for (int base = 0; base < NSLICE; base += 64) {
        const uint32_t c = b.sub_cnt[base + lane_id()], inc = wave_incl_scan32(c);
        b.sub_off[base + lane_id()] = carry + inc - c;
        carry += __shfl(inc, 63, 64);
    }
}

// One tile a block.  With ONE the launch has a single slice (every task of at
// most 64 vertices, one algorithm): no counting pass is needed, its tasks
// start at 0 and sub_pos ends as their number; the block after the last tile
// makes the binomial table.
template <bool ONE, int I>
__global__ __launch_bounds__(BIN_T) void k_bin_scatter(BinArgs b)
{
    __shared__ uint32_t cnt[NSLICE], at[NSLICE];
    const uint64_t base = (uint64_t)blockIdx.x * BIN_T * I;
    if (ONE && base >= b.total) {
        if (b.binom && threadIdx.x < 64) binom_rows(b, b.brows - 1);
        return;
    }
    for (int i = threadIdx.x; i < NSLICE; i += BIN_T) cnt[i] = 0;
    __syncthreads();
    BinCursor c(b, base);
    int fb[I];
    uint32_t rank[I], s[I];
    tile_sizes(b, c, base + threadIdx.x, s);
    {
        BinCursor cc = c;
#pragma unroll
        for (int i = 0; i < I; ++i) {
            const uint64_t gi = base + (uint64_t)i * BIN_T + threadIdx.x;
            fb[i] = -1;
            if (gi >= b.total) continue;
            cc.seek(b, gi);
            fb[i] = bin_of(b, cc, gi, s[i]);
            if (fb[i] >= 0) rank[i] = atomicAdd(&cnt[fb[i]], 1u);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NSLICE; i += BIN_T)
        if (cnt[i]) at[i] = (ONE ? 0u : b.sub_off[i]) + atomicAdd(&b.sub_pos[ONE ? 0 : i], cnt[i]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < I; ++i) {
        if (fb[i] < 0) continue;
        const uint64_t gi = base + (uint64_t)i * BIN_T + threadIdx.x;
        c.seek(b, gi);
        b.out[at[fb[i]] + rank[i]] = ((uint64_t)c.q << 32) | (uint32_t)(gi - c.begin);
    }
}

// ---- host -------------------------------------------------------------------
static const void *generic_kernel(bool pivot, bool global, bool local, bool small)
{
    if (pivot) {  // (per-vertex counts; the others have kernels of their own)
        if (!local) return nullptr;
        return global ? reinterpret_cast<const void *>(&k_count<true, true, true, false>)
                      : reinterpret_cast<const void *>(&k_count<true, false, true, false>);
    }
    static const void *const k[6] = {
        reinterpret_cast<const void *>(&k_count<false, false, false, true>),
        reinterpret_cast<const void *>(&k_count<false, false, false, false>),
        reinterpret_cast<const void *>(&k_count<false, true, false, false>),
        reinterpret_cast<const void *>(&k_count<false, false, true, true>),
        reinterpret_cast<const void *>(&k_count<false, false, true, false>),
        reinterpret_cast<const void *>(&k_count<false, true, true, false>)};
    return k[(local ? 3 : 0) + (global ? 2 : small ? 0 : 1)];
}

static const void *register_kernel(int c, bool deep)
{
    static const void *const reg[5] = {reinterpret_cast<const void *>(&k_pivot_reg<1, LEAN>),
                                       reinterpret_cast<const void *>(&k_pivot_reg<2, LEAN>),
                                       reinterpret_cast<const void *>(&k_pivot_reg<4, LEAN>),
                                       reinterpret_cast<const void *>(&k_pivot_reg<2, MFMA>),
                                       reinterpret_cast<const void *>(&k_pivot_reg<4, MFMA>)};
    return reg[deep && c > 0 ? c + 2 : c];
}

// exact C(n, r) for n <= nmax, r <= rmax; ovf[i] = 1 when it exceeds 2^64-1
static void binom_table(uint32_t nmax, uint32_t rmax, std::vector<uint64_t> &val, std::vector<uint8_t> &ovf)
{
    const uint32_t st = rmax + 1;
    val.assign((size_t)(nmax + 1) * st, 0);
    ovf.assign((size_t)(nmax + 1) * st, 0);
    for (uint32_t n = 0; n <= nmax; ++n) {
        val[(size_t)n * st] = 1;
        for (uint32_t r = 1; r <= rmax && r <= n; ++r) {
            size_t i = (size_t)n * st + r, a = (size_t)(n - 1) * st + r - 1, b = (size_t)(n - 1) * st + r;
            uint64_t s = val[a] + val[b];
            ovf[i] = ovf[a] | ovf[b] | (s < val[a]);
            val[i] = s;
        }
    }
}

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t *p, uint64_t n, uint32_t v)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// The HIP events of one run_queries call, owned here so that every return
// path destroys them.  With a fixed scratch (no allocation of any kind) there
// are none: records and elapsed times become no-ops and the launches stay on
// one stream (the side-by-side launches need events to join).
struct RunEvents {
    static constexpr int NB = 2 * NCLASS;
    hipEvent_t start = nullptr, cls = nullptr, go = nullptr, fan = nullptr, end = nullptr;
    hipEvent_t b0[NB] = {}, b1[NB] = {};
    bool on = false;
    int create()
    {
        on = true;
        hipEvent_t *all[5] = {&start, &cls, &go, &fan, &end};
        for (hipEvent_t *e : all) KC_HIP(hipEventCreate(e));
        for (int b = 0; b < NB; ++b) {
            KC_HIP(hipEventCreate(&b0[b]));
            KC_HIP(hipEventCreate(&b1[b]));
        }
        return KC_OK;
    }
    void record(hipEvent_t e, hipStream_t st) const
    {
        if (on) hipEventRecord(e, st);
    }
    float ms(hipEvent_t a, hipEvent_t b) const
    {
        float t = 0;
        if (on) hipEventElapsedTime(&t, a, b);
        return t;
    }
    ~RunEvents()
    {
        hipEvent_t all[5] = {start, cls, go, fan, end};
        for (hipEvent_t e : all)
            if (e) hipEventDestroy(e);
        for (int b = 0; b < NB; ++b) {
            if (b0[b]) hipEventDestroy(b0[b]);
            if (b1[b]) hipEventDestroy(b1[b]);
        }
    }
};

int run_queries(Scratch &scr, hipStream_t s, const std::vector<QueryRun> &qs, std::vector<kc_result> &res,
                LaunchStats *ls, uint64_t *local, uint32_t grid_share)
{
    DeviceCtx *ctx;
    int rc = device_ctx(&ctx);
    if (rc) return rc;
    const uint32_t nq = (uint32_t)qs.size();
    res.assign(nq, kc_result{});
    if (nq == 0) return KC_OK;
    if (local && nq != 1) return fail(KC_ERR_ARG, "per-vertex counts take one query per launch");
    constexpr int NB = 2 * NCLASS;  // (algo, size class) bins

    // --- query descriptors and the concatenated task space ---
    std::vector<QDesc> hq(nq);
    std::vector<uint8_t> halgo(nq);
    std::vector<uint64_t> hoff(nq + 1, 0);
    uint32_t kmax = 0, P = 1;
    for (uint32_t i = 0; i < nq; ++i) {
        const kc_oriented *o = qs[i].o;
        const kc_query &q = qs[i].q;
        hq[i] = QDesc{o->rowptr.as<uint32_t>(), o->col.as<uint32_t>(), o->src.as<uint32_t>(),
                      o->key.as<uint32_t>(), q.k, q.gran, std::max<uint32_t>(1, qs[i].sample), qs[i].sample > 1 ? qs[i].offset : 0, q.part_size};
        halgo[i] = (uint8_t)(q.algo == KC_ALGO_PIVOT);
        hoff[i + 1] = hoff[i] + (q.gran == KC_GRAN_EDGE ? o->m : o->n);
        kmax = std::max(kmax, q.k);
        // every query keeps its own partition size; the orientation DFS stacks
        // are laid out for the smallest (the most partitions per wave)
        P = i == 0 ? q.part_size : std::min(P, q.part_size);
    }
    const uint64_t total = hoff[nq];
    if (total >= (1ull << 32) * 64) return fail(KC_ERR_LIMIT, "too many tasks in one launch");
    const size_t qd_bytes = sizeof(QDesc) * nq, off_bytes = sizeof(uint64_t) * (nq + 1);
    constexpr int NS = NB * NSUB;  // size slices
    // sub_cnt[NS] bin_max[16] sub_pos[NS] sub_off[NS] qhead[NB][NQUEUE]
    const size_t meta_u32 = 3 * NS + 16 + NB * NQUEUE * QSTRIDE;
    const size_t acc_bytes = sizeof(uint64_t) * NB * NSTRIPE * ACC;
    // per query: two sums, then a flag (the sums of a single query are in the accumulators)
    const size_t q_bytes = sizeof(uint64_t) * 2 * nq + sizeof(uint32_t) * nq;
    bool any_pivot = false, any_edge = false, one_algo = true;
    // The most vertices below the root of a pivoting task (it decides whether the two-
    // and four-word kernels have the matrix cores, below)
    uint32_t depth = 0;
    uint32_t max_out = 0;  // bounds every task's size
    for (uint32_t i = 0; i < nq; ++i) {
        any_pivot |= halgo[i] != 0;
        any_edge |= hq[i].gran == KC_GRAN_EDGE;
        one_algo &= halgo[i] == halgo[0];
        if (halgo[i]) depth = std::max(depth, hq[i].k - std::min(hq[i].k, hq[i].gran == KC_GRAN_EDGE ? 2u : 1u));
        max_out = std::max(max_out, qs[i].o->max_out);
    }
    const uint32_t bstride = kmax + 1, brows = max_out + 2;
    const size_t nbin = (size_t)brows * bstride;
    if ((rc = scr.qdesc.ensure(qd_bytes + off_bytes + nq + 16)) ||
        (rc = scr.meta.ensure(meta_u32 * 4 + acc_bytes + q_bytes + 16)) ||
        (rc = scr.tasks.ensure(sizeof(uint64_t) * (total + 1))) || (any_pivot && (rc = scr.binom.ensure(nbin * 9 + 16))) ||
        (any_edge && (rc = scr.size.ensure(sizeof(uint32_t) * (total + 1)))))
        return rc;
    QDesc *dq = scr.qdesc.as<QDesc>();
    uint64_t *doff = reinterpret_cast<uint64_t *>(scr.qdesc.as<uint8_t>() + qd_bytes);
    uint8_t *dalgo = scr.qdesc.as<uint8_t>() + qd_bytes + off_bytes;
    uint32_t *m32 = scr.meta.as<uint32_t>();
    uint32_t *sub_cnt = m32, *bin_max = m32 + NS, *sub_pos = bin_max + 16, *sub_off = sub_pos + NS, *qhead = sub_off + NS;
    uint64_t *dacc = reinterpret_cast<uint64_t *>(m32 + meta_u32);
    uint64_t *qcount = dacc + NB * NSTRIPE * ACC;
    uint32_t *qovf = reinterpret_cast<uint32_t *>(qcount + 2 * (size_t)nq);
    // descriptors, task offsets and algorithms side by side: one copy
    std::vector<uint8_t> up(qd_bytes + off_bytes + nq);
    std::memcpy(up.data(), hq.data(), qd_bytes);
    std::memcpy(up.data() + qd_bytes, hoff.data(), off_bytes);
    std::memcpy(up.data() + qd_bytes + off_bytes, halgo.data(), nq);
    // accumulators, per-query sums and overflow flags lie side by side: one copy back
    std::vector<uint64_t> back((acc_bytes + q_bytes + 7) / 8);
    uint32_t h[NS + 16] = {0};
    struct WordsUse {
        AdjWords *w = nullptr;
        ~WordsUse()
        {
            if (w) w->put();
        }
    } wu;
    StreamWait wait(s);  // no return leaves a kernel running on the caller's scratch
    KC_HIP(hipMemcpyAsync(dq, up.data(), up.size(), hipMemcpyHostToDevice, s));
    {  // counters, queue heads and per-query sums start at zero (a fill kernel, no memset node)
        const uint64_t nz = (meta_u32 * 4 + acc_bytes + q_bytes) / 4;
        hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)std::min<uint64_t>(1024, (nz + 255) / 256)), dim3(256), 0, s,
                           m32, nz, 0u);
    }

    // largest pivoting task the four-word register kernel takes (the rest of
    // the 129..256 class goes to the block-wide kernel); KC_PIVOT_TOP2
    // overrides it (129..256)
    uint32_t pivot_top2 = PIVOT_TOP2;
    if (const char *e = std::getenv("KC_PIVOT_TOP2")) {
        const long v = std::strtol(e, nullptr, 10);
        if (v >= 129 && v <= 256) pivot_top2 = (uint32_t)v;
    }
    RunEvents evs;
    if (!scr.fixed && (rc = evs.create())) return rc;
    evs.record(evs.start, s);
    const int gs = (int)std::max<uint64_t>(1, std::min<uint64_t>((total + 255) / 256, (uint64_t)ctx->cu * 16));
    // edge task sizes of a single query on the graph they were last computed for are reused
    const bool sizes_cached = nq == 1 && any_edge && scr.size_uid == qs[0].o->uid && scr.size_total == total;
    scr.size_uid = 0;
    // Every task of at most 64 vertices and one algorithm: a single bin, filled
    // by one pass, and the launch reads its number of tasks on the device, so
    // that the host waits for the device once, for the result.  Otherwise it
    // reads the bins' sizes first: they choose the launches.
    const bool one_bin = one_algo && max_out <= CLASS_ROWS[0] && total < 0xFFFFFFFFull;
    // edge tasks at k = 3 add their sizes: nothing to bin, nothing to launch after
    // (lists of at most MERGE_OUT are sooner merged by a lane an edge, and binned:
    // 23,936 edges with lists of at most 8, 47 us a call against 59)
    constexpr uint32_t MERGE_OUT = 32;
    // (KC_WORDS_MIB sets the bytes of adjacency words a handle may keep, 0: none)
    uint64_t bits_limit = 2ull << 30;
    if (const char *e = std::getenv("KC_WORDS_MIB")) bits_limit = std::strtoull(e, nullptr, 10) << 20;
    const bool lists = nq == 1 && any_edge && max_out > MERGE_OUT;
    const bool triangles = lists && kmax == 3 && !local && total > 0;
    // The adjacency words (rows_from_bits) of one query on a graph with
    // long lists: they belong to the handle's scratch like the sizes, and are
    // made by the pass that makes those, of a whole count and within bits_limit.
    // With lists of at most MERGE_OUT the pass costs the first call more than a
    // later one gains (BA n=200,000: 0.63 -> 0.84 and 0.52 -> 0.41 ms); with longer
    // ones both gain (Chung-Lu n=300,000, 2 M edges: pass 0.36 ms, the launches of a
    // count at k=6 1.39 -> 0.90 ms).
    // A sample of the tasks would not earn the pass; the fixed scratch and the
    // server's workers keep to the memory they declared.
    const uint64_t nedge = qs[0].o->m;
    const uint64_t bits_bytes = nedge * sizeof(uint64_t) * std::min<uint64_t>(BITS_ROW / 64, ((uint64_t)max_out + 63) / 64);
    // Where the device has no room for them the lists are used, and a later
    // allocation of this call or of another may take them back.
    if (nq == 1 && max_out > MERGE_OUT && !triangles && !(any_edge && kmax == 3) && nedge > 0 && !scr.fixed &&
        grid_share <= 1 && scr.words && hq[0].sample <= 1 && bits_bytes <= bits_limit && scr.words->take()) {
        wu.w = scr.words;
        if (wu.w->bits.bytes < bits_bytes) wu.w->uid = 0;
    }
    const bool with_bits = wu.w && wu.w->bits.try_ensure(bits_bytes);
    const bool bits_cached = with_bits && wu.w->uid == qs[0].o->uid;
    if (wu.w && !bits_cached) wu.w->uid = 0;
    uint64_t *const bits = with_bits ? wu.w->bits.as<uint64_t>() : nullptr;
    BinArgs ba{dq, dalgo, doff, nq, pivot_top2, total, any_edge ? scr.size.as<uint32_t>() : nullptr, sub_cnt, bin_max,
               sub_pos, sub_off, scr.tasks.as<uint64_t>(), any_pivot ? scr.binom.as<uint64_t>() : nullptr, brows, bstride};
    if (total > 0) {
        if ((lists && (triangles || !sizes_cached)) || (with_bits && !bits_cached)) {
            EdgeArgs ea{hq[0].rowptr, hq[0].col, hq[0].src, (uint32_t)nedge, hq[0].sample, hq[0].offset,
                        halgo[0] ? pivot_top2 : CLASS_ROWS[2], triangles ? 1u : 0u, any_edge ? scr.size.as<uint32_t>() : nullptr,
                        dacc + (halgo[0] ? NCLASS * NSTRIPE * ACC : 0), bits_cached ? nullptr : bits};
            const unsigned eb = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((nedge + 255) / 256, (uint64_t)ctx->cu * 8));
            if (triangles) evs.record(evs.go, s);
            if (ea.bits) hipLaunchKernelGGL(k_edge_sizes<true>, dim3(eb), dim3(256), 0, s, ea);
            else hipLaunchKernelGGL(k_edge_sizes<false>, dim3(eb), dim3(256), 0, s, ea);
        } else if (any_edge && !sizes_cached) {
            hipLaunchKernelGGL(k_task_size, dim3(gs), dim3(256), 0, s, dq, doff, nq, total, scr.size.as<uint32_t>());
        }
        const bool few = total < (uint64_t)BIN_T * BIN_I * ctx->cu;  // (less than a full tile per CU)
        const int per = BIN_T * (few ? BIN_I_FEW : BIN_I);
        const unsigned tiles = (unsigned)((total + per - 1) / per);
        void *args[] = {&ba};
        auto go = [&](const void *kern, unsigned blocks, unsigned threads) {
            return hipLaunchKernel(kern, dim3(blocks), dim3(threads), args, 0, s);
        };
        if (triangles) {
        } else if (one_bin) {
            KC_HIP(go(few ? (const void *)&k_bin_scatter<true, BIN_I_FEW> : (const void *)&k_bin_scatter<true, BIN_I>,
                      tiles + 1, BIN_T));
        } else {
            KC_HIP(go(few ? (const void *)&k_bin_count<BIN_I_FEW> : (const void *)&k_bin_count<BIN_I>,
                      std::min<unsigned>(tiles, (unsigned)ctx->cu * 4), BIN_T));
            KC_HIP(go((const void *)&k_bin_offsets, 2, 64));
            KC_HIP(go(few ? (const void *)&k_bin_scatter<false, BIN_I_FEW> : (const void *)&k_bin_scatter<false, BIN_I>,
                      tiles, BIN_T));
        }
    }
    KC_HIP(hipGetLastError());
    if (nq == 1 && any_edge) {
        scr.size_uid = qs[0].o->uid;
        scr.size_total = total;
    }
    if (with_bits) wu.w->uid = qs[0].o->uid;
    uint32_t bcnt[NB] = {0}, bmax[NB] = {0}, boff[NB] = {0};
    if (triangles) {
    } else if (one_bin) {
        bcnt[halgo[0] ? NCLASS : 0] = (uint32_t)total;  // (at most)
    } else {
        KC_HIP(hipMemcpyAsync(h, m32, sizeof h, hipMemcpyDeviceToHost, s));
        KC_HIP(hipStreamSynchronize(s));
        uint64_t tot = 0;
        for (int b = 0; b < NB; ++b) {
            boff[b] = (uint32_t)tot;
            for (int sl = 0; sl < NSUB; ++sl) {
                bcnt[b] += h[b * NSUB + sl];
                tot += h[b * NSUB + sl];
            }
            bmax[b] = h[NS + b];  // (kept for the unbounded classes only)
        }
        if (tot >= 0xFFFFFFFFull) return fail(KC_ERR_LIMIT, "more than 2^32 tasks in one launch");
    }
    if (!triangles) evs.record(evs.cls, s);

    // --- one persistent launch per non-empty bin, largest tasks first ---
    // The bins of tasks of at most 256 vertices can run side by side on the
    // device's side streams (each bin has its own queue head and
    // accumulators), so the waves a bin frees while its last long tasks
    // finish take the next bin's tasks.  Larger classes (the wide kernel,
    // launches that use the shared HBM slice gscr) run first and in order on
    // s, and the side streams start after them: sharing the device with the
    // small classes delays the wide classes' long chain walks.  With
    // grid_share > 1 (a server worker) every launch stays on s.
    if (!triangles) evs.record(evs.go, s);
    // Side by side only when the register classes hold few tasks per CU: then
    // a class's last long tasks are a large part of its launch (Chung-Lu
    // n=1.7M m=11.1M, edge tasks at k=8: 8,600 per CU, one 125 ms task in a
    // 132 ms launch; the count 572 -> 526 ms).  With many tasks per CU the tail
    // is negligible and overlapping launches only contend (R-MAT scale 22,
    // edge tasks at k=5: 166,000 per CU, 3.69 -> 3.91 s).
    constexpr uint64_t FAN_MAX_TASKS_PER_CU = 1u << 15;
    uint64_t reg_tasks = 0;
    for (int b = 0; b < NB; ++b)
        if (b % NCLASS <= 2) reg_tasks += bcnt[b];
    // KC_SIDE_BY_SIDE=1 / =0 forces the choice (tests run both ways)
    const char *fan_env = std::getenv("KC_SIDE_BY_SIDE");
    const bool fan_rule = reg_tasks < FAN_MAX_TASKS_PER_CU * (uint64_t)ctx->cu;
    const bool fan = evs.on && grid_share == 1 && (fan_env && *fan_env ? *fan_env == '1' : fan_rule);
    // With at most one large task per CU the wide launches are on the device
    // whole from the start and the small classes take the CUs they leave (R-MAT
    // scale 17, node tasks at k=5: 187 large tasks, 1.5 ms before the rest, 4.8
    // -> 4.0 ms).
    uint64_t wide_tasks = 0;
    for (int b = 0; b < NB; ++b)
        if (b % NCLASS > 2) wide_tasks += bcnt[b];
    const bool few_wide = wide_tasks <= (uint64_t)ctx->cu;
    // Every launch is planned before the first one starts: the HBM slices of the
    // classes that need them are one block, sized here for the largest need.  A
    // block that grew between two launches would be released while the launch
    // before still keeps its bitmaps, chains and entry lists in it (the class
    // above 1024 vertices goes first, with few tasks; the 513..1024 class behind
    // it has smaller slices and usually more of them).
    struct Launch {
        CountArgs a;
        const void *kern;
        int b;
        uint32_t blocks, nw;
        size_t lds;
        bool global;
    };
    std::vector<Launch> plan;
    size_t slice_bytes = 0;
    bool side_waits[DeviceCtx::NSIDE] = {false}, fan_recorded = false;
    hipStream_t bin_stream[NB];
    int nside = 0;
    uint32_t variant[NB] = {0};
    bool launched[NB] = {false};
    const size_t lds_cap = ctx->lds_per_block;
    int order[NB], no = 0;
    for (int c = NCLASS - 1; c >= 0; --c) {
        order[no++] = NCLASS + c;  // pivot bins
        order[no++] = c;           // orientation bins
    }
    for (int oi = 0; oi < NB; ++oi) {
        const int b = order[oi];
        if (bcnt[b] == 0) continue;
        const bool pivot = b >= NCLASS;
        const int c = b % NCLASS;
        CountArgs a{};
        a.qd = dq;
        a.tasks = scr.tasks.as<uint64_t>() + boff[b];
        a.ntasks = bcnt[b];
        a.ntasks_p = one_bin ? sub_pos : nullptr;
        a.binom = scr.binom.as<uint64_t>();
        a.binom_ovf = scr.binom.as<uint8_t>() + nbin * 8;
        a.bstride = bstride;
        a.qhead = qhead + (size_t)b * NQUEUE * QSTRIDE;
        a.acc = dacc + (size_t)b * NSTRIPE * ACC;
        a.acc_mask = NSTRIPE - 1;
        a.bits = bits;
        a.bits_m = nedge;
        a.qcount = qcount;
        a.single = nq == 1;
        a.qovf = qovf;
        a.local = local;
        const bool lc = local != nullptr;
        bool global = (c == NCLASS - 1);
        const uint32_t rows_cap = global ? bmax[b] : CLASS_ROWS[c];
        a.rmax = rows_cap;
        a.wmax = (rows_cap + 63) / 64;
        a.levels = pivot ? kmax + 3 : std::max<uint32_t>(1, kmax - 2);
        uint32_t np = 64 / P;
        Layout L = make_layout(a.rmax, a.wmax, a.levels, np, pivot, lc);
        if (!global && !pivot) {
            while (np > 1 && L.total * 8 > lds_cap) {  // fewer partitions when the stacks do not fit
                np >>= 1;
                L = make_layout(a.rmax, a.wmax, a.levels, np, pivot, lc);
            }
        }
        if (!global && L.total * 8 > lds_cap) global = true;  // same layout in HBM
        a.nparts = np;
        const void *kern = generic_kernel(pivot, global, lc, c <= 1);
        variant[b] = global ? 3u : 1u;
        if (pivot && !global && c <= 2 && !lc) {
            // Six or more vertices below the roots: the tree is walked, and most of the time
            // goes to closing its nodes, on the matrix cores.  Up to three: most roots close
            // by themselves, and the operands' registers only cost waves and spills.  Between
            // them it turns with the tasks: at four, closures of a few long tasks are shorter
            // on the matrix cores, with many tasks the waves count; at five the few tasks'
            // nodes spend their time above the closures, except edge tasks', whose sets are
            // dense.  ms without / with matrix cores, and tasks of the class per CU:
            //   <= 3  R-MAT scale 22 edge k=5, 65..128 vertices 341 / 476, 129..256 982 / 1196
            //   4     random graph, 300 vertices, node k=5 (0.6) 0.63 / 0.49, R-MAT scale 14
            //         node (4.9) 0.42 / 0.35, Chung-Lu n=300,000 edge k=6 (20) 0.87 / 0.81, R-MAT
            //         scale 18 node (35) 2.18 / 2.32, Chung-Lu n=1.7M edge (1087) 26.7 / 30.0
            //   5     random graph, 300 vertices, node k=6 (0.6) 3.52 / 4.71, R-MAT scale 14 node
            //         (4.9) 1.29 / 1.64, scale 15 node (7.1) 2.85 / 2.65, Chung-Lu n=1M edge k=7
            //         (543) 26.6 / 24.4, R-MAT scale 14 edge (2.5) 0.97 / 0.79
            //   >= 6  R-MAT scale 14 node k=7 6.3 / 5.2, Chung-Lu n=1.7M edge k=8 434 / 345
            const uint32_t cu = (uint32_t)ctx->cu;
            constexpr uint32_t MANY_AT_4 = 24, MANY_AT_5 = 7;  // tasks per CU
            kern = register_kernel(c, depth >= 6 || (depth == 5 && (any_edge || bcnt[b] >= MANY_AT_5 * cu)) ||
                                          (depth == 4 && bcnt[b] < MANY_AT_4 * cu));
            L = make_layout(a.rmax, a.wmax, 0, 0, true);
            variant[b] = 2u;
        }
        if (pivot && !global && lc && c <= 1) {
            kern = c == 0 ? reinterpret_cast<const void *>(&k_local_reg<1>)
                          : reinterpret_cast<const void *>(&k_local_reg<2>);
            L = make_layout(a.rmax, a.wmax, 0, 0, true);
            L.total += LOCAL_CACHE * (sizeof(uint64_t) + sizeof(uint32_t) + 1) / sizeof(uint64_t);
            variant[b] = 2u;
        }
        uint32_t nw = 1;
        if (pivot && !global && c == 2 && !lc && bcnt[b] <= (uint32_t)ctx->cu * BLOCK_TASKS_PER_CU) {
            kern = reinterpret_cast<const void *>(&k_pivot_block<BLOCK_WAVES>);
            nw = BLOCK_WAVES;
            L.total = make_block_layout(nw).total;
        }
        // large tasks of pivoting: blocks of several waves sharing one bitmap
        WideLayout WL{};
        if (pivot && !lc && c >= 3) {
            // chain levels walked by wave 0 before the entries are shared: the
            // whole chain for the HBM classes (a chain left whole is one entry,
            // which one wave would walk alone), 32 levels when LDS holds them
            if (a.rmax >= 0xFFFFu)
                return fail(KC_ERR_LIMIT, "a task of %u vertices exceeds the wide kernel's 65534", a.rmax);
            a.chain = c == 3 ? 32u : std::min<uint32_t>(1024u, std::max<uint32_t>(64u, a.rmax));
            bool fits = false;
            if (c < NCLASS - 1)
                for (uint32_t t = 8; t >= 2 && !fits; t >>= 1) {
                    WL = make_wide_layout(a.rmax, a.wmax, a.levels, t, a.chain);
                    if (WL.total * 8 <= lds_cap) {
                        nw = t;
                        fits = true;
                    }
                }
            global = !fits;
            if (!fits) {
                nw = 8;
                WL = make_wide_layout(a.rmax, a.wmax, a.levels, nw, a.chain);
            }
            static const void *const wide[4] = {reinterpret_cast<const void *>(&k_pivot_wide<false, WIDE_SCT>),
                                                reinterpret_cast<const void *>(&k_pivot_wide<true, WIDE_SCT>),
                                                reinterpret_cast<const void *>(&k_pivot_wide<false, WIDE_DEEP>),
                                                reinterpret_cast<const void *>(&k_pivot_wide<true, WIDE_DEEP>)};
            // (the matrix cores from six vertices below the roots, above 512 vertices from
            // seven.  ms without / with: R-MAT scale 18, node tasks of 257..512, k=7 126 / 111,
            // k=8 634 / 429; R-MAT scale 22, 1 of 2048 node tasks at k=7, 257..512 784 / 811,
            // 513..1024 15,780 / 16,860; 1 of 8192 edge tasks at k=9, both 18,090 / 15,230)
            kern = wide[(depth >= (c == 3 ? 6u : 7u) ? 2 : 0) + (global ? 1 : 0)];
            L.total = WL.total;
            variant[b] = global ? 5u : 4u;
        }
        if (!kern) return fail(KC_ERR_DEVICE, "no kernel for tasks of %u vertices (internal error)", a.rmax);
        const size_t lds = global ? 0 : L.total * 8;
        if (!global) KC_HIP(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        int per_cu = 0;
        KC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, (int)(64 * nw), lds));
        if (per_cu < 1) per_cu = 1;
        uint64_t blocks = std::max<uint64_t>(1, (uint64_t)per_cu * ctx->cu / std::max<uint32_t>(1, grid_share));
        // one block per task while the tasks are few, else the persistent grid
        // and its queues (a server worker's share of the device is a grid size,
        // an HBM slice belongs to a block: those stay persistent)
        constexpr uint64_t DIRECT_ROUNDS = 4;
        a.direct = grid_share <= 1 && !global && bcnt[b] <= blocks * DIRECT_ROUNDS;
        a.chunk_log = (c == 0 && bcnt[b] > blocks * 64) ? 2 : 0;  // (the wide kernel takes one task per grab)
        const uint64_t chunks = ((uint64_t)bcnt[b] + (1u << a.chunk_log) - 1) >> a.chunk_log;
        blocks = a.direct ? chunks : std::min<uint64_t>(blocks, chunks);
        if (global) {
            a.gscr_words = L.total;
            // a fixed scratch holds as many slices as fit in what it has left
            const uint64_t cap = (scr.fixed ? scr.gscr.bytes : (2ull << 30)) / (L.total * 8 + 1);
            if (scr.fixed && cap == 0)
                return fail(KC_ERR_LIMIT, "a task of %u vertices needs %llu bytes of HBM workspace, more than the "
                            "%zu left in the fixed scratch", a.rmax, (unsigned long long)(L.total * 8), scr.gscr.bytes);
            blocks = std::max<uint64_t>(1, std::min<uint64_t>(blocks, cap));
            slice_bytes = std::max<size_t>(slice_bytes, blocks * L.total * 8);
        }
        plan.push_back(Launch{a, kern, b, (uint32_t)blocks, nw, lds, global});
    }
    if (slice_bytes && !scr.gscr.try_ensure(slice_bytes, true) && with_bits) {
        // the words of this very call stand in the way: the lists do
        KC_HIP(hipStreamSynchronize(s));
        wu.w->uid = 0;
        wu.w->bits.release();
        for (Launch &l : plan) l.a.bits = nullptr;
    }
    if (slice_bytes && (rc = scr.gscr.ensure(slice_bytes))) return rc;
    DevBuf::InUse in_use;  // from here to the wait below no buffer of this thread may move
    for (Launch &l : plan) {
        const int b = l.b;
        if (l.global) l.a.gscr = scr.gscr.as<uint64_t>();
        hipStream_t st = s;
        if (fan && !l.global && b % NCLASS <= 2) {
            if (!fan_recorded && !few_wide) {
                KC_HIP(hipEventRecord(evs.fan, s));  // after every launch so far on s
                fan_recorded = true;
            }
            const int si = nside++ % DeviceCtx::NSIDE;
            wait.side = ctx->side;
            st = ctx->side[si];
            if (!side_waits[si]) {
                KC_HIP(hipStreamWaitEvent(st, few_wide ? evs.go : evs.fan, 0));
                side_waits[si] = true;
            }
        }
        bin_stream[b] = st;
        if (plan.size() > 1 && !l.global)  // (two classes may share a kernel: the last plan's limit stands)
            KC_HIP(hipFuncSetAttribute(l.kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l.lds));
        void *args[] = {&l.a};
        evs.record(evs.b0[b], st);
        KC_HIP(hipLaunchKernel(l.kern, dim3(l.blocks), dim3(64 * l.nw), args, l.lds, st));
        evs.record(evs.b1[b], st);
        launched[b] = true;
    }
    for (int b = 0; b < NB; ++b)
        if (launched[b] && bin_stream[b] != s) KC_HIP(hipStreamWaitEvent(s, evs.b1[b], 0));
    evs.record(evs.end, s);
    KC_HIP(hipMemcpyAsync(back.data(), dacc, acc_bytes + q_bytes, hipMemcpyDeviceToHost, s));
    const hipError_t se = hipStreamSynchronize(s);
    if (se != hipSuccess) return fail(KC_ERR_DEVICE, "counting kernels failed: %s", hipGetErrorString(se));
    wait.done();
    uint64_t hacc[NB * ACC] = {0};
    for (int b = 0; b < NB; ++b)
        for (uint32_t c = 0; c < NSTRIPE; ++c)
            for (int i = 0; i < ACC; ++i) {
                const uint64_t v = back[((size_t)b * NSTRIPE + c) * ACC + i];
                uint64_t &h = hacc[b * ACC + i];
                h = i == 4 ? std::max(h, v) : h + v;  // [4] is the longest task
            }
    for (int b = 0; b < NB; ++b) {
        if (triangles && hacc[ACC * b + 2]) {
            launched[b] = true;
            variant[b] = 6u;
        }
        if (one_bin && hacc[ACC * b + 2] == 0) launched[b] = false;  // the bin was empty
    }
    const uint64_t *hq_sum = back.data() + NB * NSTRIPE * ACC;
    const uint32_t *hq_flag = reinterpret_cast<const uint32_t *>(hq_sum + 2 * (size_t)nq);
    float bin_ms[NB] = {0};
    const float prep_ms = evs.ms(evs.start, triangles ? evs.go : evs.cls), total_ms = evs.ms(evs.go, evs.end);
    for (int b = 0; b < NB; ++b)
        if (launched[b]) bin_ms[b] = triangles ? total_ms : evs.ms(evs.b0[b], evs.b1[b]);
    int wall_khz = 100000;
    hipDeviceGetAttribute(&wall_khz, hipDeviceAttributeWallClockRate, ctx->dev);
    if (wall_khz <= 0) wall_khz = 100000;

    for (uint32_t i = 0; i < nq; ++i) {
        kc_result &r = res[i];
        r.overflow = hq_flag[i] ? 1 : 0;
        unsigned __int128 sum = 0;
        if (nq == 1)
            for (int b = 0; b < NB; ++b) sum += hacc[ACC * b] + ((unsigned __int128)hacc[ACC * b + 6] << 32);
        else
            sum = hq_sum[2 * i] + ((unsigned __int128)hq_sum[2 * i + 1] << 32);
        r.count = (uint64_t)sum;
        if (sum >> 64) r.overflow = 1;
        r.algo = qs[i].q.algo;
        r.gran = qs[i].q.gran;
        r.part_size = qs[i].q.part_size;
    }
    if (ls) {
        *ls = LaunchStats{};
        ls->count_ms = total_ms;
        ls->prep_ms = prep_ms;
        int dom = -1;
        for (int b = 0; b < NB; ++b) {
            ls->tasks += hacc[ACC * b + 2];
            ls->alg_bytes += hacc[ACC * b + 1];
            ls->tree_nodes += hacc[ACC * b + 3];
            // the dominant launch: the one whose tasks hold the waves longest
            // (summed task durations; the side-by-side launches' spans overlap)
            if (launched[b] && (dom < 0 || hacc[ACC * b + 5] > hacc[ACC * dom + 5])) dom = b;
            const int c = b % NCLASS;
            if (!launched[b]) continue;
            ls->class_ms[c] += bin_ms[b];
            ls->class_bytes[c] += hacc[ACC * b + 1];
            ls->class_tasks[c] += hacc[ACC * b + 2];
            ls->class_kernel[c] = variant[b];
            ls->class_max_task_ms[c] = std::max(ls->class_max_task_ms[c], (double)hacc[ACC * b + 4] / wall_khz);
            ls->class_task_ms_sum[c] += (double)hacc[ACC * b + 5] / wall_khz;
        }
        if (dom >= 0) {
            ls->dominant_ms = bin_ms[dom];
            ls->dominant_bytes = hacc[ACC * dom + 1];
            ls->dominant_class = (uint32_t)(dom % NCLASS);
        }
    }
    return KC_OK;
}


// ---- OpenEngine (host) --------------------------------------------------------
OpenEngine::~OpenEngine()
{
    if (dev >= 0) hipSetDevice(dev);
    // every launch is stopped before any wait: streams sharing a hardware
    // queue would otherwise wait on a launch not stopped yet
    for (int j = 0; j < NQ; ++j)
        if (running(j) && !qs[j].stopped) stop(j);
    for (int j = 0; j < NQ; ++j) {
        if (qs[j].run) hipStreamSynchronize(qs[j].run);
        if (qs[j].done) hipEventDestroy(qs[j].done);
        if (qs[j].run) hipStreamDestroy(qs[j].run);
    }
    if (adm) {
        hipStreamSynchronize(adm);
        hipStreamDestroy(adm);
    }
    if (pinned) hipHostFree(pinned);
}

int OpenEngine::init(int device)
{
    dev = device;
    KC_HIP(hipSetDevice(dev));
    DeviceCtx *ctx;
    int rc = device_ctx(&ctx);
    if (rc) return rc;
    KC_HIP(hipStreamCreate(&adm));
    for (Queue &q : qs) {
        KC_HIP(hipStreamCreate(&q.run));
        KC_HIP(hipEventCreateWithFlags(&q.done, hipEventDisableTiming));
    }
    if ((rc = qcount.ensure(8 * SLOTS)) || (rc = qovf.ensure(4 * SLOTS)) || (rc = qdone.ensure(8 * SLOTS)) ||
        (rc = ctl.ensure(8 * CTL_WORDS * NQ)))
        return rc;
    const size_t qbytes = 16 + 16 * NSEG;  // total, nseg, then (base, slot|count) per segment
    const size_t bytes = NQ * qbytes + sizeof(OpenSlot) * SLOTS + sizeof(OpenMail) * SLOTS;
    KC_HIP(hipHostMalloc((void **)&pinned, bytes, hipHostMallocCoherent | hipHostMallocMapped));
    std::memset(pinned, 0, bytes);
    KC_HIP(hipHostGetDevicePointer((void **)&pinned_dev, pinned, 0));
    for (int j = 0; j < NQ; ++j) {
        uint64_t *h = reinterpret_cast<uint64_t *>(pinned + j * qbytes);
        qs[j].htotal = h;
        qs[j].hnseg = h + 1;
        qs[j].hseg = h + 2;
    }
    hslot = reinterpret_cast<OpenSlot *>(pinned + NQ * qbytes);
    mail = reinterpret_cast<OpenMail *>(hslot + SLOTS);
    // C(n, r) for n <= OPEN_MAX_ROWS + 1, r <= KC_MAX_K: every query a launch can take
    {
        std::vector<uint64_t> bv;
        std::vector<uint8_t> bo;
        binom_table(OPEN_MAX_ROWS + 1, KC_MAX_K, bv, bo);
        const size_t nbin = (size_t)(OPEN_MAX_ROWS + 2) * (KC_MAX_K + 1);
        if ((rc = binom.ensure(nbin * 9 + 16))) return rc;
        KC_HIP(hipMemcpyAsync(binom.p, bv.data(), nbin * 8, hipMemcpyHostToDevice, adm));
        KC_HIP(hipMemcpyAsync(binom.as<uint8_t>() + nbin * 8, bo.data(), nbin, hipMemcpyHostToDevice, adm));
        KC_HIP(hipStreamSynchronize(adm));
    }
    // per-slot sums start at zero; the flush that completes a slot zeroes them again
    hipLaunchKernelGGL(k_fill_u32, dim3(64), dim3(256), 0, adm, qcount.as<uint32_t>(), (uint64_t)2 * SLOTS, 0u);
    hipLaunchKernelGGL(k_fill_u32, dim3(64), dim3(256), 0, adm, qovf.as<uint32_t>(), (uint64_t)SLOTS, 0u);
    hipLaunchKernelGGL(k_fill_u32, dim3(64), dim3(256), 0, adm, qdone.as<uint32_t>(), (uint64_t)2 * SLOTS, 0u);
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, adm, ctl.as<uint32_t>(), (uint64_t)2 * CTL_WORDS * NQ, 0u);
    KC_HIP(hipGetLastError());
    KC_HIP(hipStreamSynchronize(adm));
    const Layout L = make_layout(OPEN_MAX_ROWS, OPEN_MAX_ROWS / 64, 0, 0, true);
    lds = L.total * 8;
    KC_HIP(hipFuncSetAttribute((const void *)k_pivot_open, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int per_cu = 0;
    KC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_pivot_open, 64, lds));
    if (per_cu < 12) return fail(KC_ERR_DEVICE, "resident launches: %d waves per CU", per_cu);
    // express: 4 waves per CU; bulk: the rest but 4, which stay free for the
    // workers' launches
    qs[0].blocks = (uint32_t)(4 * ctx->cu);
    qs[1].blocks = (uint32_t)((per_cu - 8) * ctx->cu);
    free_slots.clear();
    for (uint32_t i = SLOTS; i-- > 0;) free_slots.push_back(i);
    return KC_OK;
}

bool OpenEngine::running(int j)
{
    Queue &q = qs[j];
    if (!q.launched) return false;
    if (hipEventQuery(q.done) == hipSuccess) q.launched = false;
    return q.launched;
}

int OpenEngine::reset(int j)
{
    if (running(j) || qs[j].inflight) return fail(KC_ERR_ARG, "open queue reset while in use");
    Queue &q = qs[j];
    // the device words are cleared on the queue's own stream, ahead of its
    // next launch, and the host does not wait: more streams than hardware
    // queues share them, and a wait on a stream whose hardware queue holds
    // another resident launch would last until that launch ends -- which
    // only this thread's stop can bring about
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, q.run, ctl.as<uint32_t>() + 2 * CTL_WORDS * j,
                       (uint64_t)2 * CTL_WORDS, 0u);
    KC_HIP(hipGetLastError());
    __atomic_store_n(q.hnseg, 0ull, __ATOMIC_RELEASE);
    __atomic_store_n(q.htotal, 0ull, __ATOMIC_RELEASE);
    q.total = q.nseg = 0;
    return KC_OK;
}

static void publish_segment(OpenEngine::Queue &q, uint32_t slot, uint64_t count)
{
    q.hseg[2 * q.nseg] = q.total;
    q.hseg[2 * q.nseg + 1] = ((uint64_t)slot << 32) | count;
    q.nseg++;
    q.total += count;
}

// segments and descriptors are written before the counts that publish them;
// the segment count before the task total (a wave that sees the total finds
// its segment)
static void publish_counts(OpenEngine::Queue &q)
{
    __atomic_store_n(q.hnseg, q.nseg, __ATOMIC_RELEASE);
    __atomic_store_n(q.htotal, q.total, __ATOMIC_RELEASE);
}

void OpenEngine::admit(int j, const std::vector<OpenQueryIn> &in, std::vector<uint32_t> &slot)
{
    Queue &qq = qs[j];
    slot.assign(in.size(), ~0u);
    bool any = false;
    for (size_t i = 0; i < in.size(); ++i) {
        const OpenQueryIn &x = in[i];
        const uint64_t nt = x.q.gran == KC_GRAN_EDGE ? x.o->m : x.o->n;
        if (nt == 0) continue;
        const uint32_t sl = free_slots.back();
        free_slots.pop_back();
        slot[i] = sl;
        hslot[sl] = OpenSlot{x.o->rowptr.as<uint32_t>(), x.o->col.as<uint32_t>(), x.o->src.as<uint32_t>(), x.q.k,
                             x.q.gran, nt, x.seq, 0};
        publish_segment(qq, sl, nt);
        qq.inflight++;
        any = true;
    }
    if (any) publish_counts(qq);
}

void OpenEngine::stop(int j)
{
    Queue &q = qs[j];
    publish_segment(q, OPEN_STOP, q.blocks);
    publish_counts(q);
    q.stopped = true;
}

int OpenEngine::launch(int j)
{
    Queue &q = qs[j];
    OpenArgs oa{};
    CountArgs &a = oa.c;
    a.rmax = OPEN_MAX_ROWS;
    a.wmax = OPEN_MAX_ROWS / 64;
    a.binom = binom.as<uint64_t>();
    a.binom_ovf = binom.as<uint8_t>() + (size_t)(OPEN_MAX_ROWS + 2) * (KC_MAX_K + 1) * 8;
    a.bstride = KC_MAX_K + 1;
    a.qcount = qcount.as<uint64_t>();
    a.qovf = qovf.as<uint32_t>();
    uint64_t *c = ctl.as<uint64_t>() + CTL_WORDS * j;
    oa.counter = c;
    oa.known = c + 1;
    oa.last_poll = c + 2;
    oa.qdone = qdone.as<uint64_t>();
    auto dev_of = [&](const void *h) { return pinned_dev + (reinterpret_cast<const uint8_t *>(h) - pinned); };
    oa.htotal = reinterpret_cast<const uint64_t *>(dev_of(q.htotal));
    oa.hnseg = reinterpret_cast<const uint64_t *>(dev_of(q.hnseg));
    oa.hseg = reinterpret_cast<const uint64_t *>(dev_of(q.hseg));
    oa.hslot = reinterpret_cast<const OpenSlot *>(dev_of(hslot));
    oa.mail = reinterpret_cast<OpenMail *>(dev_of(mail));
    // a backstop only (the host ends every launch with a stop segment): 10 min
    oa.safety_ticks = 60000000000ull;
    void *args[] = {&oa};
    KC_HIP(hipLaunchKernel((const void *)k_pivot_open, dim3(q.blocks), dim3(64), args, lds, q.run));
    KC_HIP(hipEventRecord(q.done, q.run));
    q.launched = true;
    q.stopped = false;
    return KC_OK;
}

}  // namespace kc

using namespace kc;

namespace kc {
int check_query(const kc_query *q);
}
int kc::check_query(const kc_query *q)
{
    if (q->k < 1 || q->k > KC_MAX_K) return fail(KC_ERR_ARG, "k=%u outside 1..%d", q->k, KC_MAX_K);
    if (q->algo > 1 || q->gran > 1) return fail(KC_ERR_ARG, "bad algo/gran");
    const uint32_t P = q->part_size;
    if (P == 0 || P > 64 || (P & (P - 1))) return fail(KC_ERR_ARG, "partition size %u", P);
    return KC_OK;
}

// The autotuner (auto_tune = 1).  Measured on gfx950: one lane per candidate
// row / per DFS partition (P = 1) is fastest for every size class; pivoting
// with closed-form tails is never slower than the orientation DFS; edge tasks
// balance heavy-tailed degree distributions, node tasks win when every
// out-degree fits one 64-bit word and there are fewer vertices than edges to
// schedule.
namespace kc {
kc_query tune_query(const kc_oriented *o, const kc_query *q);
}
static kc_query tune(const kc_oriented *o, const kc_query *q) { return kc::tune_query(o, q); }

kc_query kc::tune_query(const kc_oriented *o, const kc_query *q)
{
    kc_query t = *q;
    if (q->auto_tune) {
        t.algo = KC_ALGO_PIVOT;
        t.part_size = 1;
        t.gran = (o->m > 0 && o->max_out > 64) ? KC_GRAN_EDGE : KC_GRAN_NODE;
    }
    return t;
}

void kc::fill_result(kc_result *r, const kc_result &res, const LaunchStats &ls)
{
    *r = res;
    r->tasks = ls.tasks;
    r->alg_bytes = ls.alg_bytes;
    r->tree_nodes = ls.tree_nodes;
    r->count_ms = ls.count_ms;
    r->dominant_ms = ls.dominant_ms;
    r->dominant_bytes = ls.dominant_bytes;
    r->dominant_class = ls.dominant_class;
    for (int c = 0; c < 6; ++c) {
        r->class_ms[c] = ls.class_ms[c];
        r->class_bytes[c] = ls.class_bytes[c];
        r->class_tasks[c] = ls.class_tasks[c];
        r->class_kernel[c] = ls.class_kernel[c];
        r->class_max_task_ms[c] = ls.class_max_task_ms[c];
        r->class_task_ms_sum[c] = ls.class_task_ms_sum[c];
    }
}

// ---- measured autotuner ---------------------------------------------------
// Both orientations are built and each (orientation, granularity) pair counts
// every 64th task at this k with pivoting; the pair with the least device
// time (classification + count of the sample) wins.  At k <= 5, where the
// orientation DFS can compete (its tree is at most three levels deep below
// the task), the same sample is then counted with the orientation DFS at
// partitions of 1, 8 and 64 lanes on the winning pair, and the algorithm and
// partition size with the least time make the plan.  (Summed task times,
// tail-free, ranked the plans worse: a sample of few large tasks runs at
// another occupancy than one of many small ones.)
int kc::autotune_measured(const kc_graph *g, uint32_t k, uint32_t degree_max_out, kc_plan *plan)
{
    constexpr uint32_t SAMPLE = 64;
    constexpr uint32_t ORIENT_DFS_MAX_K = 5;
    if (k > KC_MAX_K) return fail(KC_ERR_ARG, "k=%u outside 1..%d", k, KC_MAX_K);
    kc_oriented *o[2] = {nullptr, nullptr};
    int rc = kc_orient(g, KC_ORIENT_DEGREE, &o[0]);
    if (rc == KC_OK) rc = kc_orient(g, KC_ORIENT_DEGEN, &o[1]);
    double best = 0;
    int best_oi = 1;
    kc_query best_q{k, KC_ALGO_PIVOT, KC_GRAN_EDGE, 1, 1, 0};
    bool have = false;
    auto measure = [&](int oi, const kc_query &q) {
        QueryRun r;
        r.o = o[oi];
        r.q = q;
        r.sample = SAMPLE;
        std::vector<kc_result> res;
        LaunchStats ls;
        hipSetDevice(o[oi]->dev);
        rc = run_queries(o[oi]->scr, o[oi]->stream, {r}, res, &ls);
        const double t = ls.count_ms + ls.prep_ms;
        if (rc == KC_OK && (!have || t < best)) {
            have = true;
            best = t;
            best_oi = oi;
            best_q = q;
        }
    };
    for (int oi = 0; oi < 2 && rc == KC_OK; ++oi)
        for (uint32_t gran = KC_GRAN_NODE; gran <= KC_GRAN_EDGE && rc == KC_OK; ++gran)
            measure(oi, kc_query{k, KC_ALGO_PIVOT, gran, 1, 1, 0});
    if (k <= ORIENT_DFS_MAX_K && rc == KC_OK) {
        const int oi = best_oi;
        const uint32_t gran = best_q.gran;
        for (uint32_t P : {1u, 8u, 64u})
            if (rc == KC_OK) measure(oi, kc_query{k, KC_ALGO_ORIENT, gran, P, 1, 0});
    }
    for (kc_oriented *x : o)
        if (x) kc_oriented_free(x);
    if (rc != KC_OK) return rc;
    plan->degree_max_out = degree_max_out;
    plan->orient_mode = best_oi == 0 ? KC_ORIENT_DEGREE : KC_ORIENT_DEGEN;
    plan->algo = best_q.algo;
    plan->gran = best_q.gran;
    plan->part_size = best_q.part_size;
    return KC_OK;
}

// kc_count over the tasks whose id (vertex, or oriented edge in CSR order)
// is congruent to offset modulo stride; stride 1 counts every task.
static int count_tasks(const kc_oriented *o, const kc_query *q, uint32_t stride, uint32_t offset, kc_result *r)
{
    if (!o || !q || !r) return fail(KC_ERR_ARG, "kc_count: null argument");
    if (stride == 0 || offset >= stride) return fail(KC_ERR_ARG, "task sample offset %u, stride %u", offset, stride);
    int rc = check_query(q);
    if (rc) return rc;
    hipSetDevice(o->dev);
    const kc_query qq = tune(o, q);
    std::memset(r, 0, sizeof *r);
    if (qq.k <= 2) {
        // closed forms: every vertex is a 1-clique, every edge a 2-clique
        r->algo = qq.algo;
        r->gran = qq.gran;
        r->part_size = qq.part_size;
        const uint64_t ntasks = qq.gran == KC_GRAN_EDGE ? o->m : o->n;
        const uint64_t nsample = ntasks > offset ? (ntasks - offset + stride - 1) / stride : 0;
        r->tasks = nsample;
        if (qq.k == 1) {
            r->count = o->n > offset ? (o->n - offset + stride - 1) / stride : 0;
        } else if (qq.gran == KC_GRAN_EDGE || stride == 1) {
            r->count = stride == 1 ? o->m : nsample;
        } else {  // out-degrees of the sampled vertices
            std::vector<uint32_t> rp((size_t)o->n + 1);
            if ((rc = kc_oriented_export(o, rp.data(), nullptr, nullptr))) return rc;
            for (uint64_t u = offset; u < o->n; u += stride) r->count += rp[u + 1] - rp[u];
        }
        return KC_OK;
    }
    kc_oriented *om = const_cast<kc_oriented *>(o);
    QueryRun run{o, qq};
    run.sample = stride;
    run.offset = offset;
    std::vector<QueryRun> qs{run};
    std::vector<kc_result> res;
    LaunchStats ls;
    om->scr.words = &om->words;
    rc = run_queries(om->scr, om->stream, qs, res, &ls);
    if (rc) return rc;
    fill_result(r, res[0], ls);
    return r->overflow ? fail(KC_ERR_OVERFLOW, "k-clique count exceeds 2^64-1") : KC_OK;
}

extern "C" int kc_count(const kc_oriented *o, const kc_query *q, kc_result *r)
{
    return count_tasks(o, q, 1, 0, r);
}

extern "C" int kc_count_sampled(const kc_oriented *o, const kc_query *q, uint32_t stride, uint32_t offset,
                                kc_result *r)
{
    return count_tasks(o, q, stride, offset, r);
}

extern "C" int kc_count_local(const kc_oriented *o, const kc_query *q, uint64_t *local, kc_result *r)
{
    if (!o || !q || !r || (!local && o->n)) return fail(KC_ERR_ARG, "kc_count_local: null argument");
    int rc = check_query(q);
    if (rc) return rc;
    hipSetDevice(o->dev);
    kc_query qq = tune(o, q);
    std::memset(r, 0, sizeof *r);
    r->algo = qq.algo;
    r->gran = qq.gran;
    r->part_size = qq.part_size;
    const uint32_t n = o->n;
    if (qq.k <= 2) {
        // every vertex is in one 1-clique; in deg(v) = out + in 2-cliques
        std::vector<uint32_t> rp((size_t)n + 1), col(o->m);
        if (qq.k == 2 && (rc = kc_oriented_export(o, rp.data(), col.data(), nullptr))) return rc;
        for (uint32_t v = 0; v < n; ++v) local[v] = qq.k == 1 ? 1 : rp[v + 1] - rp[v];
        if (qq.k == 2)
            for (uint32_t x : col) local[x]++;
        r->count = qq.k == 1 ? n : o->m;
        r->tasks = qq.gran == KC_GRAN_EDGE ? o->m : o->n;
        return KC_OK;
    }
    kc_oriented *om = const_cast<kc_oriented *>(o);
    if ((rc = om->scr.local.ensure(sizeof(uint64_t) * ((size_t)n + 1)))) return rc;
    KC_HIP(hipMemsetAsync(om->scr.local.p, 0, sizeof(uint64_t) * (size_t)n, om->stream));
    std::vector<QueryRun> qs{QueryRun{o, qq}};
    std::vector<kc_result> res;
    LaunchStats ls;
    om->scr.words = &om->words;
    rc = run_queries(om->scr, om->stream, qs, res, &ls, om->scr.local.as<uint64_t>());
    if (rc) return rc;
    if (n) {
        KC_HIP(hipMemcpyAsync(local, om->scr.local.p, sizeof(uint64_t) * (size_t)n, hipMemcpyDeviceToHost, om->stream));
        KC_HIP(hipStreamSynchronize(om->stream));
    }
    fill_result(r, res[0], ls);
    return r->overflow ? fail(KC_ERR_OVERFLOW, "k-clique count exceeds 2^64-1") : KC_OK;
}

extern "C" int kc_batch_count(kc_oriented *const *gs, const kc_query *qs, size_t nq, kc_result *results,
                              kc_batch_stats *stats)
{
    if ((!gs || !qs || !results) && nq) return fail(KC_ERR_ARG, "kc_batch_count: null argument");
    std::vector<QueryRun> runs;
    std::vector<size_t> idx;
    runs.reserve(nq);
    int dev = -1;
    for (size_t i = 0; i < nq; ++i) {
        if (!gs[i]) return fail(KC_ERR_ARG, "kc_batch_count: null graph %zu", i);
        int rc = check_query(&qs[i]);
        if (rc) return rc;
        if (dev < 0) dev = gs[i]->dev;
        if (gs[i]->dev != dev) return fail(KC_ERR_ARG, "kc_batch_count: graphs on different devices");
        const kc_query t = tune(gs[i], &qs[i]);
        std::memset(&results[i], 0, sizeof(kc_result));
        results[i].algo = t.algo;
        results[i].gran = t.gran;
        results[i].part_size = t.part_size;
        if (t.k <= 2) {
            results[i].count = t.k == 1 ? gs[i]->n : gs[i]->m;
            continue;
        }
        runs.push_back(QueryRun{gs[i], t});
        idx.push_back(i);
    }
    if (stats) std::memset(stats, 0, sizeof *stats);
    if (runs.empty()) return KC_OK;
    hipSetDevice(dev);
    kc_oriented *first = runs[0].o == nullptr ? nullptr : const_cast<kc_oriented *>(runs[0].o);
    std::vector<kc_result> res;
    LaunchStats ls;
    int rc = run_queries(first->batch_scr, first->stream, runs, res, &ls);
    if (rc) return rc;
    bool ovf = false;
    for (size_t j = 0; j < runs.size(); ++j) {
        results[idx[j]].count = res[j].count;
        results[idx[j]].overflow = res[j].overflow;
        ovf |= res[j].overflow != 0;
    }
    if (stats) {
        stats->total_ms = ls.count_ms + ls.prep_ms;
        stats->count_ms = ls.count_ms;
        stats->tasks = ls.tasks;
        stats->queries = runs.size();
    }
    return ovf ? fail(KC_ERR_OVERFLOW, "a k-clique count exceeds 2^64-1") : KC_OK;
}
