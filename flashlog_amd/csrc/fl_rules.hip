// Rule-bank scoring accumulators (rules/shared_inference.py:12-245, the
// dense-accumulator branch :87-96,200-206,224-237).
//
// A chunk of rules has been grounded for every source b: a COO state
// (b, rule l, entity e, v) with v the path count (or 0/1 with Boolean paths).
// Per rank k the scores are
//   sum:  S_k[b, e] += sum over the chunk's rules, in rule order, of v * W[rule, k]
//   max:  S_k[b, e]  = max(S_k[b, e], v * W[rule, k])      (W >= 0)
// accumulated over chunks in a dense [K, B*E] buffer; then every (k, b) row
// is normalized by its sum (clamped to 1e-30) and the ranks are summed (or
// maxed with final_max) into one [B*E] score.
#include "fl_abi.h"
#include "fl_common.h"
#include "fl_scan.h"

namespace fl {

constexpr int RB_NT = 256;

// Maxima: thread per state entry; the maximum of nonnegative values is
// exact in any order (the integer order of their bits), so atomics give the
// same bits on every run.  (Sums go through fl_sparse_channel_weighted_add,
// one writer per accumulator slot.)
__global__ __launch_bounds__(RB_NT) void k_rule_accum_max(const int64_t *__restrict__ sb,
                                                         const int64_t *__restrict__ sl,
                                                         const int64_t *__restrict__ se,
                                                         const float *__restrict__ sv, int64_t nnz,
                                                         const float *__restrict__ W, int64_t K, int64_t B,
                                                         int64_t L, int64_t E, float *__restrict__ dense) {
    const int64_t i = (int64_t)blockIdx.x * RB_NT + threadIdx.x;
    if (i >= nnz) return;
    if (sb[i] < 0 || sb[i] >= B || se[i] < 0 || se[i] >= E || sl[i] < 0 || sl[i] >= L) return;  // outside the shape
    const int64_t key = sb[i] * E + se[i];
    const float v = sv[i];
    const float *wr = W + sl[i] * K;
    for (int64_t k = 0; k < K; ++k) {
        const float x = fl_mul(v, wr[k]);
        if (x > 0.0f) atomicMax((unsigned int *)(dense + k * B * E + key), __float_as_uint(x));
    }
}

// Sums through LDS (entities of a source fit a workgroup's LDS): row
// pointers of the coalesced chunk state first (thread per entry; err 1: an
// index outside [B, L, E], 2: rows out of order, 3: entities not strictly
// increasing within a row), then a workgroup per (source b, rank k) holds
// acc[e] for every entity in LDS and walks the chunk's rules in order: rule
// l's entries (distinct entities: no two lanes add into one slot) add
// v * W[l, k] to acc, a barrier between rules.  Per entity the terms are
// thus added from 0 in rule order, then the chunk's sum is added to the
// dense accumulator: the order of k_cs_weighted_add, without the merge.
constexpr int RA_NT = 256;

__global__ void k_ra_zero(unsigned long long *err) {
    if (threadIdx.x == 0) *err = 0;
}
constexpr int64_t RA_LDS_MAX_E = 16384;  // 64 KB of LDS per workgroup

__global__ __launch_bounds__(RA_NT) void k_ra_rows(const int64_t *__restrict__ sb, const int64_t *__restrict__ sl,
                                                  const int64_t *__restrict__ se, int64_t nnz, int64_t B, int64_t L,
                                                  int64_t E, int64_t *__restrict__ row_ptr,
                                                  unsigned long long *__restrict__ err) {
    const int64_t i = (int64_t)blockIdx.x * RA_NT + threadIdx.x;
    if (i >= nnz) return;
    const int64_t b = sb[i], l = sl[i], e = se[i];
    if (b < 0 || b >= B || l < 0 || l >= L || e < 0 || e >= E) {
        atomicMax(err, 1ull);
        return;
    }
    const int64_t r = b * L + l;
    int64_t rp = -1;
    if (i > 0) {
        const int64_t pb = sb[i - 1], pl = sl[i - 1];
        rp = (pb >= 0 && pb < B && pl >= 0 && pl < L) ? pb * L + pl : r;
        if (rp > r) {
            atomicMax(err, 2ull);
            return;
        }
        if (rp == r && se[i - 1] >= e) {
            atomicMax(err, 3ull);
            return;
        }
    }
    for (int64_t q = rp + 1; q <= r; ++q) row_ptr[q] = i;
    if (i == nnz - 1)
        for (int64_t q = r + 1; q <= B * L; ++q) row_ptr[q] = nnz;
}

__global__ __launch_bounds__(RA_NT) void k_ra_sum(const int64_t *__restrict__ se, const float *__restrict__ sv,
                                                 const int64_t *__restrict__ row_ptr,
                                                 const unsigned long long *__restrict__ err,
                                                 const float *__restrict__ W, int64_t K, int64_t B, int64_t L,
                                                 int64_t E, float *__restrict__ dense) {
    extern __shared__ float acc[];  // [E]
    if (*err != 0) return;          // a malformed state adds nothing
    const int64_t b = blockIdx.x, k = blockIdx.y;
    const int t = threadIdx.x;
    for (int64_t e = t; e < E; e += RA_NT) acc[e] = 0.0f;
    __syncthreads();
    for (int64_t l = 0; l < L; ++l) {
        const int64_t a = row_ptr[b * L + l], z = row_ptr[b * L + l + 1];
        const float wk = W[l * K + k];
        for (int64_t i = a + t; i < z; i += RA_NT) {
            const int64_t e = se[i];
            acc[e] = fl_add(acc[e], fl_mul(sv[i], wk));
        }
        __syncthreads();
    }
    float *drow = dense + k * B * E + b * E;
    for (int64_t e = t; e < E; e += RA_NT) {
        const float x = acc[e];
        if (x != 0.0f) drow[e] = fl_add(drow[e], x);
    }
}

// ---------------------------------------------------------------------------
// Grounding of a chunk of rules from a block of sources in one launch: a
// workgroup per (source b, rule r) walks the whole body, keeping the state
// (entity -> path count) in LDS, and leaves the final state as a segment of a
// pool; k_rg_sum then adds the segments of a source in rule order.  The
// general path (one sparse hop per operator for all rows) costs some 27
// launches and two host reads per operator, whatever the state's size.
//   Counts are integers; the sums a state holds stay below 2^24, where every
// float sum of them is exact in any order, else the row reports RG_LIMIT and
// the caller takes the general path, as it does for a row of more than
// RG_ITEMS_MAX edges in a step (which the general path spreads over the
// chip).  A chunk that overruns the pool reports how much it asks for.
// Chunks before a report are added and stay so;
// later chunks are left, and so are listed rows that begin after the report.
// (k_rg_rows reads the report as it was at its start: asked for past the L2
// by every row, 1024 sources took 2732 us instead of 2435.)
//   k_rg_rows    state in a hash table (RG_TAB slots, at most RG_CAP
//                entities): five workgroups a CU;
//   k_rg_dense   the rows that outgrow it, from a list: two dense arrays of
//                E counts.
// Bound by latency: per operator a binary search of the node's groups and
// the edges' columns, some ten dependent loads; C3, 10 sources x 42 rules:
// 1030 -> 393 us a scored head with the sums and the collection below
// (k_rg_rows 68, k_rg_dense 53, k_rg_sum 27 us).
constexpr int RG_NT = 128, RG_TAB = 2048, RG_CAP = 1536;
constexpr int RG_DENSE_NT = 512;
constexpr int RG_ITEMS_MAX = 1 << 20;
constexpr unsigned long long RG_PATHS_MAX = 1ull << 24;
enum { RG_SOURCE = 1, RG_POOL = 2, RG_LIMIT = 3 };  // the larger report stands

struct RgSeg {
    int64_t base;  // n == 0: the step, from 1, that left the row empty
    int64_t n;
};

struct RgPool {
    RgSeg *seg;               // [nb * C] final state of a row
    int32_t *ent;             // [cap]
    float *val;               // [cap]
    int64_t cap;
    int32_t *over;            // rows for k_rg_dense
    // [0] pool entries taken, [1] status, [2] listed rows, [3] next row to claim, [4] the status at the launch's start
    unsigned long long *ctr;
};
constexpr int RG_CTR = 5;

// status: [0] the worst report of the calls so far, [1] chunks added, [2] the
// pool entries that the chunk of a first RG_POOL asks for, [3] the steps that
// the added chunks would take one by one: a chunk's longest body, or as many
// as leave every row empty
__global__ void k_rg_zero(unsigned long long *ctr, const unsigned long long *status) {
    if (threadIdx.x < RG_CTR) ctr[threadIdx.x] = threadIdx.x == 1 || threadIdx.x == 4 ? *status : 0ull;
}

__global__ __launch_bounds__(RB_NT) void k_rg_status(RgPool pool, const int32_t *__restrict__ lens, int64_t C,
                                                     int64_t rows, unsigned long long *status) {
    __shared__ int steps;
    if (threadIdx.x == 0) steps = 0;
    // (the words, which the common case needs, are requested together)
    const unsigned long long taken = pool.ctr[0], report = pool.ctr[1];
    const unsigned long long before = status[0], added = status[1], done = status[3];
    int mine = 0;  // some row is left: to the end of the longest body
    for (int64_t r = threadIdx.x; r < C; r += RB_NT) mine = max(mine, (int)lens[r]);
    if (taken == 0) {
        mine = 0;
        for (int64_t r = threadIdx.x; r < rows; r += RB_NT) mine = max(mine, (int)pool.seg[r].base);
    }
    __syncthreads();
    if (mine > 0) atomicMax(&steps, mine);
    __syncthreads();
    if (threadIdx.x != 0) return;
    if (report == 0) {
        status[1] = added + 1;
        status[3] = done + steps;
    }
    if (before == 0) status[2] = taken;
    status[0] = report;
}

// Expands n entries (get(i, node, count), count 0: no entry) through relation
// rel of side s: put(entity, count) for every edge.  A batch of NT entries at
// a time: each finds its group, the edges are spread over the threads by a
// search in the batch's prefix counts.  Returns the edges (capped: a batch
// that passes RG_ITEMS_MAX is not expanded), uniform over the workgroup.
template <int NT, typename Get, typename Put>
__device__ __forceinline__ int64_t rg_expand(const fl_side &s, int rel, int n, int *pre, int32_t *first, uint32_t *cnt,
                                             int *scan_lds, Get get, Put put) {
    const int t = threadIdx.x;
    int64_t items = 0;
    for (int base = 0; base < n; base += NT) {
        int32_t node = 0, c = 0, st = 0;
        uint32_t v = 0;
        if (base + t < n) get(base + t, node, v);
        if (__syncthreads_or(v != 0) == 0) continue;  // (also: the last batch's edges are done)
        if (v != 0) {
            int64_t lo = s.row_group_ptr[node], hi = s.row_group_ptr[node + 1];
            const int64_t end = hi;
            while (lo < hi) {
                const int64_t mid = lo + ((hi - lo) >> 1);
                if ((int)s.group_rel[mid] < rel) lo = mid + 1;
                else hi = mid;
            }
            if (lo < end && (int)s.group_rel[lo] == rel) {
                c = s.group_count[lo];
                st = s.group_start[lo];
            }
        }
        int total;
        pre[t] = fl_block_excl_scan<NT>(c, scan_lds, &total);
        first[t] = st;
        cnt[t] = v;
        __syncthreads();
        items += total;
        if (items > RG_ITEMS_MAX) return items;
        for (int k = t; k < total; k += NT) {
            int lo = 0, hi = NT;  // the last entry whose prefix is at most k
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (pre[mid] <= k) lo = mid;
                else hi = mid;
            }
            put(s.col_ind[(int64_t)first[lo] + (k - pre[lo])], cnt[lo]);
        }
    }
    __syncthreads();
    return items;
}

__global__ __launch_bounds__(RG_NT) void k_rg_rows(fl_side ori, fl_side inv, const int64_t *__restrict__ sources,
                                                  const int64_t *__restrict__ ops, const int32_t *__restrict__ lens,
                                                  int64_t C, int64_t steps, int64_t E, int64_t R, int boolean,
                                                  RgPool pool) {
    __shared__ int32_t key[RG_TAB];
    __shared__ uint32_t count[RG_TAB];
    __shared__ int32_t node_of[RG_CAP + RG_NT];
    __shared__ uint32_t count_of[RG_CAP + RG_NT];
    __shared__ int pre[RG_NT];
    __shared__ int32_t first[RG_NT];
    __shared__ uint32_t vcnt[RG_NT];
    __shared__ int scan_lds[RG_NT / FL_WAVE + 1];
    __shared__ int n_lds, keys_lds, over_lds;
    __shared__ unsigned long long paths_lds, base_lds;
    const int t = threadIdx.x;
    const int64_t row = blockIdx.x, b = row / C, r = row - b * C;
    // (both are requested before either is looked at)
    const unsigned long long before = pool.ctr[4];
    const int64_t src = sources[b];
    if ((before != 0) | (src < 0) | (src >= E)) {  // uniform
        if (before == 0 && t == 0) {               // else nothing of this chunk is used
            atomicMax(&pool.ctr[1], (unsigned long long)RG_SOURCE);
            pool.seg[row] = {0, 0};
        }
        return;
    }
    if (t == 0) {
        node_of[0] = (int32_t)src;
        count_of[0] = 1;
    }
    int n = 1;
    bool limit = false, over = false;
    int step = 0;
    for (; step < lens[r] && n > 0; ++step) {
        const int64_t op = ops[r * steps + step];
        if (op == 2 * R) continue;  // the identity
        if (op < 0 || op > 2 * R) {
            n = 0;
            continue;
        }
        __syncthreads();  // the last step's list is made, and its table read
        for (int q = t; q < RG_TAB; q += RG_NT) {
            key[q] = -1;
            count[q] = 0;
        }
        if (t == 0) {
            n_lds = keys_lds = over_lds = 0;
            paths_lds = 0;
        }
        __syncthreads();
        unsigned long long paths = 0;
        const volatile int *full = &over_lds;
        const int64_t items = rg_expand<RG_NT>(
            op >= R ? inv : ori, (int)(op >= R ? op - R : op), n, pre, first, vcnt, scan_lds,
            [&](int i, int32_t &node, uint32_t &v) {
                node = node_of[i];
                v = count_of[i];
            },
            [&](int32_t e, uint32_t v) {
                paths += v;
                // a thread adds at most one entity after the table is called
                // full: at most RG_CAP + RG_NT of its RG_TAB slots are taken
                if (*full) return;
                uint32_t h = ((uint32_t)e * 2654435761u) >> 21;
                for (int probe = 0; probe < RG_TAB; ++probe, h = (h + 1) & (RG_TAB - 1)) {
                    const int32_t old = atomicCAS(&key[h], -1, e);
                    if (old == -1 && atomicAdd(&keys_lds, 1) >= RG_CAP) over_lds = 1;
                    if (old == -1 || old == e) {
                        atomicAdd(&count[h], v);
                        break;
                    }
                }
            });
        atomicAdd(&paths_lds, paths);
        __syncthreads();
        limit = items > RG_ITEMS_MAX || (!boolean && paths_lds >= RG_PATHS_MAX);
        over = over_lds != 0;
        if (limit || over) break;  // uniform
        for (int q = t; q < RG_TAB; q += RG_NT)
            if (key[q] >= 0) {
                const int i = atomicAdd(&n_lds, 1);
                node_of[i] = key[q];
                count_of[i] = boolean ? 1u : count[q];
            }
        __syncthreads();
        n = n_lds;
    }
    if (limit || over) {
        if (t == 0) {
            pool.seg[row] = {0, 0};
            if (limit) atomicMax(&pool.ctr[1], (unsigned long long)RG_LIMIT);
            else pool.over[atomicAdd(&pool.ctr[2], 1ull)] = (int32_t)row;
        }
        return;
    }
    if (t == 0) {
        base_lds = n > 0 ? atomicAdd(&pool.ctr[0], (unsigned long long)n) : (unsigned long long)step;
        const bool fits = n == 0 || (int64_t)base_lds + n <= pool.cap;
        if (!fits) atomicMax(&pool.ctr[1], (unsigned long long)RG_POOL);
        pool.seg[row] = {(int64_t)base_lds, fits ? (int64_t)n : 0};
    }
    __syncthreads();
    const int64_t base = (int64_t)base_lds;
    if (n == 0 || base + n > pool.cap) return;
    for (int i = t; i < n; i += RG_NT) {
        pool.ent[base + i] = node_of[i];
        pool.val[base + i] = (float)count_of[i];
    }
}

__global__ __launch_bounds__(RG_DENSE_NT) void k_rg_dense(fl_side ori, fl_side inv,
                                                         const int64_t *__restrict__ sources,
                                                         const int64_t *__restrict__ ops,
                                                         const int32_t *__restrict__ lens, int64_t C, int64_t steps,
                                                         int E, int64_t R, int boolean, RgPool pool) {
    extern __shared__ uint32_t rg_counts[];  // two arrays of E counts
    __shared__ int pre[RG_DENSE_NT];
    __shared__ int32_t first[RG_DENSE_NT];
    __shared__ uint32_t vcnt[RG_DENSE_NT];
    __shared__ int scan_lds[RG_DENSE_NT / FL_WAVE + 1];
    __shared__ unsigned long long paths_lds, base_lds;
    __shared__ int claim;
    const int t = threadIdx.x;
    const int rows = (int)pool.ctr[2];
    if ((int)blockIdx.x >= rows) return;
    for (;;) {
        __syncthreads();  // the last row is done with the LDS arrays
        if (t == 0) {
            // (one thread asks: the report may come while this kernel runs)
            const unsigned long long at = atomicAdd(&pool.ctr[3], 1ull);
            // (a chunk that only overran the pool is walked to its end, which tells how much it asks for)
            const unsigned long long now = __hip_atomic_load(&pool.ctr[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            claim = now != 0 && now != RG_POOL ? rows : (int)at;
        }
        __syncthreads();
        const int ci = __builtin_amdgcn_readfirstlane(claim);  // uniform: scalar registers
        if (ci >= rows) break;
        const int64_t row = pool.over[ci], b = row / C, r = row - b * C;
        uint32_t *cur = rg_counts, *nxt = rg_counts + E;
        for (int e = t; e < 2 * E; e += RG_DENSE_NT) rg_counts[e] = 0;
        __syncthreads();
        if (t == 0) cur[sources[b]] = 1;  // (k_rg_rows checked the source)
        bool limit = false, none = false;
        int step = 0;
        for (; step < lens[r] && !none; ++step) {
            const int64_t op = ops[r * steps + step];
            if (op == 2 * R) continue;
            if (op < 0 || op > 2 * R) {
                none = true;
                continue;
            }
            if (t == 0) paths_lds = 0;
            __syncthreads();
            unsigned long long paths = 0;
            const int64_t items = rg_expand<RG_DENSE_NT>(
                op >= R ? inv : ori, (int)(op >= R ? op - R : op), E, pre, first, vcnt, scan_lds,
                [&](int i, int32_t &node, uint32_t &v) {
                    node = i;
                    v = cur[i];
                },
                [&](int32_t e, uint32_t v) {
                    paths += v;
                    atomicAdd(&nxt[e], v);
                });
            atomicAdd(&paths_lds, paths);
            __syncthreads();
            limit = items > RG_ITEMS_MAX || (!boolean && paths_lds >= RG_PATHS_MAX);
            if (limit) break;  // uniform
            none = items == 0;
            for (int e = t; e < E; e += RG_DENSE_NT) {
                cur[e] = 0;
                if (boolean && nxt[e] > 1) nxt[e] = 1;
            }
            uint32_t *x = cur;
            cur = nxt;
            nxt = x;
            __syncthreads();
        }
        __syncthreads();
        int mine = 0;
        if (!limit && !none)
            for (int e = t; e < E; e += RG_DENSE_NT) mine += cur[e] != 0;
        int n;
        const int at = fl_block_excl_scan<RG_DENSE_NT>(mine, scan_lds, &n);
        if (t == 0) {
            if (limit) atomicMax(&pool.ctr[1], (unsigned long long)RG_LIMIT);
            base_lds = n > 0 ? atomicAdd(&pool.ctr[0], (unsigned long long)n) : (unsigned long long)step;
            const bool fits = n == 0 || (int64_t)base_lds + n <= pool.cap;
            if (!fits) atomicMax(&pool.ctr[1], (unsigned long long)RG_POOL);
            pool.seg[row] = {(int64_t)base_lds, fits ? (int64_t)n : 0};
        }
        __syncthreads();
        const int64_t base = (int64_t)base_lds;
        if (n == 0 || base + n > pool.cap) continue;
        int64_t o = base + at;
        for (int e = t; e < E; e += RG_DENSE_NT)
            if (cur[e] != 0) {
                pool.ent[o] = e;
                pool.val[o] = (float)cur[e];
                ++o;
            }
    }
}

// Workgroup per (source b, rank k): the source's segments in rule order into
// an accumulator of every entity in LDS (a segment's entities are distinct),
// then the chunk's sum (or maximum) into the dense accumulator: the terms and
// the order of k_ra_sum and k_rule_accum_max.  Eight segments' first entries
// are requested together, so that a rule does not wait for its own loads.
template <bool MAX>
__global__ __launch_bounds__(RA_NT) void k_rg_sum(RgPool pool, const float *__restrict__ W, int64_t K, int64_t B,
                                                 int64_t C, int64_t E, float *__restrict__ dense) {
    extern __shared__ float acc[];  // [E]
    constexpr int U = 8;
    if (pool.ctr[1] != 0) return;   // the caller does not use the accumulator
    const int64_t b = blockIdx.x, k = blockIdx.y;
    const int t = threadIdx.x;
    for (int64_t e = t; e < E; e += RA_NT) acc[e] = 0.0f;
    const RgSeg *seg = pool.seg + b * C;
    for (int64_t r0 = 0; r0 < C; r0 += U) {
        RgSeg sg[U];
        int32_t e0[U];
        float v0[U], wk[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t r = r0 + u < C ? r0 + u : C - 1;
            sg[u] = seg[r];
            wk[u] = W[r * K + k];
            if (r0 + u >= C) sg[u].n = 0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = t < sg[u].n;
            e0[u] = in ? pool.ent[sg[u].base + t] : -1;
            v0[u] = in ? pool.val[sg[u].base + t] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (sg[u].n == 0) continue;  // uniform
            __syncthreads();             // the accumulator is cleared, or the rule before is added
            auto add = [&](int32_t e, float v) {
                const float x = fl_mul(v, wk[u]);
                acc[e] = MAX ? (x > acc[e] ? x : acc[e]) : fl_add(acc[e], x);
            };
            if (e0[u] >= 0) add(e0[u], v0[u]);
            for (int64_t i = RA_NT + t; i < sg[u].n; i += RA_NT) add(pool.ent[sg[u].base + i], pool.val[sg[u].base + i]);
        }
    }
    __syncthreads();
    float *drow = dense + k * B * E + b * E;
    for (int64_t e = t; e < E; e += RA_NT) {
        const float x = acc[e];
        if (x != 0.0f) drow[e] = MAX ? (x > drow[e] ? x : drow[e]) : fl_add(drow[e], x);
    }
}

// The scored entities of [B, E]: per 256 cells their number, and after a scan
// the coordinates and scores in order.
__global__ __launch_bounds__(RB_NT) void k_rule_count(const float *__restrict__ total, int64_t n,
                                                     int32_t *__restrict__ cnt) {
    __shared__ int wsum[RB_NT / FL_WAVE];
    const int64_t q = (int64_t)blockIdx.x * RB_NT + threadIdx.x;
    const unsigned long long m = __ballot(q < n && total[q] != 0.0f);
    if (fl_lane() == 0) wsum[threadIdx.x / FL_WAVE] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int w = 0; w < RB_NT / FL_WAVE; ++w) s += wsum[w];
        cnt[blockIdx.x] = s;
    }
}

__global__ __launch_bounds__(RB_NT) void k_rule_fill(const float *__restrict__ total, int64_t n, int64_t E,
                                                    int64_t row0, const int64_t *__restrict__ off,
                                                    int64_t *__restrict__ ob, int64_t *__restrict__ oe,
                                                    float *__restrict__ ov) {
    __shared__ int wsum[RB_NT / FL_WAVE];
    const int64_t q = (int64_t)blockIdx.x * RB_NT + threadIdx.x;
    const float x = q < n ? total[q] : 0.0f;
    const unsigned long long m = __ballot(x != 0.0f);
    const int w = threadIdx.x / FL_WAVE;
    if (fl_lane() == 0) wsum[w] = __popcll(m);
    __syncthreads();
    if (x == 0.0f) return;
    int64_t o = off[blockIdx.x] + __popcll(m & ((1ull << fl_lane()) - 1));
    for (int k = 0; k < w; ++k) o += wsum[k];
    ob[o] = row0 + q / E;
    oe[o] = q % E;
    ov[o] = x;
}

__global__ void k_rule_info(const int64_t *total, const unsigned long long *status, int64_t *info) {
    info[0] = *total;
    info[1] = status ? (int64_t)*status : 0;
}

// Workgroup per (k, b): the row's sum in a fixed order.
__global__ __launch_bounds__(RB_NT) void k_rule_rowsum(const float *__restrict__ dense, int64_t E,
                                                      float *__restrict__ rowsum) {
    __shared__ float red[RB_NT];
    const float *row = dense + (int64_t)blockIdx.x * E;
    float s = 0.0f;
#pragma unroll 8
    for (int64_t e = threadIdx.x; e < E; e += RB_NT) s = fl_add(s, row[e]);
    red[threadIdx.x] = s;
    __syncthreads();
    for (int st = RB_NT / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) red[threadIdx.x] = fl_add(red[threadIdx.x], red[threadIdx.x + st]);
        __syncthreads();
    }
    if (threadIdx.x == 0) rowsum[blockIdx.x] = red[0];
}

// Thread per (b, e): the normalized ranks combined in rank order.
__global__ __launch_bounds__(RB_NT) void k_rule_combine(const float *__restrict__ dense,
                                                       const float *__restrict__ rowsum, int64_t K, int64_t B,
                                                       int64_t E, int final_max, float *__restrict__ total) {
    const int64_t q = (int64_t)blockIdx.x * RB_NT + threadIdx.x;
    if (q >= B * E) return;
    const int64_t b = q / E;
    float t = 0.0f;
    for (int64_t k = 0; k < K; ++k) {
        const float x = dense[k * B * E + q];
        if (x == 0.0f) continue;
        const float d = rowsum[k * B + b];
        const float p = __fdiv_rn(x, d < 1e-30f ? 1e-30f : d);
        t = final_max ? (p > t ? p : t) : fl_add(t, p);
    }
    total[q] = t;
}

}  // namespace fl

extern "C" {

size_t fl_rule_accumulate_bytes(int64_t nnz, int64_t B, int64_t L) {
    if (nnz < 0 || B < 0 || L < 0) return 0;
    const size_t merge = ((fl_sparse_channel_sum_bytes(nnz, B, L) + 255) & ~(size_t)255) + 256;
    const size_t lds = ((sizeof(int64_t) * (size_t)(B * L + 1) + 255) & ~(size_t)255) + 256;
    return merge > lds ? merge : lds;
}

int fl_rule_accumulate(void *stream, const int64_t *sb, const int64_t *sl, const int64_t *se, const float *sv,
                       int64_t nnz, const float *W, int64_t K, int64_t B, int64_t L, int64_t E, int is_max,
                       float *dense, void *ws, size_t ws_bytes) {
    if (nnz < 0 || K < 1 || B < 0 || L < 0 || E < 0) return fl::fl_fail(FL_ERR_ARG, "rule_accumulate: bad shape");
    if (nnz == 0) return FL_OK;
    if (!sb || !sl || !se || !sv || !W || !dense) return fl::fl_fail(FL_ERR_ARG, "rule_accumulate: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (is_max) {
        FL_LAUNCH("k_rule_accum_max", fl::k_rule_accum_max, dim3((unsigned)((nnz + fl::RB_NT - 1) / fl::RB_NT)),
                  dim3(fl::RB_NT), 0, st, sb, sl, se, sv, nnz, W, K, B, L, E, dense);
        return fl::fl_check_launch("rule_accumulate");
    }
    if (!ws || ws_bytes < fl_rule_accumulate_bytes(nnz, B, L))
        return fl::fl_fail(FL_ERR_ARG, "rule_accumulate: workspace too small");
    if (E <= fl::RA_LDS_MAX_E && B * K <= 0x7fffffff && K <= 65535) {
        // rules in order through an LDS accumulator per (source, rank)
        int64_t *row_ptr = (int64_t *)ws;
        unsigned long long *err =
            (unsigned long long *)((char *)ws + ((sizeof(int64_t) * (size_t)(B * L + 1) + 255) & ~(size_t)255));
        FL_LAUNCH("k_fill_u64", fl::k_ra_zero, dim3(1), dim3(64), 0, st, err);
        FL_LAUNCH("k_ra_rows", fl::k_ra_rows, dim3((unsigned)((nnz + fl::RA_NT - 1) / fl::RA_NT)), dim3(fl::RA_NT), 0,
                  st, sb, sl, se, nnz, B, L, E, row_ptr, err);
        FL_LAUNCH("k_ra_sum", fl::k_ra_sum, dim3((unsigned)B, (unsigned)K), dim3(fl::RA_NT),
                  sizeof(float) * (size_t)E, st, se, sv, row_ptr, err, W, K, B, L, E, dense);
        return fl::fl_check_launch("rule_accumulate");
    }
    // rank the entries of every (b, e) in rule order, then one writer per slot
    const size_t cs = (fl_sparse_channel_sum_bytes(nnz, B, L) + 255) & ~(size_t)255;
    int64_t *plan = (int64_t *)((char *)ws + cs);
    int rc = fl_sparse_channel_sum_plan(stream, sb, sl, se, nnz, B, L, E, ws, cs, plan);
    if (rc != FL_OK) return rc;
    return fl_sparse_channel_weighted_add(stream, sb, sl, se, sv, nnz, B, L, E, W, K, ws, dense);
}

// workspace of fl_rule_ground: counters, segments, overflow list, pool
static size_t rg_layout(int64_t nb, int64_t C, int64_t cap, char *base, fl::RgPool *p) {
    size_t off = 0;
    auto take = [&](size_t b) { char *q = base ? base + off : nullptr; off += (b + 255) & ~(size_t)255; return q; };
    const int64_t rows = nb * C > 0 ? nb * C : 1;
    p->ctr = (unsigned long long *)take(fl::RG_CTR * sizeof(unsigned long long));
    p->seg = (fl::RgSeg *)take(sizeof(fl::RgSeg) * (size_t)rows);
    p->over = (int32_t *)take(sizeof(int32_t) * (size_t)rows);
    p->ent = (int32_t *)take(sizeof(int32_t) * (size_t)cap);
    p->val = (float *)take(sizeof(float) * (size_t)cap);
    p->cap = cap;
    return off;
}

size_t fl_rule_ground_bytes(int64_t nb, int64_t C, int64_t pool) {
    if (nb < 0 || C < 0 || pool < 0) return 0;
    fl::RgPool p;
    return rg_layout(nb, C, pool, nullptr, &p);
}

int64_t fl_rule_ground_max_entities(void) { return fl::RA_LDS_MAX_E; }

int fl_rule_ground(void *stream, const fl_side *ori, const fl_side *inv, const int64_t *sources, int64_t nb,
                   const int64_t *operators, const int32_t *lengths, int64_t C, int64_t steps, int64_t r_size,
                   const float *W, int64_t K, int64_t E, int boolean_paths, int is_max, float *dense, int64_t pool,
                   void *ws, size_t ws_bytes, int64_t *status) {
    using namespace fl;
    if (!ori || !inv || nb < 0 || C < 0 || steps < 0 || K < 1 || E < 1 || r_size < 0 || pool < 0)
        return fl_fail(FL_ERR_ARG, "rule_ground: bad arguments");
    if (E > RA_LDS_MAX_E) return fl_fail(FL_ERR_ARG, "rule_ground: at most %lld entities", (long long)RA_LDS_MAX_E);
    if (nb * C > 0x7fffffff || K > 65535) return fl_fail(FL_ERR_ARG, "rule_ground: too many rows");
    if (nb * C == 0) return FL_OK;
    if (!sources || !lengths || !W || !dense || !ws || !status || (steps > 0 && !operators))
        return fl_fail(FL_ERR_ARG, "rule_ground: null pointer");
    for (const fl_side *s : {ori, inv})
        if (!s->row_group_ptr || (s->edges > 0 && (!s->col_ind || !s->group_rel || !s->group_start || !s->group_count)))
            return fl_fail(FL_ERR_ARG, "rule_ground: side without CSR arrays");
    if (ws_bytes < fl_rule_ground_bytes(nb, C, pool)) return fl_fail(FL_ERR_ARG, "rule_ground: workspace too small");
    RgPool p;
    (void)rg_layout(nb, C, pool, (char *)ws, &p);
    hipStream_t st = (hipStream_t)stream;
    // (status, given by the caller and zeroed by it, is that of all calls that share it)
    FL_LAUNCH("k_rg_zero", k_rg_zero, dim3(1), dim3(64), 0, st, p.ctr, (const unsigned long long *)status);
    FL_LAUNCH("k_rg_rows", k_rg_rows, dim3((unsigned)(nb * C)), dim3(RG_NT), 0, st, *ori, *inv, sources, operators,
              lengths, C, steps, E, r_size, boolean_paths, p);
    const size_t dense_lds = 2 * sizeof(uint32_t) * (size_t)E;
    if (dense_lds > 65536)
        (void)hipFuncSetAttribute((const void *)k_rg_dense, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)dense_lds);
    FL_LAUNCH("k_rg_dense", k_rg_dense, dim3((unsigned)(nb * C < 256 ? nb * C : 256)), dim3(RG_DENSE_NT), dense_lds, st,
              *ori, *inv, sources, operators, lengths, C, steps, (int)E, r_size, boolean_paths, p);
    FL_LAUNCH("k_rg_sum", is_max ? k_rg_sum<true> : k_rg_sum<false>, dim3((unsigned)nb, (unsigned)K), dim3(RA_NT),
              sizeof(float) * (size_t)E, st, p, W, K, nb, C, E, dense);
    FL_LAUNCH("k_rg_status", k_rg_status, dim3(1), dim3(RB_NT), 0, st, p, lengths, C, nb * C,
              (unsigned long long *)status);
    return fl_check_launch("rule_ground");
}

size_t fl_rule_collect_bytes(int64_t B, int64_t E) {
    if (B < 0 || E < 0) return 0;
    const int64_t blocks = (B * E + fl::RB_NT - 1) / fl::RB_NT;
    return ((sizeof(int32_t) * (size_t)(blocks + 1) + 255) & ~(size_t)255) +
           ((sizeof(int64_t) * (size_t)(blocks + 1) + 255) & ~(size_t)255) + fl::scan_tmp_bytes(blocks + 1);
}

static void rule_collect_layout(int64_t blocks, char *ws, int32_t **cnt, int64_t **off, int64_t **tmp) {
    *cnt = (int32_t *)ws;
    ws += (sizeof(int32_t) * (size_t)(blocks + 1) + 255) & ~(size_t)255;
    *off = (int64_t *)ws;
    ws += (sizeof(int64_t) * (size_t)(blocks + 1) + 255) & ~(size_t)255;
    *tmp = (int64_t *)ws;
}

int fl_rule_collect_plan(void *stream, const float *total, int64_t B, int64_t E, const int64_t *status, void *ws,
                         size_t ws_bytes, int64_t *info) {
    using namespace fl;
    if (B < 0 || E < 0 || !info) return fl_fail(FL_ERR_ARG, "rule_collect: bad arguments");
    const int64_t n = B * E, blocks = (n + RB_NT - 1) / RB_NT;
    if (!ws || ws_bytes < fl_rule_collect_bytes(B, E) || (n > 0 && !total))
        return fl_fail(FL_ERR_ARG, "rule_collect: null pointer or small workspace");
    int32_t *cnt;
    int64_t *off, *tmp;
    rule_collect_layout(blocks, (char *)ws, &cnt, &off, &tmp);
    hipStream_t st = (hipStream_t)stream;
    if (n > 0) FL_LAUNCH("k_rule_count", k_rule_count, dim3((unsigned)blocks), dim3(RB_NT), 0, st, total, n, cnt);
    const int rc = exclusive_scan(st, cnt, off, blocks, tmp);
    if (rc != FL_OK) return rc;
    FL_LAUNCH("k_rule_info", k_rule_info, dim3(1), dim3(1), 0, st, off + blocks, (const unsigned long long *)status,
              info);
    return fl_check_launch("rule_collect_plan");
}

int fl_rule_collect_fill(void *stream, const float *total, int64_t B, int64_t E, int64_t row0, void *ws,
                         int64_t *out_b, int64_t *out_e, float *out_v) {
    using namespace fl;
    if (B < 0 || E < 0) return fl_fail(FL_ERR_ARG, "rule_collect: bad shape");
    const int64_t n = B * E, blocks = (n + RB_NT - 1) / RB_NT;
    if (n == 0) return FL_OK;
    if (!total || !ws || !out_b || !out_e || !out_v) return fl_fail(FL_ERR_ARG, "rule_collect: null pointer");
    int32_t *cnt;
    int64_t *off, *tmp;
    rule_collect_layout(blocks, (char *)ws, &cnt, &off, &tmp);
    FL_LAUNCH("k_rule_fill", k_rule_fill, dim3((unsigned)blocks), dim3(RB_NT), 0, (hipStream_t)stream, total, n, E,
              row0, off, out_b, out_e, out_v);
    return fl_check_launch("rule_collect_fill");
}

int fl_rule_finalize(void *stream, const float *dense, int64_t K, int64_t B, int64_t E, int final_max,
                     float *rowsum, float *total) {
    if (K < 1 || B < 0 || E < 0) return fl::fl_fail(FL_ERR_ARG, "rule_finalize: bad shape");
    if (B * E == 0) return FL_OK;
    if (!dense || !rowsum || !total) return fl::fl_fail(FL_ERR_ARG, "rule_finalize: null pointer");
    hipStream_t st = (hipStream_t)stream;
    FL_LAUNCH("k_rule_rowsum", fl::k_rule_rowsum, dim3((unsigned)(K * B)), dim3(fl::RB_NT), 0, st, dense, E, rowsum);
    FL_LAUNCH("k_rule_combine", fl::k_rule_combine, dim3((unsigned)((B * E + fl::RB_NT - 1) / fl::RB_NT)),
              dim3(fl::RB_NT), 0, st, dense, rowsum, K, B, E, final_max, total);
    return fl::fl_check_launch("rule_finalize");
}

}  // extern "C"
