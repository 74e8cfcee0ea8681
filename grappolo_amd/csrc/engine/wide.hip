// wide.hip -- the whole-GPU persistent colored iteration (see wide.hpp).
//
// Per vertex, the decision is the reference's: the weights to the
// neighbouring communities (buildLocalMapCounter,
// Utility/utilityClusteringFunctions.cpp:172-194), the gain of each and the
// strictly positive maximum with ties to the smaller id and the singleton swap
// rule (max(), :226-259), against the state frozen at the start of the color
// step (the colored sweep, Coloring/parallelLouvainWithColoring.cpp:169-210),
// then the community degree and size updates of the move (:213-217).
#include "wide.hpp"

#include <algorithm>
#include <cstddef>
#include <cstdlib>
#include <cstring>

#include "sweep_device.hpp"

namespace glv {
namespace {

constexpr uint32_t kEmptyKey = 0xFFFFFFFFu;
constexpr int kWWaves = kWBlock / kWave;
constexpr int kWUnroll = 4;  // loads in flight per thread in the gathers
static_assert(kWMidMaxDeg * 3 <= kWMidSlots * 2, "a mid vertex overloads a wavefront's table");
static_assert(kWHeavyMaxDeg * 3 <= kWHeavySlots * 2, "a heavy vertex overloads the table");
static_assert(kWMergeLive * 3 <= kWHeavySlots * 2, "a merged giant overloads the table");
static_assert(kWMidSlots >= kWave, "light-vertex staging exceeds a wavefront's slots");

// slot of a community id in a table of T slots (multiplicative hash, then the
// high bits of the product with T)
__device__ inline uint32_t slot_of(uint32_t key, uint32_t T) {
    return (uint32_t)(((u64)(key * 0x9E3779B1u) * T) >> 32);
}

__device__ inline void lds_insert(uint32_t *keys, double *vals, uint32_t T, uint32_t key, double w) {
    uint32_t h = slot_of(key, T);
    while (true) {
        uint32_t k = keys[h];
        if (k == kEmptyKey) {
            k = atomicCAS(&keys[h], kEmptyKey, key);
            if (k == kEmptyKey) k = key;
        }
        if (k == key) {
            atomicAdd(&vals[h], w);
            return;
        }
        h = h + 1 == T ? 0 : h + 1;
    }
}

__device__ inline double lds_lookup(const uint32_t *keys, const double *vals, uint32_t T, uint32_t key) {
    uint32_t h = slot_of(key, T);
    while (true) {
        const uint32_t k = keys[h];
        if (k == key) return vals[h];
        if (k == kEmptyKey) return 0.0;
        h = h + 1 == T ? 0 : h + 1;
    }
}

// partition of a community id among P (a hash independent of slot_of's, so
// the ids of one partition still spread over a table's slots)
__device__ inline int part_of(uint32_t key, int P) {
    uint32_t h = key * 0x85EBCA6Bu;
    h ^= h >> 13;
    h *= 0xC2B2AE35u;
    h ^= h >> 16;
    return (int)(((u64)h * (u64)P) >> 32);
}

// lds_insert that gives up (false) once every slot was probed
__device__ inline bool lds_insert_bounded(uint32_t *keys, double *vals, uint32_t T, uint32_t key, double w) {
    uint32_t h = slot_of(key, T);
    for (uint32_t probes = 0; probes < T; probes++) {
        uint32_t k = keys[h];
        if (k == kEmptyKey) {
            k = atomicCAS(&keys[h], kEmptyKey, key);
            if (k == kEmptyKey) k = key;
        }
        if (k == key) {
            atomicAdd(&vals[h], w);
            return true;
        }
        h = h + 1 == T ? 0 : h + 1;
    }
    return false;
}

// LDS writes of a wavefront are visible to its other lanes after this
__device__ inline void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// __syncthreads for LDS alone: loads, stores and atomics on global memory stay
// in flight across it (__syncthreads waits for them, which put the read-ahead
// and the moves' atomics on every item's path).
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Reduction scratch of a workgroup (one slot per wavefront).
struct Red {
    double d[kWWaves];
    double e[kWWaves];
    u64 key[kWWaves];
    uint32_t id[kWWaves];
    int32_t n[kWWaves];
    int c[kWWaves];
    int last;    // giant chunk: this workgroup finished the giant's last one
    int32_t to;  // new label of the item's vertex, -1: it stays
};

// Workgroup sum in a fixed order (every thread gets it).
__device__ inline double wg_sum(double v, Red &R) {
    v = wave_sum(v);
    const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
    lds_barrier();
    if (l == 0) R.d[w] = v;
    lds_barrier();
    double r = 0;
    for (int q = 0; q < kWWaves; q++) r += R.d[q];
    return r;
}

// Exclusive prefix sum over the workgroup (one value per thread); *total
// gets the sum.  Uses R.c.
__device__ inline int wg_exscan(int x, Red &R, int *total) {
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    int incl = x;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int y = __shfl_up(incl, o);
        if (lane >= o) incl += y;
    }
    lds_barrier();
    if (lane == kWave - 1) R.c[w] = incl;
    lds_barrier();
    int before = 0, all = 0;
    for (int q = 0; q < kWWaves; q++) {
        const int t = R.c[q];
        if (q < w) before += t;
        all += t;
    }
    *total = all;
    return before + incl - x;
}

// The best move of a vertex so far: its gain as an argmax_key (0: none), the
// target community, the vertex's weight towards it and its size (for the
// singleton swap rule).
struct Cand {
    u64 key = 0;
    uint32_t id = 0xFFFFFFFFu;
    double e = 0;
    int32_t n = 0;
};

__device__ inline void offer(Cand &c, double g, uint32_t y, double e, i64 n) {
    const u64 key = argmax_key(g > 0, g);
    if (key > c.key || (key == c.key && key != 0 && y < c.id)) {
        c.key = key;
        c.id = y;
        c.e = e;
        c.n = (int32_t)n;
    }
}

// One pairing step over DPP control CTRL (or lane xor o when CTRL is 0): the
// other lane's candidate wins on a larger key or an equal key and a smaller id.
template <int CTRL>
__device__ inline void best_step(u64 &key, uint32_t &id, int o) {
    u64 ok;
    uint32_t oid;
    if (CTRL) {
        ok = dpp64<CTRL>(key);
        oid = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)id, CTRL, 0xf, 0xf, false);
    } else {
        ok = (u64)__shfl_xor((long long)key, o);
        oid = (uint32_t)__shfl_xor((int)id, o);
    }
    const bool t = ok > key || (ok == key && oid < id);
    key = t ? ok : key;
    id = t ? oid : id;
}
// Largest key (ties: smallest id) over aligned groups of W lanes (a power of
// two from 4 to 64, the same in every lane), in every lane of the group; the
// pairing is that of group_argmax_key.
__device__ inline void group_best(u64 &key, uint32_t &id, int W) {
    best_step<0xB1>(key, id, 0);               // quad_perm [1,0,3,2]
    best_step<0x4E>(key, id, 0);               // quad_perm [2,3,0,1]
    if (W >= 8) best_step<0x141>(key, id, 0);  // row_half_mirror
    if (W >= 16) best_step<0x140>(key, id, 0); // row_mirror
    if (W >= 32) best_step<0>(key, id, 16);
    if (W >= 64) best_step<0>(key, id, 32);
}
// c becomes the wavefront's best candidate in every lane (its weight and size
// read from the lane that holds it)
__device__ inline void wave_best(Cand &c) {
    u64 key = c.key;
    uint32_t id = c.id;
    group_best(key, id, kWave);
    const u64 holds = __ballot(c.key == key && c.id == id);
    const int src = __ffsll((long long)holds) - 1;
    c.e = __shfl(c.e, src);
    c.n = __shfl(c.n, src);
    c.key = key;
    c.id = id;
}

// best over the workgroup, in the first wavefront only (one barrier; R's slots are
// rewritten only after the caller's next barrier): the wavefronts' bests,
// then the first wavefront reduces the kWWaves of them
__device__ inline void wg_best0(Cand &c, Red &R) {
    wave_best(c);
    const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
    if (l == 0) {
        R.key[w] = c.key;
        R.id[w] = c.id;
        R.e[w] = c.e;
        R.n[w] = c.n;
    }
    lds_barrier();
    if (w != 0) return;
    const u64 mk = R.key[l % kWWaves];
    const uint32_t mi = R.id[l % kWWaves];
    c.key = mk;
    c.id = mi;
    group_best(c.key, c.id, kWWaves);
    const int q = __ffsll((long long)__ballot(mk == c.key && mi == c.id)) - 1;
    c.e = R.e[q % kWWaves];
    c.n = R.n[q % kWWaves];
}

// The community state of one color step: read as it was after the previous
// step, write the moves into the other buffer.
struct Step {
    const CommInfo *m;
    CommInfo *mq;
};

// The moves a workgroup made in a step, in LDS: applied to the other buffer of
// the community state in its next step (two lists, in turn).
struct Moves {
    int n;
    int32_t v[kWMoves], t[kWMoves], s[kWMoves];
    double kv[kWMoves];
};

__device__ inline void move_comm(i64 t, i64 s, double kv, CommInfo *m) {
    atomicAdd(&m[t].a, kv);
    atomicAdd(&m[s].a, -kv);
    atomicAdd((unsigned long long *)&m[t].n, 1ULL);
    atomicAdd((unsigned long long *)&m[s].n, ~0ULL);  // -1
}

// Move decision of vertex v (one thread): the best candidate, or stay; the
// swap rule of utilityClusteringFunctions.cpp:245-256 (two singletons move
// only towards the smaller id).  Returns the new label, -1 to stay.
__device__ inline int32_t decide(const WideArgs &W, const Step &S, Moves &M, int32_t v, int32_t s, double kv,
                                 i64 ns, const Cand &c, double eix, double &dein, int &moved) {
    int32_t target = s;
    if (c.key) {
        target = (int32_t)c.id;
        if (ns == 1 && c.n == 1 && target > s) target = s;
    }
    if (target == s) return -1;
    move_comm(target, s, kv, S.mq);
    dein += 2.0 * (c.e - eix);
    moved++;
    const int at = atomicAdd(&M.n, 1);
    if (at < kWMoves) {
        M.v[at] = v;
        M.t[at] = target;
        M.s[at] = s;
        M.kv[at] = kv;
        W.C[v] = target;
    } else {
        W.tgt[v] = target;
    }
    return target;
}

// Writes the new label t of vertex v into the entries that hold v's label
// (lanes `first` of `step`).  The entries belong to rows of other classes, so
// no item of this step reads them; with a coloring whose classes hold edges
// (W.defer) the labels are written after the step instead.
__device__ inline void push_label(const WideArgs &W, int32_t v, int32_t t, int first, int step) {
    for (i64 q = W.toff[v] + first, e = W.toff[v + 1]; q < e; q += step) {
        i64 at = W.tpos[q];
        if (W.tpos_hi) at |= (i64)W.tpos_hi[q] << kTposBits;
        W.lab[at] = t;
    }
}

// Empties the first T slots of an LDS table (the caller synchronises).  Every
// table is empty between items.
__device__ inline void clear_table(uint32_t *keys, double *vals, uint32_t T, int first, int step) {
    for (uint32_t i = first; i < T; i += step) {
        keys[i] = kEmptyKey;
        vals[i] = 0.0;
    }
}
// Slots for n entries of a phase with `live` communities: twice the
// communities they can meet, in steps of `step`, at most `most` (a full table
// is 2/3 occupied).
__device__ inline uint32_t table_slots(int n, int live, int step, int most) {
    const int d = 2 * (n < live ? n : live);
    const int t = (d + step - 1) / step * step;
    return (uint32_t)(t < step ? step : t < most ? t : most);
}

// Sums the entries of an item per neighbouring community into the
// workgroup's (empty) table; kWUnroll passes of loads are in flight at a time.
__device__ inline void wg_gather(const WideArgs &W, const WideItem &it, uint32_t *keys, double *vals, uint32_t T) {
    const int32_t *lab = W.lab + it.beg;
    const double *wt = W.w + it.beg;
    const unsigned len = it.len;
    for (unsigned j0 = threadIdx.x; j0 < len; j0 += kWUnroll * kWBlock) {
        uint32_t c[kWUnroll];
        double w[kWUnroll];
#pragma unroll
        for (int u = 0; u < kWUnroll; u++) {
            const unsigned j = j0 + u * kWBlock;
            c[u] = j < len ? (uint32_t)lab[j] : kEmptyKey;
            w[u] = j < len ? wt[j] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kWUnroll; u++)
            if (c[u] != kEmptyKey) lds_insert(keys, vals, T, c[u], w[u]);
    }
    lds_barrier();
}

// Scores slots [first, T) step `step` of an LDS table for vertex v: the
// degree and size of every candidate community are loaded together.
__device__ inline void score_lds(const Step &S, const uint32_t *keys, const double *vals, uint32_t T, int first,
                                 int step, uint32_t s, double kv, double eix, double ax, double cst, Cand &c) {
    for (int i0 = first; i0 < (int)T; i0 += kWUnroll * step) {
        uint32_t yk[kWUnroll];
        double ay[kWUnroll];
        i64 ny[kWUnroll];
#pragma unroll
        for (int u = 0; u < kWUnroll; u++) {
            const int i = i0 + u * step;
            yk[u] = i < (int)T ? keys[i] : kEmptyKey;
        }
#pragma unroll
        for (int u = 0; u < kWUnroll; u++) {
            const bool y = yk[u] != kEmptyKey && yk[u] != s;
            const CommInfo m = y ? S.m[yk[u]] : CommInfo{0.0, 0};
            ay[u] = m.a;
            ny[u] = m.n;
        }
#pragma unroll
        for (int u = 0; u < kWUnroll; u++) {
            if (yk[u] == kEmptyKey || yk[u] == s) continue;
            const double e = vals[i0 + u * step];
            offer(c, gain_of(e, eix, kv, ay[u], ax, cst), yk[u], e, ny[u]);
        }
    }
}

// The vertex of the workgroup's next item, read ahead: its label (it changes
// only in its own step), degree and self-loop weight.
struct VertexAhead {
    int32_t s;
    double kv, sl;
};
__device__ inline void read_ahead(const WideArgs &W, const WideItem &it, VertexAhead &p) {
    p.s = it.len > 0 ? W.C[it.v] : 0;
    p.kv = it.len > 0 ? W.k[it.v] : 0.0;
    p.sl = it.len > 0 ? W.selfw[it.v] : 0.0;
}

// A heavy vertex (the whole workgroup, LDS table).
__device__ void heavy_vertex(const WideArgs &W, const Step &S, Moves &M, const WideItem &it, const VertexAhead &p,
                             uint32_t *keys, double *vals, Red &R, double &dein, int &moved) {
    const uint32_t T = table_slots(it.len, W.live, kWBlock, kWHeavySlots);
    const CommInfo ms = S.m[p.s];
    wg_gather(W, it, keys, vals, T);
    const double eix = lds_lookup(keys, vals, T, (uint32_t)p.s) - p.sl, ax = ms.a - p.kv;
    Cand c;
    score_lds(S, keys, vals, T, threadIdx.x, kWBlock, (uint32_t)p.s, p.kv, eix, ax, W.constant, c);
    wg_best0(c, R);  // its barrier ends the reads of the table
    clear_table(keys, vals, T, threadIdx.x, kWBlock);
    if (threadIdx.x == 0) R.to = decide(W, S, M, it.v, p.s, p.kv, ms.n, c, eix, dein, moved);
    lds_barrier();
    if (R.to >= 0 && !W.defer) push_label(W, it.v, R.to, threadIdx.x, kWBlock);
}

// The pairs of giant G in segments (thread j < nchunks passes the start and
// length of chunk j's), summed in the LDS table and scored; the best in the
// first wavefront.  total: their number; false when they outgrow the table.  pc: 2 *
// kWMaxChunks + 1 ints of LDS.  eix becomes the weight to the giant's own
// community less its self-loop's (sl): *e_s, or (null) that community's sum in
// the table.
__device__ bool score_pairs(const WideArgs &W, const Step &S, const WideGiant &G, int32_t s, double kv, double sl,
                            const double *e_s, double ax, int lo, int before, int total, uint32_t *keys,
                            double *vals, int *pc, Red &R, Cand &c, double &eix) {
    __shared__ int s_fit;
    const int nc = G.nchunks;
    int *pre = pc, *seg = pc + kWMaxChunks + 1;
    lds_barrier();  // pc is free
    if (threadIdx.x < (unsigned)nc) {
        pre[threadIdx.x] = before;
        seg[threadIdx.x] = lo;
    }
    if (threadIdx.x == 0) {
        pre[nc] = total;
        s_fit = 1;
    }
    const uint32_t T = table_slots(total, W.live, kWBlock, kWHeavySlots);
    lds_barrier();
    const uint32_t *pk = W.gpk + G.pairs;
    const double *pv = W.gpv + G.pairs;
    for (int i0 = threadIdx.x; i0 < total; i0 += kWUnroll * kWBlock) {
        uint32_t k[kWUnroll];
        double x[kWUnroll];
#pragma unroll
        for (int u = 0; u < kWUnroll; u++) {
            const int i = i0 + u * kWBlock;
            k[u] = kEmptyKey;
            x[u] = 0.0;
            if (i < total) {
                int a = 0, b = nc;  // the chunk c with pre[c] <= i < pre[c + 1]
                while (b - a > 1) {
                    const int m = (a + b) / 2;
                    if (pre[m] <= i) a = m; else b = m;
                }
                const i64 at = (i64)a * kWChunk + seg[a] + (i - pre[a]);
                k[u] = ld_agent(&pk[at]);
                x[u] = ld_agent(&pv[at]);
            }
        }
#pragma unroll
        for (int u = 0; u < kWUnroll; u++)
            if (k[u] != kEmptyKey && !lds_insert_bounded(keys, vals, T, k[u], x[u])) s_fit = 0;
    }
    lds_barrier();
    const bool fit = s_fit != 0;
    eix = (e_s ? *e_s : lds_lookup(keys, vals, T, (uint32_t)s)) - sl;
    if (fit) score_lds(S, keys, vals, T, threadIdx.x, kWBlock, (uint32_t)s, kv, eix, ax, W.constant, c);
    wg_best0(c, R);
    clear_table(keys, vals, T, threadIdx.x, kWBlock);
    return fit;
}

// Chunk j of a giant: its entries summed per community in LDS, then written
// out as (community, weight) pairs.  With at most kWMergeLive communities
// left, in any order, and the workgroup writing the last chunk sums every
// chunk's pairs, scores them and decides the giant; else grouped by partition
// (bounds in gcnt), its part of the weight to the giant's own community added
// to gsc, and the last chunk marks the pairs ready for the partitions.  pc: 2
// * kWMaxChunks + 1 ints of LDS.
__device__ void giant_chunk(const WideArgs &W, const Step &S, Moves &M, const WideItem &it, const VertexAhead &p,
                            uint32_t *keys, double *vals, int *pc, Red &R, int &moved) {
    const int g = it.g, j = it.j;
    const WideGiant G = W.giants[g];
    const CommInfo ms = S.m[p.s];
    const bool merge = W.live <= kWMergeLive;
    const int P = merge ? 0 : G.nparts;
    const uint32_t T = table_slots(it.len, W.live, kWBlock, kWHeavySlots);
    for (int q = threadIdx.x; q <= P; q += kWBlock) pc[q] = 0;
    wg_gather(W, it, keys, vals, T);
    int32_t *cnt = W.gcnt + G.cnt + (i64)j * (G.nparts + 1);
    uint32_t *pk = W.gpk + G.pairs + (i64)j * kWChunk;
    double *pv = W.gpv + G.pairs + (i64)j * kWChunk;
    double es = 0;
    int total = 0;
    if (!merge) {
        es = lds_lookup(keys, vals, T, (uint32_t)p.s);
        for (uint32_t i = threadIdx.x; i < T; i += kWBlock) {
            const uint32_t k = keys[i];
            if (k != kEmptyKey) atomicAdd(&pc[part_of(k, P)], 1);
        }
        lds_barrier();
        const int ex = wg_exscan(threadIdx.x < (unsigned)P ? pc[threadIdx.x] : 0, R, &total);
        lds_barrier();  // every count was read
        if (threadIdx.x < (unsigned)P) {
            pc[threadIdx.x] = ex;
            st_agent(&cnt[threadIdx.x], ex);
        }
        if (threadIdx.x == 0) st_agent(&cnt[P], total);
        lds_barrier();
    }
    for (uint32_t i = threadIdx.x; i < T; i += kWBlock) {
        const uint32_t k = keys[i];
        if (k == kEmptyKey) continue;
        const int at = atomicAdd(&pc[merge ? 0 : part_of(k, P)], 1);
        st_agent(&pk[at], k);
        st_agent(&pv[at], vals[i]);
        keys[i] = kEmptyKey;
        vals[i] = 0.0;
    }
    // The pairs are stored past the L2 (agent scope) and read back the same way,
    // so no cache is written back or invalidated: every wavefront waits for
    // its stores, then thread 0 counts the chunk.
    stores_done();
    lds_barrier();
    if (threadIdx.x == 0) {
        if (merge) st_agent(&cnt[G.nparts], pc[0]);
        if (es != 0.0) atomicAdd(&W.gsc[g], es);
        stores_done();
        R.last = __hip_atomic_fetch_add(&W.gstate[3 * g], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
                 G.nchunks;
    }
    lds_barrier();
    if (!R.last) return;
    if (!merge) {
        if (threadIdx.x == 0)
            __hip_atomic_store(&W.gstate[3 * g + 1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    const int len =
        threadIdx.x < (unsigned)G.nchunks ? ld_agent(&W.gcnt[G.cnt + (i64)threadIdx.x * (G.nparts + 1) + G.nparts])
                                          : 0;
    const int before = wg_exscan(len, R, &total);
    Cand c;
    double eix = 0;
    // (the table holds every community left, so it does not overflow)
    score_pairs(W, S, G, p.s, p.kv, p.sl, nullptr, ms.a - p.kv, 0, before, total, keys, vals, pc, R, c, eix);
    if (threadIdx.x == 0) {
        double dg = 0;
        R.to = decide(W, S, M, it.v, p.s, p.kv, ms.n, c, eix, dg, moved);
        W.gout[g] = dg;
    }
    lds_barrier();
    if (R.to >= 0 && !W.defer) push_label(W, it.v, R.to, threadIdx.x, kWBlock);
}

// Partition p of giant g: waits for the pairs, sums the partition's pairs of
// every chunk in the LDS table and scores them; the workgroup scoring the last
// partition merges the partitions' candidates in partition order and decides
// the giant's move.  pc: 2 * kWMaxChunks + 1 ints of LDS.  Returns false when the
// wait gave up or the partition outgrew the table (abort raised: bit 1, or
// bit 2 for the table).
__device__ bool giant_part(const WideArgs &W, const Step &S, Moves &M, int g, int p, uint32_t *keys, double *vals, int *pc,
                           Red &R, int &moved) {
    __shared__ int s_ready;
    const WideGiant G = W.giants[g];
    const int32_t v = (int32_t)G.v, s = W.C[v];
    const double kv = W.k[v], sl = W.selfw[v];
    const CommInfo ms = S.m[s];
    const int P = G.nparts, nc = G.nchunks;
    if (threadIdx.x == 0) {
        int ready = 1;
        unsigned spins = 0;
        while (__hip_atomic_load(&W.gstate[3 * g + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
            if (__hip_atomic_load(&W.bar[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) || ++spins > kSpinLimit) {
                atomicOr(&W.bar[0], 1u);
                ready = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        s_ready = ready;
    }
    lds_barrier();
    if (!s_ready) return false;
    const double e_s = ld_agent(&W.gsc[g]), ax = ms.a - kv;
    // this partition's segment of every chunk
    int lo = 0, len = 0;
    if (threadIdx.x < (unsigned)nc) {
        const int32_t *cnt = W.gcnt + G.cnt + (i64)threadIdx.x * (P + 1);
        lo = ld_agent(&cnt[p]);
        len = ld_agent(&cnt[p + 1]) - lo;
    }
    int total = 0;
    const int before = wg_exscan(len, R, &total);
    Cand c;
    double eix = 0;
    if (!score_pairs(W, S, G, s, kv, sl, &e_s, ax, lo, before, total, keys, vals, pc, R, c, eix)) {
        if (threadIdx.x == 0) atomicOr(&W.bar[0], 3u);
        return false;
    }
    if (threadIdx.x == 0) {
        R.to = -1;
        const i64 at = g * W.gparts + p;
        W.gcid[at] = c.key ? (i64)c.id : -1;
        W.gcand[3 * at] = key_gain(c.key);
        W.gcand[3 * at + 1] = c.e;
        W.gcand[3 * at + 2] = (double)c.n;
        __threadfence();
        const int done = atomicAdd(&W.gstate[3 * g + 2], 1) + 1;
        if (done == P) {
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            Cand b;
            for (int q = 0; q < P; q++) {
                const i64 bq = g * W.gparts + q;
                const i64 iq = ld_agent(&W.gcid[bq]);
                if (iq < 0) continue;
                offer(b, ld_agent(&W.gcand[3 * bq]), (uint32_t)iq, ld_agent(&W.gcand[3 * bq + 1]),
                      (i64)ld_agent(&W.gcand[3 * bq + 2]));
            }
            double dg = 0;
            R.to = decide(W, S, M, v, s, kv, ms.n, b, eix, dg, moved);
            W.gout[g] = dg;
        }
    }
    lds_barrier();
    if (R.to >= 0 && !W.defer) push_label(W, v, R.to, threadIdx.x, kWBlock);
    return true;
}

// A color class as a wavefront holds it: its record, a word per lane.
__device__ inline int class_word(const WideArgs &W, int k, int lane) {
    return lane < kWClassWords ? reinterpret_cast<const int *>(W.classes + k)[lane] : 0;
}
__device__ inline int class_at(int word, int i) { return __builtin_amdgcn_readlane(word, i); }
constexpr int kCLo = 0, kCHi = 1, kCExtra = 2, kCExtra0 = 3, kCBinLo = 4, kCBinN = 10, kCGroups = 16;
static_assert(offsetof(WideClass, nextra) == 4 * kCExtra && offsetof(WideClass, extra0) == 4 * kCExtra0 &&
                  offsetof(WideClass, bin_lo) == 4 * kCBinLo && offsetof(WideClass, bin_n) == 4 * kCBinN &&
                  offsetof(WideClass, groups) == 4 * kCGroups,
              "words of a WideClass");

// A wavefront's item with what is read ahead of it: lanes per vertex, and per
// lane the vertex's row and own label and, for a light vertex, its entry.
struct WaveItem {
    int lanes;  // 4 .. 64: light vertices of that many lanes each; 0: a mid vertex; -1: none
    int32_t v, deg, s;
    double kv, sl;
    i64 beg;
    int32_t c;  // the entry's label, read in the item's own step
    double w;
};
// its row: item i of the class
__device__ inline void wave_row(const WideArgs &W, int word, int i, int lane, WaveItem &I) {
    I.lanes = -1;
    I.deg = 0;
    I.v = -1;
    i64 pos = -1;
    const int extra = class_at(word, kCExtra);
    if (i < extra) {
        pos = class_at(word, kCExtra0) + i;
        I.lanes = 0;
    } else {
        i -= extra;
#pragma unroll
        for (int b = 0; b < 6; b++) {
            const int sh = b == 0 ? 0 : b - 1;  // vertices per item: bins 6, 5: 1, bin 4: 2, .. bin 1: 16
            const int nv = class_at(word, kCBinN + b), n = (nv + (1 << sh) - 1) >> sh;
            if (I.lanes < 0 && i < n) {
                I.lanes = b == 0 ? 0 : kWave >> sh;
                const int q = (i << sh) + (b == 0 ? 0 : lane >> (6 - sh));
                if (q < nv) pos = class_at(word, kCBinLo + b) + q;
            }
            i -= n;
        }
    }
    if (pos >= 0) {
        const WideRow r = W.rows[pos];
        I.v = r.v;
        I.deg = r.deg;
        I.kv = r.k;
        I.sl = r.sl;
        I.beg = r.beg;
    }
}
// and its own label and entry's weight
__device__ inline void wave_entry(const WideArgs &W, int lane, WaveItem &I) {
    const int j = lane & (I.lanes - 1);
    I.w = I.lanes > 0 && j < I.deg ? W.w[I.beg + j] : 0.0;
    I.s = I.v >= 0 ? W.C[I.v] : -3;
}
__device__ inline void wave_label(const WideArgs &W, int lane, WaveItem &I) {
    const int j = lane & (I.lanes - 1);
    I.c = I.lanes > 0 && j < I.deg ? W.lab[I.beg + j] : -2;
}

// A mid vertex: one wavefront, its own LDS table.
__device__ inline void mid_vertex(const WideArgs &W, const Step &S, Moves &M, const WaveItem &I, uint32_t *keys,
                                  double *vals, int lane, const CommInfo &ms, double &dein, int &moved) {
    const uint32_t T = table_slots(I.deg, W.live, kWave, kWMidSlots);
    const int64_t beg = (int64_t)(((u64)(uint32_t)__builtin_amdgcn_readfirstlane((int)(I.beg >> 32)) << 32) |
                                  (uint32_t)__builtin_amdgcn_readfirstlane((int)I.beg));
    const int32_t *lab = W.lab + beg;
    const double *wt = W.w + beg;
    const unsigned deg = __builtin_amdgcn_readfirstlane(I.deg);
    for (unsigned j0 = lane; j0 < deg; j0 += kWUnroll * kWave) {
        uint32_t c[kWUnroll];
        double w[kWUnroll];
#pragma unroll
        for (int u = 0; u < kWUnroll; u++) {
            const unsigned j = j0 + u * kWave;
            c[u] = j < deg ? (uint32_t)lab[j] : kEmptyKey;
            w[u] = j < deg ? wt[j] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kWUnroll; u++)
            if (c[u] != kEmptyKey) lds_insert(keys, vals, T, c[u], w[u]);
    }
    wave_lds_sync();
    const double eix = lds_lookup(keys, vals, T, (uint32_t)I.s) - I.sl, ax = ms.a - I.kv;
    Cand c;
    score_lds(S, keys, vals, T, lane, kWave, (uint32_t)I.s, I.kv, eix, ax, W.constant, c);
    wave_best(c);
    wave_lds_sync();  // every lane is done with the table
    clear_table(keys, vals, T, lane, kWave);
    int32_t to = -1;
    if (lane == 0) to = decide(W, S, M, I.v, I.s, I.kv, ms.n, c, eix, dein, moved);
    wave_lds_sync();
    to = __builtin_amdgcn_readfirstlane(to);
    if (to >= 0 && !W.defer) push_label(W, I.v, to, lane, kWave);
}

// 64 / G light vertices, G lanes each and one entry per lane (I.c: its
// neighbour's label, -2 past the vertex's entries): every lane walks its
// group's entries in adjacency order, so the weight to a community is the
// left-to-right sum buildLocalMapCounter forms.  The entries are staged in
// the wavefront's (empty) table.
__device__ inline void light_vertices(const WideArgs &W, const Step &S, Moves &M, const WaveItem &I,
                                      uint32_t *keys, double *vals, int lane, const CommInfo &ms, double &dein, int &moved) {
    const int32_t c = I.c;
    const int G = I.lanes, gl = lane & (G - 1), gb = lane & ~(G - 1);
    const bool mine = gl < I.deg;
    keys[lane] = (uint32_t)c;
    vals[lane] = I.w;
    wave_lds_sync();
    const int4 *s_c = reinterpret_cast<const int4 *>(keys + gb);
    const double2 *s_w = reinterpret_cast<const double2 *>(vals + gb);
    double e_mine = 0;
    bool first = true;
    for (int m = 0; __ballot(m < I.deg); m += 4) {
        const int4 cm = s_c[m >> 2];
        const double2 wa = s_w[m >> 1], wb = s_w[(m >> 1) + 1];
        const bool e0 = cm.x == c, e1 = cm.y == c, e2 = cm.z == c, e3 = cm.w == c;
        e_mine += e0 ? wa.x : 0.0;
        e_mine += e1 ? wa.y : 0.0;
        e_mine += e2 ? wb.x : 0.0;
        e_mine += e3 ? wb.y : 0.0;
        if ((e0 && m < gl) || (e1 && m + 1 < gl) || (e2 && m + 2 < gl) || (e3 && m + 3 < gl)) first = false;
    }
    // the weight to the vertex's own community, from a lane that holds it
    const u64 own = (__ballot(mine && c == I.s) >> gb) & (G == kWave ? ~0ULL : (1ULL << G) - 1);
    const double at_s = __shfl(e_mine, own ? gb + __ffsll((long long)own) - 1 : lane);
    const double eix = (own ? at_s : 0.0) - I.sl;
    Cand b;
    if (mine && first && c != I.s) {
        const CommInfo mc = S.m[c];
        // max() starts from maxGain = 0 and needs a strict increase
        offer(b, gain_of(e_mine, eix, I.kv, mc.a, ms.a - I.kv, W.constant), (uint32_t)c, e_mine, mc.n);
    }
    u64 key = b.key;
    uint32_t id = b.id;
    group_best(key, id, G);
    const u64 win = (__ballot(b.key == key && b.id == id) >> gb) & (G == kWave ? ~0ULL : (1ULL << G) - 1);
    const int src = gb + __ffsll((long long)win) - 1;
    b.e = __shfl(b.e, src);
    b.n = __shfl(b.n, src);
    b.key = key;
    b.id = id;
    wave_lds_sync();  // every lane is done with the staged entries
    keys[lane] = kEmptyKey;
    vals[lane] = 0.0;
    int32_t to = -1;
    if (I.v >= 0 && gl == 0) to = decide(W, S, M, I.v, I.s, I.kv, ms.n, b, eix, dein, moved);
    wave_lds_sync();
    to = __shfl(to, gb);
    if (to >= 0 && !W.defer) push_label(W, I.v, to, gl, G);
}

__global__ __launch_bounds__(kWBlock) void k_wide_iteration(WideArgs W) {
    __shared__ __align__(16) uint32_t hkeys[kWHeavySlots];
    __shared__ __align__(16) double hvals[kWHeavySlots];
    __shared__ Red R;
    __shared__ int pc[2 * kWMaxChunks + 2];  // giant items: partition counts or chunk segments
    __shared__ Moves moves[2];
    const unsigned nb = gridDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    uint32_t *wkeys = hkeys + wave * kWMidSlots;
    double *wvals = hvals + wave * kWMidSlots;
    const i64 nv = W.nv;
    const i64 gtid = (i64)blockIdx.x * kWBlock + threadIdx.x, gstride = (i64)nb * kWBlock;
    // both buffers of the community state start equal
    for (i64 i = gtid; i < nv; i += gstride) {
        const CommInfo m{W.a[i], W.n[i]};
        W.m0[i] = m;
        W.m1[i] = m;
        W.tgt[i] = -1;
    }
    for (i64 i = gtid; i < W.ncls; i += gstride) W.over[i] = 0;
    if (threadIdx.x == 0) moves[0].n = moves[1].n = 0;
    for (i64 g = gtid; g < W.ngiants; g += gstride) {
        W.gstate[3 * g] = W.gstate[3 * g + 1] = W.gstate[3 * g + 2] = 0;
        W.gsc[g] = 0.0;
        W.gout[g] = 0.0;
    }
    clear_table(hkeys, hvals, kWHeavySlots, threadIdx.x, kWBlock);
    unsigned seq = 1;
    grid_arrive(W.bar, seq);
    // the workgroup's streams of items; the first class's record; the
    // workgroup's and the wavefront's first item read ahead
    i64 wi = W.wbeg[blockIdx.x], pi = W.pbeg[blockIdx.x];
    const i64 *wend = W.wend + (i64)blockIdx.x * W.ncls, *pend = W.pend + (i64)blockIdx.x * W.ncls;
    WideItem item = W.witems[wi];  // (a stream ends with an empty item)
    VertexAhead ahead;
    WaveItem I;
    // class k + 1's record, stream bounds and rank are read a step before
    // they are used
    int word = 0, at = 0, nword = 0, nrank = -1;
    i64 whi = wi, phi = pi, nwhi = wi, nphi = pi;
    auto read_class = [&](int k) {
        if (k >= W.ncls) return;
        nword = class_word(W, k, lane);
        nwhi = wend[k];
        nphi = pend[k];
        nrank = W.rank[(i64)k * nb + blockIdx.x];
    };
    auto look_ahead = [&](int k) {
        read_ahead(W, item, ahead);
        word = nword;
        whi = nwhi;
        phi = nphi;
        at = nrank >= 0 ? wave * class_at(word, kCGroups) + nrank : 0x3FFFFFFF;
        wave_row(W, word, at, lane, I);
        read_class(k + 1);
        wave_entry(W, lane, I);
    };
    read_class(0);
    if (W.ncls > 0) look_ahead(0);
    bool alive = grid_wait(W.bar, nb, seq);
    double dein = 0;  // this thread's movers' 2 (e_t - e_s)
    int moved = 0;
    int par = 0;
    int mlo = 0, mhi = 0;  // the previous step's class in cperm
    for (int k = 0; k < W.ncls && alive; k++) {
        Step S;
        S.m = par ? W.m1 : W.m0;
        S.mq = par ? W.m0 : W.m1;
        Moves &M = moves[k & 1], &L = moves[(k & 1) ^ 1];
        // the previous step's moves, into the buffer this step writes
        const int over = mhi > mlo ? W.over[k - 1] : 0;
        for (int q = threadIdx.x, n = min(L.n, kWMoves); q < n; q += kWBlock)
            move_comm(L.t[q], L.s[q], L.kv[q], S.mq);
        // workgroup items
        for (; wi < whi; wi++) {
            const WideItem next = W.witems[wi + 1];
            const VertexAhead p = ahead;
            read_ahead(W, next, ahead);
            if (item.g < 0) heavy_vertex(W, S, M, item, p, hkeys, hvals, R, dein, moved);
            else giant_chunk(W, S, M, item, p, hkeys, hvals, pc, R, moved);
            item = next;
        }
        // wavefront items
        wave_label(W, lane, I);
        while (I.lanes >= 0) {
            const CommInfo ms = I.s >= 0 ? S.m[I.s] : CommInfo{0.0, 0};
            WaveItem N;
            at += class_at(word, kCGroups) * kWWaves;
            wave_row(W, word, at, lane, N);
            wave_entry(W, lane, N);
            wave_label(W, lane, N);
            if (I.lanes == 0) mid_vertex(W, S, M, I, wkeys, wvals, lane, ms, dein, moved);
            else light_vertices(W, S, M, I, wkeys, wvals, lane, ms, dein, moved);
            I = N;
        }
        if (over)  // moves of the previous step beyond the workgroups' lists
            for (i64 q = mlo + gtid; q < mhi; q += gstride) {
                const i64 v = W.cperm[q];
                const int32_t t = W.tgt[v];
                if (t < 0) continue;
                move_comm(t, W.C[v], W.k[v], S.mq);
                W.C[v] = t;
                W.tgt[v] = -1;
            }
        // partitions of giants
        if (W.live > kWMergeLive) {
            if (pi < phi) lds_barrier();  // the wavefronts' tables are empty
            for (; pi < phi; pi++) {
                const int2 gp = W.pitems[pi];
                if (!giant_part(W, S, M, gp.x, gp.y, hkeys, hvals, pc, R, moved)) {
                    alive = false;
                    break;
                }
            }
            if (!alive) break;
        }
        mlo = class_at(word, kCLo);
        mhi = class_at(word, kCHi);
        lds_barrier();
        if (threadIdx.x == 0) {
            L.n = 0;
            if (M.n > kWMoves) atomicOr(&W.over[k], 1);
        }
        if (W.defer) {  // every item of the step has read its labels: write the new ones
            alive = grid_barrier(W.bar, nb, ++seq);
            if (!alive) break;
            for (int q = wave; q < min(M.n, kWMoves); q += kWWaves) push_label(W, M.v[q], M.t[q], lane, kWave);
            if (__hip_atomic_load(&W.over[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                for (i64 q = mlo + (i64)blockIdx.x * kWWaves + wave; q < mhi; q += (i64)nb * kWWaves) {
                    const int32_t v = (int32_t)W.cperm[q], t = W.tgt[v];
                    if (t >= 0) push_label(W, v, t, lane, kWave);
                }
        }
        grid_arrive(W.bar, ++seq);
        if (k + 1 < W.ncls) look_ahead(k + 1);
        alive = grid_wait(W.bar, nb, seq);
        par ^= 1;
    }
    const CommInfo *mf = par ? W.m1 : W.m0;
    // modularity partials: the movers' change of the internal weight (giants
    // in giant order) and the sum of a^2
    double exx = 0, a2 = 0;
    int live = 0;
    if (alive) {
        exx = dein;
        if (blockIdx.x == 0 && threadIdx.x == 0)
            for (i64 g = 0; g < W.ngiants; g++) exx += W.gout[g];
        for (i64 i = gtid; i < nv; i += gstride) {
            const CommInfo m = mf[i];
            a2 += m.a * m.a;
            live += m.n > 0;
            W.a[i] = m.a;
            W.n[i] = m.n;
        }
    }
    exx = wg_sum(exx, R);
    a2 = wg_sum(a2, R);
    // moves of the iteration, communities left (one atomic each per workgroup)
    __shared__ unsigned long long s_moved;
    __shared__ unsigned s_live;
    if (threadIdx.x == 0) {
        s_moved = 0;
        s_live = 0;
    }
    __syncthreads();
    if (moved) atomicAdd(&s_moved, (unsigned long long)moved);
    if (live) atomicAdd(&s_live, (unsigned)live);
    __syncthreads();
    if (threadIdx.x == 0) {
        W.part[blockIdx.x] = exx;
        W.part[nb + blockIdx.x] = a2;
        if (s_moved) atomicAdd((unsigned long long *)W.moves, s_moved);
        if (s_live) atomicAdd(&W.bar[1], s_live);
    }
    if (alive && mhi > mlo && W.over[W.ncls - 1])  // the last class's moves beyond the lists
        for (i64 q = mlo + gtid; q < mhi; q += gstride) {
            const i64 v = W.cperm[q];
            if (W.tgt[v] >= 0) W.C[v] = W.tgt[v];
        }
}

__global__ void k_wide_rows(const i64 *perm, const i64 *off, const double *k, const double *selfw, i64 lo, i64 hi,
                            WideRow *rows) {
    for (i64 q = lo + blockIdx.x * (i64)blockDim.x + threadIdx.x; q < hi; q += (i64)gridDim.x * blockDim.x) {
        const i64 v = perm[q], b = off[v];
        rows[q] = WideRow{b, k[v], selfw[v], (int32_t)v, wide_row_deg(off[v + 1] - b)};
    }
}

}  // namespace

#define GLV_LAUNCH_CHECK() GLV_HIP(hipGetLastError())

__global__ void k_narrow_ids(const i64 *src, i64 n, int32_t *dst) {
    for (i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x)
        dst[i] = (int32_t)src[i];
}
__global__ void k_widen_ids(const int32_t *src, i64 n, i64 *dst) {
    for (i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x)
        dst[i] = (i64)src[i];
}
void launch_narrow_ids(const i64 *src, i64 n, int32_t *dst, hipStream_t s) {
    if (n <= 0) return;
    k_narrow_ids<<<grid_for(n, kBlock, 16384), kBlock, 0, s>>>(src, n, dst);
    GLV_LAUNCH_CHECK();
}
void launch_widen_ids(const int32_t *src, i64 n, i64 *dst, hipStream_t s) {
    if (n <= 0) return;
    k_widen_ids<<<grid_for(n, kBlock, 16384), kBlock, 0, s>>>(src, n, dst);
    GLV_LAUNCH_CHECK();
}

bool wide_enabled() {
    static const bool on = [] {
        const char *e = std::getenv("GLV_WIDE");
        return !(e && std::strcmp(e, "0") == 0);
    }();
    return on;
}

int wide_blocks() {
    static int cached = -1;
    if (cached < 0) {
        int dev = 0, cus = 0, per = 0;
        GLV_HIP(hipGetDevice(&dev));
        GLV_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        GLV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_wide_iteration, kWBlock, 0));
        cached = per > 0 ? cus * std::min(per, 1) : 0;
    }
    return cached;
}

int wide_grid(i64 entries) {
    const int most = wide_blocks();
    int nb = kWMinGrid;
    while (nb < most && (i64)nb * kWBlock < entries) nb *= 2;
    return std::min(nb, most);
}

bool launch_wide_iteration(const WideArgs &W, int nblocks, hipStream_t s) {
    if (nblocks <= 0 || nblocks > wide_blocks()) return false;
    WideArgs w = W;
    void *args[] = {&w};
    hipError_t e = hipLaunchKernel((const void *)k_wide_iteration, dim3(nblocks), dim3(kWBlock), args, 0, s);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        trace("wide colored iteration (%d workgroups) refused: %s", nblocks, hipGetErrorString(e));
        return false;
    }
    return true;
}

void launch_wide_rows(const i64 *perm, const i64 *off, const double *k, const double *selfw, i64 lo, i64 hi,
                      WideRow *rows, hipStream_t s) {
    if (hi <= lo) return;
    k_wide_rows<<<grid_for(hi - lo, kBlock, 8192), kBlock, 0, s>>>(perm, off, k, selfw, lo, hi, rows);
    GLV_LAUNCH_CHECK();
}

}  // namespace glv
