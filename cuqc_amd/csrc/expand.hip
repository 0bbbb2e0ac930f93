// expand.hip -- gfx950 expansion of quasi-clique task records.
//
// One 64-lane wavefront owns one task record at a time and runs the whole
// per-task step of the reference host path (h_expand_level body,
// main.cu:1060-1181): lookahead, the sequential branch loop with
// remove-one-vertex, add-one-vertex with diameter and degree pruning,
// critical-vertex pruning, the clique test and the Q-ordered child write.
//
// Four forms of the same steps, by the task's size: up to 64 vertices in
// registers, with the whole subtree below (tiny_*); up to what the wave's LDS
// holds (WideLds); larger ones from the wave's HBM slab, in 16- and 32-bit
// arrays up to 4,095 vertices (WideMid), else in 32- and 64-bit ones (WideSlab).
//
// Adjacency.  Every task is a subset of the root task, so vertex ids are
// root-local (0..R-1) and the 1-hop / 2-hop relations are kept as R x R bit
// matrices in HBM (A1, A2).  Where the reference scans adjacency lists through
// its id->position map (vertex_order_map), this code tests bits: the two are
// the same relation.
//
// Semantics follow the host column of the reference (main.cu:1349-2198),
// including the two degree-update branches of a degree-pruning round
// (recompute from the remaining set when it is smaller than the removed set,
// else decrement via the removed set, main.cu:1775-1807) and the round
// structure that follows critical-vertex pruning when no candidate is
// critical-adjacent: the reference then leaves its id->position map empty
// (main.cu:1575-1602), so a recompute round sets every exdeg to 0 and a
// decrement round changes nothing.  Both effects are reproduced.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "qc_device.h"

namespace qcdev {

constexpr int WAVE = 64;

__device__ __forceinline__ int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ int lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Lane broadcasts by v_readlane (lane index uniform): no LDS round trip.
__device__ __forceinline__ int rdlane(int x, int l) { return __builtin_amdgcn_readlane(x, l); }
__device__ __forceinline__ unsigned long long rdlane64(unsigned long long x, int l) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), l);
    return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ float rdlanef(float x, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// Whole-wave reductions with DPP moves (called with all 64 lanes active).
// Quad permutes and the half-row and row mirrors combine every row of 16
// lanes; row broadcast 15 then adds row 0 into row 1 and row 2 into row 3,
// row broadcast 31 adds rows 0-1 into rows 2-3; lane 63 holds the result.
// Lanes a move does not write keep `id`, the operation's identity.
template <int CTRL, int RM>
__device__ __forceinline__ int dpp32(int id, int v) {
    return __builtin_amdgcn_update_dpp(id, v, CTRL, RM, 0xf, false);
}
template <int CTRL, int RM>
__device__ __forceinline__ unsigned long long dpp64(unsigned long long id, unsigned long long v) {
    const uint32_t lo = (uint32_t)dpp32<CTRL, RM>((int)(uint32_t)id, (int)(uint32_t)v);
    const uint32_t hi = (uint32_t)dpp32<CTRL, RM>((int)(uint32_t)(id >> 32), (int)(uint32_t)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}
template <class Op>
__device__ __forceinline__ int wave_reduce32(int v, int id, Op op) {
    v = op(v, dpp32<0xb1, 0xf>(id, v));   // quad_perm [1,0,3,2]
    v = op(v, dpp32<0x4e, 0xf>(id, v));   // quad_perm [2,3,0,1]
    v = op(v, dpp32<0x141, 0xf>(id, v));  // row_half_mirror
    v = op(v, dpp32<0x140, 0xf>(id, v));  // row_mirror
    v = op(v, dpp32<0x142, 0xa>(id, v));  // row_bcast:15 into rows 1, 3
    v = op(v, dpp32<0x143, 0xc>(id, v));  // row_bcast:31 into rows 2, 3
    return rdlane(v, WAVE - 1);
}
template <class Op>
__device__ __forceinline__ unsigned long long wave_reduce64(unsigned long long v, unsigned long long id, Op op) {
    v = op(v, dpp64<0xb1, 0xf>(id, v));
    v = op(v, dpp64<0x4e, 0xf>(id, v));
    v = op(v, dpp64<0x141, 0xf>(id, v));
    v = op(v, dpp64<0x140, 0xf>(id, v));
    v = op(v, dpp64<0x142, 0xa>(id, v));
    v = op(v, dpp64<0x143, 0xc>(id, v));
    return rdlane64(v, WAVE - 1);
}
__device__ __forceinline__ int wave_sum(int v) {
    return wave_reduce32(v, 0, [](int x, int y) { return x + y; });
}
__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
    return v;
}
__device__ __forceinline__ long long wave_sum64(long long v) {
    return (long long)wave_reduce64((unsigned long long)v, 0ull,
                                    [](unsigned long long x, unsigned long long y) { return x + y; });
}
__device__ __forceinline__ int wave_min(int v) {
    return wave_reduce32(v, INT32_MAX, [](int x, int y) { return min(x, y); });
}
__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) {
    return wave_reduce64(v, ~0ull, [](unsigned long long x, unsigned long long y) { return x < y ? x : y; });
}
__device__ __forceinline__ int wave_max(int v) {
    return wave_reduce32(v, INT32_MIN, [](int x, int y) { return max(x, y); });
}
__device__ __forceinline__ void wsync() { __syncthreads(); }

// ---------------------------------------------------------------------------
// per-task state
// ---------------------------------------------------------------------------
struct LStats {
    unsigned long long tasks, branches, children, raw, sum_t, sum_tw, sum_clq, large, beyond;
};

// The scalar fields of a DevGraph the kernels read, held in scalar
// registers for the task being expanded: read through the table pointer they
// would be reloaded from memory after every store the compiler cannot
// disambiguate.  The table pointers stay behind `p` (holding all of them in
// scalar registers spills other scalars into vector lanes).
struct GConst {
    const DevGraph* p;
    double gamma;
    int32_t min_size, max_depth;
};

__device__ __forceinline__ int32_t uni32(int32_t x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ long long uni64(long long x) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((unsigned long long)x >> 32));
    return (long long)(((unsigned long long)hi << 32) | lo);
}

__device__ __forceinline__ GConst load_graph(const DevGraph* p) {
    GConst g;
    g.p = p;
    g.gamma = __longlong_as_double(uni64(__double_as_longlong(p->gamma)));
    g.min_size = uni32(p->min_size);
    g.max_depth = uni32(p->max_depth);
    return g;
}

struct Ctx {
    const ExpandArgs* a;
    GConst g;             // tables of the instance being expanded
    int lane;
    LStats* st;           // counters of this wave (LDS; lane 0 updates them)
    uint32_t depth;
    uint32_t inst;        // instance of the task being expanded
    long long slot;       // queue slot of the task being expanded (trace)
    unsigned long long* ph;           // phase cycles (LDS, diagnostics)
    long long ph_t;                   // start of the running phase
    long long wadj_l;                 // this lane's share of W_adj (summed at flush)
    bool phase_on;                    // phase counters requested
    bool keys;                        // the task's children are written (inside the depth
                                      // window): only then is the child's lvl2adj kept
    // persistent mode: this wave's private stack (entries [pbot, ptop) of a
    // ring of priv_cap refs; uniform counters, lane 0 touches the entries)
    int shard;                        // this wave's ring shard (blockIdx % q_shards)
    TaskRef* ptopref;                 // LDS: a copy of stack entry ptopi (the last pushed), ~0u: none
    uint32_t ptopi;
    unsigned long long* clq;          // LDS, lane 0: the wave's refs and slots of the clique stream (clq_reserve)
    uint32_t* fl;                     // LDS: free block indices of the small classes, FL_LOCAL_MAX per class
    uint32_t* fln;                    // LDS: their counts
    TaskRef* pstack;
    unsigned char* pbkt;
    uint32_t pbot, ptop;
    // children given straight to the rings while waves wait (share_child)
    unsigned long long share_v;       // lane 0: the pending word as read at the last check
    int share_n;                      // children since the last check
    int share_left;                   // children still to give before the next check
    bool share_ok;                    // the running task has SHARE_MIN_T vertices or more
};

// phase accounting: charge the cycles since the last mark to phase k
__device__ __forceinline__ void ph_mark(Ctx& c, int k) {
    if (c.phase_on) {
        long long n = clock64();
        if (c.lane == 0) c.ph[k] += (unsigned long long)(n - c.ph_t);
        c.ph_t = n;
    }
}
__device__ __forceinline__ void ph_start(Ctx& c) {
    if (c.lane == 0)
        for (int k = 0; k < PH_COUNT; k++) c.ph[k] = 0;
    c.ph_t = clock64();
}
__device__ __forceinline__ void ph_flush(Ctx& c) {
    if (c.a->phase && c.lane == 0)
        for (int k = 0; k < PH_COUNT; k++)
            if (c.ph[k]) atomicAdd(&c.a->phase[k], c.ph[k]);
}

// mindeg[i] of the host table (graph_io.cpp build_tables), computed in
// registers: a per-lane table lookup is a dependent memory round trip
__device__ __forceinline__ int md(const Ctx& c, int i) {
    return i < 1 ? 0 : (int)ceil(c.g.gamma * (double)(i - 1));
}
// floor(d / gamma), the same IEEE division as on the host, in place of a table:
// a dependent load on the way to every bound
__device__ __forceinline__ int ub_quot(const Ctx& c, int d) { return (int)floor((double)d / c.g.gamma); }
__device__ __forceinline__ int get_mindeg(const Ctx& c, int s) {
    int ms = c.g.min_size;
    return s < ms ? md(c, ms) : md(c, s);
}

// W_adj bookkeeping: adjacency entries the reference's list scans visit
// (restricted to root vertices), summed over ids.  Each lane keeps its own
// partial sum; the wave sums them when the counters are flushed.
__device__ __forceinline__ void wadj_add(Ctx& c, long long x) {  // x uniform
    if (c.lane == 0) c.wadj_l += x;
}
__device__ __forceinline__ void wadj_lanes(Ctx& c, long long x) {  // x per lane
    c.wadj_l += x;
}

__device__ inline void set_mask_bit(uint64_t* mk, int b) {
    atomicOr((unsigned long long*)&mk[b >> 6], 1ull << (b & 63));
}

// ---------------------------------------------------------------------------
// emission
// ---------------------------------------------------------------------------
// A place for one raw set of `len` vertices in the clique stream: the ref's
// index and the first vertex slot.  The persistent form takes CLQ_REFS refs
// and CLQ_SLOTS slots at a time for the wave (lane 0 keeps what is left in
// c.clq: next ref, end, next slot, end), since two device-scope atomics on one
// pair of counters for each of a million raw sets cost as much as the search;
// refs it does not use are marked empty when the wave ends (clq_close).  Sets of
// more than CLQ_SLOTS / 4 vertices take their slots directly, so less than a
// quarter of a wave's slots are lost at the ends.
__device__ __attribute__((always_inline)) bool clq_reserve(Ctx& c, int len, unsigned long long& ri, unsigned long long& si) {
    const ExpandArgs& a = *c.a;
    if (c.lane == 0) {
        if (a.queue_mode) {
            ri = c.clq[0];
            if (ri == c.clq[1]) {
                ri = atomicAdd(&a.clq_ctr->items, (unsigned long long)CLQ_REFS);
                c.clq[1] = ri + CLQ_REFS;
            }
            c.clq[0] = ri + 1;
            if (len > CLQ_SLOTS / 4) {
                si = atomicAdd(&a.clq_ctr->slots, (unsigned long long)len);
            } else {
                si = c.clq[2];
                if (si + len > c.clq[3]) {
                    si = atomicAdd(&a.clq_ctr->slots, (unsigned long long)CLQ_SLOTS);
                    c.clq[3] = si + CLQ_SLOTS;
                }
                c.clq[2] = si + len;
            }
        } else {
            ri = atomicAdd(&a.clq_ctr->items, 1ull);
            si = atomicAdd(&a.clq_ctr->slots, (unsigned long long)len);
        }
    }
    ri = rdlane64(ri, 0);
    si = rdlane64(si, 0);
    if (ri >= a.clq_ref_cap || si + len > a.clq_vert_cap) {
        if (c.lane == 0) atomicOr(a.error, 1);
        return false;
    }
    return true;
}
__device__ __forceinline__ void clq_ref(Ctx& c, unsigned long long ri, unsigned long long si, int len) {
    if (c.lane == 0) {
        CliqueRef r;
        r.off = si;
        r.len = (uint32_t)len;
        r.inst = c.inst;
        c.a->clq_refs[ri] = r;
        c.st->raw++;
        c.st->sum_clq += len;
    }
}
// the vertices of the lanes in m
__device__ __forceinline__ void emit_lanes(Ctx& c, uint64_t m, uint32_t orig) {
    const int len = __popcll(m);
    unsigned long long ri = 0, si = 0;
    if (!clq_reserve(c, len, ri, si)) return;
    if ((m >> c.lane) & 1ull) c.a->clq_verts[si + lanes_below(m)] = orig;
    clq_ref(c, ri, si, len);
}
// the wave's unused refs, marked empty
__device__ __forceinline__ void clq_close(Ctx& c) {
    const ExpandArgs& a = *c.a;
    wsync();
    const unsigned long long end = min<unsigned long long>(c.clq[1], a.clq_ref_cap);
    for (unsigned long long i = c.clq[0] + c.lane; i < end; i += WAVE) a.clq_refs[i] = CliqueRef{0, 0, CLQ_NONE};
}

// Cost-model features of a record from per-lane partial values (lane 0 holds
// the row): members, candidates, min/max/mean indeg, min/max/mean exdeg, depth,
// ub - lb, mean |N2 n root| over candidates, size.  Means are
// float(sum) / float(count), as in the oracle.
__device__ __forceinline__ void feature_row(int tc, int mem, int depth, int gap, int mi, int ma, int me, int mx,
                                            long long si, long long se, long long s2, float* f) {
    mi = wave_min(mi);
    ma = wave_max(ma);
    me = wave_min(me);
    mx = wave_max(mx);
    si = wave_sum64(si);
    se = wave_sum64(se);
    s2 = wave_sum64(s2);
    if (lane_id() == 0) {
        const int cnd = tc - mem;
        f[0] = (float)mem;
        f[1] = (float)cnd;
        f[2] = (float)mi;
        f[3] = (float)ma;
        f[4] = (float)si / (float)tc;
        f[5] = (float)me;
        f[6] = (float)mx;
        f[7] = (float)se / (float)tc;
        f[8] = (float)depth;
        f[9] = (float)gap;
        f[10] = cnd > 0 ? (float)s2 / (float)cnd : 0.0f;
        f[11] = (float)tc;
    }
}

__device__ __forceinline__ float bf16f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// Bucket of a child from the cost model (12 -> 64 -> 64 -> 1 ReLU MLP,
// bf16 weights, fp32 accumulation): lane j evaluates hidden unit j of both
// layers; the prediction is compared with the bucket thresholds.
__device__ int cost_bucket(Ctx& c, const float* feat /* valid in lane 0 */) {
    const ExpandArgs& a = *c.a;
    const uint16_t* W = a.cm_w;
    const float* nrm = a.cm_norm;
    const int j = c.lane;
    float h1 = bf16f(W[12 * 64 + j]);
    for (int k = 0; k < 12; k++) {
        float f = rdlanef(feat[k], 0);
        float z = (log1pf(fmaxf(f, 0.0f)) - nrm[k]) / nrm[12 + k];
        h1 = fmaf(z, bf16f(W[k * 64 + j]), h1);
    }
    h1 = fmaxf(h1, 0.0f);
    const int ow2 = 12 * 64 + 64;
    float h2 = bf16f(W[ow2 + 64 * 64 + j]);
    for (int i = 0; i < 64; i++) h2 = fmaf(rdlanef(h1, i), bf16f(W[ow2 + i * 64 + j]), h2);
    h2 = fmaxf(h2, 0.0f);
    const int ow3 = ow2 + 64 * 64 + 64;
    float y = wave_sum_f(h2 * bf16f(W[ow3 + j])) + bf16f(W[ow3 + 64]);
    int b = 0;
    for (int q = 0; q < a.n_buckets - 1 && q < 3; q++)
        if (y > nrm[26 + q]) b = q + 1;
    return uni(b);
}

// ---------------------------------------------------------------------------
// persistent mode: vertex pool, shared rings, private stacks
// ---------------------------------------------------------------------------
constexpr unsigned long long FL_IDX = (1ull << 36) - 1;  // block index field (units); all ones = empty list

// Free blocks.  Every size class has FL_SHARDS shared lock-free stacks of
// magazines, and a wave uses shard blockIdx % FL_SHARDS (workgroups go to
// the XCDs in turn, so a shard's users share an XCD and its L2).  A
// magazine is a free head block that lists up to FL_LOCAL_MAX - 1 more
// blocks: one exchange on a shard moves up to fl_mag blocks.  The small
// classes (up to 8 units) also keep up to 2 fl_mag block indices per wave
// in LDS (lane 0 only): the free of a task's record and its children's
// allocations meet there without touching memory.
// Head block words: [0] next magazine (index), [1] block count, then the
// other blocks' indices as 32-bit words.
__device__ __forceinline__ unsigned long long* fl_shard(const ExpandArgs& a, int cl, int sh) {
    return a.fl_head + ((size_t)cl * FL_SHARDS + sh) * QSTRIDE;
}

// Pops a magazine (lane 0): its head block index, or FL_IDX when the shard
// holds none.  The next link is read from the head block before the
// exchange; if another wave takes that block meanwhile, the tag in the
// shard head changes and the exchange fails.
__device__ __attribute__((always_inline)) unsigned long long mag_pop(const ExpandArgs& a, unsigned long long* hp) {
    unsigned long long h = __hip_atomic_load(hp, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
    while ((h & FL_IDX) != FL_IDX) {
        const unsigned long long idx = h & FL_IDX;
        const unsigned long long nxt =
            __hip_atomic_load((unsigned long long*)(a.pool + idx * POOL_UNIT), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long nh = (((h >> 36) + 1ull) << 36) | (nxt & FL_IDX);
        if (__hip_atomic_compare_exchange_strong(hp, &h, nh, __ATOMIC_ACQUIRE, __ATOMIC_ACQUIRE,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return idx;
    }
    return FL_IDX;
}

// Pushes the magazine headed by block idx (lane 0; its count and member
// words are written: the release orders them, and the wave's reads of the
// blocks' old records, before any reuse).
__device__ __attribute__((always_inline)) void mag_push(const ExpandArgs& a, unsigned long long* hp, unsigned long long idx) {
    unsigned long long h = __hip_atomic_load(hp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        __hip_atomic_store((unsigned long long*)(a.pool + idx * POOL_UNIT), h & FL_IDX, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long nh = (((h >> 36) + 1ull) << 36) | idx;
        if (__hip_atomic_compare_exchange_strong(hp, &h, nh, __ATOMIC_RELEASE, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
    }
}

// The shared part of pool_alloc (out of line: it is the rare path, and
// inlined twice it costs the kernel registers).
__device__ __attribute__((noinline)) unsigned long long pool_alloc_shared(const ExpandArgs& a, uint32_t* fl, uint32_t* fln,
                                                                          int cl, uint32_t units) {
    const int sh = (int)(blockIdx.x % FL_SHARDS);
    unsigned long long m = mag_pop(a, fl_shard(a, cl, sh));
    if (m == FL_IDX) {
        const unsigned long long n = (unsigned long long)units * POOL_UNIT;
        const unsigned long long off = atomicAdd(a.pool_top, n);
        if (off + n <= a.pool_cap) return off;
        for (int k = 1; k < FL_SHARDS && m == FL_IDX; k++) m = mag_pop(a, fl_shard(a, cl, (sh + k) % FL_SHARDS));
        if (m == FL_IDX) return ~0ull;
        atomicAdd(a.pool_top, 0ull - n);  // served from a free list after all
    }
    if (cl < FL_SMALL) {
        // the other blocks of the magazine go on the (empty) LDS stack
        const unsigned long long* w = (const unsigned long long*)(a.pool + m * POOL_UNIT);
        const uint32_t cnt = (uint32_t)min<unsigned long long>(max<unsigned long long>(w[1], 1ull), FL_LOCAL_MAX);
        const uint32_t* mem = (const uint32_t*)(w + 2);
        for (uint32_t j = 0; j + 1 < cnt; j++) fl[cl * FL_LOCAL_MAX + j] = mem[j];
        fln[cl] = cnt - 1;
    }
    return m * POOL_UNIT;
}

// A block of the record's size class (lane 0): this wave's LDS stack, a
// magazine of the wave's shard, fresh units from the bump pointer, and once
// the bump region is used up, a magazine of any other shard.  Returns the
// Vrec offset, or ~0 when the pool is exhausted (the bump pointer then keeps
// the failed request: the host reads what the launch needed).
__device__ __attribute__((always_inline)) unsigned long long pool_alloc(Ctx& c, uint32_t nvrec) {
    const ExpandArgs& a = *c.a;
    uint32_t units = 0;
    const int cl = pool_class(nvrec, units);
    const bool small = cl < FL_SMALL;
    if (small) {
        const uint32_t n = c.fln[cl];
        if (n > 0) {
            c.fln[cl] = n - 1;
            return (unsigned long long)c.fl[cl * FL_LOCAL_MAX + n - 1] * POOL_UNIT;
        }
    }
    return pool_alloc_shared(a, c.fl, c.fln, cl, units);
}

// The shared part of pool_free (out of line, like pool_alloc_shared).
__device__ __attribute__((noinline)) void pool_free_shared(const ExpandArgs& a, uint32_t* fl, uint32_t* fln, int cl,
                                                           unsigned long long idx) {
    unsigned long long* w = (unsigned long long*)(a.pool + idx * POOL_UNIT);
    if (cl < FL_SMALL) {
        const uint32_t n = fln[cl];
        const uint32_t k = a.fl_mag - 1;
        uint32_t* mem = (uint32_t*)(w + 2);
        for (uint32_t j = 0; j < k; j++) mem[j] = fl[cl * FL_LOCAL_MAX + n - k + j];
        fln[cl] = n - k;
        w[1] = k + 1;
    } else {
        w[1] = 1;
    }
    mag_push(a, fl_shard(a, cl, (int)(blockIdx.x % FL_SHARDS)), idx);
}

// Gives a block back (lane 0, after the wave has read the record).  A full
// LDS stack hands the block, with the stack's fl_mag - 1 newest entries
// listed in it, to the shard as one magazine.
__device__ __attribute__((always_inline)) void pool_free(Ctx& c, unsigned long long off, uint32_t nvrec) {
    const ExpandArgs& a = *c.a;
    uint32_t units = 0;
    const int cl = pool_class(nvrec, units);
    const unsigned long long idx = off / POOL_UNIT;
    if (cl < FL_SMALL) {
        const uint32_t n = c.fln[cl];
        if (n < 2 * a.fl_mag) {
            c.fl[cl * FL_LOCAL_MAX + n] = (uint32_t)idx;
            c.fln[cl] = n + 1;
            return;
        }
    }
    pool_free_shared(a, c.fl, c.fln, cl, idx);
}

// Claims up to n (<= 64) consecutive free cells of ring b for producers
// (whole wave; lane j checks the cell of position pos + j).  Returns how
// many were claimed (0: the ring is full, or max_tries attempts lost to
// other producers), their first position in *pos.
__device__ __attribute__((always_inline)) int ring_claim(Ctx& c, int b, int n, unsigned long long* pos_out,
                                                        int max_tries = 1 << 16) {
    const ExpandArgs& a = *c.a;
    unsigned long long* tp = &a.q_tail[b * QSTRIDE];
    const unsigned long long* seq = a.q_seq + (size_t)b * a.q_cap;
    for (int tries = 0; tries < max_tries; tries++) {
        unsigned long long pos = 0;
        if (c.lane == 0) pos = __hip_atomic_load(tp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        pos = rdlane64(pos, 0);
        const unsigned long long p = pos + (unsigned long long)c.lane;
        unsigned long long sq = 0;
        if (c.lane < n) sq = __hip_atomic_load(&seq[p % a.q_cap], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t freem = ballot(c.lane < n && sq == p);
        const uint64_t fullm = ballot(c.lane < n && sq < p);
        int k = freem == ~0ull ? WAVE : __builtin_ctzll(~freem);
        k = min(k, n);
        // lane 0's cell still holds the entry of the previous lap: full.  Not free
        // otherwise (k == 0): the tail moved under us.  (Tried again without a
        // branch of its own: with one the kernel for large roots had 347 scalars in
        // vector lanes instead of 259, and a window of a million-vertex graph took
        // 10.5 ms of kernel instead of 7.0.)
        if (fullm & 1ull) return 0;
        int ok = 0;
        if (c.lane == 0 && k > 0) {
            unsigned long long e = pos;
            ok = __hip_atomic_compare_exchange_strong(tp, &e, pos + (unsigned long long)k, __ATOMIC_RELAXED,
                                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                     ? 1
                     : 0;
        }
        if (rdlane(ok, 0)) {
            *pos_out = pos;
            return k;
        }
    }
    return 0;
}

// The same with a trace, whose one ring must not wrap (positions index the
// trace rows): its cells are free for their only lap, and one add takes the
// positions.  Every task goes through the ring then: 1,024 waves that tried to
// move its tail by compare and swap for each child spent 77% of a co-expression
// window's time on it.
__device__ __forceinline__ int ring_claim_trace(Ctx& c, int n, unsigned long long* pos_out) {
    const ExpandArgs& a = *c.a;
    unsigned long long pos = 0;
    if (c.lane == 0)
        pos = __hip_atomic_fetch_add(&a.q_tail[0], (unsigned long long)n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    pos = rdlane64(pos, 0);
    *pos_out = pos;
    return pos + (unsigned long long)n <= a.q_cap ? n : 0;
}

// The ring a producer's next task goes to: this wave's own shard when waves wait
// there (head ahead of tail) or nowhere, else the shard where most wait.
__device__ __attribute__((always_inline)) int ring_for(Ctx& c, int* waiting = nullptr) {
    const ExpandArgs& a = *c.a;
    if (a.q_shards == 1) return 0;
    int w = 0;
    if (c.lane < a.q_shards) {
        const unsigned long long h = __hip_atomic_load(&a.q_head[c.lane * QSTRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long t = __hip_atomic_load(&a.q_tail[c.lane * QSTRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        w = h > t ? (int)(h - t) : 0;
    }
    int r = c.shard, n = rdlane(w, c.shard);
    if (n == 0) {
        // (the lane in the low bits: the maximum names its shard)
        const int best = wave_max(w << 6 | c.lane);
        if (best >> 6) {
            r = best & 63;
            n = best >> 6;
        }
    }
    if (waiting) *waiting = n;
    return r;
}

// Publishes positions [pos, pos + k) of ring b (their refs are written):
// one release fence for the wave's record and ref stores, then the
// sequence words (lanes < k).
__device__ __forceinline__ void ring_publish(Ctx& c, int b, unsigned long long pos, int k) {
    const ExpandArgs& a = *c.a;
    wsync();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    if (c.lane < k) {
        const unsigned long long p = pos + (unsigned long long)c.lane;
        __hip_atomic_store(&a.q_seq[(size_t)b * a.q_cap + p % a.q_cap], p + 1ull, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Dynamic order: whether this child goes to a ring instead of the wave's own
// stack.  The stack's records are handed over only between tasks, so while a
// long task runs (a root, a large first-level task) its children would wait
// on this wave while other waves have nothing.  In tasks of SHARE_MIN_T
// vertices or more, every SHARE_EVERY children the wave compares the waves
// that wait for work with the tasks the rings hold (the pending word, as the
// hand-over between tasks does) and gives up to 16 of its next children to
// the rings when they fall short.  Smaller tasks end soon enough for the
// hand-over between tasks, and sending their children through the rings
// costs more than the wait (trees of 30-vertex tasks ran slower).  The word
// is loaded at one check and read at the next, so its latency overlaps the
// children built in between; a count one interval old only delays the answer.
constexpr int SHARE_EVERY = 8;
// fewest branches of an item when waves wait (an item loads its task's record,
// which takes as long as one to three branches)
constexpr int SPLIT_FINE = 4;
constexpr uint32_t SHARE_MIN_T = 64;
__device__ __forceinline__ bool share_child(Ctx& c) {
    const ExpandArgs& a = *c.a;
    if (!c.share_ok) return false;
    if (c.share_left > 0) {
        c.share_left--;
        return true;
    }
    if (++c.share_n < SHARE_EVERY) return false;
    c.share_n = 0;
    const unsigned long long ph = rdlane64(c.share_v, 0);
    if (c.lane == 0) c.share_v = __hip_atomic_load(a.pending, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const long long hg = (long long)(ph >> 32), pd = (long long)(ph & 0xFFFFFFFFull);
    const long long waiting = pd - ((long long)gridDim.x - hg);
    const long long need = hg - (waiting > 0 ? waiting : 0);
    if (need <= 0) return false;
    c.share_left = (int)min<long long>(need, 16ll) - 1;
    return true;
}

// One task ref into a ring (shared = true first; counted in `pending` before
// anyone can take it) or this wave's private stack (covered by the wave's
// own count while it is busy).  Returns false when both are full (the launch
// then reports a capacity overflow).
__device__ __attribute__((always_inline)) bool push_ref(Ctx& c, const TaskRef& r, int bkt, bool shared, const float* feat) {
    const ExpandArgs& a = *c.a;
    for (int pass = 0; pass < 2; pass++) {
        const bool ring = (pass == 0) == (shared || !a.use_priv);
        if (ring) {
            const int rg = ring_for(c);
            unsigned long long pos = 0;
            if ((a.trace_feat ? ring_claim_trace(c, 1, &pos) : ring_claim(c, rg, 1, &pos)) == 1) {
                const unsigned long long gi = (unsigned long long)rg * a.q_cap + pos % a.q_cap;
                if (c.lane == 0) {
                    __hip_atomic_fetch_add(a.pending, 1ull, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                    a.q_refs[gi] = r;
                    if (a.trace_parent) a.trace_parent[gi] = r.b1 > 0 ? -2 : c.slot;
                    if (a.trace_feat && feat)
                        for (int k = 0; k < 12; k++) a.trace_feat[gi * 12 + k] = feat[k];
                }
                ring_publish(c, rg, pos, 1);
                return true;
            }
        } else if (a.use_priv && c.ptop - c.pbot < a.priv_cap) {
            if (c.lane == 0) {
                c.pstack[c.ptop % a.priv_cap] = r;
                c.pbkt[c.ptop % a.priv_cap] = (unsigned char)bkt;
                *c.ptopref = r;  // the entry the next pop takes, kept in LDS too
            }
            c.ptopi = c.ptop;
            c.ptop++;
            return true;
        }
    }
    if (c.lane == 0) {
        atomicAdd(a.overflow, 1ull);
        atomicOr(a.error, 1);
    }
    return false;
}

// Static order: moves the staged children on this wave's stack into the
// ring, up to 64 per claim, oldest first (lane j copies entry j; the
// barrier makes lane 0's earlier stack stores visible to the other lanes).
// Returns false when the ring took none (it is full): the wave then runs
// its staged tasks itself.
__device__ __attribute__((always_inline)) bool static_flush(Ctx& c) {
    const ExpandArgs& a = *c.a;
    bool moved = false;
    wsync();
    while (c.ptop != c.pbot) {
        unsigned long long pos = 0;
        const int k = ring_claim(c, 0, (int)min<uint32_t>(c.ptop - c.pbot, (uint32_t)WAVE), &pos);
        if (k == 0) break;
        if (c.lane < k)
            a.q_refs[(pos + c.lane) % a.q_cap] = c.pstack[(c.pbot + (uint32_t)c.lane) % a.priv_cap];
        if (c.lane == 0)
            __hip_atomic_fetch_add(a.pending, (unsigned long long)k, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        ring_publish(c, 0, pos, k);
        c.pbot += (uint32_t)k;
        moved = true;
    }
    return moved;
}

// TaskRef as eight dwords, broadcast from lane l
__device__ __forceinline__ TaskRef bcast_ref(const TaskRef& mine, int l) {
    uint32_t w[8];
    __builtin_memcpy(w, &mine, sizeof(w));
#pragma unroll
    for (int k = 0; k < 8; k++) w[k] = (uint32_t)__builtin_amdgcn_readlane((int)w[k], l);
    TaskRef r;
    __builtin_memcpy(&r, w, sizeof(r));
    return r;
}

// ---------------------------------------------------------------------------
// subtrees of at most 64 vertices, in registers
// ---------------------------------------------------------------------------
// A task of at most 64 vertices and its whole subtree need no memory: lane l
// holds one vertex (ascending id order) with its 64-bit rows of the 1-hop and
// 2-hop relations among the task's vertices, every set is a 64-bit mask in
// scalar registers, a degree is the popcount of row & set, and a child of the
// task is one 32-bit word per lane.  The rows are gathered once, when the
// subtree's root is loaded; below it a vertex keeps its lane, children wait on
// a stack in the LDS (which no other task uses meanwhile), and records are
// written only for tasks handed to other waves.  The steps are those of
// process_task; lists become masks, so only the order of the branches (the
// key below) is kept of the records' order.
//
// Bound by the issue of dependent vector and scalar instructions (one or two
// waves a SIMD).  Through records and lists in LDS a task of this size took
// 40 us on a wave (load and matrix gathers 18%, flat LDS accesses and their
// waits most of the rest), here about 12 us; whole kernels are compared at the
// dispatch in expand_persistent.
constexpr uint32_t TINY_MAX = WAVE;
constexpr int TINY_EX_MAX = 8000;  // largest exdeg the word holds (stale exdegs can pass the task's size)
constexpr int TINY_EX_MIN = -64;   // smallest at load: a subtree lowers an exdeg by at most 63 more
constexpr int TINY_BIAS = 128;

// State word of a vertex: [12:0] exdeg + 128, [18:13] indeg, [24:19] order
// (lvl2adj, or 63 - position for a task loaded from a record), [25] member,
// [26] present; 0: not in the task.
constexpr uint32_t TW_MEMBER = 1u << 25, TW_PRESENT = 1u << 26;
__device__ __forceinline__ uint32_t tiny_word(int in, int ex, int ord, bool member) {
    return (uint32_t)(ex + TINY_BIAS) | ((uint32_t)in << 13) | ((uint32_t)ord << 19) | (member ? TW_MEMBER : 0u) |
           TW_PRESENT;
}
__device__ __forceinline__ int tw_ex(uint32_t w) { return (int)(w & 0x1FFFu) - TINY_BIAS; }
__device__ __forceinline__ int tw_in(uint32_t w) { return (int)((w >> 13) & 63u); }
// Q order of candidates (main.cu:2059-2104): indeg, exdeg, lvl2adj, id, all
// descending; the lane is the rank by id, so keys are unique and the last
// branch vertex is the smallest key's lane
__device__ __forceinline__ int tiny_key(uint32_t w, int lane) {
    return (int)((((w >> 13) & 63u) << 25) | ((w & 0x1FFFu) << 12) | (((w >> 19) & 63u) << 6) | (uint32_t)lane);
}

struct Tiny {
    uint64_t r1, r2;      // rows among the basis (bit = lane)
    int id;               // root-local id (ascending over the lanes)
    uint32_t orig;        // input id
    int d1, d2;           // |N n root|, |N2 n root|
    int mdt;              // mindeg[lane]
    int ubt;              // floor(lane / gamma)
    uint32_t s;           // word of the task to run next
    uint32_t hot;         // the child pushed last, not yet in the LDS
    int fr, ff;           // lane k: removed vertex and smallest failing member of the k-th failed removal
    int nf;
    uint32_t depth, hot_depth;
    bool hot_on;
    uint32_t n, bot;      // LDS stack: n entries from place bot (a ring)
    uint32_t cap;
    uint32_t tick;
    uint32_t tasks, branches, children, beyond;  // counters since the last flush
    unsigned long long sum_t, sum_tw;
};

// mindeg[i] for a uniform i >= 0
__device__ __forceinline__ int tiny_md(const Ctx& c, const Tiny& y, int i) {
    return i < WAVE ? rdlane(y.mdt, i) : uni(md(c, i));
}

// The basis from a record of t <= 64 vertices.  False (nothing changed but y)
// when a degree does not fit the state word: the caller runs the general path.
__device__ __attribute__((always_inline)) bool tiny_load(Ctx& c, const TaskRef& ref, Tiny& y) {
    const int t = (int)ref.t;
    const int lane = c.lane;
    const bool on = lane < t;
    Vrec v{0, 0, 0, 0};
    if (on) v = c.a->in_verts[ref.off + lane];
    if (ballot(on && (v.exdeg < TINY_EX_MIN || v.exdeg > TINY_EX_MAX || (uint32_t)v.indeg > 63u))) return false;
    int rk = 0;
    for (int i = 0; i < t; i++) rk += rdlane(v.id, i) < v.id ? 1 : 0;
    const int to = (on ? rk : lane) << 2;
    const uint32_t word = on ? tiny_word(v.indeg, v.exdeg, WAVE - 1 - lane, v.label == 1) : 0u;
    y.id = __builtin_amdgcn_ds_permute(to, v.id);
    y.s = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)word);
    const int rw = c.g.p->rw;
    const uint64_t* __restrict__ A1 = c.g.p->A1;
    const uint64_t* __restrict__ A2 = c.g.p->A2;
    const int cw = y.id >> 6;
    const uint64_t cm = 1ull << (y.id & 63);
    y.d1 = on ? c.g.p->d1r[y.id] : 0;
    y.d2 = on ? c.g.p->d2r[y.id] : 0;
    y.orig = on ? c.g.p->orig[y.id] : 0u;
    y.r1 = 0;
    y.r2 = 0;
    // (RU rows at a time: 2 RU gathers in flight per lane)
    constexpr int RU = 8;
    for (int i = 0; i < t; i += RU) {
        uint64_t x[RU], z[RU];
#pragma unroll
        for (int q = 0; q < RU; q++) {
            const int k = min(i + q, t - 1);
            const size_t rb = (size_t)rdlane(y.id, k) * rw + cw;
            x[q] = A1[rb];
            z[q] = A2[rb];
        }
#pragma unroll
        for (int q = 0; q < RU; q++) {
            const uint64_t b = ballot(on && (x[q] & cm)), e = ballot(on && (z[q] & cm));
            if (lane == min(i + q, t - 1)) {
                y.r1 = b;
                y.r2 = e;
            }
        }
    }
    y.mdt = md(c, lane);
    y.ubt = ub_quot(c, lane);
    y.depth = ref.depth;
    y.hot_on = false;
    y.hot = 0;
    y.hot_depth = 0;
    y.n = 0;
    y.bot = 0;
    y.nf = 0;
    y.fr = 0;
    y.ff = 0;
    y.tick = 0;
    y.tasks = y.branches = y.children = y.beyond = 0;
    y.sum_t = y.sum_tw = 0;
    return true;
}

// W_adj of the failed removals noted so far: the reference scans N(r) in
// ascending id order and stops after the first failing member
// (main.cu:1437-1450).  Noted per lane and counted here together: the row
// loads of different removals do not wait for each other.
__device__ __attribute__((always_inline)) void tiny_failed_scans(Ctx& c, Tiny& y) {
    const int rw = c.g.p->rw;
    const uint64_t* __restrict__ A1 = c.g.p->A1;
    int rank = 0;
    for (int k = 0; k < y.nf; k++) {
        const int rid = rdlane(y.fr, k), fid = rdlane(y.ff, k);
        const uint64_t* row = A1 + (size_t)rid * rw;
        for (int wd = c.lane; wd <= (fid >> 6); wd += WAVE) {
            uint64_t x = row[wd];
            if (wd == (fid >> 6)) x &= (1ull << (fid & 63)) - 1ull;
            rank += __popcll(x);
        }
    }
    c.wadj_l += rank + (c.lane < y.nf ? 1 : 0);
    y.nf = 0;
}

// counters into the wave's (LDS)
__device__ __attribute__((always_inline)) void tiny_counters(Ctx& c, Tiny& y) {
    if (c.lane == 0) {
        c.st->tasks += y.tasks;
        c.st->branches += y.branches;
        c.st->children += y.children;
        c.st->beyond += y.beyond;
        c.st->sum_t += y.sum_t;
        c.st->sum_tw += y.sum_tw;
    }
    y.tasks = y.branches = y.children = y.beyond = 0;
    y.sum_t = y.sum_tw = 0;
}

// LU bounds (lu_bounds) and the member checks over lane masks: members M (m
// of them), `cand` the lanes whose indegrees count (nc of them), in / ex per
// lane.  True: the record fails.
__device__ __forceinline__ bool tiny_bounds(Ctx& c, const Tiny& y, uint64_t M, int m, uint64_t cand, int nc, int in,
                                            int ex, int mds, int& ub, int& lb, int& med) {
    const bool mem = (M >> c.lane) & 1ull;
    const int ms = c.g.min_size;
    auto gm = [&](int s) { return s < ms ? mds : tiny_md(c, y, s); };  // get_mindeg
    // the smallest (indeg, exdeg) pair, exdeg as an unsigned field
    const int pair = wave_min(mem ? (in << 14) | (ex & 0x3FFF) : INT32_MAX);
    const int min_in = pair >> 14;
    bool invalid = false;
    const int gmm = gm(m);
    med = gm(m + 1);
    if (min_in < tiny_md(c, y, m)) {
        const int min_in_ex = (int)((uint32_t)pair << 18) >> 18;
        int x = gmm - min_in;
        for (;;) {
            const int k = x + c.lane;
            const uint64_t bm = ballot(k > min_in_ex || min_in + k >= md(c, m + k));
            if (bm) {
                x += __builtin_ctzll(bm);
                break;
            }
            x += WAVE;
        }
        lb = x;
        if (min_in + lb < tiny_md(c, y, m + lb)) {
            lb = nc + 1;
            invalid = true;
        }
        const int min_tot = wave_min(mem ? in + ex : INT32_MAX);
        // (a stale exdeg can make the sum negative: floor(d / gamma) is then
        // below 0 and the bound too)
        // (from 63 on floor(d / gamma) + 1 - m is nc or more)
        const int tq = min_tot < 0 ? -1 : rdlane(y.ubt, min(min_tot, WAVE - 1));
        ub = tq + 1 - m;
        if (ub > nc) ub = nc;
        if (lb < ub) {
            const int sum_in = wave_sum(mem ? in : 0);
            // P(idx) = sum over v >= 1 of min(#{indeg >= v}, idx), idx = lane
            const int xin = (cand >> c.lane) & 1ull ? in : 0;
            int p = 0;
            for (int v = 1;; v++) {
                const int k = __popcll(ballot(xin >= v));
                if (k == 0) break;
                p += min(k, c.lane);
            }
            const uint64_t ok = ballot(c.lane <= ub && c.lane >= lb && sum_in + p >= m * md(c, m + c.lane));
            if (ok == 0) {
                lb = ub + 1;
                invalid = true;
            } else {
                lb = __builtin_ctzll(ok);
                ub = min(ub, 63 - __builtin_clzll(ok));
                if (lb > 1) med = gm(m + lb);
            }
        }
    } else {
        ub = nc;
        lb = m < ms ? ms - m : 0;
    }
    if (m + ub < ms || ub < 0 || ub < lb) invalid = true;
    if (invalid) return true;
    // vert_isextendable_LU (vert_ext): the checks that do not depend on the
    // lane folded into two bounds; get_mindeg(m + ex) is mindeg[m + ex] under
    // the first of them (mindeg is monotone)
    const int tot = in + ex;
    const int T = max(max(mds, med), gm(m + lb));
    const bool f = mem && (tot < T || in + ub < tiny_md(c, y, m + ub) || tot < md(c, m + ex));
    return ballot(f) != 0;
}

// degree_pruning over lane masks: `alive` are the candidates that may stay,
// `dead` the others; on return `alive` holds those that stay.  True: fails.
// again: whether the same call on what it leaves could end otherwise (the last
// bounds counted fewer candidates than stay).
__device__ __attribute__((always_inline)) bool tiny_prune(Ctx& c, const Tiny& y, uint64_t M, int m, uint64_t& alive,
                                                          uint64_t dead, int in, int& ex, bool map_empty, int mds, int& ub,
                                                          int& lb, int& med, bool& again) {
    const int ms = c.g.min_size;
    const uint64_t me = 1ull << c.lane;
    int T = 0, U = 0;
    auto bounds = [&]() {
        const int g = m + lb < ms ? mds : tiny_md(c, y, m + lb);
        T = max(max(mds, med), g);
        U = tiny_md(c, y, m + lb) - ub + 1;
    };
    auto valid = [&]() { return in + ex >= T && in >= U && in + ex >= md(c, m + ex + 1); };  // cand_valid
    uint64_t rem = alive, rmv = dead, cnt_set = alive;
    bool first = true;
    for (;;) {
        if (tiny_bounds(c, y, M, m, cnt_set, __popcll(cnt_set), in, ex, mds, ub, lb, med)) return true;
        bounds();
        const uint64_t stay = ballot((rem & me) && valid());
        rmv = first ? dead | (rem & ~stay) : rem & ~stay;
        first = false;
        rem = stay;
        if (rem == 0 || rmv == 0) break;
        // degree update, main.cu:1775-1807
        const bool rc = __popcll(rem) < __popcll(rmv);
        const uint64_t L = rc ? rem : rmv;
        if (L & me) c.wadj_l += y.d1;
        if ((M | rem) & me) {
            if (map_empty) {
                if (rc) ex = 0;
            } else {
                const int k = __popcll(y.r1 & L);
                ex = rc ? k : ex - k;
            }
        }
        // the indegrees that count: candidates valid under the old bounds
        // with the new exdeg (main.cu:1811-1815)
        cnt_set = ballot((rem & me) && valid());
    }
    alive = rem;
    again = cnt_set != rem;
    return false;
}

// One task (y.s): its branches, children pushed on the stack (the caller has
// made room for them).
__device__ __attribute__((always_inline)) void tiny_task(Ctx& c, Tiny& y, uint32_t* stk, uint16_t* sdep) {
    const int lane = c.lane;
    const uint64_t me = 1ull << lane;
    const uint32_t w = y.s;
    const uint64_t P = ballot(w & TW_PRESENT), M = ballot(w & TW_MEMBER);
    const uint64_t C = P & ~M;
    const int t0 = __popcll(P), nm = __popcll(M), nc = __popcll(C);
    const int in = tw_in(w);
    int ex = tw_ex(w);
    const int ms = c.g.min_size;
    const int mds = tiny_md(c, y, ms);
    y.tasks++;
    y.sum_t += t0;
    // ---- lookahead ----
    const int req = tiny_md(c, y, t0);
    int l2 = 0;
    if (ballot((M & me) && in + ex < req) == 0) {
        if (C & me) {
            c.wadj_l += y.d2;
            l2 = __popcll(y.r2 & C);
        }
        if (ballot((C & me) && (l2 < nc - 1 || in + ex < req)) == 0) {
            emit_lanes(c, P, y.orig);
            return;
        }
    }
    // ---- branches ----
    const int mdg = nm < ms ? mds : tiny_md(c, y, nm);  // get_mindeg(nm)
    const bool keys = !(c.g.max_depth >= 0 && (int)y.depth + 1 > c.g.max_depth);
    uint64_t Cr = C;
    const int key = tiny_key(w, lane);
    int v = 0;
    for (int b = 0; b < nc; b++) {
        if (b > 0) {
            // remove_one_vertex: the last branch's vertex
            const uint64_t vb = 1ull << v;
            Cr &= ~vb;
            const bool adj = (y.r1 & vb) != 0;
            if (adj) ex--;
            const uint64_t fail = ballot(adj && (M & me) && in + ex < mdg);
            if (fail) {
                // (lanes are in id order: the lowest failing lane is scanned first)
                const int rid = rdlane(y.id, v), fid = rdlane(y.id, __builtin_ctzll(fail));
                if (lane == y.nf) {
                    y.fr = rid;
                    y.ff = fid;
                }
                if (++y.nf == WAVE) tiny_failed_scans(c, y);
                break;
            }
            if (lane == v) c.wadj_l += y.d1;
        }
        v = wave_min((Cr & me) ? key : INT32_MAX) & (WAVE - 1);
        y.branches++;
        if (lane == v) c.wadj_l += y.d1 + y.d2;
        // the child: members and v, candidates inside N2(v)
        uint64_t Mc = M | (1ull << v);
        int m = nm + 1;
        const uint64_t rest = Cr & ~(1ull << v);
        uint64_t alive = rest & rdlane64(y.r2, v), dead = rest & ~alive;
        const int a1 = (int)((y.r1 >> v) & 1ull);
        int ci = in + a1, ce = ex - a1;
        int ub = 0, lb = 0, med = 0;
        bool map_empty = false, first = true, fails, again = true;
        for (;;) {
            fails = tiny_prune(c, y, Mc, m, alive, dead, ci, ce, map_empty, mds, ub, lb, med, again);
            if (!first || fails) break;
            first = false;
            // critical_prep
            const int thr = tiny_md(c, y, m + lb);
            const uint64_t cm = ballot((Mc & me) && ci + ce == thr && ce > 0);
            if (cm & me) c.wadj_l += y.d1;
            const uint64_t F = cm ? ballot((alive & me) && (y.r1 & cm)) : 0ull;
            dead = 0;
            if (F == 0) {
                // nothing changed: the closing degree pruning ends as the first
                // one did, unless that one's last bounds counted fewer
                if (!again) break;
                map_empty = true;
                continue;
            }
            const int ncrit = __popcll(F);
            if (F & me) c.wadj_l += y.d1 + y.d2;
            const int x1 = __popcll(y.r1 & F), x2 = __popcll(y.r2 & F);
            ci += x1;
            ce -= x1;
            if (ballot(((Mc & me) && x2 != ncrit) || ((F & me) && x2 < ncrit - 1))) {
                m = -1;  // the reference's 2: neither a clique test nor a child
                break;
            }
            Mc |= F;
            m += ncrit;
            const uint64_t left = alive & ~F;
            alive = left & ballot(x2 == ncrit);
            dead = left & ~alive;
        }
        if (m < 0) continue;
        if (m >= ms && ballot((Mc & me) && ci < tiny_md(c, y, m)) == 0) emit_lanes(c, Mc, y.orig);
        if (fails || alive == 0) continue;
        y.children++;
        y.sum_tw += m + __popcll(alive);
        if (!keys) {
            y.beyond++;
            continue;
        }
        if (y.hot_on) {
            uint32_t at = y.bot + y.n;
            if (at >= y.cap) at -= y.cap;
            stk[at * WAVE + lane] = y.hot;
            if (lane == 0) sdep[at] = (uint16_t)y.hot_depth;
            y.n++;
        }
        y.hot_on = true;
        y.hot_depth = y.depth + 1;
        y.hot = ((Mc | alive) & me) ? tiny_word(ci, ce, l2, (Mc & me) != 0) : 0u;
    }
}

// the task after this one (the child pushed last, else the top of the stack)
__device__ __forceinline__ bool tiny_next(Ctx& c, Tiny& y, const uint32_t* stk, const uint16_t* sdep) {
    if (y.hot_on) {
        y.s = y.hot;
        y.depth = y.hot_depth;
        y.hot_on = false;
        return true;
    }
    if (y.n == 0) return false;
    y.n--;
    uint32_t at = y.bot + y.n;
    if (at >= y.cap) at -= y.cap;
    wsync();
    y.s = stk[at * WAVE + c.lane];
    y.depth = (uint32_t)uni((int)sdep[at]);
    return true;
}

// place of every lane's vertex in the record of task word w: members first
// (ascending id), then the candidates in Q order
__device__ __forceinline__ int tiny_place(Ctx& c, uint32_t w, uint64_t M, uint64_t C) {
    const int key = tiny_key(w, c.lane);
    int rank = __popcll(M);
    for (uint64_t s = C; s; s &= s - 1) rank += rdlane(key, __builtin_ctzll(s)) > key ? 1 : 0;
    return (M >> c.lane) & 1ull ? lanes_below(M) : rank;
}

// The k oldest tasks of the stack become records on the wave's own task stack
// (for the rings, or because the LDS stack needs room).
__device__ __attribute__((always_inline)) void tiny_spill(Ctx& c, Tiny& y, const uint32_t* stk, const uint16_t* sdep,
                                                          uint32_t k) {
    const ExpandArgs& a = *c.a;
    wsync();
    for (; k > 0; k--) {
        const uint32_t w = stk[y.bot * WAVE + c.lane];
        const uint32_t depth = (uint32_t)uni((int)sdep[y.bot]);
        if (++y.bot == y.cap) y.bot = 0;
        y.n--;
        const uint64_t P = ballot(w & TW_PRESENT), M = ballot(w & TW_MEMBER);
        const int t = __popcll(P);
        unsigned long long si = 0;
        if (c.lane == 0) si = pool_alloc(c, (uint32_t)t);
        si = rdlane64(si, 0);
        if (si == ~0ull) {
            if (c.lane == 0) atomicOr(a.error, 1);
            continue;
        }
        const int at = tiny_place(c, w, M, P & ~M);
        if (w & TW_PRESENT) a.pool[si + at] = Vrec{y.id, (w & TW_MEMBER) ? 1 : 0, tw_in(w), tw_ex(w)};
        TaskRef r;
        r.off = si;
        r.t = (uint32_t)t;
        r.depth = (uint16_t)depth;
        r.inst = (uint16_t)c.inst;
        r.bound = 0;
        r.b0 = 0;
        r.b1 = 0;
        push_ref(c, r, 0, !a.use_priv, nullptr);
    }
}

// moves the child pushed last to the stack
__device__ __forceinline__ void tiny_unhot(Ctx& c, Tiny& y, uint32_t* stk, uint16_t* sdep) {
    if (!y.hot_on) return;
    uint32_t at = y.bot + y.n;
    if (at >= y.cap) at -= y.cap;
    stk[at * WAVE + c.lane] = y.hot;
    if (c.lane == 0) sdep[at] = (uint16_t)y.hot_depth;
    y.n++;
    y.hot_on = false;
}

// Runs the subtree; returns true when it stopped to hand tasks over (their
// records are on the wave's own stack) and has to be resumed, false when it
// is done.  One task only, its children all made records, in the static order
// (whose tasks are dealt to the waves in turn).
__device__ __attribute__((always_inline)) bool tiny_run(Ctx& c, Tiny& y, uint32_t* stk, uint16_t* sdep, bool go_on) {
    const ExpandArgs& a = *c.a;
    bool more = go_on ? tiny_next(c, y, stk, sdep) : true;
    while (more) {
        const uint32_t nc = (uint32_t)__popcll(ballot((y.s & (TW_PRESENT | TW_MEMBER)) == TW_PRESENT));
        uint32_t out = y.n + nc > y.cap ? y.n + nc - y.cap : 0u;
        bool give = false;
        // (looked at every 4 tasks while 4 or more wait on the stack, else every
        // 16: a task given from a short stack is a few us of work for 10 of
        // hand-over.  Every 4 in any case, a full search took 10.4 ms against
        // 7.8 and a power-law window 9.3 against 7.6; every 16, 3,051 tasks took
        // 0.97 against 0.68.)
        if (!a.static_sched && (++y.tick & (y.n >= 4u ? 3u : 15u)) == 0) {
            // more waves wait for work than the rings hold (as between
            // tasks of the general loop, with the word read at one check and
            // used at the next): up to 16 of the oldest tasks go out
            const unsigned long long ph = rdlane64(c.share_v, 0);
            if (c.lane == 0) c.share_v = __hip_atomic_load(a.pending, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const long long hg = (long long)(ph >> 32), pd = (long long)(ph & 0xFFFFFFFFull);
            const long long waiting = pd - ((long long)gridDim.x - hg);
            const long long need = hg - (waiting > 0 ? waiting : 0);
            // every busy wave reads the same need: each answers with the
            // chance that twice the need is met between them (a record made
            // and not taken costs its basis again)
            const long long busy = (long long)gridDim.x - hg;
            const uint32_t dice = (blockIdx.x * 0x9E3779B9u + y.tick * 0x85EBCA6Bu) >> 8;
            if (need > 0 && y.n > 0 && (2 * need >= busy || (long long)(((unsigned long long)dice * busy) >> 24) < 2 * need)) {
                give = true;
                const long long share = need / max(1ll, busy) + 1;
                out = max(out, (uint32_t)min<long long>(min<long long>(share, 16ll), (long long)y.n));
            }
        }
        if (out) tiny_spill(c, y, stk, sdep, out);
        if (give) {
            // the task to run next waits in front of the stack
            y.hot = y.s;
            y.hot_depth = y.depth;
            y.hot_on = true;
            return true;
        }
        tiny_task(c, y, stk, sdep);
        if (a.static_sched) {
            tiny_unhot(c, y, stk, sdep);
            tiny_spill(c, y, stk, sdep, y.n);
        }
        more = tiny_next(c, y, stk, sdep);
    }
    tiny_failed_scans(c, y);
    tiny_counters(c, y);
    return false;
}

// Level-synchronous form: one task, its children written to the output
// stream with one claim for all of them.
__device__ __attribute__((always_inline)) void tiny_level(Ctx& c, Tiny& y, uint32_t* stk, uint16_t* sdep) {
    const ExpandArgs& a = *c.a;
    tiny_task(c, y, stk, sdep);
    tiny_unhot(c, y, stk, sdep);
    const uint32_t n = y.n;
    const unsigned long long slots = y.beyond ? 0ull : y.sum_tw;
    tiny_failed_scans(c, y);
    tiny_counters(c, y);
    if (n == 0) return;
    unsigned long long ri = 0, si = 0;
    if (c.lane == 0) {
        ri = atomicAdd(&a.out_ctr[0].items, (unsigned long long)n);
        si = atomicAdd(&a.out_ctr[0].slots, slots);
    }
    ri = rdlane64(ri, 0);
    si = rdlane64(si, 0);
    if (ri + n > a.out_ref_cap[0] || si + slots > a.out_vert_cap[0]) {
        if (c.lane == 0) atomicOr(a.error, 1);
        return;
    }
    wsync();
    for (uint32_t k = 0; k < n; k++) {
        const uint32_t w = stk[k * WAVE + c.lane];
        const uint64_t P = ballot(w & TW_PRESENT), M = ballot(w & TW_MEMBER), C = P & ~M;
        const int t = __popcll(P), nm = __popcll(M);
        const int at = tiny_place(c, w, M, C);
        if (w & TW_PRESENT) a.out_verts[0][si + at] = Vrec{y.id, (w & TW_MEMBER) ? 1 : 0, tw_in(w), tw_ex(w)};
        // slot bound of this child's own children (see TaskRef)
        const bool kids = a.all_bounds || !(c.g.max_depth >= 0 && (int)c.depth + 2 > c.g.max_depth);
        const int bnd = wave_sum(kids && ((C >> c.lane) & 1ull) ? min(y.d2 + nm + 1, t) : 0);
        if (c.lane == 0) {
            TaskRef r;
            r.off = si;
            r.t = (uint32_t)t;
            r.depth = (uint16_t)(c.depth + 1);
            r.inst = (uint16_t)c.inst;
            r.bound = (uint64_t)bnd;
            r.b0 = 0;
            r.b1 = 0;
            a.out_refs[0][ri + k] = r;
        }
        si += t;
    }
}

// ---------------------------------------------------------------------------
// tasks of more than 64 vertices
// ---------------------------------------------------------------------------
// The steps of h_expand_level's body (main.cu:1060-1181) on a compact layout: a
// vertex's indeg and exdeg are one 32-bit word, a child vertex is that word
// and its position in the parent, 20 bytes a vertex for parent and child
// together.  With WideLds all of it is in LDS (about 1,700 vertices at 4 waves
// per CU); with WideSlab the arrays are in the wave's HBM slab, read and
// written in order, and only bit masks, rows and short sorts use the LDS.
//   * A branch reads two matrix rows (N and N2 of its vertex), loaded while
//     the branch before it runs and kept in LDS; the bits of N are kept per
//     position for the removal that follows (main.cu:1437-1450).
//   * Every access is a ds_ or global_ instruction on an array known to be
//     there; several chunks of 64 are loaded before the first is used.
//   * Removed candidates leave the arrays at once (one list of positions,
//     only written when there are any): nothing scans what was removed.
//   * The indegree counts of the LU bounds are made only when the bounds
//     get that far, and their index search stops at the first hit from
//     either end.
//   * Counts against a set of vertices walk the set's rows (one scalar row
//     address for 64 lanes, neighbouring words) while the set is small.
// The order of members and of candidates inside a child is free: the record
// written is sorted by a key that is unique.
constexpr uint32_t WIDE_LDS_MAX = WIDE_TASK_MAX;   // WideLds: positions, indegrees and the sort key's fields
constexpr int WIDE_LDS_R_MAX = 1 << 20;   // WideLds: ids in a sort key
constexpr int WIDE_ROW_WORDS = 256;       // rows up to this size (R <= 16,384) are staged in LDS

// orders this wave's LDS and memory accesses among its lanes (they execute
// in order: only the compiler is held, no outstanding load is waited for)
__device__ __forceinline__ void lsync() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

template <class T>
using gptr = __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ gptr<const T> glob(const T* p) {
    return (gptr<const T>)p;
}
template <class T>
__device__ __forceinline__ gptr<T> globw(T* p) {
    return (gptr<T>)p;
}

// Vertex word: indeg above EXB bits of exdeg + BIAS; exdeg is accepted at load
// within LIMIT of 0 (a task lowers it by less than its size after that).
template <class W, int EXB_, int BIAS_, int LIMIT_>
struct WideWord {
    using word = W;
    static constexpr int EXB = EXB_, BIAS = BIAS_, LIMIT = LIMIT_;
    static constexpr W MASK = ((W)1 << EXB) - 1;
    static constexpr W ADJ1 = ((W)1 << EXB) - 1;  // indeg + 1, exdeg - 1
    static __device__ __forceinline__ int in(W w) { return (int)(w >> EXB); }
    static __device__ __forceinline__ int ex(W w) { return (int)(w & MASK) - BIAS; }
    static __device__ __forceinline__ W make(int in, int ex) { return ((W)(uint32_t)in << EXB) | (W)(uint32_t)(ex + BIAS); }
    static __device__ __forceinline__ W set_ex(W w, int ex) { return (w & ~MASK) | (W)(uint32_t)(ex + BIAS); }
};
struct WideLds : WideWord<uint32_t, 20, 1 << 17, 1 << 16> {
    static constexpr bool slab = false;
    static constexpr int U = 2;  // chunks of 64 in flight
    static constexpr bool cw_lds = true;
    using u32p = uint32_t*;
    using wordp = uint32_t*;
    using cwordp = uint32_t*;
    using posp = uint16_t*;
    using pos_t = uint16_t;
    using keyp = uint64_t*;
};
struct WideSlab : WideWord<uint64_t, 32, 1 << 30, 1 << 29> {
    static constexpr bool slab = true;
    static constexpr int U = 4;
    using u32p = gptr<uint32_t>;
    static constexpr bool cw_lds = false;
    using wordp = gptr<uint64_t>;
    using cwordp = gptr<uint64_t>;
    using posp = gptr<uint32_t>;
    using pos_t = uint32_t;
    using keyp = gptr<uint64_t>;
};

// the slab with 16-bit ids and positions and WideLds' words: half the bytes
// that a branch reads and writes per vertex, which bound the first branches of a
// power-law graph (tasks of 3,000 vertices, 2,048 slabs: 160 -> 146 ms)
struct WideMid : WideWord<uint32_t, 20, 1 << 17, 1 << 16> {
    static constexpr bool slab = true;
    static constexpr int U = 4;
    static constexpr bool cw_lds = false;
    using u32p = gptr<uint16_t>;
    using wordp = gptr<uint32_t>;
    using cwordp = gptr<uint32_t>;
    using posp = gptr<uint16_t>;
    using pos_t = uint16_t;
    using keyp = gptr<uint64_t>;
};
// the same with the child's words in LDS, which every pass over the child's
// candidates reads: up to 3,200 vertices with 20 KB a wave
struct WideMidLds : WideMid {
    static constexpr bool cw_lds = true;
    using cwordp = uint32_t*;
};
constexpr int WIDE_MID_R_MAX = 1 << 16;

__device__ __forceinline__ bool wide_rows_staged(uint32_t rw, uint32_t lds_bytes) {
    return rw <= (uint32_t)WIDE_ROW_WORDS && 24u * rw <= lds_bytes;
}

template <class P>
struct Wide {
    uint64_t* row1;         // LDS: rows of the branch vertex (rl)
    uint64_t* row2;
    uint64_t* lmask;        // LDS: a set of vertices in root space (ml)
    uint64_t* nbits;        // N of the branch vertex by parent position (LDS; in the slab when too large)
    uint64_t* flag;         // a bit per candidate (as nbits)
    typename P::u32p pid;   // parent: root-local id
    typename P::wordp pw;   //         indeg / exdeg word
    typename P::posp pl2;   //         lvl2adj
    typename P::posp cpos;  // child: position in the parent
    typename P::cwordp cw;  //        word
    typename P::posp list;  // positions (parent) of removed candidates, and other short lists (T entries)
    typename P::posp tab;   // counts per indegree (T entries)
    typename P::keyp keys;  // sort keys (WideLds: in the place of cw, list and tab; WideSlab: 2 T entries)
    char* spare;            // LDS behind the masks and rows (WideSlab: short sorts)
    uint32_t spare_bytes;
    gptr<const uint64_t> A1, A2;
    gptr<const int32_t> d1r, d2r;
    int T;             // capacity of the arrays
    int rw;            // words per row
    int idb;           // WideLds: bits of the id in a sort key
    int mdt;           // mindeg[lane]
    int mds;           // mindeg[min_size]
    int ubt;           // floor(lane / gamma)
    bool rl;           // rows are staged in LDS
    bool ml;           // lmask has room for a row
    int tb, ub1;       // cand_valid's lane-independent bounds, from the last wide_bounds
};

template <class P>
__device__ __forceinline__ int wide_md(const Ctx& c, const Wide<P>& z, int i) {
    return i < WAVE ? rdlane(z.mdt, i) : uni(md(c, i));
}

// cand_valid (main.cu:2153-2173) with the lane-independent checks in tb, ub1
template <class P>
__device__ __forceinline__ bool wide_valid(const Ctx& c, int tb, int ub1, int m, typename P::word w) {
    const int in = P::in(w), ex = P::ex(w), tot = in + ex;
    return tot >= tb && in >= ub1 && tot >= md(c, m + ex + 1);
}

// LU bounds (main.cu:1857-1972) and the member checks of a child with members
// [0, m): nc candidates count, all of [m, m + n) or, with `sub`, those valid
// under the bounds (tb0, ub0).  True: the record fails.
template <class P>
__device__ __attribute__((always_inline)) bool wide_bounds(Ctx& c, Wide<P>& z, int m, int n, int nc, bool sub, int tb0,
                                                           int ub0, int& ub, int& lb, int& med) {
    const int ms = c.g.min_size;
    auto gm = [&](int s) { return s < ms ? z.mds : wide_md(c, z, s); };
    // smallest (indeg, exdeg) pair, exdeg compared as an unsigned value
    int min_in, min_in_ex, min_tot = INT32_MAX, sum_in = 0;
    if constexpr (sizeof(typename P::word) == 4) {
        // (in one word, compared as signed with the top bit flipped)
        int pair = INT32_MAX;
        for (int i = c.lane; i < m; i += WAVE) {
            const uint32_t w = z.cw[i];
            const int in = P::in(w), ex = P::ex(w);
            pair = min(pair, (int)((((uint32_t)in << P::EXB) | ((uint32_t)ex & P::MASK)) ^ 0x80000000u));
            min_tot = min(min_tot, in + ex);
            sum_in += in;
        }
        const uint32_t mp = (uint32_t)wave_min(pair) ^ 0x80000000u;
        min_in = (int)(mp >> P::EXB);
        min_in_ex = (int)(mp << (32 - P::EXB)) >> (32 - P::EXB);
    } else {
        uint64_t pair = ~0ull;
        for (int i = c.lane; i < m; i += WAVE) {
            const uint64_t w = z.cw[i];
            const int in = P::in(w), ex = P::ex(w);
            pair = min(pair, ((uint64_t)(uint32_t)in << 32) | (uint32_t)ex);
            min_tot = min(min_tot, in + ex);
            sum_in += in;
        }
        pair = wave_min_u64(pair);
        min_in = (int)(pair >> 32);
        min_in_ex = (int)(uint32_t)pair;
    }
    bool invalid = false;
    med = gm(m + 1);
    if (min_in < wide_md(c, z, m)) {
        int x = gm(m) - min_in;
        for (;;) {
            const int k = x + c.lane;
            const uint64_t bm = ballot(k > min_in_ex || min_in + k >= md(c, m + k));
            if (bm) {
                x += __builtin_ctzll(bm);
                break;
            }
            x += WAVE;
        }
        lb = uni(x);
        if (min_in + lb < wide_md(c, z, m + lb)) {
            lb = nc + 1;
            invalid = true;
        }
        min_tot = wave_min(min_tot);
        // (a stale exdeg can make the sum negative: floor(d / gamma) is then
        // below 0 and the bound too)
        const int tq = min_tot < 0 ? -1 : min_tot < WAVE ? rdlane(z.ubt, min_tot) : uni(ub_quot(c, min_tot));
        ub = tq + 1 - m;
        if (ub > nc) ub = nc;
        ub = uni(ub);
        if (lb < ub) {
            // (32-bit words: t <= 4,095, so degree sums and products fit 32 bits)
            using num = typename std::conditional<sizeof(typename P::word) == 8, long long, int>::type;
            num sum_all;
            if constexpr (sizeof(typename P::word) == 8)
                sum_all = wave_sum64((long long)sum_in);
            else
                sum_all = wave_sum(sum_in);
            // C[v] = #{indeg >= v}: lane v holds it while every value is
            // below 64, else a table
            int V = 0, creg = 0;
            const bool reg = m < WAVE;
            auto indeg = [&](int i) {  // of candidate i, 0 when it does not count
                if (i >= m + n) return 0;
                const typename P::word w = z.cw[i];
                return !sub || wide_valid<P>(c, tb0, ub0, m, w) ? P::in(w) : 0;
            };
            if (m <= 4 && n > 2 * WAVE) {
                // values 1 to 4, the first levels of a search: as below with
                // one word a lane and two sums
                int cnt[5] = {0, 0, 0, 0, 0};
                for (int b0 = m; b0 < m + n; b0 += 255 * WAVE) {
                    uint32_t acc = 0;
                    const int b1 = min(m + n, b0 + 255 * WAVE);
#pragma unroll 4
                    for (int base = b0; base < b1; base += WAVE) {
                        const int x = indeg(base + c.lane);
                        acc += x ? 1u << (x * 8 - 8) : 0u;
                    }
                    const uint32_t f0 = (uint32_t)wave_sum((int)(acc & 0x00FF00FFu));
                    const uint32_t f1 = (uint32_t)wave_sum((int)((acc >> 8) & 0x00FF00FFu));
                    cnt[1] += (int)(f0 & 0xFFFFu);
                    cnt[2] += (int)(f1 & 0xFFFFu);
                    cnt[3] += (int)(f0 >> 16);
                    cnt[4] += (int)(f1 >> 16);
                }
                int run = 0;
#pragma unroll
                for (int v = 4; v >= 1; v--) {
                    run += cnt[v];
                    if (run && V == 0) V = v;
                    if (c.lane == v) creg = run;
                }
            } else if (m < 16 && n > 2 * WAVE) {
                // values below 16: every lane counts its own in 8-bit fields
                // (of at most 255 chunks at a time), then sums of 16- and
                // 32-bit fields over the lanes
                int cnt[16];
#pragma unroll
                for (int v = 0; v < 16; v++) cnt[v] = 0;
                for (int b0 = m; b0 < m + n; b0 += 255 * WAVE) {
                    unsigned long long lo = 0, hi = 0;
                    const int b1 = min(m + n, b0 + 255 * WAVE);
#pragma unroll 4
                    for (int base = b0; base < b1; base += WAVE) {
                        const int x = indeg(base + c.lane);
                        const unsigned long long one = 1ull << ((x & 7) * 8);
                        lo += x < 8 ? one : 0ull;
                        hi += x < 8 ? 0ull : one;
                    }
                    constexpr unsigned long long EV = 0x00FF00FF00FF00FFull;
                    auto sum = [](unsigned long long x, unsigned long long y) { return x + y; };
                    // (64 lanes x 255 fit 16 bits)
                    const unsigned long long f0 = wave_reduce64(lo & EV, 0ull, sum);
                    const unsigned long long f1 = wave_reduce64((lo >> 8) & EV, 0ull, sum);
                    unsigned long long f2 = 0, f3 = 0;
                    if (m >= 8) {
                        f2 = wave_reduce64(hi & EV, 0ull, sum);
                        f3 = wave_reduce64((hi >> 8) & EV, 0ull, sum);
                    }
#pragma unroll
                    for (int v = 1; v < 16; v++) {
                        const unsigned long long f = v & 8 ? (v & 1 ? f3 : f2) : (v & 1 ? f1 : f0);
                        cnt[v] += (int)((f >> (((v & 7) >> 1) * 16)) & 0xFFFFull);
                    }
                }
                int run = 0;
#pragma unroll
                for (int v = 15; v >= 1; v--) {
                    run += cnt[v];
                    if (run && V == 0) V = v;
                    if (c.lane == v) creg = run;
                }
            } else if (reg) {
                for (int base = m; base < m + n; base += WAVE) {
                    const int xin = indeg(base + c.lane);
                    int v = 1;
                    for (;; v++) {
                        const int k = __popcll(ballot(xin >= v));
                        if (k == 0) break;
                        if (c.lane == v) creg += k;
                    }
                    V = max(V, v - 1);
                }
            } else {
                for (int v = 1;; v++) {
                    int k = 0;
                    for (int base = m; base < m + n; base += WAVE) k += __popcll(ballot(indeg(base + c.lane) >= v));
                    if (k == 0) break;
                    if (c.lane == 0) z.tab[v] = (typename P::pos_t)k;
                    V = v;
                }
                lsync();
            }
            // the condition for 64 values of idx, P(idx) = sum of
            // min(C[v], idx) over v >= 1; the first value that holds is looked
            // for from lb up, the last from ub down (nearly always in the
            // first 64 on either side)
            auto holds = [&](int base) -> uint64_t {
                const int idx = base + c.lane;
                num p = 0;
                if (reg) {
                    int q = 0;
                    for (int v = 1; v <= V; v++) q += min(rdlane(creg, v), idx);
                    p = q;
                } else {
                    for (int v = 1; v <= V; v++) p += min((int)z.tab[v], idx);
                }
                return ballot(idx <= ub && idx >= lb && sum_all + p >= (num)m * md(c, m + idx));
            };
            int first = -1, last = -1, base = lb & ~(WAVE - 1);
            uint64_t ok = 0;
            for (; base <= ub; base += WAVE) {
                ok = holds(base);
                if (ok) break;
            }
            if (ok) {
                first = base + __builtin_ctzll(ok);
                int top = ub & ~(WAVE - 1);
                for (; top > base; top -= WAVE) {
                    const uint64_t up = holds(top);
                    if (up) {
                        ok = up;
                        break;
                    }
                }
                last = top + 63 - __builtin_clzll(ok);
            }
            if (first < 0) {
                lb = ub + 1;
                invalid = true;
            } else {
                lb = first;
                ub = min(ub, last);
                if (lb > 1) med = gm(m + lb);
            }
        }
    } else {
        ub = nc;
        lb = m < ms ? ms - m : 0;
    }
    if (m + ub < ms || ub < 0 || ub < lb) invalid = true;
    if (invalid) return true;
    // vert_isextendable_LU (vert_ext) for the members: the checks that do not
    // depend on the vertex folded into two bounds; get_mindeg(m + ex) is
    // mindeg[m + ex] under the first of them (mindeg is monotone)
    const int g = gm(m + lb);
    const int tb = max(max(z.mds, med), g);
    const int um = wide_md(c, z, m + ub) - ub;
    bool f = false;
    for (int i = c.lane; i < m; i += WAVE) {
        const typename P::word w = z.cw[i];
        const int in = P::in(w), ex = P::ex(w), tot = in + ex;
        if (tot < tb || in < um || tot < md(c, m + ex)) f = true;
    }
    if (ballot(f)) return true;
    z.tb = tb;
    z.ub1 = wide_md(c, z, m + lb) - ub + 1;
    return false;
}

// |row(id) n L| for this lane's id against the vertices of L: lane k of
// `ids` holds L's k-th vertex of the group, nl <= 64 of them (X: A1 or A2).
__device__ __forceinline__ int wide_count(gptr<const uint64_t> X, int rw, int ids, int nl, int id) {
    const int wd = id >> 6, sh = id & 63;
    int n = 0, k = 0;
    for (; k + 4 <= nl; k += 4) {
        uint64_t x[4];
#pragma unroll
        for (int q = 0; q < 4; q++) x[q] = X[(size_t)rdlane(ids, k + q) * rw + wd];
#pragma unroll
        for (int q = 0; q < 4; q++) n += (int)((x[q] >> sh) & 1ull);
    }
    for (; k < nl; k++) n += (int)((X[(size_t)rdlane(ids, k) * rw + wd] >> sh) & 1ull);
    return n;
}
// the same for four chunks of ids: 16 words in flight, where rows are long and
// far apart (a recount of 700 candidates against each other on rows of 1,096
// words took 4 ms a chunk at a time)
struct Count4 {
    int n0, n1, n2, n3;
};
__device__ __forceinline__ Count4 wide_count4(gptr<const uint64_t> X, int rw, int ids, int nl, int i0, int i1, int i2,
                                              int i3) {
    Count4 c{0, 0, 0, 0};
    const int w0 = i0 >> 6, w1 = i1 >> 6, w2 = i2 >> 6, w3 = i3 >> 6;
    auto bit = [](uint64_t x, int i) { return (int)((x >> (i & 63)) & 1ull); };
    int k = 0;
    for (; k + 4 <= nl; k += 4) {
        uint64_t x[4][4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            gptr<const uint64_t> r = X + (size_t)rdlane(ids, k + q) * rw;
            x[q][0] = r[w0];
            x[q][1] = r[w1];
            x[q][2] = r[w2];
            x[q][3] = r[w3];
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            c.n0 += bit(x[q][0], i0);
            c.n1 += bit(x[q][1], i1);
            c.n2 += bit(x[q][2], i2);
            c.n3 += bit(x[q][3], i3);
        }
    }
    for (; k < nl; k++) {
        gptr<const uint64_t> r = X + (size_t)rdlane(ids, k) * rw;
        const uint64_t x0 = r[w0], x1 = r[w1], x2 = r[w2], x3 = r[w3];
        c.n0 += bit(x0, i0);
        c.n1 += bit(x1, i1);
        c.n2 += bit(x2, i2);
        c.n3 += bit(x3, i3);
    }
    return c;
}
// the same against a mask in LDS
__device__ __forceinline__ int wide_rowpop(gptr<const uint64_t> X, int rw, const uint64_t* mask, int id) {
    gptr<const uint64_t> r = X + (size_t)id * rw;
    int s = 0, w = 0;
    for (; w + 8 <= rw; w += 8) {
        uint64_t x[8];
#pragma unroll
        for (int q = 0; q < 8; q++) x[q] = r[w + q];
#pragma unroll
        for (int q = 0; q < 8; q++) s += __popcll(x[q] & mask[w + q]);
    }
    for (; w < rw; w++) s += __popcll(r[w] & mask[w]);
    return s;
}

// the same for 64 rows, 8 at a time: the lanes share a row's words (a lane on its
// own row touches 64 lines with every load, which the L1 does not keep until
// the row's next words are read).  Sums of two rows share a word (R <= 16,384).
// For the slab's tasks: one in LDS has no registers to spare for it, and gained
// nothing.
__device__ __forceinline__ int wide_rowpop_shared(const Ctx& c, gptr<const uint64_t> X, int rw, const uint64_t* mask, int id) {
    int out = 0;
#pragma unroll 1
    for (int g = 0; g < 8; g++) {
        uint32_t s[4] = {0, 0, 0, 0};
        gptr<const uint64_t> r[8];
#pragma unroll
        for (int k = 0; k < 8; k++) r[k] = X + (size_t)rdlane(id, g * 8 + k) * rw;
#pragma unroll 2
        for (int w0 = 0; w0 < rw; w0 += WAVE) {
            const int wd = w0 + c.lane;
            uint64_t x[8];
            uint64_t mk = 0;
            if (wd < rw) mk = mask[wd];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                x[k] = 0;
                if (wd < rw) x[k] = r[k][wd];
            }
#pragma unroll
            for (int k = 0; k < 8; k++) s[k >> 1] += (uint32_t)__popcll(x[k] & mk) << (16 * (k & 1));
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            int v = (int)s[k];
            v += dpp32<0xb1, 0xf>(0, v);
            v += dpp32<0x4e, 0xf>(0, v);
            v += dpp32<0x141, 0xf>(0, v);
            v += dpp32<0x140, 0xf>(0, v);
            s[k] = (uint32_t)v;
        }
        // lane l takes row l & 7 of the group
        const int q = (c.lane >> 1) & 3;
        uint32_t t = q == 0 ? s[0] : q == 1 ? s[1] : q == 2 ? s[2] : s[3];
        t += (uint32_t)__shfl_xor((int)t, 16, WAVE);
        t += (uint32_t)__shfl_xor((int)t, 32, WAVE);
        const int v = (int)((c.lane & 1) ? t >> 16 : t & 0xFFFFu);
        if ((c.lane >> 3) == g) out = v;
    }
    return out;
}
constexpr int WIDE_SHARED_MIN = 48;  // row words from which rows are shared (below, most lanes have no word)

// A set of nl vertices, vertex k = at(k): counts by its rows, or by a mask of
// it when it has more than two vertices per row word (a lane then reads its own
// row, 64 rows at once, instead of the same words of one row).
template <class P, class At>
__device__ __attribute__((always_inline)) bool wide_set(Ctx& c, Wide<P>& z, int nl, At at) {
    const bool mask = z.ml && nl > 2 * z.rw;
    if (mask) {
        for (int w = c.lane; w < z.rw; w += WAVE) z.lmask[w] = 0;
        lsync();
        for (int k = c.lane; k < nl; k += WAVE) set_mask_bit(z.lmask, (int)at(k));
        lsync();
    }
    return mask;
}
template <class P, class At>
__device__ __attribute__((always_inline)) int wide_in_set(Ctx& c, Wide<P>& z, gptr<const uint64_t> X, bool mask, int nl,
                                                          At at, int id) {
    if (mask && P::slab && z.rl && z.rw >= WIDE_SHARED_MIN) return wide_rowpop_shared(c, X, z.rw, z.lmask, id);
    if (mask) return wide_rowpop(X, z.rw, z.lmask, id);
    int n = 0;
    for (int g = 0; g < nl; g += WAVE) {
        const int ids = g + c.lane < nl ? (int)at(g + c.lane) : 0;
        n += wide_count(X, z.rw, ids, min(nl - g, WAVE), id);
    }
    return n;
}

// |N n set| of places [0, n), place i's id = id_of(i), given to put(i, count).
// (A task in LDS keeps its registers for the branch loop: one chunk at a time.)
template <class P, class At, class Id, class Put>
__device__ __attribute__((always_inline)) void wide_counts(Ctx& c, Wide<P>& z, bool mask, int nl, At at, int n, Id id_of,
                                                           Put put) {
    if (mask || !P::slab) {
        for (int base = 0; base < n; base += WAVE) {
            const int i = base + c.lane;
            const int k = wide_in_set(c, z, z.A1, mask, nl, at, i < n ? id_of(i) : 0);
            if (i < n) put(i, k);
        }
        return;
    }
    for (int base = 0; base < n; base += 4 * WAVE) {
        int id[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = base + u * WAVE + c.lane;
            id[u] = i < n ? id_of(i) : 0;
        }
        int k[4] = {0, 0, 0, 0};
        for (int g = 0; g < nl; g += WAVE) {
            const int ids = g + c.lane < nl ? (int)at(g + c.lane) : 0;
            const int gn = min(nl - g, WAVE);
            if (n - base <= WAVE) {
                k[0] += wide_count(z.A1, z.rw, ids, gn, id[0]);
            } else {
                const Count4 q = wide_count4(z.A1, z.rw, ids, gn, id[0], id[1], id[2], id[3]);
                k[0] += q.n0;
                k[1] += q.n1;
                k[2] += q.n2;
                k[3] += q.n3;
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = base + u * WAVE + c.lane;
            if (i < n) put(i, k[u]);
        }
    }
}

// Keeps the candidates [m, m + n) valid under (z.tb, z.ub1), in place; the
// others go on the list (their positions) from nl on.  Returns how many stay.
template <class P>
__device__ __attribute__((always_inline)) int wide_keep(Ctx& c, Wide<P>& z, int m, int n, int& nl) {
    // (most children keep every candidate: the words are only read up to the
    // first that goes)
    int from = 0;
    for (; from < n; from += P::U * WAVE) {
        bool go = false;
#pragma unroll
        for (int u = 0; u < P::U; u++) {
            const int i = from + u * WAVE + c.lane;
            if (i < n) go |= !wide_valid<P>(c, z.tb, z.ub1, m, z.cw[m + i]);
        }
        if (ballot(go)) break;
    }
    if (from >= n) return n;
    int kept = from;
    for (int base = from; base < n; base += P::U * WAVE) {
        typename P::word w[P::U];
        uint32_t p[P::U];
#pragma unroll
        for (int u = 0; u < P::U; u++) {
            const int i = base + u * WAVE + c.lane;
            w[u] = i < n ? z.cw[m + i] : (typename P::word)0;
            p[u] = i < n ? (uint32_t)z.cpos[m + i] : 0u;
        }
        lsync();
#pragma unroll
        for (int u = 0; u < P::U; u++) {
            const int i = base + u * WAVE + c.lane;
            const bool in = i < n;
            const bool ok = in && wide_valid<P>(c, z.tb, z.ub1, m, w[u]);
            const uint64_t bo = ballot(ok), bx = ballot(in && !ok);
            if (ok) {
                const int d = m + kept + lanes_below(bo);
                z.cw[d] = w[u];
                z.cpos[d] = (typename P::pos_t)p[u];
            } else if (in) {
                z.list[nl + lanes_below(bx)] = (typename P::pos_t)p[u];
            }
            kept += __popcll(bo);
            nl += __popcll(bx);
        }
        lsync();
    }
    return kept;
}

// degree_pruning (main.cu:1735-1855): members [0, m), candidates [m, m + n),
// nl removed ones on the list.  True: the record fails (n is then meaningless).
// map_empty: the reference's id->position map holds no entry during this call
// (critical-vertex pruning without critical-adjacent candidates).  again: whether
// the same call on what it leaves could end otherwise (the last bounds counted
// fewer candidates than stay).
template <class P>
__device__ __attribute__((always_inline)) bool wide_prune(Ctx& c, Wide<P>& z, int m, int& n, int nl, bool map_empty, int& ub,
                                                          int& lb, int& med, bool& again) {
    int nc = n;
    bool sub = false;
    int tb0 = 0, ub0 = 0;
    for (;;) {
        ph_mark(c, PH_PRUNE);
        const bool fail = wide_bounds(c, z, m, n, nc, sub, tb0, ub0, ub, lb, med);
        ph_mark(c, PH_LU);
        if (fail) return true;
        again = nc != n;
        if (sub) nl = 0;
        n = wide_keep(c, z, m, n, nl);
        lsync();
        ph_mark(c, PH_COMPACT);
        if (n == 0 || nl == 0) return false;
        // degree update, main.cu:1775-1807: recomputed from the remaining
        // candidates when they are fewer than the removed ones, else lowered
        const bool rc = n < nl;
        const int k = rc ? n : nl;
        auto at = [&](int q) { return z.pid[rc ? z.cpos[m + q] : z.list[q]]; };
        long long sw = 0;
        for (int q = c.lane; q < k; q += WAVE) sw += z.d1r[at(q)];
        wadj_lanes(c, sw);
        const bool mask = map_empty ? false : wide_set(c, z, k, at);
        tb0 = z.tb;
        ub0 = z.ub1;
        sub = true;
        auto put = [&](int i, int k) {
            const typename P::word w = z.cw[i];
            z.cw[i] = P::set_ex(w, rc ? k : P::ex(w) - k);
        };
        if (!map_empty) {
            wide_counts(c, z, mask, k, at, m + n, [&](int i) { return (int)z.pid[z.cpos[i]]; }, put);
        } else if (rc) {
            for (int i = c.lane; i < m + n; i += WAVE) z.cw[i] = P::set_ex(z.cw[i], 0);
        }
        lsync();
        // indegrees of the candidates valid under the old bounds with the new
        // exdeg (main.cu:1811-1815)
        nc = 0;
        for (int base = 0; base < n; base += WAVE) {
            const int i = base + c.lane;
            nc += __popcll(ballot(i < n && wide_valid<P>(c, tb0, ub0, m, z.cw[m + (i < n ? i : 0)])));
        }
        lsync();
        ph_mark(c, PH_DEGUPD);
    }
}

// critical vertex pruning (main.cu:1526-1707) up to its closing degree pruning:
// 2 when the record fails, 1 when nothing changed (no critical-adjacent
// candidates), else 0 with the candidates, the list and map_empty as that pruning
// takes them.
template <class P>
__device__ __attribute__((always_inline)) int wide_critical(Ctx& c, Wide<P>& z, int& m, int& n, int& nl, int lb,
                                                            bool& map_empty) {
    using pos_t = typename P::pos_t;
    const int thr = wide_md(c, z, m + lb);
    int ncm = 0;
    long long sw = 0;
    for (int base = 0; base < m; base += WAVE) {
        const int i = base + c.lane;
        typename P::word w = 0;
        if (i < m) w = z.cw[i];
        const bool cr = i < m && P::in(w) + P::ex(w) == thr && P::ex(w) > 0;
        const uint64_t bc = ballot(cr);
        if (cr) {
            const pos_t p = z.cpos[i];
            z.list[ncm + lanes_below(bc)] = p;
            sw += z.d1r[z.pid[p]];
        }
        ncm += __popcll(bc);
    }
    nl = 0;
    map_empty = true;
    if (ncm == 0) return 1;
    wadj_lanes(c, sw);
    lsync();
    // critical-adjacent candidates, moved to the front of the candidates: the
    // ones beyond the first ncrit places change places with the others there
    auto crit = [&](int q) { return z.pid[z.list[q]]; };
    int ncrit = 0;
    const bool cmask = wide_set(c, z, ncm, crit);
    for (int base = 0; base < n; base += WAVE) {
        const int i = base + c.lane;
        const int id = i < n ? (int)z.pid[z.cpos[m + i]] : 0;
        const int k = wide_in_set(c, z, z.A1, cmask, ncm, crit, id);
        const uint64_t bf = ballot(i < n && k > 0);
        if (c.lane == 0) z.flag[base / WAVE] = bf;
        ncrit += __popcll(bf);
    }
    if (ncrit == 0) return 1;
    map_empty = false;
    lsync();
    int na = 0, nb = 0;
    const int half = z.T / 2;  // adjacent at ncrit or beyond: list[0 ..); not adjacent before it: list[half ..)
    for (int base = 0; base < n; base += WAVE) {
        const int i = base + c.lane;
        const bool f = (z.flag[base / WAVE] >> c.lane) & 1ull;
        const bool xa = f && i >= ncrit, xb = i < n && !f && i < ncrit;
        const uint64_t ba = ballot(xa), bb = ballot(xb);
        if (xa) z.list[na + lanes_below(ba)] = (pos_t)(m + i);
        if (xb) z.list[half + nb + lanes_below(bb)] = (pos_t)(m + i);
        na += __popcll(ba);
        nb += __popcll(bb);
    }
    lsync();
    for (int k = c.lane; k < na; k += WAVE) {  // (na == nb)
        const int i = z.list[k], j = z.list[half + k];
        const typename P::word wi = z.cw[i], wj = z.cw[j];
        const pos_t pi = z.cpos[i], pj = z.cpos[j];
        z.cw[i] = wj;
        z.cpos[i] = pj;
        z.cw[j] = wi;
        z.cpos[j] = pi;
    }
    lsync();
    auto at = [&](int q) { return z.pid[z.cpos[m + q]]; };
    sw = 0;
    for (int q = c.lane; q < ncrit; q += WAVE) {
        const uint32_t id = at(q);
        sw += z.d1r[id] + z.d2r[id];
    }
    wadj_lanes(c, sw);
    const bool mask = wide_set(c, z, ncrit, at);
    // degrees and 2-hop counts against the added vertices; candidates not
    // within 2 hops of all of them leave.  (The entries of the set itself,
    // [m, m + ncrit), stay where they are: later chunks read them.)
    bool bad = false;
    const int all = m + n, fixed = m + ncrit;
    int kept = 0;
    for (int base = 0; base < all; base += WAVE) {
        const int i = base + c.lane;
        const bool in = i < all;
        typename P::word w = 0;
        uint32_t p = 0;
        int id = 0;
        if (in) {
            w = z.cw[i];
            p = z.cpos[i];
            id = (int)z.pid[p];
        }
        const int x1 = wide_in_set(c, z, z.A1, mask, ncrit, at, id);
        const int x2 = wide_in_set(c, z, z.A2, mask, ncrit, at, id);
        w += (typename P::word)x1 * P::ADJ1;
        if (in && ((i < m && x2 != ncrit) || (i >= m && i < fixed && x2 < ncrit - 1))) bad = true;
        const bool cand = in && i >= fixed;
        const bool ok = cand && x2 == ncrit;
        const uint64_t bo = ballot(ok), bx = ballot(cand && !ok);
        lsync();
        if (in && i < fixed) z.cw[i] = w;
        if (ok) {
            const int d = fixed + kept + lanes_below(bo);
            z.cw[d] = w;
            z.cpos[d] = (pos_t)p;
        } else if (cand) {
            z.list[nl + lanes_below(bx)] = (pos_t)p;
        }
        kept += __popcll(bo);
        nl += __popcll(bx);
        lsync();
    }
    if (ballot(bad)) return 2;
    m = fixed;
    n = kept;
    return 0;
}

// a raw set of `len` vertices, id_at(i) the i-th one's root-local id
template <class At>
__device__ __attribute__((always_inline)) void wide_emit(Ctx& c, int len, At id_at) {
    unsigned long long ri = 0, si = 0;
    if (!clq_reserve(c, len, ri, si)) return;
    for (int k = c.lane; k < len; k += WAVE) c.a->clq_verts[si + k] = glob(c.g.p->orig)[id_at(k)];
    clq_ref(c, ri, si, len);
}

// Descending bitonic sort of n keys, any n: every comparator has the larger key
// to the lower index, so places from n on (the smallest possible key) would
// never move.  swap_if(lo, hi) exchanges the two places when out of order.
template <class F>
__device__ __forceinline__ void wide_sort(Ctx& c, int n, F swap_if) {
    int n2 = 1;
    while (n2 < n) n2 <<= 1;
    for (int k = 2; k <= n2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int x = c.lane; x < n2 / 2; x += WAVE) {
                const int lo = ((x & ~(j - 1)) << 1) | (x & (j - 1));
                const int hi = j == k >> 1 ? (lo ^ (k - 1)) : lo + j;
                if (hi < n) swap_if(lo, hi);
            }
            lsync();
        }
    }
}

// Descending radix sort of n 64-bit keys of `bits` bits in the slab: 8 bits a
// pass, counters of a digit in LDS (256 words), the lanes of a chunk that share
// a digit found by ballots.  Returns the array that holds the result.  For the
// slab's children (thousands of candidates) the bitonic sort's 78 and more
// passes over memory were most of the child: 2 ms for 3,000 candidates and 8
// for 13,900, against 0.1 and 0.6.
__device__ __attribute__((noinline)) gptr<uint64_t> wide_radix(gptr<uint64_t> src, gptr<uint64_t> dst, int n, int bits,
                                                               uint32_t* cnt) {
    constexpr int U = 4;
    const int lane = lane_id();
    for (int s = 0; s < bits; s += 8) {
        for (int k = lane; k < 256; k += WAVE) cnt[k] = 0;
        lsync();
        for (int base = 0; base < n; base += U * WAVE) {
            uint64_t key[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = base + u * WAVE + lane;
                key[u] = i < n ? src[i] : 0;
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (base + u * WAVE + lane < n) atomicAdd(&cnt[255 - (int)((key[u] >> s) & 255)], 1u);
        }
        lsync();
        {
            uint32_t v[4], t = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                v[k] = cnt[4 * lane + k];
                t += v[k];
            }
            uint32_t before = t;
            for (int d = 1; d < WAVE; d <<= 1) {
                const uint32_t o = __shfl_up(before, d, WAVE);
                if (lane >= d) before += o;
            }
            before -= t;
            lsync();
#pragma unroll
            for (int k = 0; k < 4; k++) {
                cnt[4 * lane + k] = before;
                before += v[k];
            }
        }
        lsync();
        for (int base = 0; base < n; base += U * WAVE) {
            uint64_t key[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = base + u * WAVE + lane;
                key[u] = i < n ? src[i] : 0;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (base + u * WAVE >= n) break;
                const bool in = base + u * WAVE + lane < n;
                const int d = 255 - (int)((key[u] >> s) & 255);
                uint64_t same = ballot(in);
#pragma unroll
                for (int b = 0; b < 8; b++) {
                    const bool bit = (d >> b) & 1;
                    const uint64_t bb = ballot(bit);
                    same &= bit ? bb : ~bb;
                }
                const int rank = lanes_below(same);
                uint32_t at = 0;
                if (in) at = cnt[d] + (uint32_t)rank;
                lsync();
                if (in && rank == 0) cnt[d] = at + (uint32_t)__popcll(same);
                lsync();
                if (in) dst[at] = key[u];
            }
        }
        lsync();
        const gptr<uint64_t> t = src;
        src = dst;
        dst = t;
    }
    return src;
}

// The child's record: members, then the candidates in Q order
// (main.cu:2059-2104: indeg, exdeg, lvl2adj, id, all descending).
template <class P>
__device__ __attribute__((always_inline)) void wide_child(Ctx& c, Wide<P>& z, int m, int n, int gap) {
    const ExpandArgs& a = *c.a;
    const int tc = m + n;
    if (!c.keys) {
        // outside the depth window: counted, never expanded
        if (c.lane == 0) {
            c.st->children++;
            c.st->sum_tw += tc;
            c.st->beyond++;
            if (a.trace_beyond && c.slot >= 0) atomicAdd(&a.trace_beyond[c.slot], 1u);
        }
        return;
    }
    const bool q = a.queue_mode != 0;
    const int s = (uint32_t)tc <= a.small_max ? 0 : 1;
    int bucket = 0;
    float feat[12];
    // cost order: children that fit the LDS tile take the lowest bucket
    // without the model (their subtrees are small, and on trees of tiny
    // tasks the features and the forward pass would cost as much as the task)
    const bool predict = q && a.n_buckets > 1 && (uint32_t)tc > a.cost_min_t;
    if (q && (a.trace_feat || predict)) {
        int mi = INT32_MAX, ma = INT32_MIN, me = INT32_MAX, mx = INT32_MIN;
        long long si = 0, se = 0, s2 = 0;
        for (int i = c.lane; i < tc; i += WAVE) {
            const typename P::word w = z.cw[i];
            const int in = P::in(w), ex = P::ex(w);
            mi = min(mi, in);
            ma = max(ma, in);
            me = min(me, ex);
            mx = max(mx, ex);
            si += in;
            se += ex;
            if (i >= m) s2 += z.d2r[z.pid[z.cpos[i]]];
        }
        feature_row(tc, m, (int)c.depth + 1, gap, mi, ma, me, mx, si, se, s2, feat);
    }
    if (predict) bucket = cost_bucket(c, feat);
    unsigned long long ri = 0, si = 0;
    ph_mark(c, PH_CHILD);
    if (c.lane == 0) {
        if (q) {
            si = pool_alloc(c, (uint32_t)tc);
        } else {
            ri = atomicAdd(&a.out_ctr[s].items, 1ull);
            si = atomicAdd(&a.out_ctr[s].slots, (unsigned long long)tc);
        }
    }
    ri = rdlane64(ri, 0);
    si = rdlane64(si, 0);
    if (q ? si == ~0ull : (ri >= a.out_ref_cap[s] || si + tc > a.out_vert_cap[s])) {
        if (c.lane == 0) atomicOr(a.error, 1);
        return;
    }
    gptr<Vrec> dst = globw((q ? a.pool : a.out_verts[s]) + si);
    auto put = [&](int i, uint32_t id, int label, typename P::word w) {
        typedef int v4 __attribute__((ext_vector_type(4)));
        *(gptr<v4>)(dst + i) = v4{(int)id, label, P::in(w), P::ex(w)};
    };
    for (int i = c.lane; i < m; i += WAVE) put(i, z.pid[z.cpos[i]], 1, z.cw[i]);
    unsigned long long bnd = 0;
    // slot bound of the child's own children (see TaskRef); past the depth
    // window they are not written
    const bool kids = c.a->all_bounds || !(c.g.max_depth >= 0 && (int)c.depth + 2 > c.g.max_depth);
    auto bound_of = [&](uint32_t id) {
        if (!kids) return 0ull;
        const unsigned long long x = (unsigned long long)z.d2r[id] + m + 1;
        return x < (unsigned long long)tc ? x : (unsigned long long)tc;
    };
    lsync();
    if constexpr (!P::slab) {
        // keys in the words' place: from the top down a chunk's keys only cover
        // words that have been read, when the candidates start at word 0
        if (m > WAVE) {
            for (int base = 0; base < n; base += WAVE) {
                const int i = base + c.lane;
                uint32_t w = 0;
                if (i < n) w = z.cw[m + i];
                lsync();
                if (i < n) z.cw[i] = w;
                lsync();
            }
        }
        const int w0 = m > WAVE ? 0 : m;
        for (int base = (n - 1) & ~(WAVE - 1); base >= 0; base -= WAVE) {
            const int i = base + c.lane;
            uint64_t key = 0;
            if (i < n) {
                const uint32_t w = z.cw[w0 + i], p = z.cpos[m + i];
                const uint32_t id = z.pid[p];
                key = ((uint64_t)w << 32) | ((uint32_t)z.pl2[p] << z.idb) | id;
                if (!q) bnd += bound_of(id);
            }
            lsync();
            if (i < n) z.keys[i] = key;
            lsync();
        }
        wide_sort(c, n, [&](int lo, int hi) {
            const uint64_t u = z.keys[lo], v = z.keys[hi];
            if (u < v) {
                z.keys[lo] = v;
                z.keys[hi] = u;
            }
        });
        for (int i = c.lane; i < n; i += WAVE) {
            const uint64_t key = z.keys[i];
            put(m + i, (uint32_t)key & ((1u << z.idb) - 1u), 0, (uint32_t)(key >> 32));
        }
    } else {
        // Many candidates: indeg and exdeg above their smallest values, lvl2adj
        // and id in 64 bits.  Few, or values that need more bits: 128-bit keys
        // (word, lvl2adj and id), in LDS when they fit there.  (Up to two chunks
        // the bitonic sort has 28 passes in LDS, the radix sort 5 of several
        // trips to the slab.)
        const int rb = 32 - __builtin_clz((uint32_t)c.g.p->R);
        int in0 = 0, ex0 = 0, eb = 0, bits = 64;
        if (n > 2 * WAVE && z.spare_bytes >= 1024u) {
            int il = INT32_MAX, ih = 0, el = INT32_MAX, eh = INT32_MIN;
            for (int i = c.lane; i < n; i += WAVE) {
                const typename P::word w = z.cw[m + i];
                il = min(il, P::in(w));
                ih = max(ih, P::in(w));
                el = min(el, P::ex(w));
                eh = max(eh, P::ex(w));
            }
            in0 = wave_min(il);
            ex0 = wave_min(el);
            const uint32_t ir = (uint32_t)(wave_max(ih) - in0), er = (uint32_t)(wave_max(eh) - ex0);
            eb = er ? 32 - __builtin_clz(er) : 0;
            bits = (ir ? 32 - __builtin_clz(ir) : 0) + eb + 2 * rb;
        }
        if (bits < 64) {
            for (int i = c.lane; i < n; i += WAVE) {
                const uint32_t p = z.cpos[m + i], id = z.pid[p];
                const typename P::word w = z.cw[m + i];
                z.keys[i] = ((uint64_t)(uint32_t)(P::in(w) - in0) << (eb + 2 * rb)) |
                            ((uint64_t)(uint32_t)(P::ex(w) - ex0) << (2 * rb)) | ((uint64_t)z.pl2[p] << rb) | id;
                if (!q) bnd += bound_of(id);
            }
            lsync();
            const gptr<uint64_t> k = wide_radix(z.keys, z.keys + (size_t)z.T, n, bits, (uint32_t*)z.spare);
            for (int i = c.lane; i < n; i += WAVE) {
                const uint64_t key = k[i];
                const int ex = (int)((key >> (2 * rb)) & ((1ull << eb) - 1ull));
                put(m + i, (uint32_t)(key & ((1ull << rb) - 1ull)), 0,
                    P::make((int)(key >> (eb + 2 * rb)) + in0, ex + ex0));
            }
        }
        auto run = [&](auto khi, auto klo) {
            for (int i = c.lane; i < n; i += WAVE) {
                const uint32_t p = z.cpos[m + i], id = z.pid[p];
                khi[i] = z.cw[m + i];
                klo[i] = ((uint64_t)z.pl2[p] << 32) | id;
                if (!q) bnd += bound_of(id);
            }
            lsync();
            wide_sort(c, n, [&](int lo, int hi) {
                const uint64_t uh = khi[lo], vh = khi[hi], ul = klo[lo], vl = klo[hi];
                if (uh < vh || (uh == vh && ul < vl)) {
                    khi[lo] = vh;
                    khi[hi] = uh;
                    klo[lo] = vl;
                    klo[hi] = ul;
                }
            });
            for (int i = c.lane; i < n; i += WAVE) put(m + i, (uint32_t)klo[i], 0, khi[i]);
        };
        if (bits < 64)
            ;
        else if (16u * (uint32_t)n <= z.spare_bytes)
            run((uint64_t*)z.spare, (uint64_t*)z.spare + n);
        else
            run(z.keys, z.keys + (size_t)z.T);
    }
    TaskRef r;
    r.off = si;
    r.t = (uint32_t)tc;
    r.depth = (uint16_t)(c.depth + 1);
    r.inst = (uint16_t)c.inst;
    r.bound = 0;
    r.b0 = 0;
    r.b1 = 0;
    if (q) {
        // dynamic order: children stay on this wave's stack (depth first),
        // with their predicted bucket when a cost model orders the work;
        // static order: the stack only stages them, and the wave moves them
        // to the ring (whose positions are dealt to the waves in turn) in
        // one claim when the task ends
        const bool shared = !a.use_priv || (!a.static_sched && share_child(c));
        const bool pushed = push_ref(c, r, bucket, shared, feat);
        ph_mark(c, PH_POOL);
        if (!pushed) return;
    } else {
        bnd = (unsigned long long)wave_sum64((long long)bnd);
        if (c.lane == 0) {
            r.bound = bnd;
            a.out_refs[s][ri] = r;
        }
    }
    if (c.lane == 0) {
        c.st->children++;
        c.st->sum_tw += tc;
    }
}

// exdeg of positions [0, keep) minus their neighbours among positions
// [keep, keep + nr): several removals at once
template <class P>
__device__ __attribute__((always_inline)) void wide_bulk_remove(Ctx& c, Wide<P>& z, int keep, int nr) {
    if (nr <= 0) return;
    auto gone = [&](int q) { return z.pid[keep + q]; };
    const bool mask = wide_set(c, z, nr, gone);
    wide_counts(c, z, mask, nr, gone, keep, [&](int i) { return (int)z.pid[i]; },
                [&](int i, int k) { z.pw[i] -= (typename P::word)k; });
    lsync();
}

// W_adj of a removal that fails: the reference scans N(r) in ascending id
// order and stops after the first failing member (main.cu:1437-1450)
template <class P>
__device__ __attribute__((always_inline)) void wide_failed_scan(Ctx& c, Wide<P>& z, int rid, int fid) {
    const size_t r0 = (size_t)rid * z.rw;
    int rank = 0;
    for (int wd = c.lane; wd <= (fid >> 6); wd += WAVE) {
        uint64_t x = z.A1[r0 + wd];
        if (wd == (fid >> 6)) x &= (1ull << (fid & 63)) - 1ull;
        rank += __popcll(x);
    }
    wadj_lanes(c, rank + (c.lane == 0));
}

// Split step of a task whose branches [bbeg, bend) go to several waves: finds
// the first failing removal, counts the removals' scans, stores the record as
// it stands before the first branch of the window (with lvl2adj) and pushes
// the items, ch branches each on average.
template <class P>
__device__ __attribute__((always_inline)) void wide_split(Ctx& c, Wide<P>& z, const TaskRef& ref, int nm, int bbeg, int bend,
                                                          int ch) {
    const ExpandArgs& a = *c.a;
    const int t0 = (int)ref.t;
    // Removal k (branch b = k) takes position t0 - k.  Member i fails at
    // the removal of its need_i-th neighbour counted from the end, with
    // need_i = max(pin + pex - mindeg(nm) + 1, 1); kb = the first such
    // removal over all members (bend: none before the window's end).
    const int mdg = get_mindeg(c, nm);
    int kb = bend;
    for (int i = 0; i < nm; i++) {
        const typename P::word w = z.pw[i];
        const int need = max(P::in(w) + P::ex(w) - mdg + 1, 1);
        const size_t r0 = (size_t)z.pid[i] * z.rw;
        // removals up to kb inclusive: a member failing at the same
        // removal as an earlier one must be seen (smallest failing id)
        const int lim = min(kb, bend - 1);
        int cnt = 0, ki = INT32_MAX;
        for (int k0 = 1; k0 <= lim && ki == INT32_MAX; k0 += WAVE) {
            const int k = k0 + c.lane;
            bool adj = false;
            if (k <= lim) {
                const uint32_t id = z.pid[t0 - k];
                adj = (z.A1[r0 + (id >> 6)] >> (id & 63)) & 1ull;
            }
            const uint64_t bm = ballot(adj);
            const int pc = __popcll(bm);
            if (cnt + pc >= need) {
                const uint64_t hit = ballot(adj && cnt + lanes_below(bm) + 1 == need);
                ki = k0 + __builtin_ctzll(hit);
            }
            cnt += pc;
        }
        if (c.lane == 0) z.list[i] = (typename P::pos_t)min(ki, bend);  // (bend: none)
        kb = min(kb, ki);
    }
    lsync();
    // W_adj of the removals: full scans of N(r) for removals 1..kb-1,
    // the partial scan up to the smallest failing member for removal kb
    long long sw = 0;
    for (int k = 1 + c.lane; k < kb; k += WAVE) sw += z.d1r[z.pid[t0 - k]];
    wadj_lanes(c, sw);
    if (kb < bend) {
        int fid = INT32_MAX;
        for (int i = c.lane; i < nm; i += WAVE)
            if ((int)z.list[i] == kb) fid = min(fid, (int)z.pid[i]);
        wide_failed_scan(c, z, (int)z.pid[t0 - kb], wave_min(fid));
    }
    const int hi = min(kb, bend);
    if (hi <= bbeg) return;
    // removals 1..bbeg happen before the window: apply them once here
    const int pre = bbeg;
    const int ts = t0 - pre;
    wide_bulk_remove(c, z, ts, pre);
    // the record plus, in the pool, one Vrec after it whose id counts the items
    // still to run (the last one frees the block); the level-synchronous form
    // writes it to the stream of large tasks, every item a ref to it
    const bool q = a.queue_mode != 0;
    const int n_items = (hi - bbeg + ch - 1) / ch;
    unsigned long long slot = 0, ri = 0;
    if (c.lane == 0) {
        if (q) {
            slot = pool_alloc(c, (uint32_t)ts + 1u);
        } else {
            ri = atomicAdd(&a.out_ctr[1].items, (unsigned long long)n_items);
            slot = atomicAdd(&a.out_ctr[1].slots, (unsigned long long)ts);
        }
    }
    slot = rdlane64(slot, 0);
    ri = rdlane64(ri, 0);
    if (q ? slot == ~0ull : (ri + n_items > a.out_ref_cap[1] || slot + ts > a.out_vert_cap[1])) {
        if (c.lane == 0) atomicOr(a.error, 1);
        return;
    }
    Vrec* dst = (q ? a.pool : a.out_verts[1]) + slot;
    for (int i = c.lane; i < ts; i += WAVE) {
        const typename P::word w = z.pw[i];
        dst[i] = Vrec{(int32_t)z.pid[i], (i < nm ? 1 : 0) | ((int32_t)z.pl2[i] << 4), P::in(w), P::ex(w)};
    }
    if (q && c.lane == 0) dst[ts] = Vrec{n_items, 0, 0, 0};
    // item boundaries balance the work rather than the branch count:
    // branch b builds a child from about t0 - b vertices, so with
    // S(b) = sum of (t0 - x) over x in [bbeg, b), boundary j is the first
    // b with S(b) >= j S(hi) / n_items (kept strictly increasing).  At the
    // window's last level the children are not written, and a branch costs about
    // the same wherever it starts: items of equal counts (first branches of
    // a power-law graph 133 -> 125 ms; with equal counts on every level a
    // cost-ordered co-expression window took 19.5 ms instead of 17.0).
    const long long t0l = t0;
    const long long fall = c.keys ? 1 : 0;
    auto S = [&](long long b) { return (b - bbeg) * t0l - fall * ((b * (b - 1) - (long long)bbeg * (bbeg - 1)) / 2); };
    const long long s_tot = S(hi);
    auto boundary = [&](int j) -> int {
        if (j <= 0) return bbeg;
        if (j >= n_items) return hi;
        const long long target = s_tot * j / n_items;
        int lo = bbeg, up = hi;
        while (lo < up) {
            const int mid = (lo + up) >> 1;
            if (S(mid) >= target)
                up = mid;
            else
                lo = mid + 1;
        }
        return min(max(lo, bbeg + j), hi - (n_items - j));
    };
    auto item_ref = [&](int j) {
        TaskRef r;
        r.off = slot;
        r.t = (uint32_t)ts;
        r.depth = ref.depth;
        r.inst = ref.inst;
        r.bound = (uint64_t)c.slot;  // the task the item belongs to (trace)
        r.b0 = (uint32_t)(boundary(j) - pre);
        r.b1 = (uint32_t)(boundary(j + 1) - pre);
        return r;
    };
    if (!q) {
        for (int j = c.lane; j < n_items; j += WAVE) {
            TaskRef r = item_ref(j);
            r.bound = 0;
            if (c.keys)  // (the slots its children can take)
                for (uint32_t b = r.b0; b < r.b1; b++)
                    r.bound += (uint64_t)min((long long)z.d2r[z.pid[ts - 1 - (int)b]] + nm + 1, (long long)ts);
            a.out_refs[1][ri + j] = r;
        }
        return;
    }
    // the items go to the rings in chunks of up to 64 claimed at once
    // (lanes write the refs, one release fence per chunk), as many as wait at a
    // ring, the rest to this wave's own; what the rings cannot take stays on
    // this wave's stack
    int done = 0;
    while (done < n_items) {
        unsigned long long pos = 0;
        int waiting = 0;
        const int rg = ring_for(c, &waiting);
        const int want = min(n_items - done, waiting > 0 ? min(waiting, WAVE) : WAVE);
        const int k = a.trace_feat ? ring_claim_trace(c, want, &pos) : ring_claim(c, rg, want, &pos);
        if (k == 0) break;
        if (c.lane == 0)
            __hip_atomic_fetch_add(a.pending, (unsigned long long)k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (c.lane < k) {
            const unsigned long long gi = (unsigned long long)rg * a.q_cap + (pos + c.lane) % a.q_cap;
            if (a.trace_parent) a.trace_parent[gi] = -2;
            a.q_refs[gi] = item_ref(done + c.lane);
        }
        ring_publish(c, rg, pos, k);
        done += k;
    }
    for (; done < n_items; done++)
        if (!push_ref(c, item_ref(done), a.n_buckets - 1, false, nullptr)) break;
}

// One task or split item.  False, with nothing done, when a degree or lvl2adj
// does not fit WideLds' fields (WideSlab then runs it; its own are never
// exceeded).  The caller has checked wide_fits (WideLds) or the slab's size.
// CUT: a root may be one that a window shortened (not where the whole root fits
// the LDS, whose counts fit the fields: 43 registers in memory there, 51 with
// the check).
template <class P, bool CUT = true>
__device__ __attribute__((always_inline)) bool process_wide(Ctx& c, const TaskRef ref, char* lds, uint32_t lds_bytes,
                                                            char* slab) {
    const ExpandArgs& a = *c.a;
    const int t0 = (int)ref.t;
    const bool item = ref.b1 > 0;
    const bool root = ref.depth == 0;
    Wide<P> z;
    z.rw = c.g.p->rw;
    const uint32_t T = wide_T((uint32_t)t0);
    z.T = (int)T;
    z.rl = wide_rows_staged((uint32_t)z.rw, lds_bytes);
    z.idb = c.g.p->R <= 65536 ? 16 : 20;
    {
        char* at = lds;
        z.row1 = (uint64_t*)at;
        z.row2 = z.row1 + z.rw;
        z.lmask = z.row2 + z.rw;
        if (z.rl) at += 24 * z.rw;
        if constexpr (!P::slab) {
            z.keys = (uint64_t*)at;
            z.cw = (uint32_t*)at;
            z.list = (uint16_t*)(at + 4 * T);
            z.tab = (uint16_t*)(at + 6 * T);
            at += 8 * T;
            z.pid = (uint32_t*)at;
            at += 4 * T;
            z.pw = (uint32_t*)at;
            at += 4 * T;
            z.pl2 = (uint16_t*)at;
            at += 2 * T;
            z.cpos = (uint16_t*)at;
            at += 2 * T;
            z.nbits = (uint64_t*)at;
            z.flag = z.nbits + T / 64;
        } else {
            // (52 bytes a vertex, WideMid: 34)
            gptr<char> g = globw(slab);
            z.keys = (gptr<uint64_t>)g;
            z.pw = (typename P::wordp)(z.keys + (size_t)2 * T);
            if constexpr (P::cw_lds) {
                z.cw = (uint32_t*)at;
                at += 4 * T;
            } else {
                z.cw = z.pw + (size_t)T;
            }
            typename P::posp u = (typename P::posp)(z.pw + (size_t)2 * T);
            z.pid = u;
            z.pl2 = u + (size_t)T;
            z.cpos = u + (size_t)2 * T;
            z.list = u + (size_t)3 * T;
            z.tab = u + (size_t)4 * T;
            if ((uint32_t)(at - lds) + T / 4 <= lds_bytes) {
                z.nbits = (uint64_t*)at;
                at += T / 4;
            } else {
                z.nbits = (uint64_t*)(slab + (size_t)52 * T);
            }
            z.flag = z.nbits + T / 64;
        }
        z.spare = at;
        z.spare_bytes = lds_bytes - (uint32_t)(at - lds);
        // rows too long to be staged can still have the mask (a batch's root of
        // 17,193 vertices took 7.3 ms to apply its window's removals row by row)
        z.ml = z.rl || 8u * (uint32_t)z.rw <= z.spare_bytes;
        if (!z.rl) z.lmask = (uint64_t*)z.spare;
    }
    // ---- record ----
    bool bad = false;
    int nm = 0, cov = 0;
    gptr<const Vrec> src = glob(a.in_verts + ref.off);
    // lvl2adj has to fit its field: an item brings it with its record, a root
    // that a window shortened takes the whole root's (below), more than its own
    // vertices
    const uint32_t l2_max = sizeof(typename P::pos_t) == 4 ? 0xFFFFFFFFu : P::slab || z.idb == 16 ? 0xFFFFu : 0xFFFu;
    if (CUT && root && !item && (uint32_t)c.g.p->max_d2r > l2_max) return false;
    for (int base = 0; base < t0; base += P::U * WAVE) {
        typedef int v4 __attribute__((ext_vector_type(4)));
        v4 v[P::U];
#pragma unroll
        for (int u = 0; u < P::U; u++) {
            const int i = base + u * WAVE + c.lane;
            v[u] = v4{0, 0, 0, 0};
            if (i < t0) v[u] = *(gptr<const v4>)(src + i);
        }
#pragma unroll
        for (int u = 0; u < P::U; u++) {
            const int i = base + u * WAVE + c.lane;
            const bool in = i < t0;
            const int lab = item ? v[u].y & 15 : v[u].y;
            const uint32_t l2 = item ? (uint32_t)v[u].y >> 4 : 0u;
            if (v[u].w < -P::LIMIT || v[u].w > P::LIMIT || l2 > l2_max) bad = true;
            nm += __popcll(ballot(in && lab == 1));
            cov += __popcll(ballot(in && lab == 2));
            if (in) {
                z.pid[i] = (uint32_t)v[u].x;
                z.pw[i] = P::make(v[u].z, v[u].w);
                z.pl2[i] = (typename P::pos_t)l2;
            }
        }
    }
    if (ballot(bad)) return false;
    int nc = t0 - nm;
    const int nb = nc - cov;
    int bend = nb;
    if (root && c.g.p->root_b1 >= 0 && c.g.p->root_b1 < bend) bend = (int)c.g.p->root_b1;
    // a negative window start counts from the end of the root's branches
    const long long rb0 = c.g.p->root_b0 >= 0 ? c.g.p->root_b0 : max(0ll, (long long)nb + c.g.p->root_b0);
    const int bbeg = root ? (int)min<long long>(rb0, (long long)nb) : 0;
    c.depth = ref.depth;
    c.keys = !(c.g.max_depth >= 0 && (int)c.depth + 1 > c.g.max_depth);
    if (!item && c.lane == 0) {  // (a split item's task is counted by its prepare step)
        c.st->tasks++;
        c.st->sum_t += t0;
        if ((uint32_t)t0 > a.small_max) c.st->large++;
    }
    z.A1 = glob(c.g.p->A1);
    z.A2 = glob(c.g.p->A2);
    z.d1r = glob(c.g.p->d1r);
    z.d2r = glob(c.g.p->d2r);
    z.mdt = md(c, c.lane);
    z.mds = uni(md(c, c.g.min_size));
    z.ubt = ub_quot(c, c.lane);
    lsync();
    ph_mark(c, PH_LOAD);

    // ---- lookahead, main.cu:1349-1405 ----
    if (!item) {
        const int req = wide_md(c, z, t0);
        bool f = false;
        for (int i = c.lane; i < nm; i += WAVE) {
            const typename P::word w = z.pw[i];
            if (P::in(w) + P::ex(w) < req) f = true;
        }
        if (ballot(f) == 0) {
            // a record holding every root vertex and no member is the whole
            // root: |N2(v) n candidates| is then |N2(v) n root| = d2r[v],
            // with no row scans.  A root shortened by a window's leading
            // removals (root_cut) takes the whole root's values too: its
            // lookahead ran on the whole root, where it failed (the host
            // checked), so nothing is emitted
            const bool cut_root = nm == 0 && root && c.g.p->root_cut > 0;
            const bool whole_root = nm == 0 && (t0 == c.g.p->R || cut_root);
            auto cand = [&](int q) { return z.pid[nm + q]; };
            const bool mask = whole_root ? false : wide_set(c, z, nc, cand);
            long long sw = 0;
            bool low = false, known = false;
            // (from the end of the record, where the degrees are lowest: when
            // the children are not kept, lvl2adj only serves this test)
            for (int base = nm + ((nc - 1) & ~(WAVE - 1)); base >= nm; base -= WAVE) {
                const int i = base + c.lane;
                const int id = i < t0 ? (int)z.pid[i] : 0;
                const int d2 = i < t0 ? z.d2r[id] : 0;
                sw += d2;
                if (known) continue;
                const int l2 = whole_root ? d2 : wide_in_set(c, z, z.A2, mask, nc, cand, id);
                if (i < t0) {
                    const typename P::word w = z.pw[i];
                    z.pl2[i] = (typename P::pos_t)l2;
                    if (l2 < nc - 1 || P::in(w) + P::ex(w) < req) low = true;
                }
                known = !c.keys && ballot(low) != 0;
            }
            wadj_lanes(c, sw);
            lsync();
            if (ballot(low) == 0 && !cut_root) {
                wide_emit(c, t0, [&](int i) { return z.pid[i]; });
                ph_mark(c, PH_LOOKAHEAD);
                return true;
            }
        }
    }
    ph_mark(c, PH_LOOKAHEAD);

    // ---- branch loop, main.cu:1094-1180 ----
    // Branch ordinal b takes position t0 - 1 - b.  Branch b >= 1 first removes
    // the vertex of the branch before; a failing member ends the loop.
    int tp = t0;
    int b_lo = 0, b_hi = bend;
    if (item) {
        // removals 1..b0 at once (the prepare step found no failure before
        // the item's range); b0 and b1 count from the record it stored
        b_lo = (int)ref.b0;
        b_hi = (int)ref.b1;
        tp = t0 - b_lo;
        nc -= b_lo;
        wide_bulk_remove(c, z, tp, b_lo);
        ph_mark(c, PH_REMOVE);
    } else {
        // a root's branches are split finer, to about one item per resident
        // wave over all roots: until the roots' items produce children nothing
        // else can run
        int ch = a.split_chunk;
        if (root && ch > 0 && a.n_roots > 0) {
            const long long want = ((long long)(bend - bbeg) * a.n_roots + a.split_waves - 1) / a.split_waves;
            ch = (int)max(1ll, min((long long)ch, want));
        } else if (ch > SPLIT_FINE && a.queue_mode && !a.static_sched) {
            // other tasks too when more waves wait than the rings hold tasks
            // for: a first-level task of 13,900 vertices whose 162-branch items
            // made 162 large children each kept the other waves waiting (its
            // window 365 -> 190 ms with the sort of the slab's children, a
            // co-expression window 76 -> 57).  Not in the static order, which
            // deals items to waves in turn, waiting or not (9 -> 19 ms).
            unsigned long long ph = 0;
            if (c.lane == 0) ph = __hip_atomic_load(a.pending, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ph = rdlane64(ph, 0);
            const long long hg = (long long)(ph >> 32), pd = (long long)(ph & 0xFFFFFFFFull);
            const long long waiting = pd - ((long long)gridDim.x - hg);
            const long long need = hg - (waiting > 0 ? waiting : 0);
            if (need > 0) ch = (int)max((long long)SPLIT_FINE, min((long long)ch, (long long)(bend - bbeg) / need));
        }
        if (ch > 0 && (uint32_t)t0 > a.split_min_t && bend - bbeg > ch) {
            wide_split(c, z, ref, nm, bbeg, bend, ch);
            ph_mark(c, PH_PREPARE);
            return true;
        }
        if (bbeg > 0 && bbeg < bend) {
            // a window that starts at branch bbeg: removals 1..bbeg at once
            // (the root has no members: none of them can fail)
            long long sw = 0;
            for (int k = 1 + c.lane; k <= bbeg; k += WAVE) sw += z.d1r[z.pid[t0 - k]];
            wadj_lanes(c, sw);
            b_lo = bbeg;
            tp = t0 - bbeg;
            nc -= bbeg;
            wide_bulk_remove(c, z, tp, bbeg);
            ph_mark(c, PH_REMOVE);
        } else if (bbeg > 0) {
            // an empty window: the removals before it are counted as the
            // reference makes them, up to the window's end
            long long sw = 0;
            for (int k = 1 + c.lane; k < bend; k += WAVE) sw += z.d1r[z.pid[t0 - k]];
            wadj_lanes(c, sw);
            return true;
        }
    }
    const int ms = c.g.min_size;
    const int mdg = nm < ms ? z.mds : wide_md(c, z, nm);  // get_mindeg(nm)
    // rows of the next branch vertex, in registers until its branch starts
    constexpr int NJ = WIDE_ROW_WORDS / WAVE;
    uint64_t n1[NJ], n2[NJ];
    int nd1 = 0, nd2 = 0;  // its |N n root|, |N2 n root|
    auto fetch = [&](int p) {
        const int id = uni((int)z.pid[p]);
        nd1 = z.d1r[id];
        nd2 = z.d2r[id];
        if (!z.rl) return;
        const size_t r0 = (size_t)id * z.rw;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int wd = j * WAVE + c.lane;
            n1[j] = 0;
            n2[j] = 0;
            if (wd < z.rw) {
                n1[j] = z.A1[r0 + wd];
                n2[j] = z.A2[r0 + wd];
            }
        }
    };
    if (b_lo < b_hi) fetch(tp - 1);
    int d1v = 0;
    for (int b = b_lo; b < b_hi; b++) {
        const bool pend = b > b_lo;
        if (pend) {
            // remove_one_vertex (main.cu:1408-1462) for the last branch's
            // vertex: the members here, the candidates with the child's build
            nc--;
            tp--;
            bool fail = false;
            int fid = INT32_MAX;
            for (int i = c.lane; i < nm; i += WAVE) {
                if ((z.nbits[i >> 6] >> (i & 63)) & 1ull) {
                    const typename P::word w = z.pw[i] - 1u;
                    z.pw[i] = w;
                    if (P::in(w) + P::ex(w) < mdg) {
                        fail = true;
                        fid = min(fid, (int)z.pid[i]);
                    }
                }
            }
            if (ballot(fail)) {
                if (!item) wide_failed_scan(c, z, uni((int)z.pid[tp]), wave_min(fid));
                break;
            }
            if (!item) wadj_add(c, d1v);
            ph_mark(c, PH_REMOVE);
        }
        const int vsrc = tp - 1;
        const int vid = uni((int)z.pid[vsrc]);
        d1v = nd1;
        wadj_add(c, (long long)nd1 + nd2);
        if (z.rl) {
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int wd = j * WAVE + c.lane;
                if (wd < z.rw) {
                    z.row1[wd] = n1[j];
                    z.row2[wd] = n2[j];
                }
            }
        }
        lsync();
        if (b + 1 < b_hi) fetch(vsrc - 1);
        if (c.lane == 0) c.st->branches++;
        // the child: members, the branch vertex, then the candidates inside
        // N2(v) with their degrees updated (add_one_vertex, main.cu:1465-1523,
        // diameter pruning, main.cu:1709-1732); the others go on the list
        int m = nm + 1, n = 0, nl = 0;
        if (c.lane == 0) {
            typename P::word w = z.pw[vsrc];
            if (pend) w -= (uint32_t)(z.nbits[vsrc >> 6] >> (vsrc & 63)) & 1u;
            z.cw[nm] = w;
            z.cpos[nm] = (typename P::pos_t)vsrc;
        }
        const size_t r0 = (size_t)vid * z.rw;
        lsync();
        for (int base = 0; base < vsrc; base += P::U * WAVE) {
            uint32_t id[P::U];
            typename P::word w[P::U];
            uint64_t x1[P::U], x2[P::U], ob[P::U];
#pragma unroll
            for (int u = 0; u < P::U; u++) {
                const int i = base + u * WAVE + c.lane;
                id[u] = i < vsrc ? z.pid[i] : 0u;
                w[u] = i < vsrc ? z.pw[i] : (typename P::word)0;
                ob[u] = pend && base + u * WAVE < vsrc ? z.nbits[base / WAVE + u] : 0ull;
            }
#pragma unroll
            for (int u = 0; u < P::U; u++) {
                if (z.rl) {
                    x1[u] = z.row1[id[u] >> 6];
                    x2[u] = z.row2[id[u] >> 6];
                } else {
                    x1[u] = z.A1[r0 + (id[u] >> 6)];
                    x2[u] = z.A2[r0 + (id[u] >> 6)];
                }
            }
            lsync();
#pragma unroll
            for (int u = 0; u < P::U; u++) {
                const int i = base + u * WAVE + c.lane;
                if (base + u * WAVE >= vsrc) break;
                const bool in = i < vsrc, cand = in && i >= nm;
                const uint32_t a1 = (uint32_t)(x1[u] >> (id[u] & 63)) & 1u;
                const uint32_t a2 = (uint32_t)(x2[u] >> (id[u] & 63)) & 1u;
                const uint32_t o = (uint32_t)(ob[u] >> c.lane) & 1u;
                if (cand && o) {
                    w[u] -= 1u;
                    z.pw[i] = w[u];
                }
                const uint64_t bm = ballot(in && a1);
                if (c.lane == 0) z.nbits[base / WAVE + u] = bm;
                const typename P::word wc = w[u] + (a1 ? P::ADJ1 : (typename P::word)0);
                const bool ok = cand && a2;
                const uint64_t bo = ballot(ok), bx = ballot(cand && !a2);
                if (ok || (in && i < nm)) {
                    const int d = ok ? m + n + lanes_below(bo) : i;
                    z.cw[d] = wc;
                    z.cpos[d] = (typename P::pos_t)i;
                }
                if (bx) {
                    if (cand && !a2) z.list[nl + lanes_below(bx)] = (typename P::pos_t)i;
                    nl += __popcll(bx);
                }
                n += __popcll(bo);
            }
            lsync();
        }
        ph_mark(c, PH_ADD);
        int ub = 0, lb = 0, med = 0;
        // degree pruning, then critical-vertex pruning, which ends in a
        // second degree pruning
        bool first = true, map_empty = false, fails, again = true;
        for (;;) {
            fails = wide_prune(c, z, m, n, nl, map_empty, ub, lb, med, again);
            if (!first || fails) break;
            first = false;
            const int cr = wide_critical(c, z, m, n, nl, lb, map_empty);
            if (cr == 2) {
                m = -1;  // neither a clique test nor a child
                break;
            }
            ph_mark(c, PH_CRIT);
            // (most children: the closing degree pruning would end as the first
            // one did, on the same degrees; with it the bounds were 37% of a
            // co-expression window's time)
            if (cr == 1 && !again) break;
        }
        if (m < 0) {
            ph_mark(c, PH_CRIT);
            continue;
        }
        if (m >= ms) {
            // clique test, main.cu:1974-1995
            const int req = wide_md(c, z, m);
            bool low = false;
            for (int i = c.lane; i < m; i += WAVE) low |= P::in(z.cw[i]) < req;
            if (ballot(low) == 0) wide_emit(c, m, [&](int i) { return z.pid[z.cpos[i]]; });
        }
        ph_mark(c, PH_PRUNE);
        if (!fails && n > 0) wide_child(c, z, m, n, ub - lb);
        lsync();
        ph_mark(c, PH_CHILD);
    }
    return true;
}

// whether a task of t vertices runs from LDS
__device__ __forceinline__ bool wide_fits(const Ctx& c, uint32_t t, uint32_t lds_bytes) {
    return t <= WIDE_LDS_MAX && c.g.p->R <= WIDE_LDS_R_MAX &&
           wide_lds_bytes(t, (uint32_t)c.g.p->rw) <= lds_bytes;
}

// What a task in the slab takes from the wave's state and changes in it.
template <class T>
using lptr = __attribute__((address_space(3))) T*;
struct Far {
    const ExpandArgs* a;
    const DevGraph* g;
    char* slab;
    TaskRef ref;
    long long slot, wadj_l, ph_t;
    unsigned long long share_v;
    lptr<char> lds;
    lptr<LStats> st;
    lptr<unsigned long long> ph, clq;
    lptr<TaskRef> ptopref;
    lptr<uint32_t> fl, fln;
    uint32_t lds_bytes, inst, ptopi, pbot, ptop;
    int shard, share_n, share_left;
    bool share_ok, phase_on;
};
template <class T>
__device__ __forceinline__ T* unip(T* p) {
    return (T*)uni64((long long)p);
}
template <class T>
__device__ __forceinline__ T* unil(lptr<T> p) {
    return (T*)(lptr<T>)(uintptr_t)(uint32_t)uni32((int)(uint32_t)(uintptr_t)p);
}
// A function of its own: with its code inside the kernel the registers of both
// forms of the branch loop did not fit (116 of them in memory, 25 without), and
// the tasks in LDS paid for it, which are most.
template <class P>
__device__ __attribute__((noinline)) bool process_far(Far* f) {
    Ctx c;
    c.a = unip(f->a);
    c.g = load_graph(unip(f->g));
    c.lane = lane_id();
    c.st = unil(f->st);
    c.depth = 0;
    c.inst = (uint32_t)uni32((int)f->inst);
    c.slot = uni64(f->slot);
    c.ph = unil(f->ph);
    c.ph_t = uni64(f->ph_t);
    c.wadj_l = f->wadj_l;
    c.phase_on = uni32(f->phase_on) != 0;
    c.keys = false;
    c.shard = uni32(f->shard);
    c.ptopref = unil(f->ptopref);
    c.ptopi = (uint32_t)uni32((int)f->ptopi);
    c.clq = unil(f->clq);
    c.fl = unil(f->fl);
    c.fln = unil(f->fln);
    c.pstack = c.a->priv + (size_t)blockIdx.x * c.a->priv_cap;
    c.pbkt = c.a->priv_bkt + (size_t)blockIdx.x * c.a->priv_cap;
    c.pbot = (uint32_t)uni32((int)f->pbot);
    c.ptop = (uint32_t)uni32((int)f->ptop);
    c.share_v = f->share_v;
    c.share_n = uni32(f->share_n);
    c.share_left = uni32(f->share_left);
    c.share_ok = uni32(f->share_ok) != 0;
    const TaskRef r = bcast_ref(f->ref, 0);
    const bool ok = process_wide<P>(c, r, unil(f->lds), (uint32_t)uni32((int)f->lds_bytes), unip(f->slab));
    f->ph_t = c.ph_t;
    f->wadj_l = c.wadj_l;
    f->ptopi = c.ptopi;
    f->pbot = c.pbot;
    f->ptop = c.ptop;
    f->share_v = c.share_v;
    f->share_n = c.share_n;
    f->share_left = c.share_left;
    return ok;
}

// a task of any size and kind; FAR: the slab's forms are there (without them
// every task fits the wave's LDS, see enumerate_persistent)
template <bool FAR>
__device__ __attribute__((always_inline)) void process_task(Ctx& c, const TaskRef& ref, char* lds, uint32_t lds_bytes,
                                                            char* slab) {
    if (wide_fits(c, ref.t, lds_bytes) && process_wide<WideLds, FAR>(c, ref, lds, lds_bytes, slab)) return;
    if constexpr (!FAR) {
        if (c.lane == 0) atomicOr(c.a->error, 2);
        return;
    }
    Far f;
    f.a = c.a;
    f.g = c.g.p;
    f.slab = slab;
    f.ref = ref;
    f.slot = c.slot;
    f.wadj_l = c.wadj_l;
    f.ph_t = c.ph_t;
    f.share_v = c.share_v;
    f.lds = (lptr<char>)lds;
    f.st = (lptr<LStats>)c.st;
    f.ph = (lptr<unsigned long long>)c.ph;
    f.clq = (lptr<unsigned long long>)c.clq;
    f.ptopref = (lptr<TaskRef>)c.ptopref;
    f.fl = (lptr<uint32_t>)c.fl;
    f.fln = (lptr<uint32_t>)c.fln;
    f.lds_bytes = lds_bytes;
    f.inst = c.inst;
    f.ptopi = c.ptopi;
    f.pbot = c.pbot;
    f.ptop = c.ptop;
    f.shard = c.shard;
    f.share_n = c.share_n;
    f.share_left = c.share_left;
    f.share_ok = c.share_ok;
    f.phase_on = c.phase_on;
    // (positions and indegrees of at most 12 bits, ids of 16; degrees that do
    // not fit are found at load)
    bool done = false;
    if (ref.t <= WIDE_LDS_MAX && c.g.p->R <= WIDE_MID_R_MAX) {
        const uint32_t rw = (uint32_t)c.g.p->rw, T = wide_T(ref.t);
        // (rows, the child's words, the masks, and the radix sort's counters)
        if ((wide_rows_staged(rw, lds_bytes) ? 24u * rw : 0u) + 4u * T + T / 4u + 1024u <= lds_bytes)
            done = process_far<WideMidLds>(&f);
        else
            done = process_far<WideMid>(&f);
    }
    if (!done) process_far<WideSlab>(&f);
    c.wadj_l = f.wadj_l;
    c.ph_t = uni64(f.ph_t);
    c.ptopi = (uint32_t)uni32((int)f.ptopi);
    c.pbot = (uint32_t)uni32((int)f.pbot);
    c.ptop = (uint32_t)uni32((int)f.ptop);
    c.share_v = f.share_v;
    c.share_n = uni32(f.share_n);
    c.share_left = uni32(f.share_left);
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
__device__ __forceinline__ void flush_stats(Ctx& c, DevStats* d) {
    const unsigned long long wadj = (unsigned long long)wave_sum64(c.wadj_l);
    c.wadj_l = 0;
    if (c.lane == 0) {
        const LStats& t = *c.st;
        if (t.tasks) atomicAdd(&d->tasks, t.tasks);
        if (t.branches) atomicAdd(&d->branches, t.branches);
        if (t.children) atomicAdd(&d->children, t.children);
        if (t.raw) atomicAdd(&d->raw_cliques, t.raw);
        if (t.sum_t) atomicAdd(&d->sum_t, t.sum_t);
        if (t.sum_tw) atomicAdd(&d->sum_t_written, t.sum_tw);
        if (t.sum_clq) atomicAdd(&d->sum_clique_len, t.sum_clq);
        if (t.large) atomicAdd(&d->large_tasks, t.large);
        if (t.beyond) atomicAdd(&d->beyond, t.beyond);
        if (wadj) atomicAdd(&d->w_adj, wadj);
        *c.st = LStats{0, 0, 0, 0, 0, 0, 0, 0, 0};
    }
}
__device__ __forceinline__ void flush_stats(Ctx& c) { flush_stats(c, c.a->stats); }

// Level-synchronous form (expand_level): one wave per task of the batch.  Small
// tasks are launched with little LDS and many waves per CU, large ones with a
// quarter of a CU's LDS and a slab each.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void expand_level(
    const ExpandArgs* __restrict__ ap) {
    const ExpandArgs& a = *ap;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ uint16_t s_dep[TINY_MAX];
    __shared__ LStats s_st;
    __shared__ unsigned long long s_ph[PH_COUNT];
    Ctx c;
    c.wadj_l = 0;
    c.a = ap;
    c.g = load_graph(&ap->g);
    c.phase_on = ap->phase != nullptr;
    c.inst = 0;
    c.slot = -1;
    c.lane = lane_id();
    c.st = &s_st;
    c.ph = s_ph;
    if (c.lane == 0) s_st = LStats{0, 0, 0, 0, 0, 0, 0, 0, 0};
    ph_start(c);
    char* const slab = a.slab + (size_t)blockIdx.x * a.slab_bytes;
    const uint32_t nw = gridDim.x;
    uint32_t i;
    if (a.static_sched) {
        i = blockIdx.x;
    } else {
        uint32_t x = 0;
        if (c.lane == 0) x = atomicAdd(a.task_counter, 1u);
        i = (uint32_t)rdlane((int)x, 0);
    }
    while (i < a.n_in) {
        const TaskRef ref = a.in_refs[i];
        Tiny y;
        if (ref.t <= TINY_MAX && ref.depth > 0 && ref.b1 == 0 && tiny_load(c, ref, y)) {
            c.depth = ref.depth;
            y.cap = TINY_MAX;
            tiny_level(c, y, (uint32_t*)lds, s_dep);
        } else {
            process_task<true>(c, ref, lds, a.lds_bytes, slab);
        }
        wsync();
        if (a.static_sched) {
            i += nw;
        } else {
            uint32_t x = 0;
            if (c.lane == 0) x = atomicAdd(a.task_counter, 1u);
            i = (uint32_t)rdlane((int)x, 0);
        }
    }
    flush_stats(c);
}

// diagnostics: one task's row of the timeline
__device__ __forceinline__ void timeline_row(Ctx& c, const TaskRef& ref, long long gslot, long long start) {
    if (c.lane != 0) return;
    unsigned long long* r = c.a->timeline + 4 * (unsigned long long)gslot;
    r[0] = (unsigned long long)start;
    r[1] = (unsigned long long)wall_clock64();
    r[2] = ((unsigned long long)blockIdx.x << 32) | ref.t;
    r[3] = (unsigned long long)ref.depth | ((unsigned long long)ref.b0 << 16) | ((unsigned long long)ref.b1 << 40);
}

// The block of a task that ran: a split item's prepared record is freed by the
// last of its items (count in the Vrec after the record); roots live outside
// the pool's blocks.
__device__ __attribute__((always_inline)) void release_record(Ctx& c, const TaskRef& ref) {
    if (c.lane != 0) return;
    if (ref.b1 > 0) {
        const int left = __hip_atomic_fetch_add(&c.a->pool[ref.off + ref.t].id, -1, __ATOMIC_ACQ_REL,
                                                __HIP_MEMORY_SCOPE_AGENT);
        if (left == 1) pool_free(c, ref.off, ref.t + 1u);
    } else if (ref.depth > 0) {
        pool_free(c, ref.off, ref.t);
    }
}

// ---------------------------------------------------------------------------
// persistent kernel: every wave takes tasks from its own stack and the shared
// rings until the pending counter reaches zero
// ---------------------------------------------------------------------------
// (two resident waves per SIMD: the register allocation is held to 256)
template <bool FAR>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void expand_persistent(
    const ExpandArgs* __restrict__ ap) {
    const ExpandArgs& a = *ap;
    // a task's arrays, or the stack of a subtree of at most 64 vertices
    extern __shared__ __attribute__((aligned(16))) char lds[];
    Ctx c;
    c.wadj_l = 0;
    c.a = ap;
    c.g = load_graph(&ap->g);
    c.phase_on = ap->phase != nullptr;
    c.inst = 0;
    c.slot = -1;
    c.lane = lane_id();
    c.pstack = a.priv + (size_t)blockIdx.x * a.priv_cap;
    c.pbkt = a.priv_bkt + (size_t)blockIdx.x * a.priv_cap;
    c.pbot = 0;
    c.ptop = 0;
    c.shard = (int)(blockIdx.x % (unsigned)a.q_shards);
    // this wave's stacks of free blocks of the small classes
    __shared__ uint32_t s_fl[FL_SMALL * FL_LOCAL_MAX];
    __shared__ uint32_t s_fln[FL_SMALL];
    c.fl = s_fl;
    c.fln = s_fln;
    if (c.lane < FL_SMALL) s_fln[c.lane] = 0;
    wsync();
    char* const slab = a.slab + (size_t)blockIdx.x * a.slab_bytes;
    __shared__ LStats s_st;
    __shared__ unsigned long long s_ph[PH_COUNT];
    c.st = &s_st;
    c.ph = s_ph;
    if (c.lane == 0) s_st = LStats{0, 0, 0, 0, 0, 0, 0, 0, 0};
    ph_start(c);
    const unsigned long long G = gridDim.x;
    int idle = 0;             // consecutive empty polls (back-off)
    uint32_t idle_total = 0;  // the same, not capped, since the last look that found a working wave
    int sinst = -1;     // instance the wave's counters belong to
    // static order: this wave takes positions blockIdx.x, +G, +2G, ... of
    // the single ring
    unsigned long long spos = blockIdx.x;

    __shared__ TaskRef s_top;
    // the wave's part of the clique stream (none yet)
    __shared__ unsigned long long s_clq[4];
    c.clq = s_clq;
    if (c.lane < 4) s_clq[c.lane] = 0;
    // the subtree of at most 64 vertices in hand (tiny_run), its children's
    // depths; the children themselves use the dynamic LDS
    __shared__ uint16_t s_dep[TINY_STACK_MAX];
    Tiny y{};
    bool tiny = false;  // to be resumed after a hand-over
    c.ptopref = &s_top;
    c.ptopi = ~0u;
    c.share_v = 0;  // reads as nobody waiting
    c.share_n = 0;
    c.share_left = 0;
    c.share_ok = false;
    // the position this wave has taken in a ring and not yet run
    bool ticket = false;
    unsigned long long tpos = 0, tbase = 0;
    // `pending` counts the tasks waiting in the rings plus the waves that hold
    // work (a published position or a non-empty stack); `hungry` counts the
    // waves that hold none.  A wave changes them only when it takes work
    // from the rings, hands work to them or runs out, not per task.
    bool busy = false;
    for (;;) {
        TaskRef ref;
        long long gslot;
        if (a.static_sched && c.ptop != c.pbot && static_flush(c)) {
            continue;
        } else if (tiny || c.ptop != c.pbot) {
            // this wave's own stack (depth first)
            idle = 0;
            ph_mark(c, PH_POP);
            // (a wave with a subtree in hand can give every record away)
            const uint32_t own = tiny ? 0u : 1u;
            if (!a.static_sched && c.ptop - c.pbot > own) {
                // more waves wait for work than the rings hold: hand over
                // the oldest (shallowest, so largest) records, up to 16 at
                // once, to one ring (ring_for).  The rings hold
                // pending - (G - hungry) tasks; handing over more than the
                // waiting waves take turns the search breadth first and
                // multiplies the live records.
                unsigned long long ph = 0;
                if (c.lane == 0) ph = __hip_atomic_load(a.pending, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ph = rdlane64(ph, 0);
                const long long hg = (long long)(ph >> 32), pd = (long long)(ph & 0xFFFFFFFFull);
                const long long waiting = pd - ((long long)G - hg);
                const long long need = hg - (waiting > 0 ? waiting : 0);
                if (need > 0) {
                    const int want = (int)min<long long>(min<long long>((long long)(c.ptop - c.pbot - own), 16ll), need);
                    if (a.n_buckets > 1) {
                        // cost order: the 16 oldest records are ordered by
                        // predicted bucket, largest first (stable), so the
                        // hand-over takes the ones the model predicts largest.
                        // Lane j holds record j; its rank is the number of
                        // records before it in that order.
                        wsync();  // lane 0's stack stores, visible to every lane
                        const int span = (int)min<uint32_t>(c.ptop - c.pbot - own, 16u);
                        const uint32_t at = (c.pbot + (uint32_t)c.lane) % a.priv_cap;
                        const int bj = c.lane < span ? (int)c.pbkt[at] : -1;
                        int rank = 0;
                        for (int i = 0; i < span; i++) {
                            const int bi = rdlane(bj, i);
                            rank += (bi > bj || (bi == bj && i < c.lane)) ? 1 : 0;
                        }
                        if (ballot(c.lane < span && rank != c.lane)) {
                            TaskRef tr;
                            if (c.lane < span) tr = c.pstack[at];
                            wsync();
                            if (c.lane < span) {
                                const uint32_t to = (c.pbot + (uint32_t)rank) % a.priv_cap;
                                c.pstack[to] = tr;
                                c.pbkt[to] = (unsigned char)bj;
                            }
                            wsync();
                        }
                    }
                    const int rg = ring_for(c);
                    // a hand-over is optional: one attempt, and when another
                    // producer moved the tail first the wave keeps its records
                    // (retrying under contention cost more than the records
                    // were worth on trees of tiny tasks)
                    unsigned long long pos = 0;
                    const int k = ring_claim(c, rg, want, &pos, 2);
                    if (k > 0) {
                        // lane j copies entry j (the barrier makes lane 0's
                        // stack stores visible to the other lanes)
                        wsync();
                        if (c.lane < k)
                            a.q_refs[(unsigned long long)rg * a.q_cap + (pos + c.lane) % a.q_cap] =
                                c.pstack[(c.pbot + (uint32_t)c.lane) % a.priv_cap];
                        if (c.lane == 0)
                            __hip_atomic_fetch_add(a.pending, (unsigned long long)k,
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        ring_publish(c, rg, pos, k);
                        c.pbot += (uint32_t)k;
                        if (c.phase_on && c.lane == 0) c.ph[PH_N_GIVEN] += (unsigned long long)k;
                    }
                }
            }
            ph_mark(c, PH_GIVE);
            if (tiny) {
                tiny = tiny_run(c, y, (uint32_t*)lds, s_dep, true);
                ph_mark(c, PH_TINY);
                continue;
            }
            c.ptop--;
            TaskRef r;
            // the newest entry is usually still in LDS (pushed last)
            if (c.lane == 0) r = c.ptopi == c.ptop ? *c.ptopref : c.pstack[c.ptop % a.priv_cap];
            c.ptopi = ~0u;
            ref = bcast_ref(r, 0);
            gslot = -1;
            if (c.phase_on && c.lane == 0) c.ph[PH_N_OWN]++;
        } else {
            // ---- the shared rings ----
            // A wave without work takes a ticket, the next position of a ring
            // (one add on its head), and waits for that position's own
            // sequence word: no two waves want the same task, so a published
            // task wakes one wave and nobody retries.  (Waves that all read
            // every ring's counters and raced for each task by compare and
            // swap slowed the working ones down: with 2,048 waves a power-law
            // window took 29 ms against 13 with 1,024.)  Heads may run ahead
            // of tails by the waves that wait; hand-overs go to such rings
            // (ring_for).  Tasks pushed where nobody waits are found by the
            // pushing wave itself at the latest: it looks at every ring
            // before it waits.
            if (!ticket) {
                if (a.static_sched) {
                    tpos = spos;
                    tbase = 0;
                    spos += G;
                } else {
                    const int NS = a.q_shards;
                    unsigned long long hl = 0, tl = 0;
                    if (c.lane < NS) {
                        hl = __hip_atomic_load(&a.q_head[c.lane * QSTRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        tl = __hip_atomic_load(&a.q_tail[c.lane * QSTRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    // this wave's own shard first (its XCD's L2 holds the
                    // records its neighbours wrote), else the next one with
                    // tasks, else wait at its own
                    const uint64_t m = ballot(c.lane < NS && tl > hl);
                    int r = c.shard;
                    if (m && !((m >> r) & 1ull)) {
                        const uint64_t up = m & ~((2ull << r) - 1ull);
                        r = __builtin_ctzll(up ? up : m);
                    }
                    if (c.lane == 0)
                        tpos = __hip_atomic_fetch_add(&a.q_head[r * QSTRIDE], 1ull, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
                    tpos = rdlane64(tpos, 0);
                    tbase = (unsigned long long)r * a.q_cap;
                }
                ticket = true;
            }
            unsigned long long* const cell = &a.q_seq[tbase + tpos % a.q_cap];
            unsigned long long sq = 0;
            if (c.lane == 0) sq = __hip_atomic_load(cell, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (rdlane64(sq, 0) != tpos + 1ull) {
                if (busy) {
                    // out of work: no longer counted in pending, now hungry
                    busy = false;
                    if (c.lane == 0)
                        __hip_atomic_fetch_add(a.pending, PH_HUNGRY - 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    continue;  // look once more before sleeping
                }
                // Finished once nothing is pending (no ring task and no busy
                // wave: a wave counts itself out only when its stack is
                // empty, after pushing what it made): looked up on every
                // fourth poll by one wave in 16, which tells the others
                // through a word that is written once: with every idle wave
                // reading it, the busy ones' adds to the pending word waited.
                // A task is lost (error bit 4, and every wave leaves) when
                // tasks are pending and no wave works, for longer than one
                // that waits for its position takes to see it.  How long this
                // wave has waited says nothing: tasks may go to other rings,
                // or one wave run a root that is not split.
                // Polls are relaxed: an acquire invalidates the CU's vector L1
                // under the waves still working.
                if ((idle_total++ & 3u) == 0) {
                    int look = 0;  // 1: leave, 2: a wave works
                    if (c.lane == 0) {
                        if ((blockIdx.x & 15u) == 0) {
                            const unsigned long long pd = __hip_atomic_load(a.pending, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            int er = __hip_atomic_load(a.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            if ((pd >> 32) < G)
                                look = 2;
                            else if ((uint32_t)pd != 0 && idle_total / 4 >= a.idle_limit)
                                er |= atomicOr(a.error, 4) | 4;
                            if ((uint32_t)pd == 0 || (er & 4) != 0) look = 1;
                            if (look == 1) __hip_atomic_store(a.done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        } else {
                            look = __hip_atomic_load(a.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
                        }
                    }
                    look = rdlane(look, 0);
                    if (look == 1) break;
                    if (look == 2) idle_total = 1;
                }
                idle = idle < 8 ? idle + 1 : 8;
                for (int k = 0; k < idle; k++) __builtin_amdgcn_s_sleep(16);
                ph_mark(c, PH_IDLE);
                continue;
            }
            idle = 0;
            idle_total = 0;
            ticket = false;
            // the task leaves the ring; an idle wave becomes busy
            if (c.lane == 0) {
                const unsigned long long d = busy ? 0ull - 1ull : 0ull - PH_HUNGRY;
                __hip_atomic_fetch_add(a.pending, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            busy = true;
            // the acquire pairs with the producer's release before the
            // sequence word; the ref is read before the cell goes back for the
            // next lap, with a plain relaxed store: no release, whose
            // agent-scope form writes back this XCD's L2
            ph_mark(c, PH_POP);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            gslot = (long long)(tbase + tpos % a.q_cap);
            TaskRef r;
            if (c.lane == 0) r = a.q_refs[gslot];
            ref = bcast_ref(r, 0);
            wsync();
            if (c.lane == 0)
                __hip_atomic_store(cell, tpos + a.q_cap, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (c.phase_on && c.lane == 0) c.ph[PH_N_RING]++;
            ph_mark(c, PH_SYNC);
        }
        ph_mark(c, PH_POP);
        const long long tl_start = a.timeline ? wall_clock64() : 0;
        if (a.graphs) {
            c.g = load_graph(&a.graphs[ref.inst]);
            c.inst = ref.inst;
        }
        if (a.inst_stats && (int)ref.inst != sinst) {
            if (sinst >= 0) flush_stats(c, &a.inst_stats[sinst]);
            sinst = ref.inst;
        }
        c.slot = ref.b1 > 0 ? (long long)ref.bound : gslot;
        c.share_ok = ref.t >= SHARE_MIN_T;
        // A task that fits one vertex a lane runs with its whole subtree in
        // registers.  64 is the width of a wave and of a mask in scalar
        // registers; split items (prepared records) and the root (labels
        // other than member and candidate) take the general path.  Against
        // that path for every size (kernel, medians): a full search of 1.86
        // million tasks of 23 vertices 59 -> 22 ms, a power-law window of
        // 252,000 tasks of 29 34 -> 16 ms, 3,051 tasks of 17 16.3 -> 9.0 ms;
        // a window whose tasks are all larger is unchanged.
        if (ref.t <= TINY_MAX && ref.depth > 0 && ref.b1 == 0 && a.tiny_cap && tiny_load(c, ref, y)) {
            y.cap = a.tiny_cap;
            // (the record is in registers: its block can go back at once)
            wsync();
            if (c.lane == 0) pool_free(c, ref.off, ref.t);
            ph_mark(c, PH_LOAD);
            tiny = tiny_run(c, y, (uint32_t*)lds, s_dep, false);
            ph_mark(c, PH_TINY);
            if (a.timeline && gslot >= 0) timeline_row(c, ref, gslot, tl_start);
            continue;
        }
        y = Tiny{};  // nothing of it lives across the general path
        if (ref.t > a.slab_tcap) {
            if (c.lane == 0) atomicOr(a.error, 2);
        } else {
            process_task<FAR>(c, ref, lds, a.lds_bytes, slab);
        }
        wsync();
        if (a.timeline && gslot >= 0) timeline_row(c, ref, gslot, tl_start);
        ph_mark(c, PH_CHILD);
        release_record(c, ref);
        ph_mark(c, PH_POOL);
    }
    ph_mark(c, PH_IDLE);
    ph_flush(c);
    clq_close(c);
    if (sinst >= 0)
        flush_stats(c, &a.inst_stats[sinst]);
    else
        flush_stats(c);
}

template __global__ void expand_persistent<false>(const ExpandArgs* __restrict__);
template __global__ void expand_persistent<true>(const ExpandArgs* __restrict__);

}  // namespace qcdev
