// root.hip -- root task construction (initialize_tasks, main.cu:846-998) and
// the device tables the expansion kernels read.
//
// The degree / |N2| filter (main.cu:872-885) and the k-core peel (main.cu:889-949)
// run on the device for large graphs, else on the host, as do the cover vertex
// and covered set (main.cu:953-975) and the Q-ordered root record
// (main.cu:978-995).
// Device tables: for every root vertex, its rows of the root-space 1-hop and
// 2-hop bit matrices and its full-graph |N2| (the third Q-order key), with
// the 2-hop relation of adjToSer.cpp:115-156: N(v) u N(N(v)) minus v.
//
// Root-local ids are assigned in increasing input-id order, so comparing
// root-local ids orders vertices exactly like comparing input ids (the last
// Q-order key, main.cu:2098-2101).

#include <algorithm>
#include <chrono>
#include <cmath>
#include <mutex>
#include <thread>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "qc_internal.h"

namespace qcdev {

// One wave per root vertex.  vis: per-wave visited bitmap over all n input
// vertices (zero on entry and on exit).
__global__ __launch_bounds__(64) void root_rows(const uint64_t* __restrict__ off, const uint32_t* __restrict__ adj,
                                                const uint64_t* __restrict__ off2, const uint32_t* __restrict__ adj2,
                                                const int32_t* __restrict__ loc, const uint32_t* __restrict__ orig,
                                                int32_t R, int32_t rw, uint64_t* A1, uint64_t* A2, int32_t* n2out,
                                                unsigned long long* vis_all, uint64_t vis_words, int has_n2) {
    const int lane = threadIdx.x & 63;
    unsigned long long* vis = vis_all + (size_t)blockIdx.x * vis_words;
    for (int a = blockIdx.x; a < R; a += gridDim.x) {
        const uint32_t v = orig[a];
        unsigned long long* row1 = (unsigned long long*)(A1 + (size_t)a * rw);
        unsigned long long* row2 = (unsigned long long*)(A2 + (size_t)a * rw);
        const uint64_t b0 = off[v], b1 = off[v + 1];
        for (uint64_t j = b0 + lane; j < b1; j += 64) {
            int la = loc[adj[j]];
            if (la >= 0) atomicOr(&row1[la >> 6], 1ull << (la & 63));
        }
        if (has_n2) {
            for (uint64_t j = off2[v] + lane; j < off2[v + 1]; j += 64) {
                int la = loc[adj2[j]];
                if (la >= 0) atomicOr(&row2[la >> 6], 1ull << (la & 63));
            }
            if (lane == 0) n2out[a] = (int32_t)(off2[v + 1] - off2[v]);
            __syncthreads();
            continue;
        }
        if (lane == 0) atomicOr(&vis[v >> 6], 1ull << (v & 63));
        __syncthreads();
        int cnt = 0;
        for (uint64_t j = b0 + lane; j < b1; j += 64) {
            uint32_t u = adj[j];
            unsigned long long bit = 1ull << (u & 63);
            unsigned long long old = atomicOr(&vis[u >> 6], bit);
            if (!(old & bit)) {
                cnt++;
                int la = loc[u];
                if (la >= 0) atomicOr(&row2[la >> 6], 1ull << (la & 63));
            }
        }
        for (uint64_t j = b0; j < b1; j++) {
            uint32_t u = adj[j];
            for (uint64_t k = off[u] + lane; k < off[u + 1]; k += 64) {
                uint32_t x = adj[k];
                unsigned long long bit = 1ull << (x & 63);
                unsigned long long old = atomicOr(&vis[x >> 6], bit);
                if (!(old & bit)) {
                    cnt++;
                    int la = loc[x];
                    if (la >= 0) atomicOr(&row2[la >> 6], 1ull << (la & 63));
                }
            }
        }
        for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
        if (lane == 0) n2out[a] = cnt;
        __syncthreads();
        // restore the visited bitmap to zero
        if (lane == 0) vis[v >> 6] = 0;
        for (uint64_t j = b0 + lane; j < b1; j += 64) vis[adj[j] >> 6] = 0;
        for (uint64_t j = b0; j < b1; j++) {
            uint32_t u = adj[j];
            for (uint64_t k = off[u] + lane; k < off[u + 1]; k += 64) vis[adj[k] >> 6] = 0;
        }
        __syncthreads();
    }
}

// The same rows and counts with the visited map and the 1-hop row in LDS, for
// graphs whose map fits, and with |N n root| and |N2 n root| (root_d2).
//
// A workgroup takes vertices from a counter (their work differs by orders of
// magnitude).  The lists to walk are cut into segments of ROWS_SEG entries, as
// many tables of them as they need, and every wave takes ROWS_AT_ONCE segments
// at a time: their loads, 16 a lane, are in flight together.  (Lists walked one
// after another waited for two dependent loads each, 2 us a list whatever its
// length: 34.9 ms for the 70,088 root vertices of a power-law graph of a million,
// whose 11.7 billion entries are now walked in 10.9, 4.3 TB/s; 3.0 -> 0.5 ms for a
// co-expression graph's 1.1 billion, 1.8 -> 0.5 for 0.4 billion of a smaller
// power-law graph.)  NT threads share a vertex: 256, or 1024 when the map leaves
// room for one workgroup per CU.
constexpr int ROWS_THREADS = 256;
constexpr int ROWS_THREADS_WIDE = 1024;
constexpr int ROWS_SEG = 256;
constexpr int ROWS_AT_ONCE = 4;
constexpr int ROWS_TAB_MIN = 256;   // segments in the LDS table, at least
constexpr int ROWS_TAB_MAX = 2048;

__device__ __forceinline__ uint64_t rdl64(uint64_t x, int l) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), l);
    return ((uint64_t)hi << 32) | lo;
}

template <bool BYTES, int NT>
__global__ __launch_bounds__(NT) void root_rows_lds(const uint64_t* __restrict__ off, const uint32_t* __restrict__ adj,
                                                    const int32_t* __restrict__ loc, const uint32_t* __restrict__ orig,
                                                    int32_t R, int32_t rw, int32_t n, int32_t tab_n, uint64_t* A1,
                                                    uint64_t* A2, int32_t* n2out, int32_t* d1r, int32_t* d2r,
                                                    uint32_t* next) {
    // vis: {v} u N(v) u N(N(v)) over all n vertices, as a byte map (BYTES:
    // plain stores of 1, no read-modify-write) or a bitmap (atomics without
    // return); r1: root-space row of N(v); seg: list start << 16 | entries.
    // |N2(v)| and the A2 row are read off the map afterwards.
    extern __shared__ unsigned long long sh[];
    __shared__ uint32_t s_a, s_tot, s_cnt, s_d1, s_d2;
    const int lane = threadIdx.x & 63;
    const int tid = threadIdx.x;
    const int wv = threadIdx.x >> 6;
    constexpr int NWV = NT / 64;
    const int nw = BYTES ? (n + 7) / 8 : (n + 63) / 64;  // 64-bit words of the map
    unsigned long long* const vis = sh;
    uint32_t* const vis32 = (uint32_t*)sh;
    unsigned char* const vis8 = (unsigned char*)sh;
    unsigned long long* const r1 = sh + nw;
    unsigned long long* const seg = r1 + rw;
    auto mark = [&](uint32_t x) {
        if (BYTES)
            vis8[x] = 1;
        else
            atomicOr(&vis32[x >> 5], 1u << (x & 31));
    };
    auto seen = [&](uint32_t x) -> bool { return BYTES ? vis8[x] != 0 : ((vis32[x >> 5] >> (x & 31)) & 1u) != 0; };
    for (;;) {
        __syncthreads();  // (the vertex before is done with everything shared)
        if (tid == 0) {
            s_a = atomicAdd(next, 1u);
            s_tot = s_cnt = s_d1 = s_d2 = 0;
        }
        for (int w = tid; w < nw; w += NT) vis[w] = 0;
        for (int w = tid; w < rw; w += NT) r1[w] = 0;
        __syncthreads();
        const uint32_t a = s_a;
        if (a >= (uint32_t)R) break;
        const uint32_t v = orig[a];
        if (tid == 0) mark(v);
        const uint64_t b0 = off[v], b1 = off[v + 1];
        for (uint64_t j0 = b0; j0 < b1; j0 += NT) {
            // a neighbour per thread: marked, and its list as segments
            uint64_t st = 0, len = 0;
            if (j0 + tid < b1) {
                const uint32_t u = adj[j0 + tid];
                mark(u);
                const int la = loc[u];
                if (la >= 0) atomicOr(&r1[la >> 6], 1ull << (la & 63));
                st = off[u];
                len = off[u + 1] - st;
            }
            const uint32_t ns = (uint32_t)((len + ROWS_SEG - 1) / ROWS_SEG);
            uint32_t pos = ns;  // inclusive prefix over the wave
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = __shfl_up(pos, o, 64);
                if (lane >= o) pos += y;
            }
            uint32_t at = 0;
            if (lane == 63) at = atomicAdd(&s_tot, pos);
            pos += (uint32_t)__builtin_amdgcn_readlane((int)at, 63) - ns;
            __syncthreads();
            const uint32_t tot = s_tot;
            for (uint32_t lo = 0; lo < tot; lo += (uint32_t)tab_n) {
                const uint32_t hi = min(tot, lo + (uint32_t)tab_n);
                for (uint32_t q = max(pos, lo); q < min(pos + ns, hi); q++) {
                    const uint64_t d = (uint64_t)(q - pos) * ROWS_SEG;
                    seg[q - lo] = ((st + d) << 16) | min(len - d, (uint64_t)ROWS_SEG);
                }
                __syncthreads();
                const int m = (int)(hi - lo);
                for (int g = wv * ROWS_AT_ONCE; g < m; g += NWV * ROWS_AT_ONCE) {
                    uint64_t sg = 0;
                    if (lane < ROWS_AT_ONCE && g + lane < m) sg = seg[g + lane];
                    uint32_t x[ROWS_AT_ONCE][ROWS_SEG / 64];
#pragma unroll
                    for (int q = 0; q < ROWS_AT_ONCE; q++) {
                        const uint64_t e = rdl64(sg, q);
                        const uint32_t* const p = adj + (e >> 16);
                        const int l = (int)(e & 0xFFFFull);
#pragma unroll
                        for (int k = 0; k < ROWS_SEG / 64; k++) {
                            x[q][k] = 0xFFFFFFFFu;
                            if (k * 64 + lane < l) x[q][k] = p[k * 64 + lane];
                        }
                    }
#pragma unroll
                    for (int q = 0; q < ROWS_AT_ONCE; q++)
#pragma unroll
                        for (int k = 0; k < ROWS_SEG / 64; k++)
                            if (x[q][k] != 0xFFFFFFFFu) mark(x[q][k]);
                }
                __syncthreads();
            }
            if (tid == 0) s_tot = 0;
            __syncthreads();
        }
        __syncthreads();
        int cnt = 0, c1 = 0, c2 = 0;
        for (int w = tid; w < nw; w += NT) cnt += __popcll(vis[w]);  // bytes are 0 or 1
        for (int w = tid; w < rw; w += NT) {
            A1[(size_t)a * rw + w] = r1[w];
            c1 += __popcll(r1[w]);
        }
        for (int o = 32; o > 0; o >>= 1) {
            cnt += __shfl_xor(cnt, o, 64);
            c1 += __shfl_xor(c1, o, 64);
        }
        // A2 row: bit b iff orig[b] was reached (b != a), one ballot per
        // word; eight words per step keep eight orig loads in flight, and the
        // words leave in one store
        for (int w0 = wv * 8; w0 < rw; w0 += NWV * 8) {
            uint32_t xs[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int b = (w0 + k) * 64 + lane;
                xs[k] = (w0 + k < rw && b < R) ? orig[b] : 0xFFFFFFFFu;
            }
            unsigned long long mine = 0;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const uint32_t b = (uint32_t)((w0 + k) * 64 + lane);
                const unsigned long long word = __ballot(xs[k] != 0xFFFFFFFFu && b != a && seen(xs[k]));
                c2 += __popcll(word);
                if (lane == k) mine = word;
            }
            if (lane < 8 && w0 + lane < rw) A2[(size_t)a * rw + w0 + lane] = mine;
        }
        if (lane == 0) {
            atomicAdd(&s_cnt, (uint32_t)cnt);
            atomicAdd(&s_d1, (uint32_t)c1);
            atomicAdd(&s_d2, (uint32_t)c2);
        }
        __syncthreads();
        if (tid == 0) {
            n2out[a] = (int32_t)s_cnt - 1;  // v itself is in the map
            d1r[a] = (int32_t)s_d1;
            d2r[a] = (int32_t)s_d2;
        }
    }
}

// ---- filter and peel on the device (large graphs) ----
// State of a peel: queue lengths per round, the core's size, and how many of
// its vertices have fewer than min_size - 1 neighbours.
constexpr int PEEL_ROUNDS = 48;
struct PeelState {
    uint32_t cnt[PEEL_ROUNDS + 1];
    uint32_t R;
    uint32_t n_check;
};
constexpr int SCAN_PER = 4096;  // vertices per block of the compaction

// The degree filter (thr, and lists of min_size - 1 second neighbours when the
// graph has them), a bit per vertex: the count below reads one for every entry
// of every list, from a table that the caches hold.
__global__ __launch_bounds__(256) void peel_pass(const uint64_t* __restrict__ off, const uint64_t* __restrict__ off2,
                                                 int32_t n, int32_t thr, int64_t need2, uint64_t* __restrict__ pass) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool ok = i < n && (int64_t)(off[i + 1] - off[i]) >= thr &&
                    (!off2 || (int64_t)(off2[i + 1] - off2[i]) >= need2);
    const unsigned long long m = __ballot(ok);
    if ((threadIdx.x & 63) == 0 && i < n) pass[i >> 6] = m;
}

// Degrees inside the vertices that pass, and the first round of the peel's
// queue.  exd < 0 marks what did not pass.  A wave takes 64 vertices and walks the
// lists of those that pass, one after the other.
__global__ __launch_bounds__(256) void peel_count(const uint64_t* __restrict__ off, const uint32_t* __restrict__ adj,
                                                  const uint64_t* __restrict__ pass, int32_t n, int32_t thr,
                                                  int32_t* __restrict__ exd, uint32_t* __restrict__ queue,
                                                  PeelState* ps) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), nwave = (int64_t)gridDim.x * 4;
    for (int64_t b = wave * 64; b < n; b += nwave * 64) {
        const unsigned long long word = pass[b >> 6];
        if (b + lane < n && !((word >> lane) & 1ull)) exd[b + lane] = -1;
        for (unsigned long long m = word; m; m &= m - 1) {
            const int64_t v = b + __builtin_ctzll(m);
            const uint64_t e = off[v + 1];
            int d = 0;
#pragma unroll 4
            for (uint64_t j = off[v] + lane; j < e; j += 64) {
                const uint32_t u = adj[j];
                d += (int)((pass[u >> 6] >> (u & 63)) & 1ull);
            }
            for (int o = 32; o > 0; o >>= 1) d += __shfl_xor(d, o, 64);
            if (lane == 0) {
                exd[v] = d;
                if (d < thr) queue[atomicAdd(&ps->cnt[0], 1u)] = (uint32_t)v;
            }
        }
    }
}

// One round: the lists of the vertices queued by the round before; a neighbour
// whose degree comes down to thr - 1 joins the next round (once, since degrees
// go down by one at a time; those queued first are below already).
__global__ __launch_bounds__(256) void peel_round(const uint64_t* __restrict__ off, const uint32_t* __restrict__ adj,
                                                  int32_t thr, int32_t* exd, uint32_t* queue, PeelState* ps, int r) {
    const int lane = threadIdx.x & 63;
    const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6), nwave = gridDim.x * 4;
    uint32_t lo = 0;
    for (int k = 0; k < r; k++) lo += ps->cnt[k];
    const uint32_t hi = lo + ps->cnt[r];
    for (uint32_t q = lo + wave; q < hi; q += nwave) {
        const uint32_t v = queue[q];
        const uint64_t e = off[v + 1];
        for (uint64_t j = off[v] + lane; j < e; j += 64) {
            const uint32_t u = adj[j];
            // (what did not pass stays negative)
            if (exd[u] >= 0 && atomicSub(&exd[u], 1) == thr) queue[hi + atomicAdd(&ps->cnt[r + 1], 1u)] = u;
        }
    }
}

// The core's vertices in input order: per block, their number (first), then
// their places.
__global__ __launch_bounds__(256) void core_count(const int32_t* __restrict__ exd, int32_t n, int32_t thr,
                                                  uint32_t* __restrict__ sums) {
    __shared__ uint32_t s;
    if (threadIdx.x == 0) s = 0;
    __syncthreads();
    const int64_t b = (int64_t)blockIdx.x * SCAN_PER;
    uint32_t k = 0;
    for (int i = threadIdx.x; i < SCAN_PER; i += 256)
        if (b + i < n && exd[b + i] >= thr) k++;
    for (int o = 32; o > 0; o >>= 1) k += __shfl_xor(k, o, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(&s, k);
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}
__global__ __launch_bounds__(64) void core_scan(uint32_t* sums, int32_t nb, PeelState* ps) {
    const int lane = threadIdx.x;
    uint32_t run = 0;
    for (int b = 0; b < nb; b += 64) {
        const uint32_t x = b + lane < nb ? sums[b + lane] : 0u;
        uint32_t y = x;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(y, o, 64);
            if (lane >= o) y += t;
        }
        if (b + lane < nb) sums[b + lane] = run + y - x;
        run += (uint32_t)__builtin_amdgcn_readlane((int)y, 63);
    }
    if (lane == 0) {
        ps->R = run;
        ps->n_check = 0;
    }
}
__global__ __launch_bounds__(64) void core_write(const int32_t* __restrict__ exd, const uint64_t* __restrict__ off,
                                                 int32_t n, int32_t thr, int64_t need, const uint32_t* __restrict__ sums,
                                                 int32_t* __restrict__ loc, uint32_t* __restrict__ orig,
                                                 int32_t* __restrict__ core_deg, uint32_t* __restrict__ check,
                                                 PeelState* ps) {
    const int lane = threadIdx.x;
    const int64_t b = (int64_t)blockIdx.x * SCAN_PER;
    uint32_t at = sums[blockIdx.x];
    for (int i = 0; i < SCAN_PER && b + i < n; i += 64) {
        const int64_t v = b + i + lane;
        const int d = v < n ? exd[v] : -1;
        const bool in = v < n && d >= thr;
        const uint64_t m = __ballot(in);
        const uint32_t p = at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        if (v < n) loc[v] = in ? (int32_t)p : -1;
        if (in) {
            orig[p] = (uint32_t)v;
            core_deg[p] = d;
            if ((int64_t)(off[v + 1] - off[v]) < need) check[atomicAdd(&ps->n_check, 1u)] = (uint32_t)v;
        }
        at += (uint32_t)__popcll(m);
    }
}

// kept root vertices against the removed ones: one wave per kept vertex,
// cnt[i] = |N(ids[i]) n removed| from its A1 row and the removal mask
__global__ __launch_bounds__(64) void root_cut_deg(const uint64_t* __restrict__ A1, int32_t rw,
                                                   const uint32_t* __restrict__ ids, int32_t nk,
                                                   const uint64_t* __restrict__ mask, int32_t* __restrict__ cnt) {
    const int lane = threadIdx.x & 63;
    for (int i = blockIdx.x; i < nk; i += gridDim.x) {
        const uint64_t* row = A1 + (size_t)ids[i] * rw;
        int c = 0;
        for (int w = lane; w < rw; w += 64) c += __popcll(row[w] & mask[w]);
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
        if (lane == 0) cnt[i] = c;
    }
}

// row popcounts: |N2(a) n root| and |N(a) n root|
__global__ __launch_bounds__(64) void root_d2(const uint64_t* __restrict__ A2, const uint64_t* __restrict__ A1,
                                              int32_t R, int32_t rw, int32_t* d2r, int32_t* d1r) {
    const int lane = threadIdx.x & 63;
    for (int a = blockIdx.x; a < R; a += gridDim.x) {
        int s = 0, s1 = 0;
        for (int w = lane; w < rw; w += 64) {
            s += __popcll(A2[(size_t)a * rw + w]);
            s1 += __popcll(A1[(size_t)a * rw + w]);
        }
        for (int o = 32; o > 0; o >>= 1) {
            s += __shfl_xor(s, o, 64);
            s1 += __shfl_xor(s1, o, 64);
        }
        if (lane == 0) {
            d2r[a] = s;
            d1r[a] = s1;
        }
    }
}

}  // namespace qcdev

namespace qc {

namespace {

// The filter and the peel run on the device from this many vertices or list
// entries on: 0.3 ms or more of launches and round trips there, while the host
// took 1.9 ms for a power-law graph of 100,000 vertices and 2 million entries,
// 0.5 to 0.8 for a co-expression graph of 8,000 and 2 million, and 0.1 to 0.3 for
// the smaller ones.
constexpr int PEEL_DEVICE_MIN = 32768;
constexpr size_t PEEL_DEVICE_ENTRIES = (size_t)1 << 20;

// min(|N2(v)|, cap) over the full graph: the walk stops at the cap-th
// distinct vertex (a neighbour that is a hub would otherwise cost its whole
// list for a vertex that passed long before)
long n2_capped(const qc_graph* g, int v, std::vector<int>& mark, long cap) {
    if (g->has_n2) return std::min<long>((long)(g->off2[v + 1] - g->off2[v]), cap);
    long cnt = 0;
    mark[v] = v;
    for (uint64_t j = g->off[v]; j < g->off[v + 1]; j++) {
        uint32_t u = g->adj[j];
        if (mark[u] != v) {
            mark[u] = v;
            if (++cnt >= cap) return cnt;
        }
        for (uint64_t k = g->off[u]; k < g->off[u + 1]; k++) {
            uint32_t x = g->adj[k];
            if (mark[x] != v) {
                mark[x] = v;
                if (++cnt >= cap) return cnt;
            }
        }
    }
    return cnt;
}

inline int label_rank(int l) { return l == 1 ? 0 : l == 2 ? 1 : l == 0 ? 2 : l == 3 ? 3 : 4; }

inline int bits_of(uint32_t x) { return x ? 32 - __builtin_clz(x) : 0; }

// root-local ids in the root's Q order.  The four keys in one word where they
// fit, sorted by 11 bits a pass (70,000 vertices: 1 ms against 6 by comparing).
void q_order(int R, int max_ex, int max_l2, const std::vector<int32_t>& label, const std::vector<int32_t>& exd,
             const std::vector<int32_t>& l2, std::vector<int32_t>& order) {
    const int be = bits_of((uint32_t)max_ex), bl = bits_of((uint32_t)max_l2), bi = bits_of((uint32_t)(R - 1));
    if (3 + be + bl + bi > 64) {
        for (int a = 0; a < R; a++) order[a] = a;
        std::sort(order.begin(), order.end(), [&](int x, int y) {
            const int rx = label_rank(label[x]), ry = label_rank(label[y]);
            if (rx != ry) return rx < ry;
            if (exd[x] != exd[y]) return exd[x] > exd[y];
            if (l2[x] != l2[y]) return l2[x] > l2[y];
            return x > y;
        });
        return;
    }
    // (ascending: the descending keys as their distance from the largest)
    std::vector<uint64_t> key(R);
    for (int a = 0; a < R; a++)
        key[a] = ((((uint64_t)label_rank(label[a]) << be | (uint64_t)(max_ex - exd[a])) << bl |
                   (uint64_t)(max_l2 - l2[a]))
                  << bi) |
                 (uint64_t)(R - 1 - a);
    if (R < 4096) {
        std::sort(key.begin(), key.end());
    } else {
        std::vector<uint64_t> tmp(R);
        std::vector<uint32_t> cnt(2048);
        for (int sh = 0; sh < 3 + be + bl + bi; sh += 11) {
            std::fill(cnt.begin(), cnt.end(), 0u);
            for (uint64_t k : key) cnt[(k >> sh) & 2047]++;
            uint32_t at = 0;
            for (uint32_t& c : cnt) {
                const uint32_t x = c;
                c = at;
                at += x;
            }
            for (uint64_t k : key) tmp[cnt[(k >> sh) & 2047]++] = k;
            key.swap(tmp);
        }
    }
    for (int a = 0; a < R; a++) order[a] = R - 1 - (int)(key[a] & ((1ull << bi) - 1ull));
}

}  // namespace

namespace {
struct DevCSR {
    DBuf off, adj, off2, adj2;
};
void free_devcsr(void* p) { delete (DevCSR*)p; }

// the graph's arrays in HBM, uploaded once per graph (the batch builders
// run on several host threads and a batch may hold one graph twice: the
// check and the upload happen under one lock)
int device_csr(const qc_graph* g, DevCSR** out, hipStream_t s) {
    static std::mutex upload_mu;
    std::lock_guard<std::mutex> lock(upload_mu);
    qc_graph* mg = const_cast<qc_graph*>(g);
    if (!mg->dev) {
        DevCSR* d = new DevCSR;
        int rc;
        if ((rc = d->off.alloc(g->off.size() * 8)) || (rc = d->adj.alloc(g->adj.size() * 4))) {
            delete d;
            return rc;
        }
        if (hipMemcpyAsync(d->off.p, g->off.data(), g->off.size() * 8, hipMemcpyHostToDevice, s) != hipSuccess ||
            hipMemcpyAsync(d->adj.p, g->adj.data(), g->adj.size() * 4, hipMemcpyHostToDevice, s) != hipSuccess) {
            delete d;
            set_error("graph upload failed");
            return QC_EDEVICE;
        }
        if (g->has_n2) {
            if ((rc = d->off2.alloc(g->off2.size() * 8)) || (rc = d->adj2.alloc(g->adj2.size() * 4))) {
                delete d;
                return rc;
            }
            if (hipMemcpyAsync(d->off2.p, g->off2.data(), g->off2.size() * 8, hipMemcpyHostToDevice, s) !=
                    hipSuccess ||
                hipMemcpyAsync(d->adj2.p, g->adj2.data(), g->adj2.size() * 4, hipMemcpyHostToDevice, s) !=
                    hipSuccess) {
                delete d;
                set_error("graph upload failed");
                return QC_EDEVICE;
            }
        }
        if (hipStreamSynchronize(s) != hipSuccess) {
            delete d;
            set_error("graph upload failed");
            return QC_EDEVICE;
        }
        mg->dev = d;
        mg->dev_free = free_devcsr;
    }
    *out = (DevCSR*)mg->dev;
    return QC_OK;
}
}  // namespace

namespace {

// Filter (main.cu:872-885) and peel (main.cu:889-949).  The reference's rounds and
// queue compute the core in which every vertex has at least thr neighbours
// inside it (unique, whatever the removal order), with exd = the degree inside
// it.  Here: degrees inside the filtered set (host threads over the vertices),
// then one queue that only walks the lists of removed filtered vertices.
void peel_host(const qc_graph* g, int thr, int ms, std::vector<uint32_t>& orig, std::vector<int32_t>& core_deg,
               std::vector<int32_t>& loc) {
    const int n = g->n;
    std::vector<int32_t> lab(n), exd(n);
    std::vector<int32_t> rem;
    std::vector<int> mark(n, -1);
    for (int i = 0; i < n; i++) {
        int deg = (int)(g->off[i + 1] - g->off[i]);
        exd[i] = deg;
        bool pass = deg >= thr;
        if (pass && deg < ms - 1) pass = n2_capped(g, i, mark, ms - 1) >= ms - 1;
        if (pass && g->has_n2) pass = (long)(g->off2[i + 1] - g->off2[i]) >= ms - 1;
        lab[i] = pass ? 0 : -1;
        if (pass) rem.push_back(i);
    }
    {
        const unsigned hw = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
        const size_t nrem = rem.size();
        const unsigned nth = nrem > 65536 ? hw : 1u;
        auto count = [&](size_t lo, size_t hi) {
            for (size_t k = lo; k < hi; k++) {
                const int v = rem[k];
                int d = 0;
                for (uint64_t j = g->off[v]; j < g->off[v + 1]; j++) d += lab[g->adj[j]] == 0;
                exd[v] = d;
            }
        };
        if (nth == 1) {
            count(0, nrem);
        } else {
            std::vector<std::thread> th;
            for (unsigned t = 0; t < nth; t++)
                th.emplace_back(count, nrem * t / nth, nrem * (t + 1) / nth);
            for (auto& x : th) x.join();
        }
    }
    std::vector<int32_t> queue;
    for (int v : rem)
        if (exd[v] < thr) {
            lab[v] = -1;
            queue.push_back(v);
        }
    for (size_t k = 0; k < queue.size(); k++) {
        const int v = queue[k];
        for (uint64_t j = g->off[v]; j < g->off[v + 1]; j++) {
            const uint32_t u = g->adj[j];
            if (lab[u] == 0 && --exd[u] < thr) {
                lab[u] = -1;
                queue.push_back(u);
            }
        }
    }
    // root-local ids
    loc.assign(n, -1);
    orig.clear();
    core_deg.clear();
    for (int i = 0; i < n; i++)
        if (lab[i] == 0) {
            loc[i] = (int32_t)orig.size();
            orig.push_back((uint32_t)i);
            core_deg.push_back(exd[i]);
        }
}

// The same on the device.  Without second-neighbour lists the filter's |N2|
// >= min_size - 1 is left out there and looked up for the core's vertices of
// degree below min_size - 1: a core whose vertices all have it is the filtered
// core too (it contains that one, and is one).  done = false, to be done on the
// host: a vertex of the core does not have it, or the peel takes more rounds
// than PEEL_ROUNDS (a long chain would cost a launch for each of its vertices).
// A power-law graph of a million vertices and 30 million entries: 45 ms on 16
// host threads, 1.2 here, bound by the latency of the rounds' launches and the
// random reads of the count.
int peel_device(const qc_graph* g, const DevCSR& G, int thr, int ms, Instance& I, std::vector<int32_t>& core_deg,
                DBuf& d_loc, bool& done, hipStream_t s) {
    using namespace qcdev;
    const int n = g->n;
    done = false;
    if (thr < 0) return QC_OK;
    DBuf d_exd, d_queue, d_state, d_sums, d_deg, d_pass, d_check;
    int rc;
    const int nb = (int)(((int64_t)n + SCAN_PER - 1) / SCAN_PER);
    if ((rc = d_exd.alloc((size_t)n * 4, s)) || (rc = d_queue.alloc((size_t)n * 4, s)) ||
        (rc = d_state.alloc(sizeof(PeelState), s)) || (rc = d_sums.alloc((size_t)nb * 4, s)) ||
        (rc = d_deg.alloc((size_t)n * 4, s)) || (rc = d_loc.alloc((size_t)n * 4, s)) ||
        (rc = d_pass.alloc(((size_t)n + 63) / 64 * 8, s)) || (rc = d_check.alloc((size_t)n * 4, s)) ||
        (rc = I.d_orig.alloc((size_t)n * 4)))
        return rc;
    QC_HIP(hipMemsetAsync(d_state.p, 0, sizeof(PeelState), s));
    PeelState* ps = d_state.as<PeelState>();
    const uint64_t* off = G.off.as<uint64_t>();
    const uint32_t* adj = G.adj.as<uint32_t>();
    hipLaunchKernelGGL(peel_pass, dim3((n + 255) / 256), dim3(256), 0, s, off,
                       g->has_n2 ? G.off2.as<uint64_t>() : (const uint64_t*)nullptr, n, thr, (int64_t)ms - 1,
                       d_pass.as<uint64_t>());
    hipLaunchKernelGGL(peel_count, dim3(std::min((n + 255) / 256, 2048)), dim3(256), 0, s, off, adj,
                       d_pass.as<uint64_t>(), n, thr, d_exd.as<int32_t>(), d_queue.as<uint32_t>(), ps);
    QC_HIP(hipGetLastError());
    // (12 rounds between looks at the queue: a round of nothing takes 3 us, a look 20)
    PeelState h;
    int r = 0;
    for (;;) {
        for (int k = 0; k < 12; k++, r++)
            hipLaunchKernelGGL(peel_round, dim3(512), dim3(256), 0, s, off, adj, thr, d_exd.as<int32_t>(),
                               d_queue.as<uint32_t>(), ps, r);
        hipLaunchKernelGGL(core_count, dim3(nb), dim3(256), 0, s, d_exd.as<int32_t>(), n, thr, d_sums.as<uint32_t>());
        hipLaunchKernelGGL(core_scan, dim3(1), dim3(64), 0, s, d_sums.as<uint32_t>(), nb, ps);
        hipLaunchKernelGGL(core_write, dim3(nb), dim3(64), 0, s, d_exd.as<int32_t>(), off, n, thr,
                           g->has_n2 ? (int64_t)0 : (int64_t)ms - 1, d_sums.as<uint32_t>(), d_loc.as<int32_t>(),
                           I.d_orig.as<uint32_t>(), d_deg.as<int32_t>(), d_check.as<uint32_t>(), ps);
        QC_HIP(hipGetLastError());
        QC_HIP(hipMemcpyAsync(&h, ps, sizeof(h), hipMemcpyDeviceToHost, s));
        QC_HIP(hipStreamSynchronize(s));
        if (h.cnt[r] == 0) break;
        if (r + 12 > PEEL_ROUNDS) return QC_OK;
    }
    I.orig.resize(h.R);
    core_deg.resize(h.R);
    std::vector<uint32_t> check(h.n_check);
    if (h.R) {
        QC_HIP(hipMemcpyAsync(I.orig.data(), I.d_orig.p, (size_t)h.R * 4, hipMemcpyDeviceToHost, s));
        QC_HIP(hipMemcpyAsync(core_deg.data(), d_deg.p, (size_t)h.R * 4, hipMemcpyDeviceToHost, s));
    }
    if (h.n_check) QC_HIP(hipMemcpyAsync(check.data(), d_check.p, (size_t)h.n_check * 4, hipMemcpyDeviceToHost, s));
    QC_HIP(hipStreamSynchronize(s));
    if (!check.empty()) {
        std::vector<int> mark(n, -1);
        for (uint32_t v : check)
            if (n2_capped(g, (int)v, mark, ms - 1) < ms - 1) return QC_OK;
    }
    done = true;
    return QC_OK;
}

}  // namespace

int upload_graph(const qc_graph* g, hipStream_t s) {
    DevCSR* d = nullptr;
    return device_csr(g, &d, s);
}

int graph_device_arrays(const qc_graph* g, const uint64_t** off, const uint32_t** adj, hipStream_t s) {
    DevCSR* d = nullptr;
    const int rc = device_csr(g, &d, s);
    if (rc) return rc;
    *off = d->off.as<uint64_t>();
    *adj = d->adj.as<uint32_t>();
    return QC_OK;
}

namespace {
int build_instance_impl(const qc_graph* g, double gamma, int ms, Instance& I, hipStream_t s) {
    const auto t_start = std::chrono::steady_clock::now();
    const int n = g->n;
    I.n = n;
    I.gamma = gamma;
    I.min_size = ms;
    const int thr = (int32_t)std::ceil(gamma * (double)(ms - 1));  // mindeg[min_size]
    int rc;
    I.orig.clear();
    I.root.clear();
    // of the root's vertices, by root-local id: degree in the core
    std::vector<int32_t> exd;
    DevCSR* G = nullptr;
    DBuf d_loc;
    bool on_device = false;
    std::vector<int32_t> loc;  // (host path: in use until its copy has run)
    if (n >= PEEL_DEVICE_MIN || g->adj.size() >= PEEL_DEVICE_ENTRIES) {
        if ((rc = device_csr(g, &G, s))) return rc;
        if ((rc = peel_device(g, *G, thr, ms, I, exd, d_loc, on_device, s))) return rc;
    }
    if (!on_device) {
        peel_host(g, thr, ms, I.orig, exd, loc);
        if (!I.orig.empty()) {
            if ((rc = device_csr(g, &G, s))) return rc;
            if ((rc = d_loc.alloc((size_t)n * 4, s)) || (rc = I.d_orig.alloc(I.orig.size() * 4))) return rc;
            QC_HIP(hipMemcpyAsync(d_loc.p, loc.data(), (size_t)n * 4, hipMemcpyHostToDevice, s));
            QC_HIP(hipMemcpyAsync(I.d_orig.p, I.orig.data(), I.orig.size() * 4, hipMemcpyHostToDevice, s));
        }
    }
    const auto t_host = std::chrono::steady_clock::now();
    const int R = (int)I.orig.size();
    I.R = R;
    I.rw = (R + 63) / 64;
    if (R == 0) return QC_OK;

    // ---- device tables ----
    const size_t mat_bytes = (size_t)R * I.rw * 8;
    if ((rc = I.A1.alloc(mat_bytes))) return rc;
    if ((rc = I.A2.alloc(mat_bytes))) return rc;
    // LDS form: visited map, the 1-hop row and a table of list segments; a
    // byte map (plain stores) up to 32K vertices, a bitmap (atomics) above
    const bool byte_map = n <= 32768;
    const size_t map_words = byte_map ? ((size_t)n + 7) / 8 : ((size_t)n + 63) / 64;
    const size_t map_bytes = (map_words + (size_t)I.rw) * 8;
    int lds_max = 0, cur_dev = 0, n_cu = 0;
    QC_HIP(hipGetDevice(&cur_dev));
    if (hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, cur_dev) != hipSuccess)
        lds_max = 64 * 1024;
    QC_HIP(hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, cur_dev));
    // one workgroup per CU when two maps do not fit: then 16 waves per vertex
    const bool rows_wide = !byte_map && map_bytes * 2 > (size_t)lds_max;
    const int rows_threads = rows_wide ? qcdev::ROWS_THREADS_WIDE : qcdev::ROWS_THREADS;
    const void* rows_kernel = byte_map    ? (const void*)qcdev::root_rows_lds<true, qcdev::ROWS_THREADS>
                              : rows_wide ? (const void*)qcdev::root_rows_lds<false, qcdev::ROWS_THREADS_WIDE>
                                          : (const void*)qcdev::root_rows_lds<false, qcdev::ROWS_THREADS>;
    // the segment table takes what is left (64: the kernel's static LDS), at
    // most four segments a thread or ROWS_TAB_MAX
    const size_t left = map_bytes + 64 < (size_t)lds_max ? ((size_t)lds_max - map_bytes - 64) / 8 : 0;
    const int tab_n = (int)std::min<size_t>(left, std::min(qcdev::ROWS_TAB_MAX, 4 * rows_threads));
    const size_t lds_bytes = map_bytes + (size_t)tab_n * 8;
    bool lds_rows = !g->has_n2 && tab_n >= qcdev::ROWS_TAB_MIN;
    if (lds_rows && lds_bytes > 48 * 1024 &&
        hipFuncSetAttribute(rows_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess)
        lds_rows = false;
    int occ = 0;
    if (lds_rows && (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, rows_kernel, rows_threads, lds_bytes) !=
                         hipSuccess ||
                     occ < 1))
        lds_rows = false;
    if (!lds_rows) {
        QC_HIP(hipMemsetAsync(I.A1.p, 0, mat_bytes, s));
        QC_HIP(hipMemsetAsync(I.A2.p, 0, mat_bytes, s));
    }
    // temporaries carry the stream: released on an error return while the
    // kernels below still run, they are not handed out again before those end
    DBuf d_n2, d_vis, d_next;
    if ((rc = d_n2.alloc((size_t)R * 4, s)) || (rc = I.d_d2r.alloc((size_t)R * 4)) ||
        (rc = I.d_d1r.alloc((size_t)R * 4)))
        return rc;
    int blocks = std::min(R, 2048);
    uint64_t vis_words = ((uint64_t)n + 63) / 64;
    const bool phases = getenv("QCMINE_PHASES") != nullptr;
    auto stamp = [&]() {
        if (phases) (void)hipStreamSynchronize(s);
        return std::chrono::steady_clock::now();
    };
    const auto t_up = stamp();
    if (lds_rows) {
        if ((rc = d_next.alloc(4, s))) return rc;
        QC_HIP(hipMemsetAsync(d_next.p, 0, 4, s));
        const uint64_t* offp = G->off.as<uint64_t>();
        const uint32_t* adjp = G->adj.as<uint32_t>();
        const int32_t* locp = d_loc.as<int32_t>();
        const uint32_t* origp = I.d_orig.as<uint32_t>();
        int32_t Rv = R, rwv = I.rw, nv = n, tabv = tab_n;
        uint64_t* A1p = I.A1.as<uint64_t>();
        uint64_t* A2p = I.A2.as<uint64_t>();
        int32_t* n2p = d_n2.as<int32_t>();
        int32_t* d1p = I.d_d1r.as<int32_t>();
        int32_t* d2p = I.d_d2r.as<int32_t>();
        uint32_t* nextp = d_next.as<uint32_t>();
        void* rargs[] = {(void*)&offp, (void*)&adjp, (void*)&locp, (void*)&origp, (void*)&Rv,  (void*)&rwv, (void*)&nv,
                         (void*)&tabv, (void*)&A1p,  (void*)&A2p,  (void*)&n2p,   (void*)&d1p, (void*)&d2p, (void*)&nextp};
        QC_HIP(hipLaunchKernel(rows_kernel, dim3(std::min(R, occ * n_cu)), dim3(rows_threads), rargs, lds_bytes, s));
    } else {
        if (!g->has_n2) {
            if ((rc = d_vis.alloc((size_t)blocks * vis_words * 8, s))) return rc;
            QC_HIP(hipMemsetAsync(d_vis.p, 0, (size_t)blocks * vis_words * 8, s));
        }
        hipLaunchKernelGGL(qcdev::root_rows, dim3(blocks), dim3(64), 0, s, G->off.as<uint64_t>(),
                           G->adj.as<uint32_t>(), G->off2.as<uint64_t>(), G->adj2.as<uint32_t>(), d_loc.as<int32_t>(),
                           I.d_orig.as<uint32_t>(), R, I.rw, I.A1.as<uint64_t>(), I.A2.as<uint64_t>(),
                           d_n2.as<int32_t>(), d_vis.as<unsigned long long>(), vis_words, g->has_n2 ? 1 : 0);
        hipLaunchKernelGGL(qcdev::root_d2, dim3(blocks), dim3(64), 0, s, I.A2.as<uint64_t>(), I.A1.as<uint64_t>(), R,
                           I.rw, I.d_d2r.as<int32_t>(), I.d_d1r.as<int32_t>());
    }
    QC_HIP(hipGetLastError());
    const auto t_rows = stamp();
    I.d2r.resize(R);
    QC_HIP(hipMemcpyAsync(I.d2r.data(), I.d_d2r.p, (size_t)R * 4, hipMemcpyDeviceToHost, s));
    std::vector<int32_t> n2(R);
    QC_HIP(hipMemcpyAsync(n2.data(), d_n2.p, (size_t)R * 4, hipMemcpyDeviceToHost, s));
    QC_HIP(hipStreamSynchronize(s));
    if (phases) {
        const auto t_dev = std::chrono::steady_clock::now();
        auto ms = [](auto a, auto b) { return std::chrono::duration<double, std::milli>(b - a).count(); };
        fprintf(stderr,
                "[qcmine] root: R=%d filter/peel %.2f ms (%s), device rows %.2f ms (%s; uploads %.2f, rows %.2f, "
                "tables %.2f)\n",
                R, ms(t_start, t_host), on_device ? "device" : "host", ms(t_host, t_dev), lds_rows ? "lds" : "global",
                ms(t_host, t_up), ms(t_up, t_rows), ms(t_rows, t_dev));
    }

    // ---- cover vertex and covered set (main.cu:953-975) ----
    int maxd = 0, maxi = -1, maxl2 = 0;
    for (int a = 0; a < R; a++) {
        if (exd[a] > maxd) {
            maxd = exd[a];
            maxi = a;
        }
        maxl2 = std::max(maxl2, n2[a]);
    }
    std::vector<int32_t> label(R, 0);
    if (maxi >= 0) {
        label[maxi] = 3;
        const uint32_t v = I.orig[maxi];
        for (uint64_t j = g->off[v]; j < g->off[v + 1]; j++) {
            // (input ids ascend with root-local ones)
            const auto it = std::lower_bound(I.orig.begin(), I.orig.end(), g->adj[j]);
            if (it == I.orig.end() || *it != g->adj[j]) continue;
            const size_t la = (size_t)(it - I.orig.begin());
            if (label[la] == 0) label[la] = 2;
        }
    }
    // ---- Q order (main.cu:2059-2104); indeg is 0 for every root vertex ----
    // label rank ascending, then exdeg, |N2| and id descending
    std::vector<int32_t> order(R);
    q_order(R, maxd, maxl2, label, exd, n2, order);
    I.root.resize(R);
    for (int a = 0; a < R; a++) I.root[a] = Vrec{order[a], label[order[a]], 0, exd[order[a]]};

    I.dg.R = R;
    I.dg.rw = I.rw;
    I.dg.A1 = I.A1.as<uint64_t>();
    I.dg.A2 = I.A2.as<uint64_t>();
    I.dg.min_size = ms;
    I.dg.max_d2r = *std::max_element(I.d2r.begin(), I.d2r.end());
    I.dg.gamma = gamma;
    I.dg.orig = I.d_orig.as<uint32_t>();
    I.dg.d2r = I.d_d2r.as<int32_t>();
    I.dg.d1r = I.d_d1r.as<int32_t>();
    I.root_bound = 0;
    I.root_branches = 0;
    for (int a = 0; a < R; a++)
        if (I.root[a].label != 2) I.root_branches++;
    for (int a = 0; a < R; a++) {
        const Vrec& x = I.root[a];
        if (x.label != 1) I.root_bound += std::min<uint64_t>((uint64_t)R, (uint64_t)I.d2r[x.id] + 1);
    }
    return QC_OK;
}

}  // namespace

int build_instance(const qc_graph* g, double gamma, int ms, Instance& I, hipStream_t s) {
    const int rc = build_instance_impl(g, gamma, ms, I, s);
    // an error can leave the root kernels running on the instance's tables:
    // they finish before the caller may release the instance
    if (rc != QC_OK) (void)hipStreamSynchronize(s);
    return rc;
}

int root_window_cut(const Instance& I, long long root_begin, long long root_end, RootCut& c, hipStream_t s) {
    c = RootCut();
    c.b0 = root_begin;
    c.b1 = root_end > 0 ? root_end : -1;
    const int R = I.R;
    if (R == 0) return QC_OK;
    // the window as the expansion resolves it (branches exclude the covered
    // block; a negative start counts from the end)
    const long long nb = (long long)I.root_branches;
    const long long rb0 = root_begin >= 0 ? root_begin : std::max(0ll, nb + root_begin);
    const long long bbeg = std::min(rb0, nb);
    long long bend = nb;
    if (root_end > 0 && root_end < bend) bend = root_end;
    if (bbeg <= 0 || bbeg >= bend) return QC_OK;
    const int ts = R - (int)bbeg;
    // worth a launch only when one wave would scan many row words (kept rows
    // x row words; QCMINE_ROOT_CUT_WORDS overrides the 2^20 threshold)
    long long min_words = 1ll << 20;
    if (const char* e = getenv("QCMINE_ROOT_CUT_WORDS")) min_words = atoll(e);
    if ((long long)ts * I.rw < min_words) return QC_OK;
    // the lookahead of the whole root (main.cu:1349-1405) must fail, since the
    // expansion does not repeat it on the shorter record: every vertex needs
    // |N2 n root| >= R - 1 and indeg + exdeg >= mindeg[R] to pass
    const int req = (int)std::ceil(I.gamma * (double)(R - 1));
    bool passes = true;
    for (const Vrec& v : I.root)
        if (I.d2r[v.id] < R - 1 || v.indeg + v.exdeg < req) {
            passes = false;
            break;
        }
    if (passes) return QC_OK;
    // removed: positions [ts, R) (branches 0 .. bbeg - 1 take them from the end)
    std::vector<uint64_t> mask((size_t)I.rw, 0);
    for (int q = ts; q < R; q++) {
        const uint32_t a = (uint32_t)I.root[q].id;
        mask[a >> 6] |= 1ull << (a & 63);
    }
    std::vector<uint32_t> ids((size_t)ts);
    for (int q = 0; q < ts; q++) ids[q] = (uint32_t)I.root[q].id;
    DBuf d_mask, d_ids, d_cnt;
    int rc;
    if ((rc = d_mask.alloc((size_t)I.rw * 8, s)) || (rc = d_ids.alloc((size_t)ts * 4, s)) ||
        (rc = d_cnt.alloc((size_t)ts * 4, s)))
        return rc;
    QC_HIP(hipMemcpyAsync(d_mask.p, mask.data(), (size_t)I.rw * 8, hipMemcpyHostToDevice, s));
    QC_HIP(hipMemcpyAsync(d_ids.p, ids.data(), (size_t)ts * 4, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(qcdev::root_cut_deg, dim3(std::min(ts, 8192)), dim3(64), 0, s, I.A1.as<uint64_t>(), I.rw,
                       d_ids.as<uint32_t>(), ts, d_mask.as<uint64_t>(), d_cnt.as<int32_t>());
    QC_HIP(hipGetLastError());
    std::vector<int32_t> cnt((size_t)ts), d1r((size_t)R);
    QC_HIP(hipMemcpyAsync(cnt.data(), d_cnt.p, (size_t)ts * 4, hipMemcpyDeviceToHost, s));
    QC_HIP(hipMemcpyAsync(d1r.data(), I.d_d1r.p, (size_t)R * 4, hipMemcpyDeviceToHost, s));
    QC_HIP(hipStreamSynchronize(s));
    c.rec.assign(I.root.begin(), I.root.begin() + ts);
    for (int q = 0; q < ts; q++) c.rec[q].exdeg -= cnt[q];
    // removal k scans N(r) of root vertex r at position R - k (main.cu:
    // 1437-1450); the lookahead scanned N2 of every root vertex (1373-1381)
    for (int q = ts; q < R; q++) {
        const int a = I.root[q].id;
        c.w_adj += (uint64_t)d1r[a] + (uint64_t)I.d2r[a];
    }
    c.cut = (int32_t)bbeg;
    c.b0 = 0;
    c.b1 = bend - bbeg;
    return QC_OK;
}

}  // namespace qc
