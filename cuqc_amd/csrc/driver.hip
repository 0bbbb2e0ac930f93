// driver.hip -- the plain (level-synchronous) enumeration: the structure of
// the reference's search() loop (main.cu:606-678) on the device.
//
// Tasks wait on two LIFO stacks (vertex pool in HBM, task refs mirrored on
// the host): tasks of at most `TL` vertices, launched with many waves per CU,
// and larger ones, launched with a quarter of a CU's LDS and an HBM slab per
// wave.  Each
// host iteration pops a batch from the top of one stack (large first), runs
// one launch, and pushes the children it wrote back on top, so the search
// proceeds depth-first in batches, like the reference's width-bounded levels
// with the LIFO overflow buffer (main.cu:2926-2931).  Raw cliques stream into
// an HBM buffer that is drained to the host when more than half full
// (CLIQUES_DUMP, main.cu:56).

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <chrono>
#include <cstring>

#include "qc_internal.h"

namespace qcdev {
__global__ void expand_level(const ExpandArgs*);
}  // namespace qcdev

namespace qc {

namespace {

struct Stack {
    DBuf verts;                    // Vrec pool
    uint64_t cap = 0;              // slots
    uint64_t top = 0;              // slots in use
    std::vector<TaskRef> refs;     // host mirror, increasing off
};

}  // namespace

int enumerate_plain(const Instance& I, const qc_params& p, EnumOut& out, hipStream_t s) {
    int rc;
    out = EnumOut();
    if (I.R == 0) return QC_OK;
    const uint32_t TL = p.lds_tile == 64 ? 64 : p.lds_tile == 256 ? 256 : 128;

    // slot bound of the root's children inside the search window: branch b
    // takes root vertex R - 1 - b and writes at most min(R - b, 1 + |N2 n root|)
    // vertices
    uint64_t root_bound = 0;
    {
        const long long nb = (long long)I.root_branches;
        long long b0 = p.root_begin >= 0 ? p.root_begin : std::max(0ll, nb + (long long)p.root_begin);
        long long b1 = p.root_end > 0 ? std::min<long long>(p.root_end, nb) : nb;
        b0 = std::min(b0, nb);
        for (long long b = b0; b < b1; b++) {
            const Vrec& x = I.root[(size_t)(I.R - 1 - b)];
            root_bound += std::min<uint64_t>((uint64_t)(I.R - b), (uint64_t)I.d2r[x.id] + 1);
        }
    }

    // ---- capacities ----
    size_t freeb = 0, totalb = 0;
    QC_HIP(hipMemGetInfo(&freeb, &totalb));
    {
        int d = 0;
        QC_HIP(hipGetDevice(&d));
        freeb += pool_cached_bytes(d);
    }
    // Buffers start at 64 MB (what the block cache recycles), or near what the
    // root needs, and grow on demand up to a
    // budget; task_capacity / clique_capacity pin them instead.
    const size_t budget = std::min<size_t>(freeb / 2, (size_t)96 << 30);
    const uint64_t max_slots = budget / 5 / sizeof(Vrec);
    uint64_t stg_slot_cap = p.task_capacity ? p.task_capacity
                                            : std::min<uint64_t>(max_slots, std::max<uint64_t>(4ull << 20, 2 * root_bound));
    uint64_t pool_cap = p.task_capacity ? p.task_capacity : stg_slot_cap;
    const bool grow = p.task_capacity == 0;
    // (a child holds two vertices or more, an item's share of its task two slots:
    // refs for half the slots are enough, and not one more keeps them, and the
    // clique refs below, at the block size that is recycled: allocating and freeing
    // three larger ones was 1.2 ms of a 3.7 ms call)
    const uint64_t more = p.task_capacity ? 4096 : 0;
    uint64_t stage_refs = std::min<uint64_t>(stg_slot_cap / 2 + more, (uint64_t)128 << 20);
    uint64_t clq_slots = p.clique_capacity ? p.clique_capacity : (16ull << 20);
    if (const char* ic = getenv("QCMINE_INITIAL_CAPACITY"))  // tests: launches made again
        if (!p.clique_capacity && atoll(ic) > 0) clq_slots = std::min<uint64_t>(clq_slots, 8 * (uint64_t)atoll(ic));
    uint64_t clq_refs = std::min<uint64_t>(clq_slots / 4 + (p.clique_capacity ? 4096 : 0), (uint64_t)64 << 20);

    Stack st[2];
    for (int k = 0; k < 2; k++) {
        st[k].cap = pool_cap;
        if ((rc = st[k].verts.alloc(st[k].cap * sizeof(Vrec)))) return rc;
    }
    DBuf stg_refs[2], stg_verts[2];
    for (int k = 0; k < 2; k++) {
        if ((rc = stg_refs[k].alloc(stage_refs * sizeof(TaskRef)))) return rc;
        if ((rc = stg_verts[k].alloc(stg_slot_cap * sizeof(Vrec)))) return rc;
    }
    DBuf d_clq_refs, d_clq_verts, d_stats, d_launch;
    if ((rc = d_clq_refs.alloc(clq_refs * sizeof(CliqueRef)))) return rc;
    if ((rc = d_clq_verts.alloc(clq_slots * 4))) return rc;
    if ((rc = d_stats.alloc(sizeof(DevStats)))) return rc;
    const uint32_t max_batch = 1u << 16;
    // one launch's counters, arguments and task refs, sent with one copy
    struct Launch {
        LevelState st;
        ExpandArgs a;
    };
    const size_t refs_at = (sizeof(Launch) + 63) & ~(size_t)63;
    if ((rc = d_launch.alloc(refs_at + (size_t)max_batch * sizeof(TaskRef)))) return rc;
    std::vector<char> launch_mem(refs_at + (size_t)max_batch * sizeof(TaskRef) + alignof(Launch));
    char* const launch =
        (char*)(((uintptr_t)launch_mem.data() + alignof(Launch) - 1) & ~(uintptr_t)(alignof(Launch) - 1));
    Launch* const L = (Launch*)launch;
    Launch* const dL = d_launch.as<Launch>();
    LevelState done{};  // counters after the last launch
    QC_HIP(hipMemsetAsync(d_stats.p, 0, sizeof(DevStats), s));

    int dev = 0;
    QC_HIP(hipGetDevice(&dev));
    int n_cu = 0;
    QC_HIP(hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev));
    // HBM slabs, one per wave of a large-task launch: 4 waves per CU, as many as
    // LARGE_LDS allows.  Small tasks fit SMALL_LDS (a task of 64 vertices' children;
    // the arrays of up to 256 vertices with any rows that are staged).
    constexpr size_t LARGE_LDS = 79 * 512, SMALL_LDS = 64 * 256;
    const size_t slab_b = wide_slab_bytes((uint32_t)I.R);
    uint32_t n_slabs = (uint32_t)std::max(1, n_cu) * 4;
    while (n_slabs > 1 && (size_t)n_slabs * slab_b > budget / 8) n_slabs >>= 1;
    const uint32_t small_grid_max =
        p.workgroups > 0 ? (uint32_t)p.workgroups : (uint32_t)std::max(1, n_cu) * 16;
    // (a small task only needs its slab for degrees beyond the LDS form's fields)
    const size_t small_slab_b = wide_slab_bytes(std::min<uint32_t>(TL, (uint32_t)I.R));
    DBuf d_slab;
    if ((rc = d_slab.alloc(std::max((size_t)n_slabs * slab_b, (size_t)small_grid_max * small_slab_b)))) return rc;

    // ---- root ----
    // (a window's leading removals applied at once when they are many)
    RootCut cut;
    if ((rc = root_window_cut(I, p.root_begin, p.root_end, cut, s))) return rc;
    const std::vector<Vrec>& rrec = cut.cut ? cut.rec : I.root;
    const int rt = (int)rrec.size();
    {
        const int k = rt <= (int)TL ? 0 : 1;
        QC_HIP(hipMemcpyAsync(st[k].verts.p, rrec.data(), rrec.size() * sizeof(Vrec), hipMemcpyHostToDevice, s));
        TaskRef r{0, (uint32_t)rt, 0, 0, root_bound, 0, 0};
        st[k].refs.push_back(r);
        st[k].top = (uint64_t)rt;
    }

    ExpandArgs A;
    memset(&A, 0, sizeof(A));
    A.g = I.dg;
    A.static_sched = p.scheduling != 0;
    A.task_counter = &dL->st.next_task;
    for (int k = 0; k < 2; k++) {
        A.out_refs[k] = stg_refs[k].as<TaskRef>();
        A.out_verts[k] = stg_verts[k].as<Vrec>();
        A.out_ref_cap[k] = stage_refs;
        A.out_vert_cap[k] = stg_slot_cap;
    }
    A.out_ctr = dL->st.out;
    A.small_max = TL;
    A.clq_refs = d_clq_refs.as<CliqueRef>();
    A.clq_verts = d_clq_verts.as<uint32_t>();
    A.clq_ctr = &dL->st.clq;
    A.clq_ref_cap = clq_refs;
    A.clq_vert_cap = clq_slots;
    A.slab = d_slab.as<char>();
    A.slab_bytes = slab_b;
    A.slab_tcap = (uint32_t)I.R;
    A.stats = d_stats.as<DevStats>();
    A.error = &dL->st.error;
    // Tasks above the small size are split into items of at most 64 branches,
    // fewer when a launch has few of them (below): on one wave each, the six
    // first-level tasks of a co-expression window kept 6 of 1,024 waves busy
    // for most of its 87 ms (now 6).  Not under a caller's capacities, whose
    // launches stay as they are without: a split record stays on the stack
    // until its last item ran.
    const bool fixed = !grow || p.clique_capacity != 0;
    A.all_bounds = fixed;
    const int split = fixed || p.split_chunk < 0 ? 0 : (p.split_chunk == 0 ? 64 : p.split_chunk);
    A.split_min_t = (uint32_t)std::max<int>((int)TL, p.split_min);
    A.n_roots = 1;
    A.split_waves = n_slabs;
    A.g.root_b0 = cut.b0;
    A.g.root_b1 = cut.b1;
    A.g.root_cut = cut.cut;
    A.g.max_depth = p.max_depth > 0 ? p.max_depth : -1;

    hipEvent_t e0, e1;
    QC_HIP(hipEventCreate(&e0));
    QC_HIP(hipEventCreate(&e1));
    double kms = 0;
    std::vector<CliqueRef> hrefs;
    std::vector<uint32_t> hverts;

    // brings the clique stream to the host (done.clq holds its counters)
    auto drain = [&](bool force) -> int {
        const StreamCtr cc = done.clq;
        if (!force && cc.slots * 2 < clq_slots && cc.items * 2 < clq_refs) return QC_OK;
        if (cc.items == 0) return QC_OK;
        hrefs.resize(cc.items);
        hverts.resize(cc.slots);
        QC_HIP(hipMemcpyAsync(hrefs.data(), d_clq_refs.p, cc.items * sizeof(CliqueRef), hipMemcpyDeviceToHost, s));
        QC_HIP(hipMemcpyAsync(hverts.data(), d_clq_verts.p, cc.slots * 4, hipMemcpyDeviceToHost, s));
        QC_HIP(hipStreamSynchronize(s));
        for (auto& r : hrefs) {
            out.raw.v.insert(out.raw.v.end(), hverts.begin() + r.off, hverts.begin() + r.off + r.len);
            out.raw.off.push_back(out.raw.v.size());
        }
        done.clq = StreamCtr{0, 0};
        return QC_OK;
    };

    // QCMINE_DEBUG=1: the reference's per-level size report on stdout
    const bool debug = getenv("QCMINE_DEBUG") && atoi(getenv("QCMINE_DEBUG")) > 0;
    struct {
        uint64_t tasks = 0, buf = 0, buf_off = 0, clq = 0, clq_off = 0, child = 0, child_off = 0;
    } mx;
    std::vector<TaskRef> batch, kids[2];
    // a launch whose raw sets overflow the stream is made again with half the
    // tasks (its counters and the stream put back), down to one task on an empty
    // stream
    uint32_t most = max_batch;
    DBuf d_keep;
    if ((rc = d_keep.alloc(sizeof(DevStats)))) return rc;
    while (!st[0].refs.empty() || !st[1].refs.empty()) {
        const int k = st[1].refs.empty() ? 0 : 1;
        Stack& S = st[k];
        // batch from the top: bounded count, children fit the staging buffers
        const uint32_t bmax = std::min(most, k == 1 ? n_slabs : std::min<uint32_t>(max_batch, small_grid_max * 4));
        uint64_t vol = 0, branches = 0;
        size_t take = 0;
        while (take < S.refs.size() && take < bmax) {
            const TaskRef& r = S.refs[S.refs.size() - 1 - take];
            // (a task to be split writes its record instead of children, and at
            // most a ref per vertex: the staging holds half as many refs as slots)
            const uint64_t need = split && k == 1 && r.b1 == 0 ? std::max<uint64_t>(r.bound, 2ull * r.t) : r.bound;
            if (take > 0 && vol + need > stg_slot_cap) break;
            if (need > stg_slot_cap) {
                uint64_t want = std::max<uint64_t>(need, 2 * stg_slot_cap);
                if (!grow || need > max_slots) {
                    set_error("task of %u vertices needs %llu child slots, staging holds %llu", r.t,
                              (unsigned long long)need, (unsigned long long)stg_slot_cap);
                    return QC_EOVERFLOW;
                }
                stg_slot_cap = std::min(want, max_slots);
                stage_refs = std::min<uint64_t>(stg_slot_cap / 2 + more, (uint64_t)128 << 20);
                for (int j = 0; j < 2; j++) {
                    stg_verts[j].release();
                    stg_refs[j].release();
                    if ((rc = stg_verts[j].alloc(stg_slot_cap * sizeof(Vrec)))) return rc;
                    if ((rc = stg_refs[j].alloc(stage_refs * sizeof(TaskRef)))) return rc;
                    A.out_refs[j] = stg_refs[j].as<TaskRef>();
                    A.out_verts[j] = stg_verts[j].as<Vrec>();
                    A.out_ref_cap[j] = stage_refs;
                    A.out_vert_cap[j] = stg_slot_cap;
                }
            }
            vol += need;
            branches += r.b1 ? r.b1 - r.b0 : r.t;
            take++;
        }
        batch.assign(S.refs.end() - take, S.refs.end());
        S.refs.resize(S.refs.size() - take);
        const uint64_t base = batch.front().off;
        A.in_refs = (const TaskRef*)(d_launch.as<char>() + refs_at);
        A.in_verts = S.verts.as<Vrec>();
        A.n_in = (uint32_t)take;
        A.lds_bytes = (uint32_t)(k == 1 ? LARGE_LDS : SMALL_LDS);
        A.slab_bytes = k == 1 ? slab_b : small_slab_b;
        // items: about one per wave over the launch's branches
        A.split_chunk = split && k == 1 ? (int)std::max<uint64_t>(1, std::min<uint64_t>((uint64_t)split, branches / n_slabs)) : 0;
        L->st = LevelState{{{0, 0}, {0, 0}}, done.clq, 0, 0};
        L->a = A;
        memcpy(launch + refs_at, batch.data(), take * sizeof(TaskRef));
        QC_HIP(hipMemcpyAsync(d_launch.p, launch, refs_at + take * sizeof(TaskRef), hipMemcpyHostToDevice, s));
        if (!fixed) QC_HIP(hipMemcpyAsync(d_keep.p, d_stats.p, sizeof(DevStats), hipMemcpyDeviceToDevice, s));
        QC_HIP(hipEventRecord(e0, s));
        const uint32_t grid = std::min<uint32_t>((uint32_t)take, k == 1 ? n_slabs : small_grid_max);
        hipLaunchKernelGGL(qcdev::expand_level, dim3(grid), dim3(64), k == 1 ? LARGE_LDS : SMALL_LDS, s, &dL->a);
        QC_HIP(hipGetLastError());
        QC_HIP(hipEventRecord(e1, s));
        LevelState ls;
        QC_HIP(hipMemcpyAsync(&ls, &dL->st, sizeof(ls), hipMemcpyDeviceToHost, s));
        QC_HIP(hipStreamSynchronize(s));
        const StreamCtr* oc = ls.out;
        float ms = 0;
        QC_HIP(hipEventElapsedTime(&ms, e0, e1));
        kms += ms;
        if (ls.error == 1 && !fixed && (take > 1 || done.clq.items > 0) &&
            (ls.clq.slots > clq_slots || ls.clq.items > clq_refs)) {
            QC_HIP(hipMemcpyAsync(d_stats.p, d_keep.p, sizeof(DevStats), hipMemcpyDeviceToDevice, s));
            S.refs.insert(S.refs.end(), batch.begin(), batch.end());
            most = (uint32_t)std::max<size_t>(1, take / 2);
            if ((rc = drain(true))) return rc;
            continue;
        }
        most = max_batch;
        out.levels++;
        if (ls.error) {
            set_error("expansion buffers overflowed (error flags %d); raise task_capacity / clique_capacity", ls.error);
            return QC_EOVERFLOW;
        }
        done = ls;
        // (a split record stays while items of it wait)
        S.top = !S.refs.empty() && S.refs.back().b1 > 0 && S.refs.back().off == base ? base + batch.front().t : base;
        // push children: staging stream j -> stack j
        for (int j = 0; j < 2; j++) {
            if (oc[j].items == 0) continue;
            Stack& D = st[j];
            if (D.top + oc[j].slots > D.cap && grow && D.cap < max_slots) {
                uint64_t ncap = std::min<uint64_t>(max_slots, std::max<uint64_t>(2 * D.cap, D.top + oc[j].slots));
                DBuf nb;
                if ((rc = nb.alloc(ncap * sizeof(Vrec)))) return rc;
                if (D.top) QC_HIP(hipMemcpyAsync(nb.p, D.verts.p, D.top * sizeof(Vrec), hipMemcpyDeviceToDevice, s));
                QC_HIP(hipStreamSynchronize(s));
                D.verts.swap(nb);
                D.cap = ncap;
            }
            if (D.top + oc[j].slots > D.cap) {
                set_error("task stack overflow (%llu + %llu slots > %llu)", (unsigned long long)D.top,
                          (unsigned long long)oc[j].slots, (unsigned long long)D.cap);
                return QC_EOVERFLOW;
            }
            kids[j].resize(oc[j].items);
            QC_HIP(hipMemcpyAsync(kids[j].data(), stg_refs[j].p, oc[j].items * sizeof(TaskRef), hipMemcpyDeviceToHost, s));
            QC_HIP(hipMemcpyAsync(D.verts.as<Vrec>() + D.top, stg_verts[j].p, oc[j].slots * sizeof(Vrec),
                                  hipMemcpyDeviceToDevice, s));
        }
        if (oc[0].items || oc[1].items) QC_HIP(hipStreamSynchronize(s));
        uint64_t n_kids = 0, kid_slots = 0;  // children (items are parts of their task)
        for (int j = 0; j < 2; j++) {
            if (oc[j].items == 0) continue;
            Stack& D = st[j];
            // (items of one record stay together: their order among themselves is free)
            std::sort(kids[j].begin(), kids[j].end(), [](const TaskRef& x, const TaskRef& y) { return x.off < y.off; });
            for (auto& r : kids[j]) {
                if (r.b1 == 0) {
                    n_kids++;
                    kid_slots += r.t;
                }
                r.off += D.top;
                D.refs.push_back(r);
            }
            D.top += oc[j].slots;
        }
        if (debug) {
            // the reference's debug size report (main.cu:2635-2646): level,
            // tasks expanded (records, vertex slots), children written,
            // records waiting on the host stacks, raw cliques held
            const StreamCtr cc = done.clq;
            uint64_t bslots = 0, n_tasks = 0;
            for (const TaskRef& r : batch)
                if (r.b1 == 0) {
                    n_tasks++;
                    bslots += r.t;
                }
            if (out.levels == 1) bslots += (uint64_t)cut.cut;  // the root as built
            const uint64_t wrefs = st[0].refs.size() + st[1].refs.size(), wslots = st[0].top + st[1].top;
            printf("L: %llu T1: %llu %llu T2: %llu %llu B: %llu %llu C: %llu %llu\n\n", (unsigned long long)out.levels,
                   (unsigned long long)n_tasks, (unsigned long long)bslots, (unsigned long long)n_kids,
                   (unsigned long long)kid_slots,
                   (unsigned long long)wrefs, (unsigned long long)wslots, cc.items, cc.slots);
            mx.tasks = std::max<uint64_t>(mx.tasks, bslots);
            mx.buf = std::max<uint64_t>(mx.buf, wslots);
            mx.buf_off = std::max<uint64_t>(mx.buf_off, wrefs);
            mx.clq = std::max<uint64_t>(mx.clq, cc.slots);
            mx.clq_off = std::max<uint64_t>(mx.clq_off, cc.items);
            mx.child = std::max<uint64_t>(mx.child, kid_slots);
            mx.child_off = std::max<uint64_t>(mx.child_off, n_kids);
        }
        if ((rc = drain(false))) return rc;
    }
    if ((rc = drain(true))) return rc;
    if (debug) {
        // print_maxes (main.cu:2893-2907): the largest of each buffer over the run
        printf("\nTASKS SIZE: %llu\nBUFFER SIZE: %llu\nBUFFER OFFSET SIZE: %llu\nCLIQUES SIZE: %llu\n"
               "CLIQUES OFFSET SIZE: %llu\nWTASKS SIZE: %llu\nWTASKS OFFSET SIZE: %llu\n\n",
               (unsigned long long)mx.tasks, (unsigned long long)mx.buf, (unsigned long long)mx.buf_off,
               (unsigned long long)mx.clq, (unsigned long long)mx.clq_off, (unsigned long long)mx.child,
               (unsigned long long)mx.child_off);
        fflush(stdout);
    }
    QC_HIP(hipMemcpyAsync(&out.ds, d_stats.p, sizeof(DevStats), hipMemcpyDeviceToHost, s));
    QC_HIP(hipStreamSynchronize(s));
    root_cut_counters(cut, I.R, TL, out.ds);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    out.kernel_ms = kms;
    return QC_OK;
}

}  // namespace qc
