// collect.hip -- the raw sets of a persistent launch, brought to the host.
//
// The expansion kernels append raw sets to one clique stream (a ref
// {off, len, inst} per set, its vertices at off) in whatever order the waves
// finish them.  The reference copies its device clique buffer to the host
// and appends it to temp.txt after the enumeration timer stops
// (dump_cliques, main.cu:688, 1234-1246).  Here the sets are put in order on
// the device -- instances one after another, each instance's sets in the
// order of their vertex slots -- and packed into one contiguous array, so
// the host receives two finished arrays (offsets, vertices) and does no
// sorting or copying of its own:
// Refs that a wave took and did not use (inst CLQ_NONE) sort last.
//   1. key = inst << 40 | off per ref, radix sort of (key, ref index);
//   2. set lengths in that order, exclusive scan -> output offsets;
//   3. the vertices are gathered in that order, straight into the host's block
//      when it is pinned.

#include <cstring>

#include <rocprim/rocprim.hpp>

#include <vector>

#include "qc_internal.h"

namespace qcdev {

__global__ void rc_keys(const CliqueRef* __restrict__ refs, uint64_t k, uint64_t* __restrict__ keys,
                        uint32_t* __restrict__ idx) {
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= k) return;
    const CliqueRef r = refs[i];
    // (instances are numbered below 65535)
    keys[i] = r.inst == CLQ_NONE ? (1ull << 56) - 1 : ((uint64_t)r.inst << 40) | r.off;
    idx[i] = (uint32_t)i;
}

__global__ void rc_lens(const CliqueRef* __restrict__ refs, const uint32_t* __restrict__ sidx, uint64_t k,
                        CliqueRef* __restrict__ sets, uint64_t* __restrict__ lens) {
    const uint64_t j = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (j < k) {
        const CliqueRef r = refs[sidx[j]];
        sets[j] = r;
        lens[j] = r.len;
    }
    if (j == k) lens[k] = 0;
}

// 256 consecutive sets a workgroup; its threads take the places of their output
// one after another (reads and writes of neighbouring words), each finding its
// set among the offsets in LDS.  `out` may be host memory: the link's rate
// bounds the kernel then (57 GB/s; 194 MB of a full search 3.4 ms, against
// 1.2 for a thread per set into a device buffer, 3.4 for the copy and 0.4 for
// the buffer).
constexpr int RC_SETS = 256;
__global__ __launch_bounds__(RC_SETS) void rc_gather(const CliqueRef* __restrict__ sets, const uint64_t* __restrict__ oo,
                                                     uint64_t k, const uint32_t* __restrict__ v, uint32_t* out) {
    __shared__ uint32_t at[RC_SETS + 1];
    __shared__ uint64_t from[RC_SETS];
    const uint64_t j0 = (uint64_t)blockIdx.x * RC_SETS;
    const int n = (int)min((uint64_t)RC_SETS, k - j0);
    const uint64_t o0 = oo[j0];
    const int t = threadIdx.x;
    if (t < n) {
        from[t] = sets[j0 + t].off;
        at[t] = (uint32_t)(oo[j0 + t] - o0);
    }
    if (t == 0) at[n] = (uint32_t)(oo[j0 + n] - o0);
    __syncthreads();
    const uint32_t total = at[n];
    for (uint32_t p = t; p < total; p += RC_SETS) {
        int lo = 0, hi = n;  // at[lo] <= p < at[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (at[mid] <= p)
                lo = mid;
            else
                hi = mid;
        }
        out[o0 + p] = v[from[lo] + (p - at[lo])];
    }
}

}  // namespace qcdev

namespace qc {

#define QC_RC(x)                                                            \
    do {                                                                    \
        if ((x) != hipSuccess) {                                            \
            set_error("raw set collection: %s failed", #x);                 \
            return QC_EDEVICE;                                              \
        }                                                                   \
    } while (0)

int collect_raw(const CliqueRef* d_refs, uint64_t taken, const uint32_t* d_verts, uint64_t k, uint64_t nv,
                RawSets& raw, DBuf& sets, hipStream_t s) {
    if (k == 0) return QC_OK;
    if (taken >= 0xFFFFFFFFull || nv >= (1ull << 40)) {
        set_error("raw set collection: %llu sets of %llu vertices exceed the key fields", (unsigned long long)k,
                  (unsigned long long)nv);
        return QC_EOVERFLOW;
    }
    if (k > taken) {
        set_error("raw set collection: %llu sets in %llu refs", (unsigned long long)k, (unsigned long long)taken);
        return QC_EDEVICE;
    }
    size_t sort_b = 0, scan_b = 0;
    QC_RC(rocprim::radix_sort_pairs(nullptr, sort_b, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint32_t*)nullptr,
                                    (uint32_t*)nullptr, (size_t)taken, 0, 56, s));
    QC_RC(rocprim::exclusive_scan(nullptr, scan_b, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint64_t)0, (size_t)k + 1,
                                  rocprim::plus<uint64_t>(), s));
    DBuf keys, skeys, idx, sidx, lens, oo, out, temp;
    int rc;
    if ((rc = keys.alloc(taken * 8, s)) || (rc = skeys.alloc(taken * 8, s)) || (rc = idx.alloc(taken * 4, s)) ||
        (rc = sidx.alloc(taken * 4, s)) || (rc = lens.alloc((k + 1) * 8, s)) || (rc = oo.alloc((k + 1) * 8, s)) ||
        (rc = sets.alloc(k * sizeof(CliqueRef), s)) ||
        (rc = temp.alloc(std::max(sort_b, scan_b), s)))
        return rc;
    const unsigned nt = (unsigned)((taken + 255) / 256);
    const unsigned nb = (unsigned)((k + 256) / 256);
    hipLaunchKernelGGL(qcdev::rc_keys, dim3(nt), dim3(256), 0, s, d_refs, taken, keys.as<uint64_t>(),
                       idx.as<uint32_t>());
    QC_RC(hipGetLastError());
    QC_RC(rocprim::radix_sort_pairs(temp.p, sort_b, keys.as<uint64_t>(), skeys.as<uint64_t>(), idx.as<uint32_t>(),
                                    sidx.as<uint32_t>(), (size_t)taken, 0, 56, s));
    hipLaunchKernelGGL(qcdev::rc_lens, dim3(nb), dim3(256), 0, s, d_refs, sidx.as<uint32_t>(), k,
                       sets.as<CliqueRef>(), lens.as<uint64_t>());
    QC_RC(hipGetLastError());
    QC_RC(rocprim::exclusive_scan(temp.p, scan_b, lens.as<uint64_t>(), oo.as<uint64_t>(), (uint64_t)0, (size_t)k + 1,
                                  rocprim::plus<uint64_t>(), s));
    if ((rc = raw.off_buf.alloc((k + 1) * 8)) || (rc = raw.v_buf.alloc(std::max<uint64_t>(nv, 1) * 4))) return rc;
    void* to = nullptr;
    if (raw.v_buf.pinned && hipHostGetDevicePointer(&to, raw.v_buf.p, 0) != hipSuccess) {
        (void)hipGetLastError();
        to = nullptr;
    }
    if (!to && (rc = out.alloc(std::max<uint64_t>(nv, 1) * 4, s))) return rc;
    raw.k = k;
    raw.nv = nv;
    QC_RC(hipMemcpyAsync(raw.off_buf.p, oo.p, (k + 1) * 8, hipMemcpyDeviceToHost, s));
    auto check = [&]() -> int {
        if (raw.offp()[k] == nv) return QC_OK;
        set_error("raw set collection: the sets hold %llu vertex slots, the stream %llu",
                  (unsigned long long)raw.offp()[k], (unsigned long long)nv);
        return QC_EDEVICE;
    };
    if (to) {  // (looked at before anything is written to the host's block)
        QC_RC(hipStreamSynchronize(s));
        if ((rc = check())) return rc;
    }
    hipLaunchKernelGGL(qcdev::rc_gather, dim3((unsigned)((k + qcdev::RC_SETS - 1) / qcdev::RC_SETS)), dim3(qcdev::RC_SETS),
                       0, s, sets.as<CliqueRef>(), oo.as<uint64_t>(), k, d_verts, to ? (uint32_t*)to : out.as<uint32_t>());
    QC_RC(hipGetLastError());
    if (!to) QC_RC(hipMemcpyAsync(raw.v_buf.p, out.p, nv * 4, hipMemcpyDeviceToHost, s));
    QC_RC(hipStreamSynchronize(s));
    if ((rc = check())) return rc;
    return QC_OK;
}

}  // namespace qc
