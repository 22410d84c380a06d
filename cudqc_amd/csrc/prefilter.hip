// Device pass before the maximal-set filter (reference src/Quick_rmnonmax.cpp): drops raw
// cliques that are duplicates or one vertex short of another raw clique. Compiled as part of
// engine.hip's translation unit.
//
// Nearly all raw cliques of a batch are such (804,465 raw cliques of 64 graphs hold 37,884
// maximal sets): a branch that emits a clique goes on to children that emit it with one more
// vertex. Fetching all of them and walking them into a trie on the host took 225 ms for
// that batch, against 35 ms for its enumeration. The hash of a set is the sum of a mix of
// its ids, so the hash of a set without one of its vertices is one subtraction: every clique
// looks its one-smaller subsets up in a hash table of all cliques. Bound by the random
// accesses to that table (one probe per id of every clique): 2.3 ms for
// 330,558 cliques, and the result dump of the 804,465 takes 44 ms instead of 225. A hash hit
// counts only after the ids were compared. What has no neighbour of one vertex more is left
// to the host's filter, which gives the same maximal sets from fewer cliques.
#include "prefilter.hpp"

namespace {

constexpr uint32_t NO_SET = 0xFFFFFFFFu;
constexpr uint32_t PREFILTER_LEAST = 4096;  // fewer cliques than this: the host filter is faster alone

__device__ __forceinline__ unsigned long long set_mix(uint32_t id) {  // splitmix64 finaliser
    unsigned long long x = ((unsigned long long)id + 1ull) * 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__global__ __launch_bounds__(256) void set_hash_kernel(const int32_t* __restrict__ ids,
                                                       const unsigned long long* __restrict__ meta, uint32_t n,
                                                       unsigned long long* __restrict__ hash, uint8_t* __restrict__ dead,
                                                       uint32_t* __restrict__ table, uint32_t slots) {
    const uint32_t step = gridDim.x * 256u, first = blockIdx.x * 256u + threadIdx.x;
    for (uint32_t i = first; i < slots; i += step) table[i] = NO_SET;
    for (uint32_t s = first; s < n; s += step) {
        const unsigned long long off = meta[s] >> 24;
        const uint32_t len = (uint32_t)(meta[s] & 0xFFFFFFull);
        unsigned long long h = 0;
        for (uint32_t i = 0; i < len; ++i) h += set_mix((uint32_t)ids[off + i]);
        hash[s] = h;
        dead[s] = 0;
    }
}

// Every id of a[0, la) among b[0, lb) (distinct ids in each).
__device__ __forceinline__ bool subset_of(const int32_t* a, uint32_t la, const int32_t* b, uint32_t lb) {
    for (uint32_t i = 0; i < la; ++i) {
        bool found = false;
        for (uint32_t j = 0; j < lb && !found; ++j) found = a[i] == b[j];
        if (!found) return false;
    }
    return true;
}

// Puts every set into the table (linear probing); one that equals a set already there is dead.
__global__ __launch_bounds__(256) void set_insert_kernel(const int32_t* __restrict__ ids,
                                                         const unsigned long long* __restrict__ meta, uint32_t n,
                                                         const unsigned long long* __restrict__ hash,
                                                         uint8_t* __restrict__ dead, uint32_t* table, uint32_t slots) {
    for (uint32_t s = blockIdx.x * 256u + threadIdx.x; s < n; s += gridDim.x * 256u) {
        const unsigned long long h = hash[s], m = meta[s];
        uint32_t at = (uint32_t)(h >> 20) & (slots - 1);
        while (true) {  // (the table has twice as many slots as sets, so a free one is met)
            const uint32_t t = atomicCAS(&table[at], NO_SET, s);
            if (t == NO_SET) break;
            if (hash[t] == h && ((meta[t] ^ m) & 0xFFFFFFull) == 0 &&
                subset_of(ids + (m >> 24), (uint32_t)(m & 0xFFFFFFull), ids + (meta[t] >> 24), (uint32_t)(m & 0xFFFFFFull))) {
                dead[s] = 1;
                break;
            }
            at = (at + 1) & (slots - 1);
        }
    }
}

// Marks, for every set, the sets that lack exactly one of its vertices.
__global__ __launch_bounds__(256) void set_mark_kernel(const int32_t* __restrict__ ids,
                                                       const unsigned long long* __restrict__ meta, uint32_t n,
                                                       const unsigned long long* __restrict__ hash, uint8_t* dead,
                                                       const uint32_t* __restrict__ table, uint32_t slots) {
    for (uint32_t s = blockIdx.x * 256u + threadIdx.x; s < n; s += gridDim.x * 256u) {
        const unsigned long long off = meta[s] >> 24, h = hash[s];
        const uint32_t len = (uint32_t)(meta[s] & 0xFFFFFFull);
        for (uint32_t i = 0; i < len; ++i) {
            const unsigned long long want = h - set_mix((uint32_t)ids[off + i]);
            for (uint32_t at = (uint32_t)(want >> 20) & (slots - 1);; at = (at + 1) & (slots - 1)) {
                const uint32_t t = table[at];
                if (t == NO_SET) break;
                if (hash[t] != want || (uint32_t)(meta[t] & 0xFFFFFFull) + 1u != len) continue;
                if (!dead[t] && subset_of(ids + (meta[t] >> 24), len - 1, ids + off, len)) dead[t] = 1;
            }
        }
    }
}

// Copies the sets that are left (out_meta null: only counts them); total: (sets << 34) | ids,
// one update a workgroup.
__global__ __launch_bounds__(256) void set_compact_kernel(const int32_t* __restrict__ ids,
                                                          const unsigned long long* __restrict__ meta, uint32_t n,
                                                          const uint8_t* __restrict__ dead, int32_t* __restrict__ out_ids,
                                                          unsigned long long* __restrict__ out_meta,
                                                          unsigned long long* total) {
    __shared__ unsigned long long scan[256];
    __shared__ unsigned long long base;
    const int tid = threadIdx.x;
    for (unsigned long long s0 = 256ull * blockIdx.x; s0 < n; s0 += 256ull * gridDim.x) {
        const unsigned long long s = s0 + tid;
        const bool keep = s < n && !dead[s];
        const unsigned long long len = keep ? meta[s] & 0xFFFFFFull : 0ull;
        const unsigned long long mine = keep ? (1ull << CNT_SHIFT) | len : 0ull;
        scan[tid] = mine;
        __syncthreads();
        for (int off = 1; off < 256; off <<= 1) {
            const unsigned long long a = tid >= off ? scan[tid - off] : 0;
            __syncthreads();
            scan[tid] += a;
            __syncthreads();
        }
        if (tid == 255) base = atomicAdd(total, scan[255]);
        __syncthreads();
        if (keep && out_meta) {
            const unsigned long long at = base + scan[tid] - mine, o = at & SIZE_MASK;
            const unsigned long long from = meta[s] >> 24;
            out_meta[at >> CNT_SHIFT] = (o << 24) | len;
            for (unsigned long long i = 0; i < len; ++i) out_ids[o + i] = ids[from + i];
        }
        __syncthreads();
    }
}

}  // namespace

namespace dqc {

dqc_status fetch_candidates(dqc_handle* h, std::vector<int32_t>* graph, std::vector<int32_t>& sizes,
                            std::vector<int32_t>& ids) {
    if (!h) return DQC_E_ARG;
    hipSetDevice(h->device);
    int64_t count = 0, total = 0;
    auto fetch_all = [&]() -> dqc_status {
        dqc_status rc = dqc_fetch_cliques(h, &count, &total, nullptr, nullptr);
        if (rc != DQC_OK) return rc;
        sizes.resize((size_t)count);
        ids.resize((size_t)total);
        if (graph) graph->resize((size_t)count);
        return graph ? dqc_fetch_batch_cliques(h, &count, &total, graph->data(), sizes.data(), ids.data())
                     : dqc_fetch_cliques(h, &count, &total, sizes.data(), ids.data());
    };
    GCtr g{};
    if (!hip_ok(h, hipMemcpy(&g, h->d_g, sizeof g, hipMemcpyDeviceToHost), "ctr read")) return DQC_E_HIP;
    const unsigned long long ns = g.clq_alloc >> CNT_SHIFT;
    // the (empty) task stack's records hold the table, the marks and what is left
    unsigned long long slots = 1;
    while (slots < 2 * ns) slots <<= 1;
    auto up = [](unsigned long long x) { return (x + 255ull) & ~255ull; };
    const unsigned long long o_hash = 256, o_table = o_hash + up(8 * ns), o_dead = o_table + up(4 * slots),
                             o_meta = o_dead + up(ns), room = h->cap_spill_v * sizeof(dqc::TaskVertex);
    if (ns < PREFILTER_LEAST || ns > (1ull << 30) || h->st_t || h->def_t || !h->d_svtx || !h->host_cliques.empty() ||
        o_meta > room)
        return fetch_all();
    char* base = (char*)h->d_svtx;
    unsigned long long *d_total = (unsigned long long*)base, *d_hash = (unsigned long long*)(base + o_hash);
    uint32_t* d_table = (uint32_t*)(base + o_table);
    uint8_t* d_dead = (uint8_t*)(base + o_dead);
    const uint32_t n = (uint32_t)ns;
    const int grid = (int)std::min<unsigned long long>((ns + 255) / 256, 8192);
    if (!hip_ok(h, hipMemsetAsync(d_total, 0, sizeof *d_total, h->stream), "prefilter")) return DQC_E_HIP;
    set_hash_kernel<<<grid, 256, 0, h->stream>>>(h->d_clq_ids, h->d_clq_meta, n, d_hash, d_dead, d_table, (uint32_t)slots);
    set_insert_kernel<<<grid, 256, 0, h->stream>>>(h->d_clq_ids, h->d_clq_meta, n, d_hash, d_dead, d_table, (uint32_t)slots);
    set_mark_kernel<<<grid, 256, 0, h->stream>>>(h->d_clq_ids, h->d_clq_meta, n, d_hash, d_dead, d_table, (uint32_t)slots);
    set_compact_kernel<<<grid, 256, 0, h->stream>>>(h->d_clq_ids, h->d_clq_meta, n, d_dead, nullptr, nullptr, d_total);
    unsigned long long left = 0;
    if (!hip_ok(h, hipGetLastError(), "prefilter launch") ||
        !hip_ok(h, hipMemcpyAsync(&left, d_total, sizeof left, hipMemcpyDeviceToHost, h->stream), "prefilter") ||
        !hip_ok(h, hipStreamSynchronize(h->stream), "prefilter"))
        return DQC_E_HIP;
    const size_t ms = (size_t)(left >> CNT_SHIFT), mi = (size_t)(left & SIZE_MASK);
    const unsigned long long o_ids = o_meta + up(8 * ms);
    if (o_ids + 4 * mi > room) return fetch_all();
    unsigned long long* d_meta = (unsigned long long*)(base + o_meta);
    int32_t* d_ids = (int32_t*)(base + o_ids);
    if (!hip_ok(h, hipMemsetAsync(d_total, 0, sizeof *d_total, h->stream), "prefilter")) return DQC_E_HIP;
    set_compact_kernel<<<grid, 256, 0, h->stream>>>(h->d_clq_ids, h->d_clq_meta, n, d_dead, d_ids, d_meta, d_total);
    if (!hip_ok(h, hipGetLastError(), "prefilter launch") || !hip_ok(h, hipStreamSynchronize(h->stream), "prefilter"))
        return DQC_E_HIP;
    std::vector<unsigned long long> meta(ms);
    std::vector<int32_t> raw(mi);
    if (!hip_ok(h, hipMemcpy(meta.data(), d_meta, sizeof(unsigned long long) * ms, hipMemcpyDeviceToHost), "clique read") ||
        !hip_ok(h, hipMemcpy(raw.data(), d_ids, sizeof(int32_t) * mi, hipMemcpyDeviceToHost), "clique read"))
        return DQC_E_HIP;
    sizes.resize(ms);
    ids.resize(mi);
    if (graph) graph->resize(ms);
    size_t p = 0;
    for (size_t s = 0; s < ms; ++s) {
        const size_t off = (size_t)(meta[s] >> 24), len = (size_t)(meta[s] & 0xFFFFFFull);
        sizes[s] = (int32_t)len;
        int32_t gb = 0;
        if (graph) {
            const int32_t gi = (int32_t)(std::upper_bound(h->gbase.begin(), h->gbase.end(), len ? raw[off] : 0) - h->gbase.begin()) - 1;
            (*graph)[s] = gi;
            gb = h->gbase[gi];
        }
        for (size_t i = 0; i < len; ++i) ids[p + i] = raw[off + i] - gb;
        p += len;
    }
    return DQC_OK;
}

}  // namespace dqc
