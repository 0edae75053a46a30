// Ground-truth comparison of two partitions (compare_communities, compare.cpp:58-307, and
// compute_gini_coeff, compare.cpp:310-337).
//
// The reference counts, for every pair of vertices inside one community of C1, whether C2
// also puts them together (same-same) or not (same-diff), and for every pair inside one
// community of C2 whether C1 separates them (diff-same), by walking all pairs: O(sum of
// squared community sizes).  The counts are integers, so any order gives the same values:
// here every vertex adds one to its (C1, C2) pair, the pairs add their counts to the sizes of C1
// and C2, and C(k, 2) is summed over each group.  The pairs live in an open-addressed HBM table
// of 64-bit keys (C1 * nC2 + C2) at most half full.  Then
//   same-same = sum over (a,b) of C(n_ab, 2),
//   same-diff = sum over a of C(n_a, 2) - same-same,
//   diff-same = sum over b of C(n_b, 2) - same-same,
// exactly the reference's counts.  Precision, recall, F-score and the Gini coefficients
// (a left fold over the sorted community sizes, zero-size ids included) are formed on the
// host with the reference's expressions and order.
#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cstring>
#include <vector>

#include "vt_internal.hpp"

namespace vt {
namespace {

constexpr unsigned long long kEmptyKey = ~0ull;
constexpr int kCmpBlock = 256;

// Per-block minimum and maximum of both partitions.
__global__ void __launch_bounds__(kCmpBlock) k_cmp_range(const int64_t* __restrict__ c1, const int64_t* __restrict__ c2,
                                                         int64_t n, int64_t* __restrict__ part)
{
    __shared__ int64_t s[4][kCmpBlock];
    int64_t mn1 = INT64_MAX, mx1 = INT64_MIN, mn2 = INT64_MAX, mx2 = INT64_MIN;
    for (int64_t i = blockIdx.x * (int64_t)kCmpBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kCmpBlock) {
        const int64_t a = c1[i], b = c2[i];
        mn1 = a < mn1 ? a : mn1;
        mx1 = a > mx1 ? a : mx1;
        mn2 = b < mn2 ? b : mn2;
        mx2 = b > mx2 ? b : mx2;
    }
    s[0][threadIdx.x] = mn1;
    s[1][threadIdx.x] = mx1;
    s[2][threadIdx.x] = mn2;
    s[3][threadIdx.x] = mx2;
    __syncthreads();
    for (int o = kCmpBlock / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            const int t = threadIdx.x;
            s[0][t] = s[0][t + o] < s[0][t] ? s[0][t + o] : s[0][t];
            s[1][t] = s[1][t + o] > s[1][t] ? s[1][t + o] : s[1][t];
            s[2][t] = s[2][t + o] < s[2][t] ? s[2][t + o] : s[2][t];
            s[3][t] = s[3][t + o] > s[3][t] ? s[3][t + o] : s[3][t];
        }
        __syncthreads();
    }
    if (threadIdx.x < 4) part[4 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

// A pair of communities and its vertices, in one line of memory.
struct __align__(16) PairSlot {
    unsigned long long key, cnt;
};

__global__ void k_cmp_clear(PairSlot* __restrict__ t, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        t[i] = PairSlot{kEmptyKey, 0};
}

// cnt vertices of the pair `key`, in the table.
__device__ __forceinline__ void pair_add(PairSlot* __restrict__ pairs, int logcap, unsigned long long key,
                                         unsigned long long cnt)
{
    const unsigned long long mask = (1ull << logcap) - 1;
    unsigned long long h = (key * 0x9E3779B97F4A7C15ull) >> (64 - logcap);
    for (;;) {  // ends: at most n distinct keys in a table of at least 2n slots
        unsigned long long old = __hip_atomic_load(&pairs[h].key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (old == kEmptyKey) old = atomicCAS(&pairs[h].key, kEmptyKey, key);
        if (old == kEmptyKey || old == key) break;
        h = (h + 1) & mask;
    }
    atomicAdd(&pairs[h].cnt, cnt);
}

// Every vertex: its (C1, C2) pair's count; the communities' sizes are left to the pairs, fewer than
// the vertices where the partitions resemble each other.  Bound by the memory's atomics, some 10 ns
// each on one line, and where the communities are few a few pairs hold most of the vertices: a
// workgroup counts its chunk in an LDS table first, one slot per hash, and adds each slot once; a
// pair whose slot another one has goes to memory directly (n = 1000003 with 2, 64, 1024 and 30011
// communities: 48, 148, 183 and 81 us; an atomic per vertex took 10023, 1542, 402 and 84).
constexpr int kCmpSlots = 1024;

__global__ void __launch_bounds__(kCmpBlock) k_cmp_count(const int64_t* __restrict__ c1, const int64_t* __restrict__ c2,
                                                         int64_t n, int64_t chunk, uint64_t nc2,
                                                         PairSlot* __restrict__ pairs, int logcap)
{
    __shared__ unsigned long long s_key[kCmpSlots];
    __shared__ unsigned s_cnt[kCmpSlots];
    static_assert(kCmpSlots == 1 << (64 - 54), "slots are the hash's top bits");
    for (int i = threadIdx.x; i < kCmpSlots; i += kCmpBlock) {
        s_key[i] = kEmptyKey;
        s_cnt[i] = 0;
    }
    __syncthreads();
    const int64_t lo = blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kCmpBlock) {
        const unsigned long long key = (uint64_t)c1[i] * nc2 + (uint64_t)c2[i];
        const uint32_t h = (uint32_t)((key * 0x9E3779B97F4A7C15ull) >> 54);
        unsigned long long old = __hip_atomic_load(&s_key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (old == kEmptyKey) old = atomicCAS(&s_key[h], kEmptyKey, key);
        if (old == kEmptyKey || old == key) atomicAdd(&s_cnt[h], 1u);
        else pair_add(pairs, logcap, key, 1);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kCmpSlots; i += kCmpBlock)
        if (s_cnt[i]) pair_add(pairs, logcap, s_key[i], s_cnt[i]);
}

// The communities' sizes from the pairs' counts, and *same += C(count, 2) over the pairs.
__global__ void __launch_bounds__(kCmpBlock) k_cmp_sizes(const PairSlot* __restrict__ pairs, int64_t cap, uint64_t nc2,
                                                         unsigned long long* __restrict__ size1,
                                                         unsigned long long* __restrict__ size2,
                                                         unsigned long long* __restrict__ same)
{
    unsigned long long p = 0;
    for (int64_t i = blockIdx.x * (int64_t)kCmpBlock + threadIdx.x; i < cap; i += (int64_t)gridDim.x * kCmpBlock) {
        const PairSlot x = pairs[i];
        if (x.key == kEmptyKey) continue;
        atomicAdd(&size1[x.key / nc2], x.cnt);
        atomicAdd(&size2[x.key % nc2], x.cnt);
        p += x.cnt * (x.cnt - 1) / 2;
    }
    __shared__ unsigned long long s;
    if (threadIdx.x == 0) s = 0;
    __syncthreads();
    for (int o = 32; o > 0; o >>= 1) p += __shfl_xor(p, o);
    if ((threadIdx.x & 63) == 0 && p) atomicAdd(&s, p);
    __syncthreads();
    if (threadIdx.x == 0 && s) atomicAdd(same, s);
}

// compute_gini_coeff (compare.cpp:310-337) on sizes already sorted ascending: the one-thread
// left folds of (i+1)*size[i] and size[i], then the reference's closing expression.  The sizes carry
// `bit`; *inside = the pairs of vertices inside the communities, counted in the same loop, beside
// the adds that wait for each other (a loop of its own took 0.5 ms for a million communities).
double gini_sorted(const uint64_t* sorted, int64_t n, uint64_t bit, uint64_t* inside)
{
    const int numColors = (int)n;
    double numFunc = 0.0, denFunc = 0.0;
    uint64_t pairs = 0;
    for (int64_t i = 0; i < numColors; i++) {
        const uint64_t size = sorted[i] - bit;
        numFunc = numFunc + (double)((i + 1) * (int64_t)size);
        denFunc = denFunc + (double)size;
        pairs += size * (size - 1) / 2;
    }
    *inside = pairs;
    return ((2 * numFunc) / (numColors * denFunc)) - ((double)(numColors + 1) / (double)numColors);
}

// Both partitions' community sizes, each sorted ascending, in one sort: C2's carry the bit above
// the sizes.
__global__ void k_cmp_mark(unsigned long long* __restrict__ size, int64_t n, unsigned long long bit)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        size[i] |= bit;
}

}  // namespace
}  // namespace vt

using namespace vt;

extern "C" int vt_compare_communities(vt_ctx* ctx, int64_t n, const int64_t* truth, const int64_t* found,
                                      vt_compare_stats* out)
{
    if (!ctx || !truth || !found || !out) return VT_ERR_ARG;
    return guarded(ctx, [&] {
        if (n < 1) fail(ctx, VT_ERR_ARG, "vt_compare_communities: n = %lld, need at least one vertex", (long long)n);
        VT_HIP(ctx, hipSetDevice(ctx->device));
        DBuf<int64_t> c1(ctx, (size_t)n), c2(ctx, (size_t)n);
        h2d(ctx, c1.p, truth, 8 * (size_t)n);
        h2d(ctx, c2.p, found, 8 * (size_t)n);

        // community id ranges
        const unsigned nb = grid_for(n, kCmpBlock, 1024);
        DBuf<int64_t> part(ctx, 4 * (size_t)nb);
        VT_LAUNCH(ctx, "cmp_range", k_cmp_range, nb, kCmpBlock, 0, (const int64_t*)c1.p, (const int64_t*)c2.p, n,
                  part.p);
        std::vector<int64_t> hp(4 * (size_t)nb);
        d2h(ctx, hp.data(), part.p, 8 * hp.size());
        int64_t mn1 = INT64_MAX, mx1 = INT64_MIN, mn2 = INT64_MAX, mx2 = INT64_MIN;
        for (unsigned b = 0; b < nb; b++) {
            mn1 = std::min(mn1, hp[4 * b]);
            mx1 = std::max(mx1, hp[4 * b + 1]);
            mn2 = std::min(mn2, hp[4 * b + 2]);
            mx2 = std::max(mx2, hp[4 * b + 3]);
        }
        if (mn1 < 0 || mn2 < 0)
            fail(ctx, VT_ERR_ARG, "vt_compare_communities: community ids must be >= 0 (smallest: %lld in truth, %lld in found)",
                 (long long)mn1, (long long)mn2);
        // the reference sizes its arrays by the largest id and passes the count to the Gini
        // coefficient as an int
        if (mx1 >= INT32_MAX || mx2 >= INT32_MAX)
            fail(ctx, VT_ERR_LIMIT, "vt_compare_communities: community ids must stay below 2^31 - 1");
        const int64_t nc1 = mx1 + 1, nc2 = mx2 + 1;

        int logcap = 1;
        while ((1ll << logcap) < 2 * n) logcap++;
        const int64_t cap = 1ll << logcap;
        const int64_t nc = nc1 + nc2;
        // [0, nc1) the sizes of C1, then those of C2, then the pairs that both put together
        DBuf<unsigned long long> size(ctx, (size_t)nc + 1);
        DBuf<PairSlot> pairs(ctx, (size_t)cap);
        unsigned long long *size1 = size.p, *size2 = size.p + nc1, *same = size.p + nc;
        dzero(ctx, size.p, 8 * (size_t)(nc + 1));
        VT_LAUNCH(ctx, "cmp_clear", k_cmp_clear, grid_for(cap, 256, 8192), 256, 0, pairs.p, cap);
        // a vertex per thread until there is a workgroup per CU, 1024 vertices until there are four, then
        // those four (n = 30000 with 3750 communities: 16 us, with 1024 a workgroup 24; n = 4 * 10^6 with 2
        // communities 66, with 2048 workgroups 125)
        const int64_t chunk = std::max(std::min<int64_t>(std::max<int64_t>(256, n / 256), 1024), (n + 1023) / 1024);
        VT_LAUNCH(ctx, "cmp_count", k_cmp_count, (unsigned)((n + chunk - 1) / chunk), kCmpBlock, 0, (const int64_t*)c1.p,
                  (const int64_t*)c2.p, n, chunk, (uint64_t)nc2, pairs.p, logcap);
        VT_LAUNCH(ctx, "cmp_sizes", k_cmp_sizes, grid_for(cap, kCmpBlock, 2048), kCmpBlock, 0, (const PairSlot*)pairs.p, cap,
                  (uint64_t)nc2, size1, size2, same);
        const int bits = (int)bits_for(n);
        VT_LAUNCH(ctx, "cmp_mark", k_cmp_mark, grid_for(nc2, 256, 8192), 256, 0, size2, nc2, 1ull << bits);
        DBuf<unsigned long long> alt(ctx, (size_t)nc);
        rocprim::double_buffer<unsigned long long> kb(size.p, alt.p);
        size_t tb = 0;
        VT_HIP(ctx, rocprim::radix_sort_keys(nullptr, tb, kb, (size_t)nc, 0, bits + 1, ctx->stream));
        void* tmp = scratch(ctx, "sort_tmp", tb);
        VT_HIP(ctx, rocprim::radix_sort_keys(tmp, tb, kb, (size_t)nc, 0, bits + 1, ctx->stream));
        if (kb.current() != size.p) d2d(ctx, size.p, kb.current(), 8 * (size_t)nc);
        std::vector<uint64_t> z((size_t)nc + 1);
        d2h(ctx, z.data(), size.p, 8 * z.size());
        uint64_t ss = z[(size_t)nc], p1 = 0, p2 = 0;

        vt_compare_stats r;
        std::memset(&r, 0, sizeof(r));
        r.gini_truth = gini_sorted(z.data(), nc1, 0, &p1);
        r.gini_found = gini_sorted(z.data() + nc1, nc2, 1ull << bits, &p2);
        r.n = n;
        r.nc_truth = nc1;
        r.nc_found = nc2;
        r.same_same = (int64_t)ss;
        r.same_diff = (int64_t)(p1 - ss);
        r.diff_same = (int64_t)(p2 - ss);
        // compare.cpp:267-272, term by term
        r.precision = (double)r.same_same / (double)(r.same_same + r.diff_same);
        r.recall = (double)r.same_same / (double)(r.same_same + r.same_diff);
        r.f_score = 2.0 * ((r.precision * r.recall) / (r.precision + r.recall));
        *out = r;
    });
}
