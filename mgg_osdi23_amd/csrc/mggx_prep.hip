// Device-side preparation of a share's remote side: the compact staging order of mggx_compact_remote, computed on
// the GPU (bit-identical to the host version).
//
// The ids are sorted (only the bits that they have) and run-length encoded.  Where a table with an entry per id is affordable
// (at most DENSE_PER_EDGE entries per edge: the ids of a partitioned graph always are), one look-up per edge writes the new
// column array; sparser ids are found with a binary search per edge.  Only the number of distinct ids is asked for first: with
// a table that takes one flag per id and no sort.  Bound: random accesses to a table the caches hold, one per edge.
// 2.43 M edges, 264 K distinct ids of 1 M: the look-ups 102 -> 16 us against the binary search; counting with one atomic per edge
// in place of the sort took 118 us (the hubs' counters are one address each) and 443 us for the two calls of the whole list,
// against 371 with the sort.
#include <algorithm>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_run_length_encode.hpp>

#include "mggx_dev.h"

namespace mggx {
namespace {

__global__ void __launch_bounds__(256) k_iota(int *__restrict__ v, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) v[i] = i;
}

// order[pos] = index (into the ascending id list) of the id staged at position pos
__global__ void __launch_bounds__(256) k_rank_and_fetch(const int *__restrict__ order, const int *__restrict__ ids, int u,
                                                        int *__restrict__ rank, int *__restrict__ fetch_ids)
{
    const int pos = blockIdx.x * 256 + threadIdx.x;
    if (pos >= u) return;
    const int i = order[pos];
    rank[i] = pos;
    fetch_ids[pos] = ids[i];
}

__global__ void __launch_bounds__(256) k_remap(const int *__restrict__ col, long long n, const int *__restrict__ ids, int u,
                                              const int *__restrict__ rank, int *__restrict__ out)
{
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long long)gridDim.x * 256) {
        const int key = col[e];
        int lo = 0, hi = u;  // first index with ids[idx] >= key; key is present
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (ids[mid] < key) lo = mid + 1;
            else hi = mid;
        }
        out[e] = rank[lo];
    }
}

// ---- dense ids
constexpr long long DENSE_PER_EDGE = 4, DENSE_ALWAYS = 1 << 20;

__global__ void k_range_init(int *w, int *sum)
{
    w[0] = 0x7fffffff;
    w[1] = -0x7fffffff - 1;
    *sum = 0;
}

// w[0] = smallest, w[1] = largest of v[0..n)
__global__ void __launch_bounds__(256) k_range(const int *__restrict__ v, long long n, int *__restrict__ w)
{
    __shared__ int red[2][4];
    int lo = 0x7fffffff, hi = -0x7fffffff - 1;
    const long long step = (long long)gridDim.x * 256;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += 4 * step) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // four loads in flight; past the end the last value again
            const int x = v[min(i + j * step, n - 1)];
            lo = min(lo, x);
            hi = max(hi, x);
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
    }
    if ((threadIdx.x & 63u) == 0) {
        red[0][threadIdx.x >> 6] = lo;
        red[1][threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; ++k) {
            lo = min(lo, red[0][k]);
            hi = max(hi, red[1][k]);
        }
        atomicMin(&w[0], lo);
        atomicMax(&w[1], hi);
    }
}

__global__ void k_publish3(const int *w, const int *sum, long long *host)
{
    host[0] = w[0];
    host[1] = w[1];
    host[2] = *sum;
}

__global__ void __launch_bounds__(256) k_mark_ids(const int *__restrict__ col, long long n, unsigned char *__restrict__ flag)
{
    const long long step = (long long)gridDim.x * 256;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += step) flag[col[e]] = 1;
}

// *sum += number of flags set in flag[0 .. 16 n16)
__global__ void __launch_bounds__(256) k_sum_flags(const uint4 *__restrict__ flag, long long n16, int *__restrict__ sum)
{
    __shared__ int red[4];
    int c = 0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n16; i += (long long)gridDim.x * 256) {
        const uint4 f = flag[i];
        c += __popc(f.x) + __popc(f.y) + __popc(f.z) + __popc(f.w);
    }
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(sum, red[0] + red[1] + red[2] + red[3]);
}

// place[id] = position of the id in the staging order
__global__ void __launch_bounds__(256) k_places(const int *__restrict__ fetch_ids, int u, int *__restrict__ place)
{
    const int pos = blockIdx.x * 256 + threadIdx.x;
    if (pos < u) place[fetch_ids[pos]] = pos;
}

__global__ void __launch_bounds__(256) k_look_up(const int *__restrict__ col, long long n, const int *__restrict__ place, int *__restrict__ out)
{
    const long long step = (long long)gridDim.x * 256;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += 4 * step) {
        int c[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) c[j] = col[min(e + j * step, n - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j) c[j] = place[c[j]];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (e + j * step < n) out[e + j * step] = c[j];
    }
}

// ---- ids by falling count
//
// Stable counting passes over COUNT_BITS bits of the counts at a time: how often each digit occurs in each tile of COUNT_TILE pairs, the
// exclusive sums of that table digit by digit (the largest first), and every pair to its place.  Bound: a chain of four short launches per pass,
// two passes up to 4 M edges.  rocPRIM merges up to a million pairs, some 20 launches one behind the other, and goes digit by digit
// beyond, in passes that last 23 us however few pairs there are: it stays where merging takes few launches and where the pairs are many (both
// calls of the staging list, us, rocPRIM / this: 1,352 distinct ids 123 / 167, 32,506 219 / 226, 243 K 373 / 329, 817 K 410 / 333, 2.7 M 702 / 803, 10.3 M
// 2,673 / 3,575; set-up of an eighth of 1 M nodes 709 -> 646).
constexpr int COUNT_LEAST = 1 << 15, COUNT_MOST = 1 << 20;
constexpr int COUNT_BITS = 11, COUNT_DIGITS = 1 << COUNT_BITS, COUNT_TILE = 2048, COUNT_STEPS = COUNT_TILE / 256;

__device__ __forceinline__ int falling_digit(unsigned count, int shift) { return COUNT_DIGITS - 1 - (int)(count >> shift & (COUNT_DIGITS - 1)); }

__global__ void __launch_bounds__(256) k_count_digits(const unsigned *__restrict__ cnt, int u, int shift, int tiles, int *__restrict__ table)
{
    __shared__ int seen[COUNT_DIGITS];
    for (int d = threadIdx.x; d < COUNT_DIGITS; d += 256) seen[d] = 0;
    __syncthreads();
    const int base = (int)blockIdx.x * COUNT_TILE;
#pragma unroll
    for (int k = 0; k < COUNT_STEPS; ++k) {
        const int i = base + k * 256 + (int)threadIdx.x;
        if (i < u) atomicAdd(&seen[falling_digit(cnt[i], shift)], 1);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < COUNT_DIGITS; d += 256) table[(size_t)d * tiles + blockIdx.x] = seen[d];
}

// A wavefront goes over its quarter of the tile 64 pairs at a time, in order; a pair's place among those of its digit is what the wavefronts before
// have of that digit, what this one has seen of it, and how many lanes before it hold it.
__global__ void __launch_bounds__(256) k_place_by_digit(const unsigned *__restrict__ cnt, const int *__restrict__ ids, int u, int shift, int tiles, const int *__restrict__ table,
                                                        unsigned *__restrict__ cnt_out, int *__restrict__ ids_out)
{
    __shared__ unsigned short seen[4][COUNT_DIGITS];
    for (int d = threadIdx.x; d < 4 * COUNT_DIGITS; d += 256) (&seen[0][0])[d] = 0;
    __syncthreads();
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
    const int base = (int)blockIdx.x * COUNT_TILE + wave * (COUNT_TILE / 4);
    unsigned c[COUNT_STEPS];
    int place[COUNT_STEPS];
#pragma unroll
    for (int k = 0; k < COUNT_STEPS; ++k) {
        const int i = base + 64 * k + lane;
        c[k] = i < u ? cnt[i] : 0;
    }
#pragma unroll
    for (int k = 0; k < COUNT_STEPS; ++k) {
        const bool on = base + 64 * k + lane < u;
        const int d = falling_digit(c[k], shift);
        unsigned long long same = __ballot(on);
#pragma unroll
        for (int b = 0; b < COUNT_BITS; ++b) {
            const unsigned long long set = __ballot(d >> b & 1);
            same &= d >> b & 1 ? set : ~set;
        }
        const int before = __popcll(same & ((1ull << lane) - 1));
        place[k] = 0;
        if (on) place[k] = seen[wave][d] + before;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (on && before == 0) seen[wave][d] = (unsigned short)(seen[wave][d] + __popcll(same));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < COUNT_STEPS; ++k) {
        const int i = base + 64 * k + lane;
        if (i >= u) continue;
        const int d = falling_digit(c[k], shift);
        int to = table[(size_t)d * tiles + blockIdx.x] + place[k];
        for (int w = 0; w < wave; ++w) to += seen[w][d];
        cnt_out[to] = c[k];
        ids_out[to] = ids[i];
    }
}

struct DeviceBuffers {
    std::vector<void *> ptrs;
    ~DeviceBuffers()
    {
        for (void *p : ptrs) dev_free(p);
    }
    template <typename T>
    int get(T **p, size_t count)
    {
        void *q = nullptr;
        const int rc = dev_alloc(&q, std::max<size_t>(count, 1) * sizeof(T));
        if (rc) return rc;
        ptrs.push_back(q);
        *p = static_cast<T *>(q);
        return MGGX_OK;
    }
};

}  // namespace
}  // namespace mggx

using mggx::fail;

MGGX_EXPORT int mggx_compact_remote_device(const int *d_remote_col, int64_t n_remote, int *d_remote_col_compact, int *d_fetch_ids,
                                           int64_t *n_unique)
{
    int rc = mggx::ensure_init();
    if (rc) return rc;
    if (n_remote < 0 || (n_remote && !d_remote_col)) return fail(MGGX_EINVAL, "compact_remote_device: bad remote_col");
    if (n_remote > 0x7fffffffLL) return fail(MGGX_ELIMIT, "compact_remote_device: more than 2^31-1 edges");
    if ((d_remote_col_compact == nullptr) != (d_fetch_ids == nullptr))
        return fail(MGGX_EINVAL, "compact_remote_device: pass both output arrays or neither");
    if (n_remote == 0) {
        if (n_unique) *n_unique = 0;
        return MGGX_OK;
    }
    hipStream_t stream = mggx::state().stream;
    const size_t n = (size_t)n_remote;
    mggx::DeviceBuffers buf;
    int *range = nullptr;  // smallest and largest id, a sum
    long long *w = nullptr;
    if ((rc = buf.get(&range, 3)) || (rc = mggx::host_words(&w))) return rc;
    mggx::k_range_init<<<1, 1, 0, stream>>>(range, range + 2);
    mggx::k_range<<<(unsigned)std::min<size_t>((n + 1023) / 1024, 256), 256, 0, stream>>>(d_remote_col, (long long)n, range);
    mggx::k_publish3<<<1, 1, 0, stream>>>(range, range + 2, w);
    MGGX_LAUNCH_CHECK("compact_remote_device kernels");
    MGGX_HIP(hipStreamSynchronize(stream));
    if (w[0] < 0) return fail(MGGX_EFORMAT, "compact_remote_device: negative neighbor id %d", (int)w[0]);
    const long long table = w[1] + 1;  // entries of a table with one per id
    const bool dense = table <= std::max(mggx::DENSE_ALWAYS, mggx::DENSE_PER_EDGE * (long long)n) && table <= 0x7fffffffLL;
    const auto bits_of = [](long long v) { return v > 0 ? 64u - (unsigned)__builtin_clzll((unsigned long long)v) : 1u; };
    const unsigned edge_blocks = (unsigned)std::min<size_t>((n + 255) / 256, 256 * 16);

    if (dense && !d_fetch_ids) {  // only their number: one flag per id
        const size_t bytes = ((size_t)table + 15) & ~(size_t)15;
        unsigned char *flag = nullptr;
        if ((rc = buf.get(&flag, bytes))) return rc;
        MGGX_HIP(hipMemsetAsync(flag, 0, bytes, stream));
        mggx::k_mark_ids<<<edge_blocks, 256, 0, stream>>>(d_remote_col, (long long)n, flag);
        mggx::k_sum_flags<<<(unsigned)std::min<size_t>((bytes / 16 + 255) / 256, 256), 256, 0, stream>>>(reinterpret_cast<const uint4 *>(flag), (long long)(bytes / 16), range + 2);
        mggx::k_publish3<<<1, 1, 0, stream>>>(range, range + 2, w);
        MGGX_LAUNCH_CHECK("compact_remote_device kernels");
        MGGX_HIP(hipStreamSynchronize(stream));
        if (n_unique) *n_unique = w[2];
        return MGGX_OK;
    }

    // 1. ascending ids, 2. distinct ids and how often each occurs
    const size_t distinct = dense ? std::min(n, (size_t)table) : n;  // at most
    int *sorted = nullptr, *ids = nullptr, *runs = nullptr;
    unsigned *cnt = nullptr;
    if ((rc = buf.get(&sorted, n)) || (rc = buf.get(&ids, distinct)) || (rc = buf.get(&cnt, distinct)) || (rc = buf.get(&runs, 1))) return rc;
    const unsigned *keys_in = reinterpret_cast<const unsigned *>(d_remote_col);  // no negative ids: the same order
    unsigned *keys_out = reinterpret_cast<unsigned *>(sorted);
    size_t tmp_bytes = 0, need = 0;
    MGGX_HIP(rocprim::radix_sort_keys(nullptr, need, keys_in, keys_out, n, 0, bits_of(table - 1), stream));
    tmp_bytes = need;
    MGGX_HIP(rocprim::run_length_encode(nullptr, need, sorted, (unsigned)n, ids, cnt, runs, stream));
    tmp_bytes = std::max(tmp_bytes, need);
    char *tmp = nullptr;
    if ((rc = buf.get(&tmp, tmp_bytes))) return rc;
    need = tmp_bytes;
    MGGX_HIP(rocprim::radix_sort_keys(tmp, need, keys_in, keys_out, n, 0, bits_of(table - 1), stream));
    need = tmp_bytes;
    MGGX_HIP(rocprim::run_length_encode(tmp, need, sorted, (unsigned)n, ids, cnt, runs, stream));
    mggx::k_publish3<<<1, 1, 0, stream>>>(range, runs, w);
    MGGX_LAUNCH_CHECK("compact_remote_device kernels");
    MGGX_HIP(hipStreamSynchronize(stream));
    const int u = (int)w[2];
    if (n_unique) *n_unique = u;
    if (!d_fetch_ids) return MGGX_OK;

    // 3. staging order: most referenced first; the sort is stable, so equal counts keep ascending id.  4. the rewritten column
    // array: an edge looks its id's position up in the table, or finds the id among the ascending ones first.
    int *order = nullptr, *iota = nullptr, *place = nullptr;
    unsigned *cnt_sorted = nullptr;
    if ((rc = buf.get(&cnt_sorted, (size_t)u)) || (rc = buf.get(&place, dense ? (size_t)table : (size_t)u)) ||
        (!dense && ((rc = buf.get(&iota, (size_t)u)) || (rc = buf.get(&order, (size_t)u)))))
        return rc;
    if (!dense) mggx::k_iota<<<(u + 255) / 256, 256, 0, stream>>>(iota, u);
    const int *from = dense ? ids : iota;
    int *to = dense ? d_fetch_ids : order;
    if (u >= mggx::COUNT_LEAST && u <= mggx::COUNT_MOST) {
        const int passes = ((int)bits_of((long long)n) + mggx::COUNT_BITS - 1) / mggx::COUNT_BITS, tiles = (u + mggx::COUNT_TILE - 1) / mggx::COUNT_TILE;
        const long long entries = (long long)tiles * mggx::COUNT_DIGITS;
        int *digits = nullptr, *places = nullptr, *ids_between = nullptr;
        char *scan_tmp = nullptr;
        if ((rc = buf.get(&digits, (size_t)entries)) || (rc = buf.get(&places, (size_t)entries + 1)) || (rc = buf.get(&ids_between, (size_t)u)) ||
            (rc = buf.get(&scan_tmp, mggx::scan_tmp_bytes((int)entries))))
            return rc;
        unsigned *cnt_from = cnt, *cnt_to = cnt_sorted;
        const int *ids_from = from;
        for (int p = 0; p < passes; ++p) {
            int *ids_to = (passes - p) % 2 ? to : ids_between;  // the last pass writes `to`
            mggx::k_count_digits<<<(unsigned)tiles, 256, 0, stream>>>(cnt_from, u, p * mggx::COUNT_BITS, tiles, digits);
            if ((rc = mggx::exclusive_scan_i32_device(digits, places, (int)entries, scan_tmp))) return rc;
            mggx::k_place_by_digit<<<(unsigned)tiles, 256, 0, stream>>>(cnt_from, ids_from, u, p * mggx::COUNT_BITS, tiles, places, cnt_to, ids_to);
            std::swap(cnt_from, cnt_to);
            ids_from = ids_to;
        }
    } else {
        need = 0;
        MGGX_HIP(rocprim::radix_sort_pairs_desc(nullptr, need, cnt, cnt_sorted, from, to, (size_t)u, 0, bits_of((long long)n), stream));
        char *tmp2 = tmp;
        if (need > tmp_bytes && (rc = buf.get(&tmp2, need))) return rc;
        MGGX_HIP(rocprim::radix_sort_pairs_desc(tmp2, need, cnt, cnt_sorted, from, to, (size_t)u, 0, bits_of((long long)n), stream));
    }
    if (dense) {
        mggx::k_places<<<(u + 255) / 256, 256, 0, stream>>>(d_fetch_ids, u, place);
        mggx::k_look_up<<<edge_blocks, 256, 0, stream>>>(d_remote_col, (long long)n, place, d_remote_col_compact);
    } else {
        mggx::k_rank_and_fetch<<<(u + 255) / 256, 256, 0, stream>>>(order, ids, u, place, d_fetch_ids);
        const long long blocks = std::min<long long>(((long long)n + 255) / 256, 256 * 64);
        mggx::k_remap<<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(d_remote_col, (long long)n, ids, u, place, d_remote_col_compact);
    }
    MGGX_LAUNCH_CHECK("compact_remote_device kernels");
    MGGX_HIP(hipStreamSynchronize(stream));  // the scratch buffers are freed on return
    return MGGX_OK;
}
