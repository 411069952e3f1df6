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
    need = 0;
    MGGX_HIP(rocprim::radix_sort_pairs_desc(nullptr, need, cnt, cnt_sorted, from, to, (size_t)u, 0, bits_of((long long)n), stream));
    char *tmp2 = tmp;
    if (need > tmp_bytes && (rc = buf.get(&tmp2, need))) return rc;
    MGGX_HIP(rocprim::radix_sort_pairs_desc(tmp2, need, cnt, cnt_sorted, from, to, (size_t)u, 0, bits_of((long long)n), stream));
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
