// Neighbor partitioning on the GPU: prefix sums, the build_part arrays in the
// reference's layout, and the merged partition-descriptor list the aggregation
// kernels consume.
#include <algorithm>
#include <chrono>
#include <type_traits>

#include "mggx_dev.h"

namespace mggx {
namespace {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 4;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

// Block-wide exclusive scan of one int per thread (256 threads); returns the
// exclusive prefix and leaves the block total in *total.
__device__ __forceinline__ int block_exclusive_scan(int v, int *lds /* 256 ints */, int *total)
{
    const int t = threadIdx.x;
    lds[t] = v;
    __syncthreads();
    for (int o = 1; o < SCAN_THREADS; o <<= 1) {
        int add = t >= o ? lds[t - o] : 0;
        __syncthreads();
        lds[t] += add;
        __syncthreads();
    }
    const int incl = lds[t];
    *total = lds[SCAN_THREADS - 1];
    __syncthreads();
    return incl - v;
}

// What a scan sums: element i, read (or computed) twice rather than written out in between.
struct ScanArray {
    const int *in;
    __device__ __forceinline__ int operator()(long long i) const { return in[i]; }
};
// parts of one CSR side per row: ceil(deg/ps); both sides summed when beg_r != NULL.  Row r spans edges
// [beg[r], end[r]) (a CSR passes end = ptr + 1).
struct ScanParts {
    const int *beg_l, *end_l, *beg_r, *end_r;
    int ps;
    __device__ __forceinline__ int operator()(long long r) const
    {
        long long c = ((long long)end_l[r] - beg_l[r] + ps - 1) / ps;
        if (beg_r) c += ((long long)end_r[r] - beg_r[r] + ps - 1) / ps;
        return (int)c;
    }
};

template <typename F>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_tile_sums(const F in, int n, long long *__restrict__ tile_sum)
{
    __shared__ long long red[SCAN_THREADS];
    const long long base = (long long)blockIdx.x * SCAN_TILE;
    long long s = 0;
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        long long idx = base + (long long)threadIdx.x * SCAN_ITEMS + i;
        if (idx < n) s += in(idx);
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = SCAN_THREADS / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) tile_sum[blockIdx.x] = red[0];
}

// One block turns tile sums into exclusive tile offsets; tile_sum[num_tiles] receives the total.
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_tile_offsets(long long *__restrict__ tile_sum, int num_tiles)
{
    __shared__ long long buf[SCAN_THREADS];
    __shared__ long long carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < num_tiles; base += SCAN_THREADS) {
        const int idx = base + threadIdx.x;
        const long long v = idx < num_tiles ? tile_sum[idx] : 0;
        buf[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < SCAN_THREADS; o <<= 1) {
            long long add = threadIdx.x >= o ? buf[threadIdx.x - o] : 0;
            __syncthreads();
            buf[threadIdx.x] += add;
            __syncthreads();
        }
        const long long incl = buf[threadIdx.x];
        const long long c = carry;
        if (idx < num_tiles) tile_sum[idx] = c + incl - v;
        __syncthreads();
        if (threadIdx.x == SCAN_THREADS - 1) carry = c + incl;
        __syncthreads();
    }
    if (threadIdx.x == 0) tile_sum[num_tiles] = carry;
}

// `tile`: the tiles' exclusive offsets (sums_only = 0), or their sums (sums_only = 1: every workgroup adds up the ones before
// its own, which for up to SCAN_SUM_TILES tiles is a few KB out of the L2 and saves the launch in between).  The total goes to
// out[n] and, in 64 bits, to *host_total (pinned host memory, or NULL).
constexpr int SCAN_SUM_TILES = 1024;
template <typename F>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_apply(const F in, int *__restrict__ out, int n, long long *__restrict__ tile, int sums_only,
                                                             long long *host_total)
{
    __shared__ int lds[SCAN_THREADS];
    __shared__ long long part[SCAN_THREADS];
    const long long base = (long long)blockIdx.x * SCAN_TILE;
    long long before = 0;
    if (sums_only) {
        for (int i = threadIdx.x; i < (int)blockIdx.x; i += SCAN_THREADS) before += tile[i];
        part[threadIdx.x] = before;
        __syncthreads();
        for (int o = SCAN_THREADS / 2; o > 0; o >>= 1) {
            if (threadIdx.x < o) part[threadIdx.x] += part[threadIdx.x + o];
            __syncthreads();
        }
        before = part[0];
    } else {
        before = tile[blockIdx.x];
    }
    int v[SCAN_ITEMS];
    int local = 0;
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        long long idx = base + (long long)threadIdx.x * SCAN_ITEMS + i;
        v[i] = idx < n ? in(idx) : 0;
        local += v[i];
    }
    int total;
    int excl = block_exclusive_scan(local, lds, &total);
    long long run = before + excl;
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        long long idx = base + (long long)threadIdx.x * SCAN_ITEMS + i;
        if (idx < n) out[idx] = (int)run;
        run += v[i];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == SCAN_THREADS - 1) {
        out[n] = (int)run;
        tile[gridDim.x] = run;
        if (host_total) *host_total = run;
    }
}

// Results of a set-up call for the host: words[0] = the value at a, words[1] at b, words[2] at c, words[3] at d, words[4] at e (NULL: 0).
__global__ void k_publish(const int *a, const int *b, const int *c, long long *words, const int *d = nullptr, const int *e = nullptr)
{
    words[0] = a ? *a : 0;
    words[1] = b ? *b : 0;
    words[2] = c ? *c : 0;
    words[3] = d ? *d : 0;
    words[4] = e ? *e : 0;
}

__global__ void k_clear_plan(int *counter, int n, unsigned long long *chain, int workgroups)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) counter[i] = 0;
    for (int i = threadIdx.x; i < workgroups; i += blockDim.x) chain[i] = 0;
}

__global__ void k_zero_words(int *w, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) w[i] = 0;
}

// largest r in [0, rows) with off[r] <= q (off is non-decreasing, off[rows] > q)
__device__ __forceinline__ int row_of_part(const int *__restrict__ off, int rows, int q)
{
    int lo = 0, hi = rows;  // invariant: off[lo] <= q < off[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid] <= q) lo = mid;
        else hi = mid;
    }
    return lo;
}

__global__ void __launch_bounds__(256) k_fill_desc(const int *__restrict__ off, const int *__restrict__ beg_l,
                                                   const int *__restrict__ end_l, const int *__restrict__ beg_r,
                                                   const int *__restrict__ end_r, int rows, int ps, int num_parts,
                                                   int4 *__restrict__ desc)
{
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= num_parts) return;
    const int r = row_of_part(off, rows, q);
    const int j = q - off[r];
    const int total = off[r + 1] - off[r];
    const int nl = (int)(((long long)end_l[r] - beg_l[r] + ps - 1) / ps);
    unsigned start, len;
    if (j < nl) {
        const long long beg = (long long)beg_l[r] + (long long)j * ps;
        start = (unsigned)beg;
        len = (unsigned)min((long long)ps, (long long)end_l[r] - beg);
    } else {
        const long long beg = (long long)beg_r[r] + (long long)(j - nl) * ps;
        start = (unsigned)beg | DESC_REMOTE;
        len = (unsigned)min((long long)ps, (long long)end_r[r] - beg);
    }
    unsigned z = len;
    if (j == 0) z |= DESC_FIRST;
    if (j == total - 1) z |= DESC_LAST;
    desc[q] = make_int4((int)start, r, (int)z, 0);
}

// Column-blocked plans.  One wavefront per row: flag = 1 if some row's neighbor ids are not in non-decreasing order.
__global__ void __launch_bounds__(256) k_check_sorted(const int *__restrict__ ptr, const int *__restrict__ col, int rows,
                                                      int *__restrict__ flag)
{
    const int r = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (r >= rows) return;
    const int lane = (int)(threadIdx.x & 63u);
    bool bad = false;
    for (int e = ptr[r] + lane; e + 1 < ptr[r + 1]; e += 64) bad |= col[e] > col[e + 1];
    if (bad) *flag = 1;
}

// vbeg[c * rows + v] = first edge of row v whose neighbor id is >= lb + c * block_rows, c = 0..blocks (rows sorted)
__global__ void __launch_bounds__(256) k_block_bounds(const int *__restrict__ ptr, const int *__restrict__ col, int rows, int lb,
                                                      int block_rows, int blocks, int *__restrict__ vbeg)
{
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long long)(blocks + 1) * rows) return;
    const int c = (int)(idx / rows), v = (int)(idx % rows);
    int lo = ptr[v], hi = ptr[v + 1];
    if (c == blocks) {
        lo = hi;
    } else if (c > 0) {
        const long long key = (long long)lb + (long long)c * block_rows;
        while (lo < hi) {
            const int mid = (int)(((long long)lo + hi) >> 1);
            if (col[mid] < key) lo = mid + 1;
            else hi = mid;
        }
    }
    vbeg[idx] = lo;
}

// explicit partition arrays (reference layout) -> descriptors; lengths from row_ptr
__global__ void __launch_bounds__(256) k_desc_from_parts(const int *__restrict__ row_ptr, const int *__restrict__ part_ptr,
                                                         const int *__restrict__ part2node, int num_parts, int ps,
                                                         int4 *__restrict__ desc)
{
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= num_parts) return;
    const int r = part2node[q];
    const int beg = part_ptr[q];
    unsigned z = (unsigned)max(0, min(ps, row_ptr[r + 1] - beg));
    if (q == 0 || part2node[q - 1] != r) z |= DESC_FIRST;
    if (q == num_parts - 1 || part2node[q + 1] != r) z |= DESC_LAST;
    desc[q] = make_int4(beg, r, (int)z, 0);
}

// Explicit plans with several partitions per unit (ps < 16).  cnt[r] = units of row r = ceil(partitions of r / g).
__global__ void __launch_bounds__(256) k_units_per_row(const int *__restrict__ off_p, int rows, int g, int *__restrict__ cnt)
{
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= rows) return;
    cnt[r] = (off_p[r + 1] - off_p[r] + g - 1) / g;
}

// One descriptor per unit: unit j of row r spans the partitions off_p[r] + j g .. (at most g of them, to the end of the row),
// which build_part lays out as consecutive edge ranges of ps neighbors -- one edge range from the first one's start.
// Threads past the device-side unit count off_u[rows] (the grid is sized by a host-side bound) do nothing.
__global__ void __launch_bounds__(256) k_desc_from_units(const int *__restrict__ row_ptr, const int *__restrict__ part_ptr,
                                                         const int *__restrict__ off_p, const int *__restrict__ off_u, int rows, int ps,
                                                         int g, int4 *__restrict__ desc)
{
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= off_u[rows]) return;
    const int r = row_of_part(off_u, rows, q);
    const int j = q - off_u[r];
    const int p0 = off_p[r] + j * g;
    const int np = min(g, off_p[r + 1] - p0);
    const int beg = part_ptr[p0];
    unsigned z = (unsigned)max(0, min(np * ps, row_ptr[r + 1] - beg));
    if (j == 0) z |= DESC_FIRST;
    if (q == off_u[r + 1] - 1) z |= DESC_LAST;
    desc[q] = make_int4(beg, r, (int)z, 0);
}

// off[r] for explicit plans: first descriptor of row r = lower bound of r in part2node
__global__ void __launch_bounds__(256) k_off_from_parts(const int *__restrict__ part2node, int num_parts, int rows,
                                                        int *__restrict__ off)
{
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r > rows) return;
    int lo = 0, hi = num_parts;  // first index with part2node[idx] >= r
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (part2node[mid] < r) lo = mid + 1;
        else hi = mid;
    }
    off[r] = lo;
}

// Rows without any descriptor (counter[0] of them), and the most descriptors that one row has in *most (holds 0; NULL: not asked for).
// Few workgroups that go over the rows in strides, because each ends in an atomic on one address: with one per 256 rows those were the
// kernel (524 K rows 25 us, 2.45 M rows 111; this way 5.3 and 7.5).
constexpr int EMPTY_THREADS = 1024, EMPTY_WORKGROUPS = 256, EMPTY_AHEAD = 4;  // EMPTY_AHEAD: rows of a thread in flight
__global__ void __launch_bounds__(EMPTY_THREADS) k_collect_empty(const int *__restrict__ off, int rows, int *__restrict__ list, int *__restrict__ counter,
                                                                 int *__restrict__ most)
{
    const long long step = (long long)gridDim.x * EMPTY_THREADS;
    int longest = 0;
    for (long long r0 = (long long)blockIdx.x * EMPTY_THREADS + threadIdx.x; r0 < rows; r0 += EMPTY_AHEAD * step) {
        int n[EMPTY_AHEAD];
#pragma unroll
        for (int j = 0; j < EMPTY_AHEAD; ++j) {
            const long long r = r0 + j * step;
            n[j] = r < rows ? off[r + 1] - off[r] : -1;
        }
#pragma unroll
        for (int j = 0; j < EMPTY_AHEAD; ++j) {
            if (n[j] == 0) list[atomicAdd(counter, 1)] = (int)(r0 + j * step);
            longest = max(longest, n[j]);
        }
    }
    if (!most) return;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o));
    __shared__ int of_wave[EMPTY_THREADS / 64];
    if ((threadIdx.x & 63u) == 0) of_wave[threadIdx.x >> 6] = longest;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    longest = threadIdx.x < EMPTY_THREADS / 64 ? of_wave[threadIdx.x] : 0;
#pragma unroll
    for (int o = EMPTY_THREADS / 128; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o));
    if (threadIdx.x == 0 && longest > 0) atomicMax(most, longest);
}

// Reference-layout arrays, launched behind the scan that makes node2part, without the host: *d_total is the number of partitions as
// the scan left it (a total that is no count of 32 bits writes nothing; the host refuses it afterwards).
__global__ void __launch_bounds__(256) k_parts_ref_layout(const int *__restrict__ indptr, int *__restrict__ node2part, const long long *__restrict__ d_total,
                                                          int num_nodes, int ps, int compat, int *__restrict__ part_ptr, int *__restrict__ part2node)
{
    const long long total = *d_total;
    if (total < 0 || total > 0x7ffffffeLL) return;
    const int num_parts = (int)total;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        node2part[num_nodes + 1] = num_parts;
        const bool last_has = num_nodes > 0 && indptr[num_nodes] > indptr[num_nodes - 1];
        part_ptr[num_parts] = (compat && !last_has) ? 0 : (num_nodes > 0 ? indptr[num_nodes] : 0);
    }
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < num_parts; q += (long long)gridDim.x * 256) {
        const int p = (int)q, i = row_of_part(node2part, num_nodes, p);
        part_ptr[p] = indptr[i] + (p - node2part[i]) * ps;
        part2node[p] = i;
    }
}

// max over non-negative ints into a word that holds 0; their number is read on the device.  One atomicMax per workgroup that saw
// more than 0, all on one address: with 1,024 workgroups those were the kernel (13.7 us on a CSR without remote edges).
__global__ void __launch_bounds__(256) k_max_i32(const int *__restrict__ v, const int *__restrict__ count, int *__restrict__ out)
{
    __shared__ int red[256];
    const long long n = *count;
    int m = 0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) m = max(m, v[i]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0 && red[0] > 0) atomicMax(out, red[0]);
}

// split_CSR on the GPU, one wavefront per row.  Pass 1 counts the neighbors inside [lb,ub); pass 2 is a stable
// partition of the row (ballot + prefix popcount keeps the order inside each side).  Long rows are taken SPLIT_AHEAD
// chunks of 64 at a time, all loads in flight before the first is used: both passes last as long as the longest row,
// one memory latency per trip (125 K rows, 2.9 M neighbors, the longest
// row some thousands: 53 -> 27 us counting, 65 -> 36 us filling; one chunk at a time as before where 128 neighbors or fewer are left).
constexpr int SPLIT_AHEAD = 8;

// chunk j of up to SPLIT_AHEAD chunks of a row at e0: its neighbor for this lane, or -1 (no id: lb >= 0) past the end
template <int N>
__device__ __forceinline__ void split_load(int (&u)[N], const int *__restrict__ col, int e0, int end, int lane)
{
#pragma unroll
    for (int j = 0; j < N; ++j) u[j] = col[e0 + min(64 * j + lane, end - e0 - 1)];
#pragma unroll
    for (int j = 0; j < N; ++j) u[j] = 64 * j + lane < end - e0 ? u[j] : -1;
}

__global__ void __launch_bounds__(256) k_split_count(const int *__restrict__ ptr, const int *__restrict__ col, int lb, int ub,
                                                     int *__restrict__ cnt_l, int *__restrict__ cnt_r)
{
    const int lane = (int)(threadIdx.x & 63u);
    const int rows = ub - lb;
    for (long long r = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); r < rows; r += (long long)gridDim.x * 4) {
        const int beg = ptr[lb + r], end = ptr[lb + r + 1];
        int local = 0;
        const auto take = [&](auto ahead, int e0) {
            int u[decltype(ahead)::value];
            split_load(u, col, e0, end, lane);
#pragma unroll
            for (int j = 0; j < decltype(ahead)::value; ++j) local += u[j] >= lb && u[j] < ub ? 1 : 0;
        };
        int e0 = beg;
        for (; end - e0 > 128; e0 += min(64 * SPLIT_AHEAD, end - e0)) take(std::integral_constant<int, SPLIT_AHEAD>{}, e0);
        for (; e0 < end; e0 += min(64, end - e0)) take(std::integral_constant<int, 1>{}, e0);
        for (int o = 32; o > 0; o >>= 1) local += __shfl_xor(local, o, 64);
        if (lane == 0) {
            cnt_l[r] = local;
            cnt_r[r] = (end - beg) - local;
        }
    }
}

__global__ void __launch_bounds__(256) k_split_fill(const int *__restrict__ ptr, const int *__restrict__ col, int lb, int ub,
                                                    const int *__restrict__ lptr, const int *__restrict__ rptr,
                                                    int *__restrict__ lcol, int *__restrict__ rcol)
{
    const int lane = (int)(threadIdx.x & 63u);
    const int rows = ub - lb;
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (long long r = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); r < rows; r += (long long)gridDim.x * 4) {
        const int beg = ptr[lb + r], end = ptr[lb + r + 1];
        int lo = lptr[r], ro = rptr[r];
        const auto take = [&](auto ahead, int e0) {
            int u[decltype(ahead)::value];
            split_load(u, col, e0, end, lane);
#pragma unroll
            for (int j = 0; j < decltype(ahead)::value; ++j) {
                const bool valid = 64 * j + lane < end - e0;
                const bool is_local = valid && u[j] >= lb && u[j] < ub;
                const unsigned long long ml = __ballot(is_local), mv = __ballot(valid);
                const unsigned long long mr = mv & ~ml;
                if (is_local) lcol[lo + __popcll(ml & below)] = u[j];
                else if (valid) rcol[ro + __popcll(mr & below)] = u[j];
                lo += __popcll(ml);
                ro += __popcll(mr);
            }
        };
        int e0 = beg;
        for (; end - e0 > 128; e0 += min(64 * SPLIT_AHEAD, end - e0)) take(std::integral_constant<int, SPLIT_AHEAD>{}, e0);
        for (; e0 < end; e0 += min(64, end - e0)) take(std::integral_constant<int, 1>{}, e0);
    }
}

struct GuardArgs {
    const int *arr[4];
    long long len[4];
};

__device__ __forceinline__ unsigned long long guard_mix(unsigned long long x)
{
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// Fingerprint of up to four index arrays: the last entry of each and up to GUARD_SAMPLES entries at a fixed stride,
// each mixed with its position.  arm != 0 stores it; otherwise it is compared with the stored one, the verdict goes to
// fp[1] (read as int: 1 = unchanged) and, on a mismatch, `tag` to the host-visible flag.  One workgroup; every thread
// issues all of its loads before it uses the first, so the kernel costs one trip to memory.
constexpr int GUARD_SAMPLES = 512;
__global__ void __launch_bounds__(256) k_guard(const GuardArgs g, unsigned long long *__restrict__ fp, volatile int *host_flag, int tag, int arm)
{
    __shared__ unsigned long long red[4];
    constexpr int PER = GUARD_SAMPLES / 256;
    int v[4][PER + 1];
    long long at[4][PER + 1];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const long long n = g.arr[a] ? g.len[a] : 0;
        const long long samples = n < GUARD_SAMPLES ? n : GUARD_SAMPLES;
        const long long stride = samples > 0 ? n / samples : 1;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const long long i = (long long)threadIdx.x + 256 * j;
            at[a][j] = i < samples ? i * stride : -1;
        }
        at[a][PER] = (threadIdx.x == 0 && n > 0) ? n - 1 : -1;
#pragma unroll
        for (int j = 0; j <= PER; ++j) v[a][j] = at[a][j] >= 0 ? __builtin_nontemporal_load(g.arr[a] + at[a][j]) : 0;
    }
    unsigned long long h = 0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
        for (int j = 0; j <= PER; ++j)
            if (at[a][j] >= 0)
                h += guard_mix(((unsigned long long)(a + 1 + (j == PER ? 4 : 0)) << 56) ^ ((unsigned long long)at[a][j] << 24) ^ (unsigned)v[a][j]);
    }
    for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o, 64);
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = h;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long total = red[0] + red[1] + red[2] + red[3];
        int *ok = reinterpret_cast<int *>(fp + 1);
        if (arm) {
            fp[0] = total;
            *ok = 1;
        } else {
            const int same = fp[0] == total;
            *ok = same;
            if (!same) *host_flag = tag;
        }
    }
}

__global__ void k_set_tail(int *node2part, int num_nodes)
{
    node2part[num_nodes + 1] = node2part[num_nodes];
}

}  // namespace

bool capturing()
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(state().stream, &st) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return st == hipStreamCaptureStatusActive;
}

static int host_flag_init()
{
    State &s = state();
    if (!s.h_stale) {
        void *p = nullptr;
        if (hipHostMalloc(&p, 64, hipHostMallocMapped) != hipSuccess) return fail(MGGX_ENOMEM, "content check: pinned flag");
        s.h_stale = static_cast<volatile int *>(p);
        *s.h_stale = 0;
    }
    return MGGX_OK;
}

static int guard_launch(Guard &g, int arm)
{
    State &s = state();
    GuardArgs a;
    for (int i = 0; i < 4; ++i) {
        a.arr[i] = g.arr[i];
        a.len[i] = g.len[i];
    }
    k_guard<<<1, 256, 0, s.stream>>>(a, g.d_fp, s.h_stale, g.id, arm);
    MGGX_LAUNCH_CHECK("k_guard");
    return MGGX_OK;
}

int guard_arm(Guard &g)
{
    State &s = state();
    int rc = host_flag_init();
    if (rc) return rc;
    if (!g.d_fp) {
        if (capturing()) return fail(MGGX_EINVAL, "first use of these CSR arrays inside a stream capture: call once outside the capture first");
        if (const int rc = dev_array(&g.d_fp, 2)) return rc;
    }
    g.id = s.next_guard_id++;
    if (s.next_guard_id > 0x3fffffff) s.next_guard_id = 1;
    rc = guard_launch(g, 1);
    g.armed = rc == MGGX_OK;
    return rc;
}

int guard_check(Guard &g, Gate *gate)
{
    State &s = state();
    *gate = Gate{};
    if (!s.plan_check || !g.armed) return MGGX_OK;
    gate->cnt_l = g.cnt_l;
    gate->cnt_r = g.cnt_r;
    gate->want_l = g.want_l;
    gate->want_r = g.want_r;
    gate->flag = s.h_stale;
    gate->tag = g.id;
    if (s.plan_check >= 2) {
        const int rc = guard_launch(g, 0);
        if (rc) return rc;
        gate->ok = g.ok();
    }
    return MGGX_OK;
}

void retire_block(void *p, size_t bytes)
{
    if (!p) return;
    State &s = state();
    s.retired.push_back(p);
    s.retired_bytes += bytes;
}

void guard_free(Guard &g, bool retire)
{
    if (g.d_fp) {
        if (retire) retire_block(g.d_fp, 16);
        else dev_free(g.d_fp);
    }
    g.d_fp = nullptr;
    g.armed = false;
}

// A check that ran on the stream since the last call found arrays that no longer match their record: everything cached
// for those addresses is dropped (the next call builds it anew from what is there now) and the caller gets an error.
int stale_poll()
{
    State &s = state();
    if (!s.h_stale || !*s.h_stale) return MGGX_OK;
    const int id = *s.h_stale;
    if (capturing()) return fail(MGGX_EINVAL, "CSR arrays changed under a cached plan (found while capturing; end the capture and call mggx_forget)");
    (void)hipStreamSynchronize(s.stream);
    *s.h_stale = 0;
    const int *arrs[4] = {nullptr, nullptr, nullptr, nullptr};
    for (const GraphInfo &g : s.graphs)
        if (g.guard.id == id)
            for (int i = 0; i < 4; ++i) arrs[i] = g.guard.arr[i];
    for (const Plan *p : s.plans)
        if (p->guard.id == id)
            for (int i = 0; i < 4; ++i) arrs[i] = p->guard.arr[i];
    for (int i = 0; i < 4; ++i)
        if (arrs[i]) (void)forget_pointer(arrs[i]);
    return fail(MGGX_EINVAL, "the CSR arrays at %p changed after the library cached a plan for them: that call's kernels did nothing and the "
                             "plan was dropped; call again (and mggx_forget() before rewriting or freeing cached arrays)", (const void *)arrs[0]);
}

size_t scan_tmp_bytes(int n)
{
    const size_t tiles = ((size_t)std::max(n, 1) + SCAN_TILE - 1) / SCAN_TILE;
    return sizeof(long long) * (tiles + 1);
}

// out[0..n] = exclusive prefix sums of in(0..n-1), in 2 or 3 launches; d_tmp: scan_tmp_bytes(n)
template <typename F>
static int scan_launch(const F &in, int *d_out, int n, void *d_tmp, long long *host_total)
{
    State &s = state();
    const int tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
    long long *d_tile = static_cast<long long *>(d_tmp);
    const int sums_only = tiles <= SCAN_SUM_TILES;
    k_scan_tile_sums<F><<<tiles, SCAN_THREADS, 0, s.stream>>>(in, n, d_tile);
    if (!sums_only) k_scan_tile_offsets<<<1, SCAN_THREADS, 0, s.stream>>>(d_tile, tiles);
    k_scan_apply<F><<<tiles, SCAN_THREADS, 0, s.stream>>>(in, d_out, n, d_tile, sums_only, host_total);
    MGGX_LAUNCH_CHECK("exclusive scan");
    return MGGX_OK;
}

int exclusive_scan_i32_device(const int *d_in, int *d_out, int n, void *d_tmp)
{
    if (n <= 0) return fail(MGGX_EINVAL, "exclusive_scan: empty input");
    return scan_launch(ScanArray{d_in}, d_out, n, d_tmp, nullptr);
}

// The scan with its total on the host (synchronises).
template <typename F>
static int scan_total(const F &in, int *d_out, int n, long long *total_host)
{
    State &s = state();
    if (n <= 0) {
        MGGX_HIP(hipMemsetAsync(d_out, 0, sizeof(int), s.stream));
        if (total_host) *total_host = 0;
        return MGGX_OK;
    }
    void *tmp = nullptr;
    long long *w = nullptr;
    int rc = host_words(&w);
    if (!rc) rc = dev_alloc(&tmp, scan_tmp_bytes(n));
    if (rc) return rc;
    rc = scan_launch(in, d_out, n, tmp, w);
    const hipError_t e = hipStreamSynchronize(s.stream);
    dev_free(tmp);
    if (rc) return rc;
    if (e != hipSuccess) return fail(MGGX_EHIP, "exclusive_scan: %s", hipGetErrorString(e));
    if (w[0] > 0x7fffffffLL) return fail(MGGX_ELIMIT, "exclusive_scan: total %lld exceeds int32", w[0]);
    if (total_host) *total_host = w[0];
    return MGGX_OK;
}

int exclusive_scan_i32(const int *d_in, int *d_out, int n, long long *total_host) { return scan_total(ScanArray{d_in}, d_out, n, total_host); }

// A plan that was used inside a stream capture leaves the cache like any other, but a captured graph still holds the
// addresses of its device arrays: those are retired (freed by mggx_release_cached), not freed.
void plan_free(Plan *p)
{
    if (!p) return;
    if (p->pinned) {
        retire_block(p->d_desc, sizeof(int4) * (size_t)std::max(p->num_parts, 1));
        retire_block(p->d_off, sizeof(int) * ((size_t)p->rows + 1));
        retire_block(p->d_empty_rows, sizeof(int) * (size_t)std::max(p->rows, 1));
    } else {
        dev_free(p->d_desc);
        dev_free(p->d_off);
        dev_free(p->d_empty_rows);
    }
    dev_free(p->d_chain);  // (captured calls do not use it)
    guard_free(p->guard, p->pinned);
    delete p;
}

// Rows without partitions, and what the host needs to know of a plan, in one wait: words[1] = number of those rows,
// words[2] = *d_a, words[3] = *d_b (of plans by the library the most descriptors of a row), words[4] = largest of the *d_cnt_r ids in d_col_r,
// words[5] = *d_cnt_r (NULL: 0).  Each launch here is 4 to 5 us of a plan's build, whatever it does: everything is cleared in one.
static int plan_finish(Plan *p, const int *d_a, const int *d_b, long long **words, const int *d_col_r = nullptr, const int *d_cnt_r = nullptr)
{
    State &s = state();
    int *d_counter = nullptr;  // rows without partitions, longest row, largest remote id
    int rc = host_words(words);
    if (!rc) rc = dev_array(&d_counter, 3);
    if (!rc) rc = dev_array(&p->d_empty_rows, (size_t)p->rows);
    const bool plain = p->blocks == 1 && !p->d_part_ptr;  // (the caller's partition arrays may list a row's partitions apart)
    if (!rc && plain) rc = dev_array(&p->d_chain, FUSE_MAX_WORKGROUPS);
    if (rc) {
        dev_free(d_counter);
        return rc;
    }
    k_clear_plan<<<1, 1024, 0, s.stream>>>(d_counter, 3, p->d_chain, plain ? FUSE_MAX_WORKGROUPS : 0);
    if (d_col_r && d_cnt_r) k_max_i32<<<256, 256, 0, s.stream>>>(d_col_r, d_cnt_r, d_counter + 2);
    if (p->rows > 0) {
        const unsigned blocks = (unsigned)std::min((p->rows - 1) / EMPTY_THREADS + 1, EMPTY_WORKGROUPS);
        k_collect_empty<<<blocks, EMPTY_THREADS, 0, s.stream>>>(p->d_off, p->rows, p->d_empty_rows, d_counter, plain ? d_counter + 1 : nullptr);
    }
    long long *const w = *words + 1;  // word 0 holds the total of a scan in flight
    k_publish<<<1, 1, 0, s.stream>>>(d_counter, d_a, plain ? d_counter + 1 : d_b, w, d_counter + 2, d_cnt_r);
    const hipError_t el = hipGetLastError(), e = hipStreamSynchronize(s.stream);
    dev_free(d_counter);
    if (el != hipSuccess || e != hipSuccess) return fail(MGGX_EHIP, "plan: %s", hipGetErrorString(el != hipSuccess ? el : e));
    p->num_empty = (int)w[0];
    if (plain) p->longest = (int)w[2];
    return MGGX_OK;
}

// The cache keeps the 16 most recently used plans (front = least recently used); plans a captured graph may point at
// are never evicted.
static void cache_insert(Plan *p)
{
    State &s = state();
    const size_t max_plans = 16;
    p->bytes = sizeof(int4) * (size_t)std::max(p->num_parts, 1) + sizeof(int) * ((size_t)p->rows + 1) + sizeof(int) * (size_t)std::max(p->rows, 1);
    if (s.plans.size() >= max_plans) {
        for (size_t i = 0; i < s.plans.size(); ++i)
            if (!s.plans[i]->pinned) {
                (void)hipStreamSynchronize(s.stream);
                plan_free(s.plans[i]);
                s.plans.erase(s.plans.begin() + (long)i);
                break;
            }
    }
    s.plans.push_back(p);
}

// A cache hit: most recently used last; a plan used while capturing stays for good.
static Plan *cache_hit(size_t i)
{
    State &s = state();
    Plan *p = s.plans[i];
    if (i + 1 != s.plans.size()) {
        s.plans.erase(s.plans.begin() + (long)i);
        s.plans.push_back(p);
    }
    if (!p->pinned && capturing()) p->pinned = true;
    return p;
}

struct BuildClock {  // adds the host-clock time of a plan build to the library's set-up account
    std::chrono::steady_clock::time_point t0 = std::chrono::steady_clock::now();
    ~BuildClock() { state().plan_build_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count(); }
};
static const char *const CAPTURE_MSG = "plan: first use of this CSR and partition size inside a stream capture; call once outside the capture first";

// Plans belong to the graph record (GraphInfo) they were built under: the record vouches for what the arrays hold (its
// edge counts, its fingerprint), so a plan is found by its addresses AND that record's serial, and it goes when the record
// goes.  A later record of the same addresses -- the arrays may hold another graph by then -- builds its own.
static void drop_plans_of_record(int serial)
{
    State &s = state();
    if (serial == 0) return;
    bool synced = false;
    const auto sync_once = [&]() {
        if (!synced && s.device >= 0) (void)hipDeviceSynchronize();  // kernels in flight on either stream may still read them
        synced = true;
    };
    for (size_t i = 0; i < s.plans.size();) {
        if (s.plans[i]->graph_serial == serial) {
            sync_once();
            Plan *p = s.plans[i];
            s.plans.erase(s.plans.begin() + (long)i);
            plan_free(p);
        } else {
            ++i;
        }
    }
    std::vector<CorePlan *> gone;
    for (size_t i = 0; i < s.cores.size();) {
        if (s.cores[i]->graph_serial == serial) {
            gone.push_back(s.cores[i]);
            s.cores.erase(s.cores.begin() + (long)i);
        } else {
            ++i;
        }
    }
    if (!gone.empty()) sync_once();
    for (CorePlan *c : gone) core_plan_free(c);  // forgets the records (and so the plans) of its remainder CSR in turn
}

int plan_get(const int *d_ptr_l, const int *d_ptr_r, const int *d_col_r, int rows, int ps, int graph_serial, Plan **out)
{
    State &s = state();
    for (size_t i = 0; i < s.plans.size(); ++i) {
        const Plan *p = s.plans[i];
        if (p->d_ptr_l == d_ptr_l && p->d_ptr_r == d_ptr_r && p->d_col_r == d_col_r && p->rows == rows && p->ps == ps &&
            !p->d_part_ptr && p->blocks == 1 && !p->unsuitable && p->graph_serial == graph_serial) {
            *out = cache_hit(i);
            return MGGX_OK;
        }
    }
    if (capturing()) return fail(MGGX_EINVAL, "%s", CAPTURE_MSG);
    BuildClock clock;
    Plan *p = new Plan;
    p->graph_serial = graph_serial;
    p->d_ptr_l = d_ptr_l;
    p->d_ptr_r = d_ptr_r;
    p->d_col_r = d_col_r;  // the plan holds the largest remote id
    p->rows = rows;
    p->real_rows = rows;
    p->ps = ps;
    p->unit = unit_of(ps);
    const int unit = p->unit;  // neighbors per descriptor: whole partitions of one row and side, at most 16 neighbors (ps < 16)
    int rc = MGGX_OK;
    void *scan_tmp = nullptr;
    do {
        // One wait for everything the host needs: the number of descriptors, the edge counts, the largest remote id, the
        // number of rows without neighbors.
        if ((rc = dev_array(&p->d_off, (size_t)rows + 1))) break;
        const bool remote = d_ptr_r && rows > 0;
        if (rows > 0) {
            if ((rc = dev_alloc(&scan_tmp, scan_tmp_bytes(rows)))) break;
            long long *w = nullptr;
            if ((rc = host_words(&w))) break;
            rc = scan_launch(ScanParts{d_ptr_l, d_ptr_l + 1, d_ptr_r, d_ptr_r ? d_ptr_r + 1 : nullptr, unit}, p->d_off, rows, scan_tmp, w);
            if (rc) break;
        } else if (hipMemsetAsync(p->d_off, 0, sizeof(int), s.stream) != hipSuccess) {
            rc = fail(MGGX_EHIP, "plan: row offsets");
            break;
        }
        long long *w = nullptr;
        if ((rc = plan_finish(p, rows > 0 ? d_ptr_l + rows : nullptr, nullptr, &w, remote ? d_col_r : nullptr, remote ? d_ptr_r + rows : nullptr))) break;
        if (rows > 0) {
            if (w[0] > 0x7fffffffLL) {
                rc = fail(MGGX_ELIMIT, "exclusive_scan: total %lld exceeds int32", w[0]);
                break;
            }
            p->num_parts = (int)w[0];
            p->nnz_l = w[2];
            p->nnz_r = w[5];
            if (p->nnz_r > 0) {
                if (!d_col_r) {
                    rc = fail(MGGX_EINVAL, "plan: remote edges but no remote column array");
                    break;
                }
                p->max_col_r = (int)w[4];
            }
        }
        if ((rc = dev_array(&p->d_desc, (size_t)p->num_parts))) break;
        if (p->num_parts > 0) {
            k_fill_desc<<<(p->num_parts + 255) / 256, 256, 0, s.stream>>>(p->d_off, d_ptr_l, d_ptr_l + 1, d_ptr_r,
                                                                          d_ptr_r ? d_ptr_r + 1 : nullptr, rows, unit, p->num_parts,
                                                                          p->d_desc);
            if (hipGetLastError() != hipSuccess) rc = fail(MGGX_EHIP, "plan: descriptor kernel launch failed");
            // a cached plan may be used on another stream next: it is complete when the call that builds it goes on
            else if (hipStreamSynchronize(s.stream) != hipSuccess) rc = fail(MGGX_EHIP, "plan: descriptors");
        }
    } while (0);
    dev_free(scan_tmp);
    if (rc) {
        plan_free(p);
        return rc;
    }
    cache_insert(p);
    *out = p;
    return MGGX_OK;
}

size_t explicit_tmp_ints(int rows)
{
    // first partition of each row | units per row | scan scratch
    return 2 * ((size_t)rows + 1) + (scan_tmp_bytes(rows) + sizeof(int) - 1) / sizeof(int) + 2;
}

// Descriptors and row offsets of explicit partition arrays into caller-provided device arrays (kernels on the library's
// stream, nothing else).
int explicit_desc_fill(const int *d_row_ptr, const int *d_part_ptr, const int *d_part2node, int rows, int num_parts, int ps,
                       int4 *d_desc, int *d_off, int *d_tmp, long long *units_bound)
{
    State &s = state();
    const int g = unit_of(ps) / ps;
    if (g <= 1 || rows <= 0 || num_parts <= 0) {
        k_off_from_parts<<<(rows + 1 + 255) / 256, 256, 0, s.stream>>>(d_part2node, num_parts, rows, d_off);
        if (num_parts > 0)
            k_desc_from_parts<<<(num_parts + 255) / 256, 256, 0, s.stream>>>(d_row_ptr, d_part_ptr, d_part2node, num_parts, ps, d_desc);
        if (hipGetLastError() != hipSuccess) return fail(MGGX_EHIP, "plan: explicit descriptor kernel launch failed");
        if (units_bound) *units_bound = num_parts;
        return MGGX_OK;
    }
    int *off_p = d_tmp, *cnt = d_tmp + ((size_t)rows + 1);
    long long *scan_tmp = reinterpret_cast<long long *>((reinterpret_cast<uintptr_t>(cnt + rows + 1) + 7) & ~(uintptr_t)7);
    k_off_from_parts<<<(rows + 1 + 255) / 256, 256, 0, s.stream>>>(d_part2node, num_parts, rows, off_p);
    k_units_per_row<<<(rows + 255) / 256, 256, 0, s.stream>>>(off_p, rows, g, cnt);
    const int rc = exclusive_scan_i32_device(cnt, d_off, rows, scan_tmp);
    if (rc) return rc;
    const long long bound = explicit_units_bound(rows, num_parts, ps);
    k_desc_from_units<<<(unsigned)((bound + 255) / 256), 256, 0, s.stream>>>(d_row_ptr, d_part_ptr, off_p, d_off, rows, ps, g, d_desc);
    if (hipGetLastError() != hipSuccess) return fail(MGGX_EHIP, "plan: explicit unit kernel launch failed");
    if (units_bound) *units_bound = bound;
    return MGGX_OK;
}

int plan_get_explicit(const int *d_row_ptr, const int *d_part_ptr, const int *d_part2node, int rows, int num_parts,
                      int ps, Plan **out)
{
    State &s = state();
    for (size_t i = 0; i < s.plans.size(); ++i) {
        const Plan *p = s.plans[i];
        if (p->d_ptr_l == d_row_ptr && p->d_part_ptr == d_part_ptr && p->d_part2node == d_part2node && p->rows == rows &&
            p->ps == ps && p->caller_parts == num_parts) {
            *out = cache_hit(i);
            return MGGX_OK;
        }
    }
    if (capturing()) return fail(MGGX_EINVAL, "%s", CAPTURE_MSG);
    BuildClock clock;
    Plan *p = new Plan;
    p->d_ptr_l = d_row_ptr;
    p->d_part_ptr = d_part_ptr;
    p->d_part2node = d_part2node;
    p->rows = rows;
    p->real_rows = rows;
    p->ps = ps;
    p->unit = unit_of(ps);
    p->caller_parts = num_parts;
    p->num_parts = num_parts;
    int rc = MGGX_OK;
    int *d_tmp = nullptr;
    do {
        long long bound = num_parts;
        if ((rc = dev_array(&p->d_off, (size_t)rows + 1)) || (rc = dev_array(&p->d_desc, (size_t)num_parts)) ||
            (p->unit != ps && (rc = dev_array(&d_tmp, explicit_tmp_ints(rows)))))
            break;
        rc = explicit_desc_fill(d_row_ptr, d_part_ptr, d_part2node, rows, num_parts, ps, p->d_desc, p->d_off, d_tmp, &bound);
        if (rc) break;
        long long *w = nullptr;
        rc = plan_finish(p, rows > 0 ? d_row_ptr + rows : nullptr, rows > 0 ? p->d_off + rows : nullptr, &w);
        if (rc) break;
        const int end = (int)w[2];
        p->num_parts = rows > 0 ? (int)w[3] : 0;  // several partitions of a row per descriptor when ps < 16 (Plan::unit)
        p->nnz_l = end;
        // the descriptors depend on these three arrays (the column array is only read while aggregating)
        p->guard.arr[0] = d_row_ptr;
        p->guard.len[0] = (long long)rows + 1;
        p->guard.arr[1] = d_part_ptr;
        p->guard.len[1] = num_parts;
        p->guard.arr[2] = d_part2node;
        p->guard.len[2] = num_parts;
        p->guard.cnt_l = d_row_ptr + rows;
        p->guard.want_l = end;
        rc = guard_arm(p->guard);
    } while (0);
    dev_free(d_tmp);
    if (rc) {
        plan_free(p);
        return rc;
    }
    cache_insert(p);
    *out = p;
    return MGGX_OK;
}

int plan_get_blocked(const int *d_ptr_l, const int *d_col_l, int rows, int lb, int ps, int block_rows, int graph_serial, Plan **out)
{
    State &s = state();
    for (size_t i = 0; i < s.plans.size(); ++i) {
        const Plan *p = s.plans[i];
        if (p->d_ptr_l == d_ptr_l && p->d_col_l == d_col_l && p->real_rows == rows && p->ps == ps && p->block_rows == block_rows && p->block_lb == lb &&
            (p->blocks > 1 || p->unsuitable) && p->graph_serial == graph_serial) {
            *out = cache_hit(i);
            return MGGX_OK;
        }
    }
    if (capturing()) return fail(MGGX_EINVAL, "%s", CAPTURE_MSG);
    BuildClock clock;
    if (block_rows < 1 || rows < 1) return fail(MGGX_EINVAL, "plan: column blocks of %d rows over %d rows", block_rows, rows);
    const long long blocks = ((long long)rows + block_rows - 1) / block_rows;
    const long long vrows = blocks * rows;
    if (blocks < 2 || vrows + rows > 0x7fffffffLL) return fail(MGGX_ELIMIT, "plan: %lld column blocks over %d rows", blocks, rows);
    Plan *p = new Plan;
    p->graph_serial = graph_serial;
    p->d_ptr_l = d_ptr_l;
    p->d_col_l = d_col_l;
    p->real_rows = rows;
    p->ps = ps;
    p->unit = unit_of(ps);
    const int unit = p->unit;
    p->block_rows = block_rows;
    p->block_lb = lb;
    int rc = MGGX_OK;
    int *d_vbeg = nullptr, *d_flag = nullptr;
    void *scan_tmp = nullptr;
    long long *w = nullptr;
    do {
        if ((rc = host_words(&w)) || (rc = dev_array(&d_flag, 1))) break;
        k_zero_words<<<1, 64, 0, s.stream>>>(d_flag, 1);
        k_check_sorted<<<(rows + 3) / 4, 256, 0, s.stream>>>(d_ptr_l, d_col_l, rows, d_flag);
        k_publish<<<1, 1, 0, s.stream>>>(d_flag, nullptr, nullptr, w);
        const hipError_t e = hipStreamSynchronize(s.stream);
        if (e != hipSuccess) {
            rc = fail(MGGX_EHIP, "plan: sortedness check: %s", hipGetErrorString(e));
            break;
        }
        if (w[0]) {  // remember the answer; the caller falls back to the plain plan
            p->unsuitable = true;
            p->rows = rows;
            break;
        }
        p->rows = (int)vrows;
        p->blocks = (int)blocks;
        if ((rc = dev_array(&d_vbeg, (size_t)(vrows + rows))) || (rc = dev_array(&p->d_off, (size_t)vrows + 1)) ||
            (rc = dev_alloc(&scan_tmp, scan_tmp_bytes((int)vrows))))
            break;
        k_block_bounds<<<(unsigned)((vrows + rows + 255) / 256), 256, 0, s.stream>>>(d_ptr_l, d_col_l, rows, lb, block_rows, (int)blocks,
                                                                                   d_vbeg);
        rc = scan_launch(ScanParts{d_vbeg, d_vbeg + rows, nullptr, nullptr, unit}, p->d_off, (int)vrows, scan_tmp, w);
        if (rc) break;
        if ((rc = plan_finish(p, d_ptr_l + rows, nullptr, &w))) break;
        if (w[0] > 0x7fffffffLL) {
            rc = fail(MGGX_ELIMIT, "exclusive_scan: total %lld exceeds int32", w[0]);
            break;
        }
        p->num_parts = (int)w[0];
        p->nnz_l = w[2];
        if ((rc = dev_array(&p->d_desc, (size_t)p->num_parts))) break;
        if (p->num_parts > 0) {
            k_fill_desc<<<(p->num_parts + 255) / 256, 256, 0, s.stream>>>(p->d_off, d_vbeg, d_vbeg + rows, nullptr, nullptr, (int)vrows, unit,
                                                                          p->num_parts, p->d_desc);
            if (hipGetLastError() != hipSuccess) rc = fail(MGGX_EHIP, "plan: descriptor kernel launch failed");
            // a cached plan may be used on another stream next: it is complete when the call that builds it goes on
            else if (hipStreamSynchronize(s.stream) != hipSuccess) rc = fail(MGGX_EHIP, "plan: descriptors");
        }
    } while (0);
    dev_free(scan_tmp);
    dev_free(d_vbeg);
    dev_free(d_flag);
    if (rc) {
        plan_free(p);
        return rc;
    }
    cache_insert(p);
    *out = p;
    return MGGX_OK;
}

int graph_info(const int *d_ptr_l, const int *d_ptr_r, const int *d_col_l, const int *d_col_r, int rows, bool internal, GraphInfo **out)
{
    State &s = state();
    for (auto it = s.graphs.begin(); it != s.graphs.end(); ++it)
        if (it->d_ptr_l == d_ptr_l && it->d_ptr_r == d_ptr_r && it->d_col_l == d_col_l && it->d_col_r == d_col_r && it->rows == rows) {
            s.graphs.splice(s.graphs.end(), s.graphs, it);  // most recently used last; the record itself does not move
            if (!it->pinned && capturing()) it->pinned = true;
            *out = &*it;
            return MGGX_OK;
        }
    if (capturing()) return fail(MGGX_EINVAL, "first use of these CSR arrays inside a stream capture: call once outside the capture first");
    GraphInfo g;
    g.d_ptr_l = d_ptr_l;
    g.d_ptr_r = d_ptr_r;
    g.d_col_l = d_col_l;
    g.d_col_r = d_col_r;
    g.rows = rows;
    g.internal = internal;
    g.serial = s.next_graph_serial++;
    if (s.next_graph_serial > 0x3fffffff) s.next_graph_serial = 1;
    int ends[2] = {0, 0};
    if (rows > 0) {
        MGGX_HIP(hipStreamSynchronize(s.stream));
        MGGX_HIP(hipMemcpy(&ends[0], d_ptr_l + rows, sizeof(int), hipMemcpyDeviceToHost));
        if (d_ptr_r) MGGX_HIP(hipMemcpy(&ends[1], d_ptr_r + rows, sizeof(int), hipMemcpyDeviceToHost));
    }
    g.nnz_l = ends[0];
    g.nnz_r = ends[1];
    if (s.graphs.size() >= 32)
        for (auto it = s.graphs.begin(); it != s.graphs.end(); ++it)
            if (!it->pinned) {
                (void)hipStreamSynchronize(s.stream);  // a check kernel in flight may still write the record's verdict word
                const int serial = it->serial;
                guard_free(it->guard);
                s.graphs.erase(it);
                drop_plans_of_record(serial);  // may erase further records (the remainder CSRs of its dense-core plans)
                break;
            }
    s.graphs.push_back(g);
    GraphInfo &r = s.graphs.back();
    if (!internal && rows > 0) {
        r.guard.arr[0] = d_ptr_l;
        r.guard.len[0] = (long long)rows + 1;
        r.guard.arr[1] = d_ptr_r;
        r.guard.len[1] = d_ptr_r ? (long long)rows + 1 : 0;
        r.guard.arr[2] = g.nnz_l > 0 ? d_col_l : nullptr;
        r.guard.len[2] = g.nnz_l;
        r.guard.arr[3] = g.nnz_r > 0 ? d_col_r : nullptr;
        r.guard.len[3] = g.nnz_r;
        r.guard.cnt_l = d_ptr_l + rows;
        r.guard.want_l = ends[0];
        r.guard.cnt_r = d_ptr_r ? d_ptr_r + rows : nullptr;
        r.guard.want_r = ends[1];
        const int rc = guard_arm(r.guard);
        if (rc) {
            guard_free(r.guard);
            s.graphs.pop_back();
            return rc;
        }
    }
    *out = &r;
    return MGGX_OK;
}

// Drops every cached plan and graph record keyed by this device address (an array about to be freed or rewritten).  What a
// captured graph may still point at (records used inside a stream capture) leaves the lookup tables all the same, but its
// device blocks are retired, not freed: a replay then reads the old plan, never freed memory.
int forget_pointer(const void *d_ptr)
{
    if (!d_ptr) return MGGX_OK;  // NULL is what absent arrays are keyed by: nothing hangs on it
    State &s = state();
    bool synced = false;
    std::vector<int> orphaned;  // serials of the graph records dropped below
    for (size_t i = 0; i < s.plans.size();) {
        Plan *p = s.plans[i];
        if (p->d_ptr_l == d_ptr || p->d_ptr_r == d_ptr || p->d_col_l == d_ptr || p->d_col_r == d_ptr || p->d_part_ptr == d_ptr ||
            p->d_part2node == d_ptr) {
            if (!synced && s.device >= 0) {  // a kernel in flight may still read the plan
                MGGX_HIP(hipStreamSynchronize(s.stream));
                synced = true;
            }
            plan_free(p);
            s.plans.erase(s.plans.begin() + (long)i);
        } else {
            ++i;
        }
    }
    for (auto it = s.graphs.begin(); it != s.graphs.end();) {
        if (it->d_ptr_l == d_ptr || it->d_ptr_r == d_ptr || it->d_col_l == d_ptr || it->d_col_r == d_ptr) {
            if (!synced && s.device >= 0) {  // a check kernel in flight may still write the record's verdict word
                MGGX_HIP(hipStreamSynchronize(s.stream));
                synced = true;
            }
            guard_free(it->guard, it->pinned);
            orphaned.push_back(it->serial);
            it = s.graphs.erase(it);
        } else {
            ++it;
        }
    }
    // dense-core plans keyed by the array (freeing one forgets its own remainder arrays in turn: take them out first)
    std::vector<CorePlan *> gone;
    for (size_t i = 0; i < s.cores.size();) {
        if (s.cores[i]->d_ptr_l == d_ptr || s.cores[i]->d_col_l == d_ptr) {
            gone.push_back(s.cores[i]);
            s.cores.erase(s.cores.begin() + (long)i);
        } else {
            ++i;
        }
    }
    if (!gone.empty() && !synced && s.device >= 0) MGGX_HIP(hipStreamSynchronize(s.stream));
    for (CorePlan *c : gone) core_plan_free(c);
    for (int serial : orphaned) drop_plans_of_record(serial);  // plans of a dropped record keyed by its other arrays only
    return MGGX_OK;
}

}  // namespace mggx

using mggx::fail;

MGGX_EXPORT int mggx_forget(const void *d_ptr)
{
    if (!d_ptr) return MGGX_OK;
    return mggx::forget_pointer(d_ptr);
}

MGGX_EXPORT int mggx_build_part_device(const int *d_indptr, int num_nodes, int part_size, int compat, int *d_part_ptr,
                                       int *d_part2node, int *d_node2part, int *num_parts)
{
    if (!d_indptr || num_nodes < 0 || part_size <= 0 || !num_parts)
        return fail(MGGX_EINVAL, "build_part_device: indptr NULL, num_nodes=%d, part_size=%d", num_nodes, part_size);
    int rc = mggx::ensure_init();
    if (rc) return rc;
    mggx::State &s = mggx::state();
    int *d_n2p = d_node2part;
    bool own_n2p = false;
    if (!d_n2p) {
        rc = mggx::dev_array(&d_n2p, (size_t)num_nodes + 2);
        if (rc) return rc;
        own_n2p = true;
    }
    // One wait for the whole call: the arrays are laid out behind the scan, which leaves the number of partitions on the device.  (Asked
    // for by the host first, and waited for again behind a launch of one thread: four of the fifteen waits of a share's set-up, some 12 us each.)
    const bool layout = d_part_ptr && d_part2node;
    void *tmp = nullptr;
    long long *w = nullptr;
    do {
        if ((rc = mggx::host_words(&w)) || (rc = mggx::dev_alloc(&tmp, mggx::scan_tmp_bytes(num_nodes)))) break;
        if (num_nodes > 0) {
            rc = mggx::scan_launch(mggx::ScanParts{d_indptr, d_indptr + 1, nullptr, nullptr, part_size}, d_n2p, num_nodes, tmp, w);
            if (rc) break;
        } else {
            mggx::k_zero_words<<<1, 64, 0, s.stream>>>(d_n2p, 1);
            mggx::k_zero_words<<<1, 64, 0, s.stream>>>(static_cast<int *>(tmp), 2);
        }
        if (layout) {
            const long long *d_total = static_cast<long long *>(tmp) + (num_nodes + mggx::SCAN_TILE - 1) / mggx::SCAN_TILE;
            mggx::k_parts_ref_layout<<<1024, 256, 0, s.stream>>>(d_indptr, d_n2p, d_total, num_nodes, part_size, compat, d_part_ptr, d_part2node);
        } else if (!own_n2p) {
            mggx::k_set_tail<<<1, 1, 0, s.stream>>>(d_n2p, num_nodes);
        }
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s.stream) != hipSuccess) {
            rc = fail(MGGX_EHIP, "build_part_device: kernel failed");
            break;
        }
        const long long total = num_nodes > 0 ? w[0] : 0;
        if (total > 0x7fffffffLL) rc = fail(MGGX_ELIMIT, "exclusive_scan: total %lld exceeds int32", total);
        else if (layout && (total < 0 || total > 0x7ffffffeLL)) rc = fail(MGGX_EHIP, "build_part_device: %lld partitions", total);
        else *num_parts = (int)total;
    } while (0);
    mggx::dev_free(tmp);
    if (own_n2p) mggx::dev_free(d_n2p);
    return rc;
}

MGGX_EXPORT int mggx_split_csr_device(const int *d_ptr, const int *d_col, int lb, int ub, int *d_local_ptr,
                                      int *d_remote_ptr, int *d_local_col, int *d_remote_col, int64_t *n_local,
                                      int64_t *n_remote)
{
    if (!d_ptr || lb < 0 || ub < lb || !d_local_ptr || !d_remote_ptr)
        return fail(MGGX_EINVAL, "split_csr_device: NULL pointer or bad range [%d,%d)", lb, ub);
    int rc = mggx::ensure_init();
    if (rc) return rc;
    mggx::State &s = mggx::state();
    const int rows = ub - lb;
    const unsigned blocks = (unsigned)std::min<long long>(((long long)rows + 3) / 4 + 1, 256 * 64);
    if (!d_local_col || !d_remote_col) {
        // pass 1: per-row counts -> the two pointer arrays and the totals
        int *d_cnt = nullptr;
        rc = mggx::dev_array(&d_cnt, 2 * (size_t)rows);
        if (rc) return rc;
        long long tl = 0, tr = 0;
        void *tmp = nullptr;
        do {
            if (rows > 0) {
                if (!d_col) { rc = fail(MGGX_EINVAL, "split_csr_device: NULL column array"); break; }
                mggx::k_split_count<<<blocks, 256, 0, s.stream>>>(d_ptr, d_col, lb, ub, d_cnt, d_cnt + rows);
            }
            if (rows == 0) {
                mggx::k_zero_words<<<1, 64, 0, s.stream>>>(d_local_ptr, 1);
                mggx::k_zero_words<<<1, 64, 0, s.stream>>>(d_remote_ptr, 1);
                if (hipGetLastError() != hipSuccess) rc = fail(MGGX_EHIP, "split_csr_device: launch failed");
                break;
            }
            // both scans, one wait
            long long *w = nullptr;
            const size_t scan_bytes = mggx::scan_tmp_bytes(rows);
            if ((rc = mggx::host_words(&w)) || (rc = mggx::dev_alloc(&tmp, 2 * scan_bytes))) break;
            if ((rc = mggx::scan_launch(mggx::ScanArray{d_cnt}, d_local_ptr, rows, tmp, w)) ||
                (rc = mggx::scan_launch(mggx::ScanArray{d_cnt + rows}, d_remote_ptr, rows, static_cast<char *>(tmp) + scan_bytes, w + 1)))
                break;
            const hipError_t e = hipStreamSynchronize(s.stream);
            if (e != hipSuccess) rc = fail(MGGX_EHIP, "exclusive_scan: %s", hipGetErrorString(e));
            else if (std::max(w[0], w[1]) > 0x7fffffffLL) rc = fail(MGGX_ELIMIT, "exclusive_scan: total %lld exceeds int32", std::max(w[0], w[1]));
            tl = w[0];
            tr = w[1];
        } while (0);
        mggx::dev_free(tmp);
        mggx::dev_free(d_cnt);
        if (rc) return rc;
        if (n_local) *n_local = tl;
        if (n_remote) *n_remote = tr;
        return MGGX_OK;
    }
    // pass 2: fill, using the pointer arrays of pass 1
    if (rows > 0) {
        mggx::k_split_fill<<<blocks, 256, 0, s.stream>>>(d_ptr, d_col, lb, ub, d_local_ptr, d_remote_ptr, d_local_col, d_remote_col);
        MGGX_LAUNCH_CHECK("k_split_fill");
    }
    return MGGX_OK;
}
