// Dense cells of a power-law graph on the matrix cores.
//
// Rank the rows of a local CSR by degree and cut the (row rank, column rank) plane into cells of 512 rows x 192 columns.  Where the
// hubs meet, cells are full of edges (the 233 K-node benchmark graph: 87 % of its 228 M edges lie in cells that hold 1,400 and more), and
// one gathered row per edge, from whatever cache or LDS, is more than such a cell costs as a matrix product: 0/1 rows times the
// columns' feature rows.  The features are split exactly into three bf16 parts, x = x1 + x2 + x3 (24 mantissa bits), so every product
// is the part itself and is added in fp32: fp32 sums at the bf16 matrix cores' rate.  A cell costs the same whatever it holds; an edge
// elsewhere costs a gathered row: cells below a number of edges stay out (cells_least_edges).  Every edge outside the kept cells stays
// in a CSR of its own, which the gather kernel sums afterwards, and the kernel that finishes the rows adds the two.
//
// The matrix instruction is v_smfmac_f32_16x16x64_bf16, whose first operand is 2 : 4 sparse: of every four columns a row takes at
// most two, each named by a 2-bit index, in the time a dense instruction takes for half the columns.  The 0/1 rows are that operand.
// Every fourth column position is a column of zeros, so that a slot without a neighbor has something to name: the operand's values
// are the constant 1 then, only the indexes are read from memory and nothing is unpacked.  A row's third neighbor among three columns
// goes to a second layer, a cell of its own.  (233 K nodes, width 41, same edges in cells: dense v_mfma_f32_16x16x32_bf16 with bitmaps
// unpacked by shifts and masks, 256 x 256 cells: 13.7 ns per 65,536 positions; sparse with four real columns and a bit per slot that says
// whether it is set: 10.0, the vector ALUs as busy as the matrix cores; this form: 9.6, with a quarter fewer bytes.)
//
// Before this, the core of such a graph came from the LDS, index list by index list, beside the gather kernel (mggx_core.hip, still the
// faster one where less of a graph lies in cells): the 233 K-node benchmark graph, us per aggregation at width 16 515 -> 367, width 41 with
// the softmax 1,305 -> 931; first use of a width 22.0 and 17.7 -> 12.8 and 11.9 ms; error against 64 bits 3.1e-7 -> 1.6e-7 of the result.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <new>

#include <rocprim/device/device_radix_sort.hpp>

#include "mggx_dev.h"

namespace mggx {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v16bf __attribute__((ext_vector_type(16)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int TILE = 256;                    // column positions of a cell; position 4 k + 3 is a column of zeros: 192 ranks
constexpr int TILE_RANKS = TILE / 4 * 3;
constexpr int GROUP = 512, GROUP_SHIFT = 9;  // rows of a cell: four wavefronts of 128
constexpr int STEPS = TILE / 64;             // matrix instructions along a cell
constexpr int LANE_WORDS = 16;               // a lane's words of a cell: 8 row blocks x 2
constexpr int CELL_WORDS = 4 * 64 * LANE_WORDS;
constexpr int MAX_TILES = 640;               // ranks looked at: the 122,880 of highest degree

__host__ __device__ constexpr int position_of(int rank) { return rank + rank / 3; }

// ---- the plan ----

__global__ void __launch_bounds__(256) k_cells_deg(const int *__restrict__ ptr, int rows, int *__restrict__ deg, int *__restrict__ ids, int *__restrict__ keep)
{
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= rows) return;
    const int d = ptr[v + 1] - ptr[v];
    deg[v] = keep[v] = d;
    ids[v] = v;
}

// sorted = row ids by falling degree (ties by rising id); order[i] = row of rank i, -1 for the ranks that fill up the last tile
__global__ void __launch_bounds__(256) k_cells_rank(const int *__restrict__ sorted, int rows, int ranked, int padded, int *__restrict__ order, int *__restrict__ rank)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < padded) order[i] = i < ranked ? sorted[i] : -1;
    if (i < rows) rank[sorted[i]] = i < ranked ? i : -1;
}

constexpr int ROWS_WG = 8;  // consecutive ranks (of one row group) per workgroup of the passes over the edges

// The workgroup's 256 threads go over the edges [beg, end) of a row, four edges per thread in flight: f(e0, u, j), this thread's edges
// being e0 + 256 q + threadIdx.x, q = 0..3; u: neighbor (0-based in the share, -1 past the end), j: its rank or -1.
template <typename F>
__device__ __forceinline__ void for_edges(const int *__restrict__ col, int beg, int end, const int *__restrict__ rank, int rows, int lb, F f)
{
    for (int e0 = beg; e0 < end; e0 += 1024) {
        int u[4], j[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = e0 + q * 256 + (int)threadIdx.x;
            u[q] = e < end ? col[e] - lb : -1;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) j[q] = (unsigned)u[q] < (unsigned)rows ? rank[u[q]] : -1;
        f(e0, u, j);
    }
}

// This row's neighbors in rank space as a bitmap in LDS, tile after tile of 8 words (map: all zero on entry).  -> 1 in *twice where the
// row lists a neighbor twice, which a bitmap cannot hold.
__device__ __forceinline__ void row_map(unsigned *map, const int *__restrict__ col, int beg, int end, const int *__restrict__ rank, int rows, int lb, int *twice)
{
    for_edges(col, beg, end, rank, rows, lb, [&](int, const int (&)[4], const int (&j)[4]) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (j[q] >= 0) {
                const int at = position_of(j[q]);
                const unsigned bit = 1u << (at & 31);
                if (atomicOr(&map[at >> 5], bit) & bit) *twice = 1;
            }
    });
}
// of every four positions (4 bits of w, the highest never set) the first two that are set: all but the third of three
__device__ __forceinline__ unsigned first_two(unsigned w) { return w & ~((w & (w << 1) & (w << 2)) & 0x44444444u); }

// cnt[((group * ntiles) + tile) * 2 + layer] += edges of these rows in that cell (layer 0: the first two of every four positions)
__global__ void __launch_bounds__(256) k_cells_count(const int *__restrict__ ptr, const int *__restrict__ col, const int *__restrict__ rank,
                                                     const int *__restrict__ sorted, int ranked, int rows, int lb, int ntiles, int *__restrict__ cnt,
                                                     int *__restrict__ twice)
{
    __shared__ unsigned map[MAX_TILES * 8];
    __shared__ int hist[MAX_TILES * 2];
    const int r0 = (int)blockIdx.x * ROWS_WG;
    for (int t = threadIdx.x; t < 2 * ntiles; t += 256) hist[t] = 0;
    for (int t = threadIdx.x; t < 8 * ntiles; t += 256) map[t] = 0;
    __syncthreads();
    for (int k = 0; k < ROWS_WG && r0 + k < ranked; ++k) {
        const int v = sorted[r0 + k];
        row_map(map, col, ptr[v], ptr[v + 1], rank, rows, lb, twice);
        __syncthreads();
        for (int t = threadIdx.x; t < 8 * ntiles; t += 256) {
            const unsigned w = map[t];
            if (!w) continue;
            const int all = __popc(w), first = __popc(first_two(w));
            atomicAdd(&hist[(t >> 3) * 2], first);
            if (all > first) atomicAdd(&hist[(t >> 3) * 2 + 1], all - first);
            map[t] = 0;
        }
        __syncthreads();
    }
    int *row = cnt + (size_t)(r0 >> GROUP_SHIFT) * ntiles * 2;
    for (int t = threadIdx.x; t < 2 * ntiles; t += 256)
        if (hist[t]) atomicAdd(&row[t], hist[t]);
}

// A cell as k_cells takes it: lane (i, q) = (L % 16, L / 16) of wavefront w holds row 128 w + 16 rb + i and of every step of 64
// positions the sixteen from 16 q on, four bits per four: two indexes, 3 where there is no neighbor to name.  Two steps to a word, as the
// instruction reads them, two words per row block: word[w][rb / 2][L][2 (rb % 2) + step / 2].
__device__ __forceinline__ size_t word_at(size_t cell, int wave, int rb, int lane, int k)
{
    return cell * CELL_WORDS + (size_t)((wave * (LANE_WORDS / 4) + (rb >> 1)) * 64 + lane) * 4 + 2 * (rb & 1) + k;
}

// Rows of kept cells: writes their words and counts what the row keeps in the remaining CSR.  cell_of[(group * ntiles + tile) * 2 + layer]:
// index of the kept cell or -1.  Rows past the last one are written empty.
__global__ void __launch_bounds__(256) k_cells_fill(const int *__restrict__ ptr, const int *__restrict__ col, const int *__restrict__ rank,
                                                    const int *__restrict__ sorted, int ranked, int rows, int lb, int ntiles, const int *__restrict__ cell_of,
                                                    unsigned *__restrict__ words, int *__restrict__ keep)
{
    __shared__ unsigned map[MAX_TILES * 8];
    __shared__ int cell[MAX_TILES * 2];
    __shared__ int in_cells;
    const int r0 = (int)blockIdx.x * ROWS_WG;
    for (int t = threadIdx.x; t < 2 * ntiles; t += 256) cell[t] = cell_of[(size_t)(r0 >> GROUP_SHIFT) * ntiles * 2 + t];
    for (int t = threadIdx.x; t < 8 * ntiles; t += 256) map[t] = 0;
    if (threadIdx.x == 0) in_cells = 0;
    __syncthreads();
    for (int k = 0; k < ROWS_WG; ++k) {
        const int r = (r0 + k) & (GROUP - 1), v = r0 + k < ranked ? sorted[r0 + k] : -1;
        const int beg = v >= 0 ? ptr[v] : 0, end = v >= 0 ? ptr[v + 1] : 0;
        int ignore = 0;  // (the counting pass has refused parallel edges)
        row_map(map, col, beg, end, rank, rows, lb, &ignore);
        __syncthreads();
        int mine = 0;
        for (int p = threadIdx.x; p < ntiles * 4; p += 256) {
            const int tile = p >> 2, q = p & 3;
            if (cell[2 * tile] < 0 && cell[2 * tile + 1] < 0) continue;
#pragma unroll
            for (int layer = 0; layer < 2; ++layer) {
                const int id = cell[2 * tile + layer];
                if (id < 0) continue;
                unsigned index[2] = {0, 0};
#pragma unroll
                for (int st = 0; st < STEPS; ++st) {
                    const unsigned w = (map[tile * 8 + 2 * st + (q >> 1)] >> (16 * (q & 1))) & 0xFFFFu;
                    const unsigned on = layer ? w & ~first_two(w) : first_two(w);
                    mine += __popc(on);
#pragma unroll
                    for (int four = 0; four < 4; ++four) {
                        const unsigned m = (on >> (4 * four)) & 7u, more = m & (m - 1);
                        const unsigned lo = m ? __ffs((int)m) - 1 : 3, hi = more ? __ffs((int)more) - 1 : 3;
                        index[st >> 1] |= (lo | (hi << 2)) << (16 * (st & 1) + 4 * four);
                    }
                }
                const int lane = 16 * q + (r & 15);
                words[word_at((size_t)id, r >> 7, (r >> 4) & 7, lane, 0)] = index[0];
                words[word_at((size_t)id, r >> 7, (r >> 4) & 7, lane, 1)] = index[1];
            }
        }
        for (int o = 32; o > 0; o >>= 1) mine += __shfl_xor(mine, o, 64);
        if ((threadIdx.x & 63u) == 0 && mine) atomicAdd(&in_cells, mine);
        __syncthreads();
        for (int t = threadIdx.x; t < 8 * ntiles; t += 256) map[t] = 0;
        if (threadIdx.x == 0) {
            if (v >= 0) keep[v] = end - beg - in_cells;
            in_cells = 0;
        }
        __syncthreads();
    }
}

// The remaining CSR: every row's other edges, in edge order.  With rows of kept cells the row's bitmap says which layer an edge is in.
__global__ void __launch_bounds__(256) k_cells_rest(const int *__restrict__ ptr, const int *__restrict__ col, const int *__restrict__ rank,
                                                    const int *__restrict__ sorted, int in_groups, int rows, int lb, int ntiles, const int *__restrict__ cell_of,
                                                    const int *__restrict__ rem_ptr, int *__restrict__ rem_col)
{
    __shared__ unsigned map[MAX_TILES * 8];
    __shared__ int cell[MAX_TILES * 2];
    __shared__ int wave_kept[4];
    const int r0 = (int)blockIdx.x * ROWS_WG;
    const bool grouped = r0 < in_groups;
    if (grouped) {
        for (int t = threadIdx.x; t < 2 * ntiles; t += 256) cell[t] = cell_of[(size_t)(r0 >> GROUP_SHIFT) * ntiles * 2 + t];
        for (int t = threadIdx.x; t < 8 * ntiles; t += 256) map[t] = 0;
    }
    __syncthreads();
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int k = 0; k < ROWS_WG && r0 + k < rows; ++k) {
        const int v = sorted[r0 + k];
        const int beg = ptr[v], end = ptr[v + 1];
        int w = rem_ptr[v];
        if (!grouped || rem_ptr[v + 1] - w == end - beg) {  // every neighbor stays
            for (int e = beg + (int)threadIdx.x; e < end; e += 256) rem_col[w + (e - beg)] = col[e];
            continue;
        }
        int ignore = 0;
        row_map(map, col, beg, end, rank, rows, lb, &ignore);
        __syncthreads();
        // the map becomes the edges that are in kept cells
        for (int t = threadIdx.x; t < 8 * ntiles; t += 256) {
            const unsigned all = map[t], first = first_two(all);
            map[t] = (cell[2 * (t >> 3)] >= 0 ? first : 0u) | (cell[2 * (t >> 3) + 1] >= 0 ? all & ~first : 0u);
        }
        __syncthreads();
        for_edges(col, beg, end, rank, rows, lb, [&](int e0, const int (&u)[4], const int (&j)[4]) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // in edge order: 256 edges at a time
                const bool stays = e0 + q * 256 + (int)threadIdx.x < end && (j[q] < 0 || !(map[position_of(j[q]) >> 5] >> (position_of(j[q]) & 31) & 1u));
                const unsigned long long m = __ballot(stays);
                int at = w + __popcll(m & below), all = 0;
                if (lane == 0) wave_kept[wave] = __popcll(m);
                __syncthreads();
                for (int i = 0; i < 4; ++i) {
                    if (i < wave) at += wave_kept[i];
                    all += wave_kept[i];
                }
                __syncthreads();
                if (stays) rem_col[at] = u[q] + lb;
                w += all;
            }
        });
        for (int t = threadIdx.x; t < 8 * ntiles; t += 256) map[t] = 0;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(256) k_cells_trim(int *__restrict__ rank, int rows, int limit)
{
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v < rows && rank[v] >= limit) rank[v] = -1;
}

// ---- the features of the ranked rows, split and in operand order ----

// The parts are made of x UP, so that all of them hold every bit of x down to the smallest subnormal number.  An infinity or NaN is its
// own first part: it reaches the rows that have its column, as in plain sums (columns that a row does not name are not multiplied).
// Values from 2^103 up have no parts, and sums beyond 2^104 no place: both need a feature of HUGE_VALUE and more, which the kernel that
// splits them reports.
constexpr float UP = 16777216.0f, DOWN = 1.0f / 16777216.0f;  // 2^24
constexpr float HUGE_VALUE = 1.2e24f;                         // 2^80: 2^17 columns of less stay below 2^121

__device__ __forceinline__ void split_pair(float a, float b, unsigned (&part)[3])
{
    const v2bf q = __builtin_convertvector((v2f){a, b}, v2bf);
    __builtin_memcpy(&part[0], &q, 4);
    const float a1 = __uint_as_float(part[0] << 16), b1 = __uint_as_float(part[0] & 0xFFFF0000u);
    a = __builtin_isfinite(a1) ? a - a1 : 0.f;
    b = __builtin_isfinite(b1) ? b - b1 : 0.f;
#pragma unroll
    for (int p = 1; p < 3; ++p) {
        const v2bf r = __builtin_convertvector((v2f){a, b}, v2bf);
        __builtin_memcpy(&part[p], &r, 4);
        a -= __uint_as_float(part[p] << 16);
        b -= __uint_as_float(part[p] & 0xFFFF0000u);
    }
}

// tab[(((tile * fg + f) * 4 + step) * 3 + part) * 2 + half][lane]: the 32 bytes (two halves) lane (i, q) gives
// v_smfmac_f32_16x16x64_bf16 as second operand: feature 16 f + i of the positions 32 half + 8 q .. + 7 of that step.
// huge[unit] != 0: one of the unit's features is finite and at least HUGE_VALUE.
__global__ void __launch_bounds__(256) k_cells_stage(v4u *__restrict__ tab, int *__restrict__ huge, const float *__restrict__ in, const int *__restrict__ order,
                                                     int fg, int dim, long long ld_in, int units, const Gate gate)
{
    if (gate_closed(gate)) return;
    const int unit = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63u);  // ((tile * 4 + step) * fg + f) * 2 + half
    if (unit >= units) return;
    const int half = unit & 1, f = (unit >> 1) % fg, ts = (unit >> 1) / fg, tile = ts / STEPS, step = ts % STEPS;
    const int d = 16 * f + (lane & 15);
    const int *o = order + (ts * 64 + 32 * half + 8 * (lane >> 4)) / 4 * 3;
    int row[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) row[j] = j % 4 < 3 ? o[j / 4 * 3 + j % 4] : -1;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = row[j] >= 0 && d < dim ? in[(long long)row[j] * ld_in + d] : 0.f;
    bool any = false;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        any |= __builtin_isfinite(x[j]) && fabsf(x[j]) >= HUGE_VALUE;
        x[j] *= UP;
    }
    const int any_lane = __any(any);
    if (lane == 0) huge[unit] = any_lane;
    unsigned h[4][3];
#pragma unroll
    for (int t = 0; t < 4; ++t) split_pair(x[2 * t], x[2 * t + 1], h[t]);
    v4u *dst = tab + ((((size_t)tile * fg + f) * STEPS + step) * 6 + half) * 64 + lane;
#pragma unroll
    for (int p = 0; p < 3; ++p) dst[p * 128] = (v4u){h[0][p], h[1][p], h[2][p], h[3][p]};
}

struct CellArgs {
    const unsigned *words;
    const int *cell_tile;
    const int4 *wgs, *segs;
    const v4u *tab;
    const int *huge;   // [units] of the splitting kernel
    int units;
    float *partial;    // [slot][512][4 n4]
    int n4;
    const float *in;   // for sums the matrix cores cannot give (see below)
    const int *order;
    long long ld_in;
    int dim;
    Gate gate;
};

// Where a sum is not finite and a feature is huge, the wavefront that finds it makes its rows again from the feature rows, edge by
// edge in fp32.
constexpr int PIECES = STEPS * 6 * 64;  // 16-byte pieces of a tile's 16 features: 24 KB

// One workgroup per resident place on the chip (2 or 3 per CU by registers), each with an equal share of the cells in a row (block of
// column tiles by block, row group by row group inside), a wavefront with 128 rows x 16 FG columns of sums in registers: where a share
// passes from one row group to the next the sums go out to a slot of partial rows.  The split features of a cell's columns go
// through LDS 16 features at a time (24 KB) in two buffers, asked for in halves while the ones before are multiplied (half the registers);
// a wavefront of 128 rows reads them at half the LDS's rate.  A cell's products are summed on their own, smallest parts first, before
// they join the row's sums: four additions at the size of the sum and one, instead of a chain of hundreds (233 K nodes, width 16: one
// chain 3.5e-7 of the result, this way 1.6e-7).
// Bound: at width 41 the matrix cores are busy 61 % of the time (299 us for 22,900 cells, 13.1 ns each; 330 us with an operand read right before
// its use and the sums kept to the end of the cell), the rest goes to the end of the launch, where some shares finish up to a fifth
// earlier than others, and to waits for the LDS; 1.55 of 2.9 GB come from beyond the L2s.  At width 16 113 us, 5.5 TB/s from beyond the
// L2s, 375 MB of indexes out of memory among them.  (Shares of about two per place instead of one: 3 - 5 % slower; tiles not in blocks:
// 40 % more misses, 3 % slower at width 16.)
template <int FG, int WAVES>
__global__ void __launch_bounds__(256, WAVES) k_cells(const CellArgs a)
{
    constexpr int PER_THREAD = PIECES / 256, HALF = PER_THREAD / 2;
    __shared__ v4u buf[2][PIECES];
    if (gate_closed(a.gate)) return;
    const int4 wg = a.wgs[blockIdx.x];  // {first segment, first cell, end cell, -}
    const int lane = (int)(threadIdx.x & 63u), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int seg = wg.x;
    int4 part = a.segs[seg];            // {row group, first cell, end cell, slot}
    v4f acc[8], sum[FG][8];
    v8bf one;
#pragma unroll
    for (int i = 0; i < 8; ++i) one[i] = (__bf16)1.0f;
#pragma unroll
    for (int f = 0; f < FG; ++f)
#pragma unroll
        for (int rb = 0; rb < 8; ++rb) sum[f][rb] = (v4f){0.f, 0.f, 0.f, 0.f};
    const v4u *words = reinterpret_cast<const v4u *>(a.words) + (size_t)wave * (LANE_WORDS / 4 * 64) + lane;
    unsigned m[LANE_WORDS];
    const auto ask_words = [&](int cell) {
#pragma unroll
        for (int k = 0; k < LANE_WORDS / 4; ++k) {
            const v4u t = words[(size_t)cell * (CELL_WORDS / 4) + k * 64];
            m[4 * k] = t.x; m[4 * k + 1] = t.y; m[4 * k + 2] = t.z; m[4 * k + 3] = t.w;
        }
    };
    v4u next[HALF];
    const auto ask = [&](const v4u *src, int h) {
#pragma unroll
        for (int i = 0; i < HALF; ++i) next[i] = src[(h * HALF + i) * 256 + threadIdx.x];
    };
    const auto put = [&](int b, int h) {
#pragma unroll
        for (int i = 0; i < HALF; ++i) buf[b][threadIdx.x + (h * HALF + i) * 256] = next[i];
    };
    int tile = a.cell_tile[wg.y], b = 0;
    ask_words(wg.y);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        ask(a.tab + (size_t)tile * FG * PIECES, h);
        put(0, h);
    }
    __syncthreads();
    for (int cell = wg.y; cell < wg.z; ++cell) {
        const bool last = cell + 1 == wg.z;
        const int next_tile = last ? tile : a.cell_tile[cell + 1];
#pragma unroll
        for (int f = 0; f < FG; ++f) {
            const v4u *src = a.tab + ((size_t)(f + 1 < FG ? tile : next_tile) * FG + (f + 1) % FG) * PIECES;  // (after the last cell: not used)
            ask(src, 0);
            unsigned touched = 0;  // brings the next cell's words into the L2
            if (f == 0 && lane < LANE_WORDS * 2) touched = a.words[(size_t)(last ? cell : cell + 1) * CELL_WORDS + wave * (LANE_WORDS * 64) + lane * 32];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) acc[rb] = (v4f){0.f, 0.f, 0.f, 0.f};
            // The smallest parts of the whole cell first: what is added at the size of the sum is four products.  An operand is read from
            // the LDS while the products of the one before are on their way (left to the compiler, it is read right before its use).
            v4u x[2][2];
            const auto read = [&](int k) {  // k = 4 (2 - part) + step
                const int at = ((k & 3) * 6 + 2 * (2 - (k >> 2))) * 64 + lane;
                x[k & 1][0] = buf[b][at];
                x[k & 1][1] = buf[b][at + 64];
            };
            read(0);
#pragma unroll
            for (int k = 0; k < 3 * STEPS; ++k) {
                const int st = k & 3;
                if (k == 6) {
                    put(b ^ 1, 0);
                    ask(src, 1);
                }
                if (k + 1 < 3 * STEPS) read(k + 1);
                __builtin_amdgcn_sched_barrier(0);
                v16bf xk;
                const unsigned t[8] = {x[k & 1][0].x, x[k & 1][0].y, x[k & 1][0].z, x[k & 1][0].w, x[k & 1][1].x, x[k & 1][1].y, x[k & 1][1].z, x[k & 1][1].w};
                __builtin_memcpy(&xk, t, 32);
#pragma unroll
                for (int rb = 0; rb < 8; ++rb) {
                    const int index = (int)m[2 * rb + (st >> 1)];
                    acc[rb] = (st & 1) ? __builtin_amdgcn_smfmac_f32_16x16x64_bf16(one, xk, acc[rb], index, 0, 1)
                                       : __builtin_amdgcn_smfmac_f32_16x16x64_bf16(one, xk, acc[rb], index, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::"v"(touched));
            if (f + 1 == FG && !last) ask_words(cell + 1);
            put(b ^ 1, 1);
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) {
                sum[f][rb] += acc[rb];
                asm volatile("" : "+v"(sum[f][rb]));  // here, not after the next products: these 32 registers are theirs
            }
            b ^= 1;
            __syncthreads();
        }
        tile = next_tile;
        if (cell + 1 < part.z && !last) continue;
        // the last cell of this row group here: its sums go out
        __builtin_amdgcn_sched_barrier(0);
        const int w4 = 4 * a.n4;
        const unsigned first = (unsigned)((lane >> 4) * 4 * w4 + (lane & 15));  // this lane's place in a row block's 16 rows
        float *out = a.partial + ((size_t)part.w * GROUP + (size_t)wave * 128) * w4;
        float check = 0.f;
#pragma unroll
        for (int f = 0; f < FG; ++f) {
#pragma unroll
            for (int rb = 0; rb < 8; ++rb)
#pragma unroll
                for (int t = 0; t < 4; ++t) check += 0.f * sum[f][rb][t];
            if (16 * f + (lane & 15) < w4) {
#pragma unroll
                for (int rb = 0; rb < 8; ++rb)
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        (out + 16 * f + (16 * rb + t) * w4)[first] = sum[f][rb][t] * DOWN;
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) sum[f][rb] = (v4f){0.f, 0.f, 0.f, 0.f};
        }
        bool again = __any(!(check == 0.f));
        if (again) {
            int any = 0;
            for (int u = lane; u < a.units; u += 64) any |= a.huge[u];
            again = __any(any);
        }
        if (again) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // what follows writes the same rows again, other lanes their columns
            const int d = lane;
            const bool on = lane < 16 * FG && d < a.dim;
            for (int r = 0; r < 128; ++r) {
                float s = 0.f;
                for (int c = part.y; c < part.z; ++c) {
                    const int *cols = a.order + (size_t)a.cell_tile[c] * TILE_RANKS;
                    // a lane per four: its two indexes, and the neighbors they name
                    const int st = lane >> 4;
                    const unsigned both = a.words[word_at((size_t)c, wave, r >> 4, 16 * ((lane >> 2) & 3) + (r & 15), st >> 1)] >> (16 * (st & 1) + 4 * (lane & 3)) & 15u;
#pragma unroll
                    for (int slot = 0; slot < 2; ++slot) {
                        const int k = (int)(both >> (2 * slot)) & 3, node = k < 3 ? cols[3 * lane + k] : -1;
                        for (unsigned long long left = __ballot(node >= 0); left; left &= left - 1) {
                            const int v = __builtin_amdgcn_readlane(node, __builtin_ctzll(left));
                            if (on) s += a.in[(long long)v * a.ld_in + d];
                        }
                    }
                }
                if (lane < 16 * FG && d < w4) out[(size_t)r * w4 + d] = s;
            }
        }
        if (!last) part = a.segs[++seg];
    }
}

// The partial rows of a row group summed, in slot order, into one row per ranked row: sums[r * n4 + q].  G lanes per row.
__global__ void __launch_bounds__(256) k_cells_reduce(v4f *__restrict__ sums, const v4f *__restrict__ partial, const int *__restrict__ wg_base, int ranks, int n4,
                                                      int g_shift, const Gate gate)
{
    if (gate_closed(gate)) return;
    const int G = 1 << g_shift;
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long r_ll = idx >> g_shift;
    const int q = (int)(idx & (G - 1));
    if (r_ll >= ranks || q >= n4) return;
    const int r = (int)r_ll, group = r >> GROUP_SHIFT;
    const int s1 = wg_base[group + 1];
    int slot = wg_base[group];
    const size_t stride = (size_t)GROUP * n4;
    const v4f *src = partial + (size_t)(r & (GROUP - 1)) * n4 + q;
    v4f sum = {0.f, 0.f, 0.f, 0.f};
    for (; slot + 4 <= s1; slot += 4) {  // four partial rows in flight, summed in order
        const v4f p0 = src[(size_t)slot * stride], p1 = src[(size_t)(slot + 1) * stride];
        const v4f p2 = src[(size_t)(slot + 2) * stride], p3 = src[(size_t)(slot + 3) * stride];
        sum += p0;
        sum += p1;
        sum += p2;
        sum += p3;
    }
    for (; slot < s1; ++slot) sum += src[(size_t)slot * stride];
    sums[(size_t)r * n4 + q] = sum;
}

}  // namespace

// ---- host ----

namespace {

struct Temporaries {  // device temporaries of one plan build, given back on the way out
    std::vector<void *> ptrs;
    ~Temporaries()
    {
        for (void *q : ptrs) dev_free(q);
    }
    template <typename T>
    int get(T **q, size_t count)
    {
        const int rc = dev_array(q, count);
        if (!rc) ptrs.push_back(*q);
        return rc;
    }
};

int groups_of(int dim) { return (dim + 15) / 16; }

constexpr size_t L2_SHARE = (size_t)2800 << 10;   // split features of a block of column tiles: most of an XCD's 4 MB
int workgroups(int dim) { return 256 * (dim <= 16 ? 3 : 2); }  // as many as 256 CUs hold at once (k_cells' launch bounds)

int build(CorePlan *p, int dim, long long nnz, double least_share, double *share)
{
    State &s = state();
    const int rows = p->rows, lb = p->lb;
    const int ranked = std::min(rows, MAX_TILES * TILE_RANKS), ntiles = (ranked + TILE_RANKS - 1) / TILE_RANKS, ngroups = (ranked + GROUP - 1) / GROUP,
              padded = ntiles * TILE_RANKS;
    Temporaries tmp;
    int *deg = nullptr, *deg_sorted = nullptr, *ids = nullptr, *sorted = nullptr, *keep = nullptr, *cnt = nullptr, *cell_of = nullptr, *twice = nullptr;
    int rc;
    const size_t plane = (size_t)ngroups * ntiles * 2;
    if ((rc = tmp.get(&deg, (size_t)rows)) || (rc = tmp.get(&deg_sorted, (size_t)rows)) || (rc = tmp.get(&ids, (size_t)rows)) || (rc = tmp.get(&sorted, (size_t)rows)) ||
        (rc = tmp.get(&keep, (size_t)rows)) || (rc = tmp.get(&cnt, plane + 1)))
        return rc;
    cell_of = cnt;
    twice = cnt + plane;
    if ((rc = dev_array(&p->d_order, (size_t)padded)) || (rc = dev_array(&p->d_rank, (size_t)rows)) || (rc = dev_array(&p->d_rem_ptr, (size_t)rows + 1))) return rc;
    MGGX_HIP(hipMemsetAsync(cnt, 0, (plane + 1) * sizeof(int), s.stream));
    const unsigned row_blocks = (unsigned)((std::max(rows, padded) + 255) / 256);
    k_cells_deg<<<row_blocks, 256, 0, s.stream>>>(p->d_ptr_l, rows, deg, ids, keep);
    size_t need = 0;
    MGGX_HIP(rocprim::radix_sort_pairs_desc(nullptr, need, deg, deg_sorted, ids, sorted, (size_t)rows, 0, 32, s.stream));
    char *sort_tmp = nullptr;
    if ((rc = tmp.get(&sort_tmp, need))) return rc;
    MGGX_HIP(rocprim::radix_sort_pairs_desc(sort_tmp, need, deg, deg_sorted, ids, sorted, (size_t)rows, 0, 32, s.stream));
    k_cells_rank<<<row_blocks, 256, 0, s.stream>>>(sorted, rows, ranked, padded, p->d_order, p->d_rank);
    k_cells_count<<<(unsigned)((ranked + ROWS_WG - 1) / ROWS_WG), 256, 0, s.stream>>>(p->d_ptr_l, p->d_col_l, p->d_rank, sorted, ranked, rows, lb, ntiles, cnt, twice);
    MGGX_LAUNCH_CHECK("k_cells_count");
    std::vector<int> count(plane);
    int two = 0;
    MGGX_HIP(hipMemcpyAsync(count.data(), cnt, plane * sizeof(int), hipMemcpyDeviceToHost, s.stream));
    MGGX_HIP(hipMemcpyAsync(&two, twice, sizeof(int), hipMemcpyDeviceToHost, s.stream));
    MGGX_HIP(hipStreamSynchronize(s.stream));
    if (two) {  // parallel edges among the ranked rows
        p->unsuitable = true;
        return MGGX_OK;
    }
    const int least = p->asked;
    // Cells in the order they are worked on: blocks of column tiles whose split features stay in an XCD's L2, row group by row group.
    const int block_tiles = std::max(1, (int)(L2_SHARE / ((size_t)groups_of(dim) * PIECES * sizeof(v4u))));
    int ncells = 0, groups = 0, tiles = 0, areas = 0;
    long long in_cells = 0;
    std::vector<int> tile_of, group_end;  // group_end: end of the cells of a (block, group), as that group's number and the cell
    std::vector<int> group_of;
    for (int t0 = 0; t0 < ntiles; t0 += block_tiles)
        for (int g = 0; g < ngroups; ++g) {
            const int before = ncells;
            for (int t = 2 * t0; t < 2 * std::min(t0 + block_tiles, ntiles); ++t) {
                int &c = count[(size_t)g * ntiles * 2 + t];
                if (c < least) {
                    c = -1;
                    continue;
                }
                in_cells += c;
                areas += (t & 1) == 0;
                c = ncells++;
                tile_of.push_back(t / 2);
                tiles = std::max(tiles, t / 2 + 1);
            }
            if (ncells == before) continue;
            groups = std::max(groups, g + 1);
            group_of.push_back(g);
            group_end.push_back(ncells);
        }
    *share = (double)in_cells / (double)nnz;
    if (ncells == 0 || *share < least_share) {
        p->unsuitable = true;
        return MGGX_OK;
    }
    // Equal shares of the cells, one per resident workgroup, and where a share meets the cells of a row group a segment with a slot of
    // its own for partial rows; the slots of a group lie together.  Workgroups go to the XCDs in turn, neighbouring shares to the same one.
    const int nwg = std::min(workgroups(dim), ncells);
    std::vector<int4> launch, segs, shares;
    for (int w = 0, k = 0; w < nwg; ++w) {
        const int c0 = (int)((long long)ncells * w / nwg), c1 = (int)((long long)ncells * (w + 1) / nwg);
        shares.push_back(make_int4((int)segs.size(), c0, c1, 0));
        for (int c = c0; c < c1;) {
            while (group_end[(size_t)k] <= c) ++k;
            const int end = std::min(c1, group_end[(size_t)k]);
            segs.push_back(make_int4(group_of[(size_t)k], c, end, 0));
            c = end;
        }
    }
    std::vector<int> wg_base((size_t)groups + 1, 0);
    for (const int4 &q : segs) ++wg_base[(size_t)q.x + 1];
    for (int g = 0; g < groups; ++g) wg_base[(size_t)g + 1] += wg_base[(size_t)g];
    {
        std::vector<int> at(wg_base.begin(), wg_base.end() - 1);
        for (int4 &q : segs) q.w = at[(size_t)q.x]++;
    }
    for (int w = 0; w < nwg; ++w) launch.push_back(shares[(size_t)(nwg % 8 ? w : w % 8 * (nwg / 8) + w / 8)]);
    launch.insert(launch.end(), segs.begin(), segs.end());
    CorePlan::Cut cut;
    cut.nwg = nwg;
    cut.slots = (int)segs.size();
    if ((rc = dev_array(&p->d_words, (size_t)ncells * CELL_WORDS)) || (rc = dev_array(&p->d_cell_tile, (size_t)ncells)) || (rc = dev_array(&cut.d_wgs, launch.size()))) return rc;
    p->cuts.push_back(cut);
    if ((rc = dev_array(&p->cuts[0].d_wg_base, wg_base.size()))) return rc;
    MGGX_HIP(hipMemcpyAsync(cell_of, count.data(), plane * sizeof(int), hipMemcpyHostToDevice, s.stream));
    MGGX_HIP(hipMemcpyAsync(p->d_cell_tile, tile_of.data(), tile_of.size() * sizeof(int), hipMemcpyHostToDevice, s.stream));
    MGGX_HIP(hipMemcpyAsync(p->cuts[0].d_wgs, launch.data(), launch.size() * sizeof(int4), hipMemcpyHostToDevice, s.stream));
    MGGX_HIP(hipMemcpyAsync(p->cuts[0].d_wg_base, wg_base.data(), wg_base.size() * sizeof(int), hipMemcpyHostToDevice, s.stream));
    const int in_groups = std::min(groups * GROUP, ranked);
    k_cells_fill<<<(unsigned)(groups * GROUP / ROWS_WG), 256, 0, s.stream>>>(p->d_ptr_l, p->d_col_l, p->d_rank, sorted, ranked, rows, lb, ntiles, cell_of,
                                                                                     p->d_words, keep);
    MGGX_LAUNCH_CHECK("k_cells_fill");
    long long rem_nnz = 0;
    if ((rc = exclusive_scan_i32(keep, p->d_rem_ptr, rows, &rem_nnz))) return rc;
    if ((rc = dev_array(&p->d_rem_col, (size_t)rem_nnz))) return rc;
    k_cells_rest<<<(unsigned)((rows + ROWS_WG - 1) / ROWS_WG), 256, 0, s.stream>>>(p->d_ptr_l, p->d_col_l, p->d_rank, sorted, in_groups, rows, lb, ntiles, cell_of,
                                                                                p->d_rem_ptr, p->d_rem_col);
    MGGX_LAUNCH_CHECK("k_cells_rest");
    k_cells_trim<<<(unsigned)((rows + 255) / 256), 256, 0, s.stream>>>(p->d_rank, rows, in_groups);
    MGGX_LAUNCH_CHECK("k_cells_trim");
    MGGX_HIP(hipStreamSynchronize(s.stream));
    p->core = in_groups;
    p->ntiles = tiles;
    p->ncells = ncells;
    p->side = (int)std::sqrt((double)areas * GROUP * TILE_RANKS);
    p->core_nnz = in_cells;
    p->rem_nnz = rem_nnz;
    p->bytes = ((size_t)padded + 2 * (size_t)rows + 1 + (size_t)rem_nnz + (size_t)ncells + wg_base.size()) * sizeof(int) + launch.size() * sizeof(int4) +
               (size_t)ncells * CELL_WORDS * sizeof(unsigned);
    return MGGX_OK;
}

int units_of(const CorePlan *p, int dim) { return p->ntiles * STEPS * groups_of(dim) * 2; }  // wavefronts of k_cells_stage

size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

// Scratch of a call: the split features of the plan's column tiles, the partial rows, the sums.
int scratch(const CorePlan *p, int dim, v4u **tab, int **huge, v4f **partial, v4f **sums)
{
    const int n4 = (dim + 3) / 4;
    const size_t tab_bytes = up256((size_t)p->ntiles * STEPS * groups_of(dim) * 6 * 1024), huge_bytes = up256(sizeof(int) * (size_t)units_of(p, dim));
    const size_t part_bytes = up256((size_t)p->cuts[0].slots * GROUP * n4 * sizeof(v4f));
    const size_t sum_bytes = (size_t)p->core * n4 * sizeof(v4f);
    void *ws = nullptr;
    const int rc = core_workspace(tab_bytes + huge_bytes + part_bytes + sum_bytes, &ws);
    if (rc) return rc;
    char *q = static_cast<char *>(ws);
    *tab = reinterpret_cast<v4u *>(q);
    *huge = reinterpret_cast<int *>(q + tab_bytes);
    *partial = reinterpret_cast<v4f *>(q + tab_bytes + huge_bytes);
    *sums = reinterpret_cast<v4f *>(q + tab_bytes + huge_bytes + part_bytes);
    return MGGX_OK;
}

}  // namespace

int cells_sums(const CorePlan *p, const float *d_in, int dim, long long ld_in, const Gate &gate, hipStream_t stream, const float4 **d_sums)
{
    v4u *tab = nullptr;
    int *huge = nullptr;
    v4f *partial = nullptr, *sums = nullptr;
    int rc = scratch(p, dim, &tab, &huge, &partial, &sums);
    if (rc) return rc;
    const int fg = groups_of(dim), units = units_of(p, dim), n4 = (dim + 3) / 4;
    k_cells_stage<<<(unsigned)((units + 3) / 4), 256, 0, stream>>>(tab, huge, d_in, p->d_order, fg, dim, ld_in, units, gate);
    MGGX_LAUNCH_CHECK("k_cells_stage");
    const CorePlan::Cut &cut = p->cuts[0];
    const CellArgs a{p->d_words, p->d_cell_tile, cut.d_wgs, cut.d_wgs + cut.nwg, tab, huge, units, reinterpret_cast<float *>(partial), n4, d_in, p->d_order, ld_in, dim, gate};
    switch (fg) {
        case 1: k_cells<1, 3><<<(unsigned)cut.nwg, 256, 0, stream>>>(a); break;
        case 2: k_cells<2, 2><<<(unsigned)cut.nwg, 256, 0, stream>>>(a); break;
        case 3: k_cells<3, 2><<<(unsigned)cut.nwg, 256, 0, stream>>>(a); break;
        case 4: k_cells<4, 2><<<(unsigned)cut.nwg, 256, 0, stream>>>(a); break;
        default: return fail(MGGX_ELIMIT, "dense cells: dim %d outside 1..64", dim);
    }
    MGGX_LAUNCH_CHECK("k_cells");
    int g_shift = 0;
    while ((1 << g_shift) < n4) ++g_shift;
    const long long n = (long long)p->core << g_shift;
    k_cells_reduce<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(sums, partial, cut.d_wg_base, p->core, n4, g_shift, gate);
    MGGX_LAUNCH_CHECK("k_cells_reduce");
    *d_sums = reinterpret_cast<const float4 *>(sums);
    return MGGX_OK;
}

// p->asked: least edges of a cell.  A plan whose cells hold less than least_share of the edges and one of a CSR with parallel edges are marked
// unsuitable.  *share: what the cells hold, -1 with parallel edges or where the build did not get that far.
int cells_plan_build(CorePlan *p, int dim, long long nnz, double least_share, double *share)
{
    *share = -1.0;
    return build(p, dim, nnz, least_share, share);
}

}  // namespace mggx
