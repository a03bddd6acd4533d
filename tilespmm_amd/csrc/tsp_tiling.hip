// tsp_tiling.hip -- CSR -> tiles on the GPU (the csr2tile conversion of
// src/csr2tile.h:15-379,724-795 moved onto MI355X), bit-exact with the host
// conversion (tilespmm_amd/host/tiles.cpp).
//
//   1. Each row-block's entries are sorted by (column, position) where they
//      lie: a block of up to kSmall entries by one wave in registers.  A
//      larger one whose rows ascend, as nearly all do, is its rows merged
//      pairwise: up to kMedium entries by one workgroup through LDS, beyond
//      (a dense row of a circuit, the hubs of a power-law graph) by many
//      through memory.  Rows in another order are sorted by the workgroup or
//      by a rocPRIM radix sort.  The only scratch is one word per entry
//      (16 bytes for the largest blocks): its position inside the block, bit
//      31 set where a new column starts.  Entries of one (block, column) pair
//      keep the CSR order.
//   2. ceil(distinct / BN) tiles per block; one chained scan -> tile_ptr.
//   3. One wave per block (per kSmall sorted entries of a larger block) walks
//      its sorted entries, builds its tiles a few at a time in LDS -- values,
//      occupancy bits -- and writes them with whole lines, zeros included, so
//      no array is cleared first.  An entry's slot is (its local row, its
//      column's rank % BN) of tile rank / BN; the ranks are prefix counts of
//      the bit-31 flags.  A slot's first entry adds up its duplicates in CSR
//      order with the value type's rounding after every add (fp16: fp32 add
//      then round to half), exactly as on the host.  A tile's first sorted
//      entry is tile_nnz, its columns tile_colidx.
//
// The conversion is bound by memory traffic: it reads the column indices
// twice, the values once, the 4-byte scratch twice, and writes the tiles
// once.  RMAT scale 22 (128M entries) to tf32 8-row tiles: 4.6 ms of kernels,
// against 28 ms for a global radix sort of 8-byte keys over all entries with
// cleared output arrays filled by one thread per column run.
#include <cstring>
#include <hip/hip_runtime.h>
#include <rocprim/rocprim.hpp>
#include <limits.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>
#include <utility>

#include "../../include/tilespmm_hip.h"
#include "tsp_kernels.h"

// Scratch of the allocation-free packing entry point
// (tsp_tiles_pack_device_noalloc): per-block partial sums of the per-tile
// value counts, one int per kPackBlockTiles tiles, plus the total, and the
// 64-bit total in the last two ints (checked before any offset is formed,
// so the int offsets never wrap).  Every
// GPU the library runs on holds one copy for the life of the process; host
// code uses only its per-device address from hipGetSymbolAddress
// (tsp::scratch_init_current_device), never this name.
constexpr int kScratchInts = 1 << 18;                 // 1 MiB
static __device__ __align__(256) int scratch[kScratchInts];

namespace {

constexpr int kThreads = 256;

inline unsigned nblocks(long long n) { return (unsigned)((n + kThreads - 1) / kThreads); }

int bits_for(long long v)     // bits to hold values 0 .. v-1
{
    int b = 1;
    while (b < 62 && (1ll << b) < v) ++b;
    return b;
}

// ---- 1. the sorted entries of every row-block -------------------------------
constexpr int kSmallBits = 10;
constexpr int kSmall = 1 << kSmallBits;    // entries one wave sorts, and walks in step 3
constexpr int kMedium = 8192;              // entries one workgroup sorts (64 KB of LDS)
constexpr int kMediumThreads = 1024;
constexpr unsigned kHead = 0x80000000u;    // sorted entry that starts a new column

// kSmall sorted entries of a block with more than that: positions p0 ..,
// rank0 columns start before them, rank1 before the next unit.
struct Unit {
    int b, p0, rank0, rank1;
};
// A block with more than kSmall entries, its first unit and (global sort)
// its first entry there.
struct Big {
    int b, unit0;
    long long off;
};
// Zeroed before each conversion.
struct Counters {
    unsigned long long huge;               // (blocks << 40) + entries of the globally sorted blocks
    long long total;                       // tiles
    int bad;                               // a column outside [0, colA), or row pointers out of order
    int dups;                              // some row's columns do not ascend: a slot may have several entries
    int odd;                               // ... in a globally sorted block
    int nunits;
    int nmerge[2], nsort;                  // blocks of up to kMedium / 2 and kMedium entries; those to sort after all
    int ticket;                            // of the chained scan
};

// The CSR entries of row-block b.  (Entries outside ptr[0] .. ptr[rows]
// belong to the first and the last row.)
__device__ __forceinline__ void block_range(const int *__restrict__ ptr, int rows, int nnz, int bm, int tilem, int b,
                                            int &s, int &n)
{
    const long long r = (long long)b * bm;
    s = b == 0 ? 0 : min(max(ptr[r], 0), nnz);
    const int e = b == tilem - 1 ? nnz : min(max(ptr[r + bm], 0), nnz);
    n = max(e - s, 0);
    (void)rows;
}

template <typename K>
__device__ __forceinline__ void order(K &a, K &b)
{
    const K lo = a < b ? a : b, hi = a < b ? b : a;
    a = lo;
    b = hi;
}

// One stage of a bitonic merge over elements thread * R + r: element i meets
// element i ^ j, or i ^ (2j - 1) in the first stage of a merge (FLIP, which
// keeps every run ascending).  `other(v, d)` gives thread t the value that
// thread t ^ d passes.
template <int J, bool FLIP, int R, typename K, typename F>
__device__ __forceinline__ void merge_stage(K (&x)[R], int t, F &&other)
{
    if constexpr (J < R) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int p = FLIP ? r ^ (2 * J - 1) : r ^ J;
            if (p > r) order(x[r], x[p]);
        }
    } else {
        constexpr int D = FLIP ? 2 * J / R - 1 : J / R;
        const bool upper = (t & (J / R)) != 0;
        K y[R];
        other(x, y, D, FLIP);
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = (y[r] < x[r]) == !upper ? y[r] : x[r];
    }
}

template <int J, int R, typename K, typename F>
__device__ __forceinline__ void merge_rest(K (&x)[R], int t, F &&other)
{
    if constexpr (J >= 1) {
        merge_stage<J, false>(x, t, other);
        merge_rest<J / 2>(x, t, other);
    }
}

// Sorts N elements, ascending, held as element thread * R + r.
template <int K2, int N, int R, typename K, typename F>
__device__ __forceinline__ void bitonic(K (&x)[R], int t, F &&other)
{
    if constexpr (K2 <= N) {
        merge_stage<K2 / 2, true>(x, t, other);
        merge_rest<K2 / 4>(x, t, other);
        bitonic<K2 * 2, N>(x, t, other);
    }
}

// Sorts the n <= 64 R entries of a block at CSR position s, one wave; writes
// their sorted words and returns the number of distinct columns.
// starts: bit i set where a row starts at entry i.
template <typename K, int R>
__device__ __forceinline__ int sort_small(const int *__restrict__ idx, int s, int n, unsigned cmask, int colA, int lane,
                                          const unsigned long long *starts, unsigned *__restrict__ words, bool &bad,
                                          bool &dups)
{
    K x[R];
    int prev = -1;                         // the column before this step's first
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = r * 64 + lane;
        x[r] = ~(K)0;                      // past every entry
        int c = 0x7fffffff;
        if (i < n) {
            c = idx[s + i];
            bad |= (unsigned)c >= (unsigned)colA;
            x[r] = (K)((unsigned)c & cmask) << kSmallBits | (unsigned)i;
        }
        int before = __shfl_up(c, 1);
        if (lane == 0) before = prev;
        dups |= (__ballot(i < n && c <= before) & ~starts[r]) != 0;
        prev = __builtin_amdgcn_readlane(c, 63);
    }
    bitonic<2, 64 * R>(x, lane, [](const K (&v)[R], K (&y)[R], int d, bool flip) {
#pragma unroll
        for (int r = 0; r < R; ++r) y[r] = __shfl_xor(v[flip ? R - 1 - r : r], d);
    });
    K before = __shfl_up(x[R - 1], 1);
    int distinct = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = lane * R + r;
        const bool head = i < n && (i == 0 || (x[r] >> kSmallBits) != (before >> kSmallBits));
        before = x[r];
        distinct += __popcll(__ballot(head));
        if (i < n) words[s + i] = ((unsigned)x[r] & (kSmall - 1)) | (head ? kHead : 0u);
    }
    return distinct;
}

// One wave per row-block.  K: the type of a sort key, column << kSmallBits |
// position (32 bits for up to 2^22 columns).
template <typename K>
__global__ __launch_bounds__(kThreads) void sort_blocks_kernel(const int *__restrict__ ptr, const int *__restrict__ idx,
                                                               int rows, int nnz, int bm, int bn, int tilem,
                                                               unsigned cmask, int colA, unsigned *__restrict__ words,
                                                               int *__restrict__ nt, Big *__restrict__ medium,
                                                               int medium_cap, Big *__restrict__ huge, int huge_cap,
                                                               int unit_cap, Counters *__restrict__ cnt)
{
    const int b = (int)((blockIdx.x * (long long)kThreads + threadIdx.x) >> 6), lane = threadIdx.x & 63;
    if (b >= tilem) return;
    int s, n;
    block_range(ptr, rows, nnz, bm, tilem, b, s, n);
    s = __builtin_amdgcn_readfirstlane(s);
    n = __builtin_amdgcn_readfirstlane(n);
    bool bad = false, dups = false;
    int d = 0;
    __shared__ unsigned long long starts_all[kThreads / 64][kSmall / 64];
    unsigned long long *starts = starts_all[threadIdx.x >> 6];
    if (n > 0 && n <= kSmall) {
        if (lane < kSmall / 64) starts[lane] = 0ull;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const long long r = (long long)b * bm + lane;
        const int at = lane < bm && r < rows ? ptr[r] - s : -1;
        if (at >= 0 && at < n) atomicOr((unsigned *)starts + (at >> 5), 1u << (at & 31));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (n > kSmall) {
        if (lane == 0) {
            const int ns = (n + kSmall - 1) / kSmall;
            const int u = atomicAdd(&cnt->nunits, ns);
            bad = u < 0 || u > unit_cap - ns;    // only row pointers out of order get there
            if (!bad && n <= kMedium) {
                const int k = n > kMedium / 2 ? 1 : 0, j = atomicAdd(&cnt->nmerge[k], 1);
                bad = j < 0 || j >= medium_cap;
                if (!bad) medium[(size_t)k * medium_cap + j] = Big{b, u, 0};
            } else if (!bad) {
                const unsigned long long at = atomicAdd(&cnt->huge, (1ull << 40) + (unsigned long long)n);
                const long long j = (long long)(at >> 40);
                const long long off = (long long)(at & ((1ull << 40) - 1));
                bad = j >= huge_cap || off + n > nnz;
                if (!bad) huge[j] = Big{b, u, off};
            }
        }
    } else if (n > 512) {
        d = sort_small<K, 16>(idx, s, n, cmask, colA, lane, starts, words, bad, dups);
    } else if (n > 256) {
        d = sort_small<K, 8>(idx, s, n, cmask, colA, lane, starts, words, bad, dups);
    } else if (n > 128) {
        d = sort_small<K, 4>(idx, s, n, cmask, colA, lane, starts, words, bad, dups);
    } else if (n > 64) {
        d = sort_small<K, 2>(idx, s, n, cmask, colA, lane, starts, words, bad, dups);
    } else if (n > 0) {
        d = sort_small<K, 1>(idx, s, n, cmask, colA, lane, starts, words, bad, dups);
    }
    if (lane == 0) nt[b] = (d + bn - 1) / bn;
    if (bad) cnt->bad = 1;
    if (dups) cnt->dups = 1;
}

// Whether entry i > 0 of a block of CSR position s may share its slot with
// an earlier one: its column c does not exceed the one before it, and no row
// starts at it.
__device__ __forceinline__ bool not_ascending(const int *__restrict__ ptr, const int *__restrict__ idx, int rows, int bm,
                                              int b, int s, int i, int c)
{
    if (i == 0 || c > idx[s + i - 1]) return false;
    for (int j = 0; j < bm; ++j) {
        const long long r = (long long)b * bm + j;
        if (r < rows && ptr[r] - s == i) return false;
    }
    return true;
}

// ---- merging the rows of a block ---------------------------------------------
// A block whose rows ascend is its bm rows merged pairwise in log2(bm)
// rounds.  Keys are column << 32 | position, all different.  A thread writes
// kMergePer outputs of a round: a binary search along its diagonal of the
// two runs finds where it starts (merge path), then it takes the smaller
// head.  In LDS, element i lies at i + i / kMergePer, so that the threads'
// consecutive outputs fall in different banks.  RMAT scale 22, 8-row blocks:
// 0.61 ms for the medium blocks (31M entries), 1.25 ms for the huge ones
// (46M); sorting networks of the whole workgroup took 3.0 ms (mostly lane
// exchanges), a radix sort of 12-byte pairs 1.75 ms.
constexpr int kMergePer = 8;
__device__ __forceinline__ int lds_at(int i) { return i + i / kMergePer; }

// How many of the first k outputs come from the first of two runs in LDS
// (la keys from a, lb keys from b).
__device__ __forceinline__ int diagonal(const unsigned long long *lds, int a, int la, int b, int lb, int k)
{
    int lo = max(0, k - lb), hi = min(k, la);
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (lds[lds_at(a + mid)] < lds[lds_at(b + k - 1 - mid)]) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Outputs o .. o + kMergePer - 1 (below n) of merging runs 2gj .. 2gj + g - 1
// with runs 2gj + g .. 2gj + 2g - 1 for every j; run r is off[r] .. off[r + 1].
__device__ __forceinline__ void merge_round(const unsigned long long *lds, const int *off, int bm, int g, int n, int o,
                                            unsigned long long (&y)[kMergePer])
{
    if (o >= n) return;
    int lo = 0, hi = bm / (2 * g) - 1;                 // the last pair that starts at or before o
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (off[2 * g * mid] <= o) lo = mid;
        else hi = mid - 1;
    }
    int j = lo;
    int a = off[2 * g * j], ae = off[2 * g * j + g], b = ae, be = off[2 * g * (j + 1)];
    const int d = diagonal(lds, a, ae - a, b, be - b, o - a);
    b += o - a - d;
    a += d;
    unsigned long long ka = a < ae ? lds[lds_at(a)] : ~0ull, kb = b < be ? lds[lds_at(b)] : ~0ull;
#pragma unroll
    for (int e = 0; e < kMergePer; ++e) {
        if (o + e >= n) break;
        while (a == ae && b == be) {                   // (pairs cover all n positions)
            ++j;
            a = off[2 * g * j];
            b = ae = off[2 * g * j + g];
            be = off[2 * g * (j + 1)];
            ka = a < ae ? lds[lds_at(a)] : ~0ull;
            kb = b < be ? lds[lds_at(b)] : ~0ull;
        }
        if (ka < kb) {
            y[e] = ka;
            ++a;
            ka = a < ae ? lds[lds_at(a)] : ~0ull;
        } else {
            y[e] = kb;
            ++b;
            kb = b < be ? lds[lds_at(b)] : ~0ull;
        }
    }
}

// Workgroups share out the listed blocks, of at most THREADS * kMergePer
// entries.  One whose rows do not ascend goes on the list for
// sort_medium_kernel.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void merge_medium_kernel(const int *__restrict__ ptr, const int *__restrict__ idx,
                                                               int rows, int nnz, int bm, int bn, int tilem,
                                                               unsigned cmask, int colA, unsigned *__restrict__ words,
                                                               int *__restrict__ nt, const Big *__restrict__ list,
                                                               const int *__restrict__ nlist, int cap,
                                                               Big *__restrict__ unsorted, Unit *__restrict__ units,
                                                               Counters *__restrict__ cnt)
{
    constexpr int N = THREADS * kMergePer;
    __shared__ unsigned long long lds[N + N / kMergePer];
    __shared__ int off[65];
    __shared__ int heads[THREADS / 64];
    const int t = threadIdx.x;
    const int nl = min(*nlist, cap);
    bool bad = false;
    for (int l = blockIdx.x; l < nl; l += gridDim.x) {
        const Big m = list[l];
        int s, n;
        block_range(ptr, rows, nnz, bm, tilem, m.b, s, n);
        n = min(n, N);
        if (t <= bm) {
            const long long r = (long long)m.b * bm + t;
            off[t] = t == 0 ? 0 : t == bm || r >= rows ? n : min(max(ptr[r] - s, 0), n);
        }
#pragma unroll
        for (int r = 0; r < kMergePer; ++r) {
            const int i = r * THREADS + t;
            if (i < n) {
                const unsigned c = (unsigned)idx[s + i];
                bad |= c >= (unsigned)colA;
                lds[lds_at(i)] = (unsigned long long)(c & cmask) << 32 | (unsigned)i;
            }
        }
        __syncthreads();
        bool odd = t < bm && off[t + 1] < off[t];
#pragma unroll
        for (int r = 0; r < kMergePer; ++r) {
            const int i = r * THREADS + t;
            if (i > 0 && i < n && (lds[lds_at(i)] >> 32) <= (lds[lds_at(i - 1)] >> 32)) {
                bool start = false;
                for (int k = 1; k < bm; ++k) start |= off[k] == i;
                odd |= !start;
            }
        }
        if (__syncthreads_or(odd)) {
            if (t == 0) {
                cnt->dups = 1;
                unsorted[atomicAdd(&cnt->nsort, 1)] = m;   // each listed block once: within both lists' room
            }
            __syncthreads();
            continue;
        }
        const int o = t * kMergePer;
        unsigned long long y[kMergePer];
        for (int g = 1; g < bm; g *= 2) {
            merge_round(lds, off, bm, g, n, o, y);
            __syncthreads();
#pragma unroll
            for (int e = 0; e < kMergePer; ++e)
                if (o + e < n) lds[lds_at(o + e)] = y[e];
            __syncthreads();
        }
        unsigned before = o > 0 && o < n ? (unsigned)(lds[lds_at(o - 1)] >> 32) : 0u;
        int mine = 0;
#pragma unroll
        for (int e = 0; e < kMergePer; ++e) {
            const bool in = o + e < n;
            const bool head = in && (o + e == 0 || (unsigned)(y[e] >> 32) != before);
            before = (unsigned)(y[e] >> 32);
            mine += __popcll(__ballot(head));
            if (in) words[s + o + e] = (unsigned)y[e] | (head ? kHead : 0u);
        }
        // a wave holds 64 kMergePer sorted entries
        if ((t & 63) == 0) heads[t >> 6] = mine;
        __syncthreads();
        if (t == 0) {
            constexpr int PW = kSmall / (64 * kMergePer);
            int run = 0;
            for (int u = 0; u * kSmall < n; ++u) {
                int k = 0;
                for (int w = 0; w < PW; ++w) k += heads[u * PW + w];
                units[m.unit0 + u] = Unit{m.b, u * kSmall, run, run + k};
                run += k;
            }
            nt[m.b] = (run + bn - 1) / bn;
        }
        __syncthreads();
    }
    if (bad) cnt->bad = 1;
}

// Sorts one block of at most kMediumThreads * R entries by the workgroup,
// whatever the order of its rows' columns.
template <int R>
__device__ __forceinline__ void sort_medium(const int *__restrict__ idx, int s, int n, unsigned cmask, Big m, int bn,
                                            unsigned *__restrict__ words, int *__restrict__ nt,
                                            Unit *__restrict__ units, unsigned long long *lds, int *heads)
{
    typedef unsigned long long K;
    const int t = threadIdx.x;
    K x[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = r * kMediumThreads + t;
        x[r] = ~0ull;
        if (i < n) {
            x[r] = (K)((unsigned)idx[s + i] & cmask) << 32 | (unsigned)i;
        }
    }
    bitonic<2, kMediumThreads * R>(x, t, [&](const K (&v)[R], K (&y)[R], int d, bool flip) {
        if (d < 64) {
#pragma unroll
            for (int r = 0; r < R; ++r) y[r] = __shfl_xor(v[flip ? R - 1 - r : r], d);
        } else {
            __syncthreads();
#pragma unroll
            for (int r = 0; r < R; ++r) lds[r * kMediumThreads + t] = v[r];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < R; ++r) y[r] = lds[(flip ? R - 1 - r : r) * kMediumThreads + (t ^ d)];
        }
    });
    __syncthreads();
    lds[t] = x[R - 1];
    __syncthreads();
    K before = t > 0 ? lds[t - 1] : 0ull;
    int mine = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = t * R + r;
        const bool head = i < n && (i == 0 || (x[r] >> 32) != (before >> 32));
        before = x[r];
        mine += __popcll(__ballot(head));
        if (i < n) words[s + i] = (unsigned)x[r] | (head ? kHead : 0u);
    }
    // a wave holds 64 R sorted entries: kSmall / (64 R) waves a unit
    if ((t & 63) == 0) heads[t >> 6] = mine;
    __syncthreads();
    if (t == 0) {
        constexpr int PW = kSmall / (64 * R);
        int run = 0;
        for (int u = 0; u * kSmall < n; ++u) {
            int k = 0;
            for (int w = 0; w < PW; ++w) k += heads[u * PW + w];
            units[m.unit0 + u] = Unit{m.b, u * kSmall, run, run + k};
            run += k;
        }
        nt[m.b] = (run + bn - 1) / bn;
    }
    __syncthreads();
}

// Workgroups share out the blocks of the list.
__global__ __launch_bounds__(kMediumThreads) void sort_medium_kernel(const int *__restrict__ ptr,
                                                                     const int *__restrict__ idx, int rows, int nnz,
                                                                     int bm, int bn, int tilem, unsigned cmask,
                                                                     unsigned *__restrict__ words,
                                                                     int *__restrict__ nt,
                                                                     const Big *__restrict__ list, int cap,
                                                                     Unit *__restrict__ units,
                                                                     const Counters *__restrict__ cnt)
{
    __shared__ unsigned long long lds[kMedium];
    __shared__ int heads[kMediumThreads / 64];
    const int nl = min(cnt->nsort, cap);
    for (int j = blockIdx.x; j < nl; j += gridDim.x) {
        const Big m = list[j];
        int s, n;
        block_range(ptr, rows, nnz, bm, tilem, m.b, s, n);
        n = min(n, kMedium);
        if (n > 4 * kMediumThreads) sort_medium<8>(idx, s, n, cmask, m, bn, words, nt, units, lds, heads);
        else if (n > 2 * kMediumThreads) sort_medium<4>(idx, s, n, cmask, m, bn, words, nt, units, lds, heads);
        else sort_medium<2>(idx, s, n, cmask, m, bn, words, nt, units, lds, heads);
    }
}

// Huge blocks: grid (blocks, kHugeY) of workgroups.  MERGE: keys column << 32
// | position for the merge rounds, else block << cbits | column with the
// position apart for the radix sort.
constexpr int kHugeY = 64;
template <bool MERGE>
__global__ __launch_bounds__(kThreads) void huge_keys_kernel(const int *__restrict__ ptr, const int *__restrict__ idx,
                                                             int rows, int nnz, int bm, int tilem, int cbits, int colA,
                                                             const Big *__restrict__ huge,
                                                             unsigned long long *__restrict__ key,
                                                             unsigned *__restrict__ pos, Counters *__restrict__ cnt)
{
    const int j = blockIdx.x;
    const Big h = huge[j];
    int s, n;
    block_range(ptr, rows, nnz, bm, tilem, h.b, s, n);
    bool bad = false, odd = false;
    const unsigned long long mask = (1ull << cbits) - 1ull;
    for (long long i = blockIdx.y * kThreads + threadIdx.x; i < n; i += kHugeY * kThreads) {
        const unsigned c = (unsigned)idx[s + i];
        bad |= c >= (unsigned)colA;
        if constexpr (MERGE) {
            odd |= not_ascending(ptr, idx, rows, bm, h.b, s, (int)i, (int)c);
            key[h.off + i] = (c & mask) << 32 | (unsigned)i;
        } else {
            key[h.off + i] = (unsigned long long)j << cbits | (c & mask);
            pos[h.off + i] = (unsigned)i;
        }
    }
    if (MERGE && blockIdx.y == 0 && (int)threadIdx.x < bm) {
        // rows in order, too
        const long long r = (long long)h.b * bm + threadIdx.x;
        if (r > 0 && r < rows) odd |= ptr[r] < ptr[r - 1];
    }
    if (bad) cnt->bad = 1;
    if (odd) cnt->odd = 1;
}

// How many of the first k outputs come from the first of two runs (la keys at
// A, lb at B), by a wave: 64 probes a step.
__device__ __forceinline__ int diagonal_wave(const unsigned long long *__restrict__ A, int la,
                                             const unsigned long long *__restrict__ B, int lb, int k, int lane)
{
    int lo = max(0, k - lb), hi = min(k, la);
    while (lo < hi) {
        const int step = (int)(((long long)hi - lo + 63) / 64);
        const long long mid = lo + (long long)lane * step;
        const bool less = mid < hi && A[mid] < B[k - 1 - mid];
        const int c = __popcll(__ballot(less));            // the first c probes
        if (c == 0) {
            hi = lo;
        } else {
            const int at = lo;
            lo = at + (c - 1) * step + 1;
            hi = (int)min((long long)hi, at + (long long)c * step);
        }
    }
    return lo;
}

// One round of merging the rows of the huge blocks, in to out: a workgroup
// merges kMergeTile outputs of one pair through LDS at a time.
constexpr int kMergeTile = kThreads * kMergePer;
__global__ __launch_bounds__(kThreads) void huge_merge_kernel(const int *__restrict__ ptr, int rows, int nnz, int bm,
                                                              int tilem, int g, const Big *__restrict__ huge,
                                                              const unsigned long long *__restrict__ in,
                                                              unsigned long long *__restrict__ out,
                                                              const Counters *__restrict__ cnt)
{
    __shared__ unsigned long long lds[kMergeTile + kMergeTile / kMergePer];
    __shared__ int off[65];
    __shared__ int split[2];
    if (cnt->odd) return;                                  // the radix sort follows
    const Big h = huge[blockIdx.x];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int s, n;
    block_range(ptr, rows, nnz, bm, tilem, h.b, s, n);
    if (t <= bm) {
        const long long r = (long long)h.b * bm + t;
        off[t] = t == 0 ? 0 : t == bm || r >= rows ? n : min(max(ptr[r] - s, 0), n);
    }
    __syncthreads();
    int j = 0, first = 0;                                  // pair, and its first tile
    for (int tile = blockIdx.y;; tile += kHugeY) {
        int p = 0, m = 0, e = 0;
        for (; j < bm / (2 * g); ++j) {
            p = off[2 * g * j];
            m = off[2 * g * j + g];
            e = off[2 * g * (j + 1)];
            const int tiles = (int)(((long long)e - p + kMergeTile - 1) / kMergeTile);
            if (tile < first + tiles) break;
            first += tiles;
        }
        if (j >= bm / (2 * g)) return;
        const int k0 = (tile - first) * kMergeTile, k1 = (int)min((long long)k0 + kMergeTile, (long long)e - p);
        const unsigned long long *A = in + h.off + p, *B = in + h.off + m;
        if (wave < 2) {
            const int d = diagonal_wave(A, m - p, B, e - m, wave ? k1 : k0, lane);
            if (lane == 0) split[wave] = d;
        }
        __syncthreads();
        const int a0 = split[0], na = split[1] - a0, nb = k1 - k0 - na;
        for (int i = t; i < na; i += kThreads) lds[lds_at(i)] = A[a0 + i];
        for (int i = t; i < nb; i += kThreads) lds[lds_at(na + i)] = B[k0 - a0 + i];
        __syncthreads();
        const int o = t * kMergePer;
        if (o < na + nb) {
            int a = diagonal(lds, 0, na, na, nb, o), b = na + o - a;
            unsigned long long ka = a < na ? lds[lds_at(a)] : ~0ull, kb = b < na + nb ? lds[lds_at(b)] : ~0ull;
            unsigned long long *y = out + h.off + p + k0 + o;
#pragma unroll
            for (int x = 0; x < kMergePer; ++x) {
                if (o + x >= na + nb) break;
                if (ka < kb) {
                    y[x] = ka;
                    ++a;
                    ka = a < na ? lds[lds_at(a)] : ~0ull;
                } else {
                    y[x] = kb;
                    ++b;
                    kb = b < na + nb ? lds[lds_at(b)] : ~0ull;
                }
            }
        }
        __syncthreads();
    }
}

// The sorted words of the huge blocks, and the columns each unit starts
// (rank1; the ranks follow).
template <bool MERGE>
__global__ __launch_bounds__(kThreads) void huge_words_kernel(const int *__restrict__ ptr, int rows, int nnz, int bm,
                                                              int tilem, const Big *__restrict__ huge,
                                                              const unsigned long long *__restrict__ key,
                                                              const unsigned *__restrict__ pos,
                                                              unsigned *__restrict__ words, Unit *__restrict__ units,
                                                              const Counters *__restrict__ cnt)
{
    if (MERGE && cnt->odd) return;
    constexpr int kShift = MERGE ? 32 : 0;
    const Big h = huge[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = blockIdx.y * (kThreads / 64) + (threadIdx.x >> 6);
    int s, n;
    block_range(ptr, rows, nnz, bm, tilem, h.b, s, n);
    for (long long u = wave; u * kSmall < n; u += kHugeY * (kThreads / 64)) {
        int k = 0;
        for (int i = 0; i < kSmall; i += 64) {
            const long long p = u * kSmall + i + lane;
            const bool in = p < n;
            const unsigned long long x = in ? key[h.off + p] : 0ull;
            const bool head = in && (p == 0 || x >> kShift != key[h.off + p - 1] >> kShift);
            if (in) words[s + p] = (MERGE ? (unsigned)x : pos[h.off + p]) | (head ? kHead : 0u);
            k += __popcll(__ballot(head));
        }
        if (lane == 0) units[h.unit0 + u] = Unit{h.b, (int)(u * kSmall), 0, k};
    }
}

// One workgroup per huge block: ranks of its units, its tiles.
__global__ __launch_bounds__(kThreads) void huge_ranks_kernel(const int *__restrict__ ptr, int rows, int nnz, int bm,
                                                              int bn, int tilem, const Big *__restrict__ huge,
                                                              Unit *__restrict__ units, int *__restrict__ nt,
                                                              const Counters *__restrict__ cnt, bool merged)
{
    if (merged && cnt->odd) return;
    using BS = rocprim::block_scan<int, kThreads>;
    __shared__ typename BS::storage_type st;
    const Big h = huge[blockIdx.x];
    int s, n;
    block_range(ptr, rows, nnz, bm, tilem, h.b, s, n);
    const int nu = (int)(((long long)n + kSmall - 1) / kSmall);
    int carry = 0;
    for (int base = 0; base < nu; base += kThreads) {
        const int u = base + (int)threadIdx.x;
        const int v = u < nu ? units[h.unit0 + u].rank1 : 0;
        int ex = 0, agg = 0;
        BS().exclusive_scan(v, ex, 0, agg, st, rocprim::plus<int>());
        if (u < nu) {
            units[h.unit0 + u].rank0 = carry + ex;
            units[h.unit0 + u].rank1 = carry + ex + v;
        }
        carry += agg;
        __syncthreads();
    }
    if (threadIdx.x == 0) nt[h.b] = (carry + bn - 1) / bn;
}

// ---- 2. chained scan --------------------------------------------------------
// out[i] = in(0) + .. + in(i - 1) for i = 0 .. n, and the 64-bit total, in
// one launch: workgroups take tickets in order, publish the sum of their
// kScanBlock inputs and add up the sums published before theirs (Merrill and
// Garland's decoupled look-back).  A workgroup only waits for lower tickets,
// which run already and publish before they wait.  state: 0 = nothing yet,
// else value << 2 | 1 (the workgroup's own sum) or | 2 (the sum so far);
// state and ticket are zero at the start.
constexpr int kScanPer = 8;
constexpr int kScanBlock = kThreads * kScanPer;

template <typename F>
__global__ __launch_bounds__(kThreads) void scan_kernel(F in, int n, int *__restrict__ out,
                                                        unsigned long long *__restrict__ state,
                                                        int *__restrict__ ticket, long long *__restrict__ total)
{
    using BS = rocprim::block_scan<long long, kThreads>;
    __shared__ typename BS::storage_type st;
    __shared__ int items[kScanBlock];
    __shared__ long long before;
    __shared__ int mine;
    const int t = threadIdx.x, lane = t & 63;
    if (t == 0) mine = atomicAdd(ticket, 1);
    __syncthreads();
    const int vb = mine;
    const long long base = (long long)vb * kScanBlock;
    // read side by side, summed kScanPer in a row
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) {
        const long long i = base + j * kThreads + t;
        items[j * kThreads + t] = i < n ? in((int)i) : 0;
    }
    __syncthreads();
    int v[kScanPer];
    long long sum = 0;
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) {
        v[j] = items[t * kScanPer + j];
        sum += v[j];
    }
    long long ex = 0, agg = 0;
    BS().exclusive_scan(sum, ex, 0ll, agg, st, rocprim::plus<long long>());
    if (t < 64) {
        const auto put = [&](long long x, unsigned long long kind) {
            if (lane == 0)
                __hip_atomic_store(&state[vb], (unsigned long long)x << 2 | kind, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        };
        long long sofar = 0;
        if (vb > 0) put(agg, 1);
        // 64 workgroups at a time, the nearest in lane 0; the one before the
        // first counts as a sum so far of 0
        for (int j = vb - 1;;) {
            const unsigned long long w = j - lane < 0 ? 2ull
                                                      : __hip_atomic_load(&state[j - lane], __ATOMIC_RELAXED,
                                                                          __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long done = __ballot((w & 2) != 0);
            const int last = done ? __ffsll((long long)done) - 1 : 63;
            if (__ballot(w == 0 && lane <= last)) {
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            long long x = lane <= last ? (long long)(w >> 2) : 0;
#pragma unroll
            for (int d = 32; d >= 1; d /= 2) x += __shfl_xor(x, d);
            sofar += x;
            if (done) break;
            j -= 64;
        }
        put(sofar + agg, 2);
        if (lane == 0) {
            before = sofar;
            if (base + kScanBlock >= n) {                // the last workgroup
                *total = sofar + agg;
                out[n] = (int)min(sofar + agg, (long long)INT_MAX);
            }
        }
    }
    __syncthreads();
    long long o = before + ex;
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) {
        const long long i = base + t * kScanPer + j;
        if (i < n) out[i] = (int)min(o, (long long)INT_MAX);
        o += v[j];
    }
}
inline size_t scan_state_bytes(long long n) { return sizeof(unsigned long long) * (size_t)((n + kScanBlock - 1) / kScanBlock); }

struct IntAt {
    const int *p;
    __device__ int operator()(int i) const { return p[i]; }
};

// ---- 3. the tiles -------------------------------------------------------------
template <typename V>
__device__ __forceinline__ V add_round(V a, V b)
{
    if constexpr (sizeof(V) == 2) return (V)((float)a + (float)b);
    else return a + b;
}

typedef uint32_t tu4 __attribute__((ext_vector_type(4), may_alias));

// Wave u < tilem: the tiles of row-block u if it has at most kSmall entries;
// wave tilem + k: the tiles that start in unit k.  BM, BN: the class's tile
// shape, or 0 with any shape in bm_, bn_.  DUP: a slot may have several
// entries (some row's columns do not ascend).
// Bound by its stores when it keeps enough loads in flight: a wave reads the
// words, then the values and columns, of kBatch x 64 entries at a time (two
// round trips to memory per 256 entries), and stages a window of tiles in 4
// KB of LDS (one tile at least: 8 KB for the widest generic shape), so that
// eight workgroups of four waves fit on a CU.  RMAT scale 22, tf32 8-row
// tiles (4.6 GB written): 2.05 ms; 3.48 ms with 64 entries a time, each
// looking at its neighbours for duplicates.  16-row tiles of a power-law
// matrix (1.1 GB): 0.345 ms, before 0.530.
constexpr int kBatch = 4;
template <typename V, int BM, int BN, bool DUP>
__global__ __launch_bounds__(kThreads) void fill_kernel(const int *__restrict__ ptr, const int *__restrict__ idx,
                                                        const V *__restrict__ val, int rows, int nnz, int bm_, int bn_,
                                                        int tilem, const unsigned *__restrict__ words,
                                                        const int *__restrict__ tile_ptr,
                                                        const Unit *__restrict__ units, int nunits, int tilenum,
                                                        int *__restrict__ colidx, int *__restrict__ tile_nnz,
                                                        V *__restrict__ dense, unsigned long long *__restrict__ bitmap)
{
    const int bm = BM ? BM : bm_, bn = BN ? BN : bn_;
    constexpr int kStage = BM ? 4096 : 8192;
    constexpr int kTiles = 16;
    constexpr int kMapWords = BM && BN ? (BM * BN + 63) / 64 * (BM * BN * (int)sizeof(V) >= kStage ? 1 : kTiles) : 64;
    __shared__ __attribute__((aligned(16))) char stage_all[kThreads / 64][kStage];
    __shared__ unsigned long long map_all[kThreads / 64][kMapWords];
    __shared__ int row_all[kThreads / 64][64];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long u = (long long)blockIdx.x * (kThreads / 64) + wid;
    if (u >= (long long)tilem + nunits) return;
    if (u == 0 && lane == 0) tile_nnz[tilenum] = nnz;
    Unit un{(int)u, 0, 0, 0};
    if (u >= tilem) un = units[u - tilem];
    const int b = __builtin_amdgcn_readfirstlane(un.b);
    int s, n;
    block_range(ptr, rows, nnz, bm, tilem, b, s, n);
    s = __builtin_amdgcn_readfirstlane(s);
    n = __builtin_amdgcn_readfirstlane(n);
    if (n == 0 || (u < tilem && n > kSmall)) return;
    const int t0 = tile_ptr[b], nt = tile_ptr[b + 1] - t0;
    int q0 = __builtin_amdgcn_readfirstlane(un.p0), rk = __builtin_amdgcn_readfirstlane(un.rank0);
    // the tiles whose first column starts here
    const int tb = (rk + bn - 1) / bn;
    const int te = __builtin_amdgcn_readfirstlane((long long)q0 + kSmall >= n ? nt : min(nt, (un.rank1 + bn - 1) / bn));
    if (tb >= te) return;
    const int slots = bm * bn, mw = (slots + 63) / 64;
    const int tile_bytes = slots * (int)sizeof(V);       // a multiple of 16: bm is a multiple of 8
    const int wt = max(1, min(min(kTiles, kStage / tile_bytes), kMapWords / mw));
    char *stage = stage_all[wid];
    unsigned long long *map = map_all[wid];
    int *rowoff = row_all[wid];
    // first entry of each row; rows past the end never match
    int mine = 0x7fffffff;
    if (lane < bm) {
        const long long r = (long long)b * bm + lane;
        if (r < rows) mine = ptr[r] - s;
        rowoff[lane] = mine;
    }
    constexpr bool kScalarRows = BM == 8 || BM == 16;    // their offsets fit the scalar registers
    int off[kScalarRows ? BM : 1];
    if constexpr (kScalarRows) {
#pragma unroll
        for (int j = 0; j < BM; ++j) off[j] = __builtin_amdgcn_readlane(mine, j);
    }
    auto row_of = [&](int i) {             // the last row that starts at or before entry i
        int lo = 0;
        if constexpr (kScalarRows) {
#pragma unroll
            for (int j = 1; j < BM; ++j) lo += i >= off[j] ? 1 : 0;
        } else {
            for (int d = bm / 2; d >= 1; d /= 2)
                if (rowoff[lo + d] <= i) lo += d;
        }
        return lo;
    };
    int w0 = tb, w1 = min(tb + wt, te);    // the window
    auto clear = [&]() {
        for (int k = lane; k < (w1 - w0) * tile_bytes / 16; k += 64) ((tu4 *)stage)[k] = tu4{0u, 0u, 0u, 0u};
        for (int k = lane; k < (w1 - w0) * mw; k += 64) map[k] = 0ull;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    auto flush = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        tu4 *out = (tu4 *)((char *)dense + (size_t)(t0 + w0) * tile_bytes);
        for (int k = lane; k < (w1 - w0) * tile_bytes / 16; k += 64)
            __builtin_nontemporal_store(((const tu4 *)stage)[k], out + k);
        for (int k = lane; k < (w1 - w0) * mw; k += 64) bitmap[(size_t)(t0 + w0) * mw + k] = map[k];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    clear();
    int prow = -1;                         // row of the entry before this batch
    if (DUP && q0 > 0) prow = row_of((int)(words[s + q0 - 1] & ~kHead));
    for (; q0 < n && w0 < te; q0 += 64 * kBatch) {
        unsigned w[kBatch];
        int rank[kBatch], c[kBatch];
        V v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int q = q0 + 64 * k + lane;
            w[k] = q < n ? words[s + q] : 0u;
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int q = q0 + 64 * k + lane, i = (int)(w[k] & ~kHead);
            v[k] = q < n ? val[s + i] : (V)0;
            c[k] = (w[k] & kHead) ? idx[s + i] : 0;
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const unsigned long long hm = __ballot((w[k] & kHead) != 0);
            rank[k] = rk + __popcll(hm & ((2ull << lane) - 1ull)) - 1;
            rk += __popcll(hm);
        }
        bool skip[kBatch];                 // not the first entry of its slot
        if constexpr (DUP) {
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const int q = q0 + 64 * k + lane, row = row_of((int)(w[k] & ~kHead));
                int before = __shfl_up(row, 1);
                if (lane == 0) before = prow;
                skip[k] = !(w[k] & kHead) && before == row;
                prow = __builtin_amdgcn_readlane(row, 63);
                // the first entry of a slot adds up the ones that follow
                if (q < n && !skip[k]) {
                    v[k] = add_round((V)0, v[k]);
                    for (int j = q + 1; j < n; ++j) {
                        const unsigned wa = words[s + j];
                        if ((wa & kHead) || row_of((int)wa) != row) break;
                        v[k] = add_round(v[k], val[s + (int)wa]);
                    }
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                skip[k] = false;
                v[k] = add_round((V)0, v[k]);
            }
        }
        const int last = (rk - 1) / bn;    // the last tile reached
        for (;;) {
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const int q = q0 + 64 * k + lane, i = (int)(w[k] & ~kHead);
                const int tile = (int)((unsigned)max(rank[k], 0) / (unsigned)bn);
                if (q < n && tile >= w0 && tile < w1) {
                    const int col = rank[k] - tile * bn, tl = tile - w0;
                    if (w[k] & kHead) {
                        colidx[(size_t)t0 * bn + rank[k]] = c[k];
                        if (col == 0) tile_nnz[t0 + tile] = s + q;
                    }
                    if (!skip[k]) {
                        const int slot = row_of(i) * bn + col;
                        ((V *)stage)[tl * slots + slot] = v[k];
                        atomicOr((unsigned *)map + 2 * (tl * mw) + ((unsigned)slot >> 5), 1u << (slot & 31));
                    }
                }
            }
            if (last < w1) break;
            flush();
            w0 = w1;
            if (w0 >= te) break;
            w1 = min(w0 + wt, te);
            clear();
        }
    }
    if (w0 < te) flush();
    if (te == nt) {
        // the block's last tile repeats its last column
        const int last = idx[s + (int)(words[s + n - 1] & ~kHead)];
        for (long long k = rk + lane; k < (long long)nt * bn; k += 64) colidx[(size_t)t0 * bn + k] = last;
    }
}

// ---- bitmap-packed A -------------------------------------------------------
struct BitsAt {                            // occupied slots of a tile
    const unsigned long long *bmp;
    int words;
    __device__ int operator()(int t) const
    {
        int k = 0;
        for (int w = 0; w < words; ++w) k += __popcll(bmp[(size_t)t * words + w]);
        return k;
    }
};

// Occupied slots over all n bitmap words.
__global__ __launch_bounds__(kThreads) void count_bits_kernel(const unsigned long long *__restrict__ bmp, long long n,
                                                              unsigned long long *__restrict__ total)
{
    using BR = rocprim::block_reduce<long long, kThreads>;
    __shared__ typename BR::storage_type st;
    long long s = 0;
    for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kThreads)
        s += __popcll(bmp[i]);
    long long b = 0;
    BR().reduce(s, b, st, rocprim::plus<long long>());
    if (threadIdx.x == 0) atomicAdd(total, (unsigned long long)b);
}

// The values at the set bits of every tile, in bit (row-major) order; writes
// at or past `cap` elements are dropped.  A lane takes 16 bytes of the dense
// tiles (4 or 8 slots) in each of kPackGroups steps, all loaded at once,
// places its set values by prefix counts of the bitmap words, and the wave's
// values, which are consecutive in the packed order, go out through LDS with
// whole lines.  Bound by the reads of the dense tiles: power law 2^20 tf32
// 16-row tiles (1.1 GB) 0.276 ms; one step a wave 0.372 ms (four round trips to
// memory for 1 KB), one thread per tile, walking its bits, 0.313 ms.  gpt:
// lane groups per tile, gshift its log2 or -1.  The first wave also zeroes
// the nz padding elements after the last value.
constexpr int kPackGroups = 4;
template <typename V>
__global__ __launch_bounds__(kThreads) void pack_kernel(const V *__restrict__ dense,
                                                        const unsigned long long *__restrict__ bmp,
                                                        const int *__restrict__ vptr, int tilenum, int words, int gpt,
                                                        int gshift, V *__restrict__ pval, long long cap, int nz)
{
    constexpr int VEC = 16 / (int)sizeof(V);
    __shared__ V out_all[kThreads / 64][64 * VEC * kPackGroups];
    const int lane = threadIdx.x & 63;
    V *out = out_all[threadIdx.x >> 6];
    const long long g0 = ((long long)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6)) * (64 * kPackGroups) + lane;
    long long pos[kPackGroups];
    unsigned occ[kPackGroups];
    tu4 raw[kPackGroups];
#pragma unroll
    for (int k = 0; k < kPackGroups; ++k) {
        const long long g = g0 + 64 * k, t = gshift >= 0 ? g >> gshift : g / gpt;
        pos[k] = 0;
        occ[k] = 0;
        raw[k] = tu4{0u, 0u, 0u, 0u};
        if (t < tilenum) {
            raw[k] = *(const tu4 *)(dense + (size_t)g * VEC);
            const int bit = (int)(g - t * gpt) * VEC;
            const unsigned long long *bw = bmp + (size_t)t * words;
            const unsigned long long w = bw[bit >> 6];
            int pre = __popcll(w & ((1ull << (bit & 63)) - 1ull));
            for (int i = 0; i < bit >> 6; ++i) pre += __popcll(bw[i]);
            pos[k] = (long long)vptr[t] + pre;
            occ[k] = (unsigned)(w >> (bit & 63)) & ((1u << VEC) - 1u);
        }
    }
    const long long base = __shfl(pos[0], 0);      // lane 0 has a tile unless no lane does
    int n = 0;
#pragma unroll
    for (int k = 0; k < kPackGroups; ++k) {
        if (!occ[k]) continue;
        int o = (int)(pos[k] - base);
        V v[VEC];
        __builtin_memcpy(v, &raw[k], 16);
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            if (occ[k] >> j & 1u) out[o++] = v[j];
        n = o;                                     // (positions ascend)
    }
#pragma unroll
    for (int d = 32; d >= 1; d /= 2) n = max(n, __shfl_xor(n, d));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int k = lane; k < n; k += 64)
        if (base + k < cap) pval[base + k] = out[k];
    if (g0 < nz) {
        const long long at = (long long)vptr[tilenum] + g0;
        if (at < cap) pval[at] = V(0);
    }
}

template <typename V>
int launch_pack(const void *dense, const unsigned long long *bmp, const int *vptr, int tilenum, int words, int slots,
                void *pval, long long cap, int nz, hipStream_t s)
{
    const int gpt = slots * (int)sizeof(V) / 16;   // slots are a multiple of 8
    const int gshift = (gpt & (gpt - 1)) == 0 ? __builtin_ctz((unsigned)gpt) : -1;
    pack_kernel<V><<<nblocks(((long long)tilenum * gpt + kPackGroups - 1) / kPackGroups), kThreads, 0, s>>>((const V *)dense, bmp, vptr, tilenum, words, gpt,
                                                                         gshift, (V *)pval, cap, nz);
    return (int)hipGetLastError();
}

// ---- allocation-free packing: a three-pass scan through `scratch` -----------
// Tiles are taken in blocks of kPackBlockTiles (kPackPer consecutive tiles per
// thread).  Pass 1 stores each tile's value count in vptr[t] and each block's
// sum in sums[b]; pass 2 (one workgroup) turns sums[0..nb) into exclusive
// block offsets and stores the total in sums[nb]; pass 3 turns the counts of
// each block into exclusive offsets.  The output array vptr doubles as the
// count buffer, so the only scratch is nb + 1 ints.
constexpr int kPackPer = 8;
constexpr int kPackBlockTiles = kThreads * kPackPer;

__global__ __launch_bounds__(kThreads) void pack_count_kernel(const unsigned long long *__restrict__ bmp, int tilenum,
                                                              int words, int *__restrict__ vptr,
                                                              int *__restrict__ sums)
{
    using BR = rocprim::block_reduce<int, kThreads>;
    __shared__ typename BR::storage_type st;
    const long long base = (long long)blockIdx.x * kPackBlockTiles + (long long)threadIdx.x * kPackPer;
    int s = 0;
    for (int j = 0; j < kPackPer; ++j) {
        const long long t = base + j;
        if (t >= tilenum) break;
        int k = 0;
        for (int w = 0; w < words; ++w) k += __popcll(bmp[(size_t)t * words + w]);
        vptr[t] = k;
        s += k;
    }
    int total = 0;
    BR().reduce(s, total, st, rocprim::plus<int>());
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// The block offsets are scanned in 64 bits; the int copies in sums[] are
// only used (pass 3) when the 64-bit total stored in *total64 leaves room
// for the padding within INT_MAX, which the host checks first.
__global__ __launch_bounds__(kThreads) void pack_block_scan_kernel(int *__restrict__ sums, int nb,
                                                                   long long *__restrict__ total64)
{
    using BS = rocprim::block_scan<long long, kThreads>;
    __shared__ typename BS::storage_type st;
    long long carry = 0;
    for (int base = 0; base < nb; base += kThreads) {
        const int i = base + (int)threadIdx.x;
        const long long v = i < nb ? sums[i] : 0;
        long long ex = 0, agg = 0;
        BS().exclusive_scan(v, ex, 0ll, agg, st, rocprim::plus<long long>());
        if (i < nb) sums[i] = (int)min(carry + ex, (long long)INT_MAX);
        carry += agg;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        sums[nb] = (int)min(carry, (long long)INT_MAX);
        *total64 = carry;
    }
}

__global__ __launch_bounds__(kThreads) void pack_offsets_kernel(int *__restrict__ vptr, int tilenum,
                                                                const int *__restrict__ sums)
{
    using BS = rocprim::block_scan<int, kThreads>;
    __shared__ typename BS::storage_type st;
    const long long base = (long long)blockIdx.x * kPackBlockTiles + (long long)threadIdx.x * kPackPer;
    int c[kPackPer];
    int s = 0;
    for (int j = 0; j < kPackPer; ++j) {
        const long long t = base + j;
        c[j] = t < tilenum ? vptr[t] : 0;
        s += c[j];
    }
    int ex = 0;
    BS().exclusive_scan(s, ex, 0, st, rocprim::plus<int>());
    int o = sums[blockIdx.x] + ex;
    for (int j = 0; j < kPackPer; ++j) {
        const long long t = base + j;
        if (t < tilenum) vptr[t] = o;
        o += c[j];
    }
}

// vptr[tilenum] = total; zero the nz padding elements after the last value
template <typename V>
__global__ void pack_tail_kernel(int *__restrict__ vptr, int tilenum, const int *__restrict__ sums, int nb,
                                 V *__restrict__ pval, long long cap, int nz)
{
    const int total = sums[nb];
    if (threadIdx.x == 0) vptr[tilenum] = total;
    if ((int)threadIdx.x < nz && (long long)total + threadIdx.x < cap) pval[(long long)total + threadIdx.x] = V(0);
}

// Device buffers of one call, all used on `stream` only: given back at scope
// exit, once the stream has drained.
struct DevBufs {
    hipStream_t stream;
    void *p[4] = {};
    int n = 0;
    explicit DevBufs(hipStream_t s) : stream(s) {}
    template <typename T>
    int get(T **out, size_t bytes)
    {
        void *q = nullptr;
        const int st = tsp::dev_alloc(&q, bytes);
        if (st == 0) p[n++] = q;
        *out = (T *)q;
        return st;
    }
    ~DevBufs()
    {
        const bool waited = n > 0 && hipStreamSynchronize(stream) == hipSuccess;
        for (int i = 0; i < n; ++i) (void)tsp::dev_free(p[i], waited);
    }
};

#define TCHK(x)                                     \
    do {                                            \
        const int e_ = (int)(x);                    \
        if (e_ != 0) return e_;                     \
    } while (0)

// One allocation cut into 256-byte aligned pieces.
struct Carve {
    size_t bytes = 0;
    size_t add(size_t n)
    {
        const size_t at = bytes;
        bytes += (n + 255) / 256 * 256;
        return at;
    }
};

template <typename F>
int launch_scan(F in, int n, int *out, unsigned long long *state, int *ticket, long long *total, hipStream_t s)
{
    scan_kernel<<<(unsigned)(((long long)n + kScanBlock - 1) / kScanBlock), kThreads, 0, s>>>(in, n, out, state, ticket,
                                                                                              total);
    return (int)hipGetLastError();
}

// Merges the rows of the `nh` huge blocks (`entries` in all) and completes
// their words, units and tile counts -- unless some row's columns do not
// ascend (cnt->odd), when nothing is completed.
int merge_huge(const int *d_ptr, const int *d_idx, int rows, int nnz, int bm, int bn, int tilem, int cbits, int colA,
               const Big *huge, unsigned nh, size_t entries, unsigned *words, Unit *units, int *nt, Counters *cnt,
               hipStream_t s)
{
    Carve c;
    const size_t k0 = c.add(8 * entries), k1 = c.add(8 * entries);
    DevBufs db(s);
    char *w = nullptr;
    TCHK(db.get(&w, c.bytes));
    unsigned long long *in = (unsigned long long *)(w + k0), *out = (unsigned long long *)(w + k1);
    const dim3 grid(nh, kHugeY);
    huge_keys_kernel<true><<<grid, kThreads, 0, s>>>(d_ptr, d_idx, rows, nnz, bm, tilem, cbits, colA, huge, in, nullptr,
                                                     cnt);
    for (int g = 1; g < bm; g *= 2) {
        huge_merge_kernel<<<grid, kThreads, 0, s>>>(d_ptr, rows, nnz, bm, tilem, g, huge, in, out, cnt);
        std::swap(in, out);
    }
    huge_words_kernel<true><<<grid, kThreads, 0, s>>>(d_ptr, rows, nnz, bm, tilem, huge, in, nullptr, words, units, cnt);
    huge_ranks_kernel<<<nh, kThreads, 0, s>>>(d_ptr, rows, nnz, bm, bn, tilem, huge, units, nt, cnt, true);
    return (int)hipGetLastError();
}

// The same by a radix sort, whatever the order of the rows' columns.
int sort_huge(const int *d_ptr, const int *d_idx, int rows, int nnz, int bm, int bn, int tilem, int cbits, int colA,
              const Big *huge, unsigned nh, size_t entries, unsigned *words, Unit *units, int *nt, Counters *cnt,
              hipStream_t s)
{
    const int bits = cbits + bits_for(nh);
    unsigned long long *key = nullptr;
    unsigned *pos = nullptr;
    size_t need = 0;
    TCHK(rocprim::radix_sort_pairs(nullptr, need, key, key, pos, pos, entries, 0, bits, s));
    Carve c;
    const size_t k0 = c.add(8 * entries), k1 = c.add(8 * entries), p0 = c.add(4 * entries), p1 = c.add(4 * entries);
    const size_t t0 = c.add(need);
    DevBufs db(s);
    char *w = nullptr;
    TCHK(db.get(&w, c.bytes));
    const dim3 grid(nh, kHugeY);
    huge_keys_kernel<false><<<grid, kThreads, 0, s>>>(d_ptr, d_idx, rows, nnz, bm, tilem, cbits, colA, huge,
                                                      (unsigned long long *)(w + k0), (unsigned *)(w + p0), cnt);
    TCHK(rocprim::radix_sort_pairs(w + t0, need, (unsigned long long *)(w + k0), (unsigned long long *)(w + k1),
                                   (unsigned *)(w + p0), (unsigned *)(w + p1), entries, 0, bits, s));
    huge_words_kernel<false><<<grid, kThreads, 0, s>>>(d_ptr, rows, nnz, bm, tilem, huge, (unsigned long long *)(w + k1),
                                                       (unsigned *)(w + p1), words, units, cnt);
    huge_ranks_kernel<<<nh, kThreads, 0, s>>>(d_ptr, rows, nnz, bm, bn, tilem, huge, units, nt, cnt, false);
    return (int)hipGetLastError();
}

int tile_create_device(tsp_dev_tiles *out, int rows, int colA, long long nnz, const int *d_ptr, const int *d_idx,
                       const void *d_val, int BM, int BN, int prec, void *stream)
{
    if (!out || rows < 0 || colA <= 0 || nnz < 0 || nnz > 0x7ffffff0LL) return TSP_EINVAL;
    if ((BM != 64 && BM != 16 && BM != 8) || BN <= 0 || BN > 32) return TSP_EINVAL;
    if (prec != TSP_PREC_FP16 && prec != TSP_PREC_TF32) return TSP_EINVAL;
    if (rows > 0 && (!d_ptr || (nnz > 0 && (!d_idx || !d_val)))) return TSP_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    out->bm = BM;
    out->bn = BN;
    out->prec = prec;
    out->bitmap_words = (BM * BN + 63) / 64;
    const int tilem = (rows + BM - 1) / BM;
    out->tilem = tilem;
    const size_t vs = prec == TSP_PREC_FP16 ? 2 : 4;
    TCHK(tsp::dev_alloc((void **)&out->d_tile_ptr, sizeof(int) * ((size_t)tilem + 1)));
    if (tilem == 0 || nnz == 0) {
        // no entries: every row-block has zero tiles
        TCHK(hipMemsetAsync(out->d_tile_ptr, 0, sizeof(int) * ((size_t)tilem + 1), s));
        TCHK(tsp::dev_alloc((void **)&out->d_tile_colidx, 16));
        TCHK(tsp::dev_alloc((void **)&out->d_val, 16));
        TCHK(tsp::dev_alloc((void **)&out->d_bitmap, 16));
        TCHK(tsp::dev_alloc((void **)&out->d_tile_nnz, sizeof(int)));
        TCHK(hipMemsetAsync(out->d_tile_nnz, 0, sizeof(int), s));
        return (int)hipStreamSynchronize(s);
    }
    const int cbits = bits_for(colA);
    const unsigned cmask = (unsigned)((1ull << cbits) - 1ull);
    const int n = (int)nnz;
    // every medium block holds more than kSmall entries, every huge one more
    // than kMedium, and a block of n of them has at most 2 n / kSmall units
    const int medium_cap = n / kSmall + 1, huge_cap = n / kMedium + 1, unit_cap = 2 * (n / kSmall) + 2;
    const size_t state_bytes = scan_state_bytes(tilem);
    Carve cv;
    const size_t o_cnt = cv.add(sizeof(Counters)), o_state = cv.add(state_bytes);
    const size_t zeroed = cv.bytes;
    const size_t o_nt = cv.add(4 * (size_t)tilem), o_medium = cv.add(sizeof(Big) * 4 * (size_t)medium_cap);
    const size_t o_huge = cv.add(sizeof(Big) * (size_t)huge_cap), o_units = cv.add(sizeof(Unit) * (size_t)unit_cap);
    const size_t o_words = cv.add(4 * (size_t)n);
    DevBufs db(s);
    char *w = nullptr;
    TCHK(db.get(&w, cv.bytes));
    Counters *cnt = (Counters *)(w + o_cnt);
    unsigned long long *state = (unsigned long long *)(w + o_state);
    int *nt = (int *)(w + o_nt);
    Big *medium = (Big *)(w + o_medium), *huge = (Big *)(w + o_huge);
    Unit *units = (Unit *)(w + o_units);
    unsigned *words = (unsigned *)(w + o_words);
    TCHK(hipMemsetAsync(w, 0, zeroed, s));
    // 1. sorted entries, tiles per block
    const unsigned wave_blocks = nblocks((long long)tilem * 64);
    if (cbits + kSmallBits <= 32)
        sort_blocks_kernel<unsigned><<<wave_blocks, kThreads, 0, s>>>(d_ptr, d_idx, rows, n, BM, BN, tilem, cmask, colA,
                                                                      words, nt, medium, medium_cap, huge, huge_cap,
                                                                      unit_cap, cnt);
    else
        sort_blocks_kernel<unsigned long long><<<wave_blocks, kThreads, 0, s>>>(
            d_ptr, d_idx, rows, n, BM, BN, tilem, cmask, colA, words, nt, medium, medium_cap, huge, huge_cap, unit_cap,
            cnt);
    if (n > kSmall) {
        // medium: two lists of blocks to merge, then room for both as blocks to sort
        Big *unsorted = medium + 2 * (size_t)medium_cap;
        const unsigned groups = (unsigned)(medium_cap < 2048 ? medium_cap : 2048);
        merge_medium_kernel<kMedium / 2 / kMergePer><<<groups, kMedium / 2 / kMergePer, 0, s>>>(
            d_ptr, d_idx, rows, n, BM, BN, tilem, cmask, colA, words, nt, medium, &cnt->nmerge[0], medium_cap, unsorted,
            units, cnt);
        if (n > kMedium / 2)
            merge_medium_kernel<kMedium / kMergePer><<<groups, kMedium / kMergePer, 0, s>>>(
                d_ptr, d_idx, rows, n, BM, BN, tilem, cmask, colA, words, nt, medium + medium_cap, &cnt->nmerge[1],
                medium_cap, unsorted, units, cnt);
        sort_medium_kernel<<<groups < 512 ? groups : 512, kMediumThreads, 0, s>>>(
            d_ptr, d_idx, rows, n, BM, BN, tilem, cmask, words, nt, unsorted, 2 * medium_cap, units, cnt);
    }
    TCHK(hipGetLastError());
    // 2. tile_ptr
    Counters h;
    for (int pass = 0;; ++pass) {
        if (int st = launch_scan(IntAt{nt}, tilem, out->d_tile_ptr, state, &cnt->ticket, &cnt->total, s)) return st;
        TCHK(hipMemcpyAsync(&h, cnt, sizeof h, hipMemcpyDeviceToHost, s));
        TCHK(hipStreamSynchronize(s));
        if (h.bad) return TSP_EINVAL;       // a column outside [0, colA)
        const size_t entries = (size_t)(h.huge & ((1ull << 40) - 1ull));
        if (entries == 0 || pass == 2 || (pass == 1 && !h.odd)) break;
        const auto complete = pass ? sort_huge : merge_huge;
        if (int st = complete(d_ptr, d_idx, rows, n, BM, BN, tilem, cbits, colA, huge, (unsigned)(h.huge >> 40), entries,
                              words, units, nt, cnt, s))
            return st;
        TCHK(hipMemsetAsync(state, 0, state_bytes, s));
        TCHK(hipMemsetAsync(&cnt->ticket, 0, sizeof(int), s));
    }
    // every tile holds at least one entry
    if (h.total > nnz) return TSP_EINVAL;
    const int tilenum = (int)h.total;
    out->tilenum = tilenum;
    const size_t tn = (size_t)tilenum;
    TCHK(tsp::dev_alloc((void **)&out->d_tile_colidx, 4 * tn * BN));
    TCHK(tsp::dev_alloc((void **)&out->d_tile_nnz, 4 * (tn + 1)));
    TCHK(tsp::dev_alloc((void **)&out->d_val, vs * tn * BM * BN));
    TCHK(tsp::dev_alloc((void **)&out->d_bitmap, 8 * tn * out->bitmap_words));
    // 3. the tiles
    const unsigned fill_blocks = nblocks(((long long)tilem + h.nunits) * 64);
    const auto fill = [&](auto kernel, auto *v) {
        kernel<<<fill_blocks, kThreads, 0, s>>>(d_ptr, d_idx, v, rows, n, BM, BN, tilem, words, out->d_tile_ptr, units,
                                                h.nunits, tilenum, out->d_tile_colidx, out->d_tile_nnz,
                                                (std::remove_const_t<std::remove_pointer_t<decltype(v)>> *)out->d_val,
                                                (unsigned long long *)out->d_bitmap);
    };
    const auto shape = [&](auto dup) {
        constexpr bool DUP = decltype(dup)::value;
        if (prec == TSP_PREC_FP16) {
            const _Float16 *v = (const _Float16 *)d_val;
            if (BM == 8 && BN == 16) fill(fill_kernel<_Float16, 8, 16, DUP>, v);
            else if (BM == 16 && BN == 16) fill(fill_kernel<_Float16, 16, 16, DUP>, v);
            else if (BM == 64 && BN == 32) fill(fill_kernel<_Float16, 64, 32, DUP>, v);
            else fill(fill_kernel<_Float16, 0, 0, DUP>, v);
        } else {
            const float *v = (const float *)d_val;
            if (BM == 8 && BN == 8) fill(fill_kernel<float, 8, 8, DUP>, v);
            else if (BM == 16 && BN == 8) fill(fill_kernel<float, 16, 8, DUP>, v);
            else if (BM == 64 && BN == 16) fill(fill_kernel<float, 64, 16, DUP>, v);
            else fill(fill_kernel<float, 0, 0, DUP>, v);
        }
    };
    if (h.dups || h.odd) shape(std::true_type{});
    else shape(std::false_type{});
    TCHK(hipGetLastError());
    return (int)hipStreamSynchronize(s);
}

}  // namespace

namespace tsp {

bool pack_total_fits(long long total) { return total >= 0 && total <= (long long)INT_MAX - 4; }

// Per-device address of `scratch`, looked up with the device current (each
// GPU holds its own copy at its own address).
constexpr int kScratchDevices = 64;
static std::mutex g_scratch_mu;
static int *g_scratch_ptr[kScratchDevices];

int scratch_init_current_device(int **ptr)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kScratchDevices) return TSP_EINVAL;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return TSP_EINVAL;
        g_scratch_ptr[dev] = (int *)p;
    }
    if (ptr) *ptr = g_scratch_ptr[dev];
    return TSP_OK;
}

}  // namespace tsp

extern "C" {

int tsp_tiles_pack_device_noalloc(int tilenum, int bm, int bn, int prec, const void *d_val,
                                  const unsigned long long *d_bitmap, void *d_pval, long long pval_capacity,
                                  int *d_vptr, long long *nvals, void *stream)
{
    if (tilenum < 0 || !nvals || !d_vptr || pval_capacity < 0 || (bm != 64 && bm != 16 && bm != 8) || bn <= 0 ||
        bn > 32)
        return TSP_EINVAL;
    if (prec != TSP_PREC_FP16 && prec != TSP_PREC_TF32) return TSP_EINVAL;
    if (pval_capacity > 0 && !d_pval) return TSP_EINVAL;
    if (tilenum > 0 && (!d_bitmap || !d_val)) return TSP_EINVAL;
    if ((long long)tilenum > TSP_PACK_NOALLOC_MAX_TILES) return TSP_EINVAL;
    int *sums = nullptr;
    if (const int st = tsp::scratch_init_current_device(&sums)) return st;
    long long *total64 = (long long *)(sums + kScratchInts - 2);
    hipStream_t s = (hipStream_t)stream;
    const int words = (bm * bn + 63) / 64;
    const int nb = (int)(((long long)tilenum + kPackBlockTiles - 1) / kPackBlockTiles);
    if (nb > 0) pack_count_kernel<<<nb, kThreads, 0, s>>>(d_bitmap, tilenum, words, d_vptr, sums);
    pack_block_scan_kernel<<<1, kThreads, 0, s>>>(sums, nb, total64);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    long long total = 0;
    if ((e = hipMemcpyAsync(&total, total64, sizeof total, hipMemcpyDeviceToHost, s)) != hipSuccess) return (int)e;
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return (int)e;
    *nvals = total;
    // the values plus 4 elements of zero padding (the kernels' packed loads
    // may read past the last value) must fit, and the offsets are ints
    if (!tsp::pack_total_fits(total) || total + 4 > pval_capacity) return TSP_EINVAL;
    if (nb > 0) pack_offsets_kernel<<<nb, kThreads, 0, s>>>(d_vptr, tilenum, sums);
    if (prec == TSP_PREC_FP16) {
        pack_tail_kernel<uint16_t><<<1, 64, 0, s>>>(d_vptr, tilenum, sums, nb, (uint16_t *)d_pval, pval_capacity, 4);
        if (tilenum > 0)
            if (const int st = launch_pack<uint16_t>(d_val, d_bitmap, d_vptr, tilenum, words, bm * bn, d_pval, pval_capacity, 0, s))
                return st;
    } else {
        pack_tail_kernel<uint32_t><<<1, 64, 0, s>>>(d_vptr, tilenum, sums, nb, (uint32_t *)d_pval, pval_capacity, 4);
        if (tilenum > 0)
            if (const int st = launch_pack<uint32_t>(d_val, d_bitmap, d_vptr, tilenum, words, bm * bn, d_pval, pval_capacity, 0, s))
                return st;
    }
    if ((e = hipGetLastError()) != hipSuccess || (e = hipStreamSynchronize(s)) != hipSuccess) return (int)e;
    return TSP_OK;
}


int tsp_tile_create_device(tsp_dev_tiles *out, int rows, int colA, long long nnz, const int *d_ptr,
                           const int *d_idx, const void *d_val, int BM, int BN, int prec, void *stream)
{
    if (!out) return TSP_EINVAL;
    memset(out, 0, sizeof *out);
    const int st = tile_create_device(out, rows, colA, nnz, d_ptr, d_idx, d_val, BM, BN, prec, stream);
    if (st != TSP_OK) tsp_dev_tiles_free(out);
    return st;
}

int tsp_tiles_pack_device(int tilenum, int bm, int bn, int prec, const void *d_val,
                          const unsigned long long *d_bitmap, long long *nvals, void **d_pval, int **d_vptr,
                          void *stream)
{
    if (tilenum < 0 || !nvals || (bm != 64 && bm != 16 && bm != 8) || bn <= 0 || bn > 32) return TSP_EINVAL;
    if (prec != TSP_PREC_FP16 && prec != TSP_PREC_TF32) return TSP_EINVAL;
    if ((d_pval == nullptr) != (d_vptr == nullptr)) return TSP_EINVAL;
    if (tilenum > 0 && (!d_bitmap || (d_pval && !d_val))) return TSP_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    const int words = (bm * bn + 63) / 64;
    DevBufs db(s);
    // the scan's state and ticket, then the 64-bit total
    Carve cv;
    const size_t o_state = cv.add(scan_state_bytes(tilenum)), o_ticket = cv.add(sizeof(int));
    const size_t o_total = cv.add(sizeof(long long));
    char *w = nullptr;
    TCHK(db.get(&w, cv.bytes));
    long long *d_total = (long long *)(w + o_total);
    TCHK(hipMemsetAsync(w, 0, cv.bytes, s));
    int *vptr = nullptr;
    if (d_pval) TCHK(tsp::dev_alloc((void **)&vptr, sizeof(int) * ((size_t)tilenum + 1)));
    auto fail = [&](int st) {
        (void)tsp::dev_free(vptr, false);
        return st;
    };
    hipError_t e = hipSuccess;
    if (!d_pval) {
        const long long nw = (long long)tilenum * words;
        if (nw > 0)
            count_bits_kernel<<<(unsigned)(nw < 1024ll * kThreads ? nblocks(nw) : 1024u), kThreads, 0, s>>>(
                d_bitmap, nw, (unsigned long long *)d_total);
        e = hipGetLastError();
    } else if (tilenum > 0) {
        // (offsets past INT_MAX are held there; the total says so below)
        e = (hipError_t)launch_scan(BitsAt{d_bitmap, words}, tilenum, vptr, (unsigned long long *)(w + o_state),
                                    (int *)(w + o_ticket), d_total, s);
    } else {
        e = hipMemsetAsync(vptr, 0, sizeof(int), s);
    }
    if (e != hipSuccess) return fail((int)e);
    long long total = 0;
    if ((e = hipMemcpyAsync(&total, d_total, sizeof total, hipMemcpyDeviceToHost, s)) != hipSuccess) return fail((int)e);
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return fail((int)e);
    *nvals = total;
    // the kernels' int offsets need the values plus the padding to stay
    // within INT_MAX
    if (!tsp::pack_total_fits(total)) return fail(TSP_EINVAL);
    if (!d_pval) return TSP_OK;
    // 4 elements of zero padding: the kernels' packed loads may read past the last value
    const size_t vs = prec == TSP_PREC_FP16 ? 2 : 4;
    void *pv = nullptr;
    if (const int st = tsp::dev_alloc(&pv, vs * ((size_t)total + 4))) return fail(st);
    int st = TSP_OK;
    if (tilenum == 0)
        st = (int)hipMemsetAsync(pv, 0, vs * 4, s);
    else if (prec == TSP_PREC_FP16)
        st = launch_pack<uint16_t>(d_val, d_bitmap, vptr, tilenum, words, bm * bn, pv, total + 4, 4, s);
    else
        st = launch_pack<uint32_t>(d_val, d_bitmap, vptr, tilenum, words, bm * bn, pv, total + 4, 4, s);
    if (st == TSP_OK) st = (int)hipStreamSynchronize(s);
    if (st != TSP_OK) {
        (void)tsp::dev_free(pv, false);
        return fail(st);
    }
    *d_pval = pv;
    *d_vptr = vptr;
    return TSP_OK;
}

int tsp_dev_tiles_free(tsp_dev_tiles *t)
{
    if (!t) return TSP_OK;
    // the first one's wait covers the rest
    const bool waited = tsp::dev_free(t->d_val, false) == TSP_OK && t->d_val;
    (void)tsp::dev_free(t->d_tile_ptr, waited);
    (void)tsp::dev_free(t->d_tile_nnz, waited);
    (void)tsp::dev_free(t->d_tile_colidx, waited);
    (void)tsp::dev_free(t->d_bitmap, waited);
    memset(t, 0, sizeof *t);
    return TSP_OK;
}

}  // extern "C"
