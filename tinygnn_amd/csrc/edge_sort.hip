// edge_sort.hip -- edge_list_to_csr by partition and sort on gfx950.
//
// The edges are partitioned into buckets of 2^shift consecutive rows (at most
// 4,096 buckets, of 4,096 edges on average where that many allow it), each edge
// packed into 32 bits (row within the bucket, destination), and a workgroup
// sorts a bucket's keys in LDS and writes its rows' row_ptr, col_ind and val.
// No step does an atomic per edge outside LDS.  Every memory pass is a stream
// (src and dst twice, the keys once each way, the outputs once), except the
// partition's writes, runs of a tile's edges of one bucket; the sorts are bound
// by the vector instructions that rank the keys (about 270 per 64 keys).
// 1M nodes, 50M edges in random order: 1.16 ms (count 0.12, partition 0.27,
// sorts 0.71).  The general build in graph.hip, which counts and places edges
// by one device atomic each and sorts row by row, takes 7.8 ms (2.5 count, 2.7
// place, 2.1 sorts).  8,192 buckets: partition 0.38, sorts 0.75 ms; one sort
// kernel for all buckets at one workgroup per CU: 0.91 ms.
#include "common.hpp"
#include "device_utils.hpp"
#include "edge_sort.hpp"

#include <algorithm>

namespace tg {
namespace {

constexpr int kBinsMax = 4096;
constexpr int kBlock = 1024;
constexpr int kWaves = kBlock / kWave;
constexpr int kTileItems = 16;
constexpr int kTile = kBlock * kTileItems;  // edges per partition step
constexpr int kGrid = 256;                  // partition workgroups: one per CU (130 KB of LDS)
constexpr int kEdgesPerBin = 4096;
constexpr int kRowsPerBin = 2048;           // where rows are few edges each
// Keys per thread that a workgroup sorts in LDS: 16 leave room for two
// workgroups on a CU (80 KB of LDS, 64 registers), 32 fill one (144 KB).
constexpr int kSortItems = 16, kSortItemsLong = 32;
constexpr int kLowBits = 12;                   // first digit: 4,096 counters
constexpr int kDigitBits = 8;                  // later digits: 256 counters per wavefront
constexpr int kLongItems = 8;
// Longer buckets take the general build: one workgroup sorts a bucket through
// memory at about 1 ns per key and digit, where the general build spreads one
// long row over the chip.
constexpr int64_t kBucketMax = int64_t(1) << 18;
constexpr uint32_t kOneF = 0x3f800000u;  // 1.0f

static_assert(kLowBits <= 12 && (1 << kDigitBits) * kWaves == kBinsMax, "counter arrays");

struct Build {
    int64_t n, e, chunk;  // chunk: edges per partition workgroup
    int32_t bins, grid;
    int shift, dst_bits;
    const int32_t* src;
    const int32_t* dst;
    int32_t* counts;   // [bins][grid]
    int32_t* offsets;  // its exclusive scan, bins * grid + 1
    int32_t* longs;    // the buckets of more than kSortItems * kBlock edges
};

// The exclusive scan of cnt[0, 4096) over the workgroup, in place (4 per
// thread); cnt[4096] is not written.  Contains barriers.
__device__ __forceinline__ void scan_counters(int* cnt, int* part) {
    int c[4], sum = 0, total;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        c[j] = cnt[4 * threadIdx.x + j];
        sum += c[j];
    }
    int ex = block_exclusive_scan<kBlock>(sum, part, &total);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        cnt[4 * threadIdx.x + j] = ex;
        ex += c[j];
    }
}

// Counts a chunk's edges per bucket, and checks the endpoints: bad = the first
// invalid endpoint as 2 * edge + (0 = src, 1 = dst) (dst where check_dst),
// dst_bad = whether any destination is invalid.
__global__ __launch_bounds__(kBlock) void bucket_count_kernel(Build b, int check_dst,
                                                              EdgeSortStatus* status) {
    __shared__ int hist[kBinsMax];
    for (int i = threadIdx.x; i < b.bins; i += kBlock) hist[i] = 0;
    __syncthreads();
    constexpr int kUnroll = 8;
    const int64_t lo = static_cast<int64_t>(blockIdx.x) * b.chunk;
    const int64_t hi = min(b.e, lo + b.chunk);
    const uint32_t n = static_cast<uint32_t>(b.n);
    bool any_dst = false;
    for (int64_t i0 = lo + threadIdx.x; i0 < hi; i0 += kUnroll * kBlock) {
        int32_t s[kUnroll], d[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int64_t i = i0 + u * kBlock;
            s[u] = i < hi ? b.src[i] : 0;
            d[u] = i < hi ? b.dst[i] : 0;
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int64_t i = i0 + u * kBlock;
            if (i >= hi) continue;
            const bool sbad = static_cast<uint32_t>(s[u]) >= n;
            const bool dbad = static_cast<uint32_t>(d[u]) >= n;
            any_dst |= dbad;
            if (sbad || (dbad && check_dst))
                atomicMin(&status->bad, static_cast<unsigned long long>(2 * i + (sbad ? 0 : 1)));
            if (!sbad) atomicAdd(&hist[s[u] >> b.shift], 1);
        }
    }
    if (any_dst) atomicOr(&status->dst_bad, 1);
    __syncthreads();
    for (int i = threadIdx.x; i < b.bins; i += kBlock)
        b.counts[static_cast<int64_t>(i) * b.grid + blockIdx.x] = hist[i];
}

__global__ void status_init_kernel(EdgeSortStatus* status) {
    status->bad = ~0ull;
    status->dst_bad = 0;
    status->longest = 0;
    status->n_long = 0;
}

__global__ __launch_bounds__(256) void bucket_max_kernel(Build b, EdgeSortStatus* status) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    int len = 0;
    if (i < b.bins)
        len = b.offsets[static_cast<int64_t>(i + 1) * b.grid] -
              b.offsets[static_cast<int64_t>(i) * b.grid];
    if (len > kSortItems * kBlock) b.longs[atomicAdd(&status->n_long, 1)] = i;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) len = max(len, __shfl_xor(len, d, kWave));
    if ((threadIdx.x & (kWave - 1)) == 0 && len > 0) atomicMax(&status->longest, len);
}

// Writes every edge's key into its bucket: tile by tile, the tile's keys
// ordered by bucket in LDS so that a bucket's keys leave as one run.
__global__ __launch_bounds__(kBlock) void bucket_scatter_kernel(Build b, uint32_t* out) {
    __shared__ int start[kBinsMax + 1];  // per tile: counts, then their scan
    __shared__ int cursor[kBinsMax];
    __shared__ uint32_t keys[kTile];
    __shared__ uint16_t bin_of[kTile];
    __shared__ int part[kWaves];
    for (int i = threadIdx.x; i < b.bins; i += kBlock)
        cursor[i] = b.offsets[static_cast<int64_t>(i) * b.grid + blockIdx.x];
    const int64_t lo = static_cast<int64_t>(blockIdx.x) * b.chunk;
    const int64_t hi = min(b.e, lo + b.chunk);
    const int mask = (1 << b.shift) - 1;
    int32_t s[kTileItems], d[kTileItems];
    auto fetch = [&](int64_t t0) {
#pragma unroll
        for (int u = 0; u < kTileItems; ++u) {
            const int64_t i = t0 + u * kBlock + threadIdx.x;
            s[u] = i < hi ? b.src[i] : -1;
            d[u] = i < hi ? b.dst[i] : 0;
        }
    };
    fetch(lo);
    for (int64_t t0 = lo; t0 < hi; t0 += kTile) {
        const int cnt = static_cast<int>(min<int64_t>(kTile, hi - t0));
#pragma unroll
        for (int j = 0; j < 4; ++j) start[4 * threadIdx.x + j] = 0;
        if (threadIdx.x == 0) start[kBinsMax] = cnt;
        __syncthreads();
        int rank[kTileItems];
#pragma unroll
        for (int u = 0; u < kTileItems; ++u)
            rank[u] = s[u] >= 0 ? atomicAdd(&start[s[u] >> b.shift], 1) : 0;
        __syncthreads();
        scan_counters(start, part);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kTileItems; ++u) {
            if (s[u] >= 0) {
                const int bin = s[u] >> b.shift;
                const int p = start[bin] + rank[u];
                keys[p] = (static_cast<uint32_t>(s[u] & mask) << b.dst_bits) |
                          static_cast<uint32_t>(d[u]);
                bin_of[p] = static_cast<uint16_t>(bin);
            }
        }
        fetch(t0 + kTile);  // the next tile, behind this one's writes
        __syncthreads();
        for (int j = threadIdx.x; j < cnt; j += kBlock) {
            const int bin = bin_of[j];
            out[cursor[bin] + (j - start[bin])] = keys[j];
        }
        __syncthreads();
        for (int j = 4 * threadIdx.x; j < min(4 * static_cast<int>(threadIdx.x) + 4, b.bins); ++j)
            cursor[j] += start[j + 1] - start[j];
        __syncthreads();
    }
}

// Lanes of the wavefront, among `among`, whose digit d (of kDigitBits bits)
// equals the caller's.
__device__ __forceinline__ uint64_t match_digit(uint32_t d, uint64_t among) {
    uint32_t lo = static_cast<uint32_t>(among), hi = static_cast<uint32_t>(among >> 32);
#pragma unroll
    for (int i = 0; i < kDigitBits; ++i) {
        const uint32_t one = static_cast<uint32_t>(static_cast<int32_t>(d << (31 - i)) >> 31);
        const uint64_t bal = __ballot(one != 0);
        lo &= ~(static_cast<uint32_t>(bal) ^ one);
        hi &= ~(static_cast<uint32_t>(bal >> 32) ^ one);
    }
    return static_cast<uint64_t>(hi) << 32 | lo;
}

__device__ __forceinline__ int lanes_below(uint64_t m) {
    return static_cast<int>(__builtin_amdgcn_mbcnt_hi(
        static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u)));
}

// The rank of a wavefront's key among its earlier keys of the same digit
// (counters[d], the wavefront's own), counting it; valid keys in lane order.
__device__ __forceinline__ int count_digit(int* counters, uint32_t d, bool valid) {
    const uint64_t m = match_digit(d, __ballot(valid));
    int r = 0;
    if (valid) {
        const int before = counters[d];
        const int below = lanes_below(m);
        r = before + below;
        if (below == 0) counters[d] = before + __popcll(m);
    }
    // the counter's update before the next key's read (one wavefront's LDS
    // operations run in program order)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_sched_barrier(0);  // one key's match at a time in registers
    return r;
}

// row_ptr of the rows that start at sorted position pos (after row `prev`), up
// to kGap of them; where more are empty in a row, *wide says that every row is
// to be searched for (search_rows), so that a row's cost does not depend on its
// neighbours: 65,536 rows, 131 edges in one of them, took 1.7 ms, now 0.07.
// (Searches alone took 98 us for 1M rows of one edge on average, 92 so.)
constexpr int kGap = 64;
__device__ __forceinline__ void start_rows(int32_t* row_ptr, int prev, int row, int32_t pos,
                                           int* wide) {
    if (row - prev > kGap) *wide = 1;
    for (int r = prev + 1; r <= min(row, prev + kGap); ++r) row_ptr[r] = pos;
}

__device__ __forceinline__ void search_rows(int32_t* row_ptr, int rows, const uint32_t* sorted,
                                            int size, int dst_bits, int32_t base) {
    for (int r = threadIdx.x; r < rows; r += kBlock) {
        const uint32_t key = static_cast<uint32_t>(r) << dst_bits;
        int lo = 0, hi = size;  // the first key not below it
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (sorted[mid] < key) lo = mid + 1;
            else hi = mid;
        }
        row_ptr[r] = base + lo;
    }
}

// One workgroup sorts one bucket (ITEMS = kSortItems: the short ones; else the
// listed ones).  Up to 1,024 ITEMS keys in LDS: the first digit (12 bits)
// placed by LDS atomics in any order, the others (8 bits) stably, the
// wavefronts' counts of a digit in wavefront order.  More keys: stable passes
// of 8 bits through memory, between the two output arrays.
template <int ITEMS>
__global__ __launch_bounds__(kBlock, ITEMS == kSortItems ? 8 : 4) void bucket_sort_kernel(
    Build b, int32_t* row_ptr, uint32_t* col, uint32_t* val) {
    __shared__ uint32_t buf[ITEMS * kBlock];
    __shared__ int cnt[kBinsMax];
    // the scans' partial sums: in buf, whose keys are in registers during a scan
    int* part = reinterpret_cast<int*>(buf) + (1 << kDigitBits);
    const int bin = ITEMS == kSortItems ? static_cast<int>(blockIdx.x) : b.longs[blockIdx.x];
    const int32_t base = b.offsets[static_cast<int64_t>(bin) * b.grid];
    const int size = b.offsets[static_cast<int64_t>(bin + 1) * b.grid] - base;
    const int64_t row0 = static_cast<int64_t>(bin) << b.shift;
    const int rows = static_cast<int>(min<int64_t>(int64_t(1) << b.shift, b.n - row0));
    const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int key_bits = b.shift + b.dst_bits;
    const uint32_t dst_mask = (1u << b.dst_bits) - 1;
    int* wide = cnt;  // (the counters are done with by then)
    if (bin == b.bins - 1 && threadIdx.x == 0) row_ptr[b.n] = static_cast<int32_t>(b.e);
    row_ptr += row0;
    if (size == 0) {
        for (int r = threadIdx.x; r < rows; r += kBlock) row_ptr[r] = base;
        return;
    }
    if (ITEMS == kSortItems && size > ITEMS * kBlock) return;  // listed
    uint32_t* in = val + base;
    uint32_t* other = col + base;
    if (size <= ITEMS * kBlock) {
        const int items = (size + kBlock - 1) / kBlock;
        uint32_t k[ITEMS];
        uint32_t ranks[ITEMS / 2];  // two 16-bit ranks each
        const auto rank = [&](int i) {
            return static_cast<int>(i % 2 ? ranks[i / 2] >> 16 : ranks[i / 2] & 0xFFFF);
        };
        const int first = wave * items * kWave + lane;  // key i of the lane: first + 64 i
        // opaque, so that the 2 x ITEMS lane masks are not all kept in scalar
        // registers (spilled, they tripled the kernel's time)
        const auto valid = [&](int i) {
            int left = size - first;
            asm volatile("" : "+v"(left));
            return i * kWave < left;
        };
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            k[i] = in[min(first + i * kWave, size - 1)];
        for (int lo = 0; lo < key_bits;) {
            const int bits = min(lo == 0 ? kLowBits : kDigitBits, key_bits - lo);
            const uint32_t dm = (1u << bits) - 1;
#pragma unroll
            for (int j = 0; j < 4; ++j) cnt[4 * threadIdx.x + j] = 0;
            __syncthreads();
            if (lo == 0) {
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) {
                    int r = 0;
                    if (i < items && valid(i)) r = atomicAdd(&cnt[k[i] & dm], 1);
                    ranks[i / 2] = i % 2 ? ranks[i / 2] | r << 16 : r;
                }
                __syncthreads();
                scan_counters(cnt, part);
                __syncthreads();
#pragma unroll
                for (int i = 0; i < ITEMS; ++i)
                    if (i < items && valid(i)) buf[cnt[k[i] & dm] + rank(i)] = k[i];
            } else {
                int* mine = cnt + wave * (1 << kDigitBits);
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) {
                    int r = 0;
                    if (i < items)
                        r = count_digit(mine, (k[i] >> lo) & dm, valid(i));
                    ranks[i / 2] = i % 2 ? ranks[i / 2] | r << 16 : r;
                }
                __syncthreads();
                // digit-major, then wavefront: thread t scans wavefronts
                // 4 (t % 4).. of digit t / 4
                int c[4], sum = 0, total;
                int* col4 = cnt + (threadIdx.x & 3) * 4 * (1 << kDigitBits) + (threadIdx.x >> 2);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    c[j] = col4[j << kDigitBits];
                    sum += c[j];
                }
                int ex = block_exclusive_scan<kBlock>(sum, part, &total);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    col4[j << kDigitBits] = ex;
                    ex += c[j];
                }
                __syncthreads();
#pragma unroll
                for (int i = 0; i < ITEMS; ++i)
                    if (i < items && valid(i))
                        buf[mine[(k[i] >> lo) & dm] + rank(i)] = k[i];
            }
            __syncthreads();
            lo += bits;
            if (lo < key_bits) {
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) k[i] = buf[first + i * kWave];  // within buf
            }
        }
        if (threadIdx.x == 0) *wide = 0;
        __syncthreads();
        for (int j = threadIdx.x; j < size; j += kBlock) {
            const uint32_t x = buf[j];
            const int row = static_cast<int>(x >> b.dst_bits);
            const int prev = j > 0 ? static_cast<int>(buf[j - 1] >> b.dst_bits) : -1;
            other[j] = x & dst_mask;
            in[j] = kOneF;
            start_rows(row_ptr, prev, row, base + j, wide);
            if (j == size - 1) start_rows(row_ptr, row, rows - 1, base + size, wide);
        }
        __syncthreads();
        if (*wide) search_rows(row_ptr, rows, buf, size, b.dst_bits, base);
        return;
    }
    if constexpr (ITEMS == kSortItems) return;
    int* digit = reinterpret_cast<int*>(buf);  // next position of each digit
    int* mine = cnt + wave * (1 << kDigitBits);
    for (int lo = 0; lo < key_bits; lo += kDigitBits) {
        const int bits = min(kDigitBits, key_bits - lo);
        const uint32_t dm = (1u << bits) - 1;
        if (threadIdx.x < (1 << kDigitBits)) digit[threadIdx.x] = 0;
        __syncthreads();
        for (int j = threadIdx.x; j < size; j += kBlock) atomicAdd(&digit[(in[j] >> lo) & dm], 1);
        __syncthreads();
        int total;
        const int c = threadIdx.x < (1 << kDigitBits) ? digit[threadIdx.x] : 0;
        const int ex = block_exclusive_scan<kBlock>(c, part, &total);
        if (threadIdx.x < (1 << kDigitBits)) digit[threadIdx.x] = ex;
        for (int t0 = 0; t0 < size; t0 += kLongItems * kBlock) {
            uint32_t k[kLongItems];
            int rank[kLongItems];
            const int first = t0 + wave * kLongItems * kWave + lane;
#pragma unroll
            for (int i = 0; i < kLongItems; ++i)
                k[i] = first + i * kWave < size ? in[first + i * kWave] : 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) cnt[4 * threadIdx.x + j] = 0;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kLongItems; ++i)
                rank[i] = count_digit(mine, (k[i] >> lo) & dm, first + i * kWave < size);
            __syncthreads();
            if (threadIdx.x < (1 << kDigitBits)) {
                int at = digit[threadIdx.x];
                for (int w = 0; w < kWaves; ++w) {
                    int& x = cnt[(w << kDigitBits) + threadIdx.x];
                    const int y = x;
                    x = at;
                    at += y;
                }
                digit[threadIdx.x] = at;
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kLongItems; ++i)
                if (first + i * kWave < size) other[mine[(k[i] >> lo) & dm] + rank[i]] = k[i];
            __syncthreads();
        }
        uint32_t* t = in;
        in = other;
        other = t;
    }
    if (threadIdx.x == 0) *wide = 0;
    __syncthreads();
    for (int j = threadIdx.x; j < size; j += kBlock) {
        const int row = static_cast<int>(in[j] >> b.dst_bits);
        const int prev = j > 0 ? static_cast<int>(in[j - 1] >> b.dst_bits) : -1;
        start_rows(row_ptr, prev, row, base + j, wide);
        if (j == size - 1) start_rows(row_ptr, row, rows - 1, base + size, wide);
    }
    __syncthreads();
    if (*wide) search_rows(row_ptr, rows, in, size, b.dst_bits, base);
    __syncthreads();
    for (int j = threadIdx.x; j < size; j += kBlock) {
        const uint32_t x = in[j];
        col[base + j] = x & dst_mask;
        val[base + j] = kOneF;
    }
}

int bits_for(int64_t n) {  // bits of 0..n-1, at least 1
    int b = 1;
    while ((int64_t(1) << b) < n) ++b;
    return b;
}

Build shape(int64_t n, int64_t e) {
    Build b{};
    b.n = n;
    b.e = e;
    b.dst_bits = bits_for(n);
    const int64_t want =
        std::clamp<int64_t>(std::max(e / kEdgesPerBin, n / kRowsPerBin), 1, kBinsMax);
    while (b.shift < 32 - b.dst_bits && ceil_div(n, int64_t(1) << b.shift) > want) ++b.shift;
    b.bins = static_cast<int32_t>(ceil_div(n, int64_t(1) << b.shift));
    // few edges: shares of 1,024, since equal sources contend for an LDS counter
    // (20,000 edges ordered by source 108 us in whole tiles, 80 in shares,
    // 87 by the general build)
    b.chunk = e <= kGrid * kBlock ? kBlock : ceil_div(ceil_div(e, kTile), kGrid) * kTile;
    b.grid = static_cast<int32_t>(ceil_div(e, b.chunk));
    return b;
}

}  // namespace

// A key holds a row of its bucket and a destination in 32 bits: with 4,096
// buckets that is n <= 2^22.
bool edge_sort_fits(int64_t n, int64_t e) { return n >= 1 && n <= (int64_t(1) << 22) && e >= 1; }

size_t edge_sort_ws(int64_t n, int64_t e) {
    if (!edge_sort_fits(n, e)) return 0;
    const Build b = shape(n, e);
    const int64_t m = static_cast<int64_t>(b.bins) * b.grid;
    Carver c(nullptr, 0);
    c.take<EdgeSortStatus>(1);
    c.take<int32_t>(m);
    c.take<int32_t>(m + 1);
    c.take<int64_t>(scan_temp_elems(m));
    c.take<int32_t>(b.bins);
    return c.bytes();
}

namespace {

struct Work {
    EdgeSortStatus* status;
    int64_t* scan;
};

Build carve(int64_t n, int64_t e, const int32_t* src, const int32_t* dst, void* work,
            size_t work_bytes, Work& w) {
    Build b = shape(n, e);
    b.src = src;
    b.dst = dst;
    const int64_t m = static_cast<int64_t>(b.bins) * b.grid;
    Carver c(work, work_bytes);
    w.status = c.take<EdgeSortStatus>(1);
    b.counts = c.take<int32_t>(m);
    b.offsets = c.take<int32_t>(m + 1);
    w.scan = c.take<int64_t>(scan_temp_elems(m));
    b.longs = c.take<int32_t>(b.bins);
    return b;
}

}  // namespace

EdgeSortStatus edge_sort_count(int64_t n, int64_t e, const int32_t* src, const int32_t* dst,
                               bool check_dst, void* work, size_t work_bytes, hipStream_t s) {
    Work w;
    const Build b = carve(n, e, src, dst, work, work_bytes, w);
    status_init_kernel<<<1, 1, 0, s>>>(w.status);
    TG_LAUNCH_CHECK();
    bucket_count_kernel<<<b.grid, kBlock, 0, s>>>(b, check_dst ? 1 : 0, w.status);
    TG_LAUNCH_CHECK();
    exclusive_scan_i32(b.counts, b.offsets, static_cast<int64_t>(b.bins) * b.grid, w.scan, s);
    bucket_max_kernel<<<static_cast<unsigned>(ceil_div(b.bins, 256)), 256, 0, s>>>(b, w.status);
    TG_LAUNCH_CHECK();
    EdgeSortStatus h;
    TG_HIP(hipMemcpyAsync(&h, w.status, sizeof(h), hipMemcpyDeviceToHost, s));
    TG_HIP(hipStreamSynchronize(s));
    return h;
}

bool edge_sort_ready(const EdgeSortStatus& h) {
    return h.bad == ~0ull && h.dst_bad == 0 && h.longest <= kBucketMax;
}

void edge_sort_finish(const EdgeSortStatus& h, int64_t n, int64_t e, const int32_t* src,
                      const int32_t* dst, int32_t* row_ptr, int32_t* col_ind, float* val,
                      void* work, size_t work_bytes, hipStream_t s) {
    Work w;
    const Build b = carve(n, e, src, dst, work, work_bytes, w);
    // the keys wait in val, which the sort overwrites
    auto* keys = reinterpret_cast<uint32_t*>(val);
    auto* col = reinterpret_cast<uint32_t*>(col_ind);
    bucket_scatter_kernel<<<b.grid, kBlock, 0, s>>>(b, keys);
    TG_LAUNCH_CHECK();
    if (h.n_long > 0) {
        bucket_sort_kernel<kSortItemsLong><<<h.n_long, kBlock, 0, s>>>(b, row_ptr, col, keys);
        TG_LAUNCH_CHECK();
    }
    bucket_sort_kernel<kSortItems><<<b.bins, kBlock, 0, s>>>(b, row_ptr, col, keys);
    TG_LAUNCH_CHECK();
}

}  // namespace tg
