// Stable sort of a matrix's entries by column, on gfx950: the CSC pattern of
// the transpose kernels (each entry's CSR position, in column order).
//
// A least-significant-digit radix sort of (column, position) pairs in digits
// of at most 8 bits.  Per pass: SortCountKernel counts every digit's entries
// per tile of kSortTile, SortScanKernel turns each digit's counts into an
// exclusive scan over the tiles, and SortScatterKernel ranks a tile's entries
// stably in LDS, orders them by digit there and writes each digit's run (64
// entries on average) in one stretch.  The first pass makes its keys from
// col_ind and its positions from the entry's index, so nothing is copied
// beforehand.  Every launch can be gated on a device word: a Preprocess whose
// path decision (taken on the device) does not need the CSC pattern skips the
// sort without the host knowing.
//
// Small matrices keep hipCUB's sort (OwnSort).
//
// Bound: HBM traffic, 16 bytes per entry in the first pass (the column read
// twice, a pair written) and 20 in the others (the key twice, the position).
// Reference counterpart: sparse/spmv/arch35/spmv_kernel.cpp:861-879 orders its
// deterministic transpose by column.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <cstdint>

#include "aclsparse_internal.h"

namespace aclsp {
namespace {

constexpr int kWave = 64;
constexpr int kSortThreads = 1024;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kSortRounds = static_cast<int>(kSortTile) / kSortThreads;  // entries per thread
constexpr int kSegment = kSortRounds * kWave;                            // consecutive entries per wave
constexpr int kDigits = 1 << kSortDigitBits;
static_assert(kSortTile % kSortThreads == 0, "whole rounds");
static_assert((kSortMinNnz / kSortTile + 2) * kDigits <= kSortMinNnz, "counts fit a word per entry");

struct SortParams {
    // first pass: keys from the matrix
    const int32_t* col;
    int64_t col_stride;
    int32_t base;
    int64_t rows, cols;
    const void* norm;  // normalised row offsets (RowT)
    // later passes
    const int32_t* key_in;
    const int32_t* val_in;
    int32_t* key_out;
    int32_t* val_out;
    int64_t nnz, tiles;
    int32_t shift, digits;  // this pass's digit: (key >> shift) & (digits - 1)
    uint32_t* counts;       // [digits][tiles]: entries, then (SortScanKernel) those of the tiles before
    uint32_t* totals;       // [digits]: entries of the digit
    const uint32_t* gate;   // non-null: nothing runs when it reads 1
};

__device__ __forceinline__ bool Gated(const uint32_t* gate) { return gate != nullptr && *gate == 1U; }

// The sort key of entry k: its column, or cols when it lies outside the
// matrix's rows or columns (such entries sort after all others).
template <typename RowT, bool kFirst>
__device__ __forceinline__ uint32_t KeyAt(const SortParams& q, int64_t k, int64_t first, int64_t last)
{
    if constexpr (kFirst) {
        const int64_t c = static_cast<int64_t>(q.col[k * q.col_stride]) - q.base;
        return static_cast<uint32_t>(k >= first && k < last && c >= 0 && c < q.cols ? c : q.cols);
    } else {
        return static_cast<uint32_t>(q.key_in[k]);
    }
}

template <typename RowT, bool kFirst>
__device__ __forceinline__ void RowRange(const SortParams& q, int64_t& first, int64_t& last)
{
    if constexpr (kFirst) {
        first = static_cast<int64_t>(static_cast<const RowT*>(q.norm)[0]);
        last = static_cast<int64_t>(static_cast<const RowT*>(q.norm)[q.rows]);
    } else {
        first = last = 0;
    }
}

// counts[d * tiles + t] = entries of tile t whose digit is d.  Eight copies of
// the histogram, by lane: neighbouring entries often share a digit.
template <typename RowT, bool kFirst>
__global__ __launch_bounds__(kSortThreads) void SortCountKernel(SortParams q)
{
    constexpr int kCopies = 8;
    __shared__ uint32_t hist[kDigits * kCopies];
    if (Gated(q.gate)) return;
    const int64_t t = blockIdx.x;
    const int tid = threadIdx.x;
    for (int i = tid; i < kDigits * kCopies; i += kSortThreads) hist[i] = 0U;
    int64_t first, last;
    RowRange<RowT, kFirst>(q, first, last);
    uint32_t d[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const int64_t k = t * kSortTile + r * kSortThreads + tid;
        d[r] = k < q.nnz ? KeyAt<RowT, kFirst>(q, k, first, last) >> q.shift & (q.digits - 1) : 0xFFFFFFFFU;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        if (d[r] != 0xFFFFFFFFU) atomicAdd(&hist[d[r] * kCopies + (tid & (kCopies - 1))], 1U);
    }
    __syncthreads();
    if (tid < q.digits) {
        uint32_t n = 0U;
#pragma unroll
        for (int c = 0; c < kCopies; ++c) n += hist[tid * kCopies + c];
        q.counts[tid * q.tiles + t] = n;
    }
}

// Exclusive sum of v over the workgroup's threads (s holds a word per wave);
// total gets the sum of all.
__device__ __forceinline__ uint32_t BlockExclusive(uint32_t v, uint32_t* s, uint32_t& total)
{
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    uint32_t inc = v;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t o = __shfl_up(inc, d, kWave);
        inc += lane >= d ? o : 0U;
    }
    if (lane == kWave - 1) s[wv] = inc;
    __syncthreads();
    uint32_t before = 0U, all = 0U;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
        const uint32_t x = s[w];
        before += w < wv ? x : 0U;
        all += x;
    }
    __syncthreads();
    total = all;
    return before + inc - v;
}

// One workgroup per digit: counts of the digit -> entries in the tiles before, totals[d].
__global__ __launch_bounds__(kSortThreads) void SortScanKernel(SortParams q)
{
    __shared__ uint32_t s[kSortWaves];
    if (Gated(q.gate)) return;
    uint32_t* row = q.counts + static_cast<int64_t>(blockIdx.x) * q.tiles;
    uint32_t carry = 0U;
    for (int64_t t0 = 0; t0 < q.tiles; t0 += kSortThreads) {
        const int64_t t = t0 + threadIdx.x;
        const uint32_t v = t < q.tiles ? row[t] : 0U;
        uint32_t total;
        const uint32_t e = BlockExclusive(v, s, total);
        if (t < q.tiles) row[t] = carry + e;
        carry += total;
    }
    if (threadIdx.x == 0) q.totals[blockIdx.x] = carry;
}

// One workgroup per tile, wave w on the tile's entries [w*kSegment, ...), 64
// consecutive ones per round.  A round's lanes with equal digits find each
// other by one ballot per digit bit; a lane's rank is the wave's count of its
// digit before the round plus its equals in lower lanes, so ranks follow the
// entries' order.  LDS operations of one wave complete in order: the read of
// the count and the add of the round's entries need no wait between rounds.
template <typename RowT, bool kFirst>
__global__ __launch_bounds__(kSortThreads) void SortScatterKernel(SortParams q)
{
    __shared__ uint32_t staged[kSortTile];
    __shared__ uint32_t waveCnt[kSortWaves * kDigits];
    __shared__ uint32_t tileStart[kDigits];  // first place of each digit within the tile
    __shared__ uint32_t outBase[kDigits];    // its first output place minus that
    __shared__ uint32_t scan[kSortWaves];
    if (Gated(q.gate)) return;
    const int64_t t = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
    const int64_t k0 = t * kSortTile;
    const int n = static_cast<int>(q.nnz - k0 < kSortTile ? q.nnz - k0 : kSortTile);
    int64_t first, last;
    RowRange<RowT, kFirst>(q, first, last);
    uint32_t key[kSortRounds], val[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const int i = wv * kSegment + r * kWave + lane;
        key[r] = i < n ? KeyAt<RowT, kFirst>(q, k0 + i, first, last) : 0U;
        if constexpr (kFirst) val[r] = static_cast<uint32_t>(k0 + i);
        else val[r] = i < n ? static_cast<uint32_t>(q.val_in[k0 + i]) : 0U;
    }
    uint32_t gTotal = tid < q.digits ? q.totals[tid] : 0U;
    const uint32_t gBefore = tid < q.digits ? q.counts[tid * q.tiles + t] : 0U;
    for (int i = tid; i < kSortWaves * kDigits; i += kSortThreads) waveCnt[i] = 0U;
    __syncthreads();

    uint32_t* wc = waveCnt + wv * kDigits;
    uint32_t rank[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const bool in = wv * kSegment + r * kWave + lane < n;
        const uint32_t d = key[r] >> q.shift & (q.digits - 1);
        uint64_t peers = __ballot(in);
#pragma unroll
        for (int b = 0; b < kSortDigitBits; ++b) {
            const bool bit = (d >> b & 1U) != 0U;
            const uint64_t set = __ballot(bit);
            peers &= bit ? set : ~set;
        }
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(peers >> 32),
                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(peers), 0U));
        const uint32_t before = __hip_atomic_load(&wc[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (in && below == 0U) {
            __hip_atomic_fetch_add(&wc[d], static_cast<uint32_t>(__popcll(peers)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        rank[r] = before + below;
    }
    __syncthreads();

    // per digit: the waves' counts -> first place of each wave's entries in
    // the tile; the digit's first place in the tile and in the output
    uint32_t mine = 0U;
    if (tid < kDigits) {
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) {
            const uint32_t c = waveCnt[w * kDigits + tid];
            waveCnt[w * kDigits + tid] = mine;
            mine += c;
        }
    }
    uint32_t all;
    const uint32_t start = BlockExclusive(mine, scan, all);
    const uint32_t gStart = BlockExclusive(gTotal, scan, all);
    if (tid < kDigits) {
        tileStart[tid] = start;
        outBase[tid] = gStart + gBefore - start;
    }
    __syncthreads();

    // keys in digit order through LDS and out, then the positions the same way
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t d = key[r] >> q.shift & (q.digits - 1);
        rank[r] += tileStart[d] + wc[d];
        if (wv * kSegment + r * kWave + lane < n) staged[rank[r]] = key[r];
    }
    __syncthreads();
    uint32_t dst[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const int i = r * kSortThreads + tid;
        if (i < n) {
            const uint32_t k = staged[i];
            dst[r] = outBase[k >> q.shift & (q.digits - 1)] + static_cast<uint32_t>(i);
            q.key_out[dst[r]] = static_cast<int32_t>(k);
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        if (wv * kSegment + r * kWave + lane < n) staged[rank[r]] = val[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const int i = r * kSortThreads + tid;
        if (i < n) q.val_out[dst[r]] = static_cast<int32_t>(staged[i]);
    }
}

// Keys and positions of a small matrix, for hipCUB's sort (key_out, val_out).
template <typename RowT>
__global__ __launch_bounds__(kSortThreads) void SortKeysKernel(SortParams q)
{
    int64_t first, last;
    RowRange<RowT, true>(q, first, last);
    const int64_t k = static_cast<int64_t>(blockIdx.x) * kSortThreads + threadIdx.x;
    if (k >= q.nnz) return;
    q.key_out[k] = static_cast<int32_t>(KeyAt<RowT, true>(q, k, first, last));
    q.val_out[k] = static_cast<int32_t>(k);
}

// Sorts (c.key, c.val); the result may lie in the temporaries, which then
// change places with them (size query when temp is null).
hipError_t SmallSort(void* temp, size_t& bytes, CscSort& c, int bits, hipStream_t s)
{
    hipcub::DoubleBuffer<int32_t> keys(c.key, c.key_tmp), vals(c.val, c.val_tmp);
    const hipError_t e =
        hipcub::DeviceRadixSort::SortPairs(temp, bytes, keys, vals, static_cast<int>(c.nnz), 0, bits, s);
    c.key = keys.Current();
    c.key_tmp = keys.Alternate();
    c.val = vals.Current();
    c.val_tmp = vals.Alternate();
    return e;
}

template <typename RowT, bool kFirst>
void Pass(const SortParams& q, hipStream_t s)
{
    const dim3 tiles(static_cast<unsigned>(q.tiles)), threads(kSortThreads);
    hipLaunchKernelGGL((SortCountKernel<RowT, kFirst>), tiles, threads, 0, s, q);
    hipLaunchKernelGGL(SortScanKernel, dim3(static_cast<unsigned>(q.digits)), threads, 0, s, q);
    hipLaunchKernelGGL((SortScatterKernel<RowT, kFirst>), tiles, threads, 0, s, q);
}

}  // namespace

size_t CscSortTempBytes(int64_t cols, int64_t nnz)
{
    if (OwnSort(cols, nnz)) return 0;
    return LastResult(nnz, [](int64_t n) {
        size_t bytes = 0;
        CscSort c{};
        c.nnz = n;
        if (SmallSort(nullptr, bytes, c, 31, nullptr) != hipSuccess) {
            bytes = static_cast<size_t>(n) * 16 + (1 << 20);  // no device to ask: a generous bound
        }
        return bytes;
    });
}

int LaunchCscSort(CscSort& c, void* stream)
{
    if (c.nnz <= 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    SortParams q{};
    q.col = c.col;
    q.col_stride = c.col_stride;
    q.base = c.base;
    q.rows = c.rows;
    q.cols = c.cols;
    q.norm = c.norm;
    q.nnz = c.nnz;
    q.tiles = (c.nnz + kSortTile - 1) / kSortTile;
    q.counts = c.counts;
    q.totals = q.counts + q.tiles * kDigits;
    q.gate = c.gate;
    const int bits = SortBits(c.cols);
    if (!OwnSort(c.cols, c.nnz)) {
        q.key_out = c.key;
        q.val_out = c.val;
        const dim3 grid(static_cast<unsigned>((c.nnz + kSortThreads - 1) / kSortThreads));
        if (c.rowptr64) hipLaunchKernelGGL(SortKeysKernel<int64_t>, grid, dim3(kSortThreads), 0, s, q);
        else hipLaunchKernelGGL(SortKeysKernel<int32_t>, grid, dim3(kSortThreads), 0, s, q);
        void* temp = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(c.temp) + 255) & ~uintptr_t{255});
        size_t bytes = c.temp_bytes;
        return SmallSort(temp, bytes, c, bits, s) == hipSuccess ? 0 : 1;
    }
    const int passes = SortPasses(c.cols);
    for (int p = 0; p < passes; ++p) {
        const int w = bits / passes + (p < bits % passes ? 1 : 0);
        q.digits = 1 << w;
        const bool toFinal = (passes - 1 - p) % 2 == 0;  // the last pass writes key / val
        q.key_in = toFinal ? c.key_tmp : c.key;
        q.val_in = toFinal ? c.val_tmp : c.val;
        q.key_out = toFinal ? c.key : c.key_tmp;
        q.val_out = toFinal ? c.val : c.val_tmp;
        if (p > 0) Pass<int32_t, false>(q, s);
        else if (c.rowptr64) Pass<int64_t, true>(q, s);
        else Pass<int32_t, true>(q, s);
        q.shift += w;
    }
    return 0;
}

}  // namespace aclsp
