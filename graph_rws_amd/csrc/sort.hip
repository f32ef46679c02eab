// Stable LSD radix sort of 64-bit keys with a 32-bit payload (gfx950).
//
// Used by the device BCSR builder (key = window, column, row-in-window) and
// by the sampler's unique-and-relabel (key = global node id).  Each pass over
// one 8-bit digit is three launches:
//   1. digit histogram per tile of 256 x iters keys (wave64 match by ballot,
//      one LDS atomic per distinct digit per wave), or of 8,192 keys from 2^20
//      keys on (radix_*_big_kernel); iters is at most 16 and as small as 1 below 16k keys, so that a small sort still
//      spreads over up to 64 work-groups instead of a few long ones,
//   2. exclusive scan of the digit-major [256][tiles] histogram, which gives
//      every (digit, tile) its output base in stable order,
//   3. stable scatter: each tile re-reads its keys in index order and ranks
//      them by (wave prefix across waves, ballot rank within the wave).
// Only ceil(bits / 8) passes run, so keys that use few bits sort fast.
#include "grws_internal.h"

namespace grws {

namespace {

constexpr int kRsBlock = 256;
constexpr int kRsWaves = kRsBlock / kWave;
constexpr int kRsMaxIters = 16;

// Keys per tile: 256 x iters, iters = ceil(n / 16k) clamped to [1, 16]: up
// to 256k keys a sort has at most 64 tiles, so its 256 x tiles digit counts
// take the one-launch scan (16k elements).
inline int radix_iters(int64_t n) {
    const int64_t it = (n + 16383) / 16384;
    return (int)(it < 1 ? 1 : (it > kRsMaxIters ? kRsMaxIters : it));
}

// Lanes of the wave whose 8-bit digit equals this lane's (valid lanes only).
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid) {
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bb = __ballot(bit);
        m &= bit ? bb : ~bb;
    }
    return m;
}

__global__ __launch_bounds__(kRsBlock) void radix_hist_kernel(const uint64_t* __restrict__ keys, int64_t n, int shift,
                                                              int64_t ntiles, int iters, int32_t* __restrict__ counts) {
    __shared__ int32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kRsBlock * iters;
    for (int it = 0; it < iters; ++it) {
        const int64_t i = base + (int64_t)it * kRsBlock + threadIdx.x;
        const bool valid = i < n;
        const uint32_t d = valid ? (uint32_t)(keys[i] >> shift) & 255u : 0u;
        const uint64_t m = match_digit(d, valid);
        if (valid && (m & lanemask_lt()) == 0) atomicAdd(&h[d], (int32_t)__popcll(m));
    }
    __syncthreads();
    counts[(int64_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(kRsBlock) void radix_scatter_kernel(const uint64_t* __restrict__ kin,
                                                                 const uint32_t* __restrict__ vin, int64_t n,
                                                                 int shift, int64_t ntiles, int iters,
                                                                 const int64_t* __restrict__ offsets,
                                                                 uint64_t* __restrict__ kout,
                                                                 uint32_t* __restrict__ vout) {
    __shared__ int64_t base_off[256];
    __shared__ int32_t wcnt[kRsWaves][256];
    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    base_off[tid] = offsets[(int64_t)tid * ntiles + blockIdx.x];
    const int64_t tile0 = (int64_t)blockIdx.x * kRsBlock * iters;
    for (int it = 0; it < iters; ++it) {
        const int64_t i = tile0 + (int64_t)it * kRsBlock + tid;
        const bool valid = i < n;
        uint64_t k = 0;
        uint32_t v = 0;
        if (valid) {
            k = kin[i];
            if (vin) v = vin[i];
        }
        const uint32_t d = (uint32_t)(k >> shift) & 255u;
#pragma unroll
        for (int w = 0; w < kRsWaves; ++w) wcnt[w][tid] = 0;
        __syncthreads();
        const uint64_t m = match_digit(d, valid);
        const int rank = __popcll(m & lanemask_lt());
        if (valid && rank == 0) wcnt[wave][d] = __popcll(m);
        __syncthreads();
        int32_t tot = 0;
#pragma unroll
        for (int w = 0; w < kRsWaves; ++w) {
            const int32_t t = wcnt[w][tid];
            wcnt[w][tid] = tot;
            tot += t;
        }
        __syncthreads();
        if (valid) {
            const int64_t pos = base_off[d] + wcnt[wave][d] + rank;
            kout[pos] = k;
            if (vin) vout[pos] = v;
        }
        __syncthreads();
        base_off[tid] += tot;
    }
}

// Large sorts (kRsBigKeys keys or more): tiles of 8,192 keys.  Memory bound: 8
// bytes read to count a key, 12 read and 12 written to move it, 0.73 ms per
// pass over 115M keys at 5 TB/s.  What held the small-tile kernels to 1.54 +
// 0.32 ms per pass was one load and four barriers per 256 keys; these take
// 0.57 + 0.23 ms (4.9 and 4.0 TB/s).  Here each wave
// loads its 1,024 consecutive keys at once and ranks them against its own
// digit counters (the wave's LDS operations run in order, so no barrier
// until all are ranked); the tile is then put in digit order in LDS and
// written out in runs of ~32 keys per digit.  Consecutive tiles run on one
// XCD, so the lines that two tiles' runs share meet in its L2.
constexpr int kRbBlock = 512;
constexpr int kRbWaves = kRbBlock / kWave;
constexpr int kRbItems = 16;
constexpr int kRbTile = kRbBlock * kRbItems;
constexpr int64_t kRsBigKeys = 1 << 20;

// Tile of a work-group: work-group b runs on XCD b % 8, which takes the
// b % 8-th eighth of the tiles in order (the grid is padded to a multiple of
// 8; tiles past the end are skipped).
__device__ __forceinline__ int64_t xcd_tile(int64_t ntiles) {
    const int64_t per = (ntiles + 7) >> 3;
    const int64_t t = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    return (blockIdx.x >> 3) < per ? t : ntiles;
}

// What a pass reads: sorted pairs, or (the first pass of a COO build) the
// edge list itself, its keys made on the fly.  digit(): what the count needs
// of element i; get(): its key and payload.
struct PairSrc {
    const uint64_t* keys;
    const uint32_t* vals;
    __device__ __forceinline__ uint64_t digit(int64_t i) const { return keys[i]; }
    using Raw = uint64_t;
    __device__ __forceinline__ Raw load(int64_t i) const { return keys[i]; }
    __device__ __forceinline__ uint64_t key(Raw r, int32_t*) const { return r; }
    __device__ __forceinline__ void report(int32_t) const {}
    __device__ __forceinline__ uint32_t pay(int64_t i) const { return vals[i]; }
    __device__ __forceinline__ bool has_pay() const { return vals != nullptr; }
};

// IT: int32_t, or int64_t ids taken modulo 2^32 as a cast to int32 takes them.
template <typename IT>
struct CooSrc {
    CooEdges e;
    struct Raw {
        int32_t r, c;
    };
    __device__ __forceinline__ Raw load(int64_t i) const {
        return Raw{(int32_t) static_cast<const IT*>(e.rows)[i], (int32_t) static_cast<const IT*>(e.cols)[i]};
    }
    // a bad id counts as id 0, here as in digit()
    __device__ __forceinline__ int64_t row(int32_t r, int32_t* bad) const {
        if (r >= 0 && r < e.num_rows) return r;
        *bad |= kErrEdgeRow;
        return 0;
    }
    __device__ __forceinline__ int64_t col(int32_t c, int32_t* bad) const {
        if (c >= 0 && c < e.num_cols) return c;
        *bad |= kErrEdgeCol;
        return 0;
    }
    // the low bits of the key: the window
    __device__ __forceinline__ uint64_t digit(int64_t i) const {
        int32_t bad = 0;
        return (uint64_t)((e.transpose ? col((int32_t) static_cast<const IT*>(e.cols)[i], &bad)
                                       : row((int32_t) static_cast<const IT*>(e.rows)[i], &bad)) >>
                          4);
    }
    __device__ __forceinline__ uint64_t key(Raw q, int32_t* bad) const {
        const int64_t r = row(q.r, bad), c = col(q.c, bad);
        return e.transpose ? window_key(c, r, e.wbits) : window_key(r, c, e.wbits);
    }
    __device__ __forceinline__ void report(int32_t bad) const {
        if (bad) atomicOr(e.err, bad);
    }
    __device__ __forceinline__ uint32_t pay(int64_t i) const {
        return e.vals ? __float_as_uint(e.vals[i]) : 0x3f800000u;  // 1.0f when no values are given
    }
    __device__ __forceinline__ bool has_pay() const { return true; }
};

template <typename Src>
__global__ __launch_bounds__(kRbBlock) void radix_hist_big_kernel(Src src, int64_t n, int shift, int64_t ntiles,
                                                                  int32_t* __restrict__ counts) {
    __shared__ int32_t h[kRbWaves][256];
    const int64_t t = xcd_tile(ntiles);
    if (t >= ntiles) return;  // uniform over the work-group
    const int tid = threadIdx.x, wave = tid / kWave;
    for (int x = tid; x < kRbWaves * 256; x += kRbBlock) (&h[0][0])[x] = 0;
    __syncthreads();
    const int64_t base = t * kRbTile;
    uint64_t k[kRbItems];
#pragma unroll
    for (int it = 0; it < kRbItems; ++it) {
        const int64_t i = base + it * kRbBlock + tid;
        k[it] = i < n ? src.digit(i) : 0;
    }
#pragma unroll
    for (int it = 0; it < kRbItems; ++it)
        if (base + it * kRbBlock + tid < n) atomicAdd(&h[wave][(uint32_t)(k[it] >> shift) & 255u], 1);
    __syncthreads();
    if (tid < 256) {
        int32_t c = 0;
#pragma unroll
        for (int w = 0; w < kRbWaves; ++w) c += h[w][tid];
        counts[(int64_t)tid * ntiles + t] = c;
    }
}

template <typename Src>
__global__ __launch_bounds__(kRbBlock) void radix_scatter_big_kernel(Src src, int64_t n, int shift, int64_t ntiles,
                                                                     const int64_t* __restrict__ offsets,
                                                                     uint64_t* __restrict__ kout,
                                                                     uint32_t* __restrict__ vout) {
    __shared__ uint64_t stage[kRbTile];        // keys, then payloads, in digit order
    __shared__ int32_t wcnt[kRbWaves][256];    // the wave's count, then its first place in the tile
    __shared__ int32_t part[4];
    __shared__ uint32_t gdelta[256];           // output position - place in the tile, per digit (mod 2^32)
    const int64_t t = xcd_tile(ntiles);
    if (t >= ntiles) return;  // uniform over the work-group
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid & (kWave - 1);
    for (int x = tid; x < kRbWaves * 256; x += kRbBlock) (&wcnt[0][0])[x] = 0;
    const int64_t base = t * kRbTile + wave * (kRbItems * kWave) + lane;
    uint64_t k[kRbItems];
    uint32_t v[kRbItems];
    uint32_t place[kRbItems];
    typename Src::Raw raw[kRbItems] = {};
#pragma unroll
    for (int it = 0; it < kRbItems; ++it) {  // every load issued before the first is used
        const int64_t i = base + it * kWave;
        if (i < n) raw[it] = src.load(i);
    }
    if (src.has_pay()) {
#pragma unroll
        for (int it = 0; it < kRbItems; ++it) {
            const int64_t i = base + it * kWave;
            v[it] = i < n ? src.pay(i) : 0;
        }
    }
    int32_t bad = 0;
#pragma unroll
    for (int it = 0; it < kRbItems; ++it) k[it] = base + it * kWave < n ? src.key(raw[it], &bad) : 0;
    src.report(bad);
    __syncthreads();
    // rank among the wave's keys of the same digit, in index order
    volatile int32_t* mine = wcnt[wave];
#pragma unroll
    for (int it = 0; it < kRbItems; ++it) {
        const bool valid = base + it * kWave < n;
        const uint32_t d = (uint32_t)(k[it] >> shift) & 255u;
        const uint64_t m = match_digit(d, valid);
        const int32_t before = mine[d];
        const int32_t rank = __popcll(m & lanemask_lt());
        place[it] = (uint32_t)(before + rank);
        if (valid && rank == 0) mine[d] = before + __popcll(m);
    }
    __syncthreads();
    // a digit's first place in the tile: exclusive scan over (digit, wave)
    int32_t tot = 0, incl = 0;
    if (tid < 256) {
#pragma unroll
        for (int w = 0; w < kRbWaves; ++w) tot += wcnt[w][tid];
        incl = tot;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int32_t o = __shfl_up(incl, d, kWave);
            if (lane >= d) incl += o;
        }
        if (lane == kWave - 1) part[wave] = incl;
    }
    __syncthreads();
    if (tid < 256) {
        int32_t run = incl - tot;
        for (int w = 0; w < wave; ++w) run += part[w];
        gdelta[tid] = (uint32_t)offsets[(int64_t)tid * ntiles + t] - (uint32_t)run;
#pragma unroll
        for (int w = 0; w < kRbWaves; ++w) {
            const int32_t c = wcnt[w][tid];
            wcnt[w][tid] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kRbItems; ++it) {
        if (base + it * kWave < n) {
            place[it] += (uint32_t)wcnt[wave][(uint32_t)(k[it] >> shift) & 255u];
            stage[place[it]] = k[it];
        }
    }
    __syncthreads();
    const int64_t left = n - t * kRbTile;
    const int cnt = left < kRbTile ? (int)left : kRbTile;
    uint32_t pos[kRbItems];
#pragma unroll
    for (int it = 0; it < kRbItems; ++it) {
        const int j = it * kRbBlock + tid;
        if (j < cnt) {
            const uint64_t key = stage[j];
            pos[it] = gdelta[(uint32_t)(key >> shift) & 255u] + (uint32_t)j;
            kout[pos[it]] = key;
        }
    }
    if (!src.has_pay()) return;  // uniform
    __syncthreads();
    uint32_t* pstage = reinterpret_cast<uint32_t*>(stage);
#pragma unroll
    for (int it = 0; it < kRbItems; ++it)
        if (base + it * kWave < n) pstage[place[it]] = v[it];
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kRbItems; ++it) {
        const int j = it * kRbBlock + tid;
        if (j < cnt) vout[pos[it]] = pstage[j];
    }
}

}  // namespace

// Sized for any sort of at most n keys (callers size by a capacity and sort
// what a batch holds): up to 256k keys a sort uses at most 64 tiles (at most
// ceil(n / 256) of them), above it ceil(n / 4096).
size_t radix_sort_workspace_bytes(int64_t n) {
    const int64_t small = (n + kRsBlock - 1) / kRsBlock;
    const int64_t big = (n + (int64_t)kRsBlock * kRsMaxIters - 1) / ((int64_t)kRsBlock * kRsMaxIters);
    const int64_t ntiles = std::max(std::min<int64_t>(small, 64), big);
    Sizer s;
    s.take<int32_t>((size_t)(256 * ntiles + 1));
    s.take<int64_t>((size_t)(256 * ntiles + 2));
    s.used += scan_workspace_bytes(256 * ntiles) + 256;
    return s.used;
}

static int sort_passes(const CooEdges* coo, uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt,
                       int64_t n, int bits, void* ws, size_t ws_bytes, hipStream_t stream, bool* result_in_alt) {
    *result_in_alt = false;
    if (n <= 1 || bits <= 0) return GRWS_OK;
    if (bits > 64) bits = 64;
    const int iters = radix_iters(n);
    // the large tiles keep output positions in 32 bits
    const bool big = n >= kRsBigKeys && n <= (int64_t)UINT32_MAX;
    const int64_t tile = big ? kRbTile : (int64_t)kRsBlock * iters;
    const int64_t ntiles = (n + tile - 1) / tile;
    if (ntiles > INT32_MAX / 2) return set_error(GRWS_E_INVALID, "radix sort: %lld keys is too many", (long long)n);
    Carver cv(ws, ws_bytes);
    int32_t* counts = cv.take<int32_t>(256 * ntiles + 1);
    int64_t* offsets = cv.take<int64_t>(256 * ntiles + 2);
    const size_t scan_bytes = scan_workspace_bytes(256 * ntiles);
    char* scan_ws = cv.take<char>(scan_bytes);
    if (!cv.ok) return set_error(GRWS_E_CAPACITY, "radix sort: workspace too small (%zu < %zu)", ws_bytes, cv.used);
    uint64_t* ka = keys;
    uint32_t* va = vals;
    uint64_t* kb = keys_alt;
    uint32_t* vb = vals_alt;
    bool alt = false;
    for (int shift = 0; shift < bits; shift += 8) {
        const unsigned bgrid = (unsigned)((ntiles + 7) / 8 * 8);
        const PairSrc pairs{ka, va};
        const bool first = coo != nullptr && shift == 0;
        if (first && coo->ids64)
            hipLaunchKernelGGL(radix_hist_big_kernel<CooSrc<int64_t>>, dim3(bgrid), dim3(kRbBlock), 0, stream,
                               CooSrc<int64_t>{*coo}, n, shift, ntiles, counts);
        else if (first)
            hipLaunchKernelGGL(radix_hist_big_kernel<CooSrc<int32_t>>, dim3(bgrid), dim3(kRbBlock), 0, stream,
                               CooSrc<int32_t>{*coo}, n, shift, ntiles, counts);
        else if (big)
            hipLaunchKernelGGL(radix_hist_big_kernel<PairSrc>, dim3(bgrid), dim3(kRbBlock), 0, stream, pairs, n,
                               shift, ntiles, counts);
        else
            hipLaunchKernelGGL(radix_hist_kernel, dim3((unsigned)ntiles), dim3(kRsBlock), 0, stream, ka, n, shift,
                               ntiles, iters, counts);
        GRWS_LAUNCH_CHECK();
        GRWS_TRY(scan_i32_to_i64(counts, offsets, 256 * ntiles, false, scan_ws, scan_bytes, stream));
        if (first && coo->ids64)
            hipLaunchKernelGGL(radix_scatter_big_kernel<CooSrc<int64_t>>, dim3(bgrid), dim3(kRbBlock), 0, stream,
                               CooSrc<int64_t>{*coo}, n, shift, ntiles, offsets, kb, vb);
        else if (first)
            hipLaunchKernelGGL(radix_scatter_big_kernel<CooSrc<int32_t>>, dim3(bgrid), dim3(kRbBlock), 0, stream,
                               CooSrc<int32_t>{*coo}, n, shift, ntiles, offsets, kb, vb);
        else if (big)
            hipLaunchKernelGGL(radix_scatter_big_kernel<PairSrc>, dim3(bgrid), dim3(kRbBlock), 0, stream, pairs, n,
                               shift, ntiles, offsets, kb, vb);
        else
            hipLaunchKernelGGL(radix_scatter_kernel, dim3((unsigned)ntiles), dim3(kRsBlock), 0, stream, ka, va, n,
                               shift, ntiles, iters, offsets, kb, vb);
        GRWS_LAUNCH_CHECK();
        std::swap(ka, kb);
        std::swap(va, vb);
        alt = !alt;
    }
    *result_in_alt = alt;
    return GRWS_OK;
}

int radix_sort_pairs(uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt, int64_t n, int bits,
                     void* ws, size_t ws_bytes, hipStream_t stream, bool* result_in_alt) {
    return sort_passes(nullptr, keys, vals, keys_alt, vals_alt, n, bits, ws, ws_bytes, stream, result_in_alt);
}

bool radix_sorts_edges(int64_t n) { return n >= kRsBigKeys && n <= (int64_t)UINT32_MAX; }

int radix_sort_edges(const CooEdges& coo, uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt,
                     int64_t n, int bits, void* ws, size_t ws_bytes, hipStream_t stream, bool* result_in_alt) {
    return sort_passes(&coo, keys, vals, keys_alt, vals_alt, n, bits, ws, ws_bytes, stream, result_in_alt);
}

}  // namespace grws
