// Scans of small and medium inputs: a reduction of every tile, then a scan of every tile that adds up the totals
// of the tiles before it; up to one tile, the scan alone.
//
// The single-pass kernel (scan.hip) is made for throughput: tiles of 24,576 items leave most CUs idle below some
// millions of items, its states are cleared in a launch of their own, and a tile waits for others' publications
// (1,000,003 f32: 41 tiles, 14.9 us per call, of 4,194,304 u32 17.4; here 11.0 and 11.0, and 8.1 for 1,500 items, 11.3
// there).  Here the second launch takes the place of the clear, nothing polls, and the tiles fill the chip; the
// input's second reading comes from the caches.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace lcpp_hip {

constexpr int kSmallScanRows = 4;
// Items of a tile: BLOCK threads x 4 rows of 16 bytes.
template <typename T, int BLOCK>
constexpr uint32_t kSmallScanTile = static_cast<uint32_t>(BLOCK) * kSmallScanRows * (16 / sizeof(T));

// Row r, thread t: the t-th 16 bytes of the tile's r-th row.  Items past the end are the identity.
template <typename T, typename Op, int BLOCK>
__device__ __forceinline__ void load_small_tile(const T* in, uint64_t n, uint64_t base, bool vector_io,
                                                T (&v)[kSmallScanRows][16 / sizeof(T)]) {
    constexpr int V = 16 / sizeof(T);
    using Vec = T __attribute__((ext_vector_type(V)));
    if (vector_io && base + kSmallScanTile<T, BLOCK> <= n) {
        Vec x[kSmallScanRows];
#pragma unroll
        for (int r = 0; r < kSmallScanRows; ++r) x[r] = reinterpret_cast<const Vec*>(in + base)[r * BLOCK + threadIdx.x];
#pragma unroll
        for (int r = 0; r < kSmallScanRows; ++r)
#pragma unroll
            for (int j = 0; j < V; ++j) v[r][j] = x[r][j];
    } else {
#pragma unroll
        for (int r = 0; r < kSmallScanRows; ++r)
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const uint64_t i = base + (static_cast<uint64_t>(r) * BLOCK + threadIdx.x) * V + j;
                v[r][j] = i < n ? in[i] : Op::template identity<T>();
            }
    }
}

// totals[b] = the fold of tile b, in the order of the items.
template <typename T, typename Op, int BLOCK>
__global__ __launch_bounds__(BLOCK) void scan_small_totals_kernel(const T* __restrict__ in, uint64_t n, bool vector_io,
                                                                  T* __restrict__ totals) {
    constexpr int V = 16 / sizeof(T);
    constexpr int W = BLOCK / kWave;
    __shared__ T s_total[kSmallScanRows][W];
    const Op op{};
    T v[kSmallScanRows][V];
    load_small_tile<T, Op, BLOCK>(in, n, static_cast<uint64_t>(blockIdx.x) * kSmallScanTile<T, BLOCK>, vector_io, v);
#pragma unroll
    for (int r = 0; r < kSmallScanRows; ++r) {
#pragma unroll
        for (int j = 1; j < V; ++j) v[r][0] = op(v[r][0], v[r][j]);
        const T sum = wave_inclusive_scan(v[r][0], op);
        if (lane_id() == kWave - 1) s_total[r][threadIdx.x / kWave] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        T total = Op::template identity<T>();
        for (int r = 0; r < kSmallScanRows; ++r)
            for (int w = 0; w < W; ++w) total = op(total, s_total[r][w]);
        totals[blockIdx.x] = total;
    }
}

// Scans tile blockIdx.x behind op(init, the totals of the tiles before it).  In place when out is in.
template <typename T, bool INCLUSIVE, typename Op, int BLOCK>
__global__ __launch_bounds__(BLOCK) void scan_small_kernel(const T* in, T* out, uint64_t n, const T* totals, T init,
                                                           bool vector_io) {
    constexpr int V = 16 / sizeof(T);
    constexpr int W = BLOCK / kWave;
    using Vec = T __attribute__((ext_vector_type(V)));
    __shared__ T s_total[kSmallScanRows][W];
    __shared__ T s_before[W];
    const Op op{};
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = lane_id();
    const uint32_t wave = tid / kWave;
    const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kSmallScanTile<T, BLOCK>;
    T v[kSmallScanRows][V];
    load_small_tile<T, Op, BLOCK>(in, n, base, vector_io, v);
    // Each thread folds its share of the earlier tiles' totals, neighbouring ones, so that the order holds.
    T before = Op::template identity<T>();
    const uint32_t share = (blockIdx.x + BLOCK - 1) / BLOCK;
    for (uint32_t i = tid * share; i < (tid + 1) * share && i < blockIdx.x; ++i) before = op(before, totals[i]);
    before = wave_inclusive_scan(before, op);
    if (lane == kWave - 1) s_before[wave] = before;
    T incl[kSmallScanRows];
#pragma unroll
    for (int r = 0; r < kSmallScanRows; ++r) {
#pragma unroll
        for (int j = 1; j < V; ++j) v[r][j] = op(v[r][j - 1], v[r][j]);
        incl[r] = wave_inclusive_scan(v[r][V - 1], op);
        if (lane == kWave - 1) s_total[r][wave] = incl[r];
    }
    __syncthreads();
    T prefix = Op::template identity<T>();
#pragma unroll
    for (int w = 0; w < W; ++w) prefix = op(prefix, s_before[w]);
    T running = op(init, prefix);
    const bool full = vector_io && base + kSmallScanTile<T, BLOCK> <= n;
#pragma unroll
    for (int r = 0; r < kSmallScanRows; ++r) {
        T earlier = Op::template identity<T>(), row_total = Op::template identity<T>();
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const T x = s_total[r][w];
            if (w < static_cast<int>(wave)) earlier = op(earlier, x);
            row_total = op(row_total, x);
        }
        const T start = op(running, earlier);
        const T p = op(start, wave_shift_exclusive<T, Op>(incl[r]));
        Vec o;
        if constexpr (INCLUSIVE) {
#pragma unroll
            for (int j = 0; j < V - 1; ++j) o[j] = op(p, v[r][j]);
            o[V - 1] = op(start, incl[r]);
        } else {
            o[0] = p;
#pragma unroll
            for (int j = 1; j < V; ++j) o[j] = op(p, v[r][j - 1]);
        }
        running = op(running, row_total);
        if (full) {
            reinterpret_cast<Vec*>(out + base)[r * BLOCK + tid] = o;
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const uint64_t i = base + (static_cast<uint64_t>(r) * BLOCK + tid) * V + j;
                if (i < n) out[i] = o[j];
            }
        }
    }
}

// Tiles of the two-launch form: 8 M u32 take 19.4 us per call in one pass and 14.9 here, 12 M 21.4 and 24.6 (the second
// reading outgrows what the clear and the look-back cost); f64 at 2,441 tiles 20.6 and 21.3.
constexpr uint64_t kSmallScanTiles = 2048;
constexpr int kSmallScanBlock = 256, kOneTileScanBlock = 1024;

// Whether the input takes this route: one tile, or totals that fit the temp storage.
template <typename T>
bool scan_small_route(uint64_t n, size_t temp_bytes) {
    if (n <= kSmallScanTile<T, kOneTileScanBlock>) return true;
    const uint64_t tiles = ceil_div(n, kSmallScanTile<T, kSmallScanBlock>);
    return tiles <= kSmallScanTiles && temp_bytes >= tiles * sizeof(T);
}

template <typename T, typename Op, bool INCLUSIVE>
int scan_small(const char* name, T* totals, const T* in, T* out, uint64_t n, T init, bool vector_io, hipStream_t stream) {
    LaunchScope scope(name, stream);
    if (n <= kSmallScanTile<T, kSmallScanBlock>) {
        scan_small_kernel<T, INCLUSIVE, Op, kSmallScanBlock><<<1, kSmallScanBlock, 0, stream>>>(in, out, n, totals, init, vector_io);
    } else if (n <= kSmallScanTile<T, kOneTileScanBlock>) {
        scan_small_kernel<T, INCLUSIVE, Op, kOneTileScanBlock><<<1, kOneTileScanBlock, 0, stream>>>(in, out, n, totals, init, vector_io);
    } else {
        const unsigned tiles = static_cast<unsigned>(ceil_div(n, kSmallScanTile<T, kSmallScanBlock>));
        scan_small_totals_kernel<T, Op, kSmallScanBlock><<<tiles, kSmallScanBlock, 0, stream>>>(in, n, vector_io, totals);
        const int st = check_hip(hipGetLastError(), "scan launch");
        if (st != kOk) return st;
        scan_small_kernel<T, INCLUSIVE, Op, kSmallScanBlock><<<tiles, kSmallScanBlock, 0, stream>>>(in, out, n, totals, init, vector_io);
    }
    return check_hip(hipGetLastError(), "scan launch");
}

}  // namespace lcpp_hip
