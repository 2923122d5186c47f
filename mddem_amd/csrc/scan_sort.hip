// Device-wide exclusive scan and the placing pass of the stable counting sort
// (cell binning).
//
// The sort reproduces the order of the reference's binning
// (crates/mddem_core/src/neighbor.rs:857-889): within a cell, elements stay
// in index order. The kernel that writes the keys counts them per cell, the
// counts are scanned, elements are placed in their cell with atomics (one per
// run of equal keys inside a wavefront, since the input is mostly sorted
// already), and the kernel that uses the order ranks each element by index
// inside its cell (cell_rank), so the result is deterministic.
#include "cells.hpp"

namespace mdd {

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, int64_t n) {
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}
__global__ void k_fill_f64(double* __restrict__ p, double v, int64_t n) {
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}
__global__ void k_fill_f32(float* __restrict__ p, float v, int64_t n) {
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}

// inclusive scan across one 64-lane wavefront
__device__ inline uint32_t wave_incl_scan(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

// exclusive scan across a 256-thread block; returns the block total in *total
__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t* lds4, uint32_t* total) {
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    uint32_t inc = wave_incl_scan(v);
    if (lane == 63) lds4[w] = inc;
    __syncthreads();
    uint32_t off = 0;
    for (int k = 0; k < w; k++) off += lds4[k];
    uint32_t tot = lds4[0] + lds4[1] + lds4[2] + lds4[3];
    __syncthreads();
    *total = tot;
    return off + inc - v;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_reduce(const uint32_t* __restrict__ in,
                                                              int64_t n, uint32_t* sums) {
    __shared__ uint32_t lds4[4];
    const int64_t base = int64_t(blockIdx.x) * kScanTile + int64_t(threadIdx.x) * kScanItems;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        int64_t i = base + k;
        if (i < n) s += in[i];
    }
    uint32_t tot;
    block_excl_scan(s, lds4, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Second pass: each block first sums the block totals before it (a few
// thousand at most, read from L2), so no separate scan of the totals runs.
// add/out2: out2[i] = out[i] + add[i] as well (bin starts: particles plus
// images of each cell).
__global__ void __launch_bounds__(kScanThreads) k_scan_apply(const uint32_t* __restrict__ in,
                                                             uint32_t* __restrict__ out,
                                                             int64_t n,
                                                             const uint32_t* __restrict__ sums,
                                                             int64_t nb,
                                                             const uint32_t* __restrict__ add,
                                                             uint32_t* __restrict__ out2) {
    __shared__ uint32_t lds4[4];
    uint32_t before = 0;
    for (int64_t j = threadIdx.x; j < int64_t(blockIdx.x); j += kScanThreads) before += sums[j];
    uint32_t off, prior;
    block_excl_scan(before, lds4, &prior);
    off = prior;
    const int64_t base = int64_t(blockIdx.x) * kScanTile + int64_t(threadIdx.x) * kScanItems;
    uint32_t v[kScanItems];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        int64_t i = base + k;
        v[k] = i < n ? in[i] : 0u;
        s += v[k];
    }
    uint32_t tot;
    uint32_t run = block_excl_scan(s, lds4, &tot) + off;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        int64_t i = base + k;
        if (i < n) {
            out[i] = run;
            if (out2) out2[i] = run + add[i];
        }
        run += v[k];
    }
    if (blockIdx.x == nb - 1 && threadIdx.x == 0) {
        out[n] = off + tot;
        if (out2) out2[n] = off + tot + add[n];
    }
}

// The same in one launch, for up to kDirectScan elements: a block scans
// kDirectTile of them, four per thread, and gets the sum of those before its
// tile by adding them up itself (at most 512 KB, from L2): 4.7 us for the
// 24,400 cells of 256,000 LJ atoms and 5.3 us for 42,900 (one workgroup tile
// after tile: 9.2 and 16.7; word by word: 6.5 and 7.1), 3.0 us for 1,300.
// Beyond, two launches cost less than the sums.
constexpr int kDirectThreads = 1024;
constexpr int kDirectTile = kDirectThreads * 4;
constexpr int64_t kDirectScan = int64_t(1) << 17;

__global__ void __launch_bounds__(kDirectThreads) k_scan_direct(const uint32_t* __restrict__ in,
                                                                uint32_t* __restrict__ out,
                                                                int64_t n,
                                                                const uint32_t* __restrict__ add,
                                                                uint32_t* __restrict__ out2) {
    __shared__ uint32_t pre[kDirectThreads / 64], wsum[kDirectThreads / 64];
    const int tid = int(threadIdx.x), lane = tid & 63, w = tid >> 6;
    const int64_t i0 = int64_t(blockIdx.x) * kDirectTile + int64_t(tid) * 4;
    // (the tiles before this one are full)
    uint32_t before = 0u;
    const uint4* in4 = reinterpret_cast<const uint4*>(in);
#pragma unroll 8
    for (int j = 0; j < int(blockIdx.x); j++) {
        const uint4 q = in4[j * kDirectThreads + tid];
        before += (q.x + q.y) + (q.z + q.w);
    }
    // (four words at a time but for the end of the array)
    const bool whole = i0 + 4 <= n;
    uint32_t v[4] = {0u, 0u, 0u, 0u}, ad[4] = {0u, 0u, 0u, 0u};
    auto load4 = [&](const uint32_t* p, uint32_t* x) {
        if (whole) {
            const uint4 q = *reinterpret_cast<const uint4*>(p + i0);
            x[0] = q.x;
            x[1] = q.y;
            x[2] = q.z;
            x[3] = q.w;
        } else {
            for (int k = 0; k < 4; k++) x[k] = i0 + k < n ? p[i0 + k] : 0u;
        }
    };
    load4(in, v);
    if (out2) load4(add, ad);
    const uint32_t s = (v[0] + v[1]) + (v[2] + v[3]);
    const uint32_t inc = wave_incl_scan(s);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    if (lane == 63) {
        pre[w] = before;
        wsum[w] = inc;
    }
    __syncthreads();
    uint32_t run = inc - s, end = 0u;
#pragma unroll
    for (int k = 0; k < kDirectThreads / 64; k++) {
        run += pre[k] + (k < w ? wsum[k] : 0u);
        end += pre[k] + wsum[k];
    }
    uint32_t r[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        r[k] = run;
        run += v[k];
    }
    if (whole) {
        *reinterpret_cast<uint4*>(out + i0) = make_uint4(r[0], r[1], r[2], r[3]);
        if (out2)
            *reinterpret_cast<uint4*>(out2 + i0) =
                make_uint4(r[0] + ad[0], r[1] + ad[1], r[2] + ad[2], r[3] + ad[3]);
    } else {
        for (int k = 0; k < 4; k++) {
            if (i0 + k < n) {
                out[i0 + k] = r[k];
                if (out2) out2[i0 + k] = r[k] + ad[k];
            }
        }
    }
    if (blockIdx.x == gridDim.x - 1 && tid == 0) {
        out[n] = end;
        if (out2) out2[n] = end + add[n];
    }
}

// Elements into their cells, in any order within a cell. n taken from n_dev
// when given (device-side element count). cnt holds the cells' counts and is
// counted down to zero, ready for the next sort.
__global__ void k_scatter(const uint32_t* __restrict__ key, int64_t n,
                          const uint32_t* __restrict__ n_dev,
                          const uint32_t* __restrict__ start, uint32_t* cnt,
                          uint32_t* __restrict__ placed) {
    const int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
    const int64_t nn = n_dev ? int64_t(*n_dev) : n;
    const bool valid = i < nn;
    const uint32_t k = valid ? key[i] : 0u;
    int h, t;
    wave_runs(k, valid, h, t);
    const int lane = threadIdx.x & 63;
    uint32_t base = 0;
    if (valid && lane == t) {
        const uint32_t run = uint32_t(t - h + 1);
        base = start[k] + (atomicSub(&cnt[k], run) - run);
    }
    base = __shfl(base, t, 64);
    if (valid) placed[base + uint32_t(lane - h)] = uint32_t(i);
}

int fill_blocks(int64_t n) {
    int64_t b = (n + 255) / 256;
    if (b > 4096) b = 4096;
    return int(b > 0 ? b : 1);
}

}  // namespace

void fill_u32(Ctx& c, uint32_t* p, uint32_t v, int64_t n) {
    if (n <= 0) return;
    launch(c, k_fill_u32, fill_blocks(n), 256, p, v, n);
    MDD_HIP(hipGetLastError());
}
void fill_f64(Ctx& c, double* p, double v, int64_t n) {
    if (n <= 0) return;
    launch(c, k_fill_f64, fill_blocks(n), 256, p, v, n);
    MDD_HIP(hipGetLastError());
}
void fill_f32(Ctx& c, float* p, float v, int64_t n) {
    if (n <= 0) return;
    launch(c, k_fill_f32, fill_blocks(n), 256, p, v, n);
    MDD_HIP(hipGetLastError());
}

// out[0..n] = exclusive scan of in[0..n), out[n] = total; with add given,
// out2[i] = out[i] + add[i] for i <= n as well
void exclusive_scan(Ctx& c, const uint32_t* in, uint32_t* out, int64_t n, const uint32_t* add,
                    uint32_t* out2) {
    if (n <= kDirectScan) {
        const int64_t tiles = (n + kDirectTile - 1) / kDirectTile;
        launch(c, k_scan_direct, int(tiles > 0 ? tiles : 1), kDirectThreads, in, out, n, add, out2);
        MDD_HIP(hipGetLastError());
        return;
    }
    int64_t nb = (n + kScanTile - 1) / kScanTile;
    c.scan_tmp.resize(size_t(nb + 2));
    launch(c, k_scan_reduce, int(nb), kScanThreads, in, n, c.scan_tmp.p);
    launch(c, k_scan_apply, int(nb), kScanThreads, in, out, n,
           static_cast<const uint32_t*>(c.scan_tmp.p), nb, add, out2);
    MDD_HIP(hipGetLastError());
}

// The elements 0..n-1 (*n_dev of them when given) into their cells' places:
// start from exclusive_scan of cnt, the counts per key; cnt is zero afterwards
void place_by_key(Ctx& c, const uint32_t* key, int64_t n, const uint32_t* n_dev,
                  const uint32_t* start, uint32_t* cnt, uint32_t* placed) {
    if (n <= 0) return;
    launch(c, k_scatter, blocks_for(n, 256), 256, key, n, n_dev, start, cnt, placed);
    MDD_HIP(hipGetLastError());
}

}  // namespace mdd
