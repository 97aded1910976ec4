// Flat-tile x sweeps: what the stress and the velocity sweep share.
//
// A block owns a (z, y) column tile of an x chunk and walks x one plane at a
// time, one point of the plane per thread.  A tile is `cols` points along z
// by `rows` along y, its threads numbered point by point and row by row, so
// both take any value with cols * rows <= 512: the y extent is split evenly,
// and z into 64-point tiles that start on a 128-byte line, the last one
// taking up to 8 points more rather than leaving a sliver.
//
// Fields differentiated along x live in per-thread register queues (the x
// loop is unrolled over the queue length, so the queues rotate by name);
// fields differentiated along y or z are staged one x plane at a time in LDS
// with their halos, double buffered, the next plane's loads in flight while
// the current one computes.
//
// Every global access is a 64-bit scalar base (one per field, set once per
// block) plus a 32-bit byte offset per thread that all fields share and that
// advances by one plane: per plane the addresses cost three adds.
#pragma once

#include "common.h"

#include <algorithm>
#include <atomic>
#include <utility>

namespace opesci {

constexpr int SWEEP_THREADS = 512;   // threads of a block at most
constexpr int SWEEP_ROWS = 16;       // rows of a tile at most
constexpr int SWEEP_COLS = 64;       // z points of a tile ...
constexpr int SWEEP_LAST = 72;       // ... and of the last one at most

// LDS plane size: the largest (rows + 2M) x (cols + 2M) over the tiles above,
// at 64 or 72 columns
template <int M>
struct SweepPlane {
    static constexpr int A = (SWEEP_THREADS / SWEEP_COLS + 2 * M) * (SWEEP_COLS + 2 * M);
    static constexpr int B = (SWEEP_THREADS / (SWEEP_COLS + 1) + 2 * M) * (SWEEP_LAST + 2 * M);
    static constexpr int SIZE = A > B ? A : B;
};

// XCD-aware block remap: hardware dispatches linear block b to XCD b % 8.
// Give XCD k the logical tiles [k*per, (k+1)*per) so one XCD's blocks are
// spatial neighbours.  Returns -1 for padding blocks.
__device__ __forceinline__ int sweep_block(int nblocks) {
    const int b = blockIdx.x;
    const int per = (nblocks + 7) / 8;
    const int l = (b % 8) * per + b / 8;
    return l < nblocks ? l : -1;
}

// element at byte offset `off` of a scalar base, ordinary or non-temporal
template <typename S>
__device__ __forceinline__ const S* at_byte(const S* base, uint32_t off) {
    return reinterpret_cast<const S*>(reinterpret_cast<const char*>(base) + (uint64_t)off);
}
template <typename S>
__device__ __forceinline__ S* at_byte(S* base, uint32_t off) {
    return reinterpret_cast<S*>(reinterpret_cast<char*>(base) + (uint64_t)off);
}

// One block's tile and this thread's place in it.  Offsets are elements of
// a plane (x = 0); `own` is in bounds for every thread, the halo ones for
// the threads that have an item.
struct SweepLane {
    int xb, xe;          // x range
    bool on;             // the thread owns a point of the tile
    int z, y;            // that point
    uint32_t own;        // its element offset
    int pitch;           // LDS row pitch
    int me;              // its place in an LDS plane
    bool hy, hz, hx;     // has a y-halo / z-halo / second y-halo item
    int ly, lz, lx;      // their places in an LDS plane
    uint32_t gy, gz, gx; // their element offsets
    bool low, high;      // the tile holds the first / last interior z
    int y0, rows;        // the tile's rows
};
// whether a tile can have more y-halo points than the block has threads
// (order 8 with more than 64 columns): a second item for the first threads
template <int M>
constexpr bool sweep_second_halo() {
    return 2 * M * SWEEP_LAST > SWEEP_THREADS;
}

// Tile of logical block l of a box list.  The box is picked with constant
// indices (the list stays in kernel arguments).
template <int M>
__device__ __forceinline__ SweepLane sweep_lane(const Geom& g, const Boxes& B, int l, const SweepTile& T) {
    int first = B.first[0], x0 = B.x0[0], x1 = B.x1[0], by0 = B.y0[0], by1 = B.y1[0], tyn = B.tyn[0], xc = B.xc[0];
#pragma unroll
    for (int i = 1; i < 4; ++i)
        if (i < B.n && l >= B.first[i]) {
            first = B.first[i];
            x0 = B.x0[i];
            x1 = B.x1[i];
            by0 = B.y0[i];
            by1 = B.y1[i];
            tyn = B.tyn[i];
            xc = B.xc[i];
        }
    const int loc = l - first;
    const int bz = loc % T.ntz, by = (loc / T.ntz) % tyn, bx = loc / (T.ntz * tyn);
    SweepLane s;
    s.xb = x0 + bx * xc;
    s.xe = min(s.xb + xc, x1);
    const int z0 = M + bz * SWEEP_COLS, y0 = by0 + by * T.rows;
    const int cols = bz == T.ntz - 1 ? g.nz - M - z0 : SWEEP_COLS, rows = min(T.rows, by1 - y0);
    const int t = threadIdx.x;
    int r = t / cols, c = t - r * cols;
    s.on = r < rows;
    // halo items: M rows above and below (the tile's columns), M points left
    // and right (the tile's rows); corners are never read.  y items from the
    // first thread up, z items from the last thread down.
    s.pitch = cols + 2 * M;
    s.hy = r < 2 * M;
    const int lr = r < M ? r : r + rows;
    s.ly = lr * s.pitch + M + c;
    s.gy = (uint32_t)((y0 - M + lr) * (int)g.sy + z0 + c);
    const int q = (int)blockDim.x - 1 - t, hr = q / (2 * M), hc = q - hr * 2 * M;
    s.hz = hr < rows;
    const int u = hc < M ? hc - M : cols + hc - M;
    s.lz = (hr + M) * s.pitch + M + u;
    s.gz = (uint32_t)((y0 + hr) * (int)g.sy + z0 + u);
    s.hx = false;
    s.lx = 0;
    s.gx = 0;
    if constexpr (sweep_second_halo<M>()) {
        const int t2 = t + (int)blockDim.x, r2 = t2 / cols, c2 = t2 - r2 * cols;
        s.hx = r2 < 2 * M;
        const int lr2 = r2 < M ? r2 : r2 + rows;
        s.lx = lr2 * s.pitch + M + c2;
        s.gx = (uint32_t)((y0 - M + lr2) * (int)g.sy + z0 + c2);
    }
    s.low = bz == 0;
    s.high = bz == T.ntz - 1;
    s.y0 = y0;
    s.rows = rows;
    if (!s.on) r = c = 0;
    s.z = z0 + c;
    s.y = y0 + r;
    s.own = (uint32_t)(s.y * (int)g.sy + s.z);
    s.me = (r + M) * s.pitch + M + c;
    return s;
}

// x loop unrolled over the U phases of the register queues: step(phase, x)
// for every plane of [xb, xe)
template <int I>
struct Phase {
    static constexpr int value = I;
};
template <typename F, int... I>
__device__ __forceinline__ void sweep_planes(int xb, int xe, F&& step, std::integer_sequence<int, I...>) {
    int x = xb;
    bool more = x < xe;
    while (more) {
        ((more ? (step(Phase<I>{}, x), more = ++x < xe) : false), ...);
    }
}

// every wave's LDS writes before every wave's LDS reads; global loads in
// flight stay in flight
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ------------------------------------------------------------------ launch shape (host)
// Tile and x chunk of one launch.  z: 64-point tiles, the last of 9 to 72; y:
// as few tiles as fill the block's threads (cfg.tile_y caps the rows), split
// evenly; x: the chunk that minimises the modelled time below (cfg.x_chunk
// when given).
struct SweepShape {
    SweepTile tile;
    Boxes boxes;
    int threads = 0, nb = 0;
};

// Modelled time in microseconds of a launch of nb blocks that walk `planes`
// planes each, at most `per_cu` of them side by side on a CU.  With n blocks
// on a CU a plane takes at least lat + step * (0.6 + 0.4 n): `lat` is the
// part of the loads' round trip that misses the caches, `step` the plane's
// own chain (staging, barrier, LDS, arithmetic), of which more blocks hide
// each other's waits but not their issue.  Once they share the memory path
// it takes bw per block.  Blocks that do not fill every CU alike leave the
// memory path idle at the end: half of the missing blocks count.
struct SweepModel {
    int per_cu;
    double lat, step, bw;
    double time(long long nb, double planes) const {
        const int cus = 256;
        const long long slots = (long long)per_cu * cus;
        const long long full = nb / slots, rest = nb % slots;
        double t = (double)full * std::max(lat + step * (0.6 + 0.4 * per_cu), bw * slots);
        if (rest > 0) {
            const long long n = (rest + cus - 1) / cus;
            t += std::max(lat + step * (0.6 + 0.4 * n), bw * 0.5 * (double)(rest + n * cus));
        }
        return t * planes;
    }
};

// Blocks of `threads` threads of a kernel that fit a CU (one query per kernel
// and block size).
template <typename K>
int sweep_blocks_per_cu(K kernel, std::atomic<int>* cache, int threads) {
    std::atomic<int>& c = cache[threads / 64];
    int n = c.load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) != hipSuccess || n < 1) n = 1;
        c.store(n, std::memory_order_relaxed);
    }
    return n;
}

// `bytes`: per point and plane; `blocks_per_cu(threads)`: of the kernel;
// `row_items`: values a tile that holds a z face stages per row and face, one
// per thread.
template <int M, typename F>
SweepShape sweep_shape(const Geom& g, const InteriorLaunch& cfg, const Boxes* boxes, int bytes, int elem,
                       F&& blocks_per_cu, int row_items = 0) {
    SweepShape s;
    const int nzi = g.nz - 2 * M;
    s.tile.ntz = std::max(1, (nzi - (SWEEP_LAST - SWEEP_COLS) + SWEEP_COLS - 1) / SWEEP_COLS);
    const int last = nzi - (s.tile.ntz - 1) * SWEEP_COLS, cols = std::max(last, s.tile.ntz > 1 ? SWEEP_COLS : 0);
    Boxes& B = s.boxes;
    if (boxes) {
        B = *boxes;
    } else {
        B.n = 1;
        B.x0[0] = M;
        B.x1[0] = g.nx - M;
        B.y0[0] = M;
        B.y1[0] = g.ny - M;
    }
    int ny = 1;
    for (int i = 0; i < B.n; ++i) ny = std::max(ny, B.y1[i] - B.y0[i]);
    const int cap = std::min(SWEEP_ROWS, SWEEP_THREADS / cols);
    const int most_rows = std::min(ny, cfg.tile_y > 0 ? std::min(cap, cfg.tile_y) : cap);
    const int tiles = (ny + most_rows - 1) / most_rows;
    s.tile.rows = (ny + tiles - 1) / tiles;
    const int items = row_items * (s.tile.ntz == 1 ? 2 : 1) * s.tile.rows;
    const int need = std::max(std::max(cols * s.tile.rows, items), std::max(2 * M * cols, 2 * M * s.tile.rows));
    s.threads = std::min(SWEEP_THREADS, (need + 63) / 64 * 64);
    long long columns = 0;
    int nx = 1;
    for (int i = 0; i < B.n; ++i) {
        B.tyn[i] = std::max(0, (B.y1[i] - B.y0[i] + s.tile.rows - 1) / s.tile.rows);
        columns += (long long)s.tile.ntz * B.tyn[i];
        nx = std::max(nx, B.x1[i] - B.x0[i]);
    }
    // offsets within a chunk are 32-bit bytes (media arrays up to 8 per point)
    const long long plane = (long long)g.sx * 8;
    const int most = (int)std::min<long long>(nx, std::max<long long>(1, (1LL << 32) / plane - 2 * MAXM - 2));
    int xc = cfg.x_chunk;
    if (xc <= 0) {
        // constants fitted to chunks of 1 to 256 planes timed on 16^3 .. 256^3
        // grids, orders 2 to 8, every storage type
        SweepModel model;
        model.per_cu = blocks_per_cu(s.threads);
        model.lat = (double)g.nx * g.sx * elem * 18 > 256e6 ? 0.6 : 0.0;
        model.step = (0.45 + 0.18 * M) * (elem == 4 ? 1.0 : 1.6);
        model.bw = (double)cols * s.tile.rows * bytes / 5.0e6;
        double best = -1.0;
        for (int n = 1; n <= nx; n = n < 16 ? n + 1 : n + n / 8) {
            const int c = (nx + n - 1) / n;
            const double t = model.time(columns * ((nx + c - 1) / c), c + 1.2 + 0.15 * (2 * M - 1));
            if (best < 0.0 || t < best) {
                best = t;
                xc = c;
            }
        }
    }
    xc = std::max(1, std::min(xc, most));
    B.first[0] = 0;
    for (int i = 0; i < B.n; ++i) {
        const int xl = std::max(0, B.x1[i] - B.x0[i]);
        B.xc[i] = std::max(1, std::min(xc, xl));
        const int tx = xl > 0 ? (xl + B.xc[i] - 1) / B.xc[i] : 0;
        B.first[i + 1] = B.first[i] + s.tile.ntz * B.tyn[i] * tx;
    }
    s.nb = B.first[B.n];
    return s;
}

}  // namespace opesci
