// Boundary program, analytic initial state, L2 norms, effective media,
// layout conversion and point source / receivers.
#include "bcdev.h"

#include <algorithm>
#include <mutex>

namespace opesci {

// real_t x = dx*(i - m [+ 0.5]) of the reference loops, rounded once to R
template <typename R>
__device__ __forceinline__ double coord_of(double dx, int i, int m, int stagger) {
    const R h = (R)dx;
    return (double)(R)((double)h * ((double)(i - m) + (stagger ? 0.5 : 0.0)));
}

// ------------------------------------------------------------------ boundary program
// One launch per hazard level, blockIdx.y = statement.  Statements of a
// level write disjoint cells and never read what another statement of the
// level writes.  Terms are loaded independently and summed in term order.
template <typename R, typename S>
__global__ __launch_bounds__(256) void bc_kernel(Geom g, FieldPtrs<S> F, const BcDesc* __restrict__ desc,
                                                 const R* __restrict__ pool, int first, int t0, int t1) {
    const BcDesc* D = desc + first + blockIdx.y;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= D->npts) return;
    const int n1 = D->n1;
    bc_point<R, S>(g, F, D, pool, p, D->lo0 + p / n1, D->lo1 + p % n1, t0, t1);
}

// One boundary launch of a step: a block takes the points its entry of the
// block list names, so pieces of any size share a launch without idle blocks.
// What bounds it on small grids and edges is the chain of dependent cache
// misses (the fields have passed through the caches since the last step):
// block entry, descriptor, values, store.  The descriptor comes to LDS in
// one load of the whole block, the field pointers next to it.  On large
// grids it is the z faces, where every value is a line of its own: a group
// touches a line once per plane it reads or writes.
template <typename R, typename S>
__device__ __forceinline__ void bc_piece(const Geom& g, S* const* field, const BcPieceDesc& D,
                                         const R* __restrict__ pool, int p0, int points) {
    using C = Conv<S, R>;
    int p = p0 + (int)threadIdx.x;
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    const int nt = uniform(D.nterms), axis = uniform(D.axis), n1 = uniform(D.n1), end = uniform(D.npts);
    const int64_t so0 = axis == 0 ? g.sy : g.sx, so1 = axis == 2 ? g.sy : 1;
    S* const to = field[uniform(D.fl)];
    auto place = [&](int q, int& pp) {
        const int i0 = D.lo0 + q / n1, i1 = D.lo1 + q % n1;
        pp = (i0 - D.plo0) * D.pn1 + (i1 - D.plo1);
        return (int64_t)i0 * so0 + (int64_t)i1 * so1 + D.disp;
    };
    if (nt <= 1) {
        // images and zeros, most points of all: several per thread
        const BcPieceTerm T = D.t[0];
        const S* from = field[T.fl] + T.disp;
        const R* coef = nt && uniform(T.cslot) >= 0 ? pool + D.cpool : nullptr;
        for (const int last = min(p0 + points, end); p < last; p += BC_FEW * BC_BLOCK) {
            R v[BC_FEW];
            int64_t dst[BC_FEW];
#pragma unroll
            for (int k = 0; k < BC_FEW; ++k) {
                const int q = p + k * BC_BLOCK;
                v[k] = (R)0;
                if (q < last) {
                    int pp;
                    dst[k] = place(q, pp);
                    if (nt) v[k] = fma(coef ? coef[pp] : (R)T.coef, C::ld(from + dst[k]), v[k]);
                }
            }
#pragma unroll
            for (int k = 0; k < BC_FEW; ++k)
                if (p + k * BC_BLOCK < last) C::st(to + dst[k], v[k]);
        }
        return;
    }
    if (p >= end) return;
    int pp;
    const int64_t dst = place(p, pp);
    // terms loaded independently, summed in term order
    R v[BC_MAXT], c[BC_MAXT];
#pragma unroll
    for (int k = 0; k < BC_MAXT; ++k)
        if (k < nt) {
            const BcPieceTerm T = D.t[k];
            c[k] = (R)T.coef;
            if (uniform(T.cslot) >= 0) c[k] = pool[D.cpool + (int64_t)T.cslot * D.pnpts + pp];
            v[k] = C::ld(field[T.fl] + dst + T.disp);
        }
    R acc = (R)0;
#pragma unroll
    for (int k = 0; k < BC_MAXT; ++k)
        if (k < nt) acc = fma(c[k], v[k], acc);
    C::st(to + dst, acc);
}

template <typename R, typename S, int T1>
__device__ __forceinline__ void bc_group(const Geom& g, S* const* field, const BcGroupDesc& D,
                                         const R* __restrict__ pool, int tile, R* slot) {
    using C = Conv<S, R>;
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    constexpr int T0 = BC_BLOCK / T1, W = T1 + 2, H = T0 + 2, P = (H * W + BC_BLOCK - 1) / BC_BLOCK;
    static_assert(H * W <= BC_TILE_ROWS, "tile");
    const int t = (int)threadIdx.x, axis = uniform(D.axis);
    const int n0 = axis == 0 ? g.ny : g.nx, n1 = axis == 2 ? g.ny : g.nz;
    const int64_t so0 = axis == 0 ? g.sy : g.sx, so1 = axis == 2 ? g.sy : 1;
    const int tiles1 = uniform(D.tiles1);
    const int a0 = uniform(D.lo0) + tile / tiles1 * T0, a1 = uniform(D.lo1) + tile % tiles1 * T1;
    const int e0 = min(a0 + T0, uniform(D.hi0)), e1 = min(a1 + T1, uniform(D.hi1));   // the tile's end
    const int ns = uniform(D.nslots), own = uniform(D.own_slot), nq = uniform(D.nstmts);
    const BcGroupStmt& N = D.s[0];
    // the first statement's box and the points of it the tile takes
    const int b0 = uniform(N.plo0), c0 = b0 + uniform(N.pn0), b1 = uniform(N.plo1), c1 = b1 + uniform(N.pn1);
    const int x0 = max(a0 + uniform(D.min0), b0), y0 = min(e0 + uniform(D.max0), c0),
              x1 = max(a1 + uniform(D.min1), b1), y1 = min(e1 + uniform(D.max1), c1);
    const S* from[BC_SLOTS];
#pragma unroll
    for (int k = 0; k < BC_SLOTS; ++k) from[k] = field[D.slot_fl[k]] + D.slot_disp[k];
    R v[P][BC_SLOTS];
    bool in[P];
#pragma unroll
    for (int r = 0; r < P; ++r) {
        const int i = t + r * BC_BLOCK, i0 = a0 - 1 + i / W, i1 = a1 - 1 + i % W;
        in[r] = i < H * W && i0 >= 0 && i0 < n0 && i0 <= e0 && i1 >= 0 && i1 < n1 && i1 <= e1;
        if (!in[r]) continue;
        const int64_t at = (int64_t)i0 * so0 + (int64_t)i1 * so1;
        const bool computed = i0 >= b0 && i0 < c0 && i1 >= b1 && i1 < c1;
#pragma unroll
        for (int k = 0; k < BC_SLOTS; ++k)
            if (k < ns && !(k == own && computed)) v[r][k] = C::ld(from[k] + at);
    }
#pragma unroll
    for (int r = 0; r < P; ++r)
        if (in[r])
#pragma unroll
            for (int k = 0; k < BC_SLOTS; ++k)
                if (k < ns) slot[k * BC_TILE_ROWS + t + r * BC_BLOCK] = v[r][k];
    __syncthreads();
    // sum of statement q's terms at the point (i0, i1), place i of the tile
    auto eval = [&](const BcGroupTerm* T, int q, int i0, int i1, int i) __attribute__((always_inline)) {
        const BcGroupStmt& s = D.s[q];
        const int nt = uniform(s.nterms);
        R c[BC_GTERMS], x[BC_GTERMS];
#pragma unroll
        for (int k = 0; k < BC_GTERMS; ++k) x[k] = slot[i + T[k].at];
#pragma unroll
        for (int k = 0; k < BC_GTERMS; ++k) c[k] = (R)T[k].coef;
        if (uniform(s.pooled)) {
            const int64_t pp = s.cpool + (int64_t)(i0 - s.plo0) * s.pn1 + (i1 - s.plo1);
            const int64_t npts = (int64_t)s.pn0 * s.pn1;
#pragma unroll
            for (int k = 0; k < BC_GTERMS; ++k)
                if (k < nt && uniform(T[k].cslot) >= 0) c[k] = pool[pp + T[k].cslot * npts];
        }
        R acc = (R)0;
#pragma unroll
        for (int k = 0; k < BC_GTERMS; ++k)
            if (k < nt) acc = fma(c[k], x[k], acc);
        return acc;
    };
    BcGroupTerm T[BC_GTERMS];
#pragma unroll
    for (int k = 0; k < BC_GTERMS; ++k) T[k] = D.t[0][k];
#pragma unroll
    for (int r = 0; r < P; ++r) {
        const int i = t + r * BC_BLOCK, i0 = a0 - 1 + i / W, i1 = a1 - 1 + i % W;
        if (i0 < x0 || i0 >= y0 || i1 < x1 || i1 >= y1) continue;
        const R v = stored<S, R>(eval(T, 0, i0, i1, i));
        slot[own * BC_TILE_ROWS + i] = v;
        if (i0 >= a0 && i0 < e0 && i1 >= a1 && i1 < e1)
            C::st(field[uniform(N.fl)] + (int64_t)i0 * so0 + (int64_t)i1 * so1 + N.disp, v);
    }
    __syncthreads();
    const int i0 = a0 + t / T1, i1 = a1 + t % T1, i = (t / T1 + 1) * W + t % T1 + 1;
    if (i0 >= e0 || i1 >= e1) return;
#pragma unroll
    for (int q = 1; q < BC_GROUP; ++q)
        if (q < nq) {
            const BcGroupStmt& s = D.s[q];
#pragma unroll
            for (int k = 0; k < BC_GTERMS; ++k) T[k] = D.t[q][k];
            if (i0 >= s.lo0 && i0 < s.hi0 && i1 >= s.lo1 && i1 < s.hi1)
                C::st(field[uniform(s.fl)] + (int64_t)i0 * so0 + (int64_t)i1 * so1 + s.disp, eval(T, q, i0, i1, i));
        }
}

// GROUPS: some entry of the launch is a group
template <typename R, typename S, bool GROUPS>
__global__ __launch_bounds__(BC_BLOCK) void bc_run_kernel(Geom g, FieldPtrs<S> F, const BcPieceAny* __restrict__ pieces,
                                                          const R* __restrict__ pool,
                                                          const BcBlock* __restrict__ blocks, int points, int t0,
                                                          int t1) {
    __shared__ __align__(16) int raw[BC_WORDS];
    __shared__ S* field[2 * NF];   // by field * 2 + level, as the terms name it
    __shared__ R slot[GROUPS ? BC_SLOTS * BC_TILE_ROWS : 1];
    const BcBlock e = blocks[blockIdx.x];
    const int t = (int)threadIdx.x;
    if (t < BC_WORDS) {
        raw[t] = reinterpret_cast<const int*>(pieces + e.piece)[t];
    } else {
        S* p = nullptr;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if (t == BC_WORDS + 2 * f) p = t0 ? F.f[f][1] : F.f[f][0];
            if (t == BC_WORDS + 2 * f + 1) p = t1 ? F.f[f][1] : F.f[f][0];
        }
        if (t < BC_WORDS + 2 * NF) field[t - BC_WORDS] = p;
    }
    __syncthreads();
    const int group = __builtin_amdgcn_readfirstlane(raw[0]);   // 1 + face axis, 0: a piece
    if (GROUPS && group == 3)
        bc_group<R, S, BC_TILE1[2]>(g, field, *reinterpret_cast<const BcGroupDesc*>(raw), pool, e.p0, slot);
    else if (GROUPS && group)
        bc_group<R, S, BC_TILE1[0]>(g, field, *reinterpret_cast<const BcGroupDesc*>(raw), pool, e.p0, slot);
    else
        bc_piece<R, S>(g, field, *reinterpret_cast<const BcPieceDesc*>(raw), pool, e.p0, points);
}

// Per-point media-dependent coefficients of the statements [first,
// first+count): coef * program, rounded to R exactly as bc_point does.
template <typename R>
__global__ __launch_bounds__(256) void bc_coef_kernel(Geom g, MediaPtrs<R> md, const BcDesc* __restrict__ desc,
                                                      const OpesciExprOp* __restrict__ code, R* __restrict__ pool,
                                                      int first) {
    const BcDesc* D = desc + first + blockIdx.y;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= D->npts) return;
    const int n1 = D->n1, axis = D->axis;
    const int i0 = D->lo0 + p / n1, i1 = D->lo1 + p % n1;
    const int ax = axis == 0 ? 0 : i0;
    const int ay = axis == 0 ? i0 : (axis == 1 ? 0 : i1);
    const int az = axis == 2 ? 0 : i1;
    const double c0[3] = {0, 0, 0};
    for (int k = 0; k < D->nterms; ++k)
        if (D->t[k].cslot >= 0)
            pool[D->cpool + (int64_t)D->t[k].cslot * D->npts + p] =
                (R)((double)D->t[k].coef * vm_eval<R>(code + D->t[k].prog, D->prog_len[k], c0, 0.0, md, g, ax, ay, az));
}

// item (face, point, term): one thread each
template <typename R>
__global__ __launch_bounds__(256) void zpool_kernel(ZFaceArgs zf, const R* __restrict__ pool, R* __restrict__ zpool) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)2 * ZPOOL_TERMS * zf.npts) return;
    const int e = (int)(i % ZPOOL_TERMS), face = i >= (int64_t)ZPOOL_TERMS * zf.npts ? 1 : 0;
    const int64_t p = i / ZPOOL_TERMS - (face ? zf.npts : 0);
    zpool[i] = pool[zf.cpool[face][e >> 3] + (int64_t)(e & 7) * zf.npts + p];
}

struct SolTable {
    double dx[3];
    double t[NF];
};

// The tables of the split analytic programs: slot blockIdx.y at every index
// i along its axis, coordinates as the point kernels compute them.
template <typename R>
__global__ __launch_bounds__(256) void sol_table_kernel(Geom g, MediaPtrs<R> md, SolProg sp, SolTable tab) {
    const SolSlot S = sp.slots[blockIdx.y];
    const int n = S.axis == 0 ? g.nx : (S.axis == 1 ? g.ny : g.nz);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double c[3] = {0.0, 0.0, 0.0};
    c[S.axis] = coord_of<R>(tab.dx[S.axis], i, g.m, stag(S.field, S.axis));
    sp.tab[S.tab + i] = vm_eval<R>(sp.code + S.prog, S.len, c, tab.t[S.field], md, g, 0, 0, 0);
}

// Field f's tables for the point kernels: copied into the block's LDS when
// they fit lds_cap doubles (the launch's dynamic LDS), else read in place.
constexpr int SOL_LDS_CAP = 4096;   // doubles (32 KiB)
__device__ __forceinline__ const double* stage_tables(const SolProg& sol, int f, int lds_cap) {
    extern __shared__ double stab[];
    const int n = sol.tab_len[f];
    if (n == 0 || n > lds_cap) return sol.tab + sol.tab_base[f];
    for (int i = threadIdx.x; i < n; i += blockDim.x) stab[i] = sol.tab[sol.tab_base[f] + i];
    __syncthreads();
    return stab;
}

// ------------------------------------------------------------------ initial state, L2 norms
// Field f's analytic values at z on K rows (x[k], y[k]) of a block: the K
// points of a shallow program in one pass over its ops, the others one
// point at a time.
// Bound by the doubles of the programs' sin, cos, sqrt and divide and by their
// decoding.  A program whose factors mix media with two axes reaches depth 4
// or 5 after its tables are split off, and the one-point evaluator's indexed
// stack then goes through scratch, so the several-points form takes depth 5
// (initial state with 3-D media, FP32: 512^3 45.1 -> 12.4 ms, 256^3 5.6 ->
// 1.54 ms; L2 norms at 101^3 217 -> 110 us).
// GENERAL: some field's program needs the one-point evaluator or holds POWC,
// EXP or LOG; the plain form leaves both out of the kernel and so keeps four
// waves per SIMD instead of two.
constexpr int SOL_ROWS = 4;
template <typename R, bool GENERAL>
__device__ __forceinline__ void sol_points(const SolProg& sol, const OpesciExprOp* __restrict__ code, int f,
                                           const SolTable& tab, const MediaPtrs<R>& md, const Geom& g,
                                           const int x[SOL_ROWS], const int y[SOL_ROWS], int z,
                                           const double* tabs, double v[SOL_ROWS]) {
    const int m = g.m;
    double cx[SOL_ROWS], cy[SOL_ROWS];
#pragma unroll
    for (int k = 0; k < SOL_ROWS; ++k) {
        cx[k] = coord_of<R>(tab.dx[0], x[k], m, stag(f, 0));
        cy[k] = coord_of<R>(tab.dx[1], y[k], m, stag(f, 1));
    }
    const double cz = coord_of<R>(tab.dx[2], z, m, stag(f, 2));
    if (!GENERAL || sol.shallow[f]) {
        vm_eval_k<R, SOL_ROWS, GENERAL>(code + sol.off[f], sol.len[f], cx, cy, cz, tab.t[f], md, g, x, y, z, tabs, v);
    } else {
        for (int k = 0; k < SOL_ROWS; ++k) {
            const double c[3] = {cx[k], cy[k], cz};
            v[k] = vm_eval_tos<R>(code + sol.off[f], sol.len[f], c, tab.t[f], md, g, x[k], y[k], z, tabs);
        }
    }
}

// rows r0 .. r0 + SOL_ROWS - 1 of field f's interior (x, y) rows; past the
// last row, repeats of it flagged not ok
__device__ __forceinline__ void sol_rows(int r0, int rows, int ny, int m, int x[SOL_ROWS], int y[SOL_ROWS],
                                         bool ok[SOL_ROWS]) {
#pragma unroll
    for (int k = 0; k < SOL_ROWS; ++k) {
        const int r = min(r0 + k, rows - 1);
        ok[k] = r0 + k < rows;
        x[k] = m + r / ny;
        y[k] = m + r % ny;
    }
}

// StaggeredGrid.initialise (opesci/staggeredgrid.py:612-659): level 0,
// ranges [m, dim-m) or [m, dim-m-1) when staggered, t = dt/2 for velocities.
template <typename R, typename S, bool GENERAL>
__global__ __launch_bounds__(256) void initial_kernel(Geom g, FieldPtrs<S> F, MediaPtrs<R> md, SolProg sol,
                                                      const OpesciExprOp* __restrict__ code, SolTable tab,
                                                      int lds_cap) {
    using C = Conv<S, R>;
    const int f = blockIdx.y;
    const int m = g.m;
    const int nx = g.nx - 2 * m - stag(f, 0), ny = g.ny - 2 * m - stag(f, 1), nz = g.nz - 2 * m - stag(f, 2);
    const int rows = nx * ny;
    const double* tabs = stage_tables(sol, f, lds_cap);
    // SOL_ROWS (x, y) rows per block iteration (block-uniform indices), z across threads
    for (int r0 = blockIdx.x * SOL_ROWS; r0 < rows; r0 += gridDim.x * SOL_ROWS) {
        int x[SOL_ROWS], y[SOL_ROWS];
        bool ok[SOL_ROWS];
        sol_rows(r0, rows, ny, m, x, y, ok);
        for (int z = m + (int)threadIdx.x; z < m + nz; z += blockDim.x) {
            double v[SOL_ROWS];
            sol_points<R, GENERAL>(sol, code, f, tab, md, g, x, y, z, tabs, v);
#pragma unroll
            for (int k = 0; k < SOL_ROWS; ++k)
                if (ok[k]) C::st(F.f[f][0] + g.at(x[k], y[k], z), (R)v[k]);
        }
    }
}

// sum over the interior of (F - F_exact(t_n))^2 in double
// (StaggeredGrid.converge_test, opesci/staggeredgrid.py:892-945); wavefront
// reduction by shuffles, one partial per block.
__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <typename R, typename S, bool GENERAL>
__global__ __launch_bounds__(256) void l2_kernel(Geom g, FieldPtrs<S> F, MediaPtrs<R> md, SolProg sol,
                                                 const OpesciExprOp* __restrict__ code, SolTable tab, int level,
                                                 double* __restrict__ partial, int lds_cap) {
    using C = Conv<S, R>;
    __shared__ double red[4];
    const int f = blockIdx.y;
    const int m = g.m;
    const int nx = g.nx - 2 * m - stag(f, 0), ny = g.ny - 2 * m - stag(f, 1), nz = g.nz - 2 * m - stag(f, 2);
    const int rows = nx * ny;
    const double* tabs = stage_tables(sol, f, lds_cap);
    double acc = 0.0;
    for (int r0 = blockIdx.x * SOL_ROWS; r0 < rows; r0 += gridDim.x * SOL_ROWS) {
        int x[SOL_ROWS], y[SOL_ROWS];
        bool ok[SOL_ROWS];
        sol_rows(r0, rows, ny, m, x, y, ok);
        for (int z = m + (int)threadIdx.x; z < m + nz; z += blockDim.x) {
            double v[SOL_ROWS];
            sol_points<R, GENERAL>(sol, code, f, tab, md, g, x, y, z, tabs, v);
#pragma unroll
            for (int k = 0; k < SOL_ROWS; ++k)
                if (ok[k]) {
                    const double e = (double)C::ld(F.f[f][level] + g.at(x[k], y[k], z)) - v[k];
                    acc += e * e;
                }
        }
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[(size_t)f * gridDim.x + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// ------------------------------------------------------------------ media
// StaggeredGrid.read_data (opesci/staggeredgrid.py:522-598): beta = 1/rho,
// lambda = rho (vp^2 - 2 vs^2), mu = rho vs^2 on every cell; beta1..3 =
// arithmetic means over the +x/+y/+z neighbour, mu12/mu13/mu23 = harmonic
// means over the 4-cell faces (the last index clamps to itself).
template <typename R>
__global__ void media_base_kernel(Geom g, const float* __restrict__ rho, const float* __restrict__ vp,
                                  const float* __restrict__ vs, MediaPtrs<R> out) {
    const int64_t n = (int64_t)g.nx * g.ny * g.nz;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(p % g.nz), y = (int)((p / g.nz) % g.ny), x = (int)(p / ((int64_t)g.nz * g.ny));
        const double r = rho[p], a = vp[p], b = vs[p];
        const int64_t q = g.at(x, y, z);
        R* const* o = (R* const*)out.m;
        o[OPESCI_M_RHO][q] = (R)r;
        o[OPESCI_M_VP][q] = (R)a;
        o[OPESCI_M_VS][q] = (R)b;
        o[OPESCI_M_BETA][q] = (R)(1.0 / r);
        o[OPESCI_M_LAMBDA][q] = (R)(r * (a * a - 2.0 * b * b));
        o[OPESCI_M_MU][q] = (R)(r * (b * b));
    }
}

template <typename R>
__global__ void media_eff_kernel(Geom g, MediaPtrs<R> md) {
    const int64_t n = (int64_t)g.nx * g.ny * g.nz;
    R* const* o = (R* const*)md.m;
    const R* beta = md.m[OPESCI_M_BETA];
    const R* mu = md.m[OPESCI_M_MU];
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(p % g.nz), y = (int)((p / g.nz) % g.ny), x = (int)(p / ((int64_t)g.nz * g.ny));
        const int x1 = min(x + 1, g.nx - 1), y1 = min(y + 1, g.ny - 1), z1 = min(z + 1, g.nz - 1);
        const int64_t q = g.at(x, y, z);
        const double b0 = beta[q];
        o[OPESCI_M_BETA1][q] = (R)((b0 + (double)beta[g.at(x1, y, z)]) / 2.0);
        o[OPESCI_M_BETA2][q] = (R)((b0 + (double)beta[g.at(x, y1, z)]) / 2.0);
        o[OPESCI_M_BETA3][q] = (R)((b0 + (double)beta[g.at(x, y, z1)]) / 2.0);
        const double i0 = 1.0 / (double)mu[q];
        const double ix = 1.0 / (double)mu[g.at(x1, y, z)], iy = 1.0 / (double)mu[g.at(x, y1, z)],
                     iz = 1.0 / (double)mu[g.at(x, y, z1)];
        o[OPESCI_M_MU12][q] = (R)(1.0 / (0.25 * (i0 + ix + iy + 1.0 / (double)mu[g.at(x1, y1, z)])));
        o[OPESCI_M_MU13][q] = (R)(1.0 / (0.25 * (i0 + ix + iz + 1.0 / (double)mu[g.at(x1, y, z1)])));
        o[OPESCI_M_MU23][q] = (R)(1.0 / (0.25 * (i0 + iy + iz + 1.0 / (double)mu[g.at(x, y1, z1)])));
    }
}

// ------------------------------------------------------------------ layout
template <typename R, typename S>
__global__ void pack_kernel(Geom g, const R* __restrict__ dense, S* __restrict__ field) {
    const int64_t n = (int64_t)g.nx * g.ny * g.nz;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(p % g.nz), y = (int)((p / g.nz) % g.ny), x = (int)(p / ((int64_t)g.nz * g.ny));
        Conv<S, R>::st(field + g.at(x, y, z), dense[p]);
    }
}

template <typename R, typename S>
__global__ void unpack_kernel(Geom g, const S* __restrict__ field, R* __restrict__ dense) {
    const int64_t n = (int64_t)g.nx * g.ny * g.nz;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(p % g.nz), y = (int)((p / g.nz) % g.ny), x = (int)(p / ((int64_t)g.nz * g.ny));
        dense[p] = Conv<S, R>::ld(field + g.at(x, y, z));
    }
}

struct ZeroList {
    uint4* p[2 * NF];
};
// n16 16-byte words of each array of the list (blockIdx.y)
__global__ void zero_kernel(ZeroList list, size_t n16) {
    uint4* p = list.p[blockIdx.y];
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x)
        p[i] = make_uint4(0, 0, 0, 0);
}

// ------------------------------------------------------------------ source / receivers
// tests/src/test_ref_iso_elastic.cpp:227-290: after the velocity update record
// U, V, W and (Txx+Tyy+Tzz)/3 at every receiver, then Tnn -= w[step]/3 at the
// source.  The step counter lives on the device so a captured graph can be
// replayed.
// Receivers (tests/src/test_ref_iso_elastic.cpp:227-272): U, V, W and
// (Txx+Tyy+Tzz)/3 at each receiver's grid point after the velocity update,
// one thread per receiver, trace[step][receiver][4] in the arithmetic type R
// (FP64 contexts keep FP64 traces, so misfits of FP64 runs are not rounded).
template <typename R> struct Trace4;
template <> struct Trace4<float> {
    static __device__ void put(void* t, size_t i, float a, float b, float c, float d) {
        reinterpret_cast<float4*>(t)[i] = make_float4(a, b, c, d);
    }
};
template <> struct Trace4<double> {
    static __device__ void put(void* t, size_t i, double a, double b, double c, double d) {
        double2* p = reinterpret_cast<double2*>(t) + 2 * i;
        p[0] = make_double2(a, b);
        p[1] = make_double2(c, d);
    }
};

// then, in the last block, the point source (test_ref_iso_elastic.cpp:274-290):
// Txx -= wx[t]/3, Tyy -= wy[t]/3, Tzz -= wz[t]/3 (one trace for all three
// when ntr == 1).  The receivers in the source's cell (at_src, which the
// others' blocks leave out) are read there, ahead of it.  step[l] is the
// number of the step whose level t0 is l: a step reads its own and leaves the
// next one's, so no block reads what another writes.  As launches of their
// own the receivers took 4.8 us and the source 4.3 us of a step.
template <typename R, typename S>
__global__ __launch_bounds__(256) void record_source_kernel(Geom g, FieldPtrs<S> F, int t1, int nrec, int nat,
                                                            const int32_t* __restrict__ rec,
                                                            const int32_t* __restrict__ at_src,
                                                            void* __restrict__ trace, int ntr, int sx, int sy, int sz,
                                                            const float* __restrict__ w, int* step, int ntsteps) {
    using C = Conv<S, R>;
    const int s = step[1 - t1], t = (int)threadIdx.x;
    auto put = [&](int r, int64_t q) {
        Trace4<R>::put(trace, (size_t)s * nrec + r, C::ld(F.f[0][t1] + q), C::ld(F.f[1][t1] + q),
                       C::ld(F.f[2][t1] + q),
                       (C::ld(F.f[3][t1] + q) + C::ld(F.f[4][t1] + q) + C::ld(F.f[5][t1] + q)) / (R)3);
    };
    if (blockIdx.x + 1 < gridDim.x) {
        const int r = blockIdx.x * blockDim.x + t;
        if (s >= ntsteps || r >= nrec) return;
        const int x = rec[3 * r], y = rec[3 * r + 1], z = rec[3 * r + 2];
        if (ntr > 0 && x == sx && y == sy && z == sz) return;
        put(r, g.at(x, y, z));
        return;
    }
    if (t == 0) step[t1] = s + 1;
    if (ntr == 0 || s >= ntsteps) return;
    const int64_t q = g.at(sx, sy, sz);
    if (nat > 0) {
        for (int i = t; i < nat; i += (int)blockDim.x) put(at_src[i], q);
        __syncthreads();
    }
    if (t < 3) {
        const R v = (R)w[(ntr == 3 ? t : 0) * (size_t)ntsteps + s] / (R)3;
        S* p = (t == 0 ? F.f[3][t1] : t == 1 ? F.f[4][t1] : F.f[5][t1]) + q;
        C::st(p, C::ld(p) - v);
    }
}

// ------------------------------------------------------------------ launchers
template <typename R, typename S>
static hipError_t bc_t(const Geom& g, void* fields, const BcDesc* desc, const void* pool, const BcLevel& lv, int t0,
                       int t1, hipStream_t s) {
    if (lv.count <= 0 || lv.maxpts <= 0) return hipSuccess;
    dim3 grid((lv.maxpts + 255) / 256, lv.count);
    hipLaunchKernelGGL((bc_kernel<R, S>), grid, dim3(256), 0, s, g, *static_cast<const FieldPtrs<S>*>(fields), desc,
                       static_cast<const R*>(pool), lv.first, t0, t1);
    return hipGetLastError();
}

template <typename R, typename S>
static hipError_t bc_run_t(const Geom& g, void* fields, const BcPieceAny* pieces, const void* pool, const BcBlock* blocks,
                           const BcRun& run, int t0, int t1, hipStream_t s) {
    if (run.count <= 0) return hipSuccess;
    const dim3 grid((unsigned)run.count), block(BC_BLOCK);
    const FieldPtrs<S>& F = *static_cast<const FieldPtrs<S>*>(fields);
    const R* coef = static_cast<const R*>(pool);
    if (run.groups)
        hipLaunchKernelGGL((bc_run_kernel<R, S, true>), grid, block, 0, s, g, F, pieces, coef, blocks + run.first,
                           run.points, t0, t1);
    else
        hipLaunchKernelGGL((bc_run_kernel<R, S, false>), grid, block, 0, s, g, F, pieces, coef, blocks + run.first,
                           run.points, t0, t1);
    return hipGetLastError();
}

template <typename R>
static hipError_t bc_coef_t(const Geom& g, const void* media, const BcDesc* desc, const OpesciExprOp* code,
                            void* pool, int first, int count, int maxpts, hipStream_t s) {
    if (count <= 0 || maxpts <= 0) return hipSuccess;
    dim3 grid((maxpts + 255) / 256, count);
    hipLaunchKernelGGL((bc_coef_kernel<R>), grid, dim3(256), 0, s, g, *static_cast<const MediaPtrs<R>*>(media), desc,
                       code, static_cast<R*>(pool), first);
    return hipGetLastError();
}

hipError_t launch_bc_coef(const Geom& g, int real_bytes, const void* media, const BcDesc* d_desc,
                          const OpesciExprOp* d_code, void* pool, int first, int count, int maxpts, hipStream_t s) {
    return real_bytes == 8 ? bc_coef_t<double>(g, media, d_desc, d_code, pool, first, count, maxpts, s)
                           : bc_coef_t<float>(g, media, d_desc, d_code, pool, first, count, maxpts, s);
}

#define OPESCI_TYPED(RB, ST, CALL_F, CALL_D, CALL_H, CALL_B) \
    ((RB) == 8 ? (CALL_D) : (ST) == OPESCI_STORE_F16 ? (CALL_H) : (ST) == OPESCI_STORE_BF16 ? (CALL_B) : (CALL_F))

hipError_t launch_zpool(int real_bytes, const ZFaceArgs& zf, const void* pool, void* zpool, hipStream_t s) {
    const dim3 grid((unsigned)(((int64_t)2 * ZPOOL_TERMS * zf.npts + 255) / 256));
    if (real_bytes == 8)
        hipLaunchKernelGGL((zpool_kernel<double>), grid, dim3(256), 0, s, zf, static_cast<const double*>(pool),
                           static_cast<double*>(zpool));
    else
        hipLaunchKernelGGL((zpool_kernel<float>), grid, dim3(256), 0, s, zf, static_cast<const float*>(pool),
                           static_cast<float*>(zpool));
    return hipGetLastError();
}

hipError_t launch_bc(const Geom& g, int real_bytes, int storage, void* fields, const BcDesc* d_desc, const void* pool,
                     const BcLevel& lvl, int t0, int t1, hipStream_t s) {
    return OPESCI_TYPED(real_bytes, storage, (bc_t<float, float>(g, fields, d_desc, pool, lvl, t0, t1, s)),
                        (bc_t<double, double>(g, fields, d_desc, pool, lvl, t0, t1, s)),
                        (bc_t<float, _Float16>(g, fields, d_desc, pool, lvl, t0, t1, s)),
                        (bc_t<float, bf16_t>(g, fields, d_desc, pool, lvl, t0, t1, s)));
}

hipError_t launch_bc_run(const Geom& g, int real_bytes, int storage, void* fields, const BcPieceAny* d_pieces,
                         const void* pool, const BcBlock* blocks, const BcRun& run, int t0, int t1, hipStream_t s) {
    return OPESCI_TYPED(real_bytes, storage, (bc_run_t<float, float>(g, fields, d_pieces, pool, blocks, run, t0, t1, s)),
                        (bc_run_t<double, double>(g, fields, d_pieces, pool, blocks, run, t0, t1, s)),
                        (bc_run_t<float, _Float16>(g, fields, d_pieces, pool, blocks, run, t0, t1, s)),
                        (bc_run_t<float, bf16_t>(g, fields, d_pieces, pool, blocks, run, t0, t1, s)));
}

static SolTable make_tab(const double* dx) {
    SolTable t;
    for (int f = 0; f < NF; ++f) t.t[f] = 0.0;
    for (int a = 0; a < 3; ++a) t.dx[a] = dx[a];
    return t;
}

// doubles of dynamic LDS for the point kernels: the largest field's tables
// when within SOL_LDS_CAP (fields with larger tables read them in place)
static int sol_lds(const SolProg& sol) {
    int n = 0;
    for (int f = 0; f < NF; ++f)
        if (sol.tab_len[f] <= SOL_LDS_CAP) n = std::max(n, sol.tab_len[f]);
    return n;
}

// the tables for this launch's times (stream-ordered before the point kernel)
template <typename R>
static hipError_t sol_tables_t(const Geom& g, const void* media, const SolProg& sol, const SolTable& tab,
                               hipStream_t s) {
    if (sol.nslots <= 0) return hipSuccess;
    hipLaunchKernelGGL((sol_table_kernel<R>), dim3((sol.maxdim + 255) / 256, sol.nslots), dim3(256), 0, s, g,
                       *static_cast<const MediaPtrs<R>*>(media), sol, tab);
    return hipGetLastError();
}

template <typename R, typename S>
static hipError_t init_t(const Geom& g, void* fields, const void* media, const SolProg& sol, SolTable tab,
                         hipStream_t s) {
    if (hipError_t e = sol_tables_t<R>(g, media, sol, tab, s)) return e;
    const int cap = sol_lds(sol);
    auto kernel = sol.general ? initial_kernel<R, S, true> : initial_kernel<R, S, false>;
    hipLaunchKernelGGL(kernel, dim3(512, NF), dim3(256), cap * sizeof(double), s, g,
                       *static_cast<const FieldPtrs<S>*>(fields), *static_cast<const MediaPtrs<R>*>(media), sol,
                       sol.code, tab, cap);
    return hipGetLastError();
}

hipError_t launch_initial(const Geom& g, int real_bytes, int storage, void* fields, const void* media,
                          const SolProg& sol, const double* spacing, double dt, hipStream_t s) {
    SolTable tab = make_tab(spacing);
    for (int f = 0; f < NF; ++f) tab.t[f] = time_stag(f) ? dt / 2.0 : 0.0;
    return OPESCI_TYPED(real_bytes, storage, (init_t<float, float>(g, fields, media, sol, tab, s)),
                        (init_t<double, double>(g, fields, media, sol, tab, s)),
                        (init_t<float, _Float16>(g, fields, media, sol, tab, s)),
                        (init_t<float, bf16_t>(g, fields, media, sol, tab, s)));
}

template <typename R, typename S>
static hipError_t l2_t(const Geom& g, void* fields, const void* media, const SolProg& sol, SolTable tab,
                       int level, double* partial, int nblk, hipStream_t s) {
    if (hipError_t e = sol_tables_t<R>(g, media, sol, tab, s)) return e;
    const int cap = sol_lds(sol);
    auto kernel = sol.general ? l2_kernel<R, S, true> : l2_kernel<R, S, false>;
    hipLaunchKernelGGL(kernel, dim3(nblk, NF), dim3(256), cap * sizeof(double), s, g,
                       *static_cast<const FieldPtrs<S>*>(fields), *static_cast<const MediaPtrs<R>*>(media), sol,
                       sol.code, tab, level, partial, cap);
    return hipGetLastError();
}

hipError_t launch_l2(const Geom& g, int real_bytes, int storage, void* fields, const void* media,
                     const SolProg& sol, const double* spacing, int level, const double t_field[NF],
                     double* d_partial, int partial_cap, double* out_host, hipStream_t s) {
    SolTable tab = make_tab(spacing);
    for (int f = 0; f < NF; ++f) tab.t[f] = t_field[f];
    const int nblk = partial_cap / NF;
    hipError_t e = OPESCI_TYPED(real_bytes, storage,
                                (l2_t<float, float>(g, fields, media, sol, tab, level, d_partial, nblk, s)),
                                (l2_t<double, double>(g, fields, media, sol, tab, level, d_partial, nblk, s)),
                                (l2_t<float, _Float16>(g, fields, media, sol, tab, level, d_partial, nblk, s)),
                                (l2_t<float, bf16_t>(g, fields, media, sol, tab, level, d_partial, nblk, s)));
    if (e != hipSuccess) return e;
    std::vector<double> h((size_t)NF * nblk);
    e = hipMemcpyAsync(h.data(), d_partial, h.size() * sizeof(double), hipMemcpyDeviceToHost, s);
    if (e != hipSuccess) return e;
    e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    const double vol = spacing[0] * spacing[1] * spacing[2];
    for (int f = 0; f < NF; ++f) {
        double a = 0.0;
        for (int b = 0; b < nblk; ++b) a += h[(size_t)f * nblk + b];
        out_host[f] = sqrt(a * vol);
    }
    return hipSuccess;
}

// ------------------------------------------------------------------ L2 without allocation
// The per-block partial sums of opesci_ctx_l2_noalloc live in one
// library-owned array per device: NF x L2_BLOCKS doubles (36 KiB), held
// until the process ends and shared by every call on that device (calls
// that overlap on one device race on it).  Every block of l2_kernel writes
// its partial, so nothing needs clearing between calls.  In host code the
// array's name stands for a host-side shadow, never for device memory: the
// device address is looked up once per device with hipGetSymbolAddress and
// only that address is handed to kernels.
constexpr int L2_BLOCKS = 512;
constexpr int L2_MAX_DEVICES = 64;
static __device__ __align__(256) double l2_scratch[NF * L2_BLOCKS];

// out[f] = sqrt(vol * sum_b partial[f][b]), summed in block order like the
// host reduction of launch_l2
__global__ void l2_finish_kernel(const double* __restrict__ partial, int nblk, double vol, double* __restrict__ out) {
    const int f = threadIdx.x;
    if (f >= NF) return;
    double a = 0.0;
    for (int b = 0; b < nblk; ++b) a += partial[(size_t)f * nblk + b];
    out[f] = sqrt(a * vol);
}

static hipError_t l2_scratch_of_current_device(double** out) {
    static std::mutex mu;
    static double* addr[L2_MAX_DEVICES] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= L2_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(l2_scratch));
        if (e != hipSuccess) return e;
        addr[dev] = static_cast<double*>(p);
    }
    *out = addr[dev];
    return hipSuccess;
}

int l2_noalloc_partials() { return L2_BLOCKS; }

hipError_t launch_l2_noalloc(const Geom& g, int real_bytes, int storage, void* fields, const void* media,
                             const SolProg& sol, const double* spacing, int level, const double t_field[NF],
                             double* d_out, hipStream_t s) {
    double* partial = nullptr;
    hipError_t e = l2_scratch_of_current_device(&partial);
    if (e != hipSuccess) return e;
    SolTable tab = make_tab(spacing);
    for (int f = 0; f < NF; ++f) tab.t[f] = t_field[f];
    e = OPESCI_TYPED(real_bytes, storage,
                     (l2_t<float, float>(g, fields, media, sol, tab, level, partial, L2_BLOCKS, s)),
                     (l2_t<double, double>(g, fields, media, sol, tab, level, partial, L2_BLOCKS, s)),
                     (l2_t<float, _Float16>(g, fields, media, sol, tab, level, partial, L2_BLOCKS, s)),
                     (l2_t<float, bf16_t>(g, fields, media, sol, tab, level, partial, L2_BLOCKS, s)));
    if (e != hipSuccess) return e;
    const double vol = spacing[0] * spacing[1] * spacing[2];
    hipLaunchKernelGGL(l2_finish_kernel, dim3(1), dim3(64), 0, s, (const double*)partial, L2_BLOCKS, vol, d_out);
    return hipGetLastError();
}

hipError_t launch_media(const Geom& g, int real_bytes, const float* d_rho, const float* d_vp, const float* d_vs,
                        void* const* d_media, hipStream_t s) {
    if (real_bytes == 8) {
        MediaPtrs<double> mp;
        for (int i = 0; i < OPESCI_M_COUNT; ++i) mp.m[i] = (const double*)d_media[i];
        hipLaunchKernelGGL((media_base_kernel<double>), dim3(1024), dim3(256), 0, s, g, d_rho, d_vp, d_vs, mp);
        hipLaunchKernelGGL((media_eff_kernel<double>), dim3(1024), dim3(256), 0, s, g, mp);
    } else {
        MediaPtrs<float> mp;
        for (int i = 0; i < OPESCI_M_COUNT; ++i) mp.m[i] = (const float*)d_media[i];
        hipLaunchKernelGGL((media_base_kernel<float>), dim3(1024), dim3(256), 0, s, g, d_rho, d_vp, d_vs, mp);
        hipLaunchKernelGGL((media_eff_kernel<float>), dim3(1024), dim3(256), 0, s, g, mp);
    }
    return hipGetLastError();
}

template <typename R, typename S>
static hipError_t pack_t(const Geom& g, const void* dense, void* field, hipStream_t s) {
    hipLaunchKernelGGL((pack_kernel<R, S>), dim3(1024), dim3(256), 0, s, g, (const R*)dense, (S*)field);
    return hipGetLastError();
}
template <typename R, typename S>
static hipError_t unpack_t(const Geom& g, const void* field, void* dense, hipStream_t s) {
    hipLaunchKernelGGL((unpack_kernel<R, S>), dim3(1024), dim3(256), 0, s, g, (const S*)field, (R*)dense);
    return hipGetLastError();
}

hipError_t launch_pack(const Geom& g, int real_bytes, int storage, const void* dense, void* field, hipStream_t s) {
    return OPESCI_TYPED(real_bytes, storage, (pack_t<float, float>(g, dense, field, s)),
                        (pack_t<double, double>(g, dense, field, s)), (pack_t<float, _Float16>(g, dense, field, s)),
                        (pack_t<float, bf16_t>(g, dense, field, s)));
}

hipError_t launch_unpack(const Geom& g, int real_bytes, int storage, const void* field, void* dense, hipStream_t s) {
    return OPESCI_TYPED(real_bytes, storage, (unpack_t<float, float>(g, field, dense, s)),
                        (unpack_t<double, double>(g, field, dense, s)),
                        (unpack_t<float, _Float16>(g, field, dense, s)), (unpack_t<float, bf16_t>(g, field, dense, s)));
}

hipError_t launch_pack_media(const Geom& g, int real_bytes, const void* dense, void* media, hipStream_t s) {
    return real_bytes == 8 ? pack_t<double, double>(g, dense, media, s) : pack_t<float, float>(g, dense, media, s);
}

hipError_t launch_zero(void* p, size_t bytes, hipStream_t s) { return launch_zero_all(&p, 1, bytes, s); }

// One launch for up to 2 * NF arrays of one size: an init clears 18, a reverse
// sweep 30, and on small grids a launch costs what it clears (16^3: 18
// launches 0.2 ms of an init's 0.4).
hipError_t launch_zero_all(void* const* p, int n, size_t bytes, hipStream_t s) {
    const size_t n16 = bytes / 16;
    if (n <= 0 || n16 == 0) return hipSuccess;
    if (n > 2 * NF) return hipErrorInvalidValue;
    ZeroList list = {};
    for (int i = 0; i < n; ++i) list.p[i] = static_cast<uint4*>(p[i]);
    const unsigned blocks = (unsigned)std::min<size_t>(n > 1 ? 512 : 2048, (n16 + 255) / 256);
    hipLaunchKernelGGL(zero_kernel, dim3(blocks, (unsigned)n), dim3(256), 0, s, list, n16);
    return hipGetLastError();
}

template <typename R, typename S>
static hipError_t rec_t(const Geom& g, void* fields, int t1, int nrec, int nat, const int32_t* rec,
                        const int32_t* at_src, void* trace, int ntr, const int32_t* si, const float* w, int* step,
                        int ntsteps, hipStream_t s) {
    const FieldPtrs<S>& F = *static_cast<const FieldPtrs<S>*>(fields);
    hipLaunchKernelGGL((record_source_kernel<R, S>), dim3((nrec + 255) / 256 + 1), dim3(nrec > 0 ? 256 : 64), 0, s, g, F,
                       t1, nrec, nat, rec, at_src, trace, ntr, si[0], si[1], si[2], w, step, ntsteps);
    return hipGetLastError();
}

hipError_t launch_record_source(const Geom& g, int real_bytes, int storage, void* fields, int t1, int nrec, int nat,
                                const int32_t* d_rec, const int32_t* d_at_src, void* d_trace, int src_on,
                                const int32_t* src_idx, const float* d_wavelet, int* d_step, int ntsteps,
                                hipStream_t s) {
#define OPESCI_REC(R, S)                                                                                             \
    (rec_t<R, S>(g, fields, t1, nrec, nat, d_rec, d_at_src, d_trace, src_on, src_idx, d_wavelet, d_step, ntsteps, s))
    return OPESCI_TYPED(real_bytes, storage, OPESCI_REC(float, float), OPESCI_REC(double, double),
                        OPESCI_REC(float, _Float16), OPESCI_REC(float, bf16_t));
#undef OPESCI_REC
}

}  // namespace opesci
