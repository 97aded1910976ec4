// Stress half step as a flat-tile x sweep (sweep.h): the six stresses at t1
// from the velocities and stresses at t0 (opesci/staggeredgrid.py:728-737).
// Stencil and accumulation order as in interior.hip; its gather kernel gives
// the same bits.
//
// What bounds it: on large grids the memory path (9 reads and 6 writes per
// point: 60 bytes in FP32), on small ones a plane's chain of load, staging,
// barrier and LDS reads, with 16-bit storage the instructions.  So it keeps
// few registers (61-72 at 4th order in FP32: three blocks per CU), forms the
// addresses from shared 32-bit offsets, rotates the queues by name and sums
// the off-axis normal terms once: 184 instructions per plane and wave of 64
// points at 4th order, against 271 per 64 points for the sweep of two points
// per lane that it replaces.  Two points per lane in this form (two blocks
// per CU) measured 248 us against 239 on the 256^3 read path and 147 against
// 128 us for FP16; loads two planes ahead instead of one, and blocks of 256
// or 1024 threads, gained nothing; z tiles that do not start on a line cost
// 81 us against 58 at 160^3.  Measured before -> now (events, us), now with the
// z faces in every one and rows of 9 lines at 256^3: 256^3 4th order FP32 223
// (z faces in it) -> 190, read path 253 -> 258 (226 without the z faces), FP16
// 278 -> 125; 128^3 4th order FP64 read path 82 -> 60; 160^3 FP32 107 -> 61; 161
// x 129 x 193 8th order BF16 read path 103 -> 87; 16^3 26 -> 7.
//
// The z-face statements of the deep rows are done here for every type and
// medium: as launches they touch a line per point and statement.  Sweep +
// other launches of a step before -> after (us): 256^3 4th order read path
// 231 + 191 -> 255 + 132, 512^3 8th order read path 2090 + 274 -> 2212 + 100,
// 161 x 129 x 193 8th order BF16 78 + 42 -> 86 + 27.  The sweep's share is
// 6 us image stores and 10 us coefficients at 256^3 4th order, all image
// stores (partial lines) at 512^3.  The coefficients in the pool's term-major
// order cost 262 instead of 255 us; non-temporal image stores 261; the high
// surface's images taken from the lane below (one whole store per line) 201
// instead of 187 us on constant media, the exchange costs more than the line.
#include "bcdev.h"
#include "sweep.h"

namespace opesci {

// Coefficients by axis j.  SHARED: own[j] multiplies the difference along j
// in T_jj, off[j] in the two other normal stresses (the same for both, which
// the launcher checks, so their sums are formed once); on the read path own
// and off are one set and the media scale the sums.  Else a set per stress i
// and axis, and nine sums: what a caller of the C ABI may ask for.
template <typename R, bool SHARED>
struct StressCoefs {
    R own[3][MAXM];
    R off[3][MAXM];
    R cs[3][2][MAXM];
};
template <typename R>
struct StressCoefs<R, false> {
    R n[3][3][MAXM];
    R cs[3][2][MAXM];
};
template <typename R, typename S>
struct StressPtrs {
    const S* v[3];    // U, V, W at t0
    const S* s0[6];   // Txx, Tyy, Tzz, Txy, Tyz, Txz at t0
    S* s1[6];         // the same at t1
    const R* lam;     // read path: lambda, mu, mu12, mu23, mu13
    const R* mu;
    const R* ms[3];
};

template <typename R, typename S, int M, bool HET, bool ZF, bool SHARED>
__global__ __launch_bounds__(SWEEP_THREADS, sizeof(R) * M <= 8 ? (SHARED ? 5 : 4) : 2) void stress_flat(
    Geom g, StressPtrs<R, S> P, StressCoefs<R, SHARED> c, SweepTile T, int nblocks, Boxes B, ZFaceArgs zf) {
    using C = Conv<S, R>;
    constexpr int Q = 2 * M;
    constexpr bool ZPOOL = ZF && HET && M == 2;   // the surface recompute takes per-point coefficients
    __shared__ R lds[2][3][SweepPlane<M>::SIZE];
    __shared__ R zlds[2][ZPOOL ? ZPOOL_ITEMS : 1];
    const int l = sweep_block(nblocks);
    if (l < 0) return;
    const SweepLane s = sweep_lane<M>(g, B, l, T);
    // scalar bases at the chunk's first plane, per-thread byte offsets
    const int64_t x0 = (int64_t)s.xb * g.sx;
    const S *bU = P.v[0] + x0, *bV = P.v[1] + x0, *bW = P.v[2] + x0;
    const S* b0[6];
    S* b1[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        b0[f] = P.s0[f] + x0;
        b1[f] = P.s1[f] + x0;
    }
    const R* bm[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    if (HET) {
        bm[0] = P.lam + x0;
        bm[1] = P.mu + x0;
        for (int k = 0; k < 3; ++k) bm[2 + k] = P.ms[k] + x0;
    }
    const uint32_t plane = (uint32_t)g.sx * sizeof(S);
    uint32_t own = s.own * sizeof(S), oy = s.gy * sizeof(S), oz = s.gz * sizeof(S), ox = s.gx * sizeof(S),
             om = s.own * sizeof(R);
    // register queues, logical element i at slot (phase + i) % Q:
    // U(x + i - M), V(x + i - M + 1), W(x + i - M + 1)
    R qU[Q], qV[Q], qW[Q];
#pragma unroll
    for (int i = 0; i < Q - 1; ++i) {
        qU[i] = C::ld(at_byte(bU + (int64_t)(i - M) * g.sx, own));
        qV[i] = C::ld(at_byte(bV + (int64_t)(i - M + 1) * g.sx, own));
        qW[i] = C::ld(at_byte(bW + (int64_t)(i - M + 1) * g.sx, own));
    }
    // z-face statements: which of them this thread's point takes part in, and
    // where its images go (bytes from the point itself)
    bool deep = false, image_s = false, image_n = false, surface = false, high = false;
    uint32_t to_s = 0, to_n = 0;
    // read path: the recompute's coefficients of a plane, ZPOOL_TERMS per
    // surface point of the tile, staged through LDS one per thread: item
    // (face, row, term)
    const R* pz = nullptr;
    int zitem = 0;
    R nz = 0;
    if constexpr (ZPOOL) {
        const int per = ZPOOL_TERMS * s.rows, t = (int)threadIdx.x;
        if (zf.rec && t < ((s.low ? 1 : 0) + (s.high ? 1 : 0)) * per) {
            const int face = (s.low ? 0 : 1) + t / per, e = t % per, y = s.y0 + e / ZPOOL_TERMS;
            if (y >= zf.F && y < g.ny - zf.F)
                pz = static_cast<const R*>(zf.zpool) + (int64_t)face * ZPOOL_TERMS * zf.npts +
                     (int64_t)ZPOOL_TERMS * (y - zf.F - zf.F * zf.n1) + e % ZPOOL_TERMS;
        }
        zitem = ((s.low && s.z == M) || !s.low ? 0 : per) + ZPOOL_TERMS * (s.y - s.y0);
    }
    if constexpr (ZF) {
        const int k = s.z - M, j = g.nz - M - 1 - s.z;   // points above the low and below the high surface
        deep = s.on && s.y >= zf.F && s.y < g.ny - zf.F;
        surface = deep && (k == 0 || j == 0);
        high = deep && j == 0;
        image_s = deep && (k < M || (j >= 1 && j <= M));
        image_n = deep && ((k >= 1 && k < M) || (j >= 1 && j < M));
        to_s = (uint32_t)((k < M ? -1 - 2 * k : 2 * j - 1) * (int)sizeof(S));
        to_n = (uint32_t)((k < M ? -2 * k : 2 * j) * (int)sizeof(S));
    }
    // the next plane's values, loaded one plane ahead
    R nU, nV, nW, nT[6], nm[5], yU, yV, yW, zU, zV, zW, xU, xV, xW;
    const S* aU = bU + (int64_t)(M - 1) * g.sx;
    const S* aV = bV + (int64_t)M * g.sx;
    const S* aW = bW + (int64_t)M * g.sx;
    auto fetch = [&](int x) __attribute__((always_inline)) {
        if constexpr (ZPOOL) {
            if (pz && x >= zf.F && x < g.nx - zf.F) nz = pz[(int64_t)x * (ZPOOL_TERMS * zf.n1)];
        }
        // halos, then the point's own loads in one block (the order in which
        // they are waited for)
        if (s.hy) {
            yU = C::ld(at_byte(bU, oy));
            yV = C::ld(at_byte(bV, oy));
            yW = C::ld(at_byte(bW, oy));
        }
        if (sweep_second_halo<M>() && s.hx) {
            xU = C::ld(at_byte(bU, ox));
            xV = C::ld(at_byte(bV, ox));
            xW = C::ld(at_byte(bW, ox));
        }
        if (s.hz) {
            zU = C::ld(at_byte(bU, oz));
            zV = C::ld(at_byte(bV, oz));
            zW = C::ld(at_byte(bW, oz));
        }
        nU = C::ld(at_byte(aU, own));
        nV = C::ld(at_byte(aV, own));
        nW = C::ld(at_byte(aW, own));
#pragma unroll
        for (int f = 0; f < 6; ++f) nT[f] = C::ldnt(at_byte(b0[f], own));
        if (HET) {
#pragma unroll
            for (int k = 0; k < 5; ++k) nm[k] = Conv<R, R>::ldnt(at_byte(bm[k], om));
        }
    };
    fetch(s.xb);
    const int pitch = s.pitch;
    auto step = [&](auto phase, int x) __attribute__((always_inline)) {
        constexpr int PH = decltype(phase)::value, b = PH & 1;
        auto q = [](int i) constexpr { return (PH + i) % Q; };
        qU[q(Q - 1)] = nU;
        qV[q(Q - 1)] = nV;
        qW[q(Q - 1)] = nW;
        R T0[6], md[5];
#pragma unroll
        for (int f = 0; f < 6; ++f) T0[f] = nT[f];
        if (HET) {
#pragma unroll
            for (int k = 0; k < 5; ++k) md[k] = nm[k];
        }
        R* LU = lds[b][0];
        R* LV = lds[b][1];
        R* LW = lds[b][2];
        if (s.on) {
            LU[s.me] = qU[q(M)];
            LV[s.me] = qV[q(M - 1)];
            LW[s.me] = qW[q(M - 1)];
        }
        if (s.hy) {
            LU[s.ly] = yU;
            LV[s.ly] = yV;
            LW[s.ly] = yW;
        }
        if (sweep_second_halo<M>() && s.hx) {
            LU[s.lx] = xU;
            LV[s.lx] = xV;
            LW[s.lx] = xW;
        }
        if (s.hz) {
            LU[s.lz] = zU;
            LV[s.lz] = zV;
            LW[s.lz] = zW;
        }
        if constexpr (ZPOOL) {
            if (pz) zlds[b][threadIdx.x] = nz;
        }
        const uint32_t here = own;
        if (x + 1 < s.xe) {
            own += plane;
            oy += plane;
            oz += plane;
            ox += plane;
            om += (uint32_t)g.sx * sizeof(R);
            fetch(x + 1);
        }
        lds_barrier();
        if (s.on) {
            R so[3] = {0, 0, 0}, sf[3] = {0, 0, 0};   // sums along x, y, z with own and off coefficients
            R sn[3][3] = {};                          // or of every stress and axis
            R vy[Q];                                  // V(y - M .. y + M - 1)
#pragma unroll
            for (int i = 0; i < Q; ++i) vy[i] = i == M ? qV[q(M - 1)] : LV[s.me + (i - M) * pitch];
#pragma unroll
            for (int k = 0; k < M; ++k) {
                const R d[3] = {qU[q(M + k)] - qU[q(M - 1 - k)], vy[M + k] - vy[M - 1 - k],
                                (k == 0 ? qW[q(M - 1)] : LW[s.me + k]) - LW[s.me - 1 - k]};
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    if constexpr (SHARED) {
                        so[j] = fma(c.own[j][k], d[j], so[j]);
                        if (!HET) sf[j] = fma(c.off[j][k], d[j], sf[j]);
                    } else {
#pragma unroll
                        for (int i = 0; i < 3; ++i) sn[i][j] = fma(c.n[i][j][k], d[j], sn[i][j]);
                    }
                }
            }
            R lam = 0, l2m = 0;
            if (HET) {
                lam = md[0];
                l2m = lam + (R)2 * md[1];
            }
            R out[6];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                R acc = T0[i];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const R sum = !SHARED ? sn[i][j] : (HET || j == i) ? so[j] : sf[j];
                    acc = HET ? fma(j == i ? l2m : lam, sum, acc) : acc + sum;
                }
                out[i] = acc;
            }
            const R u0 = qU[q(M)], v0 = qV[q(M - 1)], w0 = qW[q(M - 1)];
            R sxy = 0, syz = 0, sxz = 0;
#pragma unroll
            for (int k = 0; k < M; ++k)
                sxy = fma(c.cs[0][0][k], LU[s.me + (1 + k) * pitch] - (k == 0 ? u0 : LU[s.me - k * pitch]), sxy);
#pragma unroll
            for (int k = 0; k < M; ++k) sxy = fma(c.cs[0][1][k], qV[q(M + k)] - qV[q(M - 1 - k)], sxy);
#pragma unroll
            for (int k = 0; k < M; ++k)
                syz = fma(c.cs[1][0][k], LV[s.me + 1 + k] - (k == 0 ? v0 : LV[s.me - k]), syz);
#pragma unroll
            for (int k = 0; k < M; ++k)
                syz = fma(c.cs[1][1][k], LW[s.me + (1 + k) * pitch] - (k == 0 ? w0 : LW[s.me - k * pitch]), syz);
#pragma unroll
            for (int k = 0; k < M; ++k)
                sxz = fma(c.cs[2][0][k], LU[s.me + 1 + k] - (k == 0 ? u0 : LU[s.me - k]), sxz);
#pragma unroll
            for (int k = 0; k < M; ++k) sxz = fma(c.cs[2][1][k], qW[q(M + k)] - qW[q(M - 1 - k)], sxz);
            out[3] = HET ? fma(md[2], sxy, T0[3]) : T0[3] + sxy;
            out[4] = HET ? fma(md[3], syz, T0[4]) : T0[4] + syz;
            out[5] = HET ? fma(md[4], sxz, T0[5]) : T0[5] + sxz;
            if constexpr (ZF) {
                // free-surface statements of the z faces on the deep rows:
                // the points within M of a face store their own images (the
                // negated value a later read would see), the surface point
                // takes the Levander recompute of Txx and Tyy and Tzz = 0
                if (x >= zf.F && x < g.nx - zf.F) {
                    if (image_s) {
                        C::st(at_byte(b1[4], here + to_s), (R)0 - stored<S, R>(out[4]));
                        C::st(at_byte(b1[5], here + to_s), (R)0 - stored<S, R>(out[5]));
                    }
                    if (image_n) C::st(at_byte(b1[2], here + to_n), (R)0 - stored<S, R>(out[2]));
                    if (surface) {
                        if constexpr (M == 2) {
                            if (zf.rec) {
                                const R qx[4] = {qU[q(0)], qU[q(1)], qU[q(2)], qU[q(3)]};
#pragma unroll
                                for (int i = 0; i < 2; ++i) {
                                    R r = 0;
                                    if constexpr (HET) {
                                        const R* zc = zlds[b] + zitem + 8 * i;
#pragma unroll
                                        for (int k = 0; k < 8; ++k)
                                            r = fma(zc[k], k < 4 ? qx[k] : vy[k - 4], r);
                                    } else {
                                        r = fma((R)-zf.rc.x[1][i], qx[0], r);
                                        r = fma((R)-zf.rc.x[0][i], qx[1], r);
                                        r = fma((R)zf.rc.x[0][i], qx[2], r);
                                        r = fma((R)zf.rc.x[1][i], qx[3], r);
                                        r = fma((R)-zf.rc.y[1][i], vy[0], r);
                                        r = fma((R)-zf.rc.y[0][i], vy[1], r);
                                        r = fma((R)zf.rc.y[0][i], vy[2], r);
                                        r = fma((R)zf.rc.y[1][i], vy[3], r);
                                    }
                                    out[i] = r + T0[i];
                                }
                            }
                        }
                        out[2] = 0;
                    }
                }
            }
#pragma unroll
            for (int f = 0; f < 4; ++f) C::stnt(at_byte(b1[f], here), out[f]);
            // on the high surface Tyz and Txz are images too (stored by the point below)
            if (!ZF || !(high && x >= zf.F && x < g.nx - zf.F)) {
                C::stnt(at_byte(b1[4], here), out[4]);
                C::stnt(at_byte(b1[5], here), out[5]);
            }
        }
    };
    sweep_planes(s.xb, s.xe, step, std::make_integer_sequence<int, Q>{});
}

// ------------------------------------------------------------------ launch
template <typename R, typename S, int M, bool HET, bool SHARED>
static hipError_t launch_shape(const Geom& g, const FieldPtrs<S>& F, const MediaPtrs<R>& md,
                               const StressCoefs<R, SHARED>& k, int t0, int t1, const InteriorLaunch& cfg,
                               hipStream_t s, const ZFaceArgs* zf, const Boxes* boxes) {
    const bool in_sweep = zf && zf->F > 0;
    static std::atomic<int> occ[2][SWEEP_THREADS / 64 + 1] = {};
    // 9 reads and 6 writes of the storage type, 5 media
    const SweepShape sh = sweep_shape<M>(
        g, cfg, boxes, 15 * (int)sizeof(S) + (HET ? 5 * (int)sizeof(R) : 0), sizeof(S), [&](int threads) {
            return in_sweep ? sweep_blocks_per_cu(stress_flat<R, S, M, HET, true, SHARED>, occ[1], threads)
                            : sweep_blocks_per_cu(stress_flat<R, S, M, HET, false, SHARED>, occ[0], threads);
        },
        in_sweep && HET && M == 2 && zf->rec ? ZPOOL_TERMS : 0);
    if (sh.nb == 0) return hipSuccess;
    StressPtrs<R, S> P;
    for (int i = 0; i < 3; ++i) P.v[i] = F.f[i][t0];
    for (int f = 0; f < 6; ++f) {
        P.s0[f] = F.f[3 + f][t0];
        P.s1[f] = F.f[3 + f][t1];
    }
    P.lam = md.m[OPESCI_M_LAMBDA];
    P.mu = md.m[OPESCI_M_MU];
    P.ms[0] = md.m[OPESCI_M_MU12];
    P.ms[1] = md.m[OPESCI_M_MU23];
    P.ms[2] = md.m[OPESCI_M_MU13];
    const dim3 grid((unsigned)((sh.nb + 7) / 8 * 8)), block((unsigned)sh.threads);
    if (in_sweep)
        hipLaunchKernelGGL((stress_flat<R, S, M, HET, true, SHARED>), grid, block, 0, s, g, P, k, sh.tile, sh.nb,
                           sh.boxes, *zf);
    else
        hipLaunchKernelGGL((stress_flat<R, S, M, HET, false, SHARED>), grid, block, 0, s, g, P, k, sh.tile, sh.nb,
                           sh.boxes, ZFaceArgs());
    return hipGetLastError();
}

// The sums of the off-axis normal terms are shared: cn[i][j] the same for
// both i != j, and on the read path (media outside the sums) for all three i.
// So lowered models are; with a sum per stress and axis a 256^3 step of 4th
// order takes 416 us instead of 394 on constant media and 532 instead of 527
// on the read path, where the gather kernel took 612 and 694.
template <typename R>
static bool shared_sums(const Coefs<R>& c, int M, bool het) {
    for (int j = 0; j < 3; ++j)
        for (int k = 0; k < M; ++k) {
            const R a = c.cn[(j + 1) % 3][j][k], b = c.cn[(j + 2) % 3][j][k];
            if (a != b || (het && a != c.cn[j][j][k])) return false;
        }
    return true;
}

template <typename R, typename S, int M, bool HET>
static hipError_t run_stress(const Geom& g, const FieldPtrs<S>& F, const MediaPtrs<R>& md, const Coefs<R>& c, int t0,
                             int t1, const InteriorLaunch& cfg, hipStream_t s, const ZFaceArgs* zf,
                             const Boxes* boxes) {
    auto launch = [&](auto k) {
        for (int a = 0; a < 3; ++a)
            for (int b = 0; b < 2; ++b)
                for (int i = 0; i < M; ++i) k.cs[a][b][i] = c.cs[a][b][i];
        return launch_shape<R, S, M, HET>(g, F, md, k, t0, t1, cfg, s, zf, boxes);
    };
    if (!shared_sums(c, M, HET)) {
        StressCoefs<R, false> k = {};
        for (int a = 0; a < 3; ++a)
            for (int j = 0; j < 3; ++j)
                for (int i = 0; i < M; ++i) k.n[a][j][i] = c.cn[a][j][i];
        return launch(k);
    }
    StressCoefs<R, true> k = {};
    for (int j = 0; j < 3; ++j)
        for (int i = 0; i < M; ++i) {
            k.own[j][i] = c.cn[j][j][i];
            k.off[j][i] = c.cn[(j + 1) % 3][j][i];
        }
    return launch(k);
}

template <typename R, typename S>
static hipError_t stress_m(const Geom& g, bool het, const void* fields, const void* media, const void* coefs, int t0,
                           int t1, const InteriorLaunch& cfg, hipStream_t s, const ZFaceArgs* zf, const Boxes* boxes) {
    const FieldPtrs<S>& F = *static_cast<const FieldPtrs<S>*>(fields);
    const MediaPtrs<R>& md = *static_cast<const MediaPtrs<R>*>(media);
    const Coefs<R>& c = *static_cast<const Coefs<R>*>(coefs);
#define OPESCI_CASE(MM)                                                                           \
    case MM:                                                                                      \
        return het ? run_stress<R, S, MM, true>(g, F, md, c, t0, t1, cfg, s, zf, boxes)           \
                   : run_stress<R, S, MM, false>(g, F, md, c, t0, t1, cfg, s, zf, boxes);
    switch (g.m) {
        OPESCI_CASE(1)
        OPESCI_CASE(2)
        OPESCI_CASE(3)
        OPESCI_CASE(4)
        default:
            return hipErrorInvalidValue;
    }
#undef OPESCI_CASE
}

hipError_t launch_stress_sweep(const Geom& g, int real_bytes, int storage, bool het, const void* fields,
                               const void* media, const void* coefs, int t0, int t1, const InteriorLaunch& cfg,
                               hipStream_t s, const ZFaceArgs* zf, const Boxes* boxes) {
    if (real_bytes == 8) return stress_m<double, double>(g, het, fields, media, coefs, t0, t1, cfg, s, zf, boxes);
    if (storage == OPESCI_STORE_F16)
        return stress_m<float, _Float16>(g, het, fields, media, coefs, t0, t1, cfg, s, zf, boxes);
    if (storage == OPESCI_STORE_BF16)
        return stress_m<float, bf16_t>(g, het, fields, media, coefs, t0, t1, cfg, s, zf, boxes);
    return stress_m<float, float>(g, het, fields, media, coefs, t0, t1, cfg, s, zf, boxes);
}

}  // namespace opesci
