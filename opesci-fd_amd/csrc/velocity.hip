// Velocity half step as a flat-tile x sweep (sweep.h): U, V, W at t1 from the
// stresses at t1 and the velocities at t0 (opesci/staggeredgrid.py:739-748).
// Stencil and accumulation order as in interior.hip; its gather kernel gives
// the same bits.
//
// What bounds it: as the stress sweep, the memory path on large grids (9
// reads and 3 writes per point, 48 bytes in FP32), the chain of one plane on
// small ones, instructions with 16-bit storage; 58-65 registers at 4th order
// in FP32.  Measured before (two points per lane in 128-point tiles, FP64 one)
// -> now (events, us; rows of 9 lines instead of 10 at 256^3): 256^3 4th order
// FP32 159 -> 154, read path 204 -> 181, FP16 142 -> 84, 8th order read path
// 222 -> 191; 160^3 93 -> 44; 161 x 129 x 193 8th order BF16 read path 89 ->
// 66; 61 x 47 x 53 8th order FP64 30 -> 12; 16^3 27 -> 7.
#include "sweep.h"

namespace opesci {

template <typename R>
struct VelocityCoefs {
    R cv[3][3][MAXM];
};
template <typename R, typename S>
struct VelocityPtrs {
    const S* t[6];     // Txx, Tyy, Tzz, Txy, Tyz, Txz at t1
    const S* v0[3];    // U, V, W at t0
    S* v1[3];          // the same at t1
    const R* beta[3];  // read path
};

template <typename R, typename S, int M, bool HET>
__global__ __launch_bounds__(SWEEP_THREADS, sizeof(R) * M <= 8 ? 5 : 2) void velocity_flat(
    Geom g, VelocityPtrs<R, S> P, VelocityCoefs<R> c, SweepTile T, int nblocks, Boxes B, int zero_last) {
    using C = Conv<S, R>;
    constexpr int Q = 2 * M;
    // planes: Tyy and Txy (y halo), Tzz and Txz (z halo), Tyz (both)
    __shared__ R lds[2][5][SweepPlane<M>::SIZE];
    const int l = sweep_block(nblocks);
    if (l < 0) return;
    const SweepLane s = sweep_lane<M>(g, B, l, T);
    const int64_t x0 = (int64_t)s.xb * g.sx;
    const S* bt[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) bt[f] = P.t[f] + x0;
    const S* b0[3];
    S* b1[3];
    const R* bm[3] = {nullptr, nullptr, nullptr};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        b0[i] = P.v0[i] + x0;
        b1[i] = P.v1[i] + x0;
        if (HET) bm[i] = P.beta[i] + x0;
    }
    const uint32_t plane = (uint32_t)g.sx * sizeof(S);
    uint32_t own = s.own * sizeof(S), oy = s.gy * sizeof(S), oz = s.gz * sizeof(S), ox = s.gx * sizeof(S),
             om = s.own * sizeof(R);
    // register queues, logical element i at slot (phase + i) % Q:
    // Txx(x + i - M + 1), Txy(x + i - M), Txz(x + i - M)
    R qXX[Q], qXY[Q], qXZ[Q];
#pragma unroll
    for (int i = 0; i < Q - 1; ++i) {
        qXX[i] = C::ldnt(at_byte(bt[0] + (int64_t)(i - M + 1) * g.sx, own));
        qXY[i] = C::ld(at_byte(bt[3] + (int64_t)(i - M) * g.sx, own));
        qXZ[i] = C::ld(at_byte(bt[5] + (int64_t)(i - M) * g.sx, own));
    }
    const S* aXX = bt[0] + (int64_t)M * g.sx;
    const S* aXY = bt[3] + (int64_t)(M - 1) * g.sx;
    const S* aXZ = bt[5] + (int64_t)(M - 1) * g.sx;
    // the next plane's values, loaded one plane ahead
    R nXX, nXY, nXZ, nYY, nZZ, nYZ, nv[3], nm[3], yYY, yXY, yYZ, zZZ, zXZ, zYZ, xYY, xXY, xYZ;
    auto fetch = [&]() __attribute__((always_inline)) {
        if (s.hy) {
            yYY = C::ld(at_byte(bt[1], oy));
            yXY = C::ld(at_byte(bt[3], oy));
            yYZ = C::ld(at_byte(bt[4], oy));
        }
        if (sweep_second_halo<M>() && s.hx) {
            xYY = C::ld(at_byte(bt[1], ox));
            xXY = C::ld(at_byte(bt[3], ox));
            xYZ = C::ld(at_byte(bt[4], ox));
        }
        if (s.hz) {
            zZZ = C::ld(at_byte(bt[2], oz));
            zXZ = C::ld(at_byte(bt[5], oz));
            zYZ = C::ld(at_byte(bt[4], oz));
        }
        nXY = C::ld(at_byte(aXY, own));
        nXZ = C::ld(at_byte(aXZ, own));
        nYY = C::ld(at_byte(bt[1], own));
        nZZ = C::ld(at_byte(bt[2], own));
        nYZ = C::ld(at_byte(bt[4], own));
        nXX = C::ldnt(at_byte(aXX, own));   // read along x only: streamed once
#pragma unroll
        for (int i = 0; i < 3; ++i) nv[i] = C::ldnt(at_byte(b0[i], own));
        if (HET) {
#pragma unroll
            for (int i = 0; i < 3; ++i) nm[i] = Conv<R, R>::ldnt(at_byte(bm[i], om));
        }
    };
    fetch();
    const int pitch = s.pitch;
    const bool zero_v = (zero_last & 2) && s.y == g.ny - M - 1, zero_w = (zero_last & 4) && s.z == g.nz - M - 1;
    auto step = [&](auto phase, int x) __attribute__((always_inline)) {
        constexpr int PH = decltype(phase)::value, b = PH & 1;
        auto q = [](int i) constexpr { return (PH + i) % Q; };
        qXX[q(Q - 1)] = nXX;
        qXY[q(Q - 1)] = nXY;
        qXZ[q(Q - 1)] = nXZ;
        const R v0[3] = {nv[0], nv[1], nv[2]}, oYY = nYY, oZZ = nZZ, oYZ = nYZ;
        R md[3] = {0, 0, 0};
        if (HET) {
#pragma unroll
            for (int i = 0; i < 3; ++i) md[i] = nm[i];
        }
        R* LYY = lds[b][0];
        R* LXY = lds[b][1];
        R* LYZ = lds[b][2];
        R* LZZ = lds[b][3];
        R* LXZ = lds[b][4];
        if (s.on) {
            LYY[s.me] = oYY;
            LXY[s.me] = qXY[q(M)];
            LYZ[s.me] = oYZ;
            LZZ[s.me] = oZZ;
            LXZ[s.me] = qXZ[q(M)];
        }
        if (s.hy) {
            LYY[s.ly] = yYY;
            LXY[s.ly] = yXY;
            LYZ[s.ly] = yYZ;
        }
        if (sweep_second_halo<M>() && s.hx) {
            LYY[s.lx] = xYY;
            LXY[s.lx] = xXY;
            LYZ[s.lx] = xYZ;
        }
        if (s.hz) {
            LYZ[s.lz] = zYZ;
            LZZ[s.lz] = zZZ;
            LXZ[s.lz] = zXZ;
        }
        const uint32_t here = own;
        if (x + 1 < s.xe) {
            own += plane;
            oy += plane;
            oz += plane;
            ox += plane;
            om += (uint32_t)g.sx * sizeof(R);
            fetch();
        }
        lds_barrier();
        if (s.on) {
            const R oXY = qXY[q(M)], oXZ = qXZ[q(M)];
            R su = 0, sv = 0, sw = 0;
#pragma unroll
            for (int k = 0; k < M; ++k) su = fma(c.cv[0][0][k], qXX[q(M + k)] - qXX[q(M - 1 - k)], su);
#pragma unroll
            for (int k = 0; k < M; ++k)
                su = fma(c.cv[0][1][k], (k == 0 ? oXY : LXY[s.me + k * pitch]) - LXY[s.me - (1 + k) * pitch], su);
#pragma unroll
            for (int k = 0; k < M; ++k)
                su = fma(c.cv[0][2][k], (k == 0 ? oXZ : LXZ[s.me + k]) - LXZ[s.me - 1 - k], su);
#pragma unroll
            for (int k = 0; k < M; ++k) sv = fma(c.cv[1][0][k], qXY[q(M + k)] - qXY[q(M - 1 - k)], sv);
#pragma unroll
            for (int k = 0; k < M; ++k)
                sv = fma(c.cv[1][1][k], LYY[s.me + (1 + k) * pitch] - (k == 0 ? oYY : LYY[s.me - k * pitch]), sv);
#pragma unroll
            for (int k = 0; k < M; ++k)
                sv = fma(c.cv[1][2][k], (k == 0 ? oYZ : LYZ[s.me + k]) - LYZ[s.me - 1 - k], sv);
#pragma unroll
            for (int k = 0; k < M; ++k) sw = fma(c.cv[2][0][k], qXZ[q(M + k)] - qXZ[q(M - 1 - k)], sw);
#pragma unroll
            for (int k = 0; k < M; ++k)
                sw = fma(c.cv[2][1][k], (k == 0 ? oYZ : LYZ[s.me + k * pitch]) - LYZ[s.me - (1 + k) * pitch], sw);
#pragma unroll
            for (int k = 0; k < M; ++k)
                sw = fma(c.cv[2][2][k], LZZ[s.me + 1 + k] - (k == 0 ? oZZ : LZZ[s.me - k]), sw);
            const R sum[3] = {su, sv, sw};
            const bool zero[3] = {(zero_last & 1) && x == g.nx - M - 1, zero_v, zero_w};
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const R v = HET ? fma(md[i], sum[i], v0[i]) : v0[i] + sum[i];
                C::stnt(at_byte(b1[i], here), zero[i] ? (R)0 : v);
            }
        }
    };
    sweep_planes(s.xb, s.xe, step, std::make_integer_sequence<int, Q>{});
}

// ------------------------------------------------------------------ launch
template <typename R, typename S, int M, bool HET>
static hipError_t run_velocity(const Geom& g, const FieldPtrs<S>& F, const MediaPtrs<R>& md, const Coefs<R>& c, int t0,
                               int t1, const InteriorLaunch& cfg, hipStream_t s, const Boxes* boxes,
                               int zero_last) {
    static std::atomic<int> occ[SWEEP_THREADS / 64 + 1] = {};
    // 9 reads and 3 writes of the storage type, 3 media
    const SweepShape sh = sweep_shape<M>(
        g, cfg, boxes, 12 * (int)sizeof(S) + (HET ? 3 * (int)sizeof(R) : 0), sizeof(S),
        [&](int threads) { return sweep_blocks_per_cu(velocity_flat<R, S, M, HET>, occ, threads); });
    if (sh.nb == 0) return hipSuccess;
    VelocityPtrs<R, S> P;
    for (int f = 0; f < 6; ++f) P.t[f] = F.f[3 + f][t1];
    for (int i = 0; i < 3; ++i) {
        P.v0[i] = F.f[i][t0];
        P.v1[i] = F.f[i][t1];
        P.beta[i] = md.m[OPESCI_M_BETA1 + i];
    }
    VelocityCoefs<R> k = {};
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j)
            for (int a = 0; a < M; ++a) k.cv[i][j][a] = c.cv[i][j][a];
    hipLaunchKernelGGL((velocity_flat<R, S, M, HET>), dim3((unsigned)((sh.nb + 7) / 8 * 8)), dim3((unsigned)sh.threads),
                       0, s, g, P, k, sh.tile, sh.nb, sh.boxes, zero_last);
    return hipGetLastError();
}

template <typename R, typename S>
static hipError_t velocity_m(const Geom& g, bool het, const void* fields, const void* media, const void* coefs, int t0,
                             int t1, const InteriorLaunch& cfg, hipStream_t s, const Boxes* boxes, int zero_last) {
    const FieldPtrs<S>& F = *static_cast<const FieldPtrs<S>*>(fields);
    const MediaPtrs<R>& md = *static_cast<const MediaPtrs<R>*>(media);
    const Coefs<R>& c = *static_cast<const Coefs<R>*>(coefs);
#define OPESCI_CASE(MM)                                                                       \
    case MM:                                                                                  \
        return het ? run_velocity<R, S, MM, true>(g, F, md, c, t0, t1, cfg, s, boxes, zero_last)         \
                   : run_velocity<R, S, MM, false>(g, F, md, c, t0, t1, cfg, s, boxes, zero_last);
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

hipError_t launch_velocity_sweep(const Geom& g, int real_bytes, int storage, bool het, const void* fields,
                                 const void* media, const void* coefs, int t0, int t1, const InteriorLaunch& cfg,
                                 hipStream_t s, const Boxes* boxes, int zero_last) {
    if (real_bytes == 8)
        return velocity_m<double, double>(g, het, fields, media, coefs, t0, t1, cfg, s, boxes, zero_last);
    if (storage == OPESCI_STORE_F16)
        return velocity_m<float, _Float16>(g, het, fields, media, coefs, t0, t1, cfg, s, boxes, zero_last);
    if (storage == OPESCI_STORE_BF16)
        return velocity_m<float, bf16_t>(g, het, fields, media, coefs, t0, t1, cfg, s, boxes, zero_last);
    return velocity_m<float, float>(g, het, fields, media, coefs, t0, t1, cfg, s, boxes, zero_last);
}

}  // namespace opesci
