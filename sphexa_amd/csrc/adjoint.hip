// Adjoint (vector-Jacobian product) kernels of the std density, IAD and momentum-energy passes.
//
// No counterpart in the reference. Each kernel walks the neighbour lists of the last search
// (held fixed: they are the checkpoint of the forward), recomputes the pair terms of its forward
// loop and accumulates the reverse-mode derivatives. A pair term of target i and neighbour j has
// derivatives for both. The target's are summed over its list (the ...VjpKernel of a pass). The
// neighbour's are summed by the neighbour: the pair index (AdjointPairs) lists for every particle j the
// targets that have j as neighbour, in increasing order, and the ...VjpSourceKernel walks them and
// forms each pair again from the target's side. No pair is written to memory and no atomics are
// used; results are the same bit for bit from run to run.
//
// Both walks read the other particle as one record (16-byte chunks, packed by the call for every
// particle; positions in FP64, which form the separations of both forms). What bounds them: the
// gathers of the records, one tag lookup of the vector cache per lane and chunk (about 0.23 ms per
// chunk at 2M particles), and the FP64 kernel evaluations. Measured at 2M particles, mixed form, with
// each pair's neighbour side written to memory and summed afterwards, and with this (ms):
// density 6.2 -> 1.8, IAD 6.3 -> 2.4, momentum-energy 13.7 -> 4.4.
// Kernel derivatives use the tabulated dW/dv interpolated like W (FP64) or are
// evaluated like W (FP32). Launch shape and list layout as the forward loops (pairs.hpp).
// Derivations, with r = x_i - x_j after the fold, d = |r|, v = d / h_i:
//
//  density   rho_i = K h_i^-3 (m_i + sum_j m_j W(v))
//            d/dr = K h_i^-4 m_j W'(v) r/d,   d/dh_i = -K h_i^-4 (3 rho0_i + sum_j m_j v W'(v))
//  IAD       C_i = h_i^3/K tau_i^-1, tau_i = sum_j V_j W(v) r r^T, V_j = m_j/rho_j; with G the
//            matrix cotangent of C_i (a stored off-diagonal entry stands for two matrix entries):
//            tauBar = -(K/h_i^3) C_i G C_i, dL/dh_i += 3/h_i tr(G C_i); per pair q = r^T tauBar r:
//            d/dr = V_j (W'(v) q r/(h_i d) + 2 W(v) tauBar r), d/dh_i = -V_j W'(v) q d/h_i^2,
//            d/drho_j = -m_j/rho_j^2 W(v) q
//  momentum  reverse mode through the pair term of hydro_std/momentum_energy_kern.hpp:11-134 with
//            a per-particle AV coefficient (the reference's is the constant 1):
//            a_i = K sum_j (aa C_i r + bb C_j r), du_i = -K/2 sum_j v_ij.(ae C_i r + be C_j r)
#include <cstring> // rocprim uses memset without including it
#include <rocprim/rocprim.hpp>

#include "pairs.hpp"

namespace sphx
{

namespace
{

constexpr unsigned kPackThreads = 256;

//! the target's own gradient: one lane per target, so a plain read-modify-write
template<class T>
__device__ __forceinline__ void addOwn(void* p, uint32_t i, T v)
{
    static_cast<T*>(p)[i] += v;
}

//! the targets of every particle (AdjointPairs) and the call's range of them
struct SourceRows
{
    const uint32_t *rowStart, *targets;
    uint32_t        first, last, n;
};

//! the particle of this lane, one wave per 64 consecutive particles
__device__ __forceinline__ uint32_t sourceParticle()
{
    const uint32_t g = __builtin_amdgcn_readfirstlane(xcdBlock(blockIdx.x, gridDim.x) * kVjpWaves + threadIdx.x / kWave);
    return g * kWave + laneId();
}

/*! pair(rec[i]) for every target i of the call that has j as neighbour, in increasing order: U targets and their
 * records in flight. A slot past the row reads the next row's target (the index is padded by a quad). */
template<int U, class Rec, class F>
__device__ __forceinline__ void overTargets(const SourceRows& R, uint32_t j, const Rec* __restrict__ rec, F&& pair)
{
    constexpr int   NC    = int(sizeof(Rec) / 16);
    const uint32_t  count = R.rowStart[j + 1] - R.rowStart[j];
    const uint32_t* row   = R.targets + R.rowStart[j];
    uint32_t        next[U];
    __builtin_memcpy(next, row, sizeof(next));
    for (uint32_t k = 0; k < count; k += U)
    {
        uint32_t i[U];
        uint4    w[U][NC];
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            i[u]             = next[u];
            const uint4* src = reinterpret_cast<const uint4*>(rec + i[u]);
#pragma unroll
            for (int c = 0; c < NC; ++c)
                w[u][c] = src[c];
        }
        __builtin_memcpy(next, row + min(k + U, count), sizeof(next));
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
#pragma unroll
            for (int c = 0; c < NC; ++c)
                asm volatile("" : "+v"(w[u][c].x)); // the batch's loads stay above the branches
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            if (k + u < count && i[u] >= R.first && i[u] < R.last)
            {
                Rec r;
                __builtin_memcpy(&r, w[u], sizeof(r));
                pair(r);
            }
        }
    }
}

//! separation x_i - x_j for a neighbour j that does not know whether its targets' separations wrap: the fold, with
//! the target's cut-off r, only where some lane's does
template<class T>
__device__ __forceinline__ void sourceSeparation(const DevBox& b, double r, double xi, double yi, double zi, double xj,
                                                 double yj, double zj, T& rx, T& ry, T& rz)
{
    const bool wraps = (b.pbc[0] && fabs(xi - xj) > r) || (b.pbc[1] && fabs(yi - yj) > r) || (b.pbc[2] && fabs(zi - zj) > r);
    if (ballot(wraps)) { separation<true>(b, r, xi, yi, zi, xj, yj, zj, rx, ry, rz); }
    else { separation<false>(b, r, xi, yi, zi, xj, yj, zj, rx, ry, rz); }
}

template<class T>
__device__ __forceinline__ T pow4Inv(T hInv)
{
    T h2 = hInv * hInv;
    return h2 * h2;
}

struct DensityVjpArgs
{
    const void *h, *m, *gRho;
    void *      gx, *gy, *gz, *gh;
};

//! a neighbour for the target's sums, and a target for the neighbour's
template<class T>
struct alignas(16) RecDensityVjpJ
{
    double x, y, z;
    T      m;
};
template<class T>
struct alignas(16) RecDensityVjpI
{
    double x, y, z;
    T      h, coef; // coef: K h^-4 times the cotangent of rho
};

template<class T>
__device__ __forceinline__ T densityVjpCoef(const PairArgs& a, const DensityVjpArgs& f, uint32_t i, T hInv)
{
    return ld<T>(f.gRho, i) * T(a.K) * pow4Inv(hInv);
}

template<class T>
__global__ void __launch_bounds__(kPackThreads)
    packDensityVjp(PairArgs a, DensityVjpArgs f, uint32_t first, uint32_t last, RecDensityVjpJ<T>* __restrict__ recJ,
                   RecDensityVjpI<T>* __restrict__ recI, uint32_t n)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) { return; }
    const double x = a.x[k], y = a.y[k], z = a.z[k];
    recJ[k] = {x, y, z, ld<T>(f.m, k)};
    if (k < first || k >= last) { return; }
    const T h = ld<T>(f.h, k);
    recI[k]   = {x, y, z, h, densityVjpCoef<T>(a, f, k, T(1) / h)};
}

template<class T>
__global__ void __launch_bounds__(kVjpWaves * kWave)
    densityStdVjpKernel(PairArgs a, DensityVjpArgs f, SincKernel<T> kern, const RecDensityVjpJ<T>* __restrict__ rec)
{
    const Lane t = vjpTarget(a.L);
    if (!t.valid) { return; }
    const uint32_t i    = t.i;
    const T        hi   = ld<T>(f.h, i);
    const T        hInv = T(1) / hi;
    const double   r2h  = 2.0 * double(hi);
    const double   xi = a.x[i], yi = a.y[i], zi = a.z[i];
    const T        coef = densityVjpCoef<T>(a, f, i, hInv);
    T              rho0 = ld<T>(f.m, i), sumVdW = 0, gxi = 0, gyi = 0, gzi = 0;
    withFold(waveNeedsFold(a.box, xi, yi, zi, r2h), [&](auto fold) {
        // a quad of neighbours at a time: their list entries and records load before any is used
        constexpr int U = 4;
        const TargetList list = a.L.lists.list(t.r);
        for (unsigned k0 = 0; k0 < t.n; k0 += U)
        {
            uint32_t j[U];
            list.quad(k0, j);
            RecDensityVjpJ<T> rj[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                rj[u] = rec[j[u]];
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                if (k0 + u >= t.n) { break; }
                T rx, ry, rz;
                separation<decltype(fold)::value>(a.box, r2h, xi, yi, zi, rj[u].x, rj[u].y, rj[u].z, rx, ry, rz);
                T d = sqrt(rx * rx + ry * ry + rz * rz);
                T v = d * hInv;
                T w, dw;
                kern.wAndDw(v, w, dw);
                rho0 += rj[u].m * w;
                sumVdW += rj[u].m * v * dw;
                T c = d > T(0) ? coef * rj[u].m * dw / d : T(0);
                gxi += c * rx, gyi += c * ry, gzi += c * rz;
            }
        }
    });
    addOwn<T>(f.gx, i, gxi), addOwn<T>(f.gy, i, gyi), addOwn<T>(f.gz, i, gzi);
    addOwn<T>(f.gh, i, -coef * (T(3) * rho0 + sumVdW));
}

template<class T>
__global__ void __launch_bounds__(kVjpWaves * kWave)
    densityStdVjpSourceKernel(PairArgs a, DensityVjpArgs f, SincKernel<T> kern, SourceRows rows,
                              const RecDensityVjpI<T>* __restrict__ rec)
{
    const uint32_t j = sourceParticle();
    if (j >= rows.n) { return; }
    const double xj = a.x[j], yj = a.y[j], zj = a.z[j];
    const T      mj = ld<T>(f.m, j);
    T            gx = 0, gy = 0, gz = 0;
    overTargets<4>(rows, j, rec, [&](const RecDensityVjpI<T>& ri) {
        T rx, ry, rz;
        sourceSeparation(a.box, 2.0 * double(ri.h), ri.x, ri.y, ri.z, xj, yj, zj, rx, ry, rz);
        T d = sqrt(rx * rx + ry * ry + rz * rz);
        T w, dw;
        kern.wAndDw(d * (T(1) / ri.h), w, dw);
        T c = d > T(0) ? ri.coef * mj * dw / d : T(0);
        gx -= c * rx, gy -= c * ry, gz -= c * rz;
    });
    addOwn<T>(f.gx, j, gx), addOwn<T>(f.gy, j, gy), addOwn<T>(f.gz, j, gz);
}

struct IadVjpArgs
{
    const void *h, *m, *rho, *c[6], *g[6];
    void *      gx, *gy, *gz, *gh, *grho;
};

//! a neighbour for the target's sums, and a target for the neighbour's
template<class T>
struct alignas(16) RecIadVjpJ
{
    double x, y, z;
    T      m, rho;
};
template<class T>
struct alignas(16) RecIadVjpI
{
    double x, y, z;
    T      h, B[9]; // B: tauBar
};

//! tauBar = -(K/h^3) C G C of target i; returns 3/h tr(G C)
template<class T>
__device__ __forceinline__ T iadVjpTarget(const PairArgs& a, const IadVjpArgs& f, uint32_t i, T hInv, T (&B)[9])
{
    T C6[6], G6[6];
    for (int q = 0; q < 6; ++q)
        C6[q] = ld<T>(f.c[q], i), G6[q] = ld<T>(f.g[q], i);
    const T C[3][3] = {{C6[0], C6[1], C6[2]}, {C6[1], C6[3], C6[4]}, {C6[2], C6[4], C6[5]}};
    const T G[3][3] = {{G6[0], G6[1] / 2, G6[2] / 2}, {G6[1] / 2, G6[3], G6[4] / 2}, {G6[2] / 2, G6[4] / 2, G6[5]}};
    T       CG[3][3];
    for (int p = 0; p < 3; ++p)
        for (int q = 0; q < 3; ++q)
            CG[p][q] = C[p][0] * G[0][q] + C[p][1] * G[1][q] + C[p][2] * G[2][q];
    const T s = -T(a.K) * hInv * hInv * hInv;
    for (int p = 0; p < 3; ++p)
        for (int q = 0; q < 3; ++q)
            B[3 * p + q] = s * (CG[p][0] * C[0][q] + CG[p][1] * C[1][q] + CG[p][2] * C[2][q]);
    return T(3) * hInv *
           (G6[0] * C6[0] + G6[1] * C6[1] + G6[2] * C6[2] + G6[3] * C6[3] + G6[4] * C6[4] + G6[5] * C6[5]);
}

template<class T>
__global__ void __launch_bounds__(kPackThreads)
    packIadVjp(PairArgs a, IadVjpArgs f, uint32_t first, uint32_t last, RecIadVjpJ<T>* __restrict__ recJ,
               RecIadVjpI<T>* __restrict__ recI, uint32_t n)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) { return; }
    const double x = a.x[k], y = a.y[k], z = a.z[k];
    recJ[k] = {x, y, z, ld<T>(f.m, k), ld<T>(f.rho, k)};
    if (k < first || k >= last) { return; }
    RecIadVjpI<T> r{x, y, z, ld<T>(f.h, k), {}};
    iadVjpTarget<T>(a, f, k, T(1) / r.h, r.B);
    recI[k] = r;
}

template<class T>
__global__ void __launch_bounds__(kVjpWaves * kWave)
    iadStdVjpKernel(PairArgs a, IadVjpArgs f, SincKernel<T> kern, const RecIadVjpJ<T>* __restrict__ rec)
{
    const Lane t = vjpTarget(a.L);
    if (!t.valid) { return; }
    const uint32_t i    = t.i;
    const T        hi   = ld<T>(f.h, i);
    const T        hInv = T(1) / hi;
    const double   r2h  = 2.0 * double(hi);
    const double   xi = a.x[i], yi = a.y[i], zi = a.z[i];

    T B[9];
    T ghi = iadVjpTarget<T>(a, f, i, hInv, B);
    T gxi = 0, gyi = 0, gzi = 0;
    withFold(waveNeedsFold(a.box, xi, yi, zi, r2h), [&](auto fold) {
        // a quad of neighbours at a time: their list entries and records load before any is used
        constexpr int U = 4;
        const TargetList list = a.L.lists.list(t.r);
        for (unsigned k0 = 0; k0 < t.n; k0 += U)
        {
            uint32_t j[U];
            list.quad(k0, j);
            RecIadVjpJ<T> rj[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                rj[u] = rec[j[u]];
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                if (k0 + u >= t.n) { break; }
                T r[3];
                separation<decltype(fold)::value>(a.box, r2h, xi, yi, zi, rj[u].x, rj[u].y, rj[u].z, r[0], r[1], r[2]);
                T d = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
                T v = d * hInv;
                T w, dw;
                kern.wAndDw(v, w, dw);
                T Vj = rj[u].m / rj[u].rho;
                T Br[3];
                for (int p = 0; p < 3; ++p)
                    Br[p] = B[3 * p] * r[0] + B[3 * p + 1] * r[1] + B[3 * p + 2] * r[2];
                T q      = r[0] * Br[0] + r[1] * Br[1] + r[2] * Br[2];
                T radial = d > T(0) ? Vj * dw * q * hInv / d : T(0);
                gxi += radial * r[0] + T(2) * Vj * w * Br[0];
                gyi += radial * r[1] + T(2) * Vj * w * Br[1];
                gzi += radial * r[2] + T(2) * Vj * w * Br[2];
                ghi += -Vj * dw * q * d * hInv * hInv;
            }
        }
    });
    addOwn<T>(f.gx, i, gxi), addOwn<T>(f.gy, i, gyi), addOwn<T>(f.gz, i, gzi);
    addOwn<T>(f.gh, i, ghi);
}

template<class T>
__global__ void __launch_bounds__(kVjpWaves * kWave)
    iadStdVjpSourceKernel(PairArgs a, IadVjpArgs f, SincKernel<T> kern, SourceRows rows,
                          const RecIadVjpI<T>* __restrict__ rec)
{
    const uint32_t j = sourceParticle();
    if (j >= rows.n) { return; }
    const double xj = a.x[j], yj = a.y[j], zj = a.z[j];
    const T      mj = ld<T>(f.m, j), rhoj = ld<T>(f.rho, j), Vj = mj / rhoj;
    T            gx = 0, gy = 0, gz = 0, wq = 0;
    overTargets<isMixed<T> ? 4 : 2>(rows, j, rec, [&](const RecIadVjpI<T>& ri) {
        T r[3];
        sourceSeparation(a.box, 2.0 * double(ri.h), ri.x, ri.y, ri.z, xj, yj, zj, r[0], r[1], r[2]);
        const T hInv = T(1) / ri.h;
        T       d    = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
        T       w, dw;
        kern.wAndDw(d * hInv, w, dw);
        T Br[3];
        for (int p = 0; p < 3; ++p)
            Br[p] = ri.B[3 * p] * r[0] + ri.B[3 * p + 1] * r[1] + ri.B[3 * p + 2] * r[2];
        T q      = r[0] * Br[0] + r[1] * Br[1] + r[2] * Br[2];
        T radial = d > T(0) ? Vj * dw * q * hInv / d : T(0);
        gx -= radial * r[0] + T(2) * Vj * w * Br[0];
        gy -= radial * r[1] + T(2) * Vj * w * Br[1];
        gz -= radial * r[2] + T(2) * Vj * w * Br[2];
        wq += w * q;
    });
    addOwn<T>(f.gx, j, gx), addOwn<T>(f.gy, j, gy), addOwn<T>(f.gz, j, gz);
    addOwn<T>(f.grho, j, -mj / (rhoj * rhoj) * wq);
}

struct MomVjpArgs
{
    const void *vx, *vy, *vz, *h, *m, *rho, *p, *c, *alpha, *C[6];
    const void *gax, *gay, *gaz, *gdu;
    void *      gx, *gy, *gz, *gh, *grho, *gp, *galpha, *gC[6];
};

//! stored-entry cotangent of a symmetric matrix used as M r, from the matrix cotangent u r^T
template<class T>
__device__ __forceinline__ void symOuter(const T u[3], const T r[3], T out[6])
{
    out[0] = u[0] * r[0];
    out[1] = u[0] * r[1] + u[1] * r[0];
    out[2] = u[0] * r[2] + u[2] * r[0];
    out[3] = u[1] * r[1];
    out[4] = u[1] * r[2] + u[2] * r[1];
    out[5] = u[2] * r[2];
}

//! what both sides of a pair need of a particle
template<class T>
struct MomVjpParticle
{
    double x, y, z;
    T      vx, vy, vz, h, c, alpha, C[6];
};
//! a neighbour for the target's sums, and a target for the neighbour's
template<class T>
struct alignas(16) RecMomVjpJ
{
    MomVjpParticle<T> p;
    T                 vol, m, prj; // vol: m / rho, prj: p / rho
};
template<class T>
struct alignas(16) RecMomVjpI
{
    MomVjpParticle<T> p;
    T                 vol, pro, ge, Ga[3]; // pro: p / rho^2; Ga, ge: K times the cotangents of a, -K/2 times that of du
};

template<class T>
__device__ __forceinline__ MomVjpParticle<T> loadMomVjp(const PairArgs& a, const MomVjpArgs& f, uint32_t k)
{
    MomVjpParticle<T> r{a.x[k],
                        a.y[k],
                        a.z[k],
                        ld<T>(f.vx, k),
                        ld<T>(f.vy, k),
                        ld<T>(f.vz, k),
                        ld<T>(f.h, k),
                        ld<T>(f.c, k),
                        f.alpha ? ld<T>(f.alpha, k) : T(1),
                        {}};
    for (int q = 0; q < 6; ++q)
        r.C[q] = ld<T>(f.C[q], k);
    return r;
}

template<class T>
__device__ __forceinline__ RecMomVjpJ<T> loadMomVjpJ(const PairArgs& a, const MomVjpArgs& f, uint32_t k)
{
    const T rho = ld<T>(f.rho, k), m = ld<T>(f.m, k);
    return {loadMomVjp<T>(a, f, k), m / rho, m, ld<T>(f.p, k) / rho};
}

template<class T>
__device__ __forceinline__ RecMomVjpI<T> loadMomVjpI(const PairArgs& a, const MomVjpArgs& f, uint32_t k)
{
    const T rho = ld<T>(f.rho, k);
    return {loadMomVjp<T>(a, f, k),
            ld<T>(f.m, k) / rho,
            ld<T>(f.p, k) / (rho * rho),
            f.gdu ? -T(a.K) * T(0.5) * ld<T>(f.gdu, k) : T(0),
            {T(a.K) * ld<T>(f.gax, k), T(a.K) * ld<T>(f.gay, k), T(a.K) * ld<T>(f.gaz, k)}};
}

template<class T>
__global__ void __launch_bounds__(kPackThreads)
    packMomVjp(PairArgs a, MomVjpArgs f, uint32_t first, uint32_t last, RecMomVjpJ<T>* __restrict__ recJ,
               RecMomVjpI<T>* __restrict__ recI, uint32_t n)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) { return; }
    recJ[k] = loadMomVjpJ<T>(a, f, k);
    if (k >= first && k < last) { recI[k] = loadMomVjpI<T>(a, f, k); }
}

//! C r of a symmetric matrix by its stored entries
template<class T>
__device__ __forceinline__ void symTimes(const T (&C)[6], const T (&r)[3], T (&out)[3])
{
    out[0] = C[0] * r[0] + C[1] * r[1] + C[2] * r[2];
    out[1] = C[1] * r[0] + C[3] * r[1] + C[4] * r[2];
    out[2] = C[2] * r[0] + C[4] * r[1] + C[5] * r[2];
}

//! reverse-mode derivatives of one pair term of target i and neighbour j; each side uses its own
template<class T>
struct MomPairBar
{
    T r[3];                // by x_i (and, negated, by x_j)
    T hi, hj, alpha;       // by h_i, h_j, and by either alpha
    T tAi[3], tAj[3];      // by C_i r and C_j r
    T pro, volI, volJ, prj; // by p_i / rho_i^2, the volumes, and p_j / rho_j
};

template<class T>
__device__ __forceinline__ MomPairBar<T> momPairBar(const SincKernel<T>& kern, const RecMomVjpI<T>& I,
                                                    const RecMomVjpJ<T>& J, const T (&r)[3], T hiInv, T hjInv)
{
    const MomVjpParticle<T>&i = I.p, &j = J.p;
    T d      = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
    T dInv   = d > T(0) ? T(1) / d : T(0);
    T vij[3] = {i.vx - j.vx, i.vy - j.vy, i.vz - j.vz};
    T hiInv3 = hiInv * hiInv * hiInv, hjInv3 = hjInv * hjInv * hjInv;
    T v1 = d * hiInv, v2 = d * hjInv;
    T W1, dW1, W2, dW2;
    kern.wAndDw(v1, W1, dW1);
    kern.wAndDw(v2, W2, dW2);
    T Wi = hiInv3 * W1, Wj = hjInv3 * W2;
    T tAi[3], tAj[3];
    symTimes(i.C, r, tAi);
    symTimes(j.C, r, tAj);
    T w    = (r[0] * vij[0] + r[1] * vij[1] + r[2] * vij[2]) * dInv;
    T visc = 0, dvisc_dw = 0, dvisc_dalpha = 0;
    if (w < T(0))
    {
        T a4         = (i.alpha + j.alpha) / T(4) * (i.c + j.c);
        visc         = T(0.5) * (-(a4 - T(2) * w) * w);
        dvisc_dw     = T(0.5) * (-a4 + T(4) * w);
        dvisc_dalpha = T(0.5) * (-(i.c + j.c) / T(4) * w);
    }
    T aa = Wi * (J.m * I.pro + visc * I.vol);
    T bb = J.vol * Wj * (J.prj + visc);
    T ae = Wi * (T(2) * J.m * I.pro + visc * I.vol);
    T be = visc * J.vol * Wj;

    T aaBar = I.Ga[0] * tAi[0] + I.Ga[1] * tAi[1] + I.Ga[2] * tAi[2];
    T bbBar = I.Ga[0] * tAj[0] + I.Ga[1] * tAj[1] + I.Ga[2] * tAj[2];
    T aeBar = I.ge * (vij[0] * tAi[0] + vij[1] * tAi[1] + vij[2] * tAi[2]);
    T beBar = I.ge * (vij[0] * tAj[0] + vij[1] * tAj[1] + vij[2] * tAj[2]);

    MomPairBar<T> o;
    for (int p = 0; p < 3; ++p)
    {
        o.tAi[p] = aa * I.Ga[p] + I.ge * ae * vij[p];
        o.tAj[p] = bb * I.Ga[p] + I.ge * be * vij[p];
    }
    T fromI[3], fromJ[3];
    symTimes(i.C, o.tAi, fromI);
    symTimes(j.C, o.tAj, fromJ);

    T WiBar = aaBar * (J.m * I.pro + visc * I.vol) + aeBar * (T(2) * J.m * I.pro + visc * I.vol);
    T WjBar = bbBar * J.vol * (J.prj + visc) + beBar * visc * J.vol;
    o.pro   = (aaBar + T(2) * aeBar) * Wi * J.m;
    o.volI  = (aaBar + aeBar) * Wi * visc;
    o.volJ  = bbBar * Wj * (J.prj + visc) + beBar * visc * Wj;
    o.prj   = bbBar * J.vol * Wj;
    T viscBar = (aaBar + aeBar) * Wi * I.vol + (bbBar + beBar) * J.vol * Wj;
    T wBar    = viscBar * dvisc_dw;
    o.alpha   = viscBar * dvisc_dalpha;
    T dBar    = WiBar * hiInv3 * hiInv * dW1 + WjBar * hjInv3 * hjInv * dW2;
    T radial  = (dBar - wBar * w * dInv) * dInv, along = wBar * dInv;
    for (int p = 0; p < 3; ++p)
        o.r[p] = fromI[p] + fromJ[p] + (radial * r[p] + along * vij[p]);
    o.hi = -WiBar * hiInv3 * hiInv * (T(3) * W1 + v1 * dW1);
    o.hj = -WjBar * hjInv3 * hjInv * (T(3) * W2 + v2 * dW2);
    return o;
}

template<class T>
__global__ void __launch_bounds__(kVjpWaves * kWave)
    momentumStdVjpKernel(PairArgs a, MomVjpArgs f, SincKernel<T> kern, const RecMomVjpJ<T>* __restrict__ rec)
{
    const Lane t = vjpTarget(a.L);
    if (!t.valid) { return; }
    const uint32_t      i     = t.i;
    const RecMomVjpI<T> I     = loadMomVjpI<T>(a, f, i);
    const T             hiInv = T(1) / I.p.h;
    const double        r2h   = 2.0 * double(I.p.h);

    T gr[3] = {0, 0, 0}, gh = 0, galpha = 0, pro = 0, vol = 0;
    T gC[6] = {0, 0, 0, 0, 0, 0};
    withFold(waveNeedsFold(a.box, I.p.x, I.p.y, I.p.z, r2h), [&](auto fold) {
        constexpr unsigned U = isMixed<T> ? 2 : 1; // records in flight
        const TargetList list = a.L.lists.list(t.r);
        for (unsigned k0 = 0; k0 < t.n; k0 += 4)
        {
            uint32_t j[4];
            list.quad(k0, j);
#pragma unroll
            for (unsigned s = 0; s < 4; s += U)
            {
                if (k0 + s >= t.n) { break; }
                RecMomVjpJ<T> rj[U];
#pragma unroll
                for (unsigned u = 0; u < U; ++u)
                    rj[u] = rec[j[s + u]];
#pragma unroll
                for (unsigned u = 0; u < U; ++u)
                {
                    if (k0 + s + u >= t.n) { break; }
                    T r[3];
                    separation<decltype(fold)::value>(a.box, r2h, I.p.x, I.p.y, I.p.z, rj[u].p.x, rj[u].p.y, rj[u].p.z,
                                                      r[0], r[1], r[2]);
                    const MomPairBar<T> b = momPairBar(kern, I, rj[u], r, hiInv, T(1) / rj[u].p.h);
                    for (int p = 0; p < 3; ++p)
                        gr[p] += b.r[p];
                    T c6[6];
                    symOuter(b.tAi, r, c6);
                    for (int q = 0; q < 6; ++q)
                        gC[q] += c6[q];
                    gh += b.hi, galpha += b.alpha, pro += b.pro, vol += b.volI;
                }
            }
        }
    });
    const T rho = ld<T>(f.rho, i), rho2 = rho * rho;
    addOwn<T>(f.gx, i, gr[0]), addOwn<T>(f.gy, i, gr[1]), addOwn<T>(f.gz, i, gr[2]), addOwn<T>(f.gh, i, gh);
    addOwn<T>(f.grho, i, -T(2) * pro * ld<T>(f.p, i) / (rho2 * rho) - vol * ld<T>(f.m, i) / rho2);
    addOwn<T>(f.gp, i, pro / rho2), addOwn<T>(f.galpha, i, galpha);
    for (int q = 0; q < 6; ++q)
        addOwn<T>(f.gC[q], i, gC[q]);
}

template<class T>
__global__ void __launch_bounds__(kVjpWaves * kWave)
    momentumStdVjpSourceKernel(PairArgs a, MomVjpArgs f, SincKernel<T> kern, SourceRows rows,
                               const RecMomVjpI<T>* __restrict__ rec)
{
    const uint32_t j = sourceParticle();
    if (j >= rows.n) { return; }
    const RecMomVjpJ<T> J     = loadMomVjpJ<T>(a, f, j);
    const T             hjInv = T(1) / J.p.h;

    T gr[3] = {0, 0, 0}, gh = 0, galpha = 0, prj = 0, vol = 0;
    T gC[6] = {0, 0, 0, 0, 0, 0};
    overTargets<isMixed<T> ? 2 : 1>(rows, j, rec, [&](const RecMomVjpI<T>& I) {
        T r[3];
        sourceSeparation(a.box, 2.0 * double(I.p.h), I.p.x, I.p.y, I.p.z, J.p.x, J.p.y, J.p.z, r[0], r[1], r[2]);
        const MomPairBar<T> b = momPairBar(kern, I, J, r, T(1) / I.p.h, hjInv);
        for (int p = 0; p < 3; ++p)
            gr[p] -= b.r[p];
        T c6[6];
        symOuter(b.tAj, r, c6);
        for (int q = 0; q < 6; ++q)
            gC[q] += c6[q];
        gh += b.hj, galpha += b.alpha, prj += b.prj, vol += b.volJ;
    });
    const T rho = ld<T>(f.rho, j), rho2 = rho * rho;
    addOwn<T>(f.gx, j, gr[0]), addOwn<T>(f.gy, j, gr[1]), addOwn<T>(f.gz, j, gr[2]), addOwn<T>(f.gh, j, gh);
    addOwn<T>(f.grho, j, -vol * J.m / rho2 - prj * ld<T>(f.p, j) / rho2);
    addOwn<T>(f.gp, j, prj / rho), addOwn<T>(f.galpha, j, galpha);
    for (int q = 0; q < 6; ++q)
        addOwn<T>(f.gC[q], j, gC[q]);
}

/* ---- the pair index of the adjoints --------------------------------------------------------------- */

constexpr uint32_t kTargetPad = 4; // entries behind the last row (overTargets reads whole batches)

//! stored pairs of each searched target (the last entry 0, so the exclusive scan ends with the total)
__global__ void pairCountKernel(NeighborLists lists, const uint32_t* __restrict__ nc, uint32_t nbFirst, uint32_t nt,
                                uint32_t* __restrict__ cnt)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < nt) { cnt[t] = lists.searched(t) ? min(nc[nbFirst + t] - 1u, lists.ngmax) : 0u; }
    else if (t == nt) { cnt[t] = 0; }
}

constexpr unsigned kPairsRun = 32; // entries of each list per round (pairsKernel)

/*! every stored pair p = pairStart[t] + k by its neighbour j and its target. A wave takes the 64 lists of one block, turns
 * kPairsRun entries of each in LDS and writes 128 bytes per row and half wave; with one thread per row, each writing
 * its own 4 bytes, the kernel took 5.1 ms of the 10 ms index of 2M particles (180M pairs); this takes 0.83. Bound by the
 * table lookups and 1.5 GB of writes. */
__global__ void __launch_bounds__(kVjpWaves* kWave)
    pairsKernel(NeighborLists lists, const uint32_t* __restrict__ pairStart, uint32_t nbFirst, uint32_t nt,
                uint32_t* __restrict__ js, uint32_t* __restrict__ targets)
{
    __shared__ uint32_t tile[kVjpWaves][kWave][kPairsRun + 1];
    const unsigned      w = threadIdx.x / kWave, lane = laneId();
    const uint32_t      t0 = (blockIdx.x * kVjpWaves + w) * kWave, t = t0 + lane;
    const bool          on = t < nt;
    const TargetList    list = lists.list(on ? t : 0u);
    const uint32_t      p0 = on ? pairStart[t] : 0u, n = on ? pairStart[t + 1] - p0 : 0u;
    const uint32_t      most = waveMax(n);
    for (uint32_t k0 = 0; k0 < most; k0 += kPairsRun)
    {
#pragma unroll
        for (uint32_t k = 0; k < kPairsRun; k += 4)
        {
            uint32_t j[4];
            if (k0 + k < n)
            {
                list.quad(k0 + k, j);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    tile[w][lane][k + u] = j[u];
            }
        }
        __builtin_amdgcn_wave_barrier(); // a wave's LDS accesses complete in order
        const uint32_t k = lane % kPairsRun;
        for (uint32_t row = lane / kPairsRun; row < kWave; row += kWave / kPairsRun)
        {
            const uint32_t rowN = __shfl(n, int(row), kWave), rowP = __shfl(p0, int(row), kWave);
            if (k0 + k < rowN) { js[rowP + k0 + k] = tile[w][row][k], targets[rowP + k0 + k] = nbFirst + t0 + row; }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

//! rowStart[j] = first pair of neighbour j in the pairs sorted by neighbour, j = 0 .. n; the targets' padding
__global__ void rowStartKernel(const uint32_t* __restrict__ js, uint64_t pairs, uint32_t n,
                               uint32_t* __restrict__ rowStart, uint32_t* __restrict__ targets)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < kTargetPad) { targets[pairs + j] = 0; }
    if (j > n) { return; }
    uint64_t lo = 0, hi = pairs;
    while (lo < hi)
    {
        const uint64_t mid = (lo + hi) / 2;
        if (js[mid] < j) { lo = mid + 1; }
        else { hi = mid; }
    }
    rowStart[j] = uint32_t(lo);
}

int bitsFor(uint64_t v)
{
    int b = 1;
    while (b < 64 && (v >> b) != 0) { ++b; }
    return b;
}

//! the pair index of the last search (built once per search, on the first adjoint call after it)
void buildAdjointPairs(sphx_workspace* ws)
{
    auto& A = ws->adj;
    if (A.serial == ws->searchSerial) { return; }
    const uint32_t nt = ws->nbLast - ws->nbFirst;
    const uint32_t n  = uint32_t(ws->tree.numParticles);
    SPHX_REQUIRE(uint64_t(nt) * ws->nbNgmax < (uint64_t(1) << 32), SPHX_ERR_ARG,
                 "adjoints: more than 2^32 neighbour pairs");
    A.pairStart.reserve(size_t(nt) + 1);
    // the counts, then the scan's temporaries, in the workspace scratch
    size_t tmpBytes = 0;
    SPHX_HIP(rocprim::exclusive_scan(nullptr, tmpBytes, static_cast<const uint32_t*>(nullptr), A.pairStart.get(), 0u,
                                     size_t(nt) + 1, rocprim::plus<uint32_t>(), ws->stream));
    const size_t cntBytes = ((size_t(nt) + 1) * sizeof(uint32_t) + 255) & ~size_t(255);
    char*        base     = static_cast<char*>(scratchBytes(ws, cntBytes + tmpBytes));
    uint32_t*    cnt      = reinterpret_cast<uint32_t*>(base);
    pairCountKernel<<<ceilDiv(size_t(nt) + 1, 256), 256, 0, ws->stream>>>(neighborLists(ws), ws->nbNc, ws->nbFirst, nt,
                                                                          cnt);
    SPHX_CHECK_LAUNCH();
    SPHX_HIP(rocprim::exclusive_scan(base + cntBytes, tmpBytes, cnt, A.pairStart.get(), 0u, size_t(nt) + 1,
                                     rocprim::plus<uint32_t>(), ws->stream));
    uint32_t pairs = 0;
    SPHX_HIP(hipMemcpyAsync(&pairs, A.pairStart.get() + nt, sizeof(pairs), hipMemcpyDeviceToHost, ws->stream));
    SPHX_HIP(hipStreamSynchronize(ws->stream));
    A.js.reserve(std::max<uint64_t>(pairs, 1)), A.jsSorted.reserve(std::max<uint64_t>(pairs, 1));
    A.targetsByPair.reserve(std::max<uint64_t>(pairs, 1)), A.targets.reserve(uint64_t(pairs) + kTargetPad);
    A.rowStart.reserve(size_t(n) + 1);
    if (pairs > 0)
    {
        pairsKernel<<<ceilDiv(nt, kVjpWaves * kWave), kVjpWaves * kWave, 0, ws->stream>>>(
            neighborLists(ws), A.pairStart.get(), ws->nbFirst, nt, A.js.get(), A.targetsByPair.get());
        SPHX_CHECK_LAUNCH();
        // stable: each neighbour's targets stay in increasing order
        const unsigned bits      = unsigned(bitsFor(n));
        size_t         sortBytes = 0;
        SPHX_HIP(rocprim::radix_sort_pairs(nullptr, sortBytes, A.js.get(), A.jsSorted.get(), A.targetsByPair.get(),
                                           A.targets.get(), size_t(pairs), 0, bits, ws->stream));
        void* tmp = scratchBytes(ws, sortBytes);
        SPHX_HIP(rocprim::radix_sort_pairs(tmp, sortBytes, A.js.get(), A.jsSorted.get(), A.targetsByPair.get(),
                                           A.targets.get(), size_t(pairs), 0, bits, ws->stream));
    }
    rowStartKernel<<<ceilDiv(size_t(n) + kTargetPad, 256), 256, 0, ws->stream>>>(A.jsSorted.get(), pairs, n,
                                                                                 A.rowStart.get(), A.targets.get());
    SPHX_CHECK_LAUNCH();
    A.serial = ws->searchSerial;
}

//! the records of a call: one of each kind per particle
template<class J, class I>
std::pair<J*, I*> vjpRecords(sphx_workspace* ws)
{
    static_assert(sizeof(J) % 16 == 0 && sizeof(I) % 16 == 0, "whole 16-byte chunks");
    const size_t n = ws->tree.numParticles;
    ws->adj.records.reserve((n + 1) * (sizeof(J) + sizeof(I)));
    J* j = reinterpret_cast<J*>(ws->adj.records.get());
    return {j, reinterpret_cast<I*>(j + n + 1)};
}

SourceRows sourceRows(const sphx_workspace* ws, uint32_t first, uint32_t last)
{
    return {ws->adj.rowStart.get(), ws->adj.targets.get(), first, last, uint32_t(ws->tree.numParticles)};
}

//! blocks of a walk over every particle
unsigned sourceBlocks(const sphx_workspace* ws)
{
    return unsigned(ceilDiv(ceilDiv(size_t(ws->tree.numParticles), kWave), kVjpWaves));
}

//! the adjoints take consecutive groups of 64 (no group view), the layout of their pair index
void requireConsecutive(const PairArgs& a)
{
    SPHX_REQUIRE(a.L.groups.start == nullptr, SPHX_ERR_ARG,
                 "the adjoints run over consecutive groups; clear the group view (sphx_set_groups with NULL) first");
}

void requireAll(std::initializer_list<const void*> ptrs, const char* what)
{
    for (const void* p : ptrs)
        SPHX_REQUIRE(p != nullptr, SPHX_ERR_ARG, what);
}

} // namespace

void densityStdVjp(sphx_workspace* ws, const DevBox& box, const sphx_fields_t* f, const sphx_params_t* p,
                   uint32_t first, uint32_t last, const sphx_adjoint_t* in, sphx_adjoint_t* out)
{
    PairArgs a = makePairArgs(ws, box, f, p, first, last);
    requireAll({f->h, f->m, in->rho, out->x, out->y, out->z, out->h},
               "density adjoint needs fields h, m, cotangent rho and gradients x, y, z, h");
    requireConsecutive(a);
    DensityVjpArgs d{f->h, f->m, in->rho, out->x, out->y, out->z, out->h};
    unsigned       blocks = vjpBlocks(a.L);
    if (blocks == 0) { return; }
    buildAdjointPairs(ws);
    const uint32_t n   = uint32_t(ws->tree.numParticles);
    auto           run = [&](auto zero) {
        using T           = decltype(zero);
        auto [recJ, recI] = vjpRecords<RecDensityVjpJ<T>, RecDensityVjpI<T>>(ws);
        packDensityVjp<T><<<ceilDiv(n, kPackThreads), kPackThreads, 0, ws->stream>>>(a, d, first, last, recJ, recI, n);
        SPHX_CHECK_LAUNCH();
        densityStdVjpKernel<T><<<blocks, kVjpWaves * kWave, 0, ws->stream>>>(a, d, sincKernel<T>(ws), recJ);
        SPHX_CHECK_LAUNCH();
        densityStdVjpSourceKernel<T><<<sourceBlocks(ws), kVjpWaves * kWave, 0, ws->stream>>>(
            a, d, sincKernel<T>(ws), sourceRows(ws, first, last), recI);
        SPHX_CHECK_LAUNCH();
    };
    if (p->hydro_type == SPHX_F32) { run(0.0f); }
    else { run(0.0); }
}

void iadStdVjp(sphx_workspace* ws, const DevBox& box, const sphx_fields_t* f, const sphx_params_t* p, uint32_t first,
               uint32_t last, const sphx_adjoint_t* in, sphx_adjoint_t* out)
{
    PairArgs a = makePairArgs(ws, box, f, p, first, last);
    requireAll({f->h, f->m, f->rho, f->c11, f->c12, f->c13, f->c22, f->c23, f->c33},
               "IAD adjoint needs fields h, m, rho and c11..c33");
    requireAll({in->c11, in->c12, in->c13, in->c22, in->c23, in->c33, out->x, out->y, out->z, out->h, out->rho},
               "IAD adjoint needs cotangents c11..c33 and gradients x, y, z, h, rho");
    IadVjpArgs d{f->h,
                 f->m,
                 f->rho,
                 {f->c11, f->c12, f->c13, f->c22, f->c23, f->c33},
                 {in->c11, in->c12, in->c13, in->c22, in->c23, in->c33},
                 out->x,
                 out->y,
                 out->z,
                 out->h,
                 out->rho};
    requireConsecutive(a);
    unsigned blocks = vjpBlocks(a.L);
    if (blocks == 0) { return; }
    buildAdjointPairs(ws);
    const uint32_t n   = uint32_t(ws->tree.numParticles);
    auto           run = [&](auto zero) {
        using T           = decltype(zero);
        auto [recJ, recI] = vjpRecords<RecIadVjpJ<T>, RecIadVjpI<T>>(ws);
        packIadVjp<T><<<ceilDiv(n, kPackThreads), kPackThreads, 0, ws->stream>>>(a, d, first, last, recJ, recI, n);
        SPHX_CHECK_LAUNCH();
        iadStdVjpKernel<T><<<blocks, kVjpWaves * kWave, 0, ws->stream>>>(a, d, sincKernel<T>(ws), recJ);
        SPHX_CHECK_LAUNCH();
        iadStdVjpSourceKernel<T><<<sourceBlocks(ws), kVjpWaves * kWave, 0, ws->stream>>>(
            a, d, sincKernel<T>(ws), sourceRows(ws, first, last), recI);
        SPHX_CHECK_LAUNCH();
    };
    if (p->hydro_type == SPHX_F32) { run(0.0f); }
    else { run(0.0); }
}

void momentumEnergyStdVjp(sphx_workspace* ws, const DevBox& box, const sphx_fields_t* f, const sphx_params_t* p,
                          uint32_t first, uint32_t last, const sphx_adjoint_t* in, sphx_adjoint_t* out)
{
    PairArgs a = makePairArgs(ws, box, f, p, first, last);
    requireAll({f->vx, f->vy, f->vz, f->h, f->m, f->rho, f->p, f->c, f->c11, f->c12, f->c13, f->c22, f->c23, f->c33},
               "momentum-energy adjoint needs the forward's fields");
    const bool perAlpha = (p->flags & SPHX_FLAG_STD_ALPHA) != 0;
    SPHX_REQUIRE(!perAlpha || f->alpha, SPHX_ERR_ARG, "SPHX_FLAG_STD_ALPHA set but fields.alpha is NULL");
    requireAll({in->ax, in->ay, in->az, out->x, out->y, out->z, out->h, out->rho, out->p, out->alpha, out->c11,
                out->c12, out->c13, out->c22, out->c23, out->c33},
               "momentum-energy adjoint needs cotangents ax, ay, az and gradients x, y, z, h, rho, p, alpha, "
               "c11..c33");
    MomVjpArgs d{f->vx,
                 f->vy,
                 f->vz,
                 f->h,
                 f->m,
                 f->rho,
                 f->p,
                 f->c,
                 perAlpha ? f->alpha : nullptr,
                 {f->c11, f->c12, f->c13, f->c22, f->c23, f->c33},
                 in->ax,
                 in->ay,
                 in->az,
                 in->du,
                 out->x,
                 out->y,
                 out->z,
                 out->h,
                 out->rho,
                 out->p,
                 out->alpha,
                 {out->c11, out->c12, out->c13, out->c22, out->c23, out->c33}};
    requireConsecutive(a);
    unsigned blocks = vjpBlocks(a.L);
    if (blocks == 0) { return; }
    buildAdjointPairs(ws);
    const uint32_t n   = uint32_t(ws->tree.numParticles);
    auto           run = [&](auto zero) {
        using T           = decltype(zero);
        auto [recJ, recI] = vjpRecords<RecMomVjpJ<T>, RecMomVjpI<T>>(ws);
        packMomVjp<T><<<ceilDiv(n, kPackThreads), kPackThreads, 0, ws->stream>>>(a, d, first, last, recJ, recI, n);
        SPHX_CHECK_LAUNCH();
        momentumStdVjpKernel<T><<<blocks, kVjpWaves * kWave, 0, ws->stream>>>(a, d, sincKernel<T>(ws), recJ);
        SPHX_CHECK_LAUNCH();
        momentumStdVjpSourceKernel<T><<<sourceBlocks(ws), kVjpWaves * kWave, 0, ws->stream>>>(
            a, d, sincKernel<T>(ws), sourceRows(ws, first, last), recI);
        SPHX_CHECK_LAUNCH();
    };
    if (p->hydro_type == SPHX_F32) { run(0.0f); }
    else { run(0.0); }
}

} // namespace sphx
