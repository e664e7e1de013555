// outputs.h -- what a step samples of the wavefield before it changes it:
// receivers, sections and Green's-function cells.  Device bodies shared by
// their own kernels and by the stress update's launch.
#pragma once

#include "swpc_internal.h"

// the step number: it, or with a device counter (step blocks captured in a
// graph) the counter plus it, the step's place in the block
__device__ static inline int step_number(int it, const int *d_it) { return d_it ? *d_it + it : it; }

// --------------------------------------------------------------------------
// wav__store, m_wav.f90:397-625 (one thread per station)
// --------------------------------------------------------------------------
struct WavArgs {
    Grid g;
    const float *Vx, *Vy, *Vz, *Sxx, *Syy, *Szz, *Syz, *Sxz, *Sxy;
    const int *ist, *jst, *kst;
    float *uacc, *eacc;
    float *wv, *wu, *ws, *we;
    int nst, what, ntdec, ntw;
    float M0, UC, dt;
    float r40x, r40y, r40z, r41x, r41y, r41z;
    int it;
    const int *d_it;
};

// station n of one context at step it
__device__ static inline void wav_store_body(const WavArgs &a, int n, int it)
{
    if (n >= a.nst) return;
    const Grid &g = a.g;
    const int i = a.ist[n], j = a.jst[n], k = a.kst[n];
    const long long P = g.plane;
    const int Y = g.pitch;
    const long long p = gidx(g, i, j, k);
    const float dt = a.dt;
    const int itw = (it - 1) / a.ntdec;
    const bool out = (it - 1) % a.ntdec == 0 && itw >= 0 && itw < a.ntw;
    // every load before the first store: a thread is a chain of dependent
    // loads (6.8 us for all four kinds with stores in between, 4.4 without)
    const float vx = a.Vx[p] + a.Vx[p - 1], vy = a.Vy[p] + a.Vy[p - Y], vz = a.Vz[p] + a.Vz[p - P];
    float u[3] = {}, e[6] = {}, sg[6] = {};
    if (a.what & SWPC_WAV_U) {
        u[0] = a.uacc[3 * n + 0] + vx * 0.5f * dt;
        u[1] = a.uacc[3 * n + 1] + vy * 0.5f * dt;
        u[2] = a.uacc[3 * n + 2] - vz * 0.5f * dt;
    }
    if (out && (a.what & SWPC_WAV_STRESS)) {
        sg[0] = a.Sxx[p];
        sg[1] = a.Syy[p];
        sg[2] = a.Szz[p];
        sg[3] = (a.Syz[p] + a.Syz[p - Y] + a.Syz[p - P] + a.Syz[p - Y - P]) / 4.0f;
        sg[4] = (a.Sxz[p] + a.Sxz[p - 1] + a.Sxz[p - P] + a.Sxz[p - 1 - P]) / 4.0f;
        sg[5] = (a.Sxy[p] + a.Sxy[p - Y] + a.Sxy[p - 1] + a.Sxy[p - 1 - Y]) / 4.0f;
    }
    if (a.what & SWPC_WAV_STRAIN) {
        const float *Vx = a.Vx, *Vy = a.Vy, *Vz = a.Vz;
        const float r40x = a.r40x, r40y = a.r40y, r40z = a.r40z, r41x = a.r41x, r41y = a.r41y, r41z = a.r41z;
#define AT(F, di, dj, dk) F[p + (di) + (long long)(dj) * Y + (long long)(dk) * P]
        const float dxVx = (AT(Vx, 0, 0, 0) - AT(Vx, -1, 0, 0)) * r40x - (AT(Vx, 1, 0, 0) - AT(Vx, -2, 0, 0)) * r41x;
        const float dyVy = (AT(Vy, 0, 0, 0) - AT(Vy, 0, -1, 0)) * r40y - (AT(Vy, 0, 1, 0) - AT(Vy, 0, -2, 0)) * r41y;
        const float dzVz = (AT(Vz, 0, 0, 0) - AT(Vz, 0, 0, -1)) * r40z - (AT(Vz, 0, 0, 1) - AT(Vz, 0, 0, -2)) * r41z;
        const float dxVy = ((AT(Vy, 1, 0, 0) - AT(Vy, 0, 0, 0)) * r40x - (AT(Vy, 2, 0, 0) - AT(Vy, -1, 0, 0)) * r41x
                          + (AT(Vy, 1, -1, 0) - AT(Vy, 0, -1, 0)) * r40x - (AT(Vy, 2, -1, 0) - AT(Vy, -1, -1, 0)) * r41x
                          + (AT(Vy, 0, 0, 0) - AT(Vy, -1, 0, 0)) * r40x - (AT(Vy, 1, 0, 0) - AT(Vy, -2, 0, 0)) * r41x
                          + (AT(Vy, 0, -1, 0) - AT(Vy, -1, -1, 0)) * r40x - (AT(Vy, 1, -1, 0) - AT(Vy, -2, -1, 0)) * r41x) / 4.0f;
        const float dxVz = ((AT(Vz, 1, 0, 0) - AT(Vz, 0, 0, 0)) * r40x - (AT(Vz, 2, 0, 0) - AT(Vz, -1, 0, 0)) * r41x
                          + (AT(Vz, 1, 0, -1) - AT(Vz, 0, 0, -1)) * r40x - (AT(Vz, 2, 0, -1) - AT(Vz, -1, 0, -1)) * r41x
                          + (AT(Vz, 0, 0, 0) - AT(Vz, -1, 0, 0)) * r40x - (AT(Vz, 1, 0, 0) - AT(Vz, -2, 0, 0)) * r41x
                          + (AT(Vz, 0, 0, -1) - AT(Vz, -1, 0, -1)) * r40x - (AT(Vz, 1, 0, -1) - AT(Vz, -2, 0, -1)) * r41x) / 4.0f;
        const float dyVx = ((AT(Vx, 0, 1, 0) - AT(Vx, 0, 0, 0)) * r40y - (AT(Vx, 0, 2, 0) - AT(Vx, 0, -1, 0)) * r41y
                          + (AT(Vx, -1, 1, 0) - AT(Vx, -1, 0, 0)) * r40y - (AT(Vx, -1, 2, 0) - AT(Vx, -1, -1, 0)) * r41y
                          + (AT(Vx, 0, 0, 0) - AT(Vx, 0, -1, 0)) * r40y - (AT(Vx, 0, 1, 0) - AT(Vx, 0, -2, 0)) * r41y
                          + (AT(Vx, -1, 0, 0) - AT(Vx, -1, -1, 0)) * r40y - (AT(Vx, -1, 1, 0) - AT(Vx, -1, -2, 0)) * r41y) / 4.0f;
        const float dyVz = ((AT(Vz, 0, 1, 0) - AT(Vz, 0, 0, 0)) * r40y - (AT(Vz, 0, 2, 0) - AT(Vz, 0, -1, 0)) * r41y
                          + (AT(Vz, 0, 1, -1) - AT(Vz, 0, 0, -1)) * r40y - (AT(Vz, 0, 2, -1) - AT(Vz, 0, -1, -1)) * r41y
                          + (AT(Vz, 0, 0, 0) - AT(Vz, 0, -1, 0)) * r40y - (AT(Vz, 0, 1, 0) - AT(Vz, 0, -2, 0)) * r41y
                          + (AT(Vz, 0, 0, -1) - AT(Vz, 0, -1, -1)) * r40y - (AT(Vz, 0, 1, -1) - AT(Vz, 0, -2, -1)) * r41y) / 4.0f;
        const float dzVx = ((AT(Vx, 0, 0, 1) - AT(Vx, 0, 0, 0)) * r40z - (AT(Vx, 0, 0, 2) - AT(Vx, 0, 0, -1)) * r41z
                          + (AT(Vx, -1, 0, 1) - AT(Vx, -1, 0, 0)) * r40z - (AT(Vx, -1, 0, 2) - AT(Vx, -1, 0, -1)) * r41z
                          + (AT(Vx, 0, 0, 0) - AT(Vx, 0, 0, -1)) * r40z - (AT(Vx, 0, 0, 1) - AT(Vx, 0, 0, -2)) * r41z
                          + (AT(Vx, -1, 0, 0) - AT(Vx, -1, 0, -1)) * r40z - (AT(Vx, -1, 0, 1) - AT(Vx, -1, 0, -2)) * r41z) / 4.0f;
        const float dzVy = ((AT(Vy, 0, 0, 1) - AT(Vy, 0, 0, 0)) * r40z - (AT(Vy, 0, 0, 2) - AT(Vy, 0, 0, -1)) * r41z
                          + (AT(Vy, 0, -1, 1) - AT(Vy, 0, -1, 0)) * r40z - (AT(Vy, 0, -1, 2) - AT(Vy, 0, -1, -1)) * r41z
                          + (AT(Vy, 0, 0, 0) - AT(Vy, 0, 0, -1)) * r40z - (AT(Vy, 0, 0, 1) - AT(Vy, 0, 0, -2)) * r41z
                          + (AT(Vy, 0, -1, 0) - AT(Vy, 0, -1, -1)) * r40z - (AT(Vy, 0, -1, 1) - AT(Vy, 0, -1, -2)) * r41z) / 4.0f;
#undef AT
        const float *o = a.eacc + 6 * n;
        e[0] = o[0] + dxVx * dt;
        e[1] = o[1] + dyVy * dt;
        e[2] = o[2] + dzVz * dt;
        e[3] = o[3] + (dyVz + dzVy) / 2.0f * dt;
        e[4] = o[4] + (dxVz + dzVx) / 2.0f * dt;
        e[5] = o[5] + (dxVy + dyVx) / 2.0f * dt;
    }
    if (a.what & SWPC_WAV_U) {
        for (int q = 0; q < 3; ++q) a.uacc[3 * n + q] = u[q];
    }
    if (a.what & SWPC_WAV_STRAIN) {
        for (int q = 0; q < 6; ++q) a.eacc[6 * n + q] = e[q];
    }
    if (!out) return;
    const float M0 = a.M0, UC = a.UC;
    const long long ntw = a.ntw;
    if (a.what & SWPC_WAV_V) {
        a.wv[(n * 3LL + 0) * ntw + itw] = vx / 2.0f * M0 * UC * 1e9f;
        a.wv[(n * 3LL + 1) * ntw + itw] = vy / 2.0f * M0 * UC * 1e9f;
        a.wv[(n * 3LL + 2) * ntw + itw] = -(vz / 2.0f * M0 * UC * 1e9f);
    }
    if (a.what & SWPC_WAV_U) {
        for (int q = 0; q < 3; ++q) a.wu[(n * 3LL + q) * ntw + itw] = u[q] * M0 * UC * 1e9f;
    }
    if (a.what & SWPC_WAV_STRESS) {
        for (int q = 0; q < 6; ++q) a.ws[(n * 6LL + q) * ntw + itw] = sg[q] * M0 * UC * 1e6f;
    }
    if (a.what & SWPC_WAV_STRAIN) {
        for (int q = 0; q < 6; ++q) a.we[(n * 6LL + q) * ntw + itw] = e[q] * M0 * UC * 1e-3f;
    }
}

// --------------------------------------------------------------------------
// snap__write, m_snap.f90:919-2189 (one thread per section point)
// --------------------------------------------------------------------------
#define SNAP_EPS 1.1920928955078125e-07f  // epsilon(1.0)

struct SnapArgs {
    Grid g;
    const float *Vx, *Vy, *Vz, *Syz, *Sxz, *Sxy, *lam;
    const int *kfs, *kob;
    SnapTask task[SWPC_SNP_NSECTION];
    int ntask, nblk;
    int k0_xy, i0_yz, j0_xz, idec, jdec, kdec, ntdec_s, nframe;
    float r20x, r20y, r20z, M0, UC, dt;
    int it;
    const int *d_it;
};

// correctly rounded single-precision square root, as the reference's sqrt:
// the double root of a float rounded once more to float is exact-rounded
// (53 >= 2*24 + 2 bits), which the single-precision hardware root is not
__device__ static inline float sqrt_rn(float x) { return (float)__dsqrt_rn((double)x); }

// lane of block blk (256 threads) of one context's section launch at step it
__device__ static inline void snap_body(const SnapArgs &a, int blk, int lane, int it)
{
    int t = 0;
    while (t + 1 < a.ntask && blk >= a.task[t + 1].blk0) ++t;
    const SnapTask T = a.task[t];
    const long long npt = (long long)T.ns1 * T.ns2;
    const long long p = (long long)(blk - T.blk0) * 256 + lane;
    if (p >= npt) return;
    if (it < 1) return;
    const bool out = ((it - 1) % a.ntdec_s) == 0;
    const int f = (it - 1) / a.ntdec_s;
    const bool every = (T.q == SWPC_SNP_U) || (T.q == SWPC_SNP_V && T.plane >= SWPC_SNP_FS);
    if (!(out && f < a.nframe) && !every) return;

    const int sa = (int)(p % T.ns1) + 1, sb = (int)(p / T.ns1) + 1;
    const Grid &g = a.g;
    int i, j, k;
    switch (T.plane) {
    case SWPC_SNP_XY: i = sa * a.idec - a.idec / 2; j = sb * a.jdec - a.jdec / 2; k = a.k0_xy; break;
    case SWPC_SNP_YZ: i = a.i0_yz; j = sa * a.jdec - a.jdec / 2; k = sb * a.kdec - a.kdec / 2; break;
    case SWPC_SNP_XZ: i = sa * a.idec - a.idec / 2; j = a.j0_xz; k = sb * a.kdec - a.kdec / 2; break;
    case SWPC_SNP_FS:
        i = sa * a.idec - a.idec / 2; j = sb * a.jdec - a.jdec / 2; k = a.kfs[g2idx(g, i, j)] + 1; break;
    default:
        i = sa * a.idec - a.idec / 2; j = sb * a.jdec - a.jdec / 2; k = a.kob[g2idx(g, i, j)] + 1; break;
    }
    const long long q = gidx(g, i, j, k);
    const long long P = g.plane;
    const int Y = g.pitch;
    float *fr = (out && f < a.nframe) ? T.frame + (long long)f * npt * (T.q == SWPC_SNP_PS ? 4 : 3) : nullptr;

    if (T.q == SWPC_SNP_PS) {
        // m_snap.f90:1016-1036
        float div = (a.Vx[q] - a.Vx[q - 1]) * a.r20x + (a.Vy[q] - a.Vy[q - Y]) * a.r20y
                  + (a.Vz[q] - a.Vz[q - P]) * a.r20z;
        float rot_x = (a.Vz[q + Y] - a.Vz[q]) * a.r20y - (a.Vy[q + P] - a.Vy[q]) * a.r20z;
        float rot_y = (a.Vx[q + P] - a.Vx[q]) * a.r20z - (a.Vz[q + 1] - a.Vz[q]) * a.r20x;
        float rot_z = (a.Vy[q + 1] - a.Vy[q]) * a.r20x - (a.Vx[q + Y] - a.Vx[q]) * a.r20y;
        const float lam = a.lam[q];
        div = div * lam / fabsf(lam + SNAP_EPS);
        const float syz = a.Syz[q], sxz = a.Sxz[q], sxy = a.Sxy[q];
        if (T.plane == SWPC_SNP_YZ) {
            // the yz section masks with abs(S + eps) (m_snap.f90:1028-1030)
            rot_x = rot_x * fabsf(syz) / fabsf(syz + SNAP_EPS);
            rot_y = rot_y * fabsf(sxz) / fabsf(sxz + SNAP_EPS);
            rot_z = rot_z * fabsf(sxy) / fabsf(sxy + SNAP_EPS);
        } else {
            // xz, xy, fs and ob mask with abs(S) + eps (m_snap.f90:1121-1123)
            rot_x = rot_x * fabsf(syz) / (fabsf(syz) + SNAP_EPS);
            rot_y = rot_y * fabsf(sxz) / (fabsf(sxz) + SNAP_EPS);
            rot_z = rot_z * fabsf(sxy) / (fabsf(sxy) + SNAP_EPS);
        }
        fr[p] = div * a.UC * a.M0 * 1e-3f;
        fr[p + npt] = rot_x * a.UC * a.M0 * 1e-3f;
        fr[p + 2 * npt] = rot_y * a.UC * a.M0 * 1e-3f;
        fr[p + 3 * npt] = rot_z * a.UC * a.M0 * 1e-3f;
    } else if (T.q == SWPC_SNP_V) {
        // m_snap.f90:1678-1683, maps :1697-1707
        const float b1 = a.Vx[q] * a.UC * a.M0;
        const float b2 = a.Vy[q] * a.UC * a.M0;
        const float b3 = a.Vz[q] * a.UC * a.M0;
        if (T.maxmap) {
            float *mx = T.maxmap;
            const float h = sqrt_rn(b1 * b1 + b2 * b2);
            const float az = fabsf(b3);
            const float m1 = fmaxf(mx[p], az), m2 = fmaxf(mx[p + npt], h);
            mx[p] = m1;
            mx[p + npt] = m2;
            mx[p + 2 * npt] = sqrt_rn(m1 * m1 + m2 * m2);
        }
        if (fr) {
            fr[p] = b1;
            fr[p + npt] = b2;
            fr[p + 2 * npt] = b3;
        }
    } else {
        // m_snap.f90:1857-1859 (u accumulates every step)
        float *u = T.uacc;
        const float u1 = u[p] + a.Vx[q] * a.UC * a.M0 * a.dt;
        const float u2 = u[p + npt] + a.Vy[q] * a.UC * a.M0 * a.dt;
        const float u3 = u[p + 2 * npt] + a.Vz[q] * a.UC * a.M0 * a.dt;
        u[p] = u1;
        u[p + npt] = u2;
        u[p + 2 * npt] = u3;
        if (T.maxmap) {
            float *mx = T.maxmap;
            const float h = sqrt_rn(u1 * u1 + u2 * u2);
            const float az = fabsf(u3);
            const float m1 = fmaxf(mx[p], az), m2 = fmaxf(mx[p + npt], h);
            mx[p] = m1;
            mx[p + npt] = m2;
            mx[p + 2 * npt] = sqrt_rn(m1 * m1 + m2 * m2);
        }
        if (fr) {
            fr[p] = u1;
            fr[p + npt] = u2;
            fr[p + 2 * npt] = u3;
        }
    }
}

// --------------------------------------------------------------------------
// green__store, m_green.f90:406-545 (one thread per Green's-function cell)
// --------------------------------------------------------------------------
// UC_DERIV = 10.0**(-15) and UC_BF = 10.0**(-12) as the Fortran compiler
// folds them to single precision (m_green.f90:30-31)
#define GREEN_UC_DERIV 0x1.203afcp-50f
#define GREEN_UC_BF 0x1.197998p-40f

struct GreenArgs {
    const float *Vx, *Vy, *Vz;
    const int *ig, *jg, *kg;
    float *acc;   // (12, ng): dxUx dxUy dxUz dyUx dyUy dyUz dzUx dzUy dzUz Ux Uy Uz
    float *gf;    // (ntw, ncmp*ng), Fortran order
    Grid g;
    int ng, ncmp, ntdec, ntw;
    float dt;
    float r40x, r40y, r40z, r41x, r41y, r41z;
    int it;
    const int *d_it;
};

// (F(c) - F(c-s)) * r40 - (F(c+s) - F(c-2s)) * r41: the 4th-order staggered
// derivative whose upper inner node is c, stride s along the axis
__device__ static inline float dstag(const float *F, long long c, long long s, float r40, float r41)
{
    return (F[c] - F[c - s]) * r40 - (F[c + s] - F[c - 2 * s]) * r41;
}

// green__store, m_green.f90:406-545
// GF point n of one context at step it
__device__ static inline void green_store_body(const GreenArgs &a, int n, int it)
{
    if (n >= a.ng) return;
    const Grid &g = a.g;
    const long long p = gidx(g, a.ig[n], a.jg[n], a.kg[n]);
    const long long X = 1, Y = g.pitch, Z = g.plane;
    const float *Vx = a.Vx, *Vy = a.Vy, *Vz = a.Vz;
    const float r40x = a.r40x, r40y = a.r40y, r40z = a.r40z, r41x = a.r41x, r41y = a.r41y, r41z = a.r41z;

    // m_green.f90:458-460
    const float dxVx = dstag(Vx, p, X, r40x, r41x);
    const float dyVy = dstag(Vy, p, Y, r40y, r41y);
    const float dzVz = dstag(Vz, p, Z, r40z, r41z);
    // the four staggered derivatives around the cell, m_green.f90:462-483
    const float dxVy1 = dstag(Vy, p + X, X, r40x, r41x), dxVy2 = dstag(Vy, p + X - Y, X, r40x, r41x);
    const float dxVy3 = dstag(Vy, p, X, r40x, r41x), dxVy4 = dstag(Vy, p - Y, X, r40x, r41x);
    const float dxVz1 = dstag(Vz, p + X, X, r40x, r41x), dxVz2 = dstag(Vz, p + X - Z, X, r40x, r41x);
    const float dxVz3 = dstag(Vz, p, X, r40x, r41x), dxVz4 = dstag(Vz, p - Z, X, r40x, r41x);
    const float dyVx1 = dstag(Vx, p + Y, Y, r40y, r41y), dyVx2 = dstag(Vx, p - X + Y, Y, r40y, r41y);
    const float dyVx3 = dstag(Vx, p, Y, r40y, r41y), dyVx4 = dstag(Vx, p - X, Y, r40y, r41y);
    const float dyVz1 = dstag(Vz, p + Y, Y, r40y, r41y), dyVz2 = dstag(Vz, p - Z + Y, Y, r40y, r41y);
    const float dyVz3 = dstag(Vz, p, Y, r40y, r41y), dyVz4 = dstag(Vz, p - Z, Y, r40y, r41y);
    const float dzVx1 = dstag(Vx, p + Z, Z, r40z, r41z), dzVx2 = dstag(Vx, p - X + Z, Z, r40z, r41z);
    const float dzVx3 = dstag(Vx, p, Z, r40z, r41z), dzVx4 = dstag(Vx, p - X, Z, r40z, r41z);
    const float dzVy1 = dstag(Vy, p + Z, Z, r40z, r41z), dzVy2 = dstag(Vy, p - Y + Z, Z, r40z, r41z);
    const float dzVy3 = dstag(Vy, p, Z, r40z, r41z), dzVy4 = dstag(Vy, p - Y, Z, r40z, r41z);
    // their means, m_green.f90:485-490
    const float dxVy = (dxVy1 + dxVy2 + dxVy3 + dxVy4) * 0.25f;
    const float dxVz = (dxVz1 + dxVz2 + dxVz3 + dxVz4) * 0.25f;
    const float dyVx = (dyVx1 + dyVx2 + dyVx3 + dyVx4) * 0.25f;
    const float dyVz = (dyVz1 + dyVz2 + dyVz3 + dyVz4) * 0.25f;
    const float dzVx = (dzVx1 + dzVx2 + dzVx3 + dzVx4) * 0.25f;
    const float dzVy = (dzVy1 + dzVy2 + dzVy3 + dzVy4) * 0.25f;

    // time integration, m_green.f90:492-506
    const long long ng = a.ng;
    const float dt = a.dt;
    float *acc = a.acc + n;
    const float d[9] = {dxVx, dxVy, dxVz, dyVx, dyVy, dyVz, dzVx, dzVy, dzVz};
#pragma unroll
    for (int q = 0; q < 9; ++q) acc[q * ng] = acc[q * ng] + d[q] * dt;
    const bool bforce = a.ncmp == 9;
    if (bforce) {
        acc[9 * ng] = acc[9 * ng] + 0.5f * (Vx[p] + Vx[p - X]) * dt;
        acc[10 * ng] = acc[10 * ng] + 0.5f * (Vy[p] + Vy[p - Y]) * dt;
        acc[11 * ng] = acc[11 * ng] + 0.5f * (Vz[p] + Vz[p - Z]) * dt;
    }

    // output every ntdec_w steps, m_green.f90:510-541
    if ((it - 1) % a.ntdec != 0) return;
    const int itw = (it - 1) / a.ntdec;
    if (itw < 0 || itw >= a.ntw) return;
    const float ucd = GREEN_UC_DERIV, ucb = GREEN_UC_BF;
    const long long ntw = a.ntw;
    float *gf = a.gf + (long long)n * a.ncmp * ntw + itw;
    gf[0 * ntw] = acc[0] * ucd * 1e9f;
    gf[1 * ntw] = acc[4 * ng] * ucd * 1e9f;
    gf[2 * ntw] = acc[8 * ng] * ucd * 1e9f;
    gf[3 * ntw] = (acc[5 * ng] + acc[7 * ng]) * ucd * 1e9f;
    gf[4 * ntw] = (acc[2 * ng] + acc[6 * ng]) * ucd * 1e9f;
    gf[5 * ntw] = (acc[1 * ng] + acc[3 * ng]) * ucd * 1e9f;
    if (bforce) {
        gf[6 * ntw] = acc[9 * ng] * ucb * 1e9f;
        gf[7 * ntw] = acc[10 * ng] * ucb * 1e9f;
        gf[8 * ntw] = acc[11 * ng] * ucb * 1e9f;
    }
}

// The outputs of one step that need V only, as the first blocks of the stress
// update's launch, which reads V and does not write it.  Blocks of 256 threads:
// ng for the Green's-function cells, nw for the receivers, ns for the
// sections, then idle ones up to nblk, a multiple of 8 (the tiles behind them
// keep their XCDs).
struct OutArgs {
    int ng, nw, ns, nblk;
    GreenArgs green;
    WavArgs wav;
    SnapArgs snap;
};

__device__ __forceinline__ void outputs_body(const OutArgs &o, int blk, int lane)
{
    if (blk < o.ng) {
        green_store_body(o.green, blk * 256 + lane, step_number(o.green.it, o.green.d_it));
    } else if (blk < o.ng + o.nw) {
        wav_store_body(o.wav, (blk - o.ng) * 256 + lane, step_number(o.wav.it, o.wav.d_it));
    } else if (blk < o.ng + o.nw + o.ns) {
        snap_body(o.snap, blk - o.ng - o.nw, lane, step_number(o.snap.it, o.snap.d_it));
    }
}
