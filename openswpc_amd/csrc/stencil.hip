// stencil.hip -- velocity/stress updates of OpenSWPC's 3D loop on gfx950.
//
// Each phase is one launch of z-marching tiles: the interior (4th order +
// Zener memory variables, m_kernel) and the ADE-CFS PML (2nd order,
// m_absorb_p).
// A thread owns one (i,j) column of a 64 x BY tile of full-width rows whose
// first cell sits on a 128-byte line, and marches a chunk of planes along z,
// keeping the z-neighbours of its column in a rotating register queue while
// the x/y neighbours come from the plane the tile is streaming (L1/L2
// resident).  Loop bodies are branch free and load everything before they
// store, so every load of an iteration is in flight at once: with each stress
// component loaded between the stores of its neighbours a wave made six
// memory round trips per cell (elastic 256 x 256 x 192, 20-cell PML: stress
// launch 262 us, 195 us with the loads first).  Every arithmetic expression
// keeps the reference's FP32 evaluation order; the library is compiled with
// -ffp-contract=off so no FMA changes the rounding.
//
// A whole step's Cerjan taper (m_absorb_c) is applied by the update itself
// before it stores; called routine by routine it is a sweep of its own, as in
// the reference.
#include "device_access.h"
#include "outputs.h"
#include "swpc_internal.h"

#define BX 64
#define MASK_INT 1
#define MASK_PML 2
#define MASK_TAPER 4  // the update applies the Cerjan taper to the values it stores

// Four waves per SIMD: 128 registers, which every NM <= 4 form fits without a
// spill; asking for no more lets the scheduler keep a cell's loads together.
#define WAVES4 __attribute__((amdgpu_waves_per_eu(4, 4)))
#define WAVES_NM __attribute__((amdgpu_waves_per_eu(NM <= 4 ? 4 : 3, NM <= 4 ? 4 : 3)))

// isign of m_kernel.f90:103-104: true inside the 2nd-order band
__device__ static inline bool in_band(int k, int kft, int kfb, int kot, int kob)
{
    const int a = (k - kft) * (kfb - k);
    const int b = (k - kot) * (kob - k);
    return (a > b ? a : b) >= 0;
}

// harmonic mean of mu over four cells, m_kernel.f90:293-309
__device__ static inline float hmean4(float a, float b, float c, float d, float epsl)
{
    return 4.0f * a * b * c * d / (a * b * c + a * b * d + a * c * d + b * c * d + epsl);
}

#define EPSL 1.1920928955078125e-07f  // epsilon(1.0)

// The 6*NM memory variables of one cell, value v = c*NM + m for component
// c = xx yy zz yz xz xy and mechanism m, packed as 16-byte vectors: value v
// lives in vector v/4 of stream v/4 (streams of rn float4 each), the last
// two values (6*NM mod 4 = 2) in a float2 stream after them.  One cell's
// values are loaded and stored together, so a wave moves 1 KB per access and
// the kernel keeps 6*NM/4 streams open instead of 6*NM.
template <int NM>
struct RCell {
    static constexpr int NV = 6 * NM, N4 = NV / 4, N2 = (NV % 4) / 2;
    float v[NV > 0 ? NV : 1];

    template <bool NT>
    __device__ __forceinline__ void load(const float *R, long long rn, const Loc &r)
    {
#pragma unroll
        for (int s = 0; s < N4; ++s) {
            const f4v t = ldv<NT>((const f4v *)((const char *)((const f4v *)R + (s * rn + r.u)) + 4 * r.o));
            v[4 * s] = t.x; v[4 * s + 1] = t.y; v[4 * s + 2] = t.z; v[4 * s + 3] = t.w;
        }
        if constexpr (N2 == 1) {
            const f2v t = ldv<NT>((const f2v *)((const char *)((const f2v *)(R + 4 * N4 * rn) + r.u) + 2 * r.o));
            v[4 * N4] = t.x; v[4 * N4 + 1] = t.y;
        }
    }
    template <bool NT>
    __device__ __forceinline__ void store(float *R, long long rn, const Loc &r) const
    {
#pragma unroll
        for (int s = 0; s < N4; ++s) {
            f4v t;
            t.x = v[4 * s]; t.y = v[4 * s + 1]; t.z = v[4 * s + 2]; t.w = v[4 * s + 3];
            stv<NT>((f4v *)((char *)((f4v *)R + (s * rn + r.u)) + 4 * r.o), t);
        }
        if constexpr (N2 == 1) {
            f2v t;
            t.x = v[4 * N4]; t.y = v[4 * N4 + 1];
            stv<NT>((f2v *)((char *)((f2v *)(R + 4 * N4 * rn) + r.u) + 2 * r.o), t);
        }
    }
};

struct StepArgs {
    Grid g;
    FieldPtrs f;
    // where the updated fields' old values are read: f itself (in place), or
    // other buffers, so a step can write its results next to its inputs
    FieldPtrs fin;
    MediumPtrs m;
    float *R;
    ViscoCoef v;
    Coef4 c;
    float dt;
    // PML
    float *ade;
    const float *ade_in;  // old auxiliaries (ade when in place)
    long long npml;
    PmlBox box[5];
    const float4 *gxc, *gxe, *gyc, *gye, *gzc, *gze;
    float r20x, r20y, r20z;
    const int4 *tiles;   // side-column PML tiles: (i0 | width << 20, j0, k0, k1)
    int ntiles;
    int first;           // blocks of the launch before the tiles' (the step's outputs, k_stress)
    int sideb;           // blocks of a launch that walk the side tiles (a multiple of 8, >= ntiles; 0: none)
    int has_pml, mask;
    int still;           // see aux_on
    int tau;             // NM = 0: whether taup or taus is anything but zero
    // Cerjan profiles at cell centres (c) and boundaries (b), halo of 3: entry of cell n is n + 2
    const float *cgx_c, *cgx_b, *cgy_c, *cgy_b, *cgz_c, *cgz_b;
    // interior launch shape
    const int *zc;       // first plane of each k chunk (nbz + 1 entries, last = nz + 1)
    int bx0, nbx, nby, nbz, by;
    int bxw, byi;        // interior tiles: bxw (64 or 32) cells wide, byi rows (bxw * byi = 64 * by threads)
};

// The 4th-order coefficients of a cell (near and far per axis) by its band
// state.  Both states are held in vector registers across the march: left in
// the arguments, the selects become loads at a per-lane address or, short of
// scalar registers, lane reads of spilled ones.
struct Coefs {
    float v[2][6];

    __device__ explicit Coefs(const StepArgs &a)
    {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            v[b][0] = a.c.re40x[b]; v[b][1] = a.c.re41x[b]; v[b][2] = a.c.re40y[b];
            v[b][3] = a.c.re41y[b]; v[b][4] = a.c.re40z[b]; v[b][5] = a.c.re41z[b];
#pragma unroll
            for (int q = 0; q < 6; ++q) asm("" : "+v"(v[b][q]));
        }
    }
    __device__ float at(bool in, int q) const { return in ? v[1][q] : v[0][q]; }
};

// Cerjan profile values of a column (m_absorb_c.f90:113-198).  Folded into the
// update the taper costs no traffic; as sweeps of their own the two tapers
// read and wrote all nine fields again (181 x 149 x 117: 163 us/step, 122
// folded).  TP: the launch may hold such members; other launches leave the
// test out, which cost PML runs 4-8 % on small grids.
template <bool TP>
struct Taper {
    float xc, xb, yc, yb;

    __device__ Taper(const StepArgs &a, int i, int j) : xc(1.0f), xb(1.0f), yc(1.0f), yb(1.0f)
    {
        if (!TP || !(a.mask & MASK_TAPER)) return;
        xc = ldv<false>(a.cgx_c + (i + 2)); xb = ldv<false>(a.cgx_b + (i + 2));
        yc = ldv<false>(a.cgy_c + (j + 2)); yb = ldv<false>(a.cgy_b + (j + 2));
    }
};

// ---------------------------------------------------------------------------
// ADE-CFS PML cell updates (m_absorb_p).  A column's auxiliaries are numbered
// compactly box by box; the auxiliary of plane k is q = abase + k*astride.
// ---------------------------------------------------------------------------
__device__ static inline PmlBox pick_box(const StepArgs &a, int q)
{
    return q == 0 ? a.box[0] : q == 1 ? a.box[1] : q == 2 ? a.box[2] : q == 3 ? a.box[3] : a.box[4];
}

// Whether a cell's auxiliaries of one axis take part.  Where the axis does not
// damp (profile entry 4, the gain of the auxiliary, is zero at the centre and
// at the edge) they start at zero and stay there, and a zero adds nothing to
// the derivative: neither they nor their update is needed.  Only the cells in
// the edges and corners of the zones keep all nine of a phase; a cell of a
// face keeps three, 24 of 72 bytes (us per step with all nine and with the
// ones that take part: 128^3 139 -> 132, elastic 256 x 256 x 192 522 -> 469,
// 768 x 768 x 448 13260 -> 12770).  still: no auxiliary has moved under other
// profiles (swpc_set_pml).
__device__ __forceinline__ bool aux_on(const StepArgs &a, const float4 &gc, const float4 &ge)
{
    return !(a.still && gc.w == 0.0f && ge.w == 0.0f);
}

// absorb_p__update_stress for one cell, m_absorb_p.f90:455-517.  The caller
// passes its z-queue values: V at k (and k+1 for Vx, Vy; k-1 for Vz) and mu
// on planes k, k+1.
template <bool NT, bool OOP>
__device__ __forceinline__ void pml_stress_cell(const StepArgs &a, Loc p, Loc q, int k, float vx_0,
                                                float vx_p1, float vy_0, float vy_p1, float vz_m1, float vz_0,
                                                float mu00, float mu00n, float mu10, float mu10n, float mu01,
                                                float mu01n, float mu11, float4 gxc, float4 gxe, float4 gyc,
                                                float4 gye)
{
    const float *__restrict__ Vx = a.f.Vx;
    const float *__restrict__ Vy = a.f.Vy;
    const float *__restrict__ Vz = a.f.Vz;
    const long long n = a.npml;
    float *__restrict__ A = a.ade;
    const float *__restrict__ AI = OOP ? a.ade_in : A;
    const float dt = a.dt;
    const float vx_im1 = ld(Vx, p, 0, -1), vy_jm1 = ld(Vy, p, 0, 0, -1);
    const float vy_ip1 = ld(Vy, p, 0, 1), vz_ip1 = ld(Vz, p, 0, 1);
    const float vx_jp1 = ld(Vx, p, 0, 0, 1), vz_jp1 = ld(Vz, p, 0, 0, 1);
    const float4 gzc = ldp(a.gzc + (k - 1)), gze = ldp(a.gze + (k - 1));
    const float lam0 = ld<NT>(a.m.lam, p);
    const bool onx = aux_on(a, gxc, gxe), ony = aux_on(a, gyc, gye), onz = aux_on(a, gzc, gze);
    float axVx = 0.0f, axVy = 0.0f, axVz = 0.0f;
    float ayVx = 0.0f, ayVy = 0.0f, ayVz = 0.0f;
    float azVx = 0.0f, azVy = 0.0f, azVz = 0.0f;
    if (onx) {
        fresh(q);
        axVx = ld<NT>(AI, q, A_axVx * n); axVy = ld<NT>(AI, q, A_axVy * n); axVz = ld<NT>(AI, q, A_axVz * n);
    }
    if (ony) {
        fresh(q);
        ayVx = ld<NT>(AI, q, A_ayVx * n); ayVy = ld<NT>(AI, q, A_ayVy * n); ayVz = ld<NT>(AI, q, A_ayVz * n);
    }
    if (onz) {
        fresh(q);
        azVx = ld<NT>(AI, q, A_azVx * n); azVy = ld<NT>(AI, q, A_azVy * n); azVz = ld<NT>(AI, q, A_azVz * n);
    }
    fresh(p);
    float *__restrict__ Sxx = a.f.Sxx;
    float *__restrict__ Syy = a.f.Syy;
    float *__restrict__ Szz = a.f.Szz;
    float *__restrict__ Syz = a.f.Syz;
    float *__restrict__ Sxz = a.f.Sxz;
    float *__restrict__ Sxy = a.f.Sxy;
    const float *__restrict__ SxxI = OOP ? a.fin.Sxx : Sxx;
    const float *__restrict__ SyyI = OOP ? a.fin.Syy : Syy;
    const float *__restrict__ SzzI = OOP ? a.fin.Szz : Szz;
    const float *__restrict__ SyzI = OOP ? a.fin.Syz : Syz;
    const float *__restrict__ SxzI = OOP ? a.fin.Sxz : Sxz;
    const float *__restrict__ SxyI = OOP ? a.fin.Sxy : Sxy;
    // every load before the first store (see stress_cell)
    const float sxx = ld<NT>(SxxI, p), syy = ld<NT>(SyyI, p), szz = ld<NT>(SzzI, p);
    const float syz = ld<NT>(SyzI, p), sxz = ld<NT>(SxzI, p), sxy = ld<NT>(SxyI, p);

    // normal components
    const float dxVx = (vx_0 - vx_im1) * a.r20x;
    const float dyVy = (vy_0 - vy_jm1) * a.r20y;
    const float dzVz = (vz_0 - vz_m1) * a.r20z;
    const float lam2mu_R = (lam0 + 2.0f * mu00);
    const float lam_R = lam2mu_R - 2.0f * mu00;
    const float dxVx_ade = gxc.x * dxVx + gxc.y * axVx;
    const float dyVy_ade = gyc.x * dyVy + gyc.y * ayVy;
    const float dzVz_ade = gzc.x * dzVz + gzc.y * azVz;
    st<NT>(Sxx, p, sxx + (lam2mu_R * dxVx_ade + lam_R * (dyVy_ade + dzVz_ade)) * dt);
    st<NT>(Syy, p, syy + (lam2mu_R * dyVy_ade + lam_R * (dxVx_ade + dzVz_ade)) * dt);
    st<NT>(Szz, p, szz + (lam2mu_R * dzVz_ade + lam_R * (dxVx_ade + dyVy_ade)) * dt);

    // shear components
    const float dxVy = (vy_ip1 - vy_0) * a.r20x;
    const float dxVz = (vz_ip1 - vz_0) * a.r20x;
    const float dyVx = (vx_jp1 - vx_0) * a.r20y;
    const float dyVz = (vz_jp1 - vz_0) * a.r20y;
    const float dzVx = (vx_p1 - vx_0) * a.r20z;
    const float dzVy = (vy_p1 - vy_0) * a.r20z;
    const float muxz = hmean4(mu00, mu00n, mu10, mu10n, EPSL);
    const float muxy = hmean4(mu00, mu10, mu01, mu11, EPSL);
    const float muyz = hmean4(mu00, mu00n, mu01, mu01n, EPSL);
    st<NT>(Syz, p, syz + muyz * (gye.x * dyVz + gze.x * dzVy + gye.y * ayVz + gze.y * azVy) * dt);
    st<NT>(Sxz, p, sxz + muxz * (gxe.x * dxVz + gze.x * dzVx + gxe.y * axVz + gze.y * azVx) * dt);
    st<NT>(Sxy, p, sxy + muxy * (gxe.x * dxVy + gye.x * dyVx + gxe.y * axVy + gye.y * ayVx) * dt);
    if (onx) {
        fresh(q);
        st<NT>(A, q, gxc.z * axVx + gxc.w * dxVx * dt, A_axVx * n);
        st<NT>(A, q, gxe.z * axVy + gxe.w * dxVy * dt, A_axVy * n);
        st<NT>(A, q, gxe.z * axVz + gxe.w * dxVz * dt, A_axVz * n);
    }
    if (ony) {
        fresh(q);
        st<NT>(A, q, gyc.z * ayVy + gyc.w * dyVy * dt, A_ayVy * n);
        st<NT>(A, q, gye.z * ayVx + gye.w * dyVx * dt, A_ayVx * n);
        st<NT>(A, q, gye.z * ayVz + gye.w * dyVz * dt, A_ayVz * n);
    }
    if (onz) {
        fresh(q);
        st<NT>(A, q, gzc.z * azVz + gzc.w * dzVz * dt, A_azVz * n);
        st<NT>(A, q, gze.z * azVx + gze.w * dzVx * dt, A_azVx * n);
        st<NT>(A, q, gze.z * azVy + gze.w * dzVy * dt, A_azVy * n);
    }
}

// absorb_p__update_vel for one cell, m_absorb_p.f90:267-304.  Queue values:
// Szz on k, k+1; Syz, Sxz on k-1, k; rho on k, k+1.
template <bool NT, bool OOP>
__device__ __forceinline__ void pml_vel_cell(const StepArgs &a, Loc p, Loc q, int k, float szz_0,
                                             float szz_p1, float syz_m1, float syz_0, float sxz_m1, float sxz_0,
                                             float rho0, float rho_kp, float4 gxc, float4 gxe, float4 gyc,
                                             float4 gye)
{
    const float *__restrict__ Sxx = a.f.Sxx;
    const float *__restrict__ Syy = a.f.Syy;
    const float *__restrict__ Syz = a.f.Syz;
    const float *__restrict__ Sxz = a.f.Sxz;
    const float *__restrict__ Sxy = a.f.Sxy;
    const float *__restrict__ rho = a.m.rho;
    const long long n = a.npml;
    float *__restrict__ A = a.ade;
    const float *__restrict__ AI = OOP ? a.ade_in : A;
    const float dt = a.dt;
    const float sxx_0 = ld(Sxx, p), sxx_ip1 = ld(Sxx, p, 0, 1);
    const float syy_0 = ld(Syy, p), syy_jp1 = ld(Syy, p, 0, 0, 1);
    const float syz_jm1 = ld(Syz, p, 0, 0, -1), sxz_im1 = ld(Sxz, p, 0, -1);
    const float sxy_0 = ld(Sxy, p), sxy_im1 = ld(Sxy, p, 0, -1), sxy_jm1 = ld(Sxy, p, 0, 0, -1);
    const float rho_ip = ld(rho, p, 0, 1), rho_jp = ld(rho, p, 0, 0, 1);
    const float4 gzc = ldp(a.gzc + (k - 1)), gze = ldp(a.gze + (k - 1));
    const bool onx = aux_on(a, gxc, gxe), ony = aux_on(a, gyc, gye), onz = aux_on(a, gzc, gze);
    float axSxx = 0.0f, axSxy = 0.0f, axSxz = 0.0f;
    float aySxy = 0.0f, aySyy = 0.0f, aySyz = 0.0f;
    float azSxz = 0.0f, azSyz = 0.0f, azSzz = 0.0f;
    if (onx) {
        fresh(q);
        axSxx = ld<NT>(AI, q, A_axSxx * n); axSxy = ld<NT>(AI, q, A_axSxy * n); axSxz = ld<NT>(AI, q, A_axSxz * n);
    }
    if (ony) {
        fresh(q);
        aySxy = ld<NT>(AI, q, A_aySxy * n); aySyy = ld<NT>(AI, q, A_aySyy * n); aySyz = ld<NT>(AI, q, A_aySyz * n);
    }
    if (onz) {
        fresh(q);
        azSxz = ld<NT>(AI, q, A_azSxz * n); azSyz = ld<NT>(AI, q, A_azSyz * n); azSzz = ld<NT>(AI, q, A_azSzz * n);
    }
    fresh(p);
    float *__restrict__ Vx = a.f.Vx;
    float *__restrict__ Vy = a.f.Vy;
    float *__restrict__ Vz = a.f.Vz;
    const float vx = ld<NT>(OOP ? a.fin.Vx : Vx, p), vy = ld<NT>(OOP ? a.fin.Vy : Vy, p);
    const float vz = ld<NT>(OOP ? a.fin.Vz : Vz, p);

    const float dxSxx = (sxx_ip1 - sxx_0) * a.r20x;
    const float dySyy = (syy_jp1 - syy_0) * a.r20y;
    const float dzSzz = (szz_p1 - szz_0) * a.r20z;
    const float dySyz = (syz_0 - syz_jm1) * a.r20y;
    const float dzSyz = (syz_0 - syz_m1) * a.r20z;
    const float dxSxz = (sxz_0 - sxz_im1) * a.r20x;
    const float dzSxz = (sxz_0 - sxz_m1) * a.r20z;
    const float dxSxy = (sxy_0 - sxy_im1) * a.r20x;
    const float dySxy = (sxy_0 - sxy_jm1) * a.r20y;
    const float bx = 2.0f / (rho0 + rho_ip);
    const float by = 2.0f / (rho0 + rho_jp);
    const float bz = 2.0f / (rho0 + rho_kp);

    st<NT>(Vx, p, vx + bx * (gxe.x * dxSxx + gyc.x * dySxy + gzc.x * dzSxz
                                                + gxe.y * axSxx + gyc.y * aySxy + gzc.y * azSxz) * dt);
    st<NT>(Vy, p, vy + by * (gxc.x * dxSxy + gye.x * dySyy + gzc.x * dzSyz
                                                + gxc.y * axSxy + gye.y * aySyy + gzc.y * azSyz) * dt);
    st<NT>(Vz, p, vz + bz * (gxc.x * dxSxz + gyc.x * dySyz + gze.x * dzSzz
                                                + gxc.y * axSxz + gyc.y * aySyz + gze.y * azSzz) * dt);
    if (onx) {
        fresh(q);
        st<NT>(A, q, gxe.z * axSxx + gxe.w * dxSxx * dt, A_axSxx * n);
        st<NT>(A, q, gxc.z * axSxy + gxc.w * dxSxy * dt, A_axSxy * n);
        st<NT>(A, q, gxc.z * axSxz + gxc.w * dxSxz * dt, A_axSxz * n);
    }
    if (ony) {
        fresh(q);
        st<NT>(A, q, gyc.z * aySxy + gyc.w * dySxy * dt, A_aySxy * n);
        st<NT>(A, q, gye.z * aySyy + gye.w * dySyy * dt, A_aySyy * n);
        st<NT>(A, q, gyc.z * aySyz + gyc.w * dySyz * dt, A_aySyz * n);
    }
    if (onz) {
        fresh(q);
        st<NT>(A, q, gzc.z * azSxz + gzc.w * dzSxz * dt, A_azSxz * n);
        st<NT>(A, q, gzc.z * azSyz + gzc.w * dzSyz * dt, A_azSyz * n);
        st<NT>(A, q, gze.z * azSzz + gze.w * dzSzz * dt, A_azSzz * n);
    }
}

// ---------------------------------------------------------------------------
// Interior columns (m_kernel, and the bottom PML band of the same columns).
// Tiles of 64 x BY columns over full-width aligned rows; lanes outside
// [ib,ie] x [jb,je] idle.  Chunks run over k = 1..nz: planes 1..ke take the
// interior update, planes ke+1..nz (the bottom PML, kbeg_a = nz-na+1) the
// ADE-CFS update, in two branch-free loops sharing the z queues.
// ---------------------------------------------------------------------------

// kernel__update_stress, m_kernel.f90:142-348 (normal and shear parts fused:
// both read V and write disjoint arrays)
// The velocities the stress update of one cell reads: the z, x and y lines
// through the cell (m_kernel.f90:198-333)
struct VStencil {
    float vx_m1, vx_0, vx_p1, vx_p2, vx_im2, vx_im1, vx_ip1, vx_jm1, vx_jp1, vx_jp2;
    float vy_m1, vy_0, vy_p1, vy_p2, vy_im1, vy_ip1, vy_ip2, vy_jm2, vy_jm1, vy_jp1;
    float vz_m2, vz_m1, vz_0, vz_p1, vz_im1, vz_ip1, vz_ip2, vz_jm1, vz_jp1, vz_jp2;
};

// kernel__update_stress for one cell of the interior box, m_kernel.f90:198-333:
// the normal and shear stresses and their memory variables.  p: field index,
// r: memory-variable index, in: the cell is in the 2nd-order band, mu..: mu
// at (i,j), (i+1,j), (i,j+1) on planes k and k+1 (n) and at (i+1,j+1) on
// plane k.  OOP: the old stresses are read from a.fin.
template <int NM, bool NT, bool OOP, bool TP>
__device__ __forceinline__ void stress_cell(const StepArgs &a, const Loc &p, const Loc &r, int k, bool in, const Coefs &cf,
                                            const Taper<TP> &tp, const VStencil &v,
                                            float mu00, float mu00n, float mu10, float mu10n, float mu01, float mu01n,
                                            float mu11)
{
    float *__restrict__ Sxx = a.f.Sxx;
    float *__restrict__ Syy = a.f.Syy;
    float *__restrict__ Szz = a.f.Szz;
    float *__restrict__ Syz = a.f.Syz;
    float *__restrict__ Sxz = a.f.Sxz;
    float *__restrict__ Sxy = a.f.Sxy;
    const float *__restrict__ SxxI = OOP ? a.fin.Sxx : Sxx;
    const float *__restrict__ SyyI = OOP ? a.fin.Syy : Syy;
    const float *__restrict__ SzzI = OOP ? a.fin.Szz : Szz;
    const float *__restrict__ SyzI = OOP ? a.fin.Syz : Syz;
    const float *__restrict__ SxzI = OOP ? a.fin.Sxz : Sxz;
    const float *__restrict__ SxyI = OOP ? a.fin.Sxy : Sxy;
    const float dt = a.dt;
    const float d2 = a.v.d2;
    const long long rn = a.g.rn;
    // every load comes before the first store: the fields may alias for the
    // compiler, and a load left between two stores waits for both
    const float lam1 = ld<NT>(a.m.lam, p);
    float taup1 = 0.0f, taus1 = 0.0f;
    if (NM > 0 || a.tau) {
        taup1 = ld<NT>(a.m.taup, p);
        taus1 = ld<NT>(a.m.taus, p);
    }
    float sxx = ld<NT>(SxxI, p), syy = ld<NT>(SyyI, p), szz = ld<NT>(SzzI, p);
    float syz = ld<NT>(SyzI, p), sxz = ld<NT>(SxzI, p), sxy = ld<NT>(SxyI, p);
    RCell<NM> R;
    R.template load<NT>(a.R, rn, r);

    const float re40x = cf.at(in, 0);
    const float re41x = cf.at(in, 1);
    const float re40y = cf.at(in, 2);
    const float re41y = cf.at(in, 3);
    const float re40z = cf.at(in, 4);
    const float re41z = cf.at(in, 5);

    // normal components, m_kernel.f90:198-238
    const float dxVx = (v.vx_0 - v.vx_im1) * re40x - (v.vx_ip1 - v.vx_im2) * re41x;
    const float dyVy = (v.vy_0 - v.vy_jm1) * re40y - (v.vy_jp1 - v.vy_jm2) * re41y;
    const float dzVz = (v.vz_0 - v.vz_m1) * re40z - (v.vz_p1 - v.vz_m2) * re41z;

    const float mu2 = 2.0f * mu00;
    const float lam2mu = lam1 + mu2;
    const float d3v3 = dxVx + dyVy + dzVz;
    const float dyVy_dzVz = dyVy + dzVz;
    const float dxVx_dzVz = dxVx + dzVz;
    const float dxVx_dyVy = dxVx + dyVy;

    float Rxx_n = 0.0f, Ryy_n = 0.0f, Rzz_n = 0.0f;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const float c1 = a.v.c1[m], c2 = a.v.c2[m], d1 = a.v.d1[m];
        const float nxx = c1 * R.v[0 * NM + m] - c2 * (lam2mu * taup1 * d3v3 - mu2 * taus1 * dyVy_dzVz) * dt;
        const float nyy = c1 * R.v[1 * NM + m] - c2 * (lam2mu * taup1 * d3v3 - mu2 * taus1 * dxVx_dzVz) * dt;
        const float nzz = c1 * R.v[2 * NM + m] - c2 * (lam2mu * taup1 * d3v3 - mu2 * taus1 * dxVx_dyVy) * dt;
        R.v[0 * NM + m] = nxx;
        R.v[1 * NM + m] = nyy;
        R.v[2 * NM + m] = nzz;
        Rxx_n = Rxx_n + d1 * nxx;
        Ryy_n = Ryy_n + d1 * nyy;
        Rzz_n = Rzz_n + d1 * nzz;
    }
    const float taup_plus1 = 1.0f + taup1 * (1.0f + d2);
    const float taus_plus1 = 1.0f + taus1 * (1.0f + d2);
    sxx = sxx + (lam2mu * taup_plus1 * d3v3 - mu2 * taus_plus1 * dyVy_dzVz + Rxx_n) * dt;
    syy = syy + (lam2mu * taup_plus1 * d3v3 - mu2 * taus_plus1 * dxVx_dzVz + Ryy_n) * dt;
    szz = szz + (lam2mu * taup_plus1 * d3v3 - mu2 * taus_plus1 * dxVx_dyVy + Rzz_n) * dt;

    // shear components, m_kernel.f90:285-333
    const float dxVy_dyVx = (v.vy_ip1 - v.vy_0) * re40x - (v.vy_ip2 - v.vy_im1) * re41x
                          + (v.vx_jp1 - v.vx_0) * re40y - (v.vx_jp2 - v.vx_jm1) * re41y;
    const float dxVz_dzVx = (v.vz_ip1 - v.vz_0) * re40x - (v.vz_ip2 - v.vz_im1) * re41x
                          + (v.vx_p1 - v.vx_0) * re40z - (v.vx_p2 - v.vx_m1) * re41z;
    const float dyVz_dzVy = (v.vz_jp1 - v.vz_0) * re40y - (v.vz_jp2 - v.vz_jm1) * re41y
                          + (v.vy_p1 - v.vy_0) * re40z - (v.vy_p2 - v.vy_m1) * re41z;

    const float muxz = hmean4(mu00, mu00n, mu10, mu10n, EPSL);
    const float muxy = hmean4(mu00, mu10, mu01, mu11, EPSL);
    const float muyz = hmean4(mu00, mu00n, mu01, mu01n, EPSL);

    float Ryz_n = 0.0f, Rxz_n = 0.0f, Rxy_n = 0.0f;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const float c1 = a.v.c1[m], c2 = a.v.c2[m], d1 = a.v.d1[m];
        const float nyz = c1 * R.v[3 * NM + m] - c2 * muyz * taus1 * dyVz_dzVy * dt;
        const float nxz = c1 * R.v[4 * NM + m] - c2 * muxz * taus1 * dxVz_dzVx * dt;
        const float nxy = c1 * R.v[5 * NM + m] - c2 * muxy * taus1 * dxVy_dyVx * dt;
        R.v[3 * NM + m] = nyz;
        R.v[4 * NM + m] = nxz;
        R.v[5 * NM + m] = nxy;
        Ryz_n = Ryz_n + d1 * nyz;
        Rxz_n = Rxz_n + d1 * nxz;
        Rxy_n = Rxy_n + d1 * nxy;
    }
    R.template store<NT>(a.R, rn, r);
    syz = syz + (muyz * taus_plus1 * dyVz_dzVy + Ryz_n) * dt;
    sxz = sxz + (muxz * taus_plus1 * dxVz_dzVx + Rxz_n) * dt;
    sxy = sxy + (muxy * taus_plus1 * dxVy_dyVx + Rxy_n) * dt;
    if (TP && (a.mask & MASK_TAPER)) {
        const float zc = ldv<false>(a.cgz_c + (k + 2)), zb = ldv<false>(a.cgz_b + (k + 2));
        const float ccc = tp.xc * tp.yc * zc;
        sxx = sxx * ccc;
        syy = syy * ccc;
        szz = szz * ccc;
        syz = syz * tp.xc * tp.yb * zb;
        sxz = sxz * tp.xb * tp.yc * zb;
        sxy = sxy * tp.xb * tp.yb * zc;
    }
    st<NT>(Sxx, p, sxx);
    st<NT>(Syy, p, syy);
    st<NT>(Szz, p, szz);
    st<NT>(Syz, p, syz);
    st<NT>(Sxz, p, sxz);
    st<NT>(Sxy, p, sxy);
}

// logical tile (bx, by, bz) of interior tile bid, x fastest; xcd_remap gives
// the blocks of one XCD a contiguous run of them
__device__ static inline void plain_tile(const StepArgs &a, int bid, int &bx, int &byy, int &bz)
{
    bx = bid % a.nbx;
    const int t = bid / a.nbx;
    byy = t % a.nby;
    bz = t / a.nby;
}

template <int NM, bool NT, bool OOP, bool TP>
__device__ __forceinline__ void stress_int_body(const StepArgs &a, int bx, int byy, int bz)
{
    const Grid &g = a.g;
    const int it = 1 + (a.bx0 + bx) * a.bxw, jt = g.jb + byy * a.byi;   // the tile's first cell
    const int i = it + threadIdx.x, j = jt + threadIdx.y;
    if (i < g.ib || i > g.ie || j > g.je) return;
    const int k0 = uni(ldv<false>(a.zc + bz));
    const int k1 = uni(ldv<false>(a.zc + bz + 1)) - 1;
    const int ka1 = (a.mask & MASK_INT) ? min(k1, g.ke) : k0 - 1;      // interior planes k0..ka1
    const int kb0 = max(k0, g.ke + 1);
    const int kb1 = (a.has_pml && (a.mask & MASK_PML)) ? k1 : kb0 - 1;  // bottom PML planes kb0..kb1
    if (ka1 < k0 && kb1 < kb0) return;
    const int ks = ka1 >= k0 ? k0 : kb0;

    const long long P = g.plane;
    const float *__restrict__ Vx = a.f.Vx;
    const float *__restrict__ Vy = a.f.Vy;
    const float *__restrict__ Vz = a.f.Vz;
    const float *__restrict__ mu = a.m.mu;

    Loc p = field_loc(g, it, jt, ks, threadIdx.x, threadIdx.y);
    float vx_m1 = ld(Vx, p, -P), vx_0 = ld(Vx, p), vx_p1 = ld(Vx, p, P);
    float vy_m1 = ld(Vy, p, -P), vy_0 = ld(Vy, p), vy_p1 = ld(Vy, p, P);
    float vz_m2 = ld(Vz, p, -2 * P), vz_m1 = ld(Vz, p, -P), vz_0 = ld(Vz, p);
    float mu00 = ld(mu, p), mu10 = ld(mu, p, 0, 1), mu01 = ld(mu, p, 0, 0, 1), mu11 = ld(mu, p, 0, 1, 1);

    if (ka1 >= k0) {
        const long long c2 = g2idx(g, i, j);
        const int kft = ldv<false>(a.m.kfs_top + c2), kfb = ldv<false>(a.m.kfs_bot + c2);
        const int kot = ldv<false>(a.m.kob_top + c2), kobb = ldv<false>(a.m.kob_bot + c2);
        const Coefs cf(a);
        const Taper<TP> tp(a, i, j);
        Loc r = {((long long)(k0 - g.kb) * g.nyk + (jt - g.jb)) * g.rpitch + (it - 1),
                 4u * (threadIdx.y * g.rpitch + threadIdx.x), 0u};
        for (int k = k0; k <= ka1; ++k, p.u += P, r.u += g.rplane) {
            fresh(p);
            fresh(r);
            const float vx_p2 = ld(Vx, p, 2 * P), vy_p2 = ld(Vy, p, 2 * P), vz_p1 = ld(Vz, p, P);
            const float mu00n = ld(mu, p, P), mu10n = ld(mu, p, P, 1), mu01n = ld(mu, p, P, 0, 1);
            const float mu11n = ld(mu, p, P, 1, 1);

            VStencil v;
            v.vx_m1 = vx_m1; v.vx_0 = vx_0; v.vx_p1 = vx_p1; v.vx_p2 = vx_p2;
            v.vy_m1 = vy_m1; v.vy_0 = vy_0; v.vy_p1 = vy_p1; v.vy_p2 = vy_p2;
            v.vz_m2 = vz_m2; v.vz_m1 = vz_m1; v.vz_0 = vz_0; v.vz_p1 = vz_p1;
            v.vx_im2 = ld(Vx, p, 0, -2); v.vx_im1 = ld(Vx, p, 0, -1); v.vx_ip1 = ld(Vx, p, 0, 1);
            v.vx_jm1 = ld(Vx, p, 0, 0, -1); v.vx_jp1 = ld(Vx, p, 0, 0, 1); v.vx_jp2 = ld(Vx, p, 0, 0, 2);
            v.vy_jm2 = ld(Vy, p, 0, 0, -2); v.vy_jm1 = ld(Vy, p, 0, 0, -1); v.vy_jp1 = ld(Vy, p, 0, 0, 1);
            v.vy_im1 = ld(Vy, p, 0, -1); v.vy_ip1 = ld(Vy, p, 0, 1); v.vy_ip2 = ld(Vy, p, 0, 2);
            v.vz_im1 = ld(Vz, p, 0, -1); v.vz_ip1 = ld(Vz, p, 0, 1); v.vz_ip2 = ld(Vz, p, 0, 2);
            v.vz_jm1 = ld(Vz, p, 0, 0, -1); v.vz_jp1 = ld(Vz, p, 0, 0, 1); v.vz_jp2 = ld(Vz, p, 0, 0, 2);
            stress_cell<NM, NT, OOP, TP>(a, p, r, k, in_band(k, kft, kfb, kot, kobb), cf, tp, v, mu00, mu00n, mu10, mu10n, mu01, mu01n,
                                     mu11);

            // rotate the z queues
            vx_m1 = vx_0; vx_0 = vx_p1; vx_p1 = vx_p2;
            vy_m1 = vy_0; vy_0 = vy_p1; vy_p1 = vy_p2;
            vz_m2 = vz_m1; vz_m1 = vz_0; vz_0 = vz_p1;
            mu00 = mu00n; mu10 = mu10n; mu01 = mu01n; mu11 = mu11n;
        }
    }
    if (kb1 >= kb0) {
        // bottom PML band of the interior columns (box 4)
        const PmlBox b = a.box[4];
        const long long astride = (long long)b.nxb * b.nyb;
        Loc q = {b.off + (long long)(jt - b.j0) * b.nxb + (it - b.i0) + (long long)(kb0 - b.k0) * astride,
                 4u * (threadIdx.y * b.nxb + threadIdx.x), 0u};
        const float4 gxc = ldp(a.gxc + (i - 1)), gxe = ldp(a.gxe + (i - 1));
        const float4 gyc = ldp(a.gyc + (j - 1)), gye = ldp(a.gye + (j - 1));
        for (int k = kb0; k <= kb1; ++k, p.u += P, q.u += astride) {
            fresh(p);
            fresh(q);
            const float vx_p2 = ld(Vx, p, 2 * P), vy_p2 = ld(Vy, p, 2 * P), vz_p1 = ld(Vz, p, P);
            const float mu00n = ld(mu, p, P), mu10n = ld(mu, p, P, 1), mu01n = ld(mu, p, P, 0, 1);
            const float mu11n = ld(mu, p, P, 1, 1);
            pml_stress_cell<NT, OOP>(a, p, q, k, vx_0, vx_p1, vy_0, vy_p1, vz_m1, vz_0, mu00, mu00n, mu10, mu10n, mu01,
                                mu01n, mu11, gxc, gxe, gyc, gye);
            vx_m1 = vx_0; vx_0 = vx_p1; vx_p1 = vx_p2;
            vy_m1 = vy_0; vy_0 = vy_p1; vy_p1 = vy_p2;
            vz_m2 = vz_m1; vz_m1 = vz_0; vz_0 = vz_p1;
            mu00 = mu00n; mu10 = mu10n; mu01 = mu01n; mu11 = mu11n;
        }
    }
}

// batched launch: tile = (member, bx, by, bz), member arguments in HBM
template <int NM, bool NT, bool TP>
__global__ void __launch_bounds__(256) WAVES_NM k_stress_int_b(const StepArgs *__restrict__ mem, const int4 *__restrict__ tiles)
{
    const int4 t = uni(tiles[xcd_remap(blockIdx.x, gridDim.x)]);
    stress_int_body<NM, NT, false, TP>(mem[t.x], t.y, t.z, t.w);
}

// kernel__update_vel, m_kernel.f90:75-140, then the bottom PML band.
// (Loading plane k+1 while computing plane k gained 1 % at three waves per
// SIMD and nothing at four.)
template <bool OOP, bool TP>
__device__ __forceinline__ void vel_int_body(const StepArgs &a, int bx, int byy, int bz)
{
    const Grid &g = a.g;
    const int it = 1 + (a.bx0 + bx) * a.bxw, jt = g.jb + byy * a.byi;   // the tile's first cell
    const int i = it + threadIdx.x, j = jt + threadIdx.y;
    if (i < g.ib || i > g.ie || j > g.je) return;
    const int k0 = uni(ldv<false>(a.zc + bz));
    const int k1 = uni(ldv<false>(a.zc + bz + 1)) - 1;
    const int ka1 = (a.mask & MASK_INT) ? min(k1, g.ke) : k0 - 1;
    const int kb0 = max(k0, g.ke + 1);
    const int kb1 = (a.has_pml && (a.mask & MASK_PML)) ? k1 : kb0 - 1;
    if (ka1 < k0 && kb1 < kb0) return;
    const int ks = ka1 >= k0 ? k0 : kb0;

    const long long P = g.plane;
    const float *__restrict__ Sxx = a.f.Sxx;
    const float *__restrict__ Syy = a.f.Syy;
    const float *__restrict__ Szz = a.f.Szz;
    const float *__restrict__ Syz = a.f.Syz;
    const float *__restrict__ Sxz = a.f.Sxz;
    const float *__restrict__ Sxy = a.f.Sxy;
    const float *__restrict__ rho = a.m.rho;
    float *__restrict__ Vx = a.f.Vx;
    float *__restrict__ Vy = a.f.Vy;
    float *__restrict__ Vz = a.f.Vz;
    const float dt = a.dt;

    Loc p = field_loc(g, it, jt, ks, threadIdx.x, threadIdx.y);
    float sxz_m2 = ld(Sxz, p, -2 * P), sxz_m1 = ld(Sxz, p, -P), sxz_0 = ld(Sxz, p);
    float syz_m2 = ld(Syz, p, -2 * P), syz_m1 = ld(Syz, p, -P), syz_0 = ld(Syz, p);
    float szz_m1 = ld(Szz, p, -P), szz_0 = ld(Szz, p), szz_p1 = ld(Szz, p, P);
    float rho0 = ld(rho, p);

    if (ka1 >= k0) {
        const long long c2 = g2idx(g, i, j);
        const int kft = ldv<false>(a.m.kfs_top + c2), kfb = ldv<false>(a.m.kfs_bot + c2);
        const int kot = ldv<false>(a.m.kob_top + c2), kobb = ldv<false>(a.m.kob_bot + c2);
        const Coefs cf(a);
        const Taper<TP> tp(a, i, j);
        for (int k = k0; k <= ka1; ++k, p.u += P) {
            fresh(p);
            const float sxz_p1 = ld(Sxz, p, P), syz_p1 = ld(Syz, p, P), szz_p2 = ld(Szz, p, 2 * P);
            const float rho_kp = ld(rho, p, P);

            const bool in = in_band(k, kft, kfb, kot, kobb);
            const float re40x = cf.at(in, 0);
            const float re41x = cf.at(in, 1);
            const float re40y = cf.at(in, 2);
            const float re41y = cf.at(in, 3);
            const float re40z = cf.at(in, 4);
            const float re41z = cf.at(in, 5);

            const float rho_ip = ld(rho, p, 0, 1), rho_jp = ld(rho, p, 0, 0, 1);
            const float vx = ld<true>(OOP ? a.fin.Vx : Vx, p), vy = ld<true>(OOP ? a.fin.Vy : Vy, p);
            const float vz = ld<true>(OOP ? a.fin.Vz : Vz, p);
            const float sxx_im1 = ld(Sxx, p, 0, -1), sxx_0 = ld(Sxx, p), sxx_ip1 = ld(Sxx, p, 0, 1), sxx_ip2 = ld(Sxx, p, 0, 2);
            const float sxy_0 = ld(Sxy, p);
            const float sxy_jm2 = ld(Sxy, p, 0, 0, -2), sxy_jm1 = ld(Sxy, p, 0, 0, -1), sxy_jp1 = ld(Sxy, p, 0, 0, 1);
            const float sxy_im2 = ld(Sxy, p, 0, -2), sxy_im1 = ld(Sxy, p, 0, -1), sxy_ip1 = ld(Sxy, p, 0, 1);
            const float syy_jm1 = ld(Syy, p, 0, 0, -1), syy_0 = ld(Syy, p), syy_jp1 = ld(Syy, p, 0, 0, 1), syy_jp2 = ld(Syy, p, 0, 0, 2);
            const float syz_jm2 = ld(Syz, p, 0, 0, -2), syz_jm1 = ld(Syz, p, 0, 0, -1), syz_jp1 = ld(Syz, p, 0, 0, 1);
            const float sxz_im2 = ld(Sxz, p, 0, -2), sxz_im1 = ld(Sxz, p, 0, -1), sxz_ip1 = ld(Sxz, p, 0, 1);

            const float d3Sx3 = (sxx_ip1 - sxx_0) * re40x - (sxx_ip2 - sxx_im1) * re41x
                              + (sxy_0 - sxy_jm1) * re40y - (sxy_jp1 - sxy_jm2) * re41y
                              + (sxz_0 - sxz_m1) * re40z - (sxz_p1 - sxz_m2) * re41z;
            const float d3Sy3 = (sxy_0 - sxy_im1) * re40x - (sxy_ip1 - sxy_im2) * re41x
                              + (syy_jp1 - syy_0) * re40y - (syy_jp2 - syy_jm1) * re41y
                              + (syz_0 - syz_m1) * re40z - (syz_p1 - syz_m2) * re41z;
            const float d3Sz3 = (sxz_0 - sxz_im1) * re40x - (sxz_ip1 - sxz_im2) * re41x
                              + (syz_0 - syz_jm1) * re40y - (syz_jp1 - syz_jm2) * re41y
                              + (szz_p1 - szz_0) * re40z - (szz_p2 - szz_m1) * re41z;

            float nx = vx + 2.0f / (rho0 + rho_ip) * d3Sx3 * dt;
            float ny = vy + 2.0f / (rho0 + rho_jp) * d3Sy3 * dt;
            float nz = vz + 2.0f / (rho0 + rho_kp) * d3Sz3 * dt;
            if (TP && (a.mask & MASK_TAPER)) {
                const float zc = ldv<false>(a.cgz_c + (k + 2)), zb = ldv<false>(a.cgz_b + (k + 2));
                nx = nx * tp.xb * tp.yc * zc;
                ny = ny * tp.xc * tp.yb * zc;
                nz = nz * tp.xc * tp.yc * zb;
            }
            st<true>(Vx, p, nx);
            st<true>(Vy, p, ny);
            st<true>(Vz, p, nz);

            sxz_m2 = sxz_m1; sxz_m1 = sxz_0; sxz_0 = sxz_p1;
            syz_m2 = syz_m1; syz_m1 = syz_0; syz_0 = syz_p1;
            szz_m1 = szz_0; szz_0 = szz_p1; szz_p1 = szz_p2;
            rho0 = rho_kp;
        }
    }
    if (kb1 >= kb0) {
        const PmlBox b = a.box[4];
        const long long astride = (long long)b.nxb * b.nyb;
        Loc q = {b.off + (long long)(jt - b.j0) * b.nxb + (it - b.i0) + (long long)(kb0 - b.k0) * astride,
                 4u * (threadIdx.y * b.nxb + threadIdx.x), 0u};
        const float4 gxc = ldp(a.gxc + (i - 1)), gxe = ldp(a.gxe + (i - 1));
        const float4 gyc = ldp(a.gyc + (j - 1)), gye = ldp(a.gye + (j - 1));
        for (int k = kb0; k <= kb1; ++k, p.u += P, q.u += astride) {
            fresh(p);
            fresh(q);
            const float sxz_p1 = ld(Sxz, p, P), syz_p1 = ld(Syz, p, P), szz_p2 = ld(Szz, p, 2 * P);
            const float rho_kp = ld(rho, p, P);
            pml_vel_cell<true, OOP>(a, p, q, k, szz_0, szz_p1, syz_m1, syz_0, sxz_m1, sxz_0, rho0, rho_kp, gxc, gxe, gyc, gye);
            sxz_m2 = sxz_m1; sxz_m1 = sxz_0; sxz_0 = sxz_p1;
            syz_m2 = syz_m1; syz_m1 = syz_0; syz_0 = syz_p1;
            szz_m1 = szz_0; szz_0 = szz_p1; szz_p1 = szz_p2;
            rho0 = rho_kp;
        }
    }
}

template <bool TP>
__global__ void __launch_bounds__(256) WAVES4 k_vel_int_b(const StepArgs *__restrict__ mem, const int4 *__restrict__ tiles)
{
    const int4 t = uni(tiles[xcd_remap_rev(blockIdx.x, gridDim.x)]);
    vel_int_body<false, TP>(mem[t.x], t.y, t.z, t.w);
}

// ---------------------------------------------------------------------------
// Velocity and stress in one z-march (variant bit 7).  One launch runs
// kernel__update_vel of step n and kernel__update_stress of step n+1 over the
// interior box, so the stresses cross HBM once for both updates and the new
// velocities reach the stress stencil through LDS instead of HBM.  The old
// fields are read from a.fin and the new ones written to a.f (two buffer sets
// that swap every step), so a tile recomputes the velocities of the cells
// around it from old values that no other tile overwrites.  A tile is FW x TY
// stress columns (TY = 4 SR); its 64 x (TY + 4) velocity columns (two halo
// columns and rows on each side) run two planes ahead of the stress update
// and are kept in a ring of six planes in LDS.  Velocities outside the
// interior box (side slabs, bottom band, outer halo) are read from a.f, where
// the side-column and band launches that precede this one have put them.
// ---------------------------------------------------------------------------
#define FW (BX - 4)

template <int NM, int SR>
__global__ void __launch_bounds__(256) k_fused(StepArgs a)
{
    constexpr int TY = 4 * SR, VR = TY + 4, NS = 6;
    __shared__ float vs[NS][3][VR][BX];
    int bx, byy, bz;
    plain_tile(a, xcd_remap(blockIdx.x, gridDim.x), bx, byy, bz);
    const Grid &g = a.g;
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int i0 = g.ib + bx * FW, j0 = g.jb + byy * TY;
    const int il = min(i0 + FW - 1, g.ie), jl = min(j0 + TY - 1, g.je);  // last stress column and row
    const int k0 = a.zc[bz], k1 = a.zc[bz + 1] - 1;                      // interior planes k0..k1
    const long long P = g.plane;
    const int Y = g.pitch;
    const float dt = a.dt;
    const float *__restrict__ Sxx = a.fin.Sxx;
    const float *__restrict__ Syy = a.fin.Syy;
    const float *__restrict__ Szz = a.fin.Szz;
    const float *__restrict__ Syz = a.fin.Syz;
    const float *__restrict__ Sxz = a.fin.Sxz;
    const float *__restrict__ Sxy = a.fin.Sxy;
    const float *__restrict__ rho = a.m.rho;
    const float *__restrict__ mu = a.m.mu;

    const Coefs cf(a);
    const Taper<false> tp(a, 1, 1);
    // velocity points of this thread: column iv, rows j0 - 2 + ty + 4 r.
    // vf: 0 not needed by the tile, 1 read from a.f, 2 computed, 3 computed
    // and stored (the tile's own cells)
    const int iv = i0 - 2 + tx;
    const int kq = max(k0 - 2, g.kb);   // first computed plane: the z queues start there
    int vf[SR + 1], vb[SR + 1][4];
    float sxz_m2[SR + 1], sxz_m1[SR + 1], sxz_0[SR + 1], syz_m2[SR + 1], syz_m1[SR + 1], syz_0[SR + 1];
    float szz_m1[SR + 1], szz_0[SR + 1], szz_p1[SR + 1], rho0[SR + 1];
#pragma unroll
    for (int r = 0; r <= SR; ++r) {
        const int jv = j0 - 2 + ty + 4 * r;
        const bool need = iv <= il + 2 && jv <= jl + 2;
        const bool comp = need && iv >= g.ib && iv <= g.ie && jv >= g.jb && jv <= g.je;
        const bool own = comp && iv >= i0 && iv <= il && jv >= j0 && jv <= jl;
        vf[r] = !need ? 0 : !comp ? 1 : own ? 3 : 2;
        vb[r][0] = vb[r][1] = vb[r][2] = vb[r][3] = 0;
        sxz_m2[r] = sxz_m1[r] = sxz_0[r] = syz_m2[r] = syz_m1[r] = syz_0[r] = 0.0f;
        szz_m1[r] = szz_0[r] = szz_p1[r] = rho0[r] = 0.0f;
        if (comp) {
            const long long c2 = g2idx(g, iv, jv);
            vb[r][0] = a.m.kfs_top[c2]; vb[r][1] = a.m.kfs_bot[c2];
            vb[r][2] = a.m.kob_top[c2]; vb[r][3] = a.m.kob_bot[c2];
            const long long p = gidx(g, iv, jv, kq);
            sxz_m2[r] = Sxz[p - 2 * P]; sxz_m1[r] = Sxz[p - P]; sxz_0[r] = Sxz[p];
            syz_m2[r] = Syz[p - 2 * P]; syz_m1[r] = Syz[p - P]; syz_0[r] = Syz[p];
            szz_m1[r] = Szz[p - P]; szz_0[r] = Szz[p]; szz_p1[r] = Szz[p + P];
            rho0[r] = rho[p];
        }
    }

    // stress cells of this thread: column is, rows j0 + ty + 4 s
    const int is = i0 + tx;
    bool sa[SR];
    int sb[SR][4];
    float mu00[SR], mu10[SR], mu01[SR], mu11[SR];
#pragma unroll
    for (int s = 0; s < SR; ++s) {
        const int js = j0 + ty + 4 * s;
        sa[s] = tx < FW && is <= il && js <= jl;
        sb[s][0] = sb[s][1] = sb[s][2] = sb[s][3] = 0;
        mu00[s] = mu10[s] = mu01[s] = mu11[s] = 0.0f;
        if (sa[s]) {
            const long long c2 = g2idx(g, is, js);
            sb[s][0] = a.m.kfs_top[c2]; sb[s][1] = a.m.kfs_bot[c2];
            sb[s][2] = a.m.kob_top[c2]; sb[s][3] = a.m.kob_bot[c2];
            const long long p = gidx(g, is, js, k0);
            mu00[s] = mu[p]; mu10[s] = mu[p + 1]; mu01[s] = mu[p + Y]; mu11[s] = mu[p + 1 + Y];
        }
    }

    for (int kv = k0 - 2; kv <= k1 + 2; ++kv) {
        // velocities of plane kv, kernel__update_vel (m_kernel.f90:75-140)
        const int sl = (kv - k0 + 2) % NS;
#pragma unroll
        for (int r = 0; r <= SR; ++r) {
            if (vf[r] == 0) continue;
            const int row = ty + 4 * r;
            const long long p = gidx(g, iv, j0 - 2 + row, kv);
            float vx, vy, vz;
            if (vf[r] >= 2 && kv >= g.kb && kv <= g.ke) {
                const float sxz_p1 = Sxz[p + P], syz_p1 = Syz[p + P], szz_p2 = Szz[p + 2 * P];
                const float rho_kp = rho[p + P];
                const bool in = in_band(kv, vb[r][0], vb[r][1], vb[r][2], vb[r][3]);
                const float re40x = cf.at(in, 0);
                const float re41x = cf.at(in, 1);
                const float re40y = cf.at(in, 2);
                const float re41y = cf.at(in, 3);
                const float re40z = cf.at(in, 4);
                const float re41z = cf.at(in, 5);

                const float sxx_im1 = Sxx[p - 1], sxx_0 = Sxx[p], sxx_ip1 = Sxx[p + 1], sxx_ip2 = Sxx[p + 2];
                const float sxy_0 = Sxy[p];
                const float sxy_jm2 = Sxy[p - 2 * Y], sxy_jm1 = Sxy[p - Y], sxy_jp1 = Sxy[p + Y];
                const float sxy_im2 = Sxy[p - 2], sxy_im1 = Sxy[p - 1], sxy_ip1 = Sxy[p + 1];
                const float syy_jm1 = Syy[p - Y], syy_0 = Syy[p], syy_jp1 = Syy[p + Y], syy_jp2 = Syy[p + 2 * Y];
                const float syz_jm2 = Syz[p - 2 * Y], syz_jm1 = Syz[p - Y], syz_jp1 = Syz[p + Y];
                const float sxz_im2 = Sxz[p - 2], sxz_im1 = Sxz[p - 1], sxz_ip1 = Sxz[p + 1];

                const float d3Sx3 = (sxx_ip1 - sxx_0) * re40x - (sxx_ip2 - sxx_im1) * re41x
                                  + (sxy_0 - sxy_jm1) * re40y - (sxy_jp1 - sxy_jm2) * re41y
                                  + (sxz_0[r] - sxz_m1[r]) * re40z - (sxz_p1 - sxz_m2[r]) * re41z;
                const float d3Sy3 = (sxy_0 - sxy_im1) * re40x - (sxy_ip1 - sxy_im2) * re41x
                                  + (syy_jp1 - syy_0) * re40y - (syy_jp2 - syy_jm1) * re41y
                                  + (syz_0[r] - syz_m1[r]) * re40z - (syz_p1 - syz_m2[r]) * re41z;
                const float d3Sz3 = (sxz_0[r] - sxz_im1) * re40x - (sxz_ip1 - sxz_im2) * re41x
                                  + (syz_0[r] - syz_jm1) * re40y - (syz_jp1 - syz_jm2) * re41y
                                  + (szz_p1[r] - szz_0[r]) * re40z - (szz_p2 - szz_m1[r]) * re41z;

                vx = ldv<true>(a.fin.Vx + p) + 2.0f / (rho0[r] + rho[p + 1]) * d3Sx3 * dt;
                vy = ldv<true>(a.fin.Vy + p) + 2.0f / (rho0[r] + rho[p + Y]) * d3Sy3 * dt;
                vz = ldv<true>(a.fin.Vz + p) + 2.0f / (rho0[r] + rho_kp) * d3Sz3 * dt;
                if (vf[r] == 3 && kv >= k0 && kv <= k1) {
                    stv<true>(a.f.Vx + p, vx);
                    stv<true>(a.f.Vy + p, vy);
                    stv<true>(a.f.Vz + p, vz);
                }
                sxz_m2[r] = sxz_m1[r]; sxz_m1[r] = sxz_0[r]; sxz_0[r] = sxz_p1;
                syz_m2[r] = syz_m1[r]; syz_m1[r] = syz_0[r]; syz_0[r] = syz_p1;
                szz_m1[r] = szz_0[r]; szz_0[r] = szz_p1[r]; szz_p1[r] = szz_p2;
                rho0[r] = rho_kp;
            } else {
                vx = a.f.Vx[p];
                vy = a.f.Vy[p];
                vz = a.f.Vz[p];
            }
            vs[sl][0][row][tx] = vx;
            vs[sl][1][row][tx] = vy;
            vs[sl][2][row][tx] = vz;
        }
        __syncthreads();

        // stresses of plane kv - 2 from the velocities of planes kv - 4 .. kv
        const int k = kv - 2;
        if (k < k0) continue;
        const int s0 = (k - k0 + 2) % NS, sm1 = (k - k0 + 1) % NS, sm2 = (k - k0) % NS;
        const int sp1 = (k - k0 + 3) % NS, sp2 = (k - k0 + 4) % NS;
#pragma unroll
        for (int s = 0; s < SR; ++s) {
            if (!sa[s]) continue;
            const int row = ty + 4 * s + 2, col = tx + 2;
            const int js = j0 + ty + 4 * s;
            const long long p = gidx(g, is, js, k);
            const float mu00n = mu[p + P], mu10n = mu[p + P + 1], mu01n = mu[p + P + Y];
            VStencil v;
            v.vx_m1 = vs[sm1][0][row][col]; v.vx_0 = vs[s0][0][row][col];
            v.vx_p1 = vs[sp1][0][row][col]; v.vx_p2 = vs[sp2][0][row][col];
            v.vy_m1 = vs[sm1][1][row][col]; v.vy_0 = vs[s0][1][row][col];
            v.vy_p1 = vs[sp1][1][row][col]; v.vy_p2 = vs[sp2][1][row][col];
            v.vz_m2 = vs[sm2][2][row][col]; v.vz_m1 = vs[sm1][2][row][col];
            v.vz_0 = vs[s0][2][row][col]; v.vz_p1 = vs[sp1][2][row][col];
            v.vx_im2 = vs[s0][0][row][col - 2]; v.vx_im1 = vs[s0][0][row][col - 1];
            v.vx_ip1 = vs[s0][0][row][col + 1];
            v.vx_jm1 = vs[s0][0][row - 1][col]; v.vx_jp1 = vs[s0][0][row + 1][col];
            v.vx_jp2 = vs[s0][0][row + 2][col];
            v.vy_jm2 = vs[s0][1][row - 2][col]; v.vy_jm1 = vs[s0][1][row - 1][col];
            v.vy_jp1 = vs[s0][1][row + 1][col];
            v.vy_im1 = vs[s0][1][row][col - 1]; v.vy_ip1 = vs[s0][1][row][col + 1];
            v.vy_ip2 = vs[s0][1][row][col + 2];
            v.vz_im1 = vs[s0][2][row][col - 1]; v.vz_ip1 = vs[s0][2][row][col + 1];
            v.vz_ip2 = vs[s0][2][row][col + 2];
            v.vz_jm1 = vs[s0][2][row - 1][col]; v.vz_jp1 = vs[s0][2][row + 1][col];
            v.vz_jp2 = vs[s0][2][row + 2][col];
            const long long rr = ((long long)(k - g.kb) * g.nyk + (js - g.jb)) * g.rpitch + (is - 1);
            stress_cell<NM, true, true, false>(a, Loc{p, 0u, 0u}, Loc{rr, 0u, 0u}, k, in_band(k, sb[s][0], sb[s][1], sb[s][2], sb[s][3]), cf, tp, v, mu00[s],
                                        mu00n, mu10[s], mu10n, mu01[s], mu01n, mu11[s]);
            mu00[s] = mu00n; mu10[s] = mu10n; mu01[s] = mu01n;
            mu11[s] = mu[p + P + 1 + Y];
        }
    }
}

// ---------------------------------------------------------------------------
// Side columns (kbeg_a = 1, m_global.f90:334-343): y slabs as full-row tiles,
// x slabs of interior rows as tiles na columns wide with several rows per
// wave (tiles from a host list).  Each lane marches its column through the
// tile's k chunk.
// ---------------------------------------------------------------------------
struct PmlLane {
    int i, j, kb, ke;
    Loc p, q;            // field and auxiliary places on plane kb
    long long astride;
};

__device__ static inline bool pml_lane(const StepArgs &a, const int4 tl, PmlLane &L)
{
    const Grid &g = a.g;
    const int i0 = tl.x & 0xFFFFF, w = (tl.x >> 20) & 0xFF, j0 = tl.y;
    const bool xslab = (tl.x >> 28) & 1;
    const int lane = threadIdx.y * blockDim.x + threadIdx.x;
    const int rows = (blockDim.x * blockDim.y) / w;
    if (lane >= rows * w) return false;
    const int col = lane % w, row = lane / w;
    L.i = i0 + col;
    L.j = j0 + row;
    // a tile lies in one box: x slabs hold the interior rows, y slabs their own
    const int na = g.na;
    const int q = xslab ? (i0 <= na ? 2 : 3) : (j0 <= na ? 0 : 1);
    const int jl = q == 0 ? na : q == 1 ? g.ny : g.ny - na;
    if (L.i > g.nx || L.j > jl) return false;
    const PmlBox b = pick_box(a, q);
    L.kb = tl.z;
    L.ke = min(tl.w, g.nz);
    L.astride = (long long)b.nxb * b.nyb;
    L.p = field_loc(g, i0, j0, L.kb, col, row);
    L.q = {b.off + (long long)(j0 - b.j0) * b.nxb + (i0 - b.i0) + (long long)(L.kb - b.k0) * L.astride,
           4u * (unsigned)(row * b.nxb + col), 0u};
    return L.kb <= L.ke;
}

// absorb_p__update_stress, m_absorb_p.f90:448-519.  Side tiles use ordinary
// loads and stores: a row of an x slab ends inside a 128-byte line whose rest
// belongs to an interior tile, and a non-temporal store gives the line up
// before that arrives.  us with non-temporal and ordinary accesses: 768 x 768
// x 448 688 and 588 (velocity 550 and 492), 384 x 384 x 256 206 and 178 (166
// and 149), twelve small members 3250 and 3040 per step.
template <bool OOP>
__device__ __forceinline__ void stress_pml_body(const StepArgs &a, const int4 tl)
{
    PmlLane L;
    if (!pml_lane(a, tl, L)) return;
    const Grid &g = a.g;
    const int i = L.i, j = L.j;
    const long long P = g.plane;
    const float *__restrict__ Vx = a.f.Vx;
    const float *__restrict__ Vy = a.f.Vy;
    const float *__restrict__ Vz = a.f.Vz;
    const float *__restrict__ mu = a.m.mu;
    const float4 gxc = ldp(a.gxc + (i - 1)), gxe = ldp(a.gxe + (i - 1));
    const float4 gyc = ldp(a.gyc + (j - 1)), gye = ldp(a.gye + (j - 1));

    Loc p = L.p, q = L.q;
    float vx_0 = ld(Vx, p), vy_0 = ld(Vy, p), vz_m1 = ld(Vz, p, -P);
    float mu00 = ld(mu, p), mu10 = ld(mu, p, 0, 1), mu01 = ld(mu, p, 0, 0, 1), mu11 = ld(mu, p, 0, 1, 1);
    for (int k = L.kb; k <= L.ke; ++k, p.u += P, q.u += L.astride) {
        fresh(p);
        fresh(q);
        const float vx_p1 = ld(Vx, p, P), vy_p1 = ld(Vy, p, P), vz_0 = ld(Vz, p);
        const float mu00n = ld(mu, p, P), mu10n = ld(mu, p, P, 1), mu01n = ld(mu, p, P, 0, 1);
        const float mu11n = ld(mu, p, P, 1, 1);
        pml_stress_cell<false, OOP>(a, p, q, k, vx_0, vx_p1, vy_0, vy_p1, vz_m1, vz_0, mu00, mu00n, mu10, mu10n, mu01,
                              mu01n, mu11, gxc, gxe, gyc, gye);
        vx_0 = vx_p1; vy_0 = vy_p1; vz_m1 = vz_0;
        mu00 = mu00n; mu10 = mu10n; mu01 = mu01n; mu11 = mu11n;
    }
}

// absorb_p__update_vel, m_absorb_p.f90:261-306
template <bool OOP>
__device__ __forceinline__ void vel_pml_body(const StepArgs &a, const int4 tl)
{
    PmlLane L;
    if (!pml_lane(a, tl, L)) return;
    const Grid &g = a.g;
    const int i = L.i, j = L.j;
    const long long P = g.plane;
    const float *__restrict__ Szz = a.f.Szz;
    const float *__restrict__ Syz = a.f.Syz;
    const float *__restrict__ Sxz = a.f.Sxz;
    const float *__restrict__ rho = a.m.rho;
    const float4 gxc = ldp(a.gxc + (i - 1)), gxe = ldp(a.gxe + (i - 1));
    const float4 gyc = ldp(a.gyc + (j - 1)), gye = ldp(a.gye + (j - 1));

    Loc p = L.p, q = L.q;
    float szz_0 = ld(Szz, p), syz_m1 = ld(Syz, p, -P), sxz_m1 = ld(Sxz, p, -P), rho0 = ld(rho, p);
    for (int k = L.kb; k <= L.ke; ++k, p.u += P, q.u += L.astride) {
        fresh(p);
        fresh(q);
        const float szz_p1 = ld(Szz, p, P), syz_0 = ld(Syz, p), sxz_0 = ld(Sxz, p), rho_kp = ld(rho, p, P);
        pml_vel_cell<false, OOP>(a, p, q, k, szz_0, szz_p1, syz_m1, syz_0, sxz_m1, sxz_0, rho0, rho_kp, gxc, gxe, gyc, gye);
        szz_0 = szz_p1; syz_m1 = syz_0; sxz_m1 = sxz_0; rho0 = rho_kp;
    }
}

// One launch of a phase: sideb blocks walk the side tiles, the rest the
// interior columns.  The two kinds update disjoint cells from the other
// phase's fields, so their order does not change any result.  Each kind is
// dealt to the XCDs by itself (sideb is a multiple of 8), so every XCD gets an
// eighth of both.  Launched one after the other, each kind's last blocks leave
// CUs idle: 128^3 took 140 us/step in two launches per phase and 127 in one,
// elastic 256 x 256 x 192 525 and 505, 768 x 768 x 448 13.26 and 13.21 ms.
//
// In place, the stress update's first blocks take the outputs that the step
// samples from V (outputs.h), which would otherwise be launches of 4.6 to 13
// us that leave the device idle.
template <int NM, bool NT, bool OOP, bool TP>
__global__ void __launch_bounds__(256) WAVES_NM k_stress(StepArgs a, OutArgs o)
{
    const int blk = (int)blockIdx.x - a.first;
    if constexpr (NT && !OOP) {
        if (blk < 0) {
            outputs_body(o, blockIdx.x, threadIdx.y * blockDim.x + threadIdx.x);
            return;
        }
    }
    if (blk < a.sideb) {
        const int t = xcd_remap(blk, a.sideb);
        if (t < a.ntiles) stress_pml_body<OOP>(a, uni(a.tiles[t]));
        return;
    }
    int bx, byy, bz;
    plain_tile(a, xcd_remap(blk - a.sideb, gridDim.x - a.first - a.sideb), bx, byy, bz);
    stress_int_body<NM, NT, OOP, TP>(a, bx, byy, bz);
}

// The stress update's blocks backwards: it starts on the stresses written
// last and ends on the velocities that the next stress update reads first,
// which the 256 MB cache in front of HBM still holds (us per step forwards and
// backwards: elastic 256 x 256 x 192 439 and 428, 384 x 384 x 256 1870 and
// 1838, 128^3 110.7 and 108.8, twelve small members 3105 and 3060, 768 x 768 x
// 448 within the noise).
template <bool OOP, bool TP>
__global__ void __launch_bounds__(256) WAVES4 k_vel(StepArgs a)
{
    const int n = gridDim.x - a.sideb;
    if ((int)blockIdx.x >= n) {
        const int t = xcd_remap_rev(blockIdx.x - n, a.sideb);
        if (t < a.ntiles) vel_pml_body<OOP>(a, uni(a.tiles[t]));
        return;
    }
    int bx, byy, bz;
    plain_tile(a, xcd_remap_rev(blockIdx.x, n), bx, byy, bz);
    vel_int_body<OOP, TP>(a, bx, byy, bz);
}

// batched side-column tiles: (i0 | width << 20 | xslab << 28, j0, k0 | k1 << 16, member)
__device__ static inline int4 unpack_bside(const int4 t) { return make_int4(t.x, t.y, t.z & 0xFFFF, t.z >> 16); }

__global__ void __launch_bounds__(256) k_stress_pml_b(const StepArgs *__restrict__ mem, const int4 *__restrict__ tiles)
{
    const int4 t = uni(tiles[xcd_remap(blockIdx.x, gridDim.x)]);
    stress_pml_body<false>(mem[t.w], unpack_bside(t));
}

__global__ void __launch_bounds__(256) k_vel_pml_b(const StepArgs *__restrict__ mem, const int4 *__restrict__ tiles)
{
    const int4 t = uni(tiles[xcd_remap_rev(blockIdx.x, gridDim.x)]);
    vel_pml_body<false>(mem[t.w], unpack_bside(t));
}

// one launch per phase for the tiles of both kinds: entries (m, bx, by, bz) are interior
// tiles of member m, entries (-(m+1), i0 | width << 20 | xslab << 28, j0,
// k0 | k1 << 16) its side tiles
template <int NM, bool NT, bool TP>
__global__ void __launch_bounds__(256) WAVES_NM k_stress_all_b(const StepArgs *__restrict__ mem, const int4 *__restrict__ tiles)
{
    const int4 t = uni(tiles[xcd_remap(blockIdx.x, gridDim.x)]);
    if (t.x >= 0) stress_int_body<NM, NT, false, TP>(mem[t.x], t.y, t.z, t.w);
    else stress_pml_body<false>(mem[-t.x - 1], make_int4(t.y, t.z, t.w & 0xFFFF, t.w >> 16));
}

template <bool TP>
__global__ void __launch_bounds__(256) WAVES4 k_vel_all_b(const StepArgs *__restrict__ mem, const int4 *__restrict__ tiles)
{
    const int4 t = uni(tiles[xcd_remap_rev(blockIdx.x, gridDim.x)]);
    if (t.x >= 0) vel_int_body<false, TP>(mem[t.x], t.y, t.z, t.w);
    else vel_pml_body<false>(mem[-t.x - 1], make_int4(t.y, t.z, t.w & 0xFFFF, t.w >> 16));
}

static void step_args(const swpc_ctx *c, StepArgs &a, int mask)
{
    a.g = c->g;
    a.f.Vx = c->fields[SWPC_VX]; a.f.Vy = c->fields[SWPC_VY]; a.f.Vz = c->fields[SWPC_VZ];
    a.f.Sxx = c->fields[SWPC_SXX]; a.f.Syy = c->fields[SWPC_SYY]; a.f.Szz = c->fields[SWPC_SZZ];
    a.f.Syz = c->fields[SWPC_SYZ]; a.f.Sxz = c->fields[SWPC_SXZ]; a.f.Sxy = c->fields[SWPC_SXY];
    {
        float *const *in = c->fields_in[0] ? c->fields_in : c->fields;
        a.fin.Vx = in[SWPC_VX]; a.fin.Vy = in[SWPC_VY]; a.fin.Vz = in[SWPC_VZ];
        a.fin.Sxx = in[SWPC_SXX]; a.fin.Syy = in[SWPC_SYY]; a.fin.Szz = in[SWPC_SZZ];
        a.fin.Syz = in[SWPC_SYZ]; a.fin.Sxz = in[SWPC_SXZ]; a.fin.Sxy = in[SWPC_SXY];
    }
    a.m.rho = c->rho; a.m.lam = c->lam; a.m.mu = c->mu; a.m.taup = c->taup; a.m.taus = c->taus;
    a.m.kfs_top = c->kfs_top; a.m.kfs_bot = c->kfs_bot; a.m.kob_top = c->kob_top; a.m.kob_bot = c->kob_bot;
    a.m.kob = c->kob;
    a.R = c->R;
    a.v = c->visco;
    a.c = c->coef;
    a.dt = c->desc.dt;
    a.ade = c->ade;
    a.ade_in = c->ade_in ? c->ade_in : c->ade;
    a.npml = c->npml;
    for (int q = 0; q < 5; ++q) a.box[q] = c->box[q];
    a.gxc = c->gxc; a.gxe = c->gxe; a.gyc = c->gyc; a.gye = c->gye; a.gzc = c->gzc; a.gze = c->gze;
    a.r20x = 1.0f / (float)c->desc.dx;
    a.r20y = 1.0f / (float)c->desc.dy;
    a.r20z = 1.0f / (float)c->desc.dz;
    a.tiles = (const int4 *)c->d_pml_tiles;
    a.ntiles = c->npml_tiles;
    a.first = 0;
    a.sideb = 0;
    a.cgx_c = c->cgx_c; a.cgx_b = c->cgx_b; a.cgy_c = c->cgy_c; a.cgy_b = c->cgy_b; a.cgz_c = c->cgz_c; a.cgz_b = c->cgz_b;
    a.has_pml = (c->desc.abc == SWPC_ABC_PML && c->npml > 0) ? 1 : 0;
    a.still = c->aux_still ? 1 : 0;
    a.tau = c->tau ? 1 : 0;
    a.mask = mask;
    a.by = c->by;
    a.zc = c->d_zchunks;
    const Grid &g = c->g;
    // variant bit 2: interior tiles 32 cells wide and twice as many rows, so
    // narrow grids idle fewer lanes at the tile edges
    a.bxw = (c->variant & 4) ? 32 : BX;
    a.byi = a.by * (BX / a.bxw);
    a.bx0 = (g.ib - 1) / a.bxw;
    a.nbx = (g.ie - 1) / a.bxw - a.bx0 + 1;
    a.nby = (g.nyk + a.byi - 1) / a.byi;
    a.nbz = c->nbz;
}

// One launch of a phase over the side tiles (side), over the interior columns'
// interior planes (mask & MASK_INT) and their bottom PML band (mask &
// MASK_PML), or over all of them.  The batch's and the fused launch's tiles
// use the same bodies.
static bool phase_grid(const swpc_ctx *c, StepArgs &a, int phase, bool side, int mask, dim3 &grid, dim3 &block)
{
    step_args(c, a, mask);
    if (phase == 1) a.zc = c->d_zchunks + c->nbz + 1;
    if (mask == MASK_PML) {   // the bottom band without the interior
        a.zc = c->d_zchunks + 2 * (c->nbz + 1);
        a.nbz = c->nbb;
    }
    const bool cols = c->g.nxk > 0 && c->g.nyk > 0 && ((mask & MASK_INT) || ((mask & MASK_PML) && a.has_pml));
    a.sideb = side && a.has_pml ? (c->npml_tiles + 7) & ~7 : 0;
    block = dim3(a.bxw, a.byi);
    grid = dim3(a.sideb + (cols ? a.nbx * a.nby * a.nbz : 0));
    return grid.x > 0;
}

void green_store_fill(swpc_ctx *c, GreenArgs &a, int it, const int *d_it);
void wavargs_fill(swpc_ctx *c, WavArgs &a, int it, const int *d_it);
void snap_fill(swpc_ctx *c, SnapArgs &a, int it, const int *d_it);

// The step's outputs before its stress update: returns those that read V only
// in o, for the update's launch, and launches the others (receivers that
// record stresses, sections of div and rot, which mask with S) or, where the
// launch does not take any (variant without bit 0, blocks of another size),
// all of them.
hipError_t launch_outputs(swpc_ctx *c, int it, const int *d_it, OutArgs &o)
{
    o.ng = o.nw = o.ns = o.nblk = 0;
    const bool in = (c->variant & 1) && !c->fields_in[0] && c->by * BX == 256;
    hipError_t e = hipSuccess;
    if (in && c->green_on && c->green_ng > 0) {
        green_store_fill(c, o.green, it, d_it);
        o.ng = (c->green_ng + 255) / 256;
    } else if ((e = launch_green_store(c, it, d_it)) != hipSuccess) {
        return e;
    }
    if (in && c->nst > 0 && !(c->wav_what & SWPC_WAV_STRESS)) {
        wavargs_fill(c, o.wav, it, d_it);
        o.nw = (c->nst + 255) / 256;
    } else if ((e = launch_wav_store(c, it, d_it)) != hipSuccess) {
        return e;
    }
    bool v_only = true;
    for (int t = 0; t < c->snap_ntask; ++t) v_only = v_only && c->snap_task[t].q != SWPC_SNP_PS;
    if (in && c->snap_ntask > 0 && v_only) {
        snap_fill(c, o.snap, it, d_it);
        o.ns = c->snap_nblk;
    } else if ((e = launch_snap(c, it, d_it)) != hipSuccess) {
        return e;
    }
    o.nblk = (o.ng + o.nw + o.ns + 7) & ~7;
    return hipSuccess;
}

hipError_t launch_stress(swpc_ctx *c, bool side, int mask, const OutArgs *out)
{
    StepArgs a;
    OutArgs o;
    dim3 grid, block;
    const bool tiles = phase_grid(c, a, 0, side, mask, grid, block);
    if (out && out->nblk > 0) {
        o = *out;
        a.first = o.nblk;
        grid.x += a.first;
    } else if (!tiles) {
        return hipSuccess;
    }
    const bool nt = (c->variant & 1) != 0;
    const bool oop = c->fields_in[0] != nullptr;   // out of place: non-temporal streams as well
    const bool tp = (mask & MASK_TAPER) != 0;
    c->aux_moved = true;
#define SWPC_STRESS_CASE(NMV)                                                                              \
    case NMV:                                                                                              \
        if (oop) hipLaunchKernelGGL((k_stress<NMV, true, true, false>), grid, block, 0, c->stream, a, o);       \
        else if (tp) hipLaunchKernelGGL((k_stress<NMV, true, false, true>), grid, block, 0, c->stream, a, o);   \
        else if (nt) hipLaunchKernelGGL((k_stress<NMV, true, false, false>), grid, block, 0, c->stream, a, o);  \
        else hipLaunchKernelGGL((k_stress<NMV, false, false, false>), grid, block, 0, c->stream, a, o);         \
        break;
    switch (c->g.nm) {
        SWPC_STRESS_CASE(0) SWPC_STRESS_CASE(1) SWPC_STRESS_CASE(2) SWPC_STRESS_CASE(3) SWPC_STRESS_CASE(4)
        SWPC_STRESS_CASE(5) SWPC_STRESS_CASE(6) SWPC_STRESS_CASE(7) SWPC_STRESS_CASE(8)
    default: return hipErrorInvalidValue;
    }
#undef SWPC_STRESS_CASE
    return hipGetLastError();
}

hipError_t launch_vel(swpc_ctx *c, bool side, int mask)
{
    StepArgs a;
    dim3 grid, block;
    if (!phase_grid(c, a, 1, side, mask, grid, block)) return hipSuccess;
    c->aux_moved = true;
    if (c->fields_in[0]) hipLaunchKernelGGL((k_vel<true, false>), grid, block, 0, c->stream, a);
    else if (mask & MASK_TAPER) hipLaunchKernelGGL((k_vel<false, true>), grid, block, 0, c->stream, a);
    else hipLaunchKernelGGL((k_vel<false, false>), grid, block, 0, c->stream, a);
    return hipGetLastError();
}

// the fused interior launch: c->fields holds the new fields, c->fields_in
// the old ones; tiles of FW x 4 sr columns (sr = 2 with variant bit 8)
hipError_t launch_fused(swpc_ctx *c)
{
    StepArgs a;
    step_args(c, a, MASK_INT);
    const Grid &g = c->g;
    if (g.nxk <= 0 || g.nyk <= 0 || c->nfz <= 0 || !c->fields_in[0]) return hipErrorInvalidValue;
    const int sr = (c->variant & 256) ? 2 : 1;
    a.zc = c->d_fzc;
    a.nbx = (g.nxk + FW - 1) / FW;
    a.nby = (g.nyk + 4 * sr - 1) / (4 * sr);
    a.nbz = c->nfz;
    const dim3 grid(a.nbx * a.nby * a.nbz), block(BX, 4);
    c->aux_moved = true;
#define SWPC_FUSED_CASE(NMV)                                                                          \
    case NMV:                                                                                         \
        if (sr == 2) hipLaunchKernelGGL((k_fused<NMV, 2>), grid, block, 0, c->stream, a);              \
        else hipLaunchKernelGGL((k_fused<NMV, 1>), grid, block, 0, c->stream, a);                      \
        break;
    switch (g.nm) {
        SWPC_FUSED_CASE(0) SWPC_FUSED_CASE(1) SWPC_FUSED_CASE(2) SWPC_FUSED_CASE(3) SWPC_FUSED_CASE(4)
        SWPC_FUSED_CASE(5) SWPC_FUSED_CASE(6) SWPC_FUSED_CASE(7) SWPC_FUSED_CASE(8)
    default: return hipErrorInvalidValue;
    }
#undef SWPC_FUSED_CASE
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Cerjan sponge (m_absorb_c.f90:113-198).  Profiles carry the 3-cell halo:
// entry of cell n is at n + 2.
// ---------------------------------------------------------------------------
struct CerjanArgs {
    Grid g;
    FieldPtrs f;
    const float *gx_c, *gx_b, *gy_c, *gy_b, *gz_c, *gz_b;
    int kend;
};

__device__ static inline void cerjan_stress_cell(const CerjanArgs &a, int i, int j, int k)
{
    if (i > a.g.nx || k > a.kend) return;
    const long long p = gidx(a.g, i, j, k);
    const float gxc = a.gx_c[i + 2], gxb = a.gx_b[i + 2];
    const float gyc = a.gy_c[j + 2], gyb = a.gy_b[j + 2];
    const float gzc = a.gz_c[k + 2], gzb = a.gz_b[k + 2];
    const float gcc = gxc * gyc * gzc;
    a.f.Sxx[p] = a.f.Sxx[p] * gcc;
    a.f.Syy[p] = a.f.Syy[p] * gcc;
    a.f.Szz[p] = a.f.Szz[p] * gcc;
    a.f.Syz[p] = a.f.Syz[p] * gxc * gyb * gzb;
    a.f.Sxz[p] = a.f.Sxz[p] * gxb * gyc * gzb;
    a.f.Sxy[p] = a.f.Sxy[p] * gxb * gyb * gzc;
}

__global__ void __launch_bounds__(256) k_cerjan_stress(CerjanArgs a)
{
    cerjan_stress_cell(a, 1 + blockIdx.x * blockDim.x + threadIdx.x, 1 + blockIdx.y, 1 + blockIdx.z);
}

__device__ static inline void cerjan_vel_cell(const CerjanArgs &a, int i, int j, int k)
{
    if (i > a.g.nx || k > a.kend) return;
    const long long p = gidx(a.g, i, j, k);
    const float gxc = a.gx_c[i + 2], gxb = a.gx_b[i + 2];
    const float gyc = a.gy_c[j + 2], gyb = a.gy_b[j + 2];
    const float gzc = a.gz_c[k + 2], gzb = a.gz_b[k + 2];
    a.f.Vx[p] = a.f.Vx[p] * gxb * gyc * gzc;
    a.f.Vy[p] = a.f.Vy[p] * gxc * gyb * gzc;
    a.f.Vz[p] = a.f.Vz[p] * gxc * gyc * gzb;
}

__global__ void __launch_bounds__(256) k_cerjan_vel(CerjanArgs a)
{
    cerjan_vel_cell(a, 1 + blockIdx.x * blockDim.x + threadIdx.x, 1 + blockIdx.y, 1 + blockIdx.z);
}

static void cerjan_fill(swpc_ctx *c, CerjanArgs &a, int kend)
{
    a.g = c->g;
    a.f.Vx = c->fields[SWPC_VX]; a.f.Vy = c->fields[SWPC_VY]; a.f.Vz = c->fields[SWPC_VZ];
    a.f.Sxx = c->fields[SWPC_SXX]; a.f.Syy = c->fields[SWPC_SYY]; a.f.Szz = c->fields[SWPC_SZZ];
    a.f.Syz = c->fields[SWPC_SYZ]; a.f.Sxz = c->fields[SWPC_SXZ]; a.f.Sxy = c->fields[SWPC_SXY];
    a.gx_c = c->cgx_c; a.gx_b = c->cgx_b; a.gy_c = c->cgy_c; a.gy_b = c->cgy_b; a.gz_c = c->cgz_c; a.gz_b = c->cgz_b;
    a.kend = kend;
}

hipError_t launch_cerjan_stress(swpc_ctx *c)
{
    CerjanArgs a;
    cerjan_fill(c, a, c->g.ke);
    dim3 grid((c->g.nx + 255) / 256, c->g.ny, c->g.ke);
    hipLaunchKernelGGL(k_cerjan_stress, grid, dim3(256), 0, c->stream, a);
    return hipGetLastError();
}

hipError_t launch_cerjan_vel(swpc_ctx *c)
{
    CerjanArgs a;
    cerjan_fill(c, a, c->g.nz);
    dim3 grid((c->g.nx + 255) / 256, c->g.ny, c->g.nz);
    hipLaunchKernelGGL(k_cerjan_vel, grid, dim3(256), 0, c->stream, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// batched launches: the arguments of every member live in HBM, the tile
// tables carry the member index (swpc_batch, batch.hip)
// ---------------------------------------------------------------------------
size_t step_args_size() { return sizeof(StepArgs); }

// arguments of one member for the launches of a whole step's phase, whose
// chunks start at the planes in zc
void fill_batch_args(const swpc_ctx *c, void *out, const int *zc)
{
    StepArgs a;
    step_args(c, a, MASK_INT | (c->desc.abc == SWPC_ABC_PML ? MASK_PML : MASK_TAPER));
    a.zc = zc;
    *(StepArgs *)out = a;
}

// interior-column tiles of one member's chunk: (bx, by)
void member_tiles(const swpc_ctx *c, int &nbx, int &nby)
{
    StepArgs a;
    step_args(c, a, MASK_INT | MASK_PML);
    nbx = a.nbx;
    nby = a.nby;
}

// one launch per phase for both kinds of tiles (the batch's packing 2)
hipError_t launch_batch_phase_all(int phase, int nm, int variant, bool tp, int by, int bxw, const void *d_args,
                                  const int4 *d_all, int nall, hipStream_t s)
{
    if (nall <= 0) return hipSuccess;
    const StepArgs *mem = (const StepArgs *)d_args;
    const dim3 block(bxw, by * (BX / bxw));
    const bool nt = (variant & 1) != 0;
    if (phase == 1) {
        if (tp) hipLaunchKernelGGL(k_vel_all_b<true>, dim3(nall), block, 0, s, mem, d_all);
        else hipLaunchKernelGGL(k_vel_all_b<false>, dim3(nall), block, 0, s, mem, d_all);
        return hipGetLastError();
    }
#define SWPC_BALL_CASE(NMV)                                                                                   \
    case NMV:                                                                                                 \
        if (tp) hipLaunchKernelGGL((k_stress_all_b<NMV, true, true>), dim3(nall), block, 0, s, mem, d_all);         \
        else if (nt) hipLaunchKernelGGL((k_stress_all_b<NMV, true, false>), dim3(nall), block, 0, s, mem, d_all);   \
        else hipLaunchKernelGGL((k_stress_all_b<NMV, false, false>), dim3(nall), block, 0, s, mem, d_all);          \
        break;
    switch (nm) {
        SWPC_BALL_CASE(0) SWPC_BALL_CASE(1) SWPC_BALL_CASE(2) SWPC_BALL_CASE(3) SWPC_BALL_CASE(4)
        SWPC_BALL_CASE(5) SWPC_BALL_CASE(6) SWPC_BALL_CASE(7) SWPC_BALL_CASE(8)
    default: return hipErrorInvalidValue;
    }
#undef SWPC_BALL_CASE
    return hipGetLastError();
}

hipError_t launch_batch_phase(int phase, int nm, int variant, bool tp, int by, int bxw, const void *d_args,
                              const int4 *d_cols, int ncols, const int4 *d_side, int nside, hipStream_t s)
{
    const bool nt = (variant & 1) != 0;
    const StepArgs *mem = (const StepArgs *)d_args;
    const dim3 side(BX, by), block(bxw, by * (BX / bxw));
    if (nside > 0) {
        if (phase == 0) hipLaunchKernelGGL(k_stress_pml_b, dim3(nside), side, 0, s, mem, d_side);
        else hipLaunchKernelGGL(k_vel_pml_b, dim3(nside), side, 0, s, mem, d_side);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (ncols <= 0) return hipSuccess;
    if (phase == 1) {
        if (tp) hipLaunchKernelGGL(k_vel_int_b<true>, dim3(ncols), block, 0, s, mem, d_cols);
        else hipLaunchKernelGGL(k_vel_int_b<false>, dim3(ncols), block, 0, s, mem, d_cols);
        return hipGetLastError();
    }
#define SWPC_BSTRESS_CASE(NMV)                                                                                \
    case NMV:                                                                                                 \
        if (tp) hipLaunchKernelGGL((k_stress_int_b<NMV, true, true>), dim3(ncols), block, 0, s, mem, d_cols);       \
        else if (nt) hipLaunchKernelGGL((k_stress_int_b<NMV, true, false>), dim3(ncols), block, 0, s, mem, d_cols); \
        else hipLaunchKernelGGL((k_stress_int_b<NMV, false, false>), dim3(ncols), block, 0, s, mem, d_cols);        \
        break;
    switch (nm) {
        SWPC_BSTRESS_CASE(0) SWPC_BSTRESS_CASE(1) SWPC_BSTRESS_CASE(2) SWPC_BSTRESS_CASE(3) SWPC_BSTRESS_CASE(4)
        SWPC_BSTRESS_CASE(5) SWPC_BSTRESS_CASE(6) SWPC_BSTRESS_CASE(7) SWPC_BSTRESS_CASE(8)
    default: return hipErrorInvalidValue;
    }
#undef SWPC_BSTRESS_CASE
    return hipGetLastError();
}
