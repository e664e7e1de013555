// green.hip -- reciprocity Green's-function mode of libswpc_gpu
// (src/swpc_3d/m_green.f90): the strain Green's functions sampled at the GF
// cells (green__store) and the unit force at the virtual source, a station
// (green__source).
//
// green__store is a gather of 4th-order staggered derivatives at a few
// scattered cells: one thread per GF cell, accumulators component-major so
// that each of the twelve read-modify-writes is coalesced.  Every expression
// keeps the reference's FP32 evaluation order (the FP32 build, MP = SP).
#include <cstring>

#include "outputs.h"

__global__ void __launch_bounds__(64) k_green_store(GreenArgs a)
{
    green_store_body(a, blockIdx.x * blockDim.x + threadIdx.x, step_number(a.it, a.d_it));
}

// batched: context m = blockIdx.y, its arguments in HBM
__global__ void __launch_bounds__(64) k_green_store_b(const GreenArgs *__restrict__ args, int it, const int *d_it)
{
    green_store_body(args[blockIdx.y], blockIdx.x * blockDim.x + threadIdx.x, step_number(it, d_it));
}

void green_store_fill(swpc_ctx *c, GreenArgs &a, int it, const int *d_it)
{
    a.Vx = c->fields[SWPC_VX]; a.Vy = c->fields[SWPC_VY]; a.Vz = c->fields[SWPC_VZ];
    a.ig = c->d_green_ijk;
    a.jg = c->d_green_ijk + c->green_ng;
    a.kg = c->d_green_ijk + 2 * (long long)c->green_ng;
    a.acc = c->d_green_acc;
    a.gf = c->d_gf;
    a.g = c->g;
    a.ng = c->green_ng; a.ncmp = c->green_ncmp; a.ntdec = c->green_ntdec; a.ntw = c->green_ntw;
    a.dt = c->desc.dt;
    // r40 = C40/d, r41 = C41/d with C40 = 9/8, C41 = 1/24 (m_green.f90:43-45,110-115)
    const float dx = (float)c->desc.dx, dy = (float)c->desc.dy, dz = (float)c->desc.dz;
    const float C40 = 9.0f / 8.0f, C41 = 1.0f / 24.0f;
    a.r40x = C40 / dx; a.r40y = C40 / dy; a.r40z = C40 / dz;
    a.r41x = C41 / dx; a.r41y = C41 / dy; a.r41z = C41 / dz;
    a.it = it;
    a.d_it = d_it;
}

hipError_t launch_green_store(swpc_ctx *c, int it, const int *d_it, hipStream_t s)
{
    if (!c->green_on || c->green_ng <= 0) return hipSuccess;
    GreenArgs a;
    green_store_fill(c, a, it, d_it);
    hipLaunchKernelGGL(k_green_store, dim3((c->green_ng + 63) / 64), dim3(64), 0, (s ? s : c->stream), a);
    return hipGetLastError();
}

struct GreenSrcArgs {
    float *Vx, *Vy, *Vz;
    const float *rho;
    const float *stf;
    Grid g;
    int i, j, k, nt;
    float fx1, fy1, fz1, dt_dxyz;
    int it;
    const int *d_it;
};

// green__source, m_green.f90:614-649: the force split onto the two staggered
// velocity nodes of each axis with the averaged buoyancy; all six updates
// are made, the zero ones included
__device__ static inline void green_source_body(const GreenSrcArgs &a, int it)
{
    if (it < 1 || it > a.nt) return;
    const Grid &g = a.g;
    const long long p = gidx(g, a.i, a.j, a.k);
    const long long Y = g.pitch, Z = g.plane;
    const float st = a.stf[it - 1];
    const float fx = a.fx1 * a.dt_dxyz * st;
    const float fy = a.fy1 * a.dt_dxyz * st;
    const float fz = a.fz1 * a.dt_dxyz * st;
    const float *rho = a.rho;
    const float r0 = rho[p];
    a.Vx[p] = a.Vx[p] + (2.0f / (r0 + rho[p + 1])) * fx / 2.0f;
    a.Vx[p - 1] = a.Vx[p - 1] + (2.0f / (r0 + rho[p - 1])) * fx / 2.0f;
    a.Vy[p] = a.Vy[p] + (2.0f / (r0 + rho[p + Y])) * fy / 2.0f;
    a.Vy[p - Y] = a.Vy[p - Y] + (2.0f / (r0 + rho[p - Y])) * fy / 2.0f;
    a.Vz[p] = a.Vz[p] + (2.0f / (r0 + rho[p + Z])) * fz / 2.0f;
    a.Vz[p - Z] = a.Vz[p - Z] + (2.0f / (r0 + rho[p - Z])) * fz / 2.0f;
}

__global__ void k_green_source(GreenSrcArgs a)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    green_source_body(a, step_number(a.it, a.d_it));
}

// batched: context m = blockIdx.y
__global__ void k_green_source_b(const GreenSrcArgs *__restrict__ args, int it, const int *d_it)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    green_source_body(args[blockIdx.y], step_number(it, d_it));
}

static void green_source_fill(swpc_ctx *c, GreenSrcArgs &a, int it, const int *d_it)
{
    a.Vx = c->fields[SWPC_VX]; a.Vy = c->fields[SWPC_VY]; a.Vz = c->fields[SWPC_VZ];
    a.rho = c->rho;
    a.stf = c->d_green_stf;
    a.g = c->g;
    a.i = c->green_src[0]; a.j = c->green_src[1]; a.k = c->green_src[2];
    a.nt = c->green_nt;
    a.fx1 = c->green_f[0]; a.fy1 = c->green_f[1]; a.fz1 = c->green_f[2];
    a.dt_dxyz = c->green_dt_dxyz;
    a.it = it;
    a.d_it = d_it;
}

hipError_t launch_green_source(swpc_ctx *c, int it, const int *d_it, hipStream_t s)
{
    if (!c->green_on || c->green_nt <= 0) return hipSuccess;
    GreenSrcArgs a;
    green_source_fill(c, a, it, d_it);
    hipLaunchKernelGGL(k_green_source, dim3(1), dim3(64), 0, (s ? s : c->stream), a);
    return hipGetLastError();
}

// batched Green's-function store and source (swpc_batch): per-member
// arguments, one launch for every member that has them
size_t batch_green_size(int kind) { return kind == BATCH_AUX_GREEN_STORE ? sizeof(GreenArgs) : sizeof(GreenSrcArgs); }

int batch_green_fill(swpc_ctx *c, int kind, void *out)
{
    if (!c->green_on) return 0;
    if (kind == BATCH_AUX_GREEN_STORE) {
        if (c->green_ng <= 0) return 0;
        GreenArgs a;
        green_store_fill(c, a, 0, nullptr);
        memcpy(out, &a, sizeof(a));
        return c->green_ng;
    }
    if (c->green_nt <= 0) return 0;
    GreenSrcArgs a;
    green_source_fill(c, a, 0, nullptr);
    memcpy(out, &a, sizeof(a));
    return 1;
}

hipError_t launch_batch_green(int kind, const void *d_args, int nmem, int nmax, int it, const int *d_it,
                              hipStream_t s)
{
    if (nmem <= 0 || nmax <= 0) return hipSuccess;
    if (kind == BATCH_AUX_GREEN_STORE)
        hipLaunchKernelGGL(k_green_store_b, dim3((nmax + 63) / 64, nmem), dim3(64), 0, s, (const GreenArgs *)d_args,
                           it, d_it);
    else
        hipLaunchKernelGGL(k_green_source_b, dim3(1, nmem), dim3(64), 0, s, (const GreenSrcArgs *)d_args, it, d_it);
    return hipGetLastError();
}
