// snap.hip -- wavefield sections of libswpc_gpu (snap__write,
// src/swpc_3d/m_snap.f90:919-2189, native-format semantics).
//
// Every enabled section is a task of ns1 x ns2 points; one launch per step
// covers all tasks (one thread per point).  A frame is taken when
// mod(it-1, ntdec_s) == 0 and stored in the section's frame store on the
// device (frame f = (it-1)/ntdec_s), so graph-replayed step blocks need no
// host round trip.  u sections integrate V dt every step and the fs/ob
// sections keep running maximum maps, as the reference does.
#include <cstring>

#include "outputs.h"

__global__ void __launch_bounds__(256) k_snap(SnapArgs a) { snap_body(a, blockIdx.x, threadIdx.x, step_number(a.it, a.d_it)); }

// batched: context m = blockIdx.y, its arguments in HBM; blocks beyond the
// context's own count idle
__global__ void __launch_bounds__(256) k_snap_b(const SnapArgs *__restrict__ args, int it, const int *d_it)
{
    const SnapArgs &a = args[blockIdx.y];
    if ((int)blockIdx.x >= a.nblk) return;
    snap_body(a, blockIdx.x, threadIdx.x, step_number(it, d_it));
}

void snap_fill(swpc_ctx *c, SnapArgs &a, int it, const int *d_it)
{
    a.g = c->g;
    a.Vx = c->fields[SWPC_VX]; a.Vy = c->fields[SWPC_VY]; a.Vz = c->fields[SWPC_VZ];
    a.Syz = c->fields[SWPC_SYZ]; a.Sxz = c->fields[SWPC_SXZ]; a.Sxy = c->fields[SWPC_SXY];
    a.lam = c->lam;
    a.kfs = c->d_kfs; a.kob = c->kob;
    for (int t = 0; t < c->snap_ntask; ++t) a.task[t] = c->snap_task[t];
    a.ntask = c->snap_ntask;
    a.nblk = c->snap_nblk;
    const swpc_snap_desc &d = c->snap;
    a.k0_xy = d.k0_xy; a.i0_yz = d.i0_yz; a.j0_xz = d.j0_xz;
    a.idec = d.idec; a.jdec = d.jdec; a.kdec = d.kdec; a.ntdec_s = d.ntdec_s; a.nframe = d.nframe;
    a.r20x = 1.0f / (float)c->desc.dx;
    a.r20y = 1.0f / (float)c->desc.dy;
    a.r20z = 1.0f / (float)c->desc.dz;
    a.M0 = d.M0; a.UC = d.UC; a.dt = c->desc.dt;
    a.it = it;
    a.d_it = d_it;
}

hipError_t launch_snap(swpc_ctx *c, int it, const int *d_it, hipStream_t s)
{
    if (c->snap_ntask <= 0) return hipSuccess;
    SnapArgs a;
    snap_fill(c, a, it, d_it);
    hipLaunchKernelGGL(k_snap, dim3(c->snap_nblk), dim3(256), 0, (s ? s : c->stream), a);
    return hipGetLastError();
}

// batched sections (swpc_batch): one launch for every member with sections,
// as many blocks as the member with the most section points
size_t batch_snap_size() { return sizeof(SnapArgs); }

int batch_snap_fill(swpc_ctx *c, void *out)
{
    if (c->snap_ntask <= 0) return 0;
    SnapArgs a;
    snap_fill(c, a, 0, nullptr);
    memcpy(out, &a, sizeof(a));
    return c->snap_nblk;
}

hipError_t launch_batch_snap(const void *d_args, int nmem, int maxblk, int it, const int *d_it, hipStream_t s)
{
    if (nmem <= 0 || maxblk <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_snap_b, dim3(maxblk, nmem), dim3(256), 0, s, (const SnapArgs *)d_args, it, d_it);
    return hipGetLastError();
}
