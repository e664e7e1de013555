// device_access.h -- how the per-cell kernels address global memory.
#pragma once

#include "swpc_internal.h"

typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f2v __attribute__((ext_vector_type(2)));

// Loads and stores through explicit global pointers: a batch launch reads its
// arrays' addresses from memory, where the compiler only knows generic ones
// and would make every access a flat one, which waits for all others.  NT:
// streams read or written once per step (memory variables, stress, the
// per-cell medium) bypass cache retention so the L2 keeps the V and mu rows
// that neighbouring tiles re-read.
template <typename T>
using GlobalPtr = __attribute__((address_space(1))) T *;

template <bool NT, typename T>
__device__ static inline T ldv(const T *p)
{
    const GlobalPtr<const T> q = (GlobalPtr<const T>)p;
    if constexpr (NT) return __builtin_nontemporal_load(q);
    else return *q;
}
template <bool NT, typename T>
__device__ static inline void stv(T *p, T v)
{
    const GlobalPtr<T> q = (GlobalPtr<T>)p;
    if constexpr (NT) __builtin_nontemporal_store(v, q);
    else *q = v;
}
// one cell's PML profile
__device__ static inline float4 ldp(const float4 *p)
{
    const f4v v = ldv<false>((const f4v *)p);
    return make_float4(v.x, v.y, v.z, v.w);
}

// Where a lane reads: u is the element offset all lanes of the block share
// (plane and tile origin, kept in scalar registers), o the lane's byte offset
// from there and y the bytes of a row.  F + u is a scalar pointer and o a
// 32-bit register, so an access is one instruction with the x neighbour as
// its immediate offset; y neighbours add rows to o and z neighbours planes to
// u.  No array costs 64-bit vector arithmetic or a register pair of its own:
// the NM = 3 stress update fell from 201 registers to 106 and four waves per
// SIMD instead of two (1024 x 1024 x 512 class grids: 9.22 -> 8.83 ms per
// 264 M cells; 128^3: 58 -> 50 us).
struct Loc {
    long long u;
    unsigned o, y;
};
// F d elements (the same for every lane), dx cells and dy rows from the lane's
// place; u starts two rows before the tile so that o stays positive
template <bool NT = false>
__device__ __forceinline__ float ld(const float *F, const Loc &l, long long d = 0, int dx = 0, int dy = 0)
{
    return ldv<NT>((const float *)((const char *)(F + (l.u + d)) + (l.o + (unsigned)dy * l.y)) + dx);
}
template <bool NT>
__device__ __forceinline__ void st(float *F, const Loc &l, float v, long long d = 0)
{
    stv<NT>((float *)((char *)(F + (l.u + d)) + l.o), v);
}
// The compiler selects the scalar-pointer form only where it sees the 32-bit
// offset being widened; hoisted out of the loop, the widened offset costs a
// 64-bit vector add per access.  An offset that looks new in every iteration
// is widened at its uses.
__device__ __forceinline__ void fresh(Loc &l) { asm("" : "+v"(l.o)); }

// the place of cell (i0 + col, j0 + row) on plane k, (i0, j0, k) the same for
// every lane of the block
__device__ __forceinline__ Loc field_loc(const Grid &g, int i0, int j0, int k, int col, int row)
{
    return Loc{gidx(g, i0, j0 - 2, k), 4u * (unsigned)((row + 2) * g.pitch + col), 4u * (unsigned)g.pitch};
}

// a value that every lane of the block holds, in a scalar register
__device__ static inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ static inline int4 uni(int4 v) { return make_int4(uni(v.x), uni(v.y), uni(v.z), uni(v.w)); }
