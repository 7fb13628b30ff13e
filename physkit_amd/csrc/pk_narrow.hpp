// What the narrowphase kernels share: a body's or a batch entry's shape as gshape, and the
// hand-off of GJK simplices and EPA contacts between kernels.
#pragma once
#include "pk_access.hpp"
#include "pk_gjk.hpp"

namespace pk
{

// UV: the shapes may include tagged UV spheres (a kernel built without it carries no
// code for their fast support)
template <bool UV> __device__ __forceinline__ gshape body_shape(const bodies_dev &b, const shapes_dev &s, uint32_t id)
{
    gshape g;
    g.kind = 2;
    g.a = ld3(b.pos, b.n, id);
    g.b = mk(0.0, 0.0, 0.0);
    g.q = ldq(b.quat, b.n, id);
    uint32_t sh = b.shape[id];
    g.v = s.verts + 3 * static_cast<size_t>(s.voff[sh]);
    g.nv = s.off[sh + 1] - s.off[sh];
    g.uv = UV ? s.uv[sh] : 0u;
    g.paired = 1;
    return g;
}

// GJK simplex hand-off, planar: slot 0 = point count, then per point p.xyz and the
// two support features packed in one 64-bit word (kSimplexWords doubles per hit).
__device__ __forceinline__ void st_spt(double *d, uint32_t cap, uint32_t slot, int k, const spt &p)
{
    double *b = d + static_cast<size_t>(1 + 4 * k) * cap + slot;
    b[0] = p.p.x;
    b[cap] = p.p.y;
    b[2 * static_cast<size_t>(cap)] = p.p.z;
    b[3 * static_cast<size_t>(cap)] =
        __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(p.ib) << 32) | p.ia));
}
__device__ __forceinline__ spt ld_spt(const double *d, uint32_t cap, uint32_t slot, int k)
{
    const double *b = d + static_cast<size_t>(1 + 4 * k) * cap + slot;
    spt p;
    p.p = mk(b[0], b[cap], b[2 * static_cast<size_t>(cap)]);
    uint64_t f = static_cast<uint64_t>(__double_as_longlong(b[3 * static_cast<size_t>(cap)]));
    p.ia = static_cast<uint32_t>(f);
    p.ib = static_cast<uint32_t>(f >> 32);
    return p;
}
__device__ __forceinline__ void save_simplex(double *d, uint32_t cap, uint32_t slot, const simplex &x)
{
    d[slot] = static_cast<double>(x.n);
    st_spt(d, cap, slot, 0, x.s0);
    if (x.n > 1) st_spt(d, cap, slot, 1, x.s1);
    if (x.n > 2) st_spt(d, cap, slot, 2, x.s2);
    if (x.n > 3) st_spt(d, cap, slot, 3, x.s3);
}
__device__ __forceinline__ void load_simplex(const double *d, uint32_t cap, uint32_t slot, simplex &x)
{
    x.n = static_cast<int>(d[slot]);
    x.s0 = ld_spt(d, cap, slot, 0);
    if (x.n > 1) x.s1 = ld_spt(d, cap, slot, 1);
    if (x.n > 2) x.s2 = ld_spt(d, cap, slot, 2);
    if (x.n > 3) x.s3 = ld_spt(d, cap, slot, 3);
}

__device__ __forceinline__ void write_info(double *info, uint32_t cap, uint32_t p, const double *o)
{
    for (int k = 0; k < 10; ++k) info[static_cast<size_t>(k) * cap + p] = o[k];
}

// shape i of one side of the standalone batch
__device__ __forceinline__ gshape pair_shape(const int32_t *kind, const double *prm, const uint32_t *vb, const uint32_t *ve,
                             const double *verts, const uint32_t *uv, uint32_t i)
{
    const double *q = prm + 10 * static_cast<size_t>(i);
    gshape g;
    g.kind = kind[i];
    g.v = nullptr;
    g.nv = 0;
    g.uv = 0;
    g.paired = 0;
    g.b = mk(0.0, 0.0, 0.0);
    g.q = mkq(1.0, 0.0, 0.0, 0.0);
    if (g.kind == 0)
    {
        g.a = mk(q[0], q[1], q[2]);
        g.b = mk(q[3], q[4], q[5]);
    }
    else if (g.kind == 1)
    {
        g.a = mk(q[0], q[1], q[2]);
        g.q = mkq(q[3], q[4], q[5], q[6]);
        g.b = mk(q[7], q[8], q[9]);
    }
    else
    {
        g.a = mk(q[0], q[1], q[2]);
        g.q = mkq(q[3], q[4], q[5], q[6]);
        g.v = verts + 3 * static_cast<size_t>(vb[i]);
        g.nv = ve[i] - vb[i];
        g.uv = uv ? uv[i] : 0u; // no tags: every support scans all vertices (same results)
    }
    return g;
}

} // namespace pk
