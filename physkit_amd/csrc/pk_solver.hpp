// What the contact solver's kernels share (k_solver.hip, k_island.hip): contact rows, body
// state, contact frames, colouring claims, the FP32 solve's vectors and union-find.
#pragma once
#include "pk_access.hpp"

#include <cfloat>

namespace pk
{

struct rowv
{
    v3 Jv, Jwa, Jwb;
    double Meff, bias, acc;
};
struct body_state
{
    v3 vel, ang;
    double im;
    m3 Iwi;
    bool stat;
};

__device__ __forceinline__ double row_jv(const rowv &r, const body_state &A, const body_state &B)
{ return ((dot(r.Jv, A.vel) + dot(r.Jwa, A.ang)) - dot(r.Jv, B.vel)) + dot(r.Jwb, B.ang); }

__device__ __forceinline__ void row_apply(rowv &r, double lo, double hi, body_state &A, body_state &B) // :49-72
{
    double jv = row_jv(r, A, B);
    double cfp = 0.0 * r.acc;
    double lambda = -((jv + r.bias) + cfp) * r.Meff;
    double old = r.acc;
    double v = old + lambda;
    r.acc = (v < lo) ? lo : ((hi < v) ? hi : v);
    double ap = r.acc - old;
    if (!A.stat)
    {
        A.vel = A.vel + (r.Jv * ap) * A.im;
        A.ang = A.ang + mul(A.Iwi, r.Jwa * ap);
    }
    if (!B.stat)
    {
        B.vel = B.vel + ((-r.Jv) * ap) * B.im;
        B.ang = B.ang + mul(B.Iwi, r.Jwb * ap);
    }
}

__device__ __forceinline__ void row_warm(const rowv &r, body_state &A, body_state &B) // :74-87
{
    if (r.acc == 0.0) return;
    if (!A.stat)
    {
        A.vel = A.vel + (r.Jv * r.acc) * A.im;
        A.ang = A.ang + mul(A.Iwi, r.Jwa * r.acc);
    }
    if (!B.stat)
    {
        B.vel = B.vel + ((-r.Jv) * r.acc) * B.im;
        B.ang = B.ang + mul(B.Iwi, r.Jwb * r.acc);
    }
}

__device__ __forceinline__ void friction_block(rowv &t1, rowv &t2, double mu, double nacc, double i11,
                                               double i12, double i22, body_state &A, body_state &B) // :1131-1187
{
    double maxf = mu * nacc;
    double jv1 = row_jv(t1, A, B);
    double jv2 = row_jv(t2, A, B);
    double b1 = jv1 + 0.0;
    double b2 = jv2 + 0.0;
    double l1 = -(i11 * b1 + i12 * b2);
    double l2 = -(i12 * b1 + i22 * b2);
    double o1 = t1.acc, o2 = t2.acc;
    double n1 = o1 + l1, n2 = o2 + l2;
    double mag = hypot_pk(n1, n2);
    if (mag > maxf)
    {
        n1 = n1 * (maxf / mag);
        n2 = n2 * (maxf / mag);
    }
    t1.acc = n1;
    t2.acc = n2;
    double a1 = n1 - o1, a2 = n2 - o2;
    if (!A.stat)
    {
        A.vel = A.vel + (t1.Jv * a1 + t2.Jv * a2) * A.im;
        A.ang = A.ang + mul(A.Iwi, t1.Jwa * a1 + t2.Jwa * a2);
    }
    if (!B.stat)
    {
        B.vel = B.vel + ((-t1.Jv) * a1 - t2.Jv * a2) * B.im;
        B.ang = B.ang + mul(B.Iwi, t1.Jwb * a1 + t2.Jwb * a2);
    }
}

__device__ __forceinline__ void basis(v3 n, v3 &t1, v3 &t2) // :104-113
{
    double sign = copysign(1.0, n.z);
    double a = -1.0 / (sign + n.z);
    double b = n.x * n.y * a;
    t1 = mk(1.0 + sign * n.x * n.x * a, sign * b, -sign * n.x);
    t2 = mk(b, sign + n.y * n.y * a, -n.y);
}

__device__ __forceinline__ rowv make_row(const body_state &A, const body_state &B, v3 dir, v3 ra, v3 rb)
{
    rowv r;
    r.Jv = dir;
    r.Jwa = cross(ra, dir);
    r.Jwb = -cross(rb, dir);
    v3 ka = mul(A.Iwi, r.Jwa);
    v3 kb = mul(B.Iwi, r.Jwb);
    r.Meff = 1.0 / (((A.im + B.im) + dot(r.Jwa, ka)) + dot(r.Jwb, kb));
    r.bias = 0.0;
    r.acc = 0.0;
    return r;
}

// inverse mass, inverse world inertia and the static flag (velocities come separately)
__device__ __forceinline__ body_state ld_body(const bodies_dev &b, uint32_t i)
{
    body_state s;
    s.vel = mk(0.0, 0.0, 0.0);
    s.ang = mk(0.0, 0.0, 0.0);
    s.im = b.inv_mass[i];
    s.Iwi = ld9(b.Iw_inv, b.n, i);
    s.stat = b.is_static[i] != 0;
    return s;
}

// Contact c of manifold p: world normal n and lever arms as build_contact_jacobian
// forms them (:883-890) and whether the contact makes rows (a penetration that is not
// <= 0, so a NaN one does too, as in the reference's `if (penetration <= 0) continue`).
__device__ __forceinline__ bool contact_frame(const manifolds_dev &m, uint32_t sl, int c, v3 pa, v3 pb, qt qa,
                                              qt qb, v3 &n, v3 &ra, v3 &rb, double &pen)
{
    const double *d = m.data + static_cast<size_t>(c * kMF) * m.dcap + sl;
    const size_t s = m.dcap;
    const v3 nw = normalized(mk(d[0], d[s], d[2 * s]));
    const v3 la = mk(d[3 * s], d[4 * s], d[5 * s]);
    const v3 lb = mk(d[6 * s], d[7 * s], d[8 * s]);
    const v3 lnb = rotate(conj(qb), nw);
    ra = rotate(qa, la);
    rb = rotate(qb, lb);
    n = rotate(qb, lnb);
    pen = dot((pb + rb) - (pa + ra), n);
    return !(pen <= 0.0);
}

// Claim of a manifold in a colouring round: the round (from 1) above the complement of
// mix32(p). mix32 is a bijection, so ordering by it equals ordering by the priority
// (mix32(p) << 32) | p; an atomic max keeps this round's lowest priority at each body,
// and claims left from earlier rounds lose to any claim of the current one, so the
// claim array is cleared once per colouring, not every round.
__device__ __forceinline__ uint64_t claim_of(uint32_t p, uint32_t round)
{ return (static_cast<uint64_t>(round + 1u) << 32) | (0xFFFFFFFFu - mix32(p)); }

__device__ __forceinline__ uint32_t local_index(uint32_t p, uint32_t ia, const uint32_t *world_of,
                                                const uint32_t *pair_base)
{ return pair_base ? p - pair_base[world_of[ia]] : p; }

struct f3
{
    float x, y, z;
};
__device__ __forceinline__ f3 f3m(float x, float y, float z) { return {x, y, z}; }
__device__ __forceinline__ f3 to_f3(v3 a) { return {static_cast<float>(a.x), static_cast<float>(a.y), static_cast<float>(a.z)}; }
__device__ __forceinline__ float dotf(f3 a, f3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
__device__ __forceinline__ f3 scl(f3 a, float k) { return {a.x * k, a.y * k, a.z * k}; }
__device__ __forceinline__ f3 addf(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ v3 widen(f3 a) { return mk(static_cast<double>(a.x), static_cast<double>(a.y), static_cast<double>(a.z)); }

__device__ __forceinline__ f3 mulI(const float *I, f3 v)
{ return f3m((I[0] * v.x + I[1] * v.y) + I[2] * v.z, (I[3] * v.x + I[4] * v.y) + I[5] * v.z, (I[6] * v.x + I[7] * v.y) + I[8] * v.z); }
__device__ __forceinline__ f3 fcr(f3 a, f3 b) { return f3m(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x); }
__device__ __forceinline__ void fbasis(f3 n, f3 &t1, f3 &t2)
{
    const float sign = copysignf(1.0f, n.z);
    const float a = -1.0f / (sign + n.z);
    const float b = n.x * n.y * a;
    t1 = f3m(1.0f + sign * n.x * n.x * a, sign * b, -sign * n.x);
    t2 = f3m(b, sign + n.y * n.y * a, -n.y);
}
__device__ __forceinline__ uint32_t par_ld(uint32_t *par, uint32_t x)
{ return __hip_atomic_load(&par[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__device__ uint32_t uf_find(uint32_t *par, uint32_t x)
{
    uint32_t p = par_ld(par, x);
    while (p != x)
    {
        uint32_t gp = par_ld(par, p);
        if (gp != p) __hip_atomic_store(&par[x], gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); // path halving
        x = p;
        p = gp;
    }
    return x;
}

// Union-find with hooking of the larger root under the smaller: every component's root is
// its smallest body id, whatever order the unions run in. False if it gave up.
__device__ __forceinline__ bool uf_union(uint32_t *par, uint32_t a, uint32_t c)
{
    for (uint32_t guard = 0; guard < 4096u; ++guard)
    {
        const uint32_t ra = uf_find(par, a), rc = uf_find(par, c);
        if (ra == rc) return true;
        const uint32_t hi = ra > rc ? ra : rc, lo = ra > rc ? rc : ra;
        uint32_t expect = hi;
        if (__hip_atomic_compare_exchange_strong(&par[hi], &expect, lo, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return true;
    }
    return false;
}

} // namespace pk
