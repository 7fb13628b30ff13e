// GJK and EPA of one shape pair by one 64-lane wavefront (src/collision.cpp:165-509),
// with the results of pk_gjk.hpp's one-thread solver bit for bit: the same operations in
// the same order, spread over the lanes where they are independent.
//
// Why a wavefront: a solve is a chain of dependent steps. On one lane every step of an
// EPA expansion is a trip to private memory (about 20 us per expansion), so a batch too
// small to fill the chip is bounded by its longest chain. Here
//   - lanes 0-31 search shape A's support while lanes 32-63 search B's;
//   - each lane keeps faces lane, lane + 64, ... in registers, so the visibility test of
//     every face is one step, and the face bookkeeping is read with v_readlane;
//   - the silhouette walk (a few scalar instructions per visible face), the heap's path
//     and the lists' counts are uniform, in scalar registers;
//   - the new faces of an expansion are built one per lane;
//   - the nearest face is a minimum over the registers. The heap that the one-thread solver
//     keeps only decides between live faces at the same distance: the first time it has
//     to, it is built by repeating its pushes and pops so far, and kept from then on (a
//     push or pop compares its whole path at once, one LDS round trip).
// Many hits at once are bounded by the issue of vector instructions: on 143,000 hits of
// random hulls 4,235 per hit (5,146 with a heap from the first face on and the first
// tetrahedron built by every lane), 1.35 ms (2.08).
// The solver's uniform values come from v_readlane and ballots, so its branches are
// scalar. Capacity is 64 K faces; running out of it returns 3, as does a plane distance
// that is not finite (the heap's order then depends on the order of its comparisons):
// the caller reruns the solve with the one-thread solver.
#pragma once
#include "pk_gjk.hpp"

namespace pk
{
namespace wave
{

__device__ __forceinline__ uint32_t rl32(uint32_t x, int lane)
{ return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x), lane)); }
__device__ __forceinline__ double rl64(double x, int lane)
{
    const uint64_t u = static_cast<uint64_t>(__double_as_longlong(x));
    const uint64_t lo = rl32(static_cast<uint32_t>(u), lane), hi = rl32(static_cast<uint32_t>(u >> 32), lane);
    return __longlong_as_double(static_cast<long long>(hi << 32 | lo));
}
__device__ __forceinline__ v3 rl3(v3 v, int lane) { return mk(rl64(v.x, lane), rl64(v.y, lane), rl64(v.z, lane)); }
__device__ __forceinline__ uint32_t first32(uint32_t x)
{ return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(x))); }
__device__ __forceinline__ double first64(double x)
{
    const uint64_t u = static_cast<uint64_t>(__double_as_longlong(x));
    const uint64_t lo = first32(static_cast<uint32_t>(u)), hi = first32(static_cast<uint32_t>(u >> 32));
    return __longlong_as_double(static_cast<long long>(hi << 32 | lo));
}
// by value: a conditional expression of two array elements selects between their
// addresses, which pins the array in private memory
template <class T> __device__ __forceinline__ T sel(bool c, T a, T b) { return c ? a : b; }
__device__ __forceinline__ int lowest_bit(uint64_t m) { return __ffsll(static_cast<long long>(m)) - 1; }

// x moved down the lanes by a DPP step; lanes without a source keep x
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp64(double x)
{
    const uint64_t u = static_cast<uint64_t>(__double_as_longlong(x));
    const int lo = static_cast<int>(u), hi = static_cast<int>(u >> 32);
    const uint32_t l = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false));
    const uint32_t h = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false));
    return __longlong_as_double(static_cast<long long>(static_cast<uint64_t>(h) << 32 | l));
}
// the maximum of lanes 0-31 ends in lane 31, that of lanes 32-63 in lane 63: four shifts
// inside rows of 16 lanes, then lane 15 of each row into the next
__device__ __forceinline__ double half_max(double x)
{
    x = fmax(x, dpp64<0x111, 0xf>(x));
    x = fmax(x, dpp64<0x112, 0xf>(x));
    x = fmax(x, dpp64<0x114, 0xf>(x));
    x = fmax(x, dpp64<0x118, 0xf>(x));
    return fmax(x, dpp64<0x142, 0xa>(x));
}

// the minimum of all lanes, in every lane
__device__ __forceinline__ double wave_min(double x)
{
    auto less = [](double a, double b) { return a < b ? a : b; };
    x = less(dpp64<0x111, 0xf>(x), x);
    x = less(dpp64<0x112, 0xf>(x), x);
    x = less(dpp64<0x114, 0xf>(x), x);
    x = less(dpp64<0x118, 0xf>(x), x);
    x = less(dpp64<0x142, 0xa>(x), x);
    x = less(dpp64<0x143, 0xc>(x), x);
    return rl64(x, 63);
}

// The shape of this lane's half of the wavefront (A below lane 32, B above). A mesh of at
// most 32 vertices keeps one vertex per lane in registers (own).
struct shape
{
    gshape s;
    v3 vtx;
    bool own;
};
__device__ __forceinline__ bool upper() { return __lane_id() >= 32u; }

__device__ __forceinline__ shape make_shape(const gshape &s)
{
    shape w;
    w.s = s;
    const uint32_t c = __lane_id() & 31u;
    w.own = s.kind == 2 && s.uv == 0 && s.nv <= 32u;
    w.vtx = mk(0.0, 0.0, 0.0);
    if (w.own && c < s.nv) w.vtx = ldv(s.v, c);
    return w;
}

// uv_support's candidates (pk_gjk.hpp) one per lane: lanes 0-8 of a half take the 3 x 3
// ring and sector vertices, lanes 9 and 10 the poles, lanes 16-18 the bounds of the
// candidate rings' other sectors. val, idx: this lane's candidate (idx kNoIdx for none);
// ub: this lane's bound on the vertices that are no candidates. False where the search
// needs the full scan.
__device__ __forceinline__ bool uv_candidates(const gshape &s, v3 ld, double &val, uint32_t &idx, double &ub,
                                              double &slack)
{
    const int S = static_cast<int>(s.uv >> 16), T = static_cast<int>(s.uv & 0xFFFFu);
    const uint32_t c = __lane_id() & 31u;
    if (!(isfinite(ld.x) && isfinite(ld.y) && isfinite(ld.z))) return false;
    const double rho = sqrt(ld.x * ld.x + ld.z * ld.z);
    const double dn = sqrt(rho * rho + ld.y * ld.y);
    if (!(dn > 0.0)) return false;
    const float pif = 3.14159265f;
    const float phi = atan2f(static_cast<float>(rho / dn), static_cast<float>(ld.y / dn));
    int i0 = static_cast<int>(rintf(phi * (static_cast<float>(S) / pif)));
    i0 = i0 < 1 ? 1 : (i0 > S - 1 ? S - 1 : i0);
    int j0 = 0;
    if (rho > 0.0)
    {
        const float al = atan2f(static_cast<float>(ld.z / rho), static_cast<float>(ld.x / rho));
        j0 = static_cast<int>(rintf(al * (static_cast<float>(T) / (2.0f * pif))));
        j0 = ((j0 % T) + T) % T;
    }
    const int ilo = i0 > 1 ? i0 - 1 : 1, ihi = i0 < S - 1 ? i0 + 1 : S - 1;
    const double r = s.v[1];
    slack = 1e-12 * r * (fabs(ld.x) + fabs(ld.y) + fabs(ld.z));
    ub = -__builtin_inf();
    if (ilo > 1 || ihi < S - 1) ub = r * dn * static_cast<double>(cosf(1.3f * pif / static_cast<float>(S)));
    idx = kNoIdx;
    val = -__builtin_inf();
    if (c < 9u)
    {
        const int i = ilo + static_cast<int>(c) / 3, dj = static_cast<int>(c) % 3 - 1;
        if (i <= ihi) idx = 1u + static_cast<uint32_t>((i - 1) * T + (j0 + dj + T) % T);
    }
    else if (c == 9u)
        idx = 0;
    else if (c == 10u)
        idx = s.nv - 1;
    if (idx != kNoIdx) val = dot(ldv(s.v, idx), ld);
    if (T > 3 && c >= 16u && c < 19u && ilo + static_cast<int>(c - 16u) <= ihi)
    {
        const double cs = static_cast<double>(cosf(1.3f * 2.0f * pif / static_cast<float>(T)));
        const int i = ilo + static_cast<int>(c - 16u);
        const double *p = s.v + 3 * (1 + static_cast<size_t>(i - 1) * T);
        const double u = p[0] * rho * cs + p[1] * ld.y;
        ub = u > ub ? u : ub;
    }
    return true;
}

// the lowest index among the candidates of the lanes in mask (a half's lanes)
__device__ __forceinline__ uint32_t lowest_index(uint32_t bi, uint64_t mask)
{
    uint32_t best = kNoIdx;
    while (mask)
    {
        const int l = lowest_bit(mask);
        mask &= mask - 1;
        const uint32_t k = rl32(bi, l);
        best = k < best ? k : best;
    }
    return best;
}

// s_A(d) - s_B(-d) (collision.h:41-49) for a uniform d; every lane gets the result. The
// winner is support_idx's: the greatest dot product, the lowest index among equal ones,
// vertex 0 where its own product is NaN.
template <bool UV, bool MESH> __device__ __forceinline__ spt support(const shape &w, v3 d)
{
    const bool hi = upper();
    const uint32_t c = __lane_id() & 31u;
    const v3 dd = hi ? -d : d;
    double bv = -__builtin_inf();
    uint32_t bi = kNoIdx;
    bool nan0 = false;
    const v3 ld = rotate(conj(w.s.q), dd);
    bool scan = true;
    if (!MESH && w.s.kind != 2)
    {
        scan = false;
        if (c == 0u) // the corner's code by signs: the same for every lane of the half
        {
            const v3 k = w.s.kind == 1 ? ld : dd;
            bi = (k.x >= 0 ? 1u : 0u) | (k.y >= 0 ? 2u : 0u) | (k.z >= 0 ? 4u : 0u);
            bv = 0.0;
        }
    }
    if (UV && __ballot(w.s.uv != 0))
    {
        double val = -__builtin_inf(), ub = -__builtin_inf(), slack = 0.0;
        uint32_t idx = kNoIdx;
        const bool tried = w.s.uv != 0 && uv_candidates(w.s, ld, val, idx, ub, slack);
        const bool bad = tried && idx != kNoIdx && !(val == val);
        const double vm = half_max(val), um = half_max(ub);
        const double vl = rl64(vm, 31), vu = rl64(vm, 63), ul = rl64(um, 31), uu = rl64(um, 63);
        const double vh = hi ? vu : vl, uh = hi ? uu : ul;
        const uint64_t nans = __ballot(bad), half = hi ? 0xFFFFFFFF00000000ull : 0xFFFFFFFFull;
        // certified: no vertex outside the candidates can reach the best of them
        if (tried && !(nans & half) && vh > uh + slack)
        {
            scan = false;
            bv = val;
            bi = idx;
        }
    }
    if (scan)
    {
        if (w.own)
        {
            if (c < w.s.nv)
            {
                const double t = dot(w.vtx, ld);
                if (c == 0u) nan0 = t != t;
                if (t == t)
                {
                    bv = t;
                    bi = c;
                }
            }
        }
        else
            for (uint32_t i = c; i < w.s.nv; i += 32u)
            {
                const double t = dot(ldv(w.s.v, i), ld);
                if (i == 0u) nan0 = t != t;
                if (t == t && (bi == kNoIdx || t > bv))
                {
                    bv = t;
                    bi = i;
                }
            }
    }
    const double m = half_max(bv);
    const double ml = rl64(m, 31), mu = rl64(m, 63), mh = hi ? mu : ml;
    const uint64_t eq = __ballot(bi != kNoIdx && bv == mh), n0 = __ballot(nan0);
    spt r;
    r.ia = (n0 & 0xFFFFFFFFull) ? 0u : lowest_index(bi, eq & 0xFFFFFFFFull);
    r.ib = (n0 >> 32) ? 0u : lowest_index(bi, eq & 0xFFFFFFFF00000000ull);
    const uint32_t f = hi ? r.ib : r.ia;
    v3 pt;
    if (MESH || w.s.kind == 2)
    {
        const v3 va = rl3(w.vtx, static_cast<int>(r.ia & 31u)), vb = rl3(w.vtx, 32 + static_cast<int>(r.ib & 31u));
        v3 lv = sel3(hi, vb, va);
        if (!w.own) lv = ldv(w.s.v, f);
        pt = rotate(w.s.q, lv) + w.s.a;
    }
    else
        pt = support_at(w.s, f);
    r.p = rl3(pt, 0) - rl3(pt, 32);
    return r;
}

// boolean GJK (collision.cpp:165-189); the simplex is uniform
template <bool UV, bool MESH> __device__ __forceinline__ bool gjk(const shape &w, simplex &x)
{
    x.n = 0;
    v3 dir = mk(1.0, 0.0, 0.0);
    for (int it = -1; it < 100; ++it) // pass -1 is the initial support
    {
        const spt np = support<UV, MESH>(w, dir);
        if (it < 0)
        {
            sx_push(x, np);
            if (sqn(np.p) < 1e-12) return true;
            dir = -normalized(np.p);
            continue;
        }
        if (dot(np.p, dir) <= 0.0) return false;
        sx_push(x, np);
        if (x.n == 2)
            handle_line(x, dir);
        else if (x.n == 3)
            handle_triangle(x, dir);
        else if (handle_tetrahedron(x, dir))
            return true;
    }
    return false;
}

// The part of a solve that lives in LDS: the polytope's points and the heap (node i's
// children at 2i and 2i + 1, root at 1, so two siblings are one aligned 16-byte read)
template <int K> struct store
{
    static_assert(64 * K <= 0xFFFF, "face indices are 16 bits");
    static constexpr int fcap = 64 * K, pcap = 68;
    alignas(16) double hk[fcap + 2];
    double px[pcap], py[pcap], pz[pcap];
    uint32_t pia[pcap], pib[pcap];
    uint16_t hf[fcap + 2];
};

// LDS written by some lanes of the (single) wavefront and read by others
__device__ __forceinline__ void lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr uint32_t kNoFace = 0xFFFFu;

template <int K> struct solver
{
    store<K> &m;
    // faces lane, lane + 64, ...: normal and plane distance, vertices (one byte each), the
    // faces across edges (v0, v1), (v1, v2) and (v2, v0)
    double nx[K], ny[K], nz[K], fd[K];
    uint32_t fv[K], f01[K], f2[K];
    uint64_t live[K]; // faces not obsolete (uniform)
    int npoly = 0, nfaces = 0, nheap = 0;
    uint32_t lane;
    // without a heap until two live faces are nearest at once; lane i holds expansion i's
    // face and (from bit 16) the face count after it, from which the heap can be built
    bool heaped = false;
    uint32_t hist = 0;

    __device__ explicit solver(store<K> &s) : m(s), lane(__lane_id())
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
        {
            nx[k] = ny[k] = nz[k] = fd[k] = 0.0;
            fv[k] = f01[k] = f2[k] = 0;
            live[k] = 0;
        }
    }
    __device__ __forceinline__ v3 P(int i) const { return mk(m.px[i], m.py[i], m.pz[i]); }
    __device__ __forceinline__ void put_point(int i, const spt &p)
    {
        if (lane == 0)
        {
            m.px[i] = p.p.x;
            m.py[i] = p.p.y;
            m.pz[i] = p.p.z;
            m.pia[i] = p.ia;
            m.pib[i] = p.ib;
        }
    }
    __device__ __forceinline__ uint32_t word(const uint32_t (&a)[K], int f) const
    {
        uint32_t r = rl32(a[0], f & 63);
#pragma unroll
        for (int k = 1; k < K; ++k)
            if (64 * k <= f) r = rl32(a[k], f & 63);
        return r;
    }
    __device__ __forceinline__ double real(const double (&a)[K], int f) const
    {
        double r = rl64(a[0], f & 63);
#pragma unroll
        for (int k = 1; k < K; ++k)
            if (64 * k <= f) r = rl64(a[k], f & 63);
        return r;
    }
    // of faces 0 .. 64 N
    template <int N> __device__ __forceinline__ static bool bit(const uint64_t (&s)[K], uint32_t f)
    {
        uint64_t w = s[0];
#pragma unroll
        for (int k = 1; k < N; ++k) w = sel((f >> 6) == static_cast<uint32_t>(k), s[k], w);
        return (w >> (f & 63u)) & 1u;
    }
    template <int N> __device__ __forceinline__ static void clear(uint64_t (&s)[K], uint32_t f)
    {
#pragma unroll
        for (int k = 0; k < N; ++k) s[k] &= ~(N == 1 || (f >> 6) == static_cast<uint32_t>(k) ? 1ull << (f & 63u) : 0ull);
    }

    // push_heap's sift (libstdc++): the keys do not increase towards the root, so the
    // ancestors that move down are the ones greater than d, a run from the new leaf up
    __device__ __forceinline__ void push(int f, double d)
    {
        const uint32_t n = static_cast<uint32_t>(++nheap);
        const uint32_t depth = 31u - static_cast<uint32_t>(__clz(static_cast<int>(n)));
        const bool anc = lane < depth;
        const uint32_t a = anc ? n >> (lane + 1u) : 1u;
        const double key = m.hk[a];
        const uint16_t face = m.hf[a];
        const uint32_t g = static_cast<uint32_t>(__popcll(__ballot(anc && key > d)));
        lds_sync();
        if (lane < g)
        {
            m.hk[n >> lane] = key;
            m.hf[n >> lane] = face;
        }
        if (lane == g)
        {
            m.hk[n >> g] = d;
            m.hf[n >> g] = static_cast<uint16_t>(f);
        }
        lds_sync();
    }
    // pop_heap, and the faces it skips (those before face `want`, or before the first live
    // one where that is negative): the hole runs from the root to a leaf along the
    // smaller children (the right one of equal ones), then the last element rises from
    // that leaf past the keys above its own. The path is a run of bits; of its keys, the
    // ones not above the last element's move up by one node.
    __device__ __forceinline__ int pop(int want)
    {
        while (nheap > 0)
        {
            const uint32_t n = static_cast<uint32_t>(nheap);
            const int top = static_cast<int>(first32(m.hf[1]));
            if (n > 1)
            {
                const double vd = first64(m.hk[n]);
                const uint32_t vf = first32(m.hf[n]);
                const uint32_t r = n - 1; // nodes 1..r remain
                uint64_t left[(K + 1) / 2 + 1];
#pragma unroll
                for (int k = 0; k < (K + 1) / 2 + 1; ++k)
                {
                    const uint32_t i = 64u * k + lane;
                    uint64_t lm = 0;
                    if (128u * k <= r)
                    {
                        bool lw = true; // no right child: the left one
                        if (2 * i + 1 <= r)
                        {
                            const double2 c = *reinterpret_cast<const double2 *>(&m.hk[2 * i]);
                            lw = c.y > c.x;
                        }
                        lm = __ballot(lw);
                    }
                    left[k] = lm;
                }
                uint32_t leaf = 1, len = 0;
                while (2 * leaf <= r)
                {
                    uint64_t w = left[0];
#pragma unroll
                    for (int k = 1; k < (K + 1) / 2 + 1; ++k) w = sel((leaf >> 6) == static_cast<uint32_t>(k), left[k], w);
                    leaf = 2 * leaf + (((w >> (leaf & 63u)) & 1u) ? 0u : 1u);
                    ++len;
                }
                const bool on = lane < len; // node leaf >> lane of the path, root excluded
                const uint32_t a = on ? leaf >> lane : 1u;
                const double key = m.hk[a];
                const uint16_t face = m.hf[a];
                const uint32_t g = static_cast<uint32_t>(__popcll(__ballot(on && key > vd)));
                lds_sync();
                if (on && lane >= g)
                {
                    m.hk[leaf >> (lane + 1u)] = key;
                    m.hf[leaf >> (lane + 1u)] = face;
                }
                if (lane == 0)
                {
                    m.hk[leaf >> g] = vd;
                    m.hf[leaf >> g] = static_cast<uint16_t>(vf);
                }
                lds_sync();
            }
            --nheap;
            if (want < 0 ? bit<K>(live, static_cast<uint32_t>(top)) : top == want) return top;
        }
        return -1;
    }
    __device__ __forceinline__ void push_range(int from, int to)
    {
        for (int f = from; f < to; ++f) push(f, real(fd, f));
    }
    // The face that the heap's next pop returns (-1: none), for expansion it. That is the
    // nearest live face, which the registers tell. Only where several are equally near does
    // the order of the heap's operations so far decide: it is built then, by repeating them.
    __device__ __forceinline__ int nearest(int it)
    {
        if (!heaped)
        {
            double b = __builtin_inf();
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (64 * k < nfaces)
                {
                    const double d = __builtin_amdgcn_inverse_ballot_w64(live[k]) ? fd[k] : __builtin_inf();
                    b = d < b ? d : b;
                }
            b = wave_min(b);
            int n = 0, f = -1;
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (64 * k < nfaces)
                {
                    const uint64_t eq = __ballot(fd[k] == b) & live[k];
                    n += __popcll(eq);
                    f = eq ? 64 * k + lowest_bit(eq) : f;
                }
            if (n < 2) return f;
            heaped = true;
            push_range(0, 4);
            for (int i = 0, from = 4; i < it; ++i)
            {
                const uint32_t h = rl32(hist, i);
                pop(static_cast<int>(h & 0xFFFFu));
                push_range(from, static_cast<int>(h >> 16));
                from = static_cast<int>(h >> 16);
            }
        }
        return pop(-1);
    }

    // :355-388 from the four points, face f in lane f; false when a plane distance is not
    // finite. Faces (0 1 2), (0 2 3), (0 3 1), (1 3 2) run opposite ways along the edge that
    // any two share, and still do if both are turned: a face's neighbour across an edge is the
    // one without its third vertex, if it was turned alike.
    __device__ __forceinline__ bool initial_tetrahedron(const v3 (&q)[4])
    {
        const uint32_t f = lane & 3u;
        const uint32_t i0 = f >> 1 & f, i1 = f == 0u ? 1u : (f == 1u ? 2u : 3u);
        uint32_t i2 = f == 0u ? 2u : (f == 1u ? 3u : (f == 2u ? 1u : 2u)), iv = i1;
        const uint32_t io = f == 0u ? 3u : (f == 3u ? 0u : f); // the vertex that face f lacks
        auto at = [&](uint32_t i) { return sel3(i < 2u, sel3(i == 0u, q[0], q[1]), sel3(i == 2u, q[2], q[3])); };
        const v3 pi = at(i0);
        v3 nrm = cross(at(iv) - pi, at(i2) - pi);
        if (sqn(nrm) < 1e-12)
            nrm = mk(0.0, 0.0, 0.0);
        else
            nrm = normalized(nrm);
        const bool turn = dot(nrm, at(io) - pi) > 0.0;
        if (turn)
        {
            const uint32_t t = iv;
            iv = i2;
            i2 = t;
            nrm = -nrm;
        }
        const double d = dot(nrm, pi);
        const uint32_t turned = static_cast<uint32_t>(__ballot(turn)) & 0xFu;
        auto across = [&](uint32_t third)
        {
            const uint32_t j = third == 0u ? 3u : (third == 3u ? 0u : third);
            return ((turned >> j ^ turned >> f) & 1u) ? kNoFace : j;
        };
        if (lane < 4u)
        {
            nx[0] = nrm.x;
            ny[0] = nrm.y;
            nz[0] = nrm.z;
            fd[0] = d;
            fv[0] = i0 | iv << 8 | i2 << 16;
            f01[0] = across(i2) | across(i0) << 16;
            f2[0] = across(iv);
        }
        nfaces = 4;
        live[0] = 0xFull;
        return !__ballot(!isfinite(d));
    }

    // :315-353 from face f0 and the new point p. Horizon edge h (start, end, face across:
    // 8 + 8 + 16 bits) ends in lane (nfaces + h) & 63 of edges, the lane that will hold the
    // face built on it. Returns the edge count, -1 past 64 edges or stack entries.
    template <int N> __device__ __forceinline__ int silhouette(int f0, v3 p, uint32_t &edges)
    {
        uint64_t vis[K];
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            uint64_t seen = 0;
            if (64 * k < nfaces) seen = __ballot(dot(mk(nx[k], ny[k], nz[k]), p) > fd[k] + 1e-6);
            vis[k] = seen;
        }
        clear<N>(live, static_cast<uint32_t>(f0));
        uint32_t stack = 0; // entry i in lane i
        int sp = 0, nh = 0, cur = f0;
        for (;;)
        {
            const uint32_t v = word(fv, cur), a01 = word(f01, cur), a2 = word(f2, cur);
#pragma unroll
            for (int i = 0; i < 3; ++i)
            {
                const uint32_t nb = i == 0 ? (a01 & 0xFFFFu) : (i == 1 ? a01 >> 16 : a2);
                if (nb == kNoFace || !bit<N>(live, nb)) continue;
                if (bit<N>(vis, nb))
                {
                    clear<N>(live, nb);
                    if (sp >= 64) return -1;
                    stack = lane == static_cast<uint32_t>(sp) ? nb : stack;
                    ++sp;
                }
                else
                {
                    if (nh >= 64) return -1;
                    const uint32_t s = (v >> (8 * i)) & 0xFFu, e = (v >> (8 * ((i + 1) % 3))) & 0xFFu;
                    edges = lane == static_cast<uint32_t>((nfaces + nh) & 63) ? (s | e << 8 | nb << 16) : edges;
                    ++nh;
                }
            }
            if (sp == 0) return nh;
            cur = static_cast<int>(rl32(stack, --sp));
        }
    }

    // :424-454: every lane gets the contact
    __device__ __forceinline__ void barycentric(int f, const shape &w, double *out) const
    {
        const uint32_t v = word(fv, f);
        const int i0 = static_cast<int>(v & 0xFFu), i1 = static_cast<int>((v >> 8) & 0xFFu), i2 = static_cast<int>(v >> 16);
        const v3 q0 = P(i0), q1 = P(i1), q2 = P(i2);
        const uint32_t *feat = upper() ? m.pib : m.pia;
        const v3 p0 = support_at(w.s, feat[i0]), p1 = support_at(w.s, feat[i1]), p2 = support_at(w.s, feat[i2]);
        const v3 nrm = mk(real(nx, f), real(ny, f), real(nz, f));
        const double d = real(fd, f);
        const v3 pm = nrm * d;
        const v3 v0 = q1 - q0, v1 = q2 - q0, v2 = pm - q0;
        const double d00 = dot(v0, v0), d01 = dot(v0, v1), d11 = dot(v1, v1);
        const double d20 = dot(v2, v0), d21 = dot(v2, v1);
        const double denom = d00 * d11 - d01 * d01;
        const double bv = (d11 * d20 - d01 * d21) / denom;
        const double bw = (d00 * d21 - d01 * d20) / denom;
        const double bu = 1.0 - bv - bw;
        const v3 wit = (p0 * bu + p1 * bv) + p2 * bw; // A's in the lower half, B's in the upper
        const v3 wa = rl3(wit, 0), wb = rl3(wit, 32);
        out[0] = -nrm.x;
        out[1] = -nrm.y;
        out[2] = -nrm.z;
        out[3] = wa.x;
        out[4] = wa.y;
        out[5] = wa.z;
        out[6] = wb.x;
        out[7] = wb.y;
        out[8] = wb.z;
        out[9] = d;
    }
};

// epa_solve (pk_gjk.hpp) by the wavefront: 0 no contact, 1 contact in out (every lane), 3
// rerun with the one-thread solver
template <bool UV, bool MESH, int K>
__device__ __forceinline__ int epa_solve(const shape &w, simplex &x, store<K> &st, double *out)
{
    if (x.n < 4 && !pad_simplex_with(x, [&](v3 d) { return support<UV, MESH>(w, d); })) return 0;
    solver<K> e(st);
    e.put_point(0, x.s0);
    e.put_point(1, x.s1);
    e.put_point(2, x.s2);
    e.put_point(3, x.s3);
    e.npoly = 4;
    lds_sync();
    const v3 q[4] = {x.s0.p, x.s1.p, x.s2.p, x.s3.p};
    if (!e.initial_tetrahedron(q)) return 3;
    int it = 0;
    for (; it < 64; ++it)
    {
        const int mf = e.nearest(it);
        if (mf < 0) return 0;
        const v3 nrm = mk(e.real(e.nx, mf), e.real(e.ny, mf), e.real(e.nz, mf));
        const double d = e.real(e.fd, mf);
        const spt p = support<UV, MESH>(w, nrm);
        const double pd = dot(nrm, p.p);
        if (pd - d < 1e-6)
        {
            e.barycentric(mf, w, out);
            return 1;
        }
        uint32_t edges = 0;
        const int nh = e.nfaces <= 64 ? e.template silhouette<1>(mf, p.p, edges) : e.template silhouette<K>(mf, p.p, edges);
        if (nh < 0) return 3;
        e.hist = e.lane == static_cast<uint32_t>(it) ? static_cast<uint32_t>(mf | (e.nfaces + nh) << 16) : e.hist;
        if (nh == 0)
        {
            ++it;
            break;
        }
        const int base = e.nfaces;
        if (e.npoly >= store<K>::pcap || base + nh > store<K>::fcap) return 3;
        const int pi = e.npoly++;
        e.put_point(pi, p);
        // face base + h on edge h, in lane (base + h) & 63
        const uint32_t h = (e.lane - static_cast<uint32_t>(base)) & 63u;
        const bool mine = h < static_cast<uint32_t>(nh);
        const uint32_t s_own = edges & 0xFFu, e_own = (edges >> 8) & 0xFFu;
        const v3 ps = e.P(static_cast<int>(mine ? s_own : 0u)), pe = e.P(static_cast<int>(mine ? e_own : 0u));
        v3 fn = cross(pe - ps, p.p - ps);
        if (sqn(fn) < 1e-12)
            fn = mk(0.0, 0.0, 0.0);
        else
            fn = normalized(fn);
        const double dist = dot(fn, ps);
        if (__ballot(mine && !isfinite(dist))) return 3;
        // links between the new faces (:488-498): for face x the pairs (y, x), y < x, then
        // (x, y), y > x, in that order; and the faces across the horizon (:305-313)
        uint32_t a1 = kNoFace, a2 = kNoFace;
        for (int y = 0; y < nh; ++y)
        {
            const uint32_t ey = rl32(edges, (base + y) & 63);
            const uint32_t s_y = ey & 0xFFu, e_y = (ey >> 8) & 0xFFu, across = ey >> 16;
            const uint32_t fy = static_cast<uint32_t>(base + y);
            const bool end_to_start = e_own == s_y, start_to_end = s_own == e_y; // (x, y) consecutive; (y, x)
            const bool before = static_cast<uint32_t>(y) < h;
            if (static_cast<uint32_t>(y) != h)
            {
                // pair (i, j), i < j: i's end is j's start first, else i's start is j's end
                const bool take2 = before ? start_to_end : (!end_to_start && start_to_end);
                const bool take1 = before ? (!start_to_end && end_to_start) : end_to_start;
                if (take1) a1 = fy;
                if (take2) a2 = fy;
            }
#pragma unroll
            for (int k = 0; k < K; ++k)
            {
                if (64 * k >= base) break;
                const bool own = e.lane + 64u * k == across;
                const bool at0 = (e.fv[k] & 0xFFu) == e_y, at1 = ((e.fv[k] >> 8) & 0xFFu) == e_y;
                const uint32_t n01 = sel(at0, (e.f01[k] & 0xFFFF0000u) | fy,
                                         sel(at1, (e.f01[k] & 0xFFFFu) | fy << 16, e.f01[k]));
                e.f01[k] = sel(own, n01, e.f01[k]);
                e.f2[k] = sel(own && !at0 && !at1, fy, e.f2[k]);
            }
        }
        const int slot = static_cast<int>((static_cast<uint32_t>(base) + h) >> 6);
#pragma unroll
        for (int k = 0; k < K; ++k)
        {
            if (64 * k >= base + nh || 64 * k + 64 <= base) continue;
            const bool put = mine && slot == k;
            e.nx[k] = sel(put, fn.x, e.nx[k]);
            e.ny[k] = sel(put, fn.y, e.ny[k]);
            e.nz[k] = sel(put, fn.z, e.nz[k]);
            e.fd[k] = sel(put, dist, e.fd[k]);
            e.fv[k] = sel(put, s_own | e_own << 8 | static_cast<uint32_t>(pi) << 16, e.fv[k]);
            e.f01[k] = sel(put, (edges >> 16) | a1 << 16, e.f01[k]);
            e.f2[k] = sel(put, a2, e.f2[k]);
        }
        const int end = base + nh;
#pragma unroll
        for (int k = 0; k < K; ++k)
        {
            const int lo = base > 64 * k ? base - 64 * k : 0, hi = end - 64 * k < 64 ? end - 64 * k : 64;
            e.live[k] |= lo < hi ? (~0ull >> (64 - hi)) & (~0ull << lo) : 0ull;
        }
        if (e.heaped) e.push_range(base, end);
        e.nfaces = end;
        lds_sync(); // point pi, which every lane may read from here on
    }
    const int mf = e.nearest(it);
    if (mf < 0) return 0;
    e.barycentric(mf, w, out);
    return 1;
}

} // namespace wave
} // namespace pk
