// Contact solve by islands (constraint_solver::setup_contacts / solve_constraints,
// include/physkit/collision/constraint.h:1052-1201): the row manifolds are grouped by
// connected component over dynamic bodies (an island), and one workgroup takes a chunk of
// whole islands through everything: colouring, row setup, warm start, every pass and the
// impulse write-back. Islands share no dynamic body, so a chunk needs nothing from another.
//
// What bounds it: with few bodies moving, one colour of one pass is a chain of dependent FP64
// operations (up to four contacts one after the other, a normal row and a friction block
// each) between two barriers, and passes x colours of these run in sequence. So a manifold
// takes two lanes, one for each body: a lane holds its body's inverse mass and inertia and
// lever arms, computes its half of every J.v and applies its half of every impulse, and the
// halves meet through a DPP exchange with the neighbour lane, in the order of operations of
// the sequential solve (bit for bit). A lane builds its manifold's rows from the manifold and keeps
// them across the passes; velocities are in LDS. FP32 rows fit its registers (171). FP64 rows
// of four contacts do not: both FP64 forms use all 256 that 512 threads leave a lane and
// spill 63 and 64 more to private memory (168 and 164 bytes a lane), 19 loads of which lie
// in the loop over passes and colours.
// Colours come from the same rounds as the global colouring (k_solver.hip), on LDS claims.
//
// Measured, solver stage per step, against global colouring rounds (three launches each),
// island sort, row setup, one manifold per thread and write-back as separate kernels: 64
// boxes 0.18 -> 0.09 ms, 1,024 boxes 0.47 -> 0.29, 10,000 bodies of batched worlds 0.40 ->
// 0.18, 720,000 (mixed) 0.49 -> 0.26, granular 131,072 (mixed) 0.37 -> 0.14, 16,384 hulls
// 0.95 -> 0.69, 64 pyramids 1.65 -> 0.95. A pyramid's step is 8 colours x 21 passes at about
// 5 us: three contacts at about 500 FP64 instructions of 7 cycles each on one lane.
#include "pk_solver.hpp"

#include <type_traits>

namespace pk
{
namespace
{
constexpr int kBlock = 256;
unsigned grid(size_t n) { return static_cast<unsigned>((n + kBlock - 1) / kBlock); }

// unions happen in k_row_flags
__global__ void k_island_init(uint32_t *par, uint32_t *cnt, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    par[i] = i;
    cnt[i] = 0;
}

// island root and rank inside the island of every listed manifold, manifolds per root, and
// the longest island. Lanes of a wavefront that share a root add once for the first
// few roots found (an island of many manifolds would serialise on its counter).
__global__ void __launch_bounds__(kBlock)
    k_island_roots(const uint64_t *keys, const uint32_t *list, uint32_t n_bound, bodies_dev b, uint32_t *par,
                   uint32_t *cnt, uint32_t *root_of, uint32_t *rank_of, unsigned long long *counters)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n = static_cast<uint32_t>(min(static_cast<unsigned long long>(n_bound), counters[C_NLIST]));
    uint32_t len = 0;
    if (i < n)
    {
        const uint64_t key = keys[list[i]];
        uint32_t a = static_cast<uint32_t>(key >> 32);
        if (b.is_static[a]) a = static_cast<uint32_t>(key & 0xFFFFFFFFu);
        const uint32_t r = uf_find(par, a);
        uint32_t rank = kNone;
        for (int tries = 0; tries < 4 && rank == kNone; ++tries)
        {
            const uint32_t lead = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(r)));
            const uint64_t same = __ballot(r == lead);
            if (r == lead)
            {
                const int first = __ffsll(static_cast<long long>(same)) - 1, lane = static_cast<int>(__lane_id());
                uint32_t at = 0;
                if (lane == first) at = atomicAdd(&cnt[r], static_cast<uint32_t>(__popcll(same)));
                rank = __shfl(at, first) + static_cast<uint32_t>(__popcll(same & ((1ull << lane) - 1ull)));
            }
        }
        if (rank == kNone) rank = atomicAdd(&cnt[r], 1u);
        root_of[i] = r;
        rank_of[i] = rank;
        len = rank + 1;
    }
    block_max(&counters[C_ISL_MAX], len);
}

// each island's first position: islands lie whole, in no particular order (no result depends
// on which islands share a chunk)
__global__ void __launch_bounds__(kBlock) k_island_base(const uint32_t *cnt, uint32_t n, uint32_t *base,
                                                        unsigned long long *counters)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t v = i < n ? cnt[i] : 0u;
    const unsigned long long at = block_reserve(&counters[C_ISL_CUR], v);
    if (v) base[i] = static_cast<uint32_t>(at);
}

__global__ void k_island_scatter(const uint32_t *list, uint32_t nl, const uint32_t *root_of, const uint32_t *rank_of,
                                 const uint32_t *base, uint32_t *ord, uint32_t *isl)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nl) return;
    const uint32_t r = root_of[i], at = base[r] + rank_of[i];
    ord[at] = list[i];
    isl[at] = r;
}

// ---- a manifold's two sides: S sides per lane (1: the neighbour lane has the other) ----
__device__ __forceinline__ bool side_b() { return (__lane_id() & 1u) != 0; }
__device__ __forceinline__ int swap32(int x) { return __builtin_amdgcn_update_dpp(x, x, 0xB1, 0xf, 0xf, false); } // lane ^ 1
__device__ __forceinline__ float swapped(float x) { return __int_as_float(swap32(__float_as_int(x))); }
__device__ __forceinline__ double swapped(double x)
{
    const uint64_t u = static_cast<uint64_t>(__double_as_longlong(x));
    const uint64_t lo = static_cast<uint32_t>(swap32(static_cast<int>(u))), hi = static_cast<uint32_t>(swap32(static_cast<int>(u >> 32)));
    return __longlong_as_double(static_cast<long long>(hi << 32 | lo));
}
// the values of side A and side B
template <class T> __device__ __forceinline__ void both(const T (&x)[2], T &a, T &b)
{
    a = x[0];
    b = x[1];
}
template <class T> __device__ __forceinline__ void both(const T (&x)[1], T &a, T &b)
{
    const T o = swapped(x[0]);
    a = side_b() ? o : x[0];
    b = side_b() ? x[0] : o;
}
// ((vA + wA) - vB) + wB from each side's v and w
template <class T> __device__ __forceinline__ T jv_sum(const T (&v)[2], const T (&w)[2])
{ return ((v[0] + w[0]) - v[1]) + w[1]; }
template <class T> __device__ __forceinline__ T jv_sum(const T (&v)[1], const T (&w)[1])
{
    const bool sb = side_b();
    const T sum = v[0] + w[0];
    const T o0 = swapped(sb ? v[0] : sum), o1 = swapped(w[0]);
    return ((sb ? o0 : sum) - (sb ? v[0] : o0)) + (sb ? w[0] : o1);
}
// x on side A, -x on side B
template <int S> __device__ __forceinline__ v3 flip(v3 x, int s)
{
    const bool neg = S == 2 ? s == 1 : side_b();
    return neg ? -x : x;
}
template <int S> __device__ __forceinline__ f3 flip(f3 x, int s)
{
    const bool neg = S == 2 ? s == 1 : side_b();
    return neg ? f3m(-x.x, -x.y, -x.z) : x;
}

struct side64
{
    v3 vel, ang;
    double im;
    m3 I;
    bool stat;
};
struct side32
{
    v3 vel, ang; // FP64 accumulators
    float im;
    float I[9];
    bool stat;
};
// A contact's rows: normal, the tangent basis' factor -1 / (sign + n.z), lever arms, normal
// mass and bias, friction block and impulses
template <class T, class V, int S> struct row_t
{
    V n, r[S]; // r is kept in LDS between colours where a lane holds both sides
    T a, meff, bias, i11, i12, i22, an, a1, a2;
};
// The FP32 solve of an island of more than kIslandMaxColours colours: the tangents and Jacobians
// themselves, computed in FP64 and rounded once, as the per-colour launches keep them
template <int S> struct row32_t
{
    f3 n, t1, t2, jn[S], j1[S], j2[S];
    float meff, bias, i11, i12, i22, an, a1, a2;
};

// row_apply and friction_block (pk_solver.hpp) with the Jacobians rebuilt by the operations
// of basis and make_row
template <int S>
__device__ __forceinline__ void solve_rows(row_t<double, v3, S> &k, double mu, bool warm, side64 (&b)[S])
{
    const double sign = copysign(1.0, k.n.z);
    const double bb = k.n.x * k.n.y * k.a;
    const v3 t1 = mk(1.0 + sign * k.n.x * k.n.x * k.a, sign * bb, -sign * k.n.x);
    const v3 t2 = mk(bb, sign + k.n.y * k.n.y * k.a, -k.n.y);
    v3 jn[S], j1[S], j2[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
    {
        jn[s] = flip<S>(cross(k.r[s], k.n), s);
        j1[s] = flip<S>(cross(k.r[s], t1), s);
        j2[s] = flip<S>(cross(k.r[s], t2), s);
    }
    if (warm) // row_warm
    {
        auto push = [&](v3 dir, const v3 (&j)[S], double acc)
        {
            if (acc == 0.0) return;
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (!b[s].stat)
                {
                    b[s].vel = b[s].vel + (flip<S>(dir, s) * acc) * b[s].im;
                    b[s].ang = b[s].ang + mul(b[s].I, j[s] * acc);
                }
        };
        push(k.n, jn, k.an);
        push(t1, j1, k.a1);
        push(t2, j2, k.a2);
        return;
    }
    double x[S], y[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
    {
        x[s] = dot(k.n, b[s].vel);
        y[s] = dot(jn[s], b[s].ang);
    }
    const double jv = jv_sum(x, y);
    const double cfp = 0.0 * k.an;
    const double lambda = -((jv + k.bias) + cfp) * k.meff;
    const double old = k.an, v = old + lambda;
    k.an = (v < 0.0) ? 0.0 : ((DBL_MAX < v) ? DBL_MAX : v);
    const double ap = k.an - old;
    double p[S], q[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
    {
        if (!b[s].stat)
        {
            b[s].vel = b[s].vel + (flip<S>(k.n, s) * ap) * b[s].im;
            b[s].ang = b[s].ang + mul(b[s].I, jn[s] * ap);
        }
        x[s] = dot(t1, b[s].vel);
        y[s] = dot(j1[s], b[s].ang);
        p[s] = dot(t2, b[s].vel);
        q[s] = dot(j2[s], b[s].ang);
    }
    const double maxf = mu * k.an;
    const double b1 = jv_sum(x, y) + 0.0, b2 = jv_sum(p, q) + 0.0;
    const double l1 = -(k.i11 * b1 + k.i12 * b2);
    const double l2 = -(k.i12 * b1 + k.i22 * b2);
    const double o1 = k.a1, o2 = k.a2;
    double n1 = o1 + l1, n2 = o2 + l2;
    const double mag = hypot_pk(n1, n2);
    if (mag > maxf)
    {
        n1 = n1 * (maxf / mag);
        n2 = n2 * (maxf / mag);
    }
    k.a1 = n1;
    k.a2 = n2;
    const double d1 = n1 - o1, d2 = n2 - o2;
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (!b[s].stat)
        {
            b[s].vel = b[s].vel + (flip<S>(t1, s) * d1 + flip<S>(t2, s) * d2) * b[s].im;
            b[s].ang = b[s].ang + mul(b[s].I, j1[s] * d1 + j2[s] * d2);
        }
}
// the FP32 solve: row arithmetic in FP32, increments added to the FP64 velocities. k: impulses, mass,
// bias and friction block of the rows along n, t1 and t2
template <int S, class K>
__device__ __forceinline__ void apply_rows32(K &k, f3 n, f3 t1, f3 t2, const f3 (&jn)[S], const f3 (&j1)[S],
                                             const f3 (&j2)[S], float mu, bool warm, side32 (&b)[S])
{
    auto push = [&](int s, f3 lin, f3 ang)
    {
        if (b[s].stat) return;
        b[s].vel = b[s].vel + flip<S>(widen(scl(lin, b[s].im)), s);
        b[s].ang = b[s].ang + widen(mulI(b[s].I, ang));
    };
    if (warm)
    {
#pragma unroll
        for (int s = 0; s < S; ++s)
        {
            if (k.an != 0.0f) push(s, scl(n, k.an), scl(jn[s], k.an));
            if (k.a1 != 0.0f) push(s, scl(t1, k.a1), scl(j1[s], k.a1));
            if (k.a2 != 0.0f) push(s, scl(t2, k.a2), scl(j2[s], k.a2));
        }
        return;
    }
    float x[S], y[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
    {
        x[s] = dotf(n, to_f3(b[s].vel));
        y[s] = dotf(jn[s], to_f3(b[s].ang));
    }
    const float jv = jv_sum(x, y);
    const float lambda = -(jv + k.bias) * k.meff;
    float nv = k.an + lambda;
    nv = nv < 0.0f ? 0.0f : nv;
    const float ap = nv - k.an;
    k.an = nv;
    float p[S], q[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
    {
        push(s, scl(n, ap), scl(jn[s], ap));
        const f3 vel = to_f3(b[s].vel), ang = to_f3(b[s].ang);
        x[s] = dotf(t1, vel);
        y[s] = dotf(j1[s], ang);
        p[s] = dotf(t2, vel);
        q[s] = dotf(j2[s], ang);
    }
    const float maxf = mu * k.an;
    const float b1 = jv_sum(x, y), b2 = jv_sum(p, q);
    float n1 = k.a1 - (k.i11 * b1 + k.i12 * b2), n2 = k.a2 - (k.i12 * b1 + k.i22 * b2);
    const float mag = sqrtf(n1 * n1 + n2 * n2);
    if (mag > maxf)
    {
        n1 = n1 * (maxf / mag);
        n2 = n2 * (maxf / mag);
    }
    const float d1 = n1 - k.a1, d2 = n2 - k.a2;
    k.a1 = n1;
    k.a2 = n2;
#pragma unroll
    for (int s = 0; s < S; ++s) push(s, addf(scl(t1, d1), scl(t2, d2)), addf(scl(j1[s], d1), scl(j2[s], d2)));
}
// the Jacobians rebuilt in FP32 from the rounded normal and arms
template <int S>
__device__ __forceinline__ void solve_rows(row_t<float, f3, S> &k, float mu, bool warm, side32 (&b)[S])
{
    const float sign = copysignf(1.0f, k.n.z);
    const float bb = k.n.x * k.n.y * k.a;
    const f3 t1 = f3m(1.0f + sign * k.n.x * k.n.x * k.a, sign * bb, -sign * k.n.x);
    const f3 t2 = f3m(bb, sign + k.n.y * k.n.y * k.a, -k.n.y);
    f3 jn[S], j1[S], j2[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
    {
        jn[s] = flip<S>(fcr(k.r[s], k.n), s);
        j1[s] = flip<S>(fcr(k.r[s], t1), s);
        j2[s] = flip<S>(fcr(k.r[s], t2), s);
    }
    apply_rows32<S>(k, k.n, t1, t2, jn, j1, j2, mu, warm, b);
}
template <int S>
__device__ __forceinline__ void solve_rows(row32_t<S> &k, float mu, bool warm, side32 (&b)[S])
{ apply_rows32<S>(k, k.n, k.t1, k.t2, k.jn, k.j1, k.j2, mu, warm, b); }

__device__ __forceinline__ void put_side(side64 &d, double im, const m3 &I)
{
    d.im = im;
    d.I = I;
}
__device__ __forceinline__ void put_side(side32 &d, double im, const m3 &I)
{
    d.im = static_cast<float>(im);
    for (int k = 0; k < 9; ++k) d.I[k] = static_cast<float>(I.m[k]);
}
__device__ __forceinline__ void put_v(v3 &d, v3 s) { d = s; }
__device__ __forceinline__ void put_v(f3 &d, v3 s) { d = to_f3(s); }
__device__ __forceinline__ double basis_factor(v3 n) { return -1.0 / (copysign(1.0, n.z) + n.z); }
__device__ __forceinline__ float basis_factor(f3 n) { return -1.0f / (copysignf(1.0f, n.z) + n.z); }

__device__ __forceinline__ uint16_t slot_of(const uint32_t *ids, uint32_t n_ids, uint32_t id)
{
    uint32_t lo = 0, hi = n_ids;
    while (lo < hi)
    {
        const uint32_t mid = (lo + hi) >> 1;
        if (ids[mid] < id)
            lo = mid + 1;
        else
            hi = mid;
    }
    return static_cast<uint16_t>(lo);
}

// Chunk k: the islands whose first position lies in [k window, (k + 1) window) of the island
// order (isl null: the whole list is one chunk). With islands of at most `longest`
// manifolds a chunk has at most window + longest - 1, which the launch keeps within CAP and
// within the workgroup's lanes (LANES per manifold). root: the island root at each position.
// In the FP32 solve, islands of more than kIslandMaxColours colours are left to a second launch
// (DEEP), which takes only those and keeps their rows as row32_t (208 registers; the others need
// 171); C_DEEP counts the chunks that have any.
template <bool F32, int LANES, int CAP, bool DEEP>
__global__ void __launch_bounds__(LANES *CAP)
    k_solve_chunks(const uint64_t *keys, const uint32_t *ord, const uint32_t *isl, const uint32_t *root, uint32_t nl,
                   uint32_t window, bodies_dev b, manifolds_dev m, uint32_t *colour, const uint32_t *world_of,
                   const uint32_t *pair_base, uint32_t iters, double dt, double thr, unsigned long long *counters)
{
    constexpr int S = 3 - LANES;
    using T = typename std::conditional<F32, float, double>::type;
    using V = typename std::conditional<F32, f3, v3>::type;
    using side = typename std::conditional<F32, side32, side64>::type;
    static_assert(!DEEP || (F32 && LANES == 2));
    if (DEEP && counters[C_DEEP] == 0) return;
    __shared__ uint32_t ids[2 * CAP];
    __shared__ double lv[2 * CAP][6]; // velocities; before them, the colouring's claims and taken colours
    // both sides' lever arms where one lane has them: with them the rows of four contacts
    // would not fit its registers
    __shared__ double arms[LANES == 1 ? 24 : 1][LANES == 1 ? CAP : 1];
    __shared__ uint32_t lim[3];
    __shared__ uint32_t deep[F32 ? 2 * CAP / 32 : 1]; // a bit per body slot: the root of an island left to DEEP
    const uint32_t tid = threadIdx.x, threads = blockDim.x;
    uint32_t s0 = 0, e0 = nl;
    if (tid < 3) lim[tid] = tid < 2 ? nl : 0u;
    __syncthreads();
    if (isl)
    {
        // Workgroups go to the XCDs in turn: chunk order is cut into eight contiguous parts, one
        // to an XCD, since islands of like size open chunks at a regular distance (64 pyramids:
        // every eighth, all on one XCD, 1.6 ms instead of 0.9).
        const uint32_t chunk = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
        for (uint32_t e = 0; e < 2; ++e) // the first island start from each end of the window
        {
            const uint32_t t = (chunk + e) * window + tid;
            if (t < nl && (t == 0 || isl[t] != isl[t - 1])) atomicMin(&lim[e], t);
        }
        __syncthreads();
        s0 = lim[0];
        e0 = lim[1];
        if (s0 >= e0) return; // no island starts here
    }
    const uint32_t cnt = e0 - s0;
    uint32_t n_ids = 2;
    while (n_ids < 2 * cnt) n_ids <<= 1;
    for (uint32_t i = tid; i < n_ids; i += threads)
    {
        uint32_t id = kNone;
        if (i < 2 * cnt)
        {
            const uint64_t key = keys[ord[s0 + i / 2]];
            const uint32_t x = (i & 1) ? static_cast<uint32_t>(key & 0xFFFFFFFFu) : static_cast<uint32_t>(key >> 32);
            id = x;
        }
        ids[i] = id;
    }
    __syncthreads();
    for (uint32_t size = 2; size <= n_ids; size <<= 1) // bitonic sort; a body's slot is its first position
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1)
        {
            for (uint32_t i = tid; i < n_ids; i += threads)
            {
                const uint32_t j = i ^ stride;
                if (j > i)
                {
                    const uint32_t x = ids[i], y = ids[j];
                    if ((x > y) == ((i & size) == 0))
                    {
                        ids[i] = y;
                        ids[j] = x;
                    }
                }
            }
            __syncthreads();
        }
    // this lane's manifold and sides
    uint32_t i = tid / LANES;
    bool own = i < cnt;
    uint32_t p = 0, id[2] = {0, 0}, mine[S];
    side body[S];
    uint16_t slot[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
    {
        mine[s] = 0;
        slot[s] = 0;
        body[s].stat = true;
    }
    auto take = [&] // manifold i of the chunk
    {
        p = ord[s0 + i];
        const uint64_t key = keys[p];
        id[0] = static_cast<uint32_t>(key >> 32);
        id[1] = static_cast<uint32_t>(key & 0xFFFFFFFFu);
#pragma unroll
        for (int s = 0; s < S; ++s)
        {
            mine[s] = LANES == 1 ? id[s] : (side_b() ? id[1] : id[0]);
            body[s].stat = b.is_static[mine[s]] != 0;
            slot[s] = slot_of(ids, n_ids, mine[s]);
        }
    };
    if (own) take();
    // colouring: the rounds of k_claim and k_assign
    unsigned long long *claim = reinterpret_cast<unsigned long long *>(&lv[0][0]), *used = claim + 2 * CAP;
    for (uint32_t t = tid; t < n_ids; t += threads)
    {
        claim[t] = 0;
        used[t] = 0;
    }
    __syncthreads();
    uint32_t col = kNone;
    const uint32_t lp = own ? local_index(p, id[0], world_of, pair_base) : 0u;
    for (uint32_t round = 0;; ++round)
    {
        const bool open = own && col == kNone;
        const unsigned long long pr = claim_of(lp, round);
        if (open)
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (!body[s].stat) atomicMax(&claim[slot[s]], pr);
        __syncthreads();
        if (open)
        {
            bool ok = true;
            unsigned long long u = 0;
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (!body[s].stat)
                {
                    ok = ok && claim[slot[s]] == pr;
                    u |= used[slot[s]];
                }
            if (LANES == 2)
            {
                const int other = swap32(ok ? 1 : 0);
                ok = ok && other != 0;
                u |= static_cast<unsigned long long>(static_cast<uint32_t>(swap32(static_cast<int>(u)))) |
                     static_cast<unsigned long long>(static_cast<uint32_t>(swap32(static_cast<int>(u >> 32)))) << 32;
            }
            if (ok)
            {
                col = ~u ? static_cast<uint32_t>(__ffsll(static_cast<long long>(~u)) - 1) : 64u + round;
                if (col < 64)
#pragma unroll
                    for (int s = 0; s < S; ++s)
                        if (!body[s].stat) used[slot[s]] |= 1ull << col;
            }
        }
        if (!__syncthreads_or(own && col == kNone)) break;
    }
    if (own)
    {
        atomicMax(&lim[2], col + 1);
        if (tid % LANES == 0) colour[p] = col;
    }
    __syncthreads();
    uint32_t n_colours = lim[2];
    const bool any_deep = F32 && n_colours > kIslandMaxColours;
    if (DEEP && !any_deep) return;
    if (tid == 0) atomicMax(&counters[C_NCOL], static_cast<unsigned long long>(n_colours));
    auto root_bit = [&]
    { return slot_of(ids, n_ids, root[s0 + i]); };
    if (any_deep)
    {
        if (tid < 2 * CAP / 32) deep[tid] = 0;
        __syncthreads();
        if (own && col >= kIslandMaxColours) atomicOr(&deep[root_bit() >> 5], 1u << (root_bit() & 31u));
        if (!DEEP && tid == 0) atomicAdd(&counters[C_DEEP], 1ull);
        __syncthreads();
    }
    if (threads > 64)
    {
        // Manifolds handed out again by colour, so that a colour's are in few wavefronts:
        // spread over all of them, each would run the whole solve for a few lanes, and two
        // wavefronts of a SIMD would share its issue.
        uint32_t *start = reinterpret_cast<uint32_t *>(&lv[0][0]), *perm = start + 64 + 2 * CAP; // colours below 64 + rounds
        for (uint32_t t = tid; t < n_colours; t += threads) start[t] = 0;
        __syncthreads();
        uint32_t rank = 0;
        if (own && tid % LANES == 0) rank = atomicAdd(&start[col], 1u);
        __syncthreads();
        if (tid == 0)
        {
            uint32_t run = 0;
            for (uint32_t t = 0; t < n_colours; ++t)
            {
                const uint32_t k = start[t];
                start[t] = run;
                run += k;
            }
        }
        __syncthreads();
        if (own && tid % LANES == 0) perm[start[col] + rank] = col << 16 | i;
        __syncthreads();
        if (own)
        {
            const uint32_t w = perm[tid / LANES];
            i = w & 0xFFFFu;
            col = w >> 16;
            take();
        }
        __syncthreads();
    }
    if (any_deep)
    {
        if (own) own = ((deep[root_bit() >> 5] >> (root_bit() & 31u)) & 1u) == (DEEP ? 1u : 0u);
        if (!DEEP) n_colours = kIslandMaxColours;
    }
    // velocities
    for (uint32_t t = tid; t < n_ids; t += threads)
    {
        const uint32_t x = ids[t];
        if (x != kNone && (t == 0 || ids[t - 1] != x))
        {
            const v3 v = ld3(b.vel, b.n, x), w = ld3(b.ang, b.n, x);
            lv[t][0] = v.x;
            lv[t][1] = v.y;
            lv[t][2] = v.z;
            lv[t][3] = w.x;
            lv[t][4] = w.y;
            lv[t][5] = w.z;
        }
    }
    // rows: build_contact_jacobian (:874-953) and setup_contacts (:1075-1102)
    typename std::conditional<DEEP, row32_t<S>, row_t<T, V, S>>::type k[4];
    uint32_t valid = 0, sl = 0;
    T mu = 0;
    if (own)
    {
        const int contacts = m.count[p];
        sl = m.slot[p];
        const v3 pa = ld3(b.pos, b.n, id[0]), pb = ld3(b.pos, b.n, id[1]);
        const qt qa = ldq(b.quat, b.n, id[0]), qb = ldq(b.quat, b.n, id[1]);
        const double e = smax(b.restitution[id[0]], b.restitution[id[1]]);
        mu = static_cast<T>(sqrt(b.friction[id[0]] * b.friction[id[1]]));
        double im[S];
        m3 I[S];
        v3 sv[S], sw[S];
#pragma unroll
        for (int s = 0; s < S; ++s)
        {
            im[s] = b.inv_mass[mine[s]];
            I[s] = ld9(b.Iw_inv, b.n, mine[s]);
            sv[s] = ld3(b.vel, b.n, mine[s]);
            sw[s] = ld3(b.ang, b.n, mine[s]);
            put_side(body[s], im[s], I[s]);
        }
        double ima, imb;
        both(im, ima, imb);
#pragma unroll
        for (int c = 0; c < 4; ++c)
        {
            v3 n, ra, rb;
            double pen;
            if (c >= contacts || !contact_frame(m, sl, c, pa, pb, qa, qb, n, ra, rb, pen)) continue;
            valid |= 1u << c;
            v3 r[S], t1, t2, vc[S];
            basis(n, t1, t2);
            double kn[S], k1[S], k2[S], k12[S], vx[S], vy[S], vz[S];
#pragma unroll
            for (int s = 0; s < S; ++s)
            {
                r[s] = LANES == 1 ? (s == 0 ? ra : rb) : (side_b() ? rb : ra);
                const v3 jn = flip<S>(cross(r[s], n), s), j1 = flip<S>(cross(r[s], t1), s), j2 = flip<S>(cross(r[s], t2), s);
                const v3 i2 = mul(I[s], j2);
                kn[s] = dot(jn, mul(I[s], jn));
                k1[s] = dot(j1, mul(I[s], j1));
                k2[s] = dot(j2, i2);
                k12[s] = dot(j1, i2);
                vc[s] = sv[s] + cross(sw[s], r[s]);
                vx[s] = vc[s].x;
                vy[s] = vc[s].y;
                vz[s] = vc[s].z;
            }
            double xa, xb, ya, yb, za, zb;
            both(kn, xa, xb);
            const double meff = 1.0 / (((ima + imb) + xa) + xb);
            both(k1, xa, xb);
            const double meff1 = 1.0 / (((ima + imb) + xa) + xb);
            both(k2, xa, xb);
            const double meff2 = 1.0 / (((ima + imb) + xa) + xb);
            both(k12, xa, xb);
            const double m12 = xa + xb;
            both(vx, xa, xb);
            both(vy, ya, yb);
            both(vz, za, zb);
            const double vrel = dot(mk(xa, ya, za) - mk(xb, yb, zb), n);
            double rbias = 0.0;
            if (vrel < -thr) rbias = e * vrel;
            const double baum = (-0.1 / dt) * smax(0.0, pen - 0.005);
            const double m11 = 1.0 / meff1, m22 = 1.0 / meff2;
            const double det = m11 * m22 - m12 * m12;
            double i11, i12, i22;
            if (det > 0.0)
            {
                i11 = m22 / det;
                i22 = m11 / det;
                i12 = -m12 / det;
            }
            else
            {
                i11 = meff1;
                i22 = meff2;
                i12 = 0.0;
            }
            put_v(k[c].n, n);
            if constexpr (DEEP)
            {
                put_v(k[c].t1, t1);
                put_v(k[c].t2, t2);
            }
#pragma unroll
            for (int s = 0; s < S; ++s)
            {
                if constexpr (DEEP)
                {
                    put_v(k[c].jn[s], flip<S>(cross(r[s], n), s));
                    put_v(k[c].j1[s], flip<S>(cross(r[s], t1), s));
                    put_v(k[c].j2[s], flip<S>(cross(r[s], t2), s));
                }
                else if constexpr (LANES == 1)
                {
                    arms[6 * c + 3 * s][tid] = r[s].x;
                    arms[6 * c + 3 * s + 1][tid] = r[s].y;
                    arms[6 * c + 3 * s + 2][tid] = r[s].z;
                }
                else
                    put_v(k[c].r[s], r[s]);
            }
            if constexpr (!DEEP) k[c].a = basis_factor(k[c].n);
            k[c].meff = static_cast<T>(meff);
            k[c].bias = static_cast<T>(smin(baum, rbias));
            k[c].i11 = static_cast<T>(i11);
            k[c].i12 = static_cast<T>(i12);
            k[c].i22 = static_cast<T>(i22);
            const double *d = m.data + static_cast<size_t>(c * kMF) * m.dcap + sl;
            k[c].an = static_cast<T>(d[10 * static_cast<size_t>(m.dcap)]);
            k[c].a1 = static_cast<T>(d[11 * static_cast<size_t>(m.dcap)]);
            k[c].a2 = static_cast<T>(d[12 * static_cast<size_t>(m.dcap)]);
            __builtin_amdgcn_sched_barrier(0); // one contact at a time: four at once would not fit the registers
        }
    }
    __syncthreads();
    // pass 0 warm starts, then the iterations; a colour's manifolds share no dynamic body
    for (uint32_t pass = 0; pass <= iters; ++pass)
    {
        const bool warm = pass == 0;
        for (uint32_t c = 0; c < n_colours; ++c)
        {
            if (own && col == c)
            {
#pragma unroll
                for (int s = 0; s < S; ++s)
                {
                    const double *l = lv[slot[s]];
                    body[s].vel = mk(l[0], l[1], l[2]);
                    body[s].ang = mk(l[3], l[4], l[5]);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
                {
                    if (valid & (1u << q))
                    {
                        if constexpr (LANES == 1)
                            for (int s = 0; s < S; ++s)
                                put_v(k[q].r[s], mk(arms[6 * q + 3 * s][tid], arms[6 * q + 3 * s + 1][tid],
                                                    arms[6 * q + 3 * s + 2][tid]));
                        solve_rows<S>(k[q], mu, warm, body);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int s = 0; s < S; ++s)
                    if (!body[s].stat)
                    {
                        double *l = lv[slot[s]];
                        l[0] = body[s].vel.x;
                        l[1] = body[s].vel.y;
                        l[2] = body[s].vel.z;
                        l[3] = body[s].ang.x;
                        l[4] = body[s].ang.y;
                        l[5] = body[s].ang.z;
                    }
            }
            __syncthreads();
        }
    }
    if (own && tid % LANES == 0) // :1191-1196
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (valid & (1u << c))
            {
                double *d = m.data + static_cast<size_t>(c * kMF) * m.dcap + sl;
                d[10 * static_cast<size_t>(m.dcap)] = static_cast<double>(k[c].an);
                d[11 * static_cast<size_t>(m.dcap)] = static_cast<double>(k[c].a1);
                d[12 * static_cast<size_t>(m.dcap)] = static_cast<double>(k[c].a2);
            }
    for (uint32_t t = tid; t < n_ids; t += threads)
    {
        const uint32_t x = ids[t];
        if (x != kNone && (t == 0 || ids[t - 1] != x) && !b.is_static[x])
        {
            st3(b.vel, b.n, x, mk(lv[t][0], lv[t][1], lv[t][2]));
            st3(b.ang, b.n, x, mk(lv[t][3], lv[t][4], lv[t][5]));
        }
    }
}
} // namespace

void launch_island_init(uint32_t *par, uint32_t *cnt, uint32_t n, hipStream_t st)
{
    if (n) k_island_init<<<grid(n), kBlock, 0, st>>>(par, cnt, n);
}
void launch_island_roots(const uint64_t *keys, const uint32_t *list, uint32_t n_bound, const bodies_dev &b, uint32_t *par,
                         uint32_t *cnt, uint32_t *root_of, uint32_t *rank_of, unsigned long long *counters, hipStream_t st)
{
    if (n_bound) k_island_roots<<<grid(n_bound), kBlock, 0, st>>>(keys, list, n_bound, b, par, cnt, root_of, rank_of, counters);
}
void launch_island_group(const uint32_t *list, uint32_t nl, const uint32_t *cnt, uint32_t n_bodies, const uint32_t *root_of,
                         const uint32_t *rank_of, uint32_t *base, uint32_t *ord, uint32_t *isl,
                         unsigned long long *counters, hipStream_t st)
{
    if (!nl) return;
    k_island_base<<<grid(n_bodies), kBlock, 0, st>>>(cnt, n_bodies, base, counters);
    k_island_scatter<<<grid(nl), kBlock, 0, st>>>(list, nl, root_of, rank_of, base, ord, isl);
}

void launch_solve_chunks(const uint64_t *keys, const uint32_t *ord, const uint32_t *isl, const uint32_t *root, uint32_t nl,
                         uint32_t longest, const bodies_dev &b, const manifolds_dev &m, uint32_t *colour,
                         const uint32_t *world_of, const uint32_t *pair_base, uint32_t iters, double dt, double thr,
                         bool f32, unsigned long long *counters, hipStream_t st)
{
    if (!nl) return;
    auto go = [&](auto f, auto lanes, auto capacity)
    {
        constexpr bool F = decltype(f)::value;
        constexpr int L = decltype(lanes)::value, CAP = decltype(capacity)::value;
        uint32_t window = nl, most = nl;
        if (isl)
        {
            window = std::min<uint32_t>(CAP + 1 - longest, std::max<uint32_t>(kChunkFill, (nl + 511) / 512));
            most = window + longest - 1;
        }
        const unsigned threads = (std::min<uint32_t>(most, CAP) * L + 63) / 64 * 64;
        const unsigned nb = isl ? ((nl + window - 1) / window + 7) / 8 * 8 : 1u;
        k_solve_chunks<F, L, CAP, false><<<nb, threads, 0, st>>>(keys, ord, isl, root, nl, window, b, m, colour, world_of,
                                                                 pair_base, iters, dt, thr, counters);
        if constexpr (F)
            if (longest > kIslandMaxColours) // a colour takes a manifold of the island's
                k_solve_chunks<F, L, CAP, true><<<nb, threads, 0, st>>>(keys, ord, isl, root, nl, window, b, m, colour,
                                                                        world_of, pair_base, iters, dt, thr, counters);
    };
    using std::integral_constant;
    using std::bool_constant;
    if (f32)
        go(bool_constant<true>{}, integral_constant<int, 2>{}, integral_constant<int, kChunkMax32>{});
    else if (longest <= kChunkTwoLanes && (isl || nl <= kChunkTwoLanes))
        go(bool_constant<false>{}, integral_constant<int, 2>{}, integral_constant<int, kChunkTwoLanes>{});
    else
        go(bool_constant<false>{}, integral_constant<int, 1>{}, integral_constant<int, kChunkMax>{});
}

} // namespace pk
