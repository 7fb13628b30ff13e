// Narrowphase kernels that give each pair a wavefront (pk_wave.hpp): the step's GJK and
// EPA for pair lists too short to fill the chip one thread per pair, EPA reruns, and the
// standalone batch. Results are those of the one-thread kernels in k_narrow.hip.
#include "pk_narrow.hpp"
#include "pk_wave.hpp"

namespace pk
{
namespace
{
constexpr int kWave = 64;
// faces a wavefront holds per lane: 3 (192 faces) for a step's solves, as the one-thread
// kernel's first store; 8 (512) for reruns and for the batch, whose meshes are the caller's
constexpr int kStepSlots = 3, kBatchSlots = 8;

// the shape of this lane's side of pair `key`
template <bool UV>
__device__ __forceinline__ wave::shape pair_side(const bodies_dev &b, const shapes_dev &s, uint64_t key)
{
    const uint32_t id = wave::upper() ? static_cast<uint32_t>(key & 0xFFFFFFFFu) : static_cast<uint32_t>(key >> 32);
    return wave::make_shape(body_shape<UV>(b, s, id));
}

// the contact or the status of hit h (pair p); an overflow is listed with its simplex
template <bool UV, int K>
__device__ __forceinline__ void solve_hit(const wave::shape &w, simplex &x, wave::store<K> &st, uint32_t p, uint32_t h,
                                          const gjk_out_dev &g, uint32_t *ovf_list, unsigned long long *ovf_count)
{
    double out[10];
    const int r = wave::epa_solve<UV, true, K>(w, x, st, out);
    if (__lane_id() == 0)
    {
        if (r == 1) write_info(g.info, g.cap, h, out);
        g.status[p] = static_cast<uint8_t>(r == 1 ? 1 : (r == 0 ? 2 : 3));
        if (r == 3)
        {
            save_simplex(g.simplex, g.cap, h, x);
            ovf_list[atomicAdd(ovf_count, 1ull)] = h;
        }
    }
}

// GJK and EPA of the listed pairs, one wavefront each: bounded by the longest pair's chain
// (about 1.9 us per EPA expansion, 64 at most; 20 us on one thread with its store in private
// memory), not by throughput. kWavePairs tells which lists take it. Entry i of the list is hit i if it
// hits: its contact goes to entry i of the hit arrays, so no slot is reserved per hit; each
// wavefront adds its hits to the counter once. Of a list longer than the arrays or than
// kWavePairs nothing is done: the host sees its count and runs the stage again with larger
// arrays or as separate kernels. (88,500 hull pairs listed a step after 1: GJK and EPA 5.5 ms when
// 256 wavefronts walked them twice, 0.9 so.)
template <bool UV>
__global__ void __launch_bounds__(kWave)
    k_gjk_epa_wave(const uint64_t *keys, const uint32_t *list, int list_slot, bodies_dev b, shapes_dev s, gjk_out_dev g,
                   uint32_t *ovf_list, unsigned long long *counters)
{
    __shared__ wave::store<kStepSlots> st;
    const uint32_t n_list = static_cast<uint32_t>(counters[list_slot]);
    if (n_list > g.cap || n_list > kWavePairs) return;
    uint32_t hits = 0;
    for (uint32_t i = blockIdx.x; i < n_list; i += gridDim.x)
    {
        const uint32_t p = wave::first32(list[i]);
        const wave::shape w = pair_side<UV>(b, s, keys[p]);
        simplex x;
        const bool hit = wave::gjk<UV, true>(w, x);
        if (hit) ++hits;
        if (hit)
        {
            if (__lane_id() == 0)
            {
                g.hit_list[i] = p;
                g.hit_of[p] = i;
            }
            solve_hit<UV, kStepSlots>(w, x, st, p, i, g, ovf_list, &counters[C_EPA_OVF]);
        }
        else if (__lane_id() == 0)
            g.status[p] = 0;
    }
    if (__lane_id() == 0 && hits) atomicAdd(&counters[C_HITS], static_cast<unsigned long long>(hits));
}

// EPA of hits in_list[0..n) (0..n-1 when null), one wavefront each: 0.12 ms on 8,400 hull hits
// (one thread each 0.45), 0.44 on 56,000 mixed hits (0.96), 0.13 on 17,880 box hits (0.36) and
// 1.35 on 143,000 hull hits (2.07). Four wavefronts a SIMD without UV spheres, though 13
// registers then spill (143,000 hull hits 1.56 -> 1.35 ms); with them too many do (56,000 mixed
// hits 0.44 -> 0.49).
template <bool UV, int K>
__global__ void __launch_bounds__(kWave, K == kStepSlots && !UV ? 4 : 1)
    k_epa_wave(const uint64_t *keys, const uint32_t *in_list, uint32_t first, uint32_t n, bodies_dev b, shapes_dev s,
               gjk_out_dev g, uint32_t *ovf_list, unsigned long long *ovf_count)
{
    __shared__ wave::store<K> st;
    const uint32_t i = first + blockIdx.x;
    if (i >= n) return;
    const uint32_t h = in_list ? wave::first32(in_list[i]) : i;
    const uint32_t p = wave::first32(g.hit_list[h]);
    const wave::shape w = pair_side<UV>(b, s, keys[p]);
    simplex x;
    x.s1 = x.s2 = x.s3 = spt{mk(0.0, 0.0, 0.0), 0u, 0u};
    load_simplex(g.simplex, g.cap, h, x);
    x.n = static_cast<int>(wave::first32(static_cast<uint32_t>(x.n)));
    solve_hit<UV, K>(w, x, st, p, h, g, ovf_list, ovf_count);
}

// ---- standalone batch ----
// words as k_batch_dev_big (k_narrow.hip) reads them. The kernel is bound by the issue of its
// dependent FP64 chains. One thread per pair took 7.9 ms on 65,536 pairs of boxes, hulls and
// 482-vertex spheres (each lane scanning 2 x 482 vertices per support, the wavefront waiting
// for its longest lane) and sent every solve past 192 faces to k_batch_dev_big, 29.7 ms on two
// threads; a wavefront per pair with 512 faces takes 1.5 ms in all.
template <bool UV>
__global__ void __launch_bounds__(kWave)
    k_batch_wave(shape_pair_dev sp, uint32_t n, uint32_t n_verts, double *out, int32_t *hit, uint32_t *words,
                 uint32_t *ovf_list, uint32_t first)
{
    __shared__ wave::store<kBatchSlots> st;
    const uint32_t i = blockIdx.x;
    if (i >= n) return;
    const bool up = wave::upper(), lead = __lane_id() == 0;
    const int k = up ? sp.kind_b[i] : sp.kind_a[i];
    const uint32_t vb = up ? sp.vbeg_b[i] : sp.vbeg_a[i], ve = up ? sp.vend_b[i] : sp.vend_a[i];
    if (__ballot(k < 0 || k > 2 || (k == 2 && (ve <= vb || ve > n_verts))))
    {
        if (lead)
        {
            hit[i] = -1;
            atomicAdd(&words[0], 1u);
        }
        return;
    }
    const wave::shape w =
        wave::make_shape(up ? pair_shape(sp.kind_b, sp.prm_b, sp.vbeg_b, sp.vend_b, sp.verts, UV ? sp.uv_b : nullptr, i)
                            : pair_shape(sp.kind_a, sp.prm_a, sp.vbeg_a, sp.vend_a, sp.verts, UV ? sp.uv_a : nullptr, i));
    simplex x;
    if (!wave::gjk<UV, false>(w, x))
    {
        if (lead) hit[i] = 0;
        return;
    }
    double o[10];
    const int r = wave::epa_solve<UV, false, kBatchSlots>(w, x, st, o);
    if (!lead) return;
    if (r == 1)
        for (int c = 0; c < 10; ++c) out[10 * static_cast<size_t>(i) + c] = o[c];
    hit[i] = r == 1 ? 1 : (r == 0 ? 2 : 3);
    if (r == 3) ovf_list[atomicAdd(&words[1], 1u)] = first + i;
}

// one workgroup of a wavefront per item, at most per_launch of them in a launch
template <class Launch> void in_parts(uint32_t n, uint32_t per_launch, Launch &&launch)
{
    for (uint64_t first = 0; first < n; first += per_launch)
        launch(static_cast<uint32_t>(first), static_cast<uint32_t>(std::min<uint64_t>(per_launch, n - first)));
}
} // namespace

void launch_gjk_epa_wave(const uint64_t *keys, const uint32_t *list, int list_slot, uint32_t waves, const bodies_dev &b,
                         const shapes_dev &s, bool uv, const gjk_out_dev &g, uint32_t *ovf_list,
                         unsigned long long *counters, hipStream_t st)
{
    const uint32_t gr = std::max<uint32_t>(waves, 256u);
    if (uv)
        k_gjk_epa_wave<true><<<gr, kWave, 0, st>>>(keys, list, list_slot, b, s, g, ovf_list, counters);
    else
        k_gjk_epa_wave<false><<<gr, kWave, 0, st>>>(keys, list, list_slot, b, s, g, ovf_list, counters);
}

void launch_epa_wave(const uint64_t *keys, const uint32_t *in_list, uint32_t n, const bodies_dev &b, const shapes_dev &s,
                     bool uv, bool rerun, const gjk_out_dev &g, uint32_t *ovf_list, unsigned long long *ovf_count,
                     uint32_t per_launch, hipStream_t st)
{
    auto go = [&](auto slots)
    {
        constexpr int K = decltype(slots)::value;
        in_parts(n, per_launch,
                 [&](uint32_t first, uint32_t wgs)
                 {
                     if (uv)
                         k_epa_wave<true, K><<<wgs, kWave, 0, st>>>(keys, in_list, first, n, b, s, g, ovf_list, ovf_count);
                     else
                         k_epa_wave<false, K><<<wgs, kWave, 0, st>>>(keys, in_list, first, n, b, s, g, ovf_list, ovf_count);
                 });
    };
    if (rerun)
        go(std::integral_constant<int, kBatchSlots>{});
    else
        go(std::integral_constant<int, kStepSlots>{});
}

void launch_batch_wave(const shape_pair_dev &sp, uint32_t n, uint32_t n_verts, double *out, int32_t *hit, uint32_t *words,
                       uint32_t *ovf_list, uint32_t per_launch, hipStream_t st)
{
    in_parts(n, per_launch,
             [&](uint32_t first, uint32_t wgs)
             {
                 shape_pair_dev part = sp; // entries first, first + 1, ...
                 for (const int32_t **p : {&part.kind_a, &part.kind_b}) *p += first;
                 for (const uint32_t **p : {&part.vbeg_a, &part.vend_a, &part.vbeg_b, &part.vend_b}) *p += first;
                 for (const double **p : {&part.prm_a, &part.prm_b}) *p += 10 * static_cast<size_t>(first);
                 if (sp.uv_a)
                 {
                     part.uv_a += first;
                     part.uv_b += first;
                 }
                 auto kernel = sp.uv_a ? k_batch_wave<true> : k_batch_wave<false>;
                 kernel<<<wgs, kWave, 0, st>>>(part, wgs, n_verts, out + 10 * static_cast<size_t>(first), hit + first, words,
                                               ovf_list, first);
             });
}

} // namespace pk
