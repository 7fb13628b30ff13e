// The standalone narrowphase (pkg_gjk_epa_batch, pkg_gjk_epa_batch_device) with a wavefront
// per pair (pk_wave.hpp).
#include "pk_narrow.hpp"
#include "pk_wave.hpp"

namespace pk
{
namespace
{
constexpr int kWave = 64;
constexpr int kBatchSlots = 8; // faces per lane: 512, enough for nearly every 64-expansion solve

// words as k_batch_dev_big (k_narrow.hip) reads them. The kernel is bound by the issue of its
// dependent FP64 chains. One thread per pair took 7.9 ms on 65,536 pairs of boxes, hulls and
// 482-vertex spheres (each lane scanning 2 x 482 vertices per support, the wavefront waiting
// for its longest lane) and sent every solve past 192 faces to k_batch_dev_big, 29.7 ms on two
// threads; a wavefront per pair with 512 faces takes 1.5 ms in all.
template <bool UV>
__global__ void __launch_bounds__(kWave)
    k_batch_wave(shape_pair_dev sp, uint32_t n, uint32_t n_verts, double *out, int32_t *hit, uint32_t *words,
                 uint32_t *ovf_list)
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
    if (r == 3) ovf_list[atomicAdd(&words[1], 1u)] = i;
}
} // namespace

void launch_batch_wave(const shape_pair_dev &sp, uint32_t n, uint32_t n_verts, double *out, int32_t *hit, uint32_t *words,
                       uint32_t *ovf_list, hipStream_t st)
{
    if (!n) return;
    if (sp.uv_a)
        k_batch_wave<true><<<n, kWave, 0, st>>>(sp, n, n_verts, out, hit, words, ovf_list);
    else
        k_batch_wave<false><<<n, kWave, 0, st>>>(sp, n, n_verts, out, hit, words, ovf_list);
}

} // namespace pk
