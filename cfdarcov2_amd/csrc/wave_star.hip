// Fused acoustic step in star form (variant 0) on an exactly uniform mesh; see
// star.hpp for the form and star_wave.hpp for the step.
//
// Bound by its arithmetic (104 operations per cell against the march's 59) and
// the launch: 48^3 FP32 2.9 us of kernel per step (3.3 to 4.2 launched one by
// one, the host's cost), 128^3 FP32 13.1 (5.1 TB/s), 90x77x123 FP64 12.2 us/step
// against 167 for the 16-row march tile, whose 30 workgroups left most of the
// chip idle.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"
#include "star_wave.hpp"

namespace cfd {

template <class T, int W, bool PW, bool KF>
__global__ void __launch_bounds__(256)
wave_star_k(UniformGeo<T> g, const T* __restrict__ p, const T* __restrict__ u, const T* __restrict__ v,
            const T* __restrict__ w, T* __restrict__ po, T* __restrict__ uo, T* __restrict__ vo, T* __restrict__ wo,
            T K, const T* __restrict__ Kf, T dt, star::Plan pl) {
    star::Place at;
    if (star::place<W>(pl, at))
        star::wave_cells<T, W, PW, KF, 0>(g, p, u, v, w, po, uo, vo, wo, K, Kf, dt, pl, at);
}

template <class T, int W, bool PW>
static void launch_star(const UniformGeo<T>& g, void* const* in, void* const* out, double K, const void* Kf, double dt,
                        hipStream_t s) {
    const star::Plan pl = star::make_plan(g.X, g.Y, g.Z, W);
    auto* kern = Kf ? wave_star_k<T, W, PW, true> : wave_star_k<T, W, PW, false>;
    kern<<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(
        g, (const T*)in[0], (const T*)in[1], (const T*)in[2], (const T*)in[3], (T*)out[0], (T*)out[1], (T*)out[2],
        (T*)out[3], T(K), (const T*)Kf, T(dt), pl);
    CFD_HIP(hipGetLastError());
}

template <class T>
void launch_wave_star(const UniformGeo<T>& g, void* const* in, void* const* out, double K, const void* Kf, double dt,
                      hipStream_t s) {
    constexpr int W = star::kWidth<T>;
    if (star::vector_form<T>(g.Y, g.Z) && !star::narrow<T>(g.X * g.Y * g.Z)) {
        if (g.vol_pow2) launch_star<T, W, true>(g, in, out, K, Kf, dt, s);
        else launch_star<T, W, false>(g, in, out, K, Kf, dt, s);
    } else {
        if (g.vol_pow2) launch_star<T, 1, true>(g, in, out, K, Kf, dt, s);
        else launch_star<T, 1, false>(g, in, out, K, Kf, dt, s);
    }
}

template void launch_wave_star<float>(const UniformGeo<float>&, void* const*, void* const*, double, const void*,
                                      double, hipStream_t);
template void launch_wave_star<double>(const UniformGeo<double>&, void* const*, void* const*, double, const void*,
                                       double, hipStream_t);

}  // namespace cfd
