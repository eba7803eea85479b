// Star form (star.hpp) of the acoustic adjoint's two per-step kernels on an
// exactly uniform mesh of any extents, constant K or a K field (form 0):
//   MODE 1, the forward step that records p' at the sensors and, for the K
//           gradient's recomputation, the divergence S of every cell;
//   MODE 2, the transposed step lam_t -> lam_{t-1}, adding the trace
//           gradients at the sensors;
//   MODE 3, MODE 2 that also adds (lam_p dt) S_t to the K gradient.
//
// At 128^3 FP32 with a K field (us/step): transposed step with the K gradient
// 64 one cell per thread with three velocity fields read back, 22 here;
// recomputed forward step 29 and 16.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"
#include "star_wave.hpp"

namespace cfd {

template <class T, int W, bool PW, bool KF, int MODE>
__global__ void __launch_bounds__(256)
wave_star_aux_k(UniformGeo<T> g, const T* __restrict__ p, const T* __restrict__ u, const T* __restrict__ v,
                const T* __restrict__ w, T* __restrict__ po, T* __restrict__ uo, T* __restrict__ vo,
                T* __restrict__ wo, T K, const T* __restrict__ Kf, T dt, star::Plan pl, star::SensorSet sens,
                star::WaveAux<T> aux) {
    star::Place at;
    if (star::place<W>(pl, at))
        star::wave_cells<T, W, PW, KF, MODE>(g, p, u, v, w, po, uo, vo, wo, K, Kf, dt, pl, at, &sens, &aux);
}

star::SensorSet sensor_set(const cfd_mesh_s* m, const SensorList& l) {
    star::SensorSet s{};
    s.n = l.n;
    while (((m->X - 1) >> s.shift) >= 256) ++s.shift;
    for (int j = 0; j < l.n; ++j) {
        s.x[j] = l.x[j];
        s.y[j] = l.y[j];
        s.z[j] = l.z[j];
        const int b = l.x[j] >> s.shift;
        s.planes[b >> 6] |= uint64_t(1) << (b & 63);
    }
    return s;
}

template <class T>
void launch_wave_star_aux(const cfd_mesh_s* m, int mode, const void* const in[4], void* const out[4], double K,
                          const void* Kf, double dt, const star::SensorSet& sens, const star::WaveAux<T>& aux,
                          hipStream_t s) {
    const UniformGeo<T>& g = [&]() -> const UniformGeo<T>& {
        if constexpr (sizeof(T) == 4) return m->ug32; else return m->ug64;
    }();
    auto run = [&](auto w, auto pw, auto kf, auto md) {
        constexpr int W = decltype(w)::value;
        const star::Plan pl = star::make_plan(g.X, g.Y, g.Z, W);
        wave_star_aux_k<T, W, decltype(pw)::value, decltype(kf)::value, decltype(md)::value>
            <<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(
                g, (const T*)in[0], (const T*)in[1], (const T*)in[2], (const T*)in[3], (T*)out[0], (T*)out[1],
                (T*)out[2], (T*)out[3], T(K), (const T*)Kf, T(dt), pl, sens, aux);
        CFD_HIP(hipGetLastError());
    };
    auto with_mode = [&](auto w, auto pw, auto kf) {
        if (mode == 1) run(w, pw, kf, std::integral_constant<int, 1>{});
        else if (aux.gK) run(w, pw, kf, std::integral_constant<int, 3>{});
        else run(w, pw, kf, std::integral_constant<int, 2>{});
    };
    auto with_geo = [&](auto w) {
        if (g.vol_pow2) {
            if (Kf) with_mode(w, std::true_type{}, std::true_type{});
            else with_mode(w, std::true_type{}, std::false_type{});
        } else {
            if (Kf) with_mode(w, std::false_type{}, std::true_type{});
            else with_mode(w, std::false_type{}, std::false_type{});
        }
    };
    if (star::vector_form<T>(g.Y, g.Z) && !star::narrow<T>(g.X * g.Y * g.Z))
        with_geo(std::integral_constant<int, star::kWidth<T>>{});
    else with_geo(std::integral_constant<int, 1>{});
}

template void launch_wave_star_aux<float>(const cfd_mesh_s*, int, const void* const[4], void* const[4], double,
                                          const void*, double, const star::SensorSet&, const star::WaveAux<float>&,
                                          hipStream_t);
template void launch_wave_star_aux<double>(const cfd_mesh_s*, int, const void* const[4], void* const[4], double,
                                           const void*, double, const star::SensorSet&,
                                           const star::WaveAux<double>&, hipStream_t);

}  // namespace cfd
