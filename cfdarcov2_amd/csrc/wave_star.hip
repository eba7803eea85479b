// Fused acoustic step in star form (variant 0) on an exactly uniform mesh; see
// star.hpp for the form.
//   u' = dt*(-Gx(p)) + u, v' = dt*(-Gy(p)) + v, w' = dt*(-Gz(p)) + w
//   p' = dt*(K*((Gx(u') + Gy(v')) + Gz(w'))) + p
// p' needs u' at x+-1, v' at y+-1 and w' at z+-1, which each thread recomputes
// from p (distance 2) and the old velocities; the recomputation is the
// neighbour's own operation sequence, so the result equals the sequential
// (Gauss-Seidel across equations) evaluation bit for bit.  Walls: the normal
// velocity's face value is zero; p is zero-gradient (neighbour = self), which
// clamped rows and planes give by themselves.
//
// Bound by its arithmetic (104 operations per cell against the march's 59) and
// the launch: 48^3 FP32 4.0 us/step, 128^3 FP32 14.5 (4.6 TB/s), 90x77x123
// FP64 12.0 us/step against 167 for the 16-row march tile, whose 30 workgroups
// left most of the chip idle.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"
#include "march.hpp"
#include "star.hpp"

namespace cfd {

template <class T, int W, bool PW, bool KF>
__global__ void __launch_bounds__(256)
wave_star_k(UniformGeo<T> g, const T* __restrict__ p, const T* __restrict__ u, const T* __restrict__ v,
            const T* __restrict__ w, T* __restrict__ po, T* __restrict__ uo, T* __restrict__ vo, T* __restrict__ wo,
            T K, const T* __restrict__ Kf, T dt, star::Plan pl) {
    using star::load;
    using star::load1;
    int x, y, z0;
    if (!star::place<W>(pl, x, y, z0)) return;
    const int X = pl.X, Y = pl.Y, Z = pl.Z;
    const T Ax = g.area[0], Ay = g.area[1], Az = g.area[2];
    const VolDiv<T, PW> Vd{g.vol, g.inv_vol};
    const star::Offsets<W> o = star::offsets<W>(pl, x, y, z0);
    using O = star::Off<W>;
    const int64_t SX = int64_t(Y) * Z;
    const int64_t x0 = o.x0, xm1 = o.xm1, xp1 = o.xp1;
    const int64_t xm2 = x >= 2 ? xm1 - SX : xm1, xp2 = x + 2 < X ? xp1 + SX : xp1;
    const O uz = O(Z);
    const O o0 = o.o0, ym1 = o.ym1, yp1 = o.yp1, zm1 = o.zm1, zp1 = o.zp1;
    const O ym2 = y >= 2 ? ym1 - uz : ym1, yp2 = y + 2 < Y ? yp1 + uz : yp1;
    const O zm2 = z0 >= 2 ? zm1 - 1 : zm1, zp2 = z0 + W + 1 < Z ? zp1 + 1 : zp1;
    const T* const pc = p + x0;

    T P[W], Pxm1[W], Pxm2[W], Pxp1[W], Pxp2[W], Pym1[W], Pym2[W], Pyp1[W], Pyp2[W];
    T U0[W], Um[W], Up[W], V0[W], Vm[W], Vp[W], W0[W], kf[W];
    load<T, W>(pc, o0, P);
    load<T, W>(p + xm1, o0, Pxm1);
    load<T, W>(p + xp1, o0, Pxp1);
    load<T, W>(pc, ym1, Pym1);
    load<T, W>(pc, yp1, Pyp1);
    load<T, W>(u + x0, o0, U0);
    load<T, W>(v + x0, o0, V0);
    load<T, W>(w + x0, o0, W0);
    const T Pz[4] = {load1(pc, zm2), load1(pc, zm1), load1(pc, zp1), load1(pc, zp2)};
    load<T, W>(p + xm2, o0, Pxm2);
    load<T, W>(p + xp2, o0, Pxp2);
    load<T, W>(pc, ym2, Pym2);
    load<T, W>(pc, yp2, Pyp2);
    load<T, W>(u + xm1, o0, Um);
    load<T, W>(u + xp1, o0, Up);
    load<T, W>(v + x0, ym1, Vm);
    load<T, W>(v + x0, yp1, Vp);
    const T Wz[2] = {load1(w + x0, zm1), load1(w + x0, zp1)};
    if constexpr (KF) load<T, W>(Kf + x0, o0, kf);

    // p and w along the row, with the halo: entry j is cell z0 - 2 + j (p), z0 - 1 + j (w)
    T pr[W + 4], wr[W + 2];
    pr[0] = Pz[0]; pr[1] = Pz[1]; pr[W + 2] = Pz[2]; pr[W + 3] = Pz[3];
    wr[0] = Wz[0]; wr[W + 1] = Wz[1];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        pr[i + 2] = P[i];
        wr[i + 1] = W0[i];
    }
    T wn[W + 2];
#pragma unroll
    for (int j = 0; j < W + 2; ++j) wn[j] = mvel(pr[j], pr[j + 1], pr[j + 2], wr[j], Az, Vd, dt);

    T pn[W], un[W], vn[W], wc[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        un[i] = mvel(Pxm1[i], P[i], Pxp1[i], U0[i], Ax, Vd, dt);
        const T ul = mvel(Pxm2[i], Pxm1[i], P[i], Um[i], Ax, Vd, dt);
        const T uh = mvel(P[i], Pxp1[i], Pxp2[i], Up[i], Ax, Vd, dt);
        vn[i] = mvel(Pym1[i], P[i], Pyp1[i], V0[i], Ay, Vd, dt);
        const T vl = mvel(Pym2[i], Pym1[i], P[i], Vm[i], Ay, Vd, dt);
        const T vh = mvel(P[i], Pyp1[i], Pyp2[i], Vp[i], Ay, Vd, dt);
        wc[i] = wn[i + 1];
        const T fx_lo = x == 0 ? T(0) : mlin(un[i], ul);
        const T fx_hi = x == X - 1 ? T(0) : mlin(un[i], uh);
        const T fy_lo = y == 0 ? T(0) : mlin(vn[i], vl);
        const T fy_hi = y == Y - 1 ? T(0) : mlin(vn[i], vh);
        const T fz_lo = (i == 0 && z0 == 0) ? T(0) : mlin(wc[i], wn[i]);
        const T fz_hi = (i == W - 1 && z0 + W == Z) ? T(0) : mlin(wc[i], wn[i + 2]);
        T S = mggp(fx_lo, fx_hi, Ax, Vd);
        S = S + mggp(fy_lo, fy_hi, Ay, Vd);
        S = S + mggp(fz_lo, fz_hi, Az, Vd);
        const T k = KF ? kf[i] : K;
        pn[i] = dt * (k * S) + P[i];
    }
    star::store<T, W>(po + x0, o0, pn);
    star::store<T, W>(uo + x0, o0, un);
    star::store<T, W>(vo + x0, o0, vn);
    star::store<T, W>(wo + x0, o0, wc);
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
    if (star::vector_form<T>(g.Y, g.Z)) {
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
