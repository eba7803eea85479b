// The fused acoustic step of a thread's W cells in star form (star.hpp), and
// its trace-recording and transposed forms; used by wave_star.hip and
// adj_star.hip.
//   u' = dt*(-Gx(p)) + u, v' = dt*(-Gy(p)) + v, w' = dt*(-Gz(p)) + w
//   p' = dt*(K*((Gx(u') + Gy(v')) + Gz(w'))) + p
// p' needs u' at x+-1, v' at y+-1 and w' at z+-1, which each thread recomputes
// from p (distance 2) and the old velocities; the recomputation is the
// neighbour's own operation sequence, so the result equals the sequential
// (Gauss-Seidel across equations) evaluation bit for bit.  Walls: the normal
// velocity's face value is zero; p is zero-gradient (neighbour = self), which
// clamped rows and planes give by themselves.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"
#include "march.hpp"
#include "star.hpp"

namespace cfd {

namespace star {

// Sensors as a kernel argument: cell coordinates and, per bucket of x-planes
// (x >> shift, at most 256 buckets), whether any sensor lies there, so a
// workgroup without sensors learns it from one scalar bit.
struct SensorSet {
    int n, shift;
    uint64_t planes[4];
    int x[kMaxSensors], y[kMaxSensors], z[kMaxSensors];
};

// Extra inputs and outputs of the trace-recording step (MODE 1) and of the
// transposed step (MODE 2; MODE 3 with the K gradient).
template <class T> struct WaveAux {
    T* trace;       // MODE 1: p' at the sensors (nullable)
    T* s_out;       // MODE 1: the velocity divergence S of every cell (nullable)
    int state_out;  // MODE 1: 0 = the state is not stored (a step whose S alone is wanted)
    const T* src;   // MODE 2/3: added to nu_p at the sensors (nullable)
    const T* s_in;  // MODE 3: the forward step's S
    T* gK;          // MODE 3: gK += (lam_p dt) S
};

// MODE 0: the step.  MODE 1: the step, recording p' at the sensors and S.
// MODE 2: the transposed step of the adjoint; with (p, u, v, w) read as
// (lam_p, lam_u, lam_v, lam_w) and q = (dt K) lam_p,
//   mu_a = lam_a - G_a(q),  nu_p = dt (Dx mu_x + Dy mu_y + Dz mu_z) + lam_p.
template <class T, int W, bool PW, bool KF, int MODE>
__device__ __forceinline__ void wave_cells(const UniformGeo<T>& g, const T* __restrict__ p, const T* __restrict__ u,
                                  const T* __restrict__ v, const T* __restrict__ w, T* __restrict__ po,
                                  T* __restrict__ uo, T* __restrict__ vo, T* __restrict__ wo, T K,
                                  const T* __restrict__ Kf, T dt, const Plan& pl, const Place& at, const SensorSet* sens = nullptr,
                                  const WaveAux<T>* aux = nullptr) {
    constexpr bool ADJ = MODE >= 2;
    const int x = at.x, y = at.y, z0 = at.z0;
    const int X = pl.X, Y = pl.Y, Z = pl.Z;
    const T Ax = g.area[0], Ay = g.area[1], Az = g.area[2];
    const VolDiv<T, PW> Vd{g.vol, g.inv_vol};
    const Offsets<W> o = offsets<W>(pl, at);
    using O = Off<W>;
    const int64_t SX = int64_t(Y) * Z;
    const int64_t x0 = o.x0, xm1 = o.xm1, xp1 = o.xp1;
    const int64_t xm2 = x >= 2 ? xm1 - SX : xm1, xp2 = x + 2 < X ? xp1 + SX : xp1;
    const O uz = O(Z);
    const O o0 = o.o0, ym1 = o.ym1, yp1 = o.yp1, zm1 = o.zm1, zp1 = o.zp1;
    const O ym2 = y >= 2 ? ym1 - uz : ym1, yp2 = y + 2 < Y ? yp1 + uz : yp1;
    const O zm2 = z0 >= 2 ? zm1 - 1 : zm1, zp2 = z0 + W + 1 < Z ? zp1 + 1 : zp1;
    const T* const pc = p + x0;

    // the pressure slot's values: p, or q = (dt K) lam_p of the transposed step
    const T dK = dt * K;
    auto get = [&](int64_t plane, O off, T(&r)[W]) {
        load<T, W>(p + plane, off, r);
        if constexpr (ADJ && KF) {
            T k[W];
            load<T, W>(Kf + plane, off, k);
#pragma unroll
            for (int i = 0; i < W; ++i) r[i] = (dt * k[i]) * r[i];
        } else if constexpr (ADJ) {
#pragma unroll
            for (int i = 0; i < W; ++i) r[i] = dK * r[i];
        }
    };
    auto get1 = [&](O off) -> T {
        const T r = load1(pc, off);
        if constexpr (ADJ && KF) return (dt * load1(Kf + x0, off)) * r;
        else if constexpr (ADJ) return dK * r;
        else return r;
    };
    auto vel = [&](T lo, T c, T hi, T q, T A) -> T {
        if constexpr (ADJ) return q - mggp(mlin(c, lo), mlin(c, hi), A, Vd);
        else return mvel(lo, c, hi, q, A, Vd, dt);
    };

    T P[W], Pxm1[W], Pxm2[W], Pxp1[W], Pxp2[W], Pym1[W], Pym2[W], Pyp1[W], Pyp2[W];
    T U0[W], Um[W], Up[W], V0[W], Vm[W], Vp[W], W0[W], kf[W], R[W], St[W], gk[W];
    get(x0, o0, P);
    get(xm1, o0, Pxm1);
    get(xp1, o0, Pxp1);
    get(x0, ym1, Pym1);
    get(x0, yp1, Pyp1);
    load<T, W>(u + x0, o0, U0);
    load<T, W>(v + x0, o0, V0);
    load<T, W>(w + x0, o0, W0);
    const T Pz[4] = {get1(zm2), get1(zm1), get1(zp1), get1(zp2)};
    get(xm2, o0, Pxm2);
    get(xp2, o0, Pxp2);
    get(x0, ym2, Pym2);
    get(x0, yp2, Pyp2);
    load<T, W>(u + xm1, o0, Um);
    load<T, W>(u + xp1, o0, Up);
    load<T, W>(v + x0, ym1, Vm);
    load<T, W>(v + x0, yp1, Vp);
    const T Wz[2] = {load1(w + x0, zm1), load1(w + x0, zp1)};
    if constexpr (KF && !ADJ) load<T, W>(Kf + x0, o0, kf);
    if constexpr (ADJ) load<T, W>(pc, o0, R);  // lam_p as it is
    if constexpr (MODE == 3) {
        load<T, W>(aux->s_in + x0, o0, St);
        load<T, W>(aux->gK + x0, o0, gk);
    }

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
    for (int j = 0; j < W + 2; ++j) wn[j] = vel(pr[j], pr[j + 1], pr[j + 2], wr[j], Az);

    T pn[W], un[W], vn[W], wc[W], Sv[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        un[i] = vel(Pxm1[i], P[i], Pxp1[i], U0[i], Ax);
        const T ul = vel(Pxm2[i], Pxm1[i], P[i], Um[i], Ax);
        const T uh = vel(P[i], Pxp1[i], Pxp2[i], Up[i], Ax);
        vn[i] = vel(Pym1[i], P[i], Pyp1[i], V0[i], Ay);
        const T vl = vel(Pym2[i], Pym1[i], P[i], Vm[i], Ay);
        const T vh = vel(P[i], Pyp1[i], Pyp2[i], Vp[i], Ay);
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
        Sv[i] = S;
        if constexpr (ADJ) {
            pn[i] = dt * S + R[i];
        } else {
            const T k = KF ? kf[i] : K;
            pn[i] = dt * (k * S) + P[i];
        }
    }
    if constexpr (MODE != 0) {
        const int bucket = x >> sens->shift;
        if ((ADJ ? aux->src != nullptr : aux->trace != nullptr) && ((sens->planes[bucket >> 6] >> (bucket & 63)) & 1)) {
            for (int j = 0; j < sens->n; ++j) {
                if (sens->x[j] != x) continue;
                if (y != sens->y[j]) continue;
                const int zz = sens->z[j];
#pragma unroll
                for (int i = 0; i < W; ++i)
                    if (zz == z0 + i) {
                        if constexpr (ADJ) pn[i] = pn[i] + aux->src[j];
                        else aux->trace[j] = pn[i];
                    }
            }
        }
    }
    if constexpr (MODE == 3) {
#pragma unroll
        for (int i = 0; i < W; ++i) gk[i] = gk[i] + (R[i] * dt) * St[i];
    }
    if constexpr (MODE == 1) {
        if (aux->s_out) store<T, W>(aux->s_out + x0, o0, Sv);
        if (!aux->state_out) return;
    }
    store<T, W>(po + x0, o0, pn);
    store<T, W>(uo + x0, o0, un);
    store<T, W>(vo + x0, o0, vn);
    store<T, W>(wo + x0, o0, wc);
    if constexpr (MODE == 3) {
        // gK is updated in place, so the cells a row's last unit shares with
        // the unit before are left to that one
        if (at.skip == 0) {
            store<T, W>(aux->gK + x0, o0, gk);
        } else {
#pragma unroll
            for (int i = 1; i < W; ++i)
                if (i >= at.skip) aux->gK[x0 + int64_t(o0) + i] = gk[i];
        }
    }
}

}  // namespace star

}  // namespace cfd
