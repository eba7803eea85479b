// Gradient, Laplacian and heat step in star form (star.hpp) on exactly uniform
// meshes and axis-aligned lattices, the stabilisation on the former and the
// acoustic step on the latter.
//
// GEO 0 / 1: uniform, volume a power of two or not; the constants are kernel
// arguments, so only the fields cross memory.  GEO 2: lattice (LatticeGeo);
// the volume is read per cell, the widths and alpha_d per layer, where the
// general form reads the normal, area and alpha_d of each of a cell's six faces.
//
// Measured against one cell per thread with 64-bit indices (GEO 0/1) and the
// general form (GEO 2): heat step 64^3 FP64 2.8 us against 3.5 (the launch and
// one memory round trip), decimal 100^3 FP64 6.8 against 38.4 us (the general
// form moves 144 bytes per cell, this one 24); gradient, Laplacian and
// stabilisation of 200^3 FP32 together 68 against 151 us; acoustic step on a
// decimal 120x100x80 FP32 lattice 14.3 against 49.0 us.
//
// The arithmetic is the reference's (src/fvm3d.cpp:825-829,902-906 and
// :690-692 with include/grad_utils.hpp:23-125) in its order.  Clamped
// neighbours give the walls' neighbour = self rule by themselves: the
// Laplacian's difference is then an exact zero.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"
#include "march.hpp"
#include "star.hpp"

namespace cfd {

namespace {

template <class T, int GEO> struct GeoArg { using type = UniformGeo<T>; };
template <class T> struct GeoArg<T, 2> { using type = LatticeGeo<T>; };

// whether the lower / upper face of cell i along axis a is on the wall
struct AtWall {
    bool lo[3], hi[3];
};
__device__ inline AtWall at_wall(const star::Plan& pl, const star::Place& q, int i) {
    return {{q.x == 0, q.y == 0, q.z0 + i == 0}, {q.x == pl.X - 1, q.y == pl.Y - 1, q.z0 + i == pl.Z - 1}};
}

// interpolated face values of cell i, zero on the walls normal to wall_axis
template <class T, int W>
__device__ inline star::Faces<T> lin_faces(const star::Star7<T, W>& s, const AtWall& w, int wall_axis, int i) {
    star::Faces<T> f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        f.lo[a] = mlin(s.c(i), star::face_nb(s, a, false, i));
        f.hi[a] = mlin(s.c(i), star::face_nb(s, a, true, i));
        if (wall_axis == a) {
            if (w.lo[a]) f.lo[a] = T(0);
            if (w.hi[a]) f.hi[a] = T(0);
        }
    }
    return f;
}

// Laplacian of cell i over the selected axes, from 0 in the order x, y, z
template <class T, int W, int GEO>
__device__ inline T lapl_cell(const typename GeoArg<T, GEO>::type& g, const star::LatticeCells<T, W>& lc,
                              const star::Star7<T, W>& s, int mask, int i) {
    if constexpr (GEO != 2) {
        return star::lapl_uniform<T, W, GEO == 0>(g, s, mask, i);
    } else {
        const T pc = s.c(i);
        T res = T(0);
        star::Faces<T> f;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            f.lo[a] = (-pc + star::face_nb(s, a, false, i)) * (a == 0 ? lc.ax[0] : a == 1 ? lc.ay[0] : lc.az[i]);
            f.hi[a] = (-pc + star::face_nb(s, a, true, i)) * (a == 0 ? lc.ax[1] : a == 1 ? lc.ay[1] : lc.az[i + 1]);
        }
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if (mask & (1 << a)) res = res + star::lattice_gauss<T, W, false>(lc, f, a, i);
        return res;
    }
}

}  // namespace

template <class T, int W, int GEO>
__global__ void __launch_bounds__(256) grad_star_k(typename GeoArg<T, GEO>::type g, const T* __restrict__ phi,
                                                   T* __restrict__ out, int mask, int wall_axis, star::Plan pl) {
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const star::Star7<T, W> s = star::load7<T, W>(phi, o);
    star::LatticeCells<T, W> lc;
    if constexpr (GEO == 2) lc = star::load_lattice<T, W, false>(g, o, q);
    T r[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const star::Faces<T> f = lin_faces(s, at_wall(pl, q, i), wall_axis, i);
        T res = T(0);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (!(mask & (1 << a))) continue;
            if constexpr (GEO == 2) {
                res = res + star::lattice_gauss<T, W, true>(lc, f, a, i);
            } else {
                const VolDiv<T, GEO == 0> Vd{g.vol, g.inv_vol};
                res = res + mggp(f.lo[a], f.hi[a], g.area[a], Vd);
            }
        }
        r[i] = res;
    }
    star::store<T, W>(out + o.x0, o.o0, r);
}

template <class T, int W, int GEO>
__global__ void __launch_bounds__(256) lapl_star_k(typename GeoArg<T, GEO>::type g, const T* __restrict__ phi,
                                                   T* __restrict__ out, int mask, star::Plan pl) {
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const star::Star7<T, W> s = star::load7<T, W>(phi, o);
    star::LatticeCells<T, W> lc;
    if constexpr (GEO == 2) lc = star::load_lattice<T, W, true>(g, o, q);
    T r[W];
#pragma unroll
    for (int i = 0; i < W; ++i) r[i] = lapl_cell<T, W, GEO>(g, lc, s, mask, i);
    star::store<T, W>(out + o.x0, o.o0, r);
}

// T' = dt * (alpha * lapl(T)) + T (DtVar::extract order, src/fvm3d.cpp:690-692)
template <class T, int W, int GEO, bool AF>
__global__ void __launch_bounds__(256) heat_star_k(typename GeoArg<T, GEO>::type g, const T* __restrict__ Tin,
                                                   T* __restrict__ Tout, T alpha, const T* __restrict__ alpha_f, T dt,
                                                   star::Plan pl) {
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const star::Star7<T, W> s = star::load7<T, W>(Tin, o);
    star::LatticeCells<T, W> lc;
    if constexpr (GEO == 2) lc = star::load_lattice<T, W, true>(g, o, q);
    T af[W];
    if constexpr (AF) star::load<T, W>(alpha_f + o.x0, o.o0, af);
    T r[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const T k = AF ? af[i] : alpha;
        r[i] = dt * (k * lapl_cell<T, W, GEO>(g, lc, s, 7, i)) + s.c(i);
    }
    star::store<T, W>(Tout + o.x0, o.o0, r);
}

// StabVar on a uniform mesh (src/fvm3d.cpp:909-936) in one pass.  Per selected
// axis: the Green-Gauss gradient of the cell and of its two neighbours on the
// axis from phi at up to two cells away, the upwind face values
// phi + (len * g) * n_out of the cell against the neighbour's at the same face
// (at a wall the cell's own at its opposite face, i.e. the neighbour is the
// cell itself), 0.5 * jump, Gauss sum.  Along z the gradients of W + 2 cells
// serve all W cells.  Bound by its arithmetic, 108 operations per cell: 200^3
// FP32 23 us against 48 for a march along x with the plane in LDS.
template <class T, int W, bool PW>
__global__ void __launch_bounds__(256) stab_star_k(UniformGeo<T> g, const T* __restrict__ phi, T* __restrict__ out,
                                                   int mask, star::Plan pl) {
    using star::load;
    using star::load1;
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    using O = star::Off<W>;
    const VolDiv<T, PW> Vd{g.vol, g.inv_vol};
    const O uz = O(pl.Z);
    const int64_t SX = int64_t(pl.Y) * pl.Z;
    const T* const f0 = phi + o.x0;
    T c[W], r[W];
    load<T, W>(f0, o.o0, c);
#pragma unroll
    for (int i = 0; i < W; ++i) r[i] = T(0);
    auto grad = [&](T lo, T pc, T hi, int a) { return mggp(mlin(pc, lo), mlin(pc, hi), g.area[a], Vd); };
    // the axis' term from the cell's, the lower and the upper neighbour's value and gradient
    auto term = [&](int a, T pc, T gc, T pl_, T gl, T ph, T gh) {
        const T L = g.len[a];
        const T own_lo = pc + (L * gc) * T(-1);
        const T col_lo = pl_ + (L * gl) * T(1);
        const T own_hi = pc + (L * gc) * T(1);
        const T col_hi = ph + (L * gh) * T(-1);
        const T f_lo = T(0.5) * (own_lo - col_lo);
        const T f_hi = T(0.5) * (own_hi - col_hi);
        return Vd(f_lo * g.area[a] + f_hi * g.area[a]);
    };
    // x and y: values at -2, -1, 1, 2 along the axis (clamped)
    auto axis = [&](int a, const T(&m2)[W], const T(&m1)[W], const T(&p1)[W], const T(&p2)[W], bool wl, bool wh) {
#pragma unroll
        for (int i = 0; i < W; ++i) {
            const T gc = grad(m1[i], c[i], p1[i], a);
            const T gl = wl ? gc : grad(m2[i], m1[i], c[i], a);
            const T gh = wh ? gc : grad(c[i], p1[i], p2[i], a);
            r[i] = r[i] + term(a, c[i], gc, m1[i], gl, p1[i], gh);
        }
    };
    // every load is issued before any axis is summed
    T xm2[W], xm1[W], xp1[W], xp2[W], ym2[W], ym1[W], yp1[W], yp2[W];
    load<T, W>(phi + o.xm1, o.o0, xm1);
    load<T, W>(phi + o.xp1, o.o0, xp1);
    load<T, W>(f0, o.ym1, ym1);
    load<T, W>(f0, o.yp1, yp1);
    load<T, W>(phi + (q.x >= 2 ? o.xm1 - SX : o.xm1), o.o0, xm2);
    load<T, W>(phi + (q.x + 2 < pl.X ? o.xp1 + SX : o.xp1), o.o0, xp2);
    load<T, W>(f0, q.y >= 2 ? o.ym1 - uz : o.ym1, ym2);
    load<T, W>(f0, q.y + 2 < pl.Y ? o.yp1 + uz : o.yp1, yp2);
    T pr[W + 4], gr[W + 2];  // entry j is cell z0 - 2 + j (pr), z0 - 1 + j (gr)
    pr[0] = load1(f0, q.z0 >= 2 ? o.zm1 - 1 : o.zm1);
    pr[1] = load1(f0, o.zm1);
    pr[W + 2] = load1(f0, o.zp1);
    pr[W + 3] = load1(f0, q.z0 + W + 1 < pl.Z ? o.zp1 + 1 : o.zp1);
    if (mask & 1) axis(0, xm2, xm1, xp1, xp2, q.x == 0, q.x == pl.X - 1);
    if (mask & 2) axis(1, ym2, ym1, yp1, yp2, q.y == 0, q.y == pl.Y - 1);
    if (mask & 4) {
#pragma unroll
        for (int i = 0; i < W; ++i) pr[i + 2] = c[i];
#pragma unroll
        for (int j = 0; j < W + 2; ++j) gr[j] = grad(pr[j], pr[j + 1], pr[j + 2], 2);
#pragma unroll
        for (int i = 0; i < W; ++i) {
            const T gl = (i == 0 && q.z0 == 0) ? gr[i + 1] : gr[i];
            const T gh = (i == W - 1 && q.z0 + W == pl.Z) ? gr[i + 1] : gr[i + 2];
            r[i] = r[i] + term(2, c[i], gr[i + 1], pr[i + 1], gl, pr[i + 3], gh);
        }
    }
    star::store<T, W>(out + o.x0, o.o0, r);
}

// Acoustic step on a lattice, as the general form runs it: the three velocity
// equations from p, then the pressure equation from the new velocities.  (One
// pass would recompute the neighbours' velocities from p; the general form's
// gradients turn NaN wherever any face value of the cell is not finite, which
// a neighbour's recomputation could not see without loading all its faces.)
template <class T, int W>
__global__ void __launch_bounds__(256) wave_vel_lattice_k(LatticeGeo<T> g, const T* __restrict__ p,
                                                          const T* __restrict__ u, const T* __restrict__ v,
                                                          const T* __restrict__ w, T* __restrict__ uo,
                                                          T* __restrict__ vo, T* __restrict__ wo, T dt,
                                                          star::Plan pl) {
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const star::Star7<T, W> s = star::load7<T, W>(p, o);
    const star::LatticeCells<T, W> lc = star::load_lattice<T, W, false>(g, o, q);
    T n[3][W];
    star::load<T, W>(u + o.x0, o.o0, n[0]);
    star::load<T, W>(v + o.x0, o.o0, n[1]);
    star::load<T, W>(w + o.x0, o.o0, n[2]);
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const star::Faces<T> f = lin_faces(s, AtWall{}, -1, i);
#pragma unroll
        for (int a = 0; a < 3; ++a) n[a][i] = dt * (-star::lattice_gauss<T, W, true>(lc, f, a, i)) + n[a][i];
    }
    star::store<T, W>(uo + o.x0, o.o0, n[0]);
    star::store<T, W>(vo + o.x0, o.o0, n[1]);
    star::store<T, W>(wo + o.x0, o.o0, n[2]);
}

template <class T, int W, bool KF>
__global__ void __launch_bounds__(256) wave_p_lattice_k(LatticeGeo<T> g, const T* __restrict__ u,
                                                        const T* __restrict__ v, const T* __restrict__ w,
                                                        const T* __restrict__ p, T* __restrict__ po, T K,
                                                        const T* __restrict__ Kf, T dt, star::Plan pl) {
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const star::Star7<T, W> s[3] = {star::load7<T, W>(u, o), star::load7<T, W>(v, o), star::load7<T, W>(w, o)};
    const star::LatticeCells<T, W> lc = star::load_lattice<T, W, false>(g, o, q);
    T pc[W], kf[W];
    star::load<T, W>(p + o.x0, o.o0, pc);
    if constexpr (KF) star::load<T, W>(Kf + o.x0, o.o0, kf);
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const AtWall wl = at_wall(pl, q, i);
        T S = T(0);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const T G = star::lattice_gauss<T, W, true>(lc, lin_faces(s[a], wl, a, i), a, i);
            S = a == 0 ? G : S + G;
        }
        const T k = KF ? kf[i] : K;
        pc[i] = dt * (k * S) + pc[i];
    }
    star::store<T, W>(po + o.x0, o.o0, pc);
}

namespace {

template <class T> const UniformGeo<T>& ug(const cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->ug32; else return m->ug64;
}
template <class T> const LatticeGeo<T>& lg(const cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->lg32; else return m->lg64;
}

// Calls f with the mesh's plan, vector width and geometry: f(plan, width,
// geometry kind, geometry), the two in the middle as integral constants.
template <class T, class F> void with_star(const cfd_mesh_s* m, F f) {
    auto with_width = [&](auto w) {
        const star::Plan pl = star::make_plan(m->X, m->Y, m->Z, w());
        if (!m->uniform) f(pl, w, std::integral_constant<int, 2>{}, lg<T>(m));
        else if (ug<T>(m).vol_pow2) f(pl, w, std::integral_constant<int, 0>{}, ug<T>(m));
        else f(pl, w, std::integral_constant<int, 1>{}, ug<T>(m));
    };
    if (star::vector_form<T>(m->Y, m->Z)) with_width(std::integral_constant<int, star::kWidth<T>>{});
    else with_width(std::integral_constant<int, 1>{});
    CFD_HIP(hipGetLastError());
}

}  // namespace

template <class T>
void launch_grad_star(const cfd_mesh_s* m, const void* phi, void* out, int mask, int wall, hipStream_t s) {
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto geo, const auto& g) {
        grad_star_k<T, decltype(w)::value, decltype(geo)::value>
            <<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)phi, (T*)out, mask, wall, pl);
    });
}

template <class T> void launch_lapl_star(const cfd_mesh_s* m, const void* phi, void* out, int mask, hipStream_t s) {
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto geo, const auto& g) {
        lapl_star_k<T, decltype(w)::value, decltype(geo)::value>
            <<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)phi, (T*)out, mask, pl);
    });
}

template <class T> void launch_stab_star(const cfd_mesh_s* m, const void* phi, void* out, int mask, hipStream_t s) {
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto geo, const auto& g) {
        if constexpr (decltype(geo)::value != 2)
            stab_star_k<T, decltype(w)::value, decltype(geo)::value == 0>
                <<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)phi, (T*)out, mask, pl);
    });
}

template <class T>
void launch_heat_star(const cfd_mesh_s* m, const void* in, void* out, double alpha, const void* af, double dt,
                      hipStream_t s) {
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto geo, const auto& g) {
        constexpr int W = decltype(w)::value, GEO = decltype(geo)::value;
        auto* kern = af ? heat_star_k<T, W, GEO, true> : heat_star_k<T, W, GEO, false>;
        kern<<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)in, (T*)out, T(alpha), (const T*)af,
                                                                T(dt), pl);
    });
}

template <class T>
void launch_wave_lattice(const cfd_mesh_s* m, void* const* in, void* const* out, double K, const void* Kf, double dt,
                         hipStream_t s) {
    auto run = [&](auto w) {
        constexpr int W = decltype(w)::value;
        const star::Plan pl = star::make_plan(m->X, m->Y, m->Z, W);
        const LatticeGeo<T>& g = lg<T>(m);
        wave_vel_lattice_k<T, W><<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(
            g, (const T*)in[0], (const T*)in[1], (const T*)in[2], (const T*)in[3], (T*)out[1], (T*)out[2], (T*)out[3],
            T(dt), pl);
        CFD_HIP(hipGetLastError());
        auto* kern = Kf ? wave_p_lattice_k<T, W, true> : wave_p_lattice_k<T, W, false>;
        kern<<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(
            g, (const T*)out[1], (const T*)out[2], (const T*)out[3], (const T*)in[0], (T*)out[0], T(K), (const T*)Kf,
            T(dt), pl);
        CFD_HIP(hipGetLastError());
    };
    if (star::vector_form<T>(m->Y, m->Z)) run(std::integral_constant<int, star::kWidth<T>>{});
    else run(std::integral_constant<int, 1>{});
}

#define CFD_INSTANTIATE(T)                                                                                         \
    template void launch_grad_star<T>(const cfd_mesh_s*, const void*, void*, int, int, hipStream_t);              \
    template void launch_lapl_star<T>(const cfd_mesh_s*, const void*, void*, int, hipStream_t);                   \
    template void launch_stab_star<T>(const cfd_mesh_s*, const void*, void*, int, hipStream_t);                   \
    template void launch_heat_star<T>(const cfd_mesh_s*, const void*, void*, double, const void*, double,         \
                                      hipStream_t);                                                                \
    template void launch_wave_lattice<T>(const cfd_mesh_s*, void* const*, void* const*, double, const void*,      \
                                         double, hipStream_t);
CFD_INSTANTIATE(float)
CFD_INSTANTIATE(double)

}  // namespace cfd
