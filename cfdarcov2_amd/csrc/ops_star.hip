// Gradient, Laplacian, stabilisation and heat step in star form (star.hpp) on
// exactly uniform meshes (ops_faces.hip: the others).  The geometry is a
// handful of constants in the kernel arguments, so only the fields cross
// memory; PW: the cell volume is a power of two.
//
// Measured against one cell per thread with 64-bit indices: heat step 64^3
// FP64 2.8 us against 3.5 (2.6 as one of two per launch); gradient,
// Laplacian and stabilisation of 200^3 FP32 together 68 against 151 us.
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

}  // namespace

// SOME: an operator over some axes loads only their neighbours.  On fields that
// stay in the last-level cache the other loads cost nothing (they bring lines
// that other workgroups read: one-axis gradient 256^3 FP64 39.3 us with all, 48
// with the axis' own), beyond it they cross memory (one-axis gradient FP64
// 512x256x256 128 / 100, 300^3 118 / 94).
template <class T, int W, bool PW, bool SOME>
__global__ void __launch_bounds__(256) grad_star_k(UniformGeo<T> g, const T* __restrict__ phi,
                                                   T* __restrict__ out, int mask, int wall_axis, star::Plan pl) {
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const star::Star7<T, W> s = SOME ? star::load_axes<T, W>(phi, o, mask) : star::load7<T, W>(phi, o);
    const VolDiv<T, PW> Vd{g.vol, g.inv_vol};
    T r[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const star::Faces<T> f = lin_faces(s, at_wall(pl, q, i), wall_axis, i);
        T res = T(0);
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if (mask & (1 << a)) res = res + mggp(f.lo[a], f.hi[a], g.area[a], Vd);
        r[i] = res;
    }
    star::store<T, W>(out + o.x0, o.o0, r);
}

template <class T, int W, bool PW, bool SOME>
__global__ void __launch_bounds__(256) lapl_star_k(UniformGeo<T> g, const T* __restrict__ phi,
                                                   T* __restrict__ out, int mask, star::Plan pl) {
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const star::Star7<T, W> s = SOME ? star::load_axes<T, W>(phi, o, mask) : star::load7<T, W>(phi, o);
    T r[W];
#pragma unroll
    for (int i = 0; i < W; ++i) r[i] = star::lapl_uniform<T, W, PW>(g, s, mask, i);
    star::store<T, W>(out + o.x0, o.o0, r);
}

// T' = dt * (alpha * lapl(T)) + T (DtVar::extract order, src/fvm3d.cpp:690-692)
template <class T, int W, bool PW, bool AF>
__global__ void __launch_bounds__(256) heat_star_k(UniformGeo<T> g, const T* __restrict__ Tin,
                                                   T* __restrict__ Tout, T alpha, const T* __restrict__ alpha_f, T dt,
                                                   star::Plan pl) {
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const star::Star7<T, W> s = star::load7<T, W>(Tin, o);
    T af[W];
    if constexpr (AF) star::load<T, W>(alpha_f + o.x0, o.o0, af);
    T r[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const T k = AF ? af[i] : alpha;
        r[i] = dt * (k * star::lapl_uniform<T, W, PW>(g, s, 7, i)) + s.c(i);
    }
    star::store<T, W>(Tout + o.x0, o.o0, r);
}

// Two heat steps in one launch: a thread recomputes the first step's values of
// its cells' neighbours (W + 2 cells of its row and W of each adjacent one)
// from the rows up to two cells away, each with its own operation sequence, so
// the bits are those of two launches. us per step against
// one step per launch: 16^3 FP32 1.4 / 2.2, 48^3 1.7 / 2.5, 64^3 2.1 / 2.6,
// 16^3 FP64 1.6 / 2.3, 64^3 2.65 / 2.85.  Bound by the launch (2 us) and by
// one wavefront's serial work, so only for meshes that a launch outlasts: the
// redundant steps make 80^3 (3.3 / 3.2 FP32, 4.5 / 3.8 FP64) slower.
template <class T, int W, bool PW, bool AF>
__global__ void __launch_bounds__(256) heat2_star_k(UniformGeo<T> g, const T* __restrict__ Tin,
                                                    T* __restrict__ Tout, T alpha, const T* __restrict__ alpha_f,
                                                    T dt, star::Plan pl) {
    using star::load;
    using star::load1;
    using O = star::Off<W>;
    star::Place q;
    if (!star::place<W>(pl, q)) return;
    const star::Offsets<W> o = star::offsets<W>(pl, q);
    const VolDiv<T, PW> Vd{g.vol, g.inv_vol};
    const int64_t SX = int64_t(pl.Y) * pl.Z;
    const O uz = O(pl.Z), zl = O(o.o0 - o.zm1), zh = O(o.zp1 - o.o0);
    // W values of a row with one cell on each side
    auto wide = [&](const T* f, O off, T(&r)[W + 2]) {
        T c[W];
        load<T, W>(f, off, c);
        r[0] = load1(f, O(off - zl));
        r[W + 1] = load1(f, O(off + zh));
#pragma unroll
        for (int i = 0; i < W; ++i) r[i + 1] = c[i];
    };
    const T *const f0 = Tin + o.x0, *const fl = Tin + o.xm1, *const fh = Tin + o.xp1;
    T c[W + 2], xl[W + 2], xh[W + 2], yl[W + 2], yh[W + 2];
    T xl2[W], xh2[W], yl2[W], yh2[W], ll[W], lh[W], hl[W], hh[W];
    wide(f0, o.o0, c);
    wide(fl, o.o0, xl);
    wide(fh, o.o0, xh);
    wide(f0, o.ym1, yl);
    wide(f0, o.yp1, yh);
    const T zl2 = load1(f0, q.z0 >= 2 ? o.zm1 - 1 : o.zm1);
    const T zh2 = load1(f0, q.z0 + W + 1 < pl.Z ? o.zp1 + 1 : o.zp1);
    load<T, W>(q.x >= 2 ? fl - SX : fl, o.o0, xl2);
    load<T, W>(q.x + 2 < pl.X ? fh + SX : fh, o.o0, xh2);
    load<T, W>(f0, q.y >= 2 ? o.ym1 - uz : o.ym1, yl2);
    load<T, W>(f0, q.y + 2 < pl.Y ? o.yp1 + uz : o.yp1, yh2);
    load<T, W>(fl, o.ym1, ll);  // rows (x-1, y-1), (x-1, y+1), (x+1, y-1), (x+1, y+1)
    load<T, W>(fl, o.yp1, lh);
    load<T, W>(fh, o.ym1, hl);
    load<T, W>(fh, o.yp1, hh);
    T kc[W + 2], kxl[W], kxh[W], kyl[W], kyh[W];
    if constexpr (AF) {
        wide(alpha_f + o.x0, o.o0, kc);
        load<T, W>(alpha_f + o.xm1, o.o0, kxl);
        load<T, W>(alpha_f + o.xp1, o.o0, kxh);
        load<T, W>(alpha_f + o.x0, o.ym1, kyl);
        load<T, W>(alpha_f + o.x0, o.yp1, kyh);
    }
    auto step = [&](T pc, T a0, T a1, T b0, T b1, T d0, T d1, T k) {
        const T lo[3] = {a0, b0, d0}, hi[3] = {a1, b1, d1};
        T L = T(0);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const T s_lo = (-pc + lo[a]) * g.alpha[a];
            const T s_hi = (-pc + hi[a]) * g.alpha[a];
            L = L + Vd(s_lo * g.area[a] + s_hi * g.area[a]);
        }
        return dt * (k * L) + pc;
    };
    const bool wxl = q.x == 0, wxh = q.x == pl.X - 1, wyl = q.y == 0, wyh = q.y == pl.Y - 1;
    T n[W + 2];  // the row after the first step
#pragma unroll
    for (int j = 0; j < W + 2; ++j)
        n[j] = step(c[j], xl[j], xh[j], yl[j], yh[j], j ? c[j - 1] : zl2, j < W + 1 ? c[j + 1] : zh2,
                    AF ? kc[j] : alpha);
    if (q.z0 == 0) n[0] = n[1];
    if (q.z0 + W == pl.Z) n[W + 1] = n[W];
    T r[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const int j = i + 1;
        const T a0 = step(xl[j], xl2[i], c[j], ll[i], lh[i], xl[j - 1], xl[j + 1], AF ? kxl[i] : alpha);
        const T a1 = step(xh[j], c[j], xh2[i], hl[i], hh[i], xh[j - 1], xh[j + 1], AF ? kxh[i] : alpha);
        const T b0 = step(yl[j], ll[i], hl[i], yl2[i], c[j], yl[j - 1], yl[j + 1], AF ? kyl[i] : alpha);
        const T b1 = step(yh[j], lh[i], hh[i], c[j], yh2[i], yh[j - 1], yh[j + 1], AF ? kyh[i] : alpha);
        r[i] = step(n[j], wxl ? n[j] : a0, wxh ? n[j] : a1, wyl ? n[j] : b0, wyh ? n[j] : b1, n[j - 1], n[j + 1],
                    AF ? kc[j] : alpha);
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

namespace {

template <class T> const UniformGeo<T>& ug(const cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->ug32; else return m->ug64;
}

// Calls f(plan, vector width, whether the volume is a power of two, geometry),
// the two in the middle as integral constants.
template <class T, class F> void with_star(const cfd_mesh_s* m, F f, bool narrow = false) {
    auto with_width = [&](auto w) {
        const star::Plan pl = star::make_plan(m->X, m->Y, m->Z, w());
        if (ug<T>(m).vol_pow2) f(pl, w, std::true_type{}, ug<T>(m));
        else f(pl, w, std::false_type{}, ug<T>(m));
    };
    if (star::vector_form<T>(m->Y, m->Z) && !narrow) with_width(std::integral_constant<int, star::kWidth<T>>{});
    else with_width(std::integral_constant<int, 1>{});
    CFD_HIP(hipGetLastError());
}

// whether an operator over `mask` loads the neighbours of its axes only (see grad_star_k)
template <class T> bool some_axes(const cfd_mesh_s* m, int mask) {
    return mask != 7 && 2 * m->N * int64_t(sizeof(T)) > kLastLevelCacheBytes;
}

}  // namespace

template <class T>
void launch_grad_star(const cfd_mesh_s* m, const void* phi, void* out, int mask, int wall, hipStream_t s) {
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto pw, const auto& g) {
        constexpr int W = decltype(w)::value;
        constexpr bool PW = decltype(pw)::value;
        auto* kern = some_axes<T>(m, mask) ? grad_star_k<T, W, PW, true> : grad_star_k<T, W, PW, false>;
        kern<<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)phi, (T*)out, mask, wall, pl);
    });
}

template <class T> void launch_lapl_star(const cfd_mesh_s* m, const void* phi, void* out, int mask, hipStream_t s) {
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto pw, const auto& g) {
        constexpr int W = decltype(w)::value;
        constexpr bool PW = decltype(pw)::value;
        auto* kern = some_axes<T>(m, mask) ? lapl_star_k<T, W, PW, true> : lapl_star_k<T, W, PW, false>;
        kern<<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)phi, (T*)out, mask, pl);
    });
}

template <class T> void launch_stab_star(const cfd_mesh_s* m, const void* phi, void* out, int mask, hipStream_t s) {
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto pw, const auto& g) {
        stab_star_k<T, decltype(w)::value, decltype(pw)::value>
            <<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)phi, (T*)out, mask, pl);
    });
}

template <class T>
void launch_heat_star(const cfd_mesh_s* m, const void* in, void* out, double alpha, const void* af, double dt,
                      hipStream_t s) {
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto pw, const auto& g) {
        constexpr int W = decltype(w)::value;
        constexpr bool PW = decltype(pw)::value;
        auto* kern = af ? heat_star_k<T, W, PW, true> : heat_star_k<T, W, PW, false>;
        kern<<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)in, (T*)out, T(alpha), (const T*)af,
                                                                T(dt), pl);
    });
}

template <class T>
void launch_heat2_star(const cfd_mesh_s* m, const void* in, void* out, double alpha, const void* af, double dt,
                       hipStream_t s) {
    static_assert(kHeat2Cells <= int64_t(1) << 18, "two-step meshes are narrow in FP32");
    with_star<T>(m, [&](const star::Plan& pl, auto w, auto pw, const auto& g) {
        constexpr int W = decltype(w)::value;
        constexpr bool PW = decltype(pw)::value;
        if constexpr (sizeof(T) == 8 || W == 1) {  // FP32 is narrow wherever two steps are taken
            auto* kern = af ? heat2_star_k<T, W, PW, true> : heat2_star_k<T, W, PW, false>;
            kern<<<star::plan_grid(pl), star::plan_block(pl), 0, s>>>(g, (const T*)in, (T*)out, T(alpha),
                                                                    (const T*)af, T(dt), pl);
        }
    }, star::narrow<T>(m->N));
}

#define CFD_INSTANTIATE(T)                                                                                         \
    template void launch_grad_star<T>(const cfd_mesh_s*, const void*, void*, int, int, hipStream_t);              \
    template void launch_lapl_star<T>(const cfd_mesh_s*, const void*, void*, int, hipStream_t);                   \
    template void launch_stab_star<T>(const cfd_mesh_s*, const void*, void*, int, hipStream_t);                   \
    template void launch_heat_star<T>(const cfd_mesh_s*, const void*, void*, double, const void*, double,         \
                                      hipStream_t);                                                                \
    template void launch_heat2_star<T>(const cfd_mesh_s*, const void*, void*, double, const void*, double,        \
                                       hipStream_t);
CFD_INSTANTIATE(float)
CFD_INSTANTIATE(double)

}  // namespace cfd
