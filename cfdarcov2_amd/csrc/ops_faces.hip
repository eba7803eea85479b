// Gradient, Laplacian, stabilisation, heat and acoustic steps in star form
// (star.hpp) on meshes with face geometry:
//   GEO 2, axis-aligned lattices (LatticeGeo): widths and alpha_d per layer,
//          volume per cell; normals are the unit vectors;
//   GEO 3, general structured meshes (GeneralGeo): normal, area and alpha_d
//          per face of each family, volume per cell.
// A thread's W cells along z read whole vectors of face values: the y- and
// x-faces of a row lie at consecutive places, its z-faces are W + 1 values.
// Consecutive planes run on one XCD, so both cells of a face find its geometry
// in one L2.
//
// Bound by the geometry: beside its 16 bytes of state an FP64 heat cell of a
// general mesh moves 128 (three faces of normal, area and alpha_d, 120, and the
// volume), of a lattice 8.  us before (one cell per thread, 64-bit indices,
// planes spread over the XCDs) and now, 200^3 FP32: perturbed mesh, gradient 156
// / 99, Laplacian 180 / 122, stabilisation 526 / 288; on a decimal lattice 527 /
// 128; FP64 perturbed 292 / 194, 328 / 239, 994 / 583 and decimal 994 / 278.
// Steps on decimal lattices: heat 100^3 FP64 38.4 / 6.6, acoustic 120x100x80
// FP32 49.0 / 14.0.
//
// The arithmetic is the reference's (src/fvm3d.cpp:825-829,902-942 and
// :690-692 with include/grad_utils.hpp:23-125) in its order, sums over the six
// faces from 0 in the local order z-, z+, y-, y+, x-, x+.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"
#include "march.hpp"
#include "star.hpp"

namespace cfd {

namespace {

using star::Offsets;
using star::Place;
using star::Plan;
using star::Star7;

template <class T, int GEO> struct FaceArg { using type = LatticeGeo<T>; };
template <class T> struct FaceArg<T, 3> { using type = GeneralGeo<T>; };

// axis of local face fc
__device__ constexpr int axis_of(int fc) { return 2 - (fc >> 1); }

template <class T, int W, int GEO, class O> struct CellGeo;

template <class T, int W, class O> struct CellGeo<T, W, 2, O> {
    star::LatticeCells<T, W> c;
    __device__ CellGeo(const LatticeGeo<T>& g, const Plan&, const Place& q, const Offsets<W, O>& o)
        : c(star::load_lattice<T, W, true>(g, o, q)) {}
    __device__ void alphas(T (&al)[6][W]) const {
#pragma unroll
        for (int i = 0; i < W; ++i) {
            al[0][i] = c.az[i]; al[1][i] = c.az[i + 1];
            al[2][i] = c.ay[0]; al[3][i] = c.ay[1];
            al[4][i] = c.ax[0]; al[5][i] = c.ax[1];
        }
    }
    __device__ void normals(int d, T (&n)[6][W]) const {
#pragma unroll
        for (int fc = 0; fc < 6; ++fc)
#pragma unroll
            for (int i = 0; i < W; ++i) n[fc][i] = T(axis_of(fc) == d);
    }
    template <bool OUTWARD> __device__ void gauss(const T (&fv)[6][W], const T (&)[6][W], int d, T (&r)[W]) const {
#pragma unroll
        for (int i = 0; i < W; ++i) {
            const star::Faces<T> f{{fv[4][i], fv[2][i], fv[0][i]}, {fv[5][i], fv[3][i], fv[1][i]}};
            r[i] = d == 0 ? star::lattice_gauss<T, W, OUTWARD>(c, f, 0, i)
                 : d == 1 ? star::lattice_gauss<T, W, OUTWARD>(c, f, 1, i)
                          : star::lattice_gauss<T, W, OUTWARD>(c, f, 2, i);
        }
    }
};

template <class T, int W, class O> struct CellGeo<T, W, 3, O> {
    const GeneralGeo<T>& g;
    int64_t zb, yb, xb, SX;  // plane bases of the z-, y- and x-faces
    O zo, co, Z;             // the first cell's z-face, and its cell and lower y- and x-face, within a plane
    T A[6][W], V[W];
    __device__ CellGeo(const GeneralGeo<T>& geo, const Plan& pl, const Place& q, const Offsets<W, O>& o) : g(geo) {
        SX = int64_t(pl.Y) * pl.Z;
        zb = int64_t(q.x) * pl.Y * (pl.Z + 1);
        yb = int64_t(q.x) * (pl.Y + 1) * pl.Z;
        xb = o.x0;
        Z = O(pl.Z);
        zo = O(q.y) * O(pl.Z + 1) + O(q.z0);
        co = o.o0;
        faces(g.farea, A);
        star::load<T, W>(g.vol + o.x0, o.o0, V);
    }
    // the six faces' values of an array per family
    __device__ void faces(const T* const (&fam)[3], T (&v)[6][W]) const {
        star::load<T, W>(fam[0] + zb, zo, v[0]);
        const T last = star::load1(fam[0] + zb, O(zo + O(W)));
#pragma unroll
        for (int i = 0; i + 1 < W; ++i) v[1][i] = v[0][i + 1];
        v[1][W - 1] = last;
        star::load<T, W>(fam[1] + yb, co, v[2]);
        star::load<T, W>(fam[1] + yb, O(co + Z), v[3]);
        star::load<T, W>(fam[2] + xb, co, v[4]);
        star::load<T, W>(fam[2] + xb + SX, co, v[5]);
    }
    __device__ void alphas(T (&al)[6][W]) const { faces(g.falpha, al); }
    __device__ void normals(int d, T (&n)[6][W]) const {
        const T* const fam[3] = {g.fn[0][d], g.fn[1][d], g.fn[2][d]};
        faces(fam, n);
    }
    template <bool OUTWARD> __device__ void gauss(const T (&fv)[6][W], const T (&n)[6][W], int, T (&r)[W]) const {
#pragma unroll
        for (int i = 0; i < W; ++i) {
            T acc = T(0);
#pragma unroll
            for (int fc = 0; fc < 6; ++fc) {
                T t = fv[fc][i] * ((OUTWARD && !(fc & 1)) ? -n[fc][i] : n[fc][i]);
                t = t * A[fc][i];
                acc = acc + t;
            }
            r[i] = acc / V[i];
        }
    }
};

template <class T, int W> __device__ inline T nb_of(const Star7<T, W>& s, int fc, int i) {
    return star::face_nb(s, axis_of(fc), fc & 1, i);
}

// whether local face fc of cell i lies on the wall
__device__ inline bool on_wall(const Plan& pl, const Place& q, int fc, int i) {
    const int a = axis_of(fc);
    const int k = a == 0 ? q.x : a == 1 ? q.y : q.z0 + i, n = a == 0 ? pl.X : a == 1 ? pl.Y : pl.Z;
    return (fc & 1) ? k == n - 1 : k == 0;
}

// interpolated face values, zero on the walls normal to wall_axis
template <class T, int W>
__device__ inline void lin_faces(const Star7<T, W>& s, const Plan& pl, const Place& q, int wall_axis,
                                 T (&fv)[6][W]) {
#pragma unroll
    for (int fc = 0; fc < 6; ++fc)
#pragma unroll
        for (int i = 0; i < W; ++i) {
            fv[fc][i] = mlin(s.c(i), nb_of(s, fc, i));
            if (wall_axis == axis_of(fc) && on_wall(pl, q, fc, i)) fv[fc][i] = T(0);
        }
}

// Laplacian over the selected axes, from 0 in the order x, y, z
template <class T, int W, int GEO, class O>
__device__ inline void lapl_of(const CellGeo<T, W, GEO, O>& c, const Star7<T, W>& s, int mask, T (&res)[W]) {
    T fv[6][W], n[6][W], r[W];
    c.alphas(fv);
#pragma unroll
    for (int fc = 0; fc < 6; ++fc)
#pragma unroll
        for (int i = 0; i < W; ++i) fv[fc][i] = (-s.c(i) + nb_of(s, fc, i)) * fv[fc][i];
#pragma unroll
    for (int i = 0; i < W; ++i) res[i] = T(0);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (!(mask & (1 << d))) continue;
        c.normals(d, n);
        c.template gauss<false>(fv, n, d, r);
#pragma unroll
        for (int i = 0; i < W; ++i) res[i] = res[i] + r[i];
    }
}

}  // namespace

#define CFD_STAR_HEAD                                 \
    Place q;                                          \
    if (!star::place<W>(pl, q)) return;               \
    const Offsets<W, O> o = star::offsets<W, O>(pl, q);

template <class T, int W, int GEO, class O>
__global__ void __launch_bounds__(256) fgrad_k(typename FaceArg<T, GEO>::type g, const T* __restrict__ phi,
                                               T* __restrict__ out, int mask, int wall_axis, Plan pl) {
    CFD_STAR_HEAD
    const Star7<T, W> s = star::load7<T, W>(phi, o);
    const CellGeo<T, W, GEO, O> c(g, pl, q, o);
    T fv[6][W], n[6][W], r[W], res[W];
    lin_faces(s, pl, q, wall_axis, fv);
#pragma unroll
    for (int i = 0; i < W; ++i) res[i] = T(0);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (!(mask & (1 << d))) continue;
        c.normals(d, n);
        c.template gauss<true>(fv, n, d, r);
#pragma unroll
        for (int i = 0; i < W; ++i) res[i] = res[i] + r[i];
    }
    star::store<T, W>(out + o.x0, o.o0, res);
}

template <class T, int W, int GEO, class O>
__global__ void __launch_bounds__(256) flapl_k(typename FaceArg<T, GEO>::type g, const T* __restrict__ phi,
                                               T* __restrict__ out, int mask, Plan pl) {
    CFD_STAR_HEAD
    const Star7<T, W> s = star::load7<T, W>(phi, o);
    const CellGeo<T, W, GEO, O> c(g, pl, q, o);
    T res[W];
    lapl_of(c, s, mask, res);
    star::store<T, W>(out + o.x0, o.o0, res);
}

// T' = dt * (alpha * lapl(T)) + T (DtVar::extract order, src/fvm3d.cpp:690-692)
template <class T, int W, int GEO, class O, bool AF>
__global__ void __launch_bounds__(256) fheat_k(typename FaceArg<T, GEO>::type g, const T* __restrict__ Tin,
                                               T* __restrict__ Tout, T alpha, const T* __restrict__ alpha_f, T dt,
                                               Plan pl) {
    CFD_STAR_HEAD
    const Star7<T, W> s = star::load7<T, W>(Tin, o);
    const CellGeo<T, W, GEO, O> c(g, pl, q, o);
    T af[W], res[W];
    if constexpr (AF) star::load<T, W>(alpha_f + o.x0, o.o0, af);
    lapl_of(c, s, 7, res);
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const T k = AF ? af[i] : alpha;
        res[i] = dt * (k * res[i]) + s.c(i);
    }
    star::store<T, W>(Tout + o.x0, o.o0, res);
}

// Kernels of three outputs store them after all loads where the registers
// allow it, since a store keeps back the loads after it (acoustic step of
// perturbed 64^3 FP32, one cell per thread 8.8 / 8.4 us; with vectors it costs:
// lattice 200^3 FP64 199 / 206).
template <class T, int W> constexpr bool kLateStores = sizeof(T) == 4 && W == 1;

// StabVar, first stage: the three gradient components
template <class T, int W, int GEO, class O>
__global__ void __launch_bounds__(256) fgrad3_k(typename FaceArg<T, GEO>::type g, const T* __restrict__ phi,
                                                T* __restrict__ gx, T* __restrict__ gy, T* __restrict__ gz, Plan pl) {
    CFD_STAR_HEAD
    const Star7<T, W> s = star::load7<T, W>(phi, o);
    const CellGeo<T, W, GEO, O> c(g, pl, q, o);
    T* const out[3] = {gx, gy, gz};
    T fv[6][W], n[6][W], r[3][W];
    lin_faces(s, pl, q, -1, fv);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        c.normals(d, n);
        c.template gauss<true>(fv, n, d, r[d]);
        if constexpr (!kLateStores<T, W>) star::store<T, W>(out[d] + o.x0, o.o0, r[d]);
    }
    if constexpr (kLateStores<T, W>)
#pragma unroll
        for (int d = 0; d < 3; ++d) star::store<T, W>(out[d] + o.x0, o.o0, r[d]);
}

// StabVar, second stage: per selected component d the upwind face value
// phi + (len * g_d) * n_out of the cell against the neighbour's at the same face
// (which it sees as its opposite local face; on a wall the neighbour is the
// cell itself, at its own opposite face), 0.5 * jump, axis-normal Gauss sum.
// len: six centre-to-face distances per cell, fc-major.
template <class T, int W, int GEO, class O>
__global__ void __launch_bounds__(256) fstab_k(typename FaceArg<T, GEO>::type g, const T* __restrict__ len,
                                               const T* __restrict__ phi, const T* __restrict__ gx,
                                               const T* __restrict__ gy, const T* __restrict__ gz,
                                               T* __restrict__ out, int mask, Plan pl) {
    CFD_STAR_HEAD
    const int64_t N = int64_t(pl.X) * pl.Y * pl.Z;
    const Star7<T, W> s = star::load7<T, W>(phi, o);
    const CellGeo<T, W, GEO, O> c(g, pl, q, o);
    const T* const gd[3] = {gx, gy, gz};
    // own lengths, and the neighbours' at their opposite local faces (the
    // clamped neighbour of a wall cell is the cell itself, as its rule asks)
    T own[6][W], col[6][W];
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) star::load<T, W>(len + fc * N + o.x0, o.o0, own[fc]);
    star::load<T, W>(len + 5 * N + o.xm1, o.o0, col[4]);
    star::load<T, W>(len + 4 * N + o.xp1, o.o0, col[5]);
    star::load<T, W>(len + 3 * N + o.x0, o.ym1, col[2]);
    star::load<T, W>(len + 2 * N + o.x0, o.yp1, col[3]);
    col[0][0] = star::load1(len + 1 * N + o.x0, o.zm1);
    col[1][W - 1] = star::load1(len + o.x0, o.zp1);
#pragma unroll
    for (int i = 0; i + 1 < W; ++i) {
        col[0][i + 1] = own[1][i];
        col[1][i] = own[0][i + 1];
    }
    T res[W];
#pragma unroll
    for (int i = 0; i < W; ++i) res[i] = T(0);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (!(mask & (1 << d))) continue;
        const Star7<T, W> sg = star::load7<T, W>(gd[d], o);
        T n[6][W], fv[6][W], r[W];
        c.normals(d, n);
#pragma unroll
        for (int fc = 0; fc < 6; ++fc)
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const T n_own = (fc & 1) ? n[fc][i] : -n[fc][i];
                T n_col = (fc & 1) ? -n[fc][i] : n[fc][i];
                if (on_wall(pl, q, fc, i)) n_col = (fc & 1) ? -n[fc ^ 1][i] : n[fc ^ 1][i];
                const T vo = s.c(i) + (own[fc][i] * sg.c(i)) * n_own;
                const T vc = nb_of(s, fc, i) + (col[fc][i] * nb_of(sg, fc, i)) * n_col;
                fv[fc][i] = T(0.5) * (vo - vc);
            }
        c.template gauss<false>(fv, n, d, r);
#pragma unroll
        for (int i = 0; i < W; ++i) res[i] = res[i] + r[i];
    }
    star::store<T, W>(out + o.x0, o.o0, res);
}

// Acoustic step: skewed face normals make every gradient component depend on
// all six faces, so the three velocity equations (from p) and the pressure
// equation (from the new velocities) are two launches.  Lattices keep them too:
// one pass would recompute the neighbours' velocities from p, and these turn
// NaN wherever any face value of that cell is not finite, which the
// recomputation could not see without loading all its faces.
template <class T, int W, int GEO, class O>
__global__ void __launch_bounds__(256) fwave_vel_k(typename FaceArg<T, GEO>::type g, const T* __restrict__ p,
                                                   const T* __restrict__ u, const T* __restrict__ v,
                                                   const T* __restrict__ w, T* __restrict__ uo, T* __restrict__ vo,
                                                   T* __restrict__ wo, T dt, Plan pl) {
    CFD_STAR_HEAD
    const Star7<T, W> s = star::load7<T, W>(p, o);
    const CellGeo<T, W, GEO, O> c(g, pl, q, o);
    const T* const in[3] = {u, v, w};
    T* const out[3] = {uo, vo, wo};
    T fv[6][W], n[6][W], r[W], vel[3][W];
#pragma unroll
    for (int d = 0; d < 3; ++d) star::load<T, W>(in[d] + o.x0, o.o0, vel[d]);
    lin_faces(s, pl, q, -1, fv);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        c.normals(d, n);
        c.template gauss<true>(fv, n, d, r);
#pragma unroll
        for (int i = 0; i < W; ++i) vel[d][i] = dt * (-r[i]) + vel[d][i];
        if constexpr (!kLateStores<T, W>) star::store<T, W>(out[d] + o.x0, o.o0, vel[d]);
    }
    if constexpr (kLateStores<T, W>)
#pragma unroll
        for (int d = 0; d < 3; ++d) star::store<T, W>(out[d] + o.x0, o.o0, vel[d]);
}

template <class T, int W, int GEO, class O, bool KF>
__global__ void __launch_bounds__(256) fwave_p_k(typename FaceArg<T, GEO>::type g, const T* __restrict__ u,
                                                 const T* __restrict__ v, const T* __restrict__ w,
                                                 const T* __restrict__ p, T* __restrict__ po, T K,
                                                 const T* __restrict__ Kf, T dt, Plan pl) {
    CFD_STAR_HEAD
    const CellGeo<T, W, GEO, O> c(g, pl, q, o);
    const T* const in[3] = {u, v, w};
    T pc[W], kf[W], S[W];
    star::load<T, W>(p + o.x0, o.o0, pc);
    if constexpr (KF) star::load<T, W>(Kf + o.x0, o.o0, kf);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const Star7<T, W> s = star::load7<T, W>(in[a], o);
        T fv[6][W], n[6][W], r[W];
        lin_faces(s, pl, q, a, fv);
        c.normals(a, n);
        c.template gauss<true>(fv, n, a, r);
#pragma unroll
        for (int i = 0; i < W; ++i) S[i] = a == 0 ? r[i] : S[i] + r[i];
    }
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const T k = KF ? kf[i] : K;
        pc[i] = dt * (k * S[i]) + pc[i];
    }
    star::store<T, W>(po + o.x0, o.o0, pc);
}

#undef CFD_STAR_HEAD

namespace {

template <class T> const LatticeGeo<T>& lg(const cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->lg32; else return m->lg64;
}
template <class T> const GeneralGeo<T>& gg(const cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->gg32; else return m->gg64;
}

enum class Op { grad, lapl, stab, heat, wave };

// The largest mesh, in cells, on which an operator takes one cell per thread.
// Small meshes because a launch then lasts about as long as one wavefront's
// chain of operations, which is W times as long with vectors; in FP32 larger
// perturbed ones too, because their kernels with vectors hold few wavefronts
// (three to five per SIMD) while the face arrays stay in the last-level cache.
// Time with vectors / with one cell per thread, in a captured graph:
//               40^3  56^3  64^3  80^3  100^3 128^3 160^3
//   lattice   grad  1.12  1.12  1.02  0.98  0.73  0.74  0.52
//   FP32      lapl  1.13  1.15  1.06  1.10  0.86  0.90  0.58
//             stab  1.18  1.17  1.08  1.14  0.95  1.05  0.83
//             heat  1.11  1.16  1.03  1.06  0.85  0.89  0.66
//             wave  1.22  1.22  1.11  1.15  0.96  1.07  0.89
//   perturbed grad  1.29  1.20  1.13  1.07  0.99  1.09  1.09 (200^3 0.97)
//   FP32      lapl  1.14  1.12  1.01  1.01  0.97  1.03  0.81
//             stab  1.28  1.16  1.21  1.19  1.03  1.07  0.80
//             heat  1.15  1.19  1.14  1.21  1.09  1.14  0.89
//             wave  1.35  1.23  1.27  1.20  1.08  1.16  0.85
//               16^3  24^3  32^3  36^3  40^3  48^3  56^3
//   lattice   heat  1.02  0.98  0.98  0.94  0.95  0.97  0.86 (the others within 0.04 but
//   FP64      wave  1.12  1.08  1.08  1.01  0.96  1.01  0.84  of 16^3 to 20^3, up to 1.07)
//   perturbed heat  1.10  1.04  1.03  0.99  0.92  0.91  0.79 (grad 1.06 to 0.77, lapl
//   FP64      wave  1.27  1.21  1.20  1.11  1.01  0.98  0.84  1.05 to 0.78, stab 1.13 to 0.80)
template <class T> int64_t one_cell_limit(Op op, bool lattice) {
    int bits;
    if (sizeof(T) == 8) bits = op == Op::wave && !lattice ? 16 : 15;
    else if (lattice) bits = op == Op::grad ? 18 : 19;
    else bits = op == Op::grad ? 22 : 21;
    return int64_t(1) << bits;
}

// f(plan, grid, block, width, geometry kind, offset, geometry): width and kind
// as integral constants, the offset a value of its type
template <class T, class F> void with_faces(const cfd_mesh_s* m, Op op, F f) {
    // Face arrays beyond half the last-level cache on meshes long in z: runs of
    // columns (us, cut in x / z: heat step FP64 40x40x1000 44.9 / 39.6, 60x60x2000
    // 246 / 216, FP32 40x40x2000 45.2 / 39.7; below that size FP32 40x40x1000 22.1
    // / 24.6).  The steps take one cell per thread there (with vectors / one, both
    // cut in z: acoustic step FP64 40x40x1000 95.5 / 87.8, 60x60x2000 480 / 472,
    // 64x64x512 130 / 134, FP32 40x40x2000 90.7 / 83.1; heat step FP64 39.6 / 37.1,
    // 216 / 214, 57.8 / 58.9).
    const bool long_z = !m->lattice && m->Z >= 8 * std::max(m->X, m->Y) &&
                        2 * 17 * m->N * int64_t(sizeof(T)) > kLastLevelCacheBytes;
    const bool one = m->N <= one_cell_limit<T>(op, m->lattice) || (long_z && (op == Op::heat || op == Op::wave));
    auto with_width = [&](auto w, auto off) {
        const Plan pl = star::make_plan(m->X, m->Y, m->Z, w(), 0, long_z);
        const dim3 grid = star::plan_grid(pl), block = star::plan_block(pl);
        if (m->lattice) f(pl, grid, block, w, std::integral_constant<int, 2>{}, off, lg<T>(m));
        else f(pl, grid, block, w, std::integral_constant<int, 3>{}, off, gg<T>(m));
    };
    // Offsets of one cell per thread: 32 bits in FP32, 64 in FP64 (us per acoustic
    // step of perturbed meshes with 64 / 32: FP32 48^3 6.30 / 5.87, 64^3 8.39 /
    // 8.08; FP64 48^3 9.08 / 9.57, 128^3 130 / 140).
    // (A plane's y- and z-faces are one row or column more than its cells.)
    const bool small = star::small_plane<T>(m->Y + 1, m->Z + 1);
    if (m->Z >= star::kWidth<T> && small && !one) {
        with_width(std::integral_constant<int, star::kWidth<T>>{}, uint32_t(0));
    } else {
        bool done = false;
        if constexpr (sizeof(T) == 4) {
            if (small) {
                with_width(std::integral_constant<int, 1>{}, uint32_t(0));
                done = true;
            }
        }
        if (!done) with_width(std::integral_constant<int, 1>{}, uint64_t(0));
    }
    CFD_HIP(hipGetLastError());
}

}  // namespace

template <class T>
void launch_grad_faces(const cfd_mesh_s* m, const void* phi, void* out, int mask, int wall, hipStream_t s) {
    with_faces<T>(m, Op::grad, [&](const Plan& pl, dim3 gr, dim3 bl, auto w, auto geo, auto off, const auto& g) {
        fgrad_k<T, decltype(w)::value, decltype(geo)::value, decltype(off)>
            <<<gr, bl, 0, s>>>(g, (const T*)phi, (T*)out, mask, wall, pl);
    });
}

template <class T> void launch_lapl_faces(const cfd_mesh_s* m, const void* phi, void* out, int mask, hipStream_t s) {
    with_faces<T>(m, Op::lapl, [&](const Plan& pl, dim3 gr, dim3 bl, auto w, auto geo, auto off, const auto& g) {
        flapl_k<T, decltype(w)::value, decltype(geo)::value, decltype(off)>
            <<<gr, bl, 0, s>>>(g, (const T*)phi, (T*)out, mask, pl);
    });
}

template <class T>
void launch_stab_faces(const cfd_mesh_s* m, const void* phi, void* out, int mask, void* scratch3, hipStream_t s) {
    T* gx = (T*)scratch3;
    T* gy = gx + m->N;
    T* gz = gy + m->N;
    with_faces<T>(m, Op::stab, [&](const Plan& pl, dim3 gr, dim3 bl, auto w, auto geo, auto off, const auto& g) {
        constexpr int W = decltype(w)::value, GEO = decltype(geo)::value;
        using O = decltype(off);
        fgrad3_k<T, W, GEO, O><<<gr, bl, 0, s>>>(g, (const T*)phi, gx, gy, gz, pl);
        CFD_HIP(hipGetLastError());
        fstab_k<T, W, GEO, O><<<gr, bl, 0, s>>>(g, gg<T>(m).len, (const T*)phi, gx, gy, gz, (T*)out, mask, pl);
    });
}

template <class T>
void launch_heat_faces(const cfd_mesh_s* m, const void* in, void* out, double alpha, const void* af, double dt,
                       hipStream_t s) {
    with_faces<T>(m, Op::heat, [&](const Plan& pl, dim3 gr, dim3 bl, auto w, auto geo, auto off, const auto& g) {
        constexpr int W = decltype(w)::value, GEO = decltype(geo)::value;
        using O = decltype(off);
        auto* kern = af ? fheat_k<T, W, GEO, O, true> : fheat_k<T, W, GEO, O, false>;
        kern<<<gr, bl, 0, s>>>(g, (const T*)in, (T*)out, T(alpha), (const T*)af, T(dt), pl);
    });
}

template <class T>
void launch_wave_faces(const cfd_mesh_s* m, void* const* in, void* const* out, double K, const void* Kf, double dt,
                       hipStream_t s) {
    with_faces<T>(m, Op::wave, [&](const Plan& pl, dim3 gr, dim3 bl, auto w, auto geo, auto off, const auto& g) {
        constexpr int W = decltype(w)::value, GEO = decltype(geo)::value;
        using O = decltype(off);
        fwave_vel_k<T, W, GEO, O><<<gr, bl, 0, s>>>(g, (const T*)in[0], (const T*)in[1], (const T*)in[2],
                                                 (const T*)in[3], (T*)out[1], (T*)out[2], (T*)out[3], T(dt), pl);
        CFD_HIP(hipGetLastError());
        auto* kern = Kf ? fwave_p_k<T, W, GEO, O, true> : fwave_p_k<T, W, GEO, O, false>;
        kern<<<gr, bl, 0, s>>>(g, (const T*)out[1], (const T*)out[2], (const T*)out[3], (const T*)in[0], (T*)out[0],
                               T(K), (const T*)Kf, T(dt), pl);
    });
}

#define CFD_INSTANTIATE(T)                                                                                           \
    template void launch_grad_faces<T>(const cfd_mesh_s*, const void*, void*, int, int, hipStream_t);               \
    template void launch_lapl_faces<T>(const cfd_mesh_s*, const void*, void*, int, hipStream_t);                    \
    template void launch_stab_faces<T>(const cfd_mesh_s*, const void*, void*, int, void*, hipStream_t);             \
    template void launch_heat_faces<T>(const cfd_mesh_s*, const void*, void*, double, const void*, double,          \
                                       hipStream_t);                                                                 \
    template void launch_wave_faces<T>(const cfd_mesh_s*, void* const*, void* const*, double, const void*, double,  \
                                       hipStream_t);
CFD_INSTANTIATE(float)
CFD_INSTANTIATE(double)

}  // namespace cfd
