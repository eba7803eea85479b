// Star form of the stencil kernels: no march and no LDS.  Each thread owns W
// consecutive z-cells of one row (16 bytes: 4 in FP32, 2 in FP64), loads every
// value its stencil reads straight from the caches with 16-byte accesses and
// recomputes what its neighbours also compute.  All loads are independent, so
// a launch lasts one memory round trip plus its arithmetic: the form for
// meshes whose fields stay in the caches, where a march along x would leave
// most of the chip idle.
//
// Any extents: rows need not start on 16-byte boundaries (global memory takes
// multi-word accesses at element alignment), and the last unit of a row whose
// extent is not a multiple of W is moved back to end with the row, so the
// cells it shares with the unit before are computed twice with equal results
// (a kernel that updates a field in place must leave them to one of the two).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "march.hpp"

namespace cfd {

namespace star {

template <class T, int W> struct VecOf {
    typedef T type __attribute__((ext_vector_type(W), aligned(sizeof(T))));
};

// Offsets within a plane.  The vector form keeps them in 32 bits (planes below
// 4 GiB), so an address is a base uniform over the workgroup plus one
// register; rows shorter than a vector and larger planes take W = 1 with 64
// (or with 32, where a kernel's launch chooses the type O of its offsets).
template <int W> struct OffOf { using type = uint32_t; };
template <> struct OffOf<1> { using type = uint64_t; };
template <int W> using Off = typename OffOf<W>::type;

template <class T, class O> __device__ inline T load1(const T* base, O off) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + O(off * O(sizeof(T))));
}
// W values at an element offset from a uniform pointer
template <class T, int W, class O> __device__ inline void load(const T* base, O off, T (&v)[W]) {
    if constexpr (W == 1) {
        v[0] = load1(base, off);
    } else {
        using V = typename VecOf<T, W>::type;
        const V r = *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + O(off * O(sizeof(T))));
#pragma unroll
        for (int i = 0; i < W; ++i) v[i] = r[i];
    }
}
template <class T, int W, class O> __device__ inline void store(T* base, O off, const T (&v)[W]) {
    char* const a = reinterpret_cast<char*>(base) + O(off * O(sizeof(T)));
    if constexpr (W == 1) {
        *reinterpret_cast<T*>(a) = v[0];
    } else {
        using V = typename VecOf<T, W>::type;
        V r;
#pragma unroll
        for (int i = 0; i < W; ++i) r[i] = v[i];
        *reinterpret_cast<V*>(a) = r;
    }
}

// Division of 0 <= k < 2^31 by a constant n >= 1: the product with the
// reciprocal rounded up to 32 significant bits, exact for these k (the
// hardware has no integer division, and a workgroup's first loads wait for it).
struct Div {
    uint32_t n, m, s;  // k / n = (k m) >> (31 + s)
    __device__ int operator()(int k) const { return int(__umulhi(uint32_t(k) << 1, m) >> s); }
};
inline Div make_div(int64_t n) {
    Div d{};
    d.n = uint32_t(n);
    while ((int64_t(1) << d.s) < n) ++d.s;
    d.m = uint32_t(((uint64_t(1) << (31 + d.s)) + uint64_t(n) - 1) / uint64_t(n));
    return d;
}

// Launch geometry: workgroups of bx units x by rows of one x-plane, nzb x nyb
// of them per plane, X planes; the grid is padded to a multiple of 8 and each
// XCD (round-robin dispatch) takes a contiguous run, so what neighbouring
// workgroups share is in its own L2.
struct Plan {
    int X, Y, Z;
    int bx, by, nzb, nyb;
    int blocks;  // workgroups with work, before the padding
    int cut;     // the axis whose blocks the runs divide (outermost in the run)
    Div d0, d1;  // by the number of innermost blocks, and of the next
};

// The runs divide x.  Slabs of a few planes share most of what they read with
// the next XCD's, so where y is at least four times as long the runs divide y
// (us, cut in x / y: acoustic step FP64 64x256x256 61.3 / 43.0, 40x1000x40
// 22.1 / 19.4, FP32 20x300x300 15.3 / 13.1; perturbed heat step FP64 40x1000x40
// 45.6 / 35.0; at twice as long neither is better: 64x128x128 FP64 14.2 / 13.9,
// perturbed 57.4 / 58.0).  z only on demand (long_z: its columns make a row's
// halo, so only face arrays that leave the cache repay it).
inline Plan make_plan(int64_t X, int64_t Y, int64_t Z, int W, int threads = 0, bool long_z = false) {
    Plan p{};
    p.X = int(X); p.Y = int(Y); p.Z = int(Z);
    const int units = int((Z + W - 1) / W);
    if (!threads) {  // 256 threads, fewer on meshes that would not give each CU a workgroup
        const int64_t all = X * Y * units;
        threads = all >= 256 * 256 ? 256 : all >= 128 * 256 ? 128 : 64;
    }
    auto split = [&](int nzb) {
        p.nzb = nzb;
        p.bx = (units + nzb - 1) / nzb;
        p.by = int(std::min<int64_t>(threads / p.bx, Y));
        if (p.by < 1) p.by = 1;
    };
    const int columns = (units + threads - 1) / threads;
    split(columns);
    // A row just over half a workgroup would leave the rest of it idle: three
    // times the columns then (FP64 z = 300, 150 units: stabilisation of 300^3 201
    // us as 150 threads, 185 as 5 rows of 50; 160^3 one cell per thread, lattice
    // heat step FP64 31.0 / 26.5).
    if (threads == 256 && p.by == 1 && Y >= 4 && 3 * p.bx < 2 * threads) split(3 * columns);
    if (long_z && units >= 64) {
        split(std::max(8, columns));  // at least one column per XCD; more have more halo (60x60x2000 FP64 241 / 216)
        p.cut = 2;
    } else {
        p.cut = Y >= 4 * X ? 1 : 0;
    }
    p.nyb = int((Y + p.by - 1) / p.by);
    const int64_t n = int64_t(p.nzb) * p.nyb * X;
    CFD_REQUIRE(n < (int64_t(1) << 31) - 8, "star grid too large");
    p.blocks = int(n);
    p.d0 = make_div(p.cut == 2 ? p.nyb : p.nzb);
    p.d1 = make_div(p.cut == 0 ? p.nyb : p.X);
    return p;
}
inline dim3 plan_grid(const Plan& p) { return dim3(unsigned((p.blocks + 7) / 8 * 8)); }
inline dim3 plan_block(const Plan& p) { return dim3(unsigned(p.bx), unsigned(p.by)); }

// Whether rows and planes suit the vector form of T
template <class T> constexpr int kWidth = 16 / int(sizeof(T));
template <class T> inline bool small_plane(int64_t Y, int64_t Z) {  // 32-bit offsets reach all of it
    return Y * Z * int64_t(sizeof(T)) < (int64_t(1) << 32);
}
template <class T> inline bool vector_form(int64_t Y, int64_t Z) { return Z >= kWidth<T> && small_plane<T>(Y, Z); }

// Whether a step of a mesh of this size is better with one cell per thread: a
// launch then lasts about as long as one wavefront's chain of operations, and
// the chain of W cells is longer than the chip needs to be filled.  Kernel times
// (steps replayed from a graph; a run launched step by step takes the host's 3
// to 4 us per launch where that is longer), us with one cell per thread / with
// vectors: acoustic step FP32 16^3 2.5 / 3.0, 48^3 2.9 / 3.3, 80^3 5.3 / 5.9,
// 100^3 8.5 / 7.9; FP64 16^3 2.5 / 3.2, 48^3 4.1 / 4.1, 56^3 5.7 / 4.8; transposed
// step FP32 48^3 4.8 / 5.5, 72^3 6.8 / 6.7, FP64 48^3 5.8 / 5.6.
template <class T> inline bool narrow(int64_t cells) {
    return cells <= (sizeof(T) == 4 ? int64_t(1) << 19 : int64_t(1) << 17);
}

// A thread's place: plane x (uniform), row y, first cell z0.  The first `skip`
// of its cells belong to the unit before as well.
struct Place {
    int x, y, z0, skip;
};
// The place of thread (tx, ty) of block `b` of a grid of `padded` blocks (a
// multiple of 8, as plan_grid's); false without work.
template <int W> __device__ inline bool place_at(const Plan& p, int b, int padded, int tx, int ty, Place& q) {
    const int lin = (b % 8) * (padded / 8) + b / 8;
    if (lin >= p.blocks) return false;
    // blocks of the run's cut axis outermost: (x, y, z), (y, x, z) or (z, x, y)
    const int row = p.d0(lin), in = lin - row * int(p.d0.n);
    const int out = p.d1(row), mid = row - out * int(p.d1.n);
    int zb = in, yb = mid;
    q.x = out;
    if (p.cut) {
        q.x = mid;
        yb = p.cut == 1 ? out : in;
        if (p.cut == 2) zb = out;
    }
    q.y = yb * p.by + ty;
    const int zi = zb * p.bx + tx;
    if (ty >= p.by || q.y >= p.Y || zi * W >= p.Z) return false;
    q.z0 = min(zi * W, p.Z - W);
    q.skip = zi * W - q.z0;
    return true;
}
template <int W> __device__ inline bool place(const Plan& p, Place& q) {
    return place_at<W>(p, int(blockIdx.x), int(gridDim.x), int(threadIdx.x), int(threadIdx.y), q);
}

// Element offsets of a thread's cells and of their six neighbours, clamped to
// the mesh: a neighbour beyond a wall is the cell itself (the reference rule).
template <int W, class O = Off<W>> struct Offsets {
    int64_t x0, xm1, xp1;      // planes
    O o0, ym1, yp1, zm1, zp1;  // within a plane: the W cells, rows y-1 and y+1, cells z0-1 and z0+W
};
template <int W, class O = Off<W>> __device__ inline Offsets<W, O> offsets(const Plan& p, const Place& q) {
    const int x = q.x, y = q.y, z0 = q.z0;
    Offsets<W, O> o;
    const int64_t SX = int64_t(p.Y) * p.Z;
    o.x0 = int64_t(x) * SX;
    o.xm1 = x >= 1 ? o.x0 - SX : o.x0;
    o.xp1 = x + 1 < p.X ? o.x0 + SX : o.x0;
    const O uz = O(p.Z);
    o.o0 = O(y) * uz + O(z0);
    o.ym1 = y >= 1 ? o.o0 - uz : o.o0;
    o.yp1 = y + 1 < p.Y ? o.o0 + uz : o.o0;
    o.zm1 = z0 >= 1 ? o.o0 - 1 : o.o0;
    const O last = o.o0 + O(W - 1);
    o.zp1 = z0 + W < p.Z ? last + 1 : last;
    return o;
}

// The values of a field that a seven-point stencil of W cells reads; r holds
// the row with one cell on each side (r[j] is cell z0 - 1 + j).
template <class T, int W> struct Star7 {
    T xm[W], xp[W], ym[W], yp[W], r[W + 2];
    __device__ T c(int i) const { return r[i + 1]; }
};
template <class T, int W, class O>
__device__ inline Star7<T, W> load7(const T* __restrict__ f, const Offsets<W, O>& o) {
    Star7<T, W> s;
    T c[W];
    const T* const f0 = f + o.x0;
    load<T, W>(f0, o.o0, c);
    load<T, W>(f + o.xm1, o.o0, s.xm);
    load<T, W>(f + o.xp1, o.o0, s.xp);
    load<T, W>(f0, o.ym1, s.ym);
    load<T, W>(f0, o.yp1, s.yp);
    s.r[0] = load1(f0, o.zm1);
    s.r[W + 1] = load1(f0, o.zp1);
#pragma unroll
    for (int i = 0; i < W; ++i) s.r[i + 1] = c[i];
    return s;
}

// The same for an operator over the axes of `mask`: the others' neighbours are
// not loaded and read as the cell itself.
template <class T, int W, class O>
__device__ inline Star7<T, W> load_axes(const T* __restrict__ f, const Offsets<W, O>& o, int mask) {
    Star7<T, W> s;
    T c[W];
    const T* const f0 = f + o.x0;
    const bool x = mask & 1, y = mask & 2, z = mask & 4;
    load<T, W>(f0, o.o0, c);
    if (x) {
        load<T, W>(f + o.xm1, o.o0, s.xm);
        load<T, W>(f + o.xp1, o.o0, s.xp);
    }
    if (y) {
        load<T, W>(f0, o.ym1, s.ym);
        load<T, W>(f0, o.yp1, s.yp);
    }
    if (z) {
        s.r[0] = load1(f0, o.zm1);
        s.r[W + 1] = load1(f0, o.zp1);
    }
#pragma unroll
    for (int i = 0; i < W; ++i) {
        s.r[i + 1] = c[i];
        if (!x) s.xm[i] = s.xp[i] = c[i];
        if (!y) s.ym[i] = s.yp[i] = c[i];
    }
    if (!z) {
        s.r[0] = c[0];
        s.r[W + 1] = c[W - 1];
    }
    return s;
}

// Value across the lower or upper face of cell i along axis a
template <class T, int W> __device__ inline T face_nb(const Star7<T, W>& s, int a, bool upper, int i) {
    if (a == 0) return upper ? s.xp[i] : s.xm[i];
    if (a == 1) return upper ? s.yp[i] : s.ym[i];
    return upper ? s.r[i + 2] : s.r[i];
}

// Laplacian of cell i of a uniform mesh over the selected axes, from 0 in the
// order x, y, z (a wall's neighbour is the cell itself, so its difference is an
// exact zero whatever the wall's alpha_d)
template <class T, int W, bool PW>
__device__ inline T lapl_uniform(const UniformGeo<T>& g, const Star7<T, W>& s, int mask, int i) {
    const VolDiv<T, PW> Vd{g.vol, g.inv_vol};
    const T pc = s.c(i);
    T res = T(0);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (!(mask & (1 << a))) continue;
        const T s_lo = (-pc + face_nb(s, a, false, i)) * g.alpha[a];
        const T s_hi = (-pc + face_nb(s, a, true, i)) * g.alpha[a];
        res = res + Vd(s_lo * g.area[a] + s_hi * g.area[a]);
    }
    return res;
}

// Geometry of a thread's cells on an axis-aligned lattice (LatticeGeo).
template <class T, int W> struct LatticeCells {
    T wx, wy, wz[W];
    T V[W];
    T ax[2], ay[2], az[W + 1];  // alpha_d of the lower and upper faces (az: of the W + 1 z-faces)
    __device__ T area(int a, int i) const { return a == 0 ? wy * wz[i] : a == 1 ? wx * wz[i] : wx * wy; }
};
template <class T, int W, bool ALPHA, class O>
__device__ inline LatticeCells<T, W> load_lattice(const LatticeGeo<T>& g, const Offsets<W, O>& o, const Place& q) {
    const int x = q.x, y = q.y, z0 = q.z0;
    LatticeCells<T, W> c;
    load<T, W>(g.vol + o.x0, o.o0, c.V);
    c.wx = g.w[0][x];
    c.wy = g.w[1][y];
    load<T, W>(g.w[2], O(z0), c.wz);
    if constexpr (ALPHA) {
        T lo[W];
        c.ax[0] = g.alpha[0][x];
        c.ax[1] = g.alpha[0][x + 1];
        c.ay[0] = g.alpha[1][y];
        c.ay[1] = g.alpha[1][y + 1];
        load<T, W>(g.alpha[2], O(z0), lo);
#pragma unroll
        for (int i = 0; i < W; ++i) c.az[i] = lo[i];
        c.az[W] = g.alpha[2][z0 + W];
    }
    return c;
}

// Six face values of a cell, lower and upper per axis
template <class T> struct Faces {
    T lo[3], hi[3];
};

// f * 0, which is not 0 where f is infinite or NaN
template <class T> __device__ inline T zero_of(T lo, T hi) {
    if constexpr (sizeof(T) == 4) return __builtin_fmaf(hi, T(0), lo * T(0));
    else return __builtin_fma(hi, T(0), lo * T(0));
}

// Gauss sum of component a on a lattice, outward (the gradient's) or axis
// normals (the Laplacian's).  The reference sums all six faces, the other
// axes' with a zero normal component: they add nothing to a finite sum and
// make it NaN where a face value is not finite.
template <class T, int W, bool OUTWARD>
__device__ inline T lattice_gauss(const LatticeCells<T, W>& c, const Faces<T>& f, int a, int i) {
    const int b = a == 0 ? 1 : 0, d = a == 2 ? 1 : 2;
    const T A = c.area(a, i);
    const T zeros = zero_of(f.lo[b], f.hi[b]) + zero_of(f.lo[d], f.hi[d]);
    T acc = T(0) + (OUTWARD ? -f.lo[a] : f.lo[a]) * A;
    acc = acc + f.hi[a] * A;
    acc = acc + zeros;
    return acc / c.V[i];
}

}  // namespace star

}  // namespace cfd
