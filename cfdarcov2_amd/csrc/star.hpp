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
// cells it shares with the unit before are computed twice with equal results.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace cfd {

namespace star {

template <class T, int W> struct VecOf {
    typedef T type __attribute__((ext_vector_type(W), aligned(sizeof(T))));
};
template <class T> struct VecOf<T, 1> { typedef T type; };

// W values at an element offset of a row-plane pointer.  The pointer is uniform
// over the workgroup and the offset 32 bits wide (star_fits), so an address is
// one register.
template <class T, int W> __device__ inline void load(const T* base, uint32_t off, T (&v)[W]) {
    using V = typename VecOf<T, W>::type;
    const V r = *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + size_t(off * uint32_t(sizeof(T))));
    if constexpr (W == 1) {
        v[0] = r;
    } else {
#pragma unroll
        for (int i = 0; i < W; ++i) v[i] = r[i];
    }
}
template <class T> __device__ inline T load1(const T* base, uint32_t off) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + size_t(off * uint32_t(sizeof(T))));
}
template <class T, int W> __device__ inline void store(T* base, uint32_t off, const T (&v)[W]) {
    using V = typename VecOf<T, W>::type;
    V r;
    if constexpr (W == 1) {
        r = v[0];
    } else {
#pragma unroll
        for (int i = 0; i < W; ++i) r[i] = v[i];
    }
    *reinterpret_cast<V*>(reinterpret_cast<char*>(base) + size_t(off * uint32_t(sizeof(T)))) = r;
}

// Launch geometry: workgroups of bx units x by rows of one x-plane, nzb x nyb
// of them per plane, X planes; the grid is padded to a multiple of 8 and each
// XCD (round-robin dispatch) takes a contiguous run, so the planes that a
// stencil shares are in its own L2.
struct Plan {
    int X, Y, Z;
    int bx, by, nzb, nyb;
    int blocks;  // workgroups with work, before the padding
};

inline Plan make_plan(int64_t X, int64_t Y, int64_t Z, int W) {
    Plan p{};
    p.X = int(X); p.Y = int(Y); p.Z = int(Z);
    const int units = int((Z + W - 1) / W);
    // 256 threads, fewer on meshes that would not give each CU a workgroup
    const int64_t all = X * Y * units;
    const int threads = all >= 256 * 256 ? 256 : all >= 128 * 256 ? 128 : 64;
    p.nzb = (units + threads - 1) / threads;
    p.bx = (units + p.nzb - 1) / p.nzb;
    p.by = threads / p.bx;
    if (p.by < 1) p.by = 1;
    if (p.by > Y) p.by = int(Y);
    p.nyb = int((Y + p.by - 1) / p.by);
    const int64_t n = int64_t(p.nzb) * p.nyb * X;
    CFD_REQUIRE(n < (int64_t(1) << 31) - 8, "star grid too large");
    p.blocks = int(n);
    return p;
}
inline dim3 plan_grid(const Plan& p) { return dim3(unsigned((p.blocks + 7) / 8 * 8)); }
inline dim3 plan_block(const Plan& p) { return dim3(unsigned(p.bx), unsigned(p.by)); }

// Whether a plane's byte offsets fit 32 bits
inline bool fits(int64_t Y, int64_t Z, size_t elem) { return Y * Z * int64_t(elem) < (int64_t(1) << 32); }

// The thread's place: plane x (uniform), row y, first cell z0; false without work.
template <int W> __device__ inline bool place(const Plan& p, int& x, int& y, int& z0) {
    const int lin = int((blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8);
    if (lin >= p.blocks) return false;
    const int row = p.nzb == 1 ? lin : lin / p.nzb;
    const int zb = p.nzb == 1 ? 0 : lin - row * p.nzb;
    x = row / p.nyb;
    y = (row - x * p.nyb) * p.by + int(threadIdx.y);
    const int zi = zb * p.bx + int(threadIdx.x);
    if (y >= p.Y || zi * W >= p.Z) return false;
    z0 = min(zi * W, p.Z - W);
    return true;
}

}  // namespace star

}  // namespace cfd
