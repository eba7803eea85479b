// Compressible Euler with a Rusanov face flux on the hex mesh (no reference
// counterpart; the reference's Sod driver, examples/main_3d_sod_shock.cpp:150-167,
// runs a central predictor with stabilisation instead).
//
// State: five SoA fields (rho, rho u, rho v, rho w, E).  One thread per cell;
// each thread rebuilds the primitive state of itself and its six neighbours,
// evaluates the six face fluxes in the lower-cell -> upper-cell orientation (so
// both cells of a face compute bit-identical fluxes and the scheme stays
// conservative without scatter or atomics on the fields), and updates
//   U <- U - (dt * net) * (1 / V),  net = ((Gx+ - Gx-) + (Gy+ - Gy-)) + (Gz+ - Gz-),
// every product that is added to something rounded once as a fused
// multiply-add, in the same nesting as the oracle's stepper.
//
// Time step, all on the device: the step kernel reads dt from a rotating slot,
// and from the cell's new state computes V / sum_f A_f (|u.n_f| + a), reduces
// the block minimum and folds it into the next slot with one atomic minimum
// per block.  A third slot is reset to +inf for the step after, so the loop
// needs no host round trip.
#include <hip/hip_runtime.h>

#include <cmath>
#include <limits>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "hexmesh.hpp"
#include "kernels.hpp"
#include "umesh.hpp"

namespace cfd {

template <class T> using Bits = std::conditional_t<sizeof(T) == 4, unsigned int, unsigned long long>;

__device__ inline float from_bits(unsigned int b) { return __uint_as_float(b); }
__device__ inline double from_bits(unsigned long long b) { return __longlong_as_double((long long)b); }
__device__ inline unsigned int to_bits(float v) { return __float_as_uint(v); }
__device__ inline unsigned long long to_bits(double v) { return (unsigned long long)__double_as_longlong(v); }
template <class T> __device__ inline Bits<T> inf_bits() { return to_bits(std::numeric_limits<T>::infinity()); }

template <class T> struct EIn { const T* u[5]; };
template <class T> struct EOut { T* u[5]; };

template <class T> struct Prim { T ux, uy, uz, p, a; };

// the rotating dt sets of one step
template <class T> struct EulerSlots {
    const Bits<T>* cur;
    Bits<T>* next;
    Bits<T>* reset;
};

// a * b + c rounded once (the fused multiply-add the scheme's rounding is
// defined with; the oracle uses std::fma in the same places)
template <class T> __device__ inline T fmul_add(T a, T b, T c) {
    if constexpr (sizeof(T) == 4) return __builtin_fmaf(a, b, c);
    else return __builtin_fma(a, b, c);
}

// u . n of a velocity and a face normal
template <class T> __device__ inline T un_of(T ux, T uy, T uz, T nx, T ny, T nz) {
    return fmul_add(uz, nz, fmul_add(uy, ny, ux * nx));
}

// Primitive state with one division: the reciprocal density multiplies the
// momenta and the sound-speed argument (the oracle's euler_prim, operation
// for operation).
template <class T> __device__ inline Prim<T> prim(T gamma, const T U[5]) {
    Prim<T> q;
    const T ir = T(1) / U[0];
    q.ux = U[1] * ir;
    q.uy = U[2] * ir;
    q.uz = U[3] * ir;
    const T q2 = fmul_add(q.uz, q.uz, fmul_add(q.uy, q.uy, q.ux * q.ux));
    q.p = (gamma - T(1)) * fmul_add(-(T(0.5) * U[0]), q2, U[4]);
    q.a = sqrt((gamma * q.p) * ir);
    return q;
}

// Rusanov flux through a face of unit +axis normal n and area A, L = lower cell
// (the oracle's rusanov_flux, operation for operation)
template <class T>
__device__ inline void rusanov(const T UL[5], const Prim<T>& L, const T UR[5], const Prim<T>& R, T nx, T ny, T nz,
                               T A, T G[5]) {
    const T unL = un_of(L.ux, L.uy, L.uz, nx, ny, nz);
    const T unR = un_of(R.ux, R.uy, R.uz, nx, ny, nz);
    const T FL[5] = {UL[0] * unL, fmul_add(UL[1], unL, L.p * nx), fmul_add(UL[2], unL, L.p * ny),
                     fmul_add(UL[3], unL, L.p * nz), (UL[4] + L.p) * unL};
    const T FR[5] = {UR[0] * unR, fmul_add(UR[1], unR, R.p * nx), fmul_add(UR[2], unR, R.p * ny),
                     fmul_add(UR[3], unR, R.p * nz), (UR[4] + R.p) * unR};
    const T lam = fmax(fabs(unL) + L.a, fabs(unR) + R.a);
    const T hA = T(0.5) * A;
#pragma unroll
    for (int k = 0; k < 5; ++k) G[k] = fmul_add(-lam, UR[k] - UL[k], FL[k] + FR[k]) * hA;
}

// family and family-local index of local face fc of cell (x, y, z)
template <class T>
__device__ inline int64_t fv_face(const FvGeo<T>& g, int64_t x, int64_t y, int64_t z, int fc, int& fam) {
    switch (fc) {
        case 0: fam = 0; return x * g.Y * (g.Z + 1) + y * (g.Z + 1) + z;
        case 1: fam = 0; return x * g.Y * (g.Z + 1) + y * (g.Z + 1) + z + 1;
        case 2: fam = 1; return x * (g.Y + 1) * g.Z + y * g.Z + z;
        case 3: fam = 1; return x * (g.Y + 1) * g.Z + (y + 1) * g.Z + z;
        case 4: fam = 2; return x * g.Y * g.Z + y * g.Z + z;
        default: fam = 2; return (x + 1) * g.Y * g.Z + y * g.Z + z;
    }
}

// V / sum over fc = 0..5 of A_f (|u.n_f| + a)
template <class T>
__device__ inline T local_dt(const FvGeo<T>& g, int64_t x, int64_t y, int64_t z, int64_t c, const Prim<T>& q) {
    T s = T(0);
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) {
        int fam;
        const int64_t f = fv_face(g, x, y, z, fc, fam);
        const T un = un_of(q.ux, q.uy, q.uz, g.n[fam][0][f], g.n[fam][1][f], g.n[fam][2][f]);
        s = fmul_add(g.A[fam][f], fabs(un) + q.a, s);
    }
    return g.vol[c] / s;
}

// The same value from the six faces' geometry already at hand, in the local
// face order z-, z+, y-, y+, x-, x+ (f[fc] = {nx, ny, nz, A})
template <class T> __device__ inline T local_dt_faces(T V, const Prim<T>& q, const T (&f)[6][4]) {
    T s = T(0);
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) {
        const T un = un_of(q.ux, q.uy, q.uz, f[fc][0], f[fc][1], f[fc][2]);
        s = fmul_add(f[fc][3], fabs(un) + q.a, s);
    }
    return V / s;
}

// The next time step is the minimum over all cells, folded with atomics.  All
// workgroups on one address would queue there (12 ns each, measured: 100 us
// for the 8,192 workgroups of a per-cell kernel at 512x64x64), so a slot is a
// set of kDtSlots values on cache lines of their own, workgroups spread over
// them, and every wave that needs the minimum reads the whole set, one value
// per lane.  Non-negative floats order like their bit patterns.
constexpr int kDtSlots = 64, kDtStride = 32;  // values, elements between them
constexpr int kDtSet = kDtSlots * kDtStride;

// minimum over the block (64 x blockDim.y threads, one wave per y row), folded
// into the set by thread (0, 0) with one atomic per block
template <class T> __device__ inline void block_min_into(T v, Bits<T>* set) {
    __shared__ T red[16];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    const int lane = threadIdx.x, wave = threadIdx.y;
    if (lane == 0) red[wave] = v;
    __syncthreads();
    if (lane == 0 && wave == 0) {
        T m = red[0];
        for (int w = 1; w < int(blockDim.y); ++w) m = fmin(m, red[w]);
        const unsigned wg = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        if (m < std::numeric_limits<T>::infinity()) atomicMin(set + (wg % kDtSlots) * kDtStride, to_bits(m));
    }
}

// the minimum of a set (every lane of a wave takes part)
template <class T> __device__ inline T set_min(const Bits<T>* set) {
    Bits<T> b = set[int(threadIdx.x) * kDtStride];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const Bits<T> c = to_bits(__shfl_xor(from_bits(b), o, 64));
        b = c < b ? c : b;
    }
    return from_bits(b);
}

// thread (0..63, 0) of the first workgroup clears a set
template <class T> __device__ inline void set_reset(Bits<T>* set) { set[int(threadIdx.x) * kDtStride] = inf_bits<T>(); }

template <class T>
__global__ void __launch_bounds__(256) euler_dt_k(FvGeo<T> g, EIn<T> in, T gamma, Bits<T>* slot) {
    const int64_t z = int64_t(blockIdx.x) * 64 + threadIdx.x;
    const int64_t y = int64_t(blockIdx.y) * 4 + threadIdx.y;
    const int64_t x = blockIdx.z;
    T loc = std::numeric_limits<T>::infinity();
    if (z < g.Z && y < g.Y) {
        const int64_t c = (x * g.Y + y) * g.Z + z;
        T U[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) U[k] = in.u[k][c];
        loc = local_dt(g, x, y, z, c, prim(gamma, U));
    }
    block_min_into(loc, slot);
}

template <class T>
__global__ void __launch_bounds__(256) euler_step_k(FvGeo<T> g, EIn<T> in, EOut<T> out, T gamma, T cfl,
                                                   const Bits<T>* dt_cur, Bits<T>* dt_next, Bits<T>* dt_reset,
                                                   T* dt_hist, int64_t step) {
    const int64_t z = int64_t(blockIdx.x) * 64 + threadIdx.x;
    const int64_t y = int64_t(blockIdx.y) * 4 + threadIdx.y;
    const int64_t x = blockIdx.z;
    const T dt = cfl * set_min<T>(dt_cur);
    if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.y == 0) {
        set_reset<T>(dt_reset);
        if (dt_hist && threadIdx.x == 0) dt_hist[step] = dt;
    }
    T loc = std::numeric_limits<T>::infinity();
    if (z < g.Z && y < g.Y) {
        const int64_t c = (x * g.Y + y) * g.Z + z;
        T Ui[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) Ui[k] = in.u[k][c];
        const Prim<T> qi = prim(gamma, Ui);
        const int64_t crd[3] = {z, y, x};           // fc >> 1 = 0 z, 1 y, 2 x
        const int64_t ext[3] = {g.Z, g.Y, g.X};
        const int64_t str[3] = {1, g.Z, g.Y * g.Z};
        T net[5] = {T(0), T(0), T(0), T(0), T(0)};
        // axis pairs in the order x, y, z: net = ((x+ - x-) + (y+ - y-)) + (z+ - z-)
#pragma unroll
        for (int pair = 2; pair >= 0; --pair) {
            T Gp[2][5];
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const int fc = 2 * pair + side;
                const bool upper = side == 1;
                const bool wall = upper ? crd[pair] == ext[pair] - 1 : crd[pair] == 0;
                T Un[5];
                if (wall) {
#pragma unroll
                    for (int k = 0; k < 5; ++k) Un[k] = Ui[k];
                    Un[3 - pair] = -Ui[3 - pair];
                } else {
                    const int64_t nb = upper ? c + str[pair] : c - str[pair];
#pragma unroll
                    for (int k = 0; k < 5; ++k) Un[k] = in.u[k][nb];
                }
                const Prim<T> qn = prim(gamma, Un);
                int fam;
                const int64_t f = fv_face(g, x, y, z, fc, fam);
                const T nx = g.n[fam][0][f], ny = g.n[fam][1][f], nz = g.n[fam][2][f], A = g.A[fam][f];
                if (upper) rusanov(Ui, qi, Un, qn, nx, ny, nz, A, Gp[side]);
                else rusanov(Un, qn, Ui, qi, nx, ny, nz, A, Gp[side]);
            }
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const T d = Gp[1][k] - Gp[0][k];
                net[k] = pair == 2 ? d : net[k] + d;
            }
        }
        const T V = g.vol[c];
        const T iV = T(1) / V;
        T Un[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            Un[k] = fmul_add(-(dt * net[k]), iV, Ui[k]);
            out.u[k][c] = Un[k];
        }
        loc = local_dt(g, x, y, z, c, prim(gamma, Un));
    }
    block_min_into(loc, dt_next);
}

// The same step as a 2.5D march: a workgroup owns TY rows x 64 z-columns and
// walks `L` x-planes.  Each cell's state and primitives go to LDS once per
// plane (with a one-cell y/z halo loaded by edge threads), the y/z face fluxes
// read the neighbours from there, and the x-face flux between planes x and x+1
// is carried in registers to the next plane, so each cell converts its state
// to primitives once instead of seven times.  Every face flux is evaluated with
// the lower cell as L, exactly as in euler_step_k, so both give the same bits.
template <class T> __device__ inline void mirror(const T U[5], const Prim<T>& q, int axis, T Um[5], Prim<T>& qm) {
#pragma unroll
    for (int k = 0; k < 5; ++k) Um[k] = U[k];
    Um[1 + axis] = -U[1 + axis];  // axis 0 x, 1 y, 2 z
    qm = q;
    if (axis == 0) qm.ux = -q.ux;
    else if (axis == 1) qm.uy = -q.uy;
    else qm.uz = -q.uz;
}

template <class T, int TY>
__global__ void __launch_bounds__(64 * TY) euler_march_k(FvGeo<T> g, EIn<T> in, EOut<T> out, T gamma, T cfl,
                                                        const Bits<T>* dt_cur, Bits<T>* dt_next, Bits<T>* dt_reset,
                                                        T* dt_hist, int64_t step, int L, int nzt, int nyt) {
    constexpr int TZ = 64;
    constexpr int PZ = TZ + 2;
    constexpr int PS = (TY + 2) * PZ;
    __shared__ T sh[2][10][PS];  // U0..U4, ux, uy, uz, p, a per slot, double-buffered

    const int64_t X = g.X, Y = g.Y, Z = g.Z, SX = Y * Z;
    const int64_t lin = blockIdx.x;
    const int64_t zt = lin % nzt;
    const int64_t yt = (lin / nzt) % nyt;
    const int64_t xc = lin / (int64_t(nzt) * nyt);
    const int lz = threadIdx.x, ly = threadIdx.y;
    const int64_t z = zt * TZ + lz, y = yt * TY + ly;
    const bool valid = z < Z && y < Y;
    const int64_t col = valid ? y * Z + z : 0;
    const int64_t x0 = xc * L;
    const int64_t x1 = (x0 + L < X) ? x0 + L : X;
    const T dt = cfl * set_min<T>(dt_cur);
    if (lin == 0 && ly == 0) {
        set_reset<T>(dt_reset);
        if (dt_hist && lz == 0) dt_hist[step] = dt;
    }
    const int own = (ly + 1) * PZ + (lz + 1);
    // halo cells: row -1 (ly 0) / row TY (ly 1) at this column, column -1
    // (lane 0) / column 64 (lane 63) at this row; -1 where outside the domain
    int64_t hy_col = -1, hz_col = -1;
    int hy_slot = 0, hz_slot = 0;
    if (ly < 2 && z < Z) {
        const int64_t yy = ly == 0 ? yt * TY - 1 : yt * TY + TY;
        if (yy >= 0 && yy < Y) {
            hy_col = yy * Z + z;
            hy_slot = (ly == 0 ? 0 : TY + 1) * PZ + (lz + 1);
        }
    }
    if ((lz == 0 || lz == TZ - 1) && y < Y) {
        const int64_t zz = lz == 0 ? zt * TZ - 1 : zt * TZ + TZ;
        if (zz >= 0 && zz < Z) {
            hz_col = y * Z + zz;
            hz_slot = (ly + 1) * PZ + (lz == 0 ? 0 : TZ + 1);
        }
    }
    // Addresses: a pointer uniform over the workgroup (the field plus the
    // plane's offset) and a 32-bit byte offset per lane (the launcher checks
    // that a plane fits 32-bit byte offsets)
    auto at = [](const T* base, uint32_t boff) {
        return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + boff);
    };
    const uint32_t bcol = uint32_t(col) * uint32_t(sizeof(T));
    const uint32_t bzf = valid ? uint32_t(y * (Z + 1) + z) * uint32_t(sizeof(T)) : 0;  // z-face of (y, z)
    auto load = [&](int64_t plane, uint32_t boff, T U[5]) {
#pragma unroll
        for (int k = 0; k < 5; ++k) U[k] = at(in.u[k] + plane * SX, boff);
    };
    auto put = [&](T* const* S, int slot, const T U[5], const Prim<T>& q) {
#pragma unroll
        for (int k = 0; k < 5; ++k) S[k][slot] = U[k];
        S[5][slot] = q.ux; S[6][slot] = q.uy; S[7][slot] = q.uz; S[8][slot] = q.p; S[9][slot] = q.a;
    };
    auto get = [&](T* const* S, int slot, T U[5], Prim<T>& q) {
#pragma unroll
        for (int k = 0; k < 5; ++k) U[k] = S[k][slot];
        q.ux = S[5][slot]; q.uy = S[6][slot]; q.uz = S[7][slot]; q.p = S[8][slot]; q.a = S[9][slot];
    };
    // face geometry: family fam, faces from `first` (uniform), lane offset boff
    auto face4 = [&](int fam, int64_t first, uint32_t boff, T (&o)[4]) {
        o[0] = at(g.n[fam][0] + first, boff);
        o[1] = at(g.n[fam][1] + first, boff);
        o[2] = at(g.n[fam][2] + first, boff);
        o[3] = at(g.A[fam] + first, boff);
    };

    T Uc[5] = {}, Un[5] = {}, Gxl[5] = {};
    T fg[6][4] = {};  // this cell's face geometry in local face order; fg[4] carried along x
    Prim<T> qc{}, qn{};
    if (valid) {  // warm-up: state of plane x0 and the flux through its lower x-face
        load(x0, bcol, Uc);
        qc = prim(gamma, Uc);
        face4(2, x0 * SX, bcol, fg[4]);
        T Ul[5];
        Prim<T> ql;
        if (x0 == 0) mirror(Uc, qc, 0, Ul, ql);
        else {
            load(x0 - 1, bcol, Ul);
            ql = prim(gamma, Ul);
        }
        rusanov(Ul, ql, Uc, qc, fg[4][0], fg[4][1], fg[4][2], fg[4][3], Gxl);
    }
    T loc = std::numeric_limits<T>::infinity();
    // Everything a plane reads is loaded one plane ahead (the state of plane
    // x + 1, the halo cells, the face geometry), so no plane waits for a load
    // that it has just issued.
    const uint32_t bhy = hy_col >= 0 ? uint32_t(hy_col) * uint32_t(sizeof(T)) : 0;
    const uint32_t bhz = hz_col >= 0 ? uint32_t(hz_col) * uint32_t(sizeof(T)) : 0;
    T Uy[5] = {}, Uz[5] = {}, Uf[5] = {}, fn[6][4] = {}, Vn = T(1);
    auto fetch = [&](int64_t x) {
        if (valid && x + 1 < X) load(x + 1, bcol, Uf);
        if (hy_col >= 0) load(x, bhy, Uy);
        if (hz_col >= 0) load(x, bhz, Uz);
        if (valid) {
            face4(2, (x + 1) * SX, bcol, fn[5]);
            face4(1, x * (Y + 1) * Z, bcol, fn[2]);
            face4(1, x * (Y + 1) * Z + Z, bcol, fn[3]);
            const int64_t fz = x * Y * (Z + 1);
            face4(0, fz, bzf, fn[0]);
            face4(0, fz + 1, bzf, fn[1]);
            Vn = at(g.vol + x * SX, bcol);
        }
    };
    if (x0 < x1) fetch(x0);
    int b = 0;
#pragma unroll 1
    for (int64_t x = x0; x < x1; ++x, b ^= 1) {
        T* S[10];
#pragma unroll
        for (int k = 0; k < 10; ++k) S[k] = sh[b][k];
        const T V = Vn;
#pragma unroll
        for (int f = 0; f < 6; ++f)
            if (f != 4)
#pragma unroll
                for (int k = 0; k < 4; ++k) fg[f][k] = fn[f][k];
#pragma unroll
        for (int k = 0; k < 5; ++k) Un[k] = Uf[k];
        if (valid && x + 1 < X) qn = prim(gamma, Un);
        if (hy_col >= 0) put(S, hy_slot, Uy, prim(gamma, Uy));
        if (hz_col >= 0) put(S, hz_slot, Uz, prim(gamma, Uz));
        if (valid) put(S, own, Uc, qc);
        if (x + 1 < x1) fetch(x + 1);
        __syncthreads();
        if (valid) {
            T Um[5], G1[5], G2[5], acc[5];
            Prim<T> qm;
            // net = ((Gx+ - Gx-) + (Gy+ - Gy-)) + (Gz+ - Gz-), accumulated one
            // axis at a time; the upper x flux becomes the next plane's lower.
            // The six faces' geometry stays in registers for the next dt.
            if (x == X - 1) {
                mirror(Uc, qc, 0, Um, qm);
                rusanov(Uc, qc, Um, qm, fg[5][0], fg[5][1], fg[5][2], fg[5][3], G1);
            } else {
                rusanov(Uc, qc, Un, qn, fg[5][0], fg[5][1], fg[5][2], fg[5][3], G1);
            }
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                acc[k] = G1[k] - Gxl[k];
                Gxl[k] = G1[k];
            }
            // y faces
            if (y == 0) mirror(Uc, qc, 1, Um, qm);
            else get(S, own - PZ, Um, qm);
            rusanov(Um, qm, Uc, qc, fg[2][0], fg[2][1], fg[2][2], fg[2][3], G1);
            if (y == Y - 1) mirror(Uc, qc, 1, Um, qm);
            else get(S, own + PZ, Um, qm);
            rusanov(Uc, qc, Um, qm, fg[3][0], fg[3][1], fg[3][2], fg[3][3], G2);
#pragma unroll
            for (int k = 0; k < 5; ++k) acc[k] = acc[k] + (G2[k] - G1[k]);
            // z faces
            if (z == 0) mirror(Uc, qc, 2, Um, qm);
            else get(S, own - 1, Um, qm);
            rusanov(Um, qm, Uc, qc, fg[0][0], fg[0][1], fg[0][2], fg[0][3], G1);
            if (z == Z - 1) mirror(Uc, qc, 2, Um, qm);
            else get(S, own + 1, Um, qm);
            rusanov(Uc, qc, Um, qm, fg[1][0], fg[1][1], fg[1][2], fg[1][3], G2);
            const T iV = T(1) / V;
            T Unew[5];
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const T net = acc[k] + (G2[k] - G1[k]);
                Unew[k] = fmul_add(-(dt * net), iV, Uc[k]);
                *reinterpret_cast<T*>(reinterpret_cast<char*>(out.u[k] + x * SX) + bcol) = Unew[k];
            }
            loc = fmin(loc, local_dt_faces(V, prim(gamma, Unew), fg));
#pragma unroll
            for (int k = 0; k < 5; ++k) Uc[k] = Un[k];
            qc = qn;
#pragma unroll
            for (int k = 0; k < 4; ++k) fg[4][k] = fg[5][k];
        }
    }
    block_min_into(loc, dt_next);
}

// ---------------------------------------------------------------------------
// The Rusanov step as a march along x over tiles of consecutive cells of a
// plane (variant 1 where a row is at most half a tile).
//
// A workgroup owns B consecutive cells c = y*Z + z of each of its L planes, so
// any Z fills its lanes (tiles of whole 64-cell columns leave 45% of them idle
// at Z = 70).  Each cell's state and primitives go to LDS once per plane with
// Z halo cells on either side, at most one per thread; the y and z neighbours
// are the slots Z and 1 away, a wall's neighbour is the cell itself with the
// normal momentum's sign flipped.  The flux between planes x and x+1 is carried
// in registers, and all a plane reads is loaded one plane ahead.  Every face
// flux is evaluated with the lower cell as L, as in euler_step_k, so both give
// the same bits.
//
// GEO 0: face normals, areas and volumes per face and cell (FvGeo).
// GEO 1 / 2: axis-aligned meshes (FvAxis), whose normals are exactly the unit
// vectors: constants for the areas and the volume (1), or areas as products of
// layer widths and the volume per cell (2).  A cell's two fluxes along an axis
// then share its own flux vector and wave speed.
// ---------------------------------------------------------------------------
namespace {

template <class T, int GEO> struct TileGeo { using type = FvAxis<T>; };
template <class T> struct TileGeo<T, 0> { using type = FvGeo<T>; };

// a slot's state and primitives, moved as pairs
template <class T> struct Pair { typedef T type __attribute__((ext_vector_type(2))); };
constexpr int kSlot = 10;

template <class T> __device__ inline void put10(T* slot, const T (&U)[5], const Prim<T>& q) {
    using P = typename Pair<T>::type;
    P* const d = reinterpret_cast<P*>(slot);
    d[0] = P{U[0], U[1]};
    d[1] = P{U[2], U[3]};
    d[2] = P{U[4], q.ux};
    d[3] = P{q.uy, q.uz};
    d[4] = P{q.p, q.a};
}
template <class T> __device__ inline void get10(const T* slot, T (&U)[5], Prim<T>& q) {
    using P = typename Pair<T>::type;
    const P* const d = reinterpret_cast<const P*>(slot);
    const P a = d[0], b = d[1], c = d[2], e = d[3], f = d[4];
    U[0] = a[0]; U[1] = a[1]; U[2] = b[0]; U[3] = b[1]; U[4] = c[0];
    q.ux = c[1]; q.uy = e[0]; q.uz = e[1]; q.p = f[0]; q.a = f[1];
}

template <class T> __device__ inline T at(const T* base, uint32_t boff) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + boff);
}

template <class T>
__device__ inline void axis_faces(T Ax, T Ay, T Az, T (&f)[6][4]) {
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) {
        const int a = 2 - (fc >> 1);
        f[fc][0] = T(a == 0);
        f[fc][1] = T(a == 1);
        f[fc][2] = T(a == 2);
        f[fc][3] = a == 0 ? Ax : a == 1 ? Ay : Az;
    }
}

}  // namespace

template <class T, int B, int GEO>
__global__ void __launch_bounds__(B) euler_tile_k(typename TileGeo<T, GEO>::type g, EIn<T> in, EOut<T> out, int64_t X,
                                                  int Y, int Z, T gamma, T cfl, const Bits<T>* dt_cur,
                                                  Bits<T>* dt_next, Bits<T>* dt_reset, T* dt_hist, int64_t step, int L,
                                                  int ntile) {
    extern __shared__ __align__(16) char lds_raw[];
    T* const lds = reinterpret_cast<T*>(lds_raw);
    const int NS = B + 2 * Z;  // slots of one plane; two planes, used in turn
    const int plane = Y * Z;
    const int64_t SX = plane;
    const int lin = blockIdx.x;
    const int tile = lin % ntile;
    const int64_t x0 = int64_t(lin / ntile) * L;
    const int64_t x1 = (x0 + L < X) ? x0 + L : X;
    const int tid = threadIdx.y * 64 + threadIdx.x;
    const int c0 = tile * B, c = c0 + tid;
    const bool valid = c < plane;
    const int y = valid ? c / Z : 0, z = valid ? c - y * Z : 0;
    const bool zlo = z == 0, zhi = z == Z - 1, ylo = y == 0, yhi = y == Y - 1;
    const T dt = cfl * set_min<T>(dt_cur);
    if (lin == 0 && threadIdx.y == 0) {
        set_reset<T>(dt_reset);
        if (dt_hist && threadIdx.x == 0) dt_hist[step] = dt;
    }
    const int own = (Z + tid) * kSlot;
    // the neighbours' slots, the cell's own at a wall
    const int szl = zlo ? own : own - kSlot, szh = zhi ? own : own + kSlot;
    const int syl = ylo ? own : own - Z * kSlot, syh = yhi ? own : own + Z * kSlot;
    // halo cell of this thread: Z cells before the tile, Z cells after it
    const int hc = tid < Z ? c0 - Z + tid : c0 + B + tid - Z;
    const bool halo = tid < 2 * Z && hc >= 0 && hc < plane;
    const int hslot = (tid < Z ? tid : B + tid) * kSlot;
    // addresses: a pointer uniform over the workgroup and a 32-bit byte offset
    // per lane (the launcher checks that a plane fits)
    const uint32_t bc = uint32_t(valid ? c : 0) * uint32_t(sizeof(T));
    const uint32_t bh = uint32_t(halo ? hc : 0) * uint32_t(sizeof(T));
    const uint32_t bzf = uint32_t(y * (Z + 1) + z) * uint32_t(sizeof(T));
    auto load = [&](int64_t p, uint32_t boff, T (&U)[5]) {
#pragma unroll
        for (int k = 0; k < 5; ++k) U[k] = at(in.u[k] + p * SX, boff);
    };
    auto face4 = [&](int fam, int64_t first, uint32_t boff, T (&o)[4]) {
        if constexpr (GEO == 0) {
            o[0] = at(g.n[fam][0] + first, boff);
            o[1] = at(g.n[fam][1] + first, boff);
            o[2] = at(g.n[fam][2] + first, boff);
            o[3] = at(g.A[fam] + first, boff);
        }
    };

    T fg[6][4] = {};
    T wyz = T(0), wy = T(0), wz = T(0);
    if constexpr (GEO == 1) axis_faces<T>(g.A[0], g.A[1], g.A[2], fg);
    if constexpr (GEO == 2) {
        wy = g.w[1][y];
        wz = g.w[2][z];
        wyz = wy * wz;
    }
    T Uc[5] = {}, Gxl[5] = {};
    Prim<T> qc{};
    T Uh[5] = {}, Uf[5] = {}, fn[6][4] = {}, Vn = T(1);
    auto fetch = [&](int64_t x) {  // for plane x: its halo cell and geometry, the state of plane x + 1
        if (valid && x + 1 < X) load(x + 1, bc, Uf);
        if (halo) load(x, bh, Uh);
        if (valid) {
            if constexpr (GEO == 0) {
                face4(2, (x + 1) * SX, bc, fn[5]);
                face4(1, x * int64_t(Y + 1) * Z, bc, fn[2]);
                face4(1, x * int64_t(Y + 1) * Z + Z, bc, fn[3]);
                const int64_t fz = x * int64_t(Y) * (Z + 1);
                face4(0, fz, bzf, fn[0]);
                face4(0, fz + 1, bzf, fn[1]);
            }
            if constexpr (GEO != 1) Vn = at(g.vol + x * SX, bc);
        }
    };
    T Ul[5] = {};
    if (valid) {  // warm-up: state of plane x0 and the flux through its lower x-face
        load(x0, bc, Uc);
        if (x0 > 0) load(x0 - 1, bc, Ul);
        face4(2, x0 * SX, bc, fg[4]);
    }
    fetch(x0);
    if constexpr (GEO == 2) axis_faces<T>(wyz, T(0), T(0), fg);
    {
        qc = prim(gamma, Uc);
        Prim<T> ql = qc;
        if (x0 == 0) {
#pragma unroll
            for (int k = 0; k < 5; ++k) Ul[k] = Uc[k];
            Ul[1] = -Uc[1];
            ql.ux = -qc.ux;
        } else {
            ql = prim(gamma, Ul);
        }
        rusanov(Ul, ql, Uc, qc, fg[4][0], fg[4][1], fg[4][2], fg[4][3], Gxl);
    }
    T loc = std::numeric_limits<T>::infinity();
    int b = 0;
#pragma unroll 1
    for (int64_t x = x0; x < x1; ++x, b ^= 1) {
        T* const S = lds + b * NS * kSlot;
        T V = Vn;
        if constexpr (GEO == 1) V = g.V;
        if constexpr (GEO == 0) {
#pragma unroll
            for (int f = 0; f < 6; ++f)
                if (f != 4)
#pragma unroll
                    for (int k = 0; k < 4; ++k) fg[f][k] = fn[f][k];
        }
        if constexpr (GEO == 2) {
            const T wx = g.w[0][x];
            axis_faces<T>(wyz, wx * wz, wx * wy, fg);
        }
        T Un[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) Un[k] = Uf[k];
        if (halo) put10(S + hslot, Uh, prim(gamma, Uh));
        put10(S + own, Uc, qc);
        if (x + 1 < x1) fetch(x + 1);
        __syncthreads();
        if (valid) {
            T Um[5], G1[5], G2[5], acc[5];
            Prim<T> qn, qm;
            // net = ((Gx+ - Gx-) + (Gy+ - Gy-)) + (Gz+ - Gz-), accumulated one
            // axis at a time; the upper x flux becomes the next plane's lower
            if (x == X - 1) {
#pragma unroll
                for (int k = 0; k < 5; ++k) Un[k] = Uc[k];
                Un[1] = -Uc[1];
                qn = qc;
                qn.ux = -qc.ux;
            } else {
                qn = prim(gamma, Un);
            }
            rusanov(Uc, qc, Un, qn, fg[5][0], fg[5][1], fg[5][2], fg[5][3], G1);
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                acc[k] = G1[k] - Gxl[k];
                Gxl[k] = G1[k];
            }
            get10(S + syl, Um, qm);
            if (ylo) { Um[2] = -Um[2]; qm.uy = -qm.uy; }
            rusanov(Um, qm, Uc, qc, fg[2][0], fg[2][1], fg[2][2], fg[2][3], G1);
            get10(S + syh, Um, qm);
            if (yhi) { Um[2] = -Um[2]; qm.uy = -qm.uy; }
            rusanov(Uc, qc, Um, qm, fg[3][0], fg[3][1], fg[3][2], fg[3][3], G2);
#pragma unroll
            for (int k = 0; k < 5; ++k) acc[k] = acc[k] + (G2[k] - G1[k]);
            get10(S + szl, Um, qm);
            if (zlo) { Um[3] = -Um[3]; qm.uz = -qm.uz; }
            rusanov(Um, qm, Uc, qc, fg[0][0], fg[0][1], fg[0][2], fg[0][3], G1);
            get10(S + szh, Um, qm);
            if (zhi) { Um[3] = -Um[3]; qm.uz = -qm.uz; }
            rusanov(Uc, qc, Um, qm, fg[1][0], fg[1][1], fg[1][2], fg[1][3], G2);
            const T iV = T(1) / V;
            T Unew[5];
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const T net = acc[k] + (G2[k] - G1[k]);
                Unew[k] = fmul_add(-(dt * net), iV, Uc[k]);
                *reinterpret_cast<T*>(reinterpret_cast<char*>(out.u[k] + x * SX) + bc) = Unew[k];
            }
            loc = fmin(loc, local_dt_faces(V, prim(gamma, Unew), fg));
#pragma unroll
            for (int k = 0; k < 5; ++k) Uc[k] = Un[k];
            qc = qn;
            if constexpr (GEO == 0) {
#pragma unroll
                for (int k = 0; k < 4; ++k) fg[4][k] = fg[5][k];
            }
        }
    }
    block_min_into(loc, dt_next);
}

// the time step of the initial state on an axis-aligned mesh
template <class T, int GEO>
__global__ void __launch_bounds__(256) euler_dt_axis_k(FvAxis<T> g, EIn<T> in, int Y, int Z, T gamma, Bits<T>* slot) {
    const int c = int(blockIdx.x) * 256 + int(threadIdx.y) * 64 + int(threadIdx.x);
    const int64_t x = blockIdx.y;
    T loc = std::numeric_limits<T>::infinity();
    if (c < Y * Z) {
        const int64_t i = x * (int64_t(Y) * Z) + c;
        T U[5], fg[6][4], V = g.V;
#pragma unroll
        for (int k = 0; k < 5; ++k) U[k] = in.u[k][i];
        if constexpr (GEO == 1) {
            axis_faces<T>(g.A[0], g.A[1], g.A[2], fg);
        } else {
            const int y = c / Z, z = c - y * Z;
            const T wx = g.w[0][x], wy = g.w[1][y], wz = g.w[2][z];
            axis_faces<T>(wy * wz, wx * wz, wx * wy, fg);
            V = g.vol[i];
        }
        loc = local_dt_faces(V, prim(gamma, U), fg);
    }
    block_min_into(loc, slot);
}

template <class T>
static void launch_euler_dt_axis(const cfd_mesh_s* m, const FvAxis<T>& g, const EIn<T>& in, T gamma, Bits<T>* slot,
                          hipStream_t s) {
    const dim3 grid(unsigned((m->Y * m->Z + 255) / 256), unsigned(m->X));
    if (g.vol) euler_dt_axis_k<T, 2><<<grid, dim3(64, 4), 0, s>>>(g, in, int(m->Y), int(m->Z), gamma, slot);
    else euler_dt_axis_k<T, 1><<<grid, dim3(64, 4), 0, s>>>(g, in, int(m->Y), int(m->Z), gamma, slot);
    CFD_HIP(hipGetLastError());
}

static bool euler_tile_supported(const cfd_mesh_s* m, int rows) {
    return 2 * m->Z <= 64 * rows && m->Y * (m->Z + 1) * 8 < (int64_t(1) << 31);
}

// Tile and chunk by size: the time of a step goes as the rounds of workgroups
// the chip needs times the planes of one, L and about 1.7 more for its start,
// at the builds' waves per SIMD (FP32 2, FP64 1; axis-aligned 4 and 2).  The
// smallest product was the fastest shape measured, or within 4% of it, at all
// of 512x64x64, 300x40x70, 242x18x21, 80x33x27 and 45x70x76, both precisions,
// all geometries (FP32 us/step against 4 rows x 16 planes throughout:
// perturbed 40.5 / 43.8, 25.4 / 35.4, 8.8 / 32.8, 8.7 / 33.5, 11.9 / 35.0).
// Equal products go to the larger tile (fewer halo cells) on meshes of 2^19
// cells and more.
static void euler_tile_shape(const cfd_mesh_s* m, bool axis, int& rows, int& L) {
    const bool f32 = m->dtype == CFD_F32;
    const int waves = (f32 ? 2 : 1) * (axis ? 2 : 1);
    const bool large = m->N >= (int64_t(1) << 19);
    const bool any = euler_tile_supported(m, f32 ? 8 : 4);
    double best = std::numeric_limits<double>::infinity();
    for (int k = 0; k < 3; ++k) {
        const int r = large ? 8 >> k : (k == 0 ? 4 : k == 1 ? 8 : 2);
        if ((r == 8 && !f32) || (any && !euler_tile_supported(m, r))) continue;
        const int64_t B = 64 * r;
        const int64_t tiles = any ? (m->Y * m->Z + B - 1) / B : ((m->Z + 63) / 64) * ((m->Y + r - 1) / r);
        const int64_t room = 256 * 4 * waves / r;
        for (int l = 32; l >= 1; l /= 2) {
            const int64_t wg = tiles * ((m->X + l - 1) / l);
            const double t = double((wg + room - 1) / room) * (l + 1.7);
            if (t < best) {
                best = t;
                rows = r;
                L = l;
            }
        }
    }
}

// One step; rows = 2, 4 or 8 (FP32) gives tiles of 64 * rows cells.  Exactly
// one of `faces` and `axis` is given.
template <class T>
static void launch_euler_tile(const cfd_mesh_s* m, const FvGeo<T>* faces, const FvAxis<T>* axis, const EIn<T>& in,
                       const EOut<T>& out, T gamma, T cfl, const EulerSlots<T>& sl, T* dt_hist, int64_t step, int rows,
                       int L, hipStream_t s) {
    const int B = 64 * rows, Z = int(m->Z);
    const int64_t ntile = (m->Y * m->Z + B - 1) / B;
    const int64_t nwg = ntile * ((m->X + L - 1) / L);
    CFD_REQUIRE(nwg < (int64_t(1) << 31), "euler march grid too large");
    const size_t lds = size_t(2) * (B + 2 * Z) * kSlot * sizeof(T);
    auto run = [&](auto kern, const auto& g) {
        if (lds > 65536)
            CFD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                        int(lds)));
        kern<<<dim3(unsigned(nwg)), dim3(64, unsigned(rows)), lds, s>>>(g, in, out, m->X, int(m->Y), Z, gamma, cfl,
                                                                       sl.cur, sl.next, sl.reset, dt_hist, step, L,
                                                                       int(ntile));
        CFD_HIP(hipGetLastError());
    };
    auto with_rows = [&](auto r) {
        constexpr int BB = 64 * decltype(r)::value;
        if (faces) run(euler_tile_k<T, BB, 0>, *faces);
        else if (axis->vol) run(euler_tile_k<T, BB, 2>, *axis);
        else run(euler_tile_k<T, BB, 1>, *axis);
    };
    switch (rows) {
        case 2: with_rows(std::integral_constant<int, 2>{}); break;
        case 4: with_rows(std::integral_constant<int, 4>{}); break;
        case 8:
            if constexpr (sizeof(T) == 4) {
                with_rows(std::integral_constant<int, 8>{});
                break;
            }
            [[fallthrough]];
        default: throw Error(CFD_E_INVALID, "euler tiles have 2, 4 or 8 (2 or 4 in FP64) times 64 cells");
    }
}

template <class B> __global__ void fill_bits_k(B* p, int n, B v) {
    const int i = int(blockIdx.x) * int(blockDim.x) + int(threadIdx.x);
    if (i < n) p[i] = v;
}

// Device geometry of the stepper, built on first use from the mesh's vertices:
// the stepper's host arrays, then on the device either what an axis-aligned
// mesh needs of them or all of them.
template <class T> struct FvHost {
    HexGeometry<T> g;
    std::vector<T> v;
    int64_t off_fam[3], off_vol;
};

template <class T> static void build_fv_host(const cfd_mesh_s* m, FvHost<T>& h) {
    build_hex_geometry<T>(h.g, m->X, m->Y, m->Z, T(m->dx), T(m->dy), T(m->dz),
                          m->has_offsets ? m->vertex_offsets.data() : nullptr);
    build_fv_geometry<T>(h.g, h.v, h.off_fam, h.off_vol);
}

static void* fv_upload(cfd_mesh_s* m, const void* host, int64_t bytes, hipStream_t s) {
    void* dev = pool_alloc(m->ctx, bytes, s);
    hipError_t e = hipMemcpyAsync(dev, host, size_t(bytes), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        pool_free(m->ctx, dev, s);
        CFD_HIP(e);
    }
    return dev;
}

template <class T> static FvGeo<T>& fv_of(cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->fv32; else return m->fv64;
}
template <class T> static FvAxis<T>& fa_of(cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->fa32; else return m->fa64;
}

template <class T> static void upload_faces(cfd_mesh_s* m, const FvHost<T>& h, hipStream_t s) {
    const int64_t bytes = int64_t(h.v.size() * sizeof(T));
    const T* d = (const T*)(m->fv_block = fv_upload(m, h.v.data(), bytes, s));
    m->fv_bytes = bytes;
    FvGeo<T>& fv = fv_of<T>(m);
    fv.X = m->X; fv.Y = m->Y; fv.Z = m->Z;
    for (int fam = 0; fam < 3; ++fam) {
        const int64_t nf = h.g.nf[fam];
        for (int k = 0; k < 3; ++k) fv.n[fam][k] = d + h.off_fam[fam] + k * nf;
        fv.A[fam] = d + h.off_fam[fam] + 3 * nf;
    }
    fv.vol = d + h.off_vol;
}

template <class T> static const FvGeo<T>& fv_geometry(cfd_mesh_s* m, hipStream_t s) {
    if (!m->fv_block) {
        FvHost<T> h;
        build_fv_host(m, h);
        upload_faces(m, h, s);
    }
    return fv_of<T>(m);
}

// The axis-aligned form, or null.  Every normal must be a unit vector exactly,
// and the areas (and the volume of a uniform mesh) what the kernels form.
template <class T> static const FvAxis<T>* fv_axis(cfd_mesh_s* m, hipStream_t s) {
    FvAxis<T>& fa = fa_of<T>(m);
    if (m->fv_axis) return m->fv_axis == 1 ? &fa : nullptr;
    if (!m->uniform && !m->lattice) {
        m->fv_axis = 2;
        return nullptr;
    }
    FvHost<T> h;
    build_fv_host(m, h);
    const HexGeometry<T>& g = h.g;
    const int64_t vs[3] = {(g.Y + 1) * (g.Z + 1), g.Z + 1, 1}, ext[3] = {g.X, g.Y, g.Z};
    const std::vector<T>* vert[3] = {&g.vx, &g.vy, &g.vz};
    std::vector<T> w[3];
    for (int a = 0; a < 3; ++a)
        for (int64_t k = 0; k < ext[a]; ++k)
            w[a].push_back((*vert[a])[size_t((k + 1) * vs[a])] - (*vert[a])[size_t(k * vs[a])]);
    int bad = 0;
    FvAxis<T> f{};
    for (int fam = 0; fam < 3 && !bad; ++fam) {
        const int axis = 2 - fam;
        const T* d = h.v.data() + h.off_fam[fam];
        const int64_t nf = g.nf[fam];
        f.A[axis] = d[3 * nf];
        const int64_t nx = g.X + (axis == 0), ny = g.Y + (axis == 1), nz = g.Z + (axis == 2);
#pragma omp parallel for schedule(static) reduction(+ : bad)
        for (int64_t x = 0; x < nx; ++x)
            for (int64_t y = 0; y < ny; ++y)
                for (int64_t z = 0; z < nz; ++z) {
                    const int64_t i = fam == 0 ? g.zface(x, y, z) : fam == 1 ? g.yface(x, y, z) : g.xface(x, y, z);
                    for (int k = 0; k < 3; ++k) bad += !(d[k * nf + i] == (k == axis ? T(1) : T(0)));
                    const T A = m->uniform ? f.A[axis]
                              : axis == 0 ? w[1][y] * w[2][z] : axis == 1 ? w[0][x] * w[2][z] : w[0][x] * w[1][y];
                    bad += !(d[3 * nf + i] == A);
                }
    }
    const T* vol = h.v.data() + h.off_vol;
    f.V = vol[0];
    if (m->uniform)
        for (int64_t i = 0; i < g.N; ++i) bad += !(vol[i] == f.V);
    if (bad) {
        m->fv_axis = 2;
        if (!m->fv_block) upload_faces(m, h, s);
        return nullptr;
    }
    if (!m->uniform) {
        m->fa_block = fv_upload(m, vol, g.N * int64_t(sizeof(T)), s);
        f.vol = (const T*)m->fa_block;
        const LatticeGeo<T>& lg = [&]() -> const LatticeGeo<T>& {
            if constexpr (sizeof(T) == 4) return m->lg32; else return m->lg64;
        }();
        for (int a = 0; a < 3; ++a) f.w[a] = lg.w[a];
    }
    fa = f;
    m->fv_axis = 1;
    return &fa;
}

// The geometry that the mesh's shape reads, built where it is not there yet:
// the axis-aligned form where it exists and the tiles take the mesh, else the
// face arrays.
template <class T> struct EulerGeometry {
    const FvAxis<T>* axis = nullptr;
    const FvGeo<T>* faces = nullptr;
};
template <class T> static EulerGeometry<T> euler_geometry(cfd_mesh_s* m, hipStream_t s) {
    EulerGeometry<T> g;
    const int rows = m->euler_variant < 0 ? (sizeof(T) == 4 ? 8 : 4) : m->euler_ty;
    if (m->euler_variant != 0 && euler_tile_supported(m, rows)) g.axis = fv_axis<T>(m, s);
    if (!g.axis) g.faces = &fv_geometry<T>(m, s);
    return g;
}

// Builds what a newly set shape reads on a mesh that has run already, so that
// its next run can be captured in a graph like any further run.
template <class T> void euler_shape_changed(cfd_mesh_s* m) {
    if (m->fv_block || m->fv_axis == 1) euler_geometry<T>(m, nullptr);
}
template void euler_shape_changed<float>(cfd_mesh_s*);
template void euler_shape_changed<double>(cfd_mesh_s*);

template <class T>
void launch_euler(cfd_mesh_s* m, void* const a[5], void* const b[5], double gamma, double cfl, int64_t nsteps,
                  void* dt_hist, hipStream_t s) {
    int ty = m->euler_ty, L = m->euler_L;
    const bool march = m->euler_variant != 0, chosen = m->euler_variant < 0;
    const EulerGeometry<T> geo = euler_geometry<T>(m, s);
    const FvAxis<T>* const axis = geo.axis;
    const FvGeo<T>* const faces = geo.faces;
    if (chosen) euler_tile_shape(m, axis != nullptr, ty, L);
    const bool tile = march && euler_tile_supported(m, ty);
    Bits<T>* slots = (Bits<T>*)pool_alloc(m->ctx, 3 * kDtSet * sizeof(Bits<T>), s);
    try {
        const dim3 block(64, 4, 1);
        const dim3 grid(unsigned((m->Z + 63) / 64), unsigned((m->Y + 3) / 4), unsigned(m->X));
        const Bits<T> inf = sizeof(T) == 4 ? Bits<T>(0x7f800000u) : Bits<T>(0x7ff0000000000000ull);
        fill_bits_k<Bits<T>><<<3 * kDtSet / 256, 256, 0, s>>>(slots, 3 * kDtSet, inf);
        EIn<T> in{};
        EOut<T> out{};
        for (int k = 0; k < 5; ++k) in.u[k] = (const T*)a[k];
        if (axis) launch_euler_dt_axis<T>(m, *axis, in, T(gamma), slots, s);
        else euler_dt_k<T><<<grid, block, 0, s>>>(*faces, in, T(gamma), slots);
        CFD_HIP(hipGetLastError());
        const int nzt = int((m->Z + 63) / 64), nyt = int((m->Y + ty - 1) / ty);
        CFD_REQUIRE(!march || m->Y * (m->Z + 1) * int64_t(sizeof(T)) < (int64_t(1) << 32),
                    "Euler march: a plane of this mesh exceeds 32-bit byte offsets (use the per-thread form)");
        const int64_t nwg = int64_t(nzt) * nyt * ((m->X + L - 1) / L);
        CFD_REQUIRE(nwg < (int64_t(1) << 31), "euler march grid too large");
        for (int64_t st = 0; st < nsteps; ++st) {
            void* const* src = (st & 1) ? b : a;
            void* const* dst = (st & 1) ? a : b;
            for (int k = 0; k < 5; ++k) {
                in.u[k] = (const T*)src[k];
                out.u[k] = (T*)dst[k];
            }
            Bits<T>* cur = slots + (st % 3) * kDtSet;
            Bits<T>* nxt = slots + ((st + 1) % 3) * kDtSet;
            Bits<T>* rst = slots + ((st + 2) % 3) * kDtSet;
            if (!march) {
                euler_step_k<T><<<grid, block, 0, s>>>(*faces, in, out, T(gamma), T(cfl), cur, nxt, rst, (T*)dt_hist,
                                                       st);
                continue;
            }
            if (tile) {
                launch_euler_tile<T>(m, faces, axis, in, out, T(gamma), T(cfl), EulerSlots<T>{cur, nxt, rst},
                                     (T*)dt_hist, st, ty, L, s);
                continue;
            }
            const dim3 mgrid{unsigned(nwg), 1u, 1u};
#define CFD_EULER_MARCH(TYV)                                                                                    \
    euler_march_k<T, TYV><<<mgrid, dim3(64, TYV), 0, s>>>(*faces, in, out, T(gamma), T(cfl), cur, nxt, rst,     \
                                                         (T*)dt_hist, st, L, nzt, nyt)
            switch (ty) {
                case 2: CFD_EULER_MARCH(2); break;
                case 4: CFD_EULER_MARCH(4); break;
                case 8:
                    // FP32 only: the FP64 8-row build spills registers, and the
                    // kernel's dt reduction reads other lanes' registers
                    if constexpr (sizeof(T) == 4) {
                        CFD_EULER_MARCH(8);
                        break;
                    }
                    [[fallthrough]];
                default: throw Error(CFD_E_INVALID, "euler march tile rows must be 2, 4 or 8 (2 or 4 in FP64)");
            }
#undef CFD_EULER_MARCH
        }
        CFD_HIP(hipGetLastError());
    } catch (...) {
        pool_free(m->ctx, slots, s);
        throw;
    }
    pool_free(m->ctx, slots, s);
}

// ---------------------------------------------------------------------------
// The same stepper on a mesh given by its connectivity (cfd_mesh_create_
// unstructured): one thread per cell in the mesh's reverse Cuthill-McKee
// numbering, the neighbours through the (local face, cell) ids, the
// stepper's geometry per face (build_ufv_geometry).  Each cell evaluates its
// six face fluxes with the lower cell of the face's axis pair as L, in the
// per-thread kernel's order, so results equal the oracle's on the same
// connectivity.
// ---------------------------------------------------------------------------

// each XCD (round-robin dispatch) takes a contiguous run of blocks
__device__ inline int64_t ucell() {
    const int b = int((blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8);
    return int64_t(b) * 256 + threadIdx.y * 64 + threadIdx.x;
}

// V / sum over fc = 0..5 of A_f (|u.n_f| + a), the faces through the ids
template <class T> __device__ inline T ulocal_dt(const UnstructGeo<T>& g, int64_t i, const Prim<T>& q) {
    T s = T(0);
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) {
        const auto r = face_rec(g.srec, g.face[int64_t(fc) * g.N + i]);
        const T un = un_of(q.ux, q.uy, q.uz, r[0], r[1], r[2]);
        s = fmul_add(r[3], fabs(un) + q.a, s);
    }
    return g.svol[i] / s;
}

template <class T>
__global__ void __launch_bounds__(256) ueuler_dt_k(UnstructGeo<T> g, EIn<T> in, T gamma, Bits<T>* slot) {
    const int64_t i = ucell();
    T loc = std::numeric_limits<T>::infinity();
    if (i < g.N) {
        T U[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) U[k] = in.u[k][i];
        loc = ulocal_dt(g, i, prim(gamma, U));
    }
    block_min_into(loc, slot);
}

template <class T>
__global__ void __launch_bounds__(256) ueuler_step_k(UnstructGeo<T> g, EIn<T> in, EOut<T> out, T gamma, T cfl,
                                                    const Bits<T>* dt_cur, Bits<T>* dt_next, Bits<T>* dt_reset,
                                                    T* dt_hist, int64_t step) {
    const int64_t i = ucell();
    const T dt = cfl * set_min<T>(dt_cur);
    if (blockIdx.x == 0 && threadIdx.y == 0) {
        set_reset<T>(dt_reset);
        if (dt_hist && threadIdx.x == 0) dt_hist[step] = dt;
    }
    T loc = std::numeric_limits<T>::infinity();
    if (i < g.N) {
        T Ui[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) Ui[k] = in.u[k][i];
        const Prim<T> qi = prim(gamma, Ui);
        T net[5] = {T(0), T(0), T(0), T(0), T(0)};
        // axis pairs in the order x, y, z: net = ((x+ - x-) + (y+ - y-)) + (z+ - z-)
#pragma unroll
        for (int pair = 2; pair >= 0; --pair) {
            T Gp[2][5];
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const int fc = 2 * pair + side;
                const int64_t k6 = int64_t(fc) * g.N + i;
                const int32_t nb = g.nbr[k6];
                T Un[5];
                if (nb < 0) {  // wall: the mirrored state
#pragma unroll
                    for (int k = 0; k < 5; ++k) Un[k] = Ui[k];
                    Un[3 - pair] = -Ui[3 - pair];
                } else {
#pragma unroll
                    for (int k = 0; k < 5; ++k) Un[k] = in.u[k][nb];
                }
                const Prim<T> qn = prim(gamma, Un);
                const auto r = face_rec(g.srec, g.face[k6]);
                if (side == 1) rusanov<T>(Ui, qi, Un, qn, r[0], r[1], r[2], r[3], Gp[side]);
                else rusanov<T>(Un, qn, Ui, qi, r[0], r[1], r[2], r[3], Gp[side]);
            }
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const T d = Gp[1][k] - Gp[0][k];
                net[k] = pair == 2 ? d : net[k] + d;
            }
        }
        const T iV = T(1) / g.svol[i];
        T Un[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            Un[k] = fmul_add(-(dt * net[k]), iV, Ui[k]);
            out.u[k][i] = Un[k];
        }
        loc = ulocal_dt(g, i, prim(gamma, Un));
    }
    block_min_into(loc, dt_next);
}

namespace {

template <class T> UnstructGeo<T>& ugeo_e(cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->uu32; else return m->uu64;
}

// the stepper's geometry of an unstructured mesh, built and uploaded on first
// use into one pool block (faces and cells in the mesh's numbering)
template <class T> const UnstructGeo<T>& ufv_geometry(cfd_mesh_s* m, hipStream_t s) {
    UnstructGeo<T>& u = ugeo_e<T>(m);
    if (u.svol) return u;
    const UConn& c = m->uconn;
    UGeometry<T> g;
    build_ugeometry<T>(g, c);
    std::vector<T> sv, svol;
    build_ufv_geometry<T>(c, g, sv, svol);
    const int64_t N = c.N, F = c.F;
    std::vector<T> host(size_t(4 * F + N));
    for (int64_t n = 0; n < F; ++n) {
        const int64_t f = m->face_dev[n];
        for (int k = 0; k < 4; ++k) host[size_t(4 * n + k)] = sv[size_t(k * F + f)];
    }
    for (int64_t n = 0; n < N; ++n) host[size_t(4 * F + n)] = svol[size_t(m->cell_perm[n])];
    const int64_t bytes = int64_t(host.size() * sizeof(T));
    void* dev = pool_alloc(m->ctx, bytes, s);
    hipError_t e = hipMemcpyAsync(dev, host.data(), size_t(bytes), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        pool_free(m->ctx, dev, s);
        CFD_HIP(e);
    }
    const T* d = static_cast<const T*>(dev);
    u.srec = d;
    u.svol = d + 4 * F;
    m->fv_block = dev;
    m->fv_bytes = bytes;
    return u;
}

}  // namespace

template <class T>
void launch_ueuler(cfd_mesh_s* m, void* const a[5], void* const b[5], double gamma, double cfl, int64_t nsteps,
                   void* dt_hist, hipStream_t s) {
    const UnstructGeo<T>& g = ufv_geometry<T>(m, s);
    Bits<T>* slots = (Bits<T>*)pool_alloc(m->ctx, 3 * kDtSet * sizeof(Bits<T>), s);
    try {
        const dim3 block(64, 4, 1);
        const dim3 grid(unsigned((m->N + 2047) / 2048 * 8));
        const Bits<T> inf = sizeof(T) == 4 ? Bits<T>(0x7f800000u) : Bits<T>(0x7ff0000000000000ull);
        fill_bits_k<Bits<T>><<<3 * kDtSet / 256, 256, 0, s>>>(slots, 3 * kDtSet, inf);
        EIn<T> in{};
        EOut<T> out{};
        for (int k = 0; k < 5; ++k) in.u[k] = (const T*)a[k];
        ueuler_dt_k<T><<<grid, block, 0, s>>>(g, in, T(gamma), slots);
        CFD_HIP(hipGetLastError());
        for (int64_t st = 0; st < nsteps; ++st) {
            void* const* src = (st & 1) ? b : a;
            void* const* dst = (st & 1) ? a : b;
            for (int k = 0; k < 5; ++k) {
                in.u[k] = (const T*)src[k];
                out.u[k] = (T*)dst[k];
            }
            ueuler_step_k<T><<<grid, block, 0, s>>>(g, in, out, T(gamma), T(cfl), slots + (st % 3) * kDtSet,
                                                    slots + ((st + 1) % 3) * kDtSet, slots + ((st + 2) % 3) * kDtSet, (T*)dt_hist, st);
            CFD_HIP(hipGetLastError());
        }
    } catch (...) {
        pool_free(m->ctx, slots, s);
        throw;
    }
    pool_free(m->ctx, slots, s);
}

template void launch_ueuler<float>(cfd_mesh_s*, void* const[5], void* const[5], double, double, int64_t, void*,
                                   hipStream_t);
template void launch_ueuler<double>(cfd_mesh_s*, void* const[5], void* const[5], double, double, int64_t, void*,
                                    hipStream_t);

template void launch_euler<float>(cfd_mesh_s*, void* const[5], void* const[5], double, double, int64_t, void*,
                                  hipStream_t);
template void launch_euler<double>(cfd_mesh_s*, void* const[5], void* const[5], double, double, int64_t, void*,
                                   hipStream_t);

}  // namespace cfd
