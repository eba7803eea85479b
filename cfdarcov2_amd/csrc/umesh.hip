// Unstructured hex meshes (cfd_mesh_create_unstructured): the reference's
// operators on a mesh given by its connectivity (no lattice), cells reordered
// for locality, as cell-centred gathers.
//
// Device layout (cells and faces in the mesh's reordered numbering):
//   per (local face fc, cell), fc-major, int32: the neighbour across the face
//   (-1 on the boundary) and the face id, its top bit set where the face
//   normal points into the cell;
//   per face: the normal (first three vertices) and area as one record of
//   four values, and alpha_d;
//   per cell: the volume; per (fc, cell): the centre-to-face distance (the
//   stabilisation's upwind extrapolation).
// Each cell reads its own six faces and neighbours and writes only itself:
// no atomics and no scatter.  A face's value is formed by each of its two
// cells in that cell's own operation order, which is the reference's per
// (cell, fc) evaluation (include/grad_utils.hpp:23-125), so the results equal
// the reference semantics bit for bit whatever the numbering.  Reverse
// Cuthill-McKee numbering keeps the six neighbours of a cell, and so the
// gathered values, within a few cache lines of the cell's own.
//
// Bound by the gathers: 96^3 FP64 moves 193 algorithmic bytes per cell and
// heat step (ids 48, volume 8, state 16, three faces' records and alpha 121) at
// 6.7 TB/s from the last-level cache.  us/step at 96^3, heat / acoustic, FP64 (FP32): blocks in
// launch order, faces by their lowest cell, one array per component 43.6 / 86.6
// (26.2 / 55.2); contiguous runs of blocks per XCD, so a face's second gather
// hits that L2, 29.6 / 64.1 (20.9 / 45.3); faces by local index and cell,
// normal and area in one record 25.4 / 59.0 (16.5 / 37.2).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"
#include "umesh.hpp"

namespace cfd {

namespace {

constexpr int kUBlock = 256;

// The thread's cell.  Each XCD (round-robin dispatch) takes a contiguous run
// of blocks, so cells a matrix bandwidth apart meet in one L2.
__device__ inline int64_t ucell_of_thread() {
    const int b = int((blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8);
    return int64_t(b) * kUBlock + threadIdx.x;
}

// a cell's six faces: neighbours, face ids (with the sign bit), normal and area
template <class T> struct UFaces {
    int32_t nb[6], f[6];
    typename FaceRec<T>::type r[6];
};
template <class T> __device__ inline void uload(const UnstructGeo<T>& g, int64_t i, UFaces<T>& c) {
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) {
        const int64_t k = int64_t(fc) * g.N + i;
        c.nb[fc] = g.nbr[k];
        c.f[fc] = g.face[k];
    }
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) c.r[fc] = face_rec(g.rec, c.f[fc]);
}

template <class T> __device__ inline T ugauss(const UnstructGeo<T>& g, const T (&fv)[6], const UFaces<T>& c, int d,
                                              int64_t i, bool axis) {
    // sum over fc = 0..5 of (fv * n) * area from 0, then / V; n is the axis
    // normal (+n on fc 2, 3, -n on the others) or the outward normal
    T acc = T(0);
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) {
        const T n = d == 0 ? c.r[fc][0] : d == 1 ? c.r[fc][1] : c.r[fc][2];
        const bool neg = axis ? !(fc == 2 || fc == 3) : c.f[fc] < 0;
        T t = fv[fc] * (neg ? -n : n);
        t = t * c.r[fc][3];
        acc = acc + t;
    }
    return acc / g.vol[i];
}

}  // namespace

// GradVar: face value (phi_c + phi_nb) / 2 (neighbour = self on the boundary,
// or 0 on boundary faces normal to wall_axis), outward Gauss sum per selected
// axis, res = 0 + g_x (+ g_y) (+ g_z).
template <class T>
__global__ void __launch_bounds__(kUBlock) ugrad_k(UnstructGeo<T> g, const T* __restrict__ phi, T* __restrict__ out,
                                                   int mask, int wall) {
    const int64_t i = ucell_of_thread();
    if (i >= g.N) return;
    UFaces<T> c;
    uload(g, i, c);
    const T pc = phi[i];
    T fv[6];
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) {
        const bool bnd = c.nb[fc] < 0;
        fv[fc] = (wall >= 0 && bnd && (fc >> 1) == 2 - wall) ? T(0) : (pc + (bnd ? pc : phi[c.nb[fc]])) * T(0.5);
    }
    T res = T(0);
    for (int d = 0; d < 3; ++d)
        if (mask & (1 << d)) res = res + ugauss(g, fv, c, d, i, false);
    out[i] = res;
}

// Grad2Var: (-phi_c + phi_nb) * alpha_d, axis-normal Gauss sum per selected axis.
template <class T> __device__ inline T ulapl_cell(const UnstructGeo<T>& g, const T* __restrict__ phi, int64_t i,
                                                  int mask) {
    UFaces<T> c;
    uload(g, i, c);
    const T pc = phi[i];
    T fv[6];
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) fv[fc] = (-pc + (c.nb[fc] < 0 ? pc : phi[c.nb[fc]])) * g.alpha[c.f[fc] & kFaceId];
    T res = T(0);
    for (int d = 0; d < 3; ++d)
        if (mask & (1 << d)) res = res + ugauss(g, fv, c, d, i, true);
    return res;
}

template <class T>
__global__ void __launch_bounds__(kUBlock) ulapl_k(UnstructGeo<T> g, const T* __restrict__ phi, T* __restrict__ out,
                                                   int mask) {
    const int64_t i = ucell_of_thread();
    if (i >= g.N) return;
    out[i] = ulapl_cell(g, phi, i, mask);
}

// d1t(T) = alpha * lapl(T): T <- dt * (alpha * L) + T
template <class T>
__global__ void __launch_bounds__(kUBlock) uheat_k(UnstructGeo<T> g, const T* __restrict__ Tin, T* __restrict__ Tout,
                                                   T alpha, const T* __restrict__ alpha_f, T dt) {
    const int64_t i = ucell_of_thread();
    if (i >= g.N) return;
    const T L = ulapl_cell(g, Tin, i, 7);
    const T k = alpha_f ? alpha_f[i] : alpha;
    Tout[i] = dt * (k * L) + Tin[i];
}

namespace {

template <class T> const UnstructGeo<T>& ugeo_u(const cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->uu32; else return m->uu64;
}
template <class T> UnstructGeo<T>& ugeo_u(cfd_mesh_s* m) {
    if constexpr (sizeof(T) == 4) return m->uu32; else return m->uu64;
}
dim3 ugrid(int64_t N) { return dim3(unsigned((N + 8 * kUBlock - 1) / (8 * kUBlock) * 8)); }

}  // namespace

template <class T> void launch_ugrad(const cfd_mesh_s* m, const void* phi, void* out, int mask, int wall, hipStream_t s) {
    ugrad_k<T><<<ugrid(m->N), kUBlock, 0, s>>>(ugeo_u<T>(m), (const T*)phi, (T*)out, mask, wall);
    CFD_HIP(hipGetLastError());
}
template <class T> void launch_ulapl(const cfd_mesh_s* m, const void* phi, void* out, int mask, hipStream_t s) {
    ulapl_k<T><<<ugrid(m->N), kUBlock, 0, s>>>(ugeo_u<T>(m), (const T*)phi, (T*)out, mask);
    CFD_HIP(hipGetLastError());
}
// StabVar, first stage: the three outward-Gauss gradient components of phi
// with the reference face rule (neighbour = self on the boundary), each
// written as computed (no 0 + g), as the reference keeps them per axis.
template <class T>
__global__ void __launch_bounds__(kUBlock) ustab_grad_k(UnstructGeo<T> g, const T* __restrict__ phi,
                                                        T* __restrict__ gx, T* __restrict__ gy, T* __restrict__ gz) {
    const int64_t i = ucell_of_thread();
    if (i >= g.N) return;
    UFaces<T> c;
    uload(g, i, c);
    const T pc = phi[i];
    T fv[6];
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) fv[fc] = (pc + (c.nb[fc] < 0 ? pc : phi[c.nb[fc]])) * T(0.5);
    gx[i] = ugauss(g, fv, c, 0, i, false);
    gy[i] = ugauss(g, fv, c, 1, i, false);
    gz[i] = ugauss(g, fv, c, 2, i, false);
}

// StabVar, second stage (include/grad_utils.hpp:38-80, src/fvm3d.cpp:915-936):
// per selected axis d, the upwind face value phi + len * g_d * n_out,d of the
// cell on face fc against the neighbour's on its opposite local face fc ^ 1
// (self on the boundary), 0.5 * (own - neighbour's), axis-normal Gauss sum,
// res = 0 + S_x (+ S_y) (+ S_z).  The neighbour's value is recomputed from its
// phi, gradient and face geometry, as its own cell forms it.
template <class T>
__global__ void __launch_bounds__(kUBlock) ustab_k(UnstructGeo<T> g, const T* __restrict__ phi,
                                                   const T* __restrict__ gx, const T* __restrict__ gy,
                                                   const T* __restrict__ gz, T* __restrict__ out, int mask) {
    const int64_t i = ucell_of_thread();
    if (i >= g.N) return;
    UFaces<T> c;
    uload(g, i, c);
    const T* const gd[3] = {gx, gy, gz};
    auto upwind = [&](int d, int64_t j, int fc) {
        const int64_t k = int64_t(fc) * g.N + j;
        const int32_t f = g.face[k];
        const T n = g.rec[4 * int64_t(f & kFaceId) + d];
        const T na = f < 0 ? -n : n;
        return phi[j] + g.len[k] * gd[d][j] * na;
    };
    T res = T(0);
    for (int d = 0; d < 3; ++d) {
        if (!(mask & (1 << d))) continue;
        T fv[6];
#pragma unroll
        for (int fc = 0; fc < 6; ++fc) {
            const int64_t j = c.nb[fc] < 0 ? i : int64_t(c.nb[fc]);
            const T own = upwind(d, i, fc);
            const T col = upwind(d, j, fc ^ 1);
            fv[fc] = T(0.5) * (own - col);
        }
        res = res + ugauss(g, fv, c, d, i, true);
    }
    out[i] = res;
}

// The fused acoustic step (the reference operators' composition, as the
// structured kernels run it): first every cell's velocities
//   u_d' = dt * (-(0 + G_d(p))) + u_d   (face values (p_c + p_nb) / 2, neighbour = self)
// then the pressure from the new velocities
//   p' = dt * (K * ((D_x(u') + D_y(v')) + D_z(w'))) + p
// with D_a = 0 + the outward Gauss sum of velocity a under the reflective-wall
// face rule (zero on boundary faces of the axis-a pair of local faces).
template <class T>
__global__ void __launch_bounds__(kUBlock) uwave_vel_k(UnstructGeo<T> g, const T* __restrict__ p,
                                                       const T* __restrict__ u, const T* __restrict__ v,
                                                       const T* __restrict__ w, T* __restrict__ uo,
                                                       T* __restrict__ vo, T* __restrict__ wo, T dt) {
    const int64_t i = ucell_of_thread();
    if (i >= g.N) return;
    UFaces<T> c;
    uload(g, i, c);
    const T pc = p[i];
    T fv[6];
#pragma unroll
    for (int fc = 0; fc < 6; ++fc) fv[fc] = (pc + (c.nb[fc] < 0 ? pc : p[c.nb[fc]])) * T(0.5);
    const T* const vin[3] = {u, v, w};
    T* const vout[3] = {uo, vo, wo};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T gd = T(0) + ugauss(g, fv, c, d, i, false);
        vout[d][i] = dt * (-gd) + vin[d][i];
    }
}

template <class T>
__global__ void __launch_bounds__(kUBlock) uwave_pres_k(UnstructGeo<T> g, const T* __restrict__ p,
                                                        const T* __restrict__ u, const T* __restrict__ v,
                                                        const T* __restrict__ w, T* __restrict__ po, T K,
                                                        const T* __restrict__ Kf, T dt) {
    const int64_t i = ucell_of_thread();
    if (i >= g.N) return;
    UFaces<T> c;
    uload(g, i, c);
    const T* const vel[3] = {u, v, w};
    T div[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T* q = vel[d];
        const T qc = q[i];
        T fv[6];
#pragma unroll
        for (int fc = 0; fc < 6; ++fc) {
            const bool bnd = c.nb[fc] < 0;
            fv[fc] = (bnd && (fc >> 1) == 2 - d) ? T(0) : (qc + (bnd ? qc : q[c.nb[fc]])) * T(0.5);
        }
        div[d] = T(0) + ugauss(g, fv, c, d, i, false);
    }
    const T S = (div[0] + div[1]) + div[2];
    const T k = Kf ? Kf[i] : K;
    po[i] = dt * (k * S) + p[i];
}

template <class T>
void launch_uwave(const cfd_mesh_s* m, void* const a[4], void* const b[4], double K, const void* Kf, double dt,
                  int64_t nsteps, hipStream_t s) {
    for (int64_t t = 0; t < nsteps; ++t) {
        void* const* in = (t & 1) ? b : a;
        void* const* out = (t & 1) ? a : b;
        uwave_vel_k<T><<<ugrid(m->N), kUBlock, 0, s>>>(ugeo_u<T>(m), (const T*)in[0], (const T*)in[1],
                                                       (const T*)in[2], (const T*)in[3], (T*)out[1], (T*)out[2],
                                                       (T*)out[3], T(dt));
        CFD_HIP(hipGetLastError());
        uwave_pres_k<T><<<ugrid(m->N), kUBlock, 0, s>>>(ugeo_u<T>(m), (const T*)in[0], (const T*)out[1],
                                                        (const T*)out[2], (const T*)out[3], (T*)out[0], T(K),
                                                        (const T*)Kf, T(dt));
        CFD_HIP(hipGetLastError());
    }
}

template <class T>
void launch_ustab(const cfd_mesh_s* m, const void* phi, void* out, int mask, void* work, hipStream_t s) {
    T* w = static_cast<T*>(work);
    const int64_t N = m->N;
    ustab_grad_k<T><<<ugrid(N), kUBlock, 0, s>>>(ugeo_u<T>(m), (const T*)phi, w, w + N, w + 2 * N);
    CFD_HIP(hipGetLastError());
    ustab_k<T><<<ugrid(N), kUBlock, 0, s>>>(ugeo_u<T>(m), (const T*)phi, w, w + N, w + 2 * N, (T*)out, mask);
    CFD_HIP(hipGetLastError());
}

template <class T>
void launch_uheat(const cfd_mesh_s* m, void* Ta, void* Tb, double alpha, const void* af, double dt, int64_t nsteps,
                  hipStream_t s) {
    for (int64_t k = 0; k < nsteps; ++k) {
        const T* in = (const T*)((k & 1) ? Tb : Ta);
        T* out = (T*)((k & 1) ? Ta : Tb);
        uheat_k<T><<<ugrid(m->N), kUBlock, 0, s>>>(ugeo_u<T>(m), in, out, T(alpha), (const T*)af, T(dt));
        CFD_HIP(hipGetLastError());
    }
}

// Geometry, numbering and upload of an unstructured mesh.  Device block: the
// faces' records (4F), alpha (F), vol (N), len (6N), then nbr and face (6N
// int32 each).
template <class T> void create_unstructured(cfd_mesh_s* m, int reorder) {
    const UConn& c = m->uconn;
    check_uconn(c);
    UGeometry<T> g;
    build_ugeometry<T>(g, c);
    const int64_t N = c.N, F = c.F;
    if (reorder) {
        m->cell_perm = rcm_order(c);
    } else {
        m->cell_perm.resize(N);
        for (int64_t i = 0; i < N; ++i) m->cell_perm[i] = i;
    }
    m->cell_iperm.assign(N, 0);
    for (int64_t n = 0; n < N; ++n) m->cell_iperm[m->cell_perm[n]] = n;
    m->face_perm = face_order(c, m->cell_iperm);
    // The device arrays hold the faces by the local index fc they have in
    // their lowest cell, and by that cell within one fc: consecutive cells
    // then find face fc at consecutive places (a wave's 64 FP64 values in 4
    // cache lines; in the order of face_perm, where a cell's own faces lie
    // side by side, in 12).
    // per (new cell, fc): the face and the new neighbour, gathered once
    struct Side { int32_t f, nb; };
    std::vector<Side> side(size_t(6 * N));
#pragma omp parallel for schedule(static)
    for (int64_t n = 0; n < N; ++n) {
        const int64_t i = m->cell_perm[n];
        for (int fc = 0; fc < 6; ++fc) {
            const int64_t f = c.cell_faces[6 * i + fc];
            const int64_t a = c.face_cells[2 * f], b = c.face_cells[2 * f + 1];
            const int64_t other = b < 0 ? -1 : (a == i ? b : a);
            side[size_t(6 * n + fc)] = {int32_t(f), other < 0 ? -1 : int32_t(m->cell_iperm[other])};
        }
    }
    std::vector<int32_t> place(size_t(F), -1);  // of each of the caller's faces in the device arrays
    m->face_dev.clear();
    m->face_dev.reserve(F);
    for (int fc = 0; fc < 6; ++fc)
        for (int64_t n = 0; n < N; ++n) {
            const Side sd = side[size_t(6 * n + fc)];
            if (sd.nb >= 0 && sd.nb < n) continue;
            if (place[size_t(sd.f)] >= 0) continue;
            place[size_t(sd.f)] = int32_t(m->face_dev.size());
            m->face_dev.push_back(sd.f);
        }
    for (int64_t f = 0; f < F; ++f)  // faces that their lowest cell does not list
        if (place[size_t(f)] < 0) {
            place[size_t(f)] = int32_t(m->face_dev.size());
            m->face_dev.push_back(f);
        }

    const size_t ib = 6 * size_t(N) * sizeof(int32_t);
    const size_t tb = (5 * size_t(F) + 7 * size_t(N)) * sizeof(T);
    const int64_t bytes = int64_t(2 * ib + tb);
    std::vector<char> host(static_cast<size_t>(bytes));
    T* tv = reinterpret_cast<T*>(host.data());
    int32_t* nbr = reinterpret_cast<int32_t*>(host.data() + tb);
    int32_t* fid = nbr + 6 * N;
#pragma omp parallel for schedule(static)
    for (int64_t n = 0; n < N; ++n) {
        const int64_t i = m->cell_perm[n];
        for (int fc = 0; fc < 6; ++fc) {
            const Side sd = side[size_t(6 * n + fc)];
            nbr[fc * N + n] = sd.nb;
            fid[fc * N + n] = place[size_t(sd.f)] | (g.out_sign[6 * i + fc] < 0 ? ~kFaceId : 0);
        }
    }
#pragma omp parallel for schedule(static)
    for (int64_t n = 0; n < F; ++n) {
        const int64_t f = m->face_dev[n];
        T* r = tv + 4 * n;
        r[0] = g.fnx[f];
        r[1] = g.fny[f];
        r[2] = g.fnz[f];
        r[3] = g.farea[f];
        tv[4 * F + n] = g.falpha[f];
    }
    T* lv = tv + 5 * F + N;
#pragma omp parallel for schedule(static)
    for (int64_t n = 0; n < N; ++n) {
        const int64_t i = m->cell_perm[n];
        tv[5 * F + n] = g.vol[i];
        for (int fc = 0; fc < 6; ++fc) lv[fc * N + n] = g.len[6 * i + fc];
    }

    hipStream_t s = nullptr;
    m->dev_block = pool_alloc(m->ctx, bytes, s);
    m->device_bytes = bytes;
    CFD_HIP(hipMemcpyAsync(m->dev_block, host.data(), size_t(bytes), hipMemcpyHostToDevice, s));
    CFD_HIP(hipStreamSynchronize(s));
    char* d = static_cast<char*>(m->dev_block);
    UnstructGeo<T>& u = ugeo_u<T>(m);
    u.N = N;
    u.F = F;
    const T* dt = reinterpret_cast<const T*>(d);
    u.rec = dt;
    u.alpha = dt + 4 * F;
    u.vol = dt + 5 * F;
    u.len = dt + 5 * F + N;
    u.nbr = reinterpret_cast<const int32_t*>(d + tb);
    u.face = u.nbr + 6 * N;
}

// Reference-layout tables of an unstructured mesh (N x 6 column-major), cells
// in the mesh's numbering when `perm` is given (perm[new] = old), else in the
// caller's.
template <class T>
void unstructured_table(const UConn& c, const int64_t* perm, const int64_t* iperm, int which, void* out) {
    check_uconn(c);
    UGeometry<T> g;
    build_ugeometry<T>(g, c);
    const int64_t N = c.N;
    T* ot = static_cast<T*>(out);
    int64_t* oi = static_cast<int64_t*>(out);
    for (int64_t n = 0; n < N; ++n) {
        const int64_t i = perm ? perm[n] : n;
        switch (which) {
            case CFD_T_VOL: ot[n] = g.vol[i]; continue;
            case CFD_T_CCX: ot[n] = g.ccx[i]; continue;
            case CFD_T_CCY: ot[n] = g.ccy[i]; continue;
            case CFD_T_CCZ: ot[n] = g.ccz[i]; continue;
            default: break;
        }
        bool bnd = false;
        for (int fc = 0; fc < 6; ++fc) {
            const int64_t f = c.cell_faces[6 * i + fc];
            const int64_t a = c.face_cells[2 * f], b = c.face_cells[2 * f + 1];
            const bool fb = b < 0;
            bnd = bnd || fb;
            const int64_t other = fb ? i : (a == i ? b : a);
            const int64_t k = int64_t(fc) * N + n;
            const P3<T> nf{g.fnx[f], g.fny[f], g.fnz[f]};
            const P3<T> ax = HexGeometry<T>::axis_normal(nf, fc);
            const T so = T(g.out_sign[6 * i + fc]);
            switch (which) {
                case CFD_T_IDS: oi[k] = iperm ? iperm[other] : other; break;
                case CFD_T_IDS_BF: oi[k] = fb ? -1 : (iperm ? iperm[other] : other); break;
                case CFD_T_NX: ot[k] = ax.x; break;
                case CFD_T_NY: ot[k] = ax.y; break;
                case CFD_T_NZ: ot[k] = ax.z; break;
                case CFD_T_NAX: ot[k] = so > 0 ? nf.x : -nf.x; break;
                case CFD_T_NAY: ot[k] = so > 0 ? nf.y : -nf.y; break;
                case CFD_T_NAZ: ot[k] = so > 0 ? nf.z : -nf.z; break;
                case CFD_T_AREA: ot[k] = g.farea[f]; break;
                case CFD_T_ALPHA: ot[k] = g.falpha[f]; break;
                case CFD_T_LEN: ot[k] = g.len[6 * i + fc]; break;
                default: break;
            }
        }
        if (which == CFD_T_IS_BND) ot[n] = bnd ? T(1) : T(0);
    }
    CFD_REQUIRE(which >= CFD_T_IDS && which <= CFD_T_CCZ, "unstructured meshes have the reference tables 0 to 15");
}

#define CFD_U_INSTANTIATE(T)                                                                                   \
    template void launch_ugrad<T>(const cfd_mesh_s*, const void*, void*, int, int, hipStream_t);              \
    template void launch_ulapl<T>(const cfd_mesh_s*, const void*, void*, int, hipStream_t);                   \
    template void launch_ustab<T>(const cfd_mesh_s*, const void*, void*, int, void*, hipStream_t);            \
    template void launch_uwave<T>(const cfd_mesh_s*, void* const[4], void* const[4], double, const void*,      \
                                  double, int64_t, hipStream_t);                                               \
    template void launch_uheat<T>(const cfd_mesh_s*, void*, void*, double, const void*, double, int64_t,       \
                                  hipStream_t);                                                                \
    template void create_unstructured<T>(cfd_mesh_s*, int);                                                    \
    template void unstructured_table<T>(const UConn&, const int64_t*, const int64_t*, int, void*);
CFD_U_INSTANTIATE(float)
CFD_U_INSTANTIATE(double)

}  // namespace cfd
