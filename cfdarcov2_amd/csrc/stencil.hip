// Operators and explicit steps on the structured hex mesh: Green-Gauss
// gradient, Laplacian, stabilisation, heat and acoustic steps, and the heat
// step's adjoint.  Three geometry forms:
//   uniform  - exactly uniform meshes; geometry is a handful of constants and
//              neighbours are implicit, so only state crosses HBM
//              (ops_star.hip, wave_*.hip, heat_row.hip, heat_multi.hip);
//   lattice  - axis-aligned faces (any spacing): widths and alpha_d per cell
//              layer, volume per cell (ops_faces.hip);
//   general  - per-face SoA geometry (face families z, y, x) for perturbed
//              meshes; neighbours are still implicit (ops_faces.hip).
// All arithmetic follows the reference operation order (see the oracle and
// src/fvm3d.cpp / include/grad_utils.hpp cited per kernel) and the library is
// built with -ffp-contract=off, so FP64 results are bit-identical to a CPU
// evaluation in the same order.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"

namespace cfd {

// ---------------------------------------------------------------------------
// indexing helpers
// ---------------------------------------------------------------------------
struct Cell {
    int64_t x, y, z, id;
    bool valid;
};

template <class G> __device__ inline Cell cell_of_thread(const G& g) {
    Cell c;
    c.z = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    c.y = int64_t(blockIdx.y) * blockDim.y + threadIdx.y;
    c.x = int64_t(blockIdx.z);
    c.valid = c.z < g.Z && c.y < g.Y && c.x < g.X;
    c.id = (c.x * g.Y + c.y) * g.Z + c.z;
    return c;
}

// Neighbour of cell c across its lower / upper face on axis a (0 = x, 1 = y,
// 2 = z); the cell itself on a boundary face (reference rule).
template <class G> __device__ inline int64_t nb_lo(const G& g, const Cell& c, int a) {
    if (a == 0) return c.x > 0 ? c.id - g.Y * g.Z : c.id;
    if (a == 1) return c.y > 0 ? c.id - g.Z : c.id;
    return c.z > 0 ? c.id - 1 : c.id;
}
template <class G> __device__ inline int64_t nb_hi(const G& g, const Cell& c, int a) {
    if (a == 0) return c.x < g.X - 1 ? c.id + g.Y * g.Z : c.id;
    if (a == 1) return c.y < g.Y - 1 ? c.id + g.Z : c.id;
    return c.z < g.Z - 1 ? c.id + 1 : c.id;
}
template <class G> __device__ inline bool at_lo(const G& g, const Cell& c, int a) {
    return a == 0 ? c.x == 0 : a == 1 ? c.y == 0 : c.z == 0;
}
template <class G> __device__ inline bool at_hi(const G& g, const Cell& c, int a) {
    return a == 0 ? c.x == g.X - 1 : a == 1 ? c.y == g.Y - 1 : c.z == g.Z - 1;
}

// ---------------------------------------------------------------------------
// launch helpers
// ---------------------------------------------------------------------------
template <class G> inline dim3 grid_for(const G& g, dim3 blk) {
    return dim3(unsigned((g.Z + blk.x - 1) / blk.x), unsigned((g.Y + blk.y - 1) / blk.y), unsigned(g.X));
}
static const dim3 kBlock(64, 4, 1);

template <class T> const UniformGeo<T>& ugeo(const cfd_mesh_s* m);
template <> const UniformGeo<float>& ugeo<float>(const cfd_mesh_s* m) { return m->ug32; }
template <> const UniformGeo<double>& ugeo<double>(const cfd_mesh_s* m) { return m->ug64; }
inline void check_launch() { CFD_HIP(hipGetLastError()); }

template <class T> void launch_grad(const cfd_mesh_s* m, const void* phi, void* out, int mask, int wall, hipStream_t s) {
    if (m->uniform) launch_grad_star<T>(m, phi, out, mask, wall, s);
    else launch_grad_faces<T>(m, phi, out, mask, wall, s);
}

template <class T> void launch_lapl(const cfd_mesh_s* m, const void* phi, void* out, int mask, hipStream_t s) {
    if (m->uniform) launch_lapl_star<T>(m, phi, out, mask, s);
    else launch_lapl_faces<T>(m, phi, out, mask, s);
}

// scratch3 (3N entries, the first stage's gradients) is needed by meshes with
// face geometry only: uniform meshes run the one-pass kernel
template <class T>
void launch_stab(const cfd_mesh_s* m, const void* phi, void* out, int mask, void* scratch3, hipStream_t s) {
    if (m->uniform) {
        launch_stab_star<T>(m, phi, out, mask, s);
    } else {
        CFD_REQUIRE(scratch3 != nullptr, "stabilisation on a general mesh needs 3N scratch entries");
        launch_stab_faces<T>(m, phi, out, mask, scratch3, s);
    }
}

template <class T>
void launch_heat(const cfd_mesh_s* m, void* Ta, void* Tb, double alpha, const void* af, double dt, int64_t nsteps,
                 hipStream_t s) {
    int64_t k0 = 0;
    if (m->uniform && !af && m->heat_variant == 2 && nsteps > 0) {
        // up to K steps per launch in LDS, reading one buffer and writing the
        // other: the number of launches has the parity of nsteps, so the
        // state ends where single steps leave it, and the steps are spread
        // evenly over the launches
        const auto& g = ugeo<T>(m);
        const int K = m->heat_L;
        int64_t launches = (nsteps + K - 1) / K;
        if ((launches - nsteps) % 2 != 0) ++launches;
        for (int64_t l = 0; l < launches; ++l) {
            const int64_t done = nsteps * l / launches, next = nsteps * (l + 1) / launches;
            const void* in = (l & 1) ? Tb : Ta;
            void* out = (l & 1) ? Ta : Tb;
            launch_heat_multi<T>(g, in, out, alpha, dt, m->heat_nw, K, int(next - done), s);
        }
        return;
    }
    if (m->uniform && !af && m->heat_variant == 1) {
        // two steps per launch, in pairs (Ta -> Tb -> Ta) so the state ends
        // where single steps leave it; the remaining steps run one per launch
        const auto& g = ugeo<T>(m);
        for (; k0 + 4 <= nsteps; k0 += 4) {
            if (!launch_heat_row2<T>(g, Ta, Tb, alpha, dt, m->heat_nw, m->heat_L, s)) break;
            launch_heat_row2<T>(g, Tb, Ta, alpha, dt, m->heat_nw, m->heat_L, s);
        }
    }
    // meshes that a launch outlasts (heat2_star_k): two steps per launch, in
    // pairs for the same reason
    if (m->uniform && m->heat_variant == 0 && m->N <= kHeat2Cells) {
        for (; k0 + 4 <= nsteps; k0 += 4) {
            launch_heat2_star<T>(m, Ta, Tb, alpha, af, dt, s);
            launch_heat2_star<T>(m, Tb, Ta, alpha, af, dt, s);
        }
    }
    for (int64_t k = k0; k < nsteps; ++k) {
        const T* in = (const T*)((k & 1) ? Tb : Ta);
        T* out = (T*)((k & 1) ? Ta : Tb);
        if (m->uniform) launch_heat_star<T>(m, in, out, alpha, af, dt, s);
        else launch_heat_faces<T>(m, in, out, alpha, af, dt, s);
    }
}

template <class T>
void launch_wave(const cfd_mesh_s* m, void* const a[4], void* const b[4], double K, const void* Kf, double dt,
                 int64_t nsteps, hipStream_t s) {
    if (!m->uniform) {
        for (int64_t k = 0; k < nsteps; ++k)
            launch_wave_faces<T>(m, (k & 1) ? b : a, (k & 1) ? a : b, K, Kf, dt, s);
        return;
    }
    launch_wave_march<T>(m, a, b, K, Kf, dt, nsteps, m->wave_variant, m->wave_ty, m->wave_L, m->wave_remap, s);
}

// ---------------------------------------------------------------------------
// Adjoint of the heat step on uniform meshes (no reference counterpart).
// The step is H = I + dt K L, K = diag(k) with k the constant alpha or the
// alpha field, L the Laplacian of heat_star_k.  On a uniform mesh L is
// symmetric (an interior face couples its two cells with the same
// alpha_d A / V, a wall face couples nothing), so H^T = I + dt L K:
//   constant alpha:  H^T = H, the forward kernels themselves;
//   alpha field:     (H^T mu)_i = dt L(k o mu)_i + mu_i   (heat_adj_field_k).
// dL/dk_i = sum over steps t of mu_t,i dt L(T_{t-1})_i (heat_grad_alpha_k),
// the forward states T_{t-1} recomputed from checkpoints.
// ---------------------------------------------------------------------------

// L(k o f) at cell c (L(f) when kf is null), heat_star_k's operation
// order; on a wall the neighbour is the cell itself and its term is zero
template <class T, bool PW>
__device__ inline T lapl_scaled(const UniformGeo<T>& g, const Cell& c, const T* __restrict__ f,
                                const T* __restrict__ kf) {
    auto val = [&](int64_t j) { return kf ? kf[j] * f[j] : f[j]; };
    const T pc = val(c.id);
    T L = T(0);
    for (int a = 0; a < 3; ++a) {
        const T al_lo = at_lo(g, c, a) ? g.alpha_b[a] : g.alpha[a];
        const T al_hi = at_hi(g, c, a) ? g.alpha_b[a] : g.alpha[a];
        const T s_lo = (-pc + val(nb_lo(g, c, a))) * al_lo;
        const T s_hi = (-pc + val(nb_hi(g, c, a))) * al_hi;
        const T num = s_lo * g.area[a] + s_hi * g.area[a];
        if constexpr (PW) L = L + num * g.inv_vol;
        else L = L + num / g.vol;
    }
    return L;
}

template <class T, bool PW>
__global__ void __launch_bounds__(256) heat_adj_field_k(UniformGeo<T> g, const T* __restrict__ mu,
                                                        T* __restrict__ out, const T* __restrict__ kf, T dt) {
    const Cell c = cell_of_thread(g);
    if (!c.valid) return;
    out[c.id] = dt * lapl_scaled<T, PW>(g, c, mu, kf) + mu[c.id];
}

template <class T, bool PW>
__global__ void __launch_bounds__(256) heat_grad_alpha_k(UniformGeo<T> g, const T* __restrict__ mu,
                                                         const T* __restrict__ Tprev, T* __restrict__ gk, T dt) {
    const Cell c = cell_of_thread(g);
    if (!c.valid) return;
    gk[c.id] = gk[c.id] + (dt * lapl_scaled<T, PW>(g, c, Tprev, nullptr)) * mu[c.id];
}

template <class T> __global__ void gather_sensors_k(const T* __restrict__ f, SensorList s, T* __restrict__ out) {
    const int j = int(threadIdx.x);
    if (j < s.n) out[j] = f[s.cell[j]];
}

// nsteps heat steps from Ta, ping-pong with Tb; after step t (1-based) T at
// the sensors goes to traces[(t-1) * n]; before steps 0, every, 2 every, ...
// the state is copied to checkpoint k.
template <class T>
void run_heat_traces(const cfd_mesh_s* m, void* Ta, void* Tb, double alpha, const void* af, double dt,
                     int64_t nsteps, const SensorList& sens, void* traces, void* ckpt, int64_t every,
                     hipStream_t s) {
    const size_t field = size_t(m->N) * sizeof(T);
    for (int64_t t = 0; t < nsteps; ++t) {
        void* in = (t & 1) ? Tb : Ta;
        void* out = (t & 1) ? Ta : Tb;
        if (ckpt && t % every == 0)
            CFD_HIP(hipMemcpyAsync((char*)ckpt + size_t(t / every) * field, in, field, hipMemcpyDeviceToDevice, s));
        launch_heat<T>(m, in, out, alpha, af, dt, 1, s);
        if (traces && sens.n) {
            gather_sensors_k<T><<<1, 64, 0, s>>>((const T*)out, sens, (T*)traces + t * sens.n);
            check_launch();
        }
    }
}

// The transposed steps in reverse order from adj_a (the adjoint of the final
// state), the trace gradients of step t added at the sensors before the
// transposed step t; the result is in adj_a (nsteps even) or adj_b (odd).
template <class T>
void run_heat_adjoint(const cfd_mesh_s* m, void* la, void* lb, double alpha, const void* af, double dt,
                      int64_t nsteps, const SensorList& sens, const void* tgrad, const void* ckpt, int64_t every,
                      void* gA, hipStream_t s) {
    const auto& g = ugeo<T>(m);
    const size_t field = size_t(m->N) * sizeof(T);
    void* ws = nullptr;  // the forward states of one checkpoint segment
    if (gA) ws = pool_alloc(m->ctx, int64_t(every) * int64_t(field), s);
    try {
        int64_t done = 0;
        auto step = [&](int64_t t, const void* Tprev) {
            void* in = (done & 1) ? lb : la;
            void* out = (done & 1) ? la : lb;
            if (tgrad) launch_scatter_add<T>(in, sens, (const T*)tgrad + (t - 1) * sens.n, s);
            if (gA) {
                if (g.vol_pow2)
                    heat_grad_alpha_k<T, true><<<grid_for(g, kBlock), kBlock, 0, s>>>(g, (const T*)in, (const T*)Tprev,
                                                                                   (T*)gA, T(dt));
                else
                    heat_grad_alpha_k<T, false><<<grid_for(g, kBlock), kBlock, 0, s>>>(g, (const T*)in,
                                                                                    (const T*)Tprev, (T*)gA, T(dt));
                check_launch();
            }
            if (af) {
                if (g.vol_pow2)
                    heat_adj_field_k<T, true><<<grid_for(g, kBlock), kBlock, 0, s>>>(g, (const T*)in, (T*)out,
                                                                                  (const T*)af, T(dt));
                else
                    heat_adj_field_k<T, false><<<grid_for(g, kBlock), kBlock, 0, s>>>(g, (const T*)in, (T*)out,
                                                                                   (const T*)af, T(dt));
                check_launch();
            } else {
                launch_heat<T>(m, in, out, alpha, nullptr, dt, 1, s);
            }
            ++done;
        };
        int64_t t = nsteps;
        while (t >= 1) {
            if (!gA) {
                step(t, nullptr);
                --t;
                continue;
            }
            // states T_{t0} .. T_{t-1} of this segment, from its checkpoint
            const int64_t seg = (t - 1) / every, t0 = seg * every, len = t - t0;
            CFD_HIP(hipMemcpyAsync(ws, (const char*)ckpt + size_t(seg) * field, field, hipMemcpyDeviceToDevice, s));
            for (int64_t k = 1; k < len; ++k)
                launch_heat<T>(m, (char*)ws + size_t(k - 1) * field, (char*)ws + size_t(k) * field, alpha, af, dt, 1,
                               s);
            for (int64_t tt = t; tt > t0; --tt) step(tt, (const char*)ws + size_t(tt - 1 - t0) * field);
            t = t0;
        }
    } catch (...) {
        if (ws) pool_free(m->ctx, ws, s);
        throw;
    }
    if (ws) pool_free(m->ctx, ws, s);
}

#define CFD_INSTANTIATE(T)                                                                                       \
    template void run_heat_traces<T>(const cfd_mesh_s*, void*, void*, double, const void*, double, int64_t,     \
                                     const SensorList&, void*, void*, int64_t, hipStream_t);                    \
    template void run_heat_adjoint<T>(const cfd_mesh_s*, void*, void*, double, const void*, double, int64_t,    \
                                      const SensorList&, const void*, const void*, int64_t, void*, hipStream_t); \
    template void launch_grad<T>(const cfd_mesh_s*, const void*, void*, int, int, hipStream_t);                \
    template void launch_lapl<T>(const cfd_mesh_s*, const void*, void*, int, hipStream_t);                     \
    template void launch_stab<T>(const cfd_mesh_s*, const void*, void*, int, void*, hipStream_t);              \
    template void launch_heat<T>(const cfd_mesh_s*, void*, void*, double, const void*, double, int64_t,         \
                                 hipStream_t);                                                                   \
    template void launch_wave<T>(const cfd_mesh_s*, void* const*, void* const*, double, const void*, double,    \
                                 int64_t, hipStream_t);
CFD_INSTANTIATE(float)
CFD_INSTANTIATE(double)

}  // namespace cfd
