// Adjoint of the fused acoustic step on uniform meshes (no reference
// counterpart), for gradients of sensor-trace misfits with respect to the
// initial pressure and a per-cell K = -c^2 field.
//
// Forward step S (the fused step of the wave kernels, same operation order):
//   u' = u - dt Gx p,  v' = v - dt Gy p,  w' = w - dt Gz p
//   p' = p + dt K (Dx u' + Dy v' + Dz w')
// G_a is the Green-Gauss gradient with the reference boundary rule
// (neighbour = self) and D_a the same with zero normal velocity on the walls.
// On a uniform mesh the two are negative transposes of each other
// (summation by parts: interior rows are h (q_{i+1} - q_{i-1}), the boundary
// rows of G are h (q_1 - q_0) and h (q_{n-1} - q_{n-2}), those of D are
// h (q_0 + q_1) and -h (q_{n-2} + q_{n-1}), h = A / 2V), so G^T = -D and
// D^T = -G, and the transposed step S^T is again a fused two-stage stencil:
//   mu_a = lam_a - G_a(q),  q = (dt K) lam_p
//   nu_p = lam_p + dt (Dx mu_x + Dy mu_y + Dz mu_z)
// The K gradient adds lam_p(t) dt (D . vel(s_t)) per step, with the forward
// velocities of step t recomputed from checkpoints.
//
// Sensor traces: the forward kernel writes p' at up to 64 sensor cells, the
// adjoint kernel adds the trace gradients of the previous step to nu_p there.
// Kernels: adj_star.hip (form 0) and adj_row.hip (form 1).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"
#include "row.hpp"
#include "star_wave.hpp"

namespace cfd {

// star form (adj_star.hip)
star::SensorSet sensor_set(const cfd_mesh_s* m, const SensorList& l);
template <class T>
void launch_wave_star_aux(const cfd_mesh_s* m, int mode, const void* const in[4], void* const out[4], double K,
                          const void* Kf, double dt, const star::SensorSet& sens, const star::WaveAux<T>& aux,
                          hipStream_t s);

// row form (adj_row.hip)
template <class T> bool adj_row_usable(const cfd_mesh_s* m, const void* const* fields, int n, bool grad_K);
template <class T>
void launch_wave_row_aux(const cfd_mesh_s* m, int mode, const void* const in[4], void* const out[4], double K,
                         const void* Kf, double dt, const SensorList* sens, const row::RowAux<T>& aux, int rev,
                         hipStream_t s);

// A device copy of the sensor list for the row-form kernels, which read it
// from memory the caches keep (the kernel-argument copy of 1.5 KB costs each
// workgroup a slow first read), followed by the single-step row tiles' per-tile
// sensor masks.  One pool block; the copy is waited for, so the host staging
// vector may go.
template <class T> std::vector<uint64_t> adj_row_tile_sensors(const cfd_mesh_s* m, const SensorList& sens);
struct DevSensors {
    const SensorList* list = nullptr;
    const uint64_t* tiles = nullptr;
    void* block = nullptr;
};
template <class T> static DevSensors upload_sensors(const cfd_mesh_s* m, const SensorList& sens, hipStream_t s) {
    const std::vector<uint64_t> tiles = adj_row_tile_sensors<T>(m, sens);
    const size_t lb = (sizeof(SensorList) + 255) / 256 * 256;
    std::vector<char> host(lb + tiles.size() * sizeof(uint64_t), 0);
    std::memcpy(host.data(), &sens, sizeof(SensorList));
    std::memcpy(host.data() + lb, tiles.data(), tiles.size() * sizeof(uint64_t));
    DevSensors d;
    d.block = pool_alloc(m->ctx, int64_t(host.size()), s);
    hipError_t e = hipMemcpyAsync(d.block, host.data(), host.size(), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        pool_free(m->ctx, d.block, s);
        CFD_HIP(e);
    }
    d.list = static_cast<const SensorList*>(d.block);
    d.tiles = reinterpret_cast<const uint64_t*>(static_cast<char*>(d.block) + lb);
    return d;
}

// lam_p[sensor j] += src[j]
template <class T> __global__ void scatter_add_k(T* __restrict__ lp, SensorList sens, const T* __restrict__ src) {
    const int j = threadIdx.x;
    if (j < sens.n) {
        const int64_t cell = sens.cell[j];
        lp[cell] = lp[cell] + src[j];
    }
}

SensorList make_sensors(const cfd_mesh_s* m, const int64_t* cells, int n) {
    CFD_REQUIRE(n >= 0 && n <= kMaxSensors, "sensor count must be in [0, 64]");
    CFD_REQUIRE(n == 0 || cells != nullptr, "null sensor list");
    CFD_REQUIRE(m->X * m->Y <= int64_t(0x7fffffff), "mesh too large for sensor rows");
    SensorList s{};
    s.n = n;
    for (int j = 0; j < n; ++j) {
        CFD_REQUIRE(cells[j] >= 0 && cells[j] < m->N, "sensor cell out of range");
        for (int i = 0; i < j; ++i) CFD_REQUIRE(cells[i] != cells[j], "duplicate sensor cell");
        s.cell[j] = cells[j];
        s.row[j] = int(cells[j] / m->Z);
        s.x[j] = int(cells[j] / (m->Z * m->Y));
        s.y[j] = int((cells[j] / m->Z) % m->Y);
        s.z[j] = int(cells[j] % m->Z);
    }
    return s;
}

template <class T> void launch_scatter_add(void* lp, const SensorList& sens, const void* src, hipStream_t s) {
    if (sens.n == 0) return;
    scatter_add_k<T><<<1, 64, 0, s>>>((T*)lp, sens, (const T*)src);
}

// ---------------------------------------------------------------------------
// host drivers
// ---------------------------------------------------------------------------

// nsteps forward steps from state_a, ping-pong with state_b; after step t
// (1-based) p at the sensors goes to traces[(t-1) * n]; before steps
// 0, every, 2 every, ... the state {p,u,v,w} is copied to checkpoint k.
template <class T>
void run_wave_traces(const cfd_mesh_s* m, void* const a[4], void* const b[4], double K, const void* Kf, double dt,
                     int64_t nsteps, const SensorList& sens, void* traces, void* ckpt, int64_t every,
                     hipStream_t s) {
    const size_t field = size_t(m->N) * sizeof(T);
    const void* fields[9] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3], Kf};
    const bool rowf = adj_row_usable<T>(m, fields, 9, false);
    auto trace_row = [&](int64_t t) -> T* { return traces ? (T*)traces + t * sens.n : nullptr; };
    const DevSensors ds = rowf ? upload_sensors<T>(m, sens, s) : DevSensors{};
    const SensorList* dsens = ds.list;
    const star::SensorSet set = rowf ? star::SensorSet{} : sensor_set(m, sens);
    try {
        for (int64_t t = 0; t < nsteps; ++t) {
            void* const* in = (t & 1) ? b : a;
            void* const* out = (t & 1) ? a : b;
            if (ckpt && t % every == 0) {
                char* dst = (char*)ckpt + size_t(t / every) * 4 * field;
                for (int f = 0; f < 4; ++f)
                    CFD_HIP(hipMemcpyAsync(dst + f * field, in[f], field, hipMemcpyDeviceToDevice, s));
            }
            T* tr = trace_row(t);
            if (rowf) {
                const row::RowAux<T> aux{T(0), tr, nullptr, nullptr, nullptr, nullptr, ds.tiles};
                launch_wave_row_aux<T>(m, 1, (const void* const*)in, out, K, Kf, dt, dsens, aux, int(t & 1), s);
            } else {
                const star::WaveAux<T> aux{tr, nullptr, 1, nullptr, nullptr, nullptr};
                launch_wave_star_aux<T>(m, 1, (const void* const*)in, out, K, Kf, dt, set, aux, s);
            }
        }
        CFD_HIP(hipGetLastError());
    } catch (...) {
        pool_free(m->ctx, ds.block, s);
        throw;
    }
    pool_free(m->ctx, ds.block, s);
}

// Reverse loop in row form (constant K).  With grad_K, each checkpoint
// segment is recomputed forward in row form, keeping every step's divergence S
// (one field per step) for the K-gradient term (lam_p dt) S_t, and the state
// in two ping-pong buffers.
template <class T>
static void run_wave_adjoint_row(const cfd_mesh_s* m, void* const la[4], void* const lb[4], double K, double dt,
                                 int64_t nsteps, const SensorList& sens, const void* tgrad, const void* ckpt,
                                 int64_t every, void* gK, hipStream_t s) {
    const size_t field = size_t(m->N) * sizeof(T);
    const T dK = T(T(dt) * T(K));
    void* ws = nullptr;     // S of each step of one segment: every fields
    void* st = nullptr;     // recomputed state: 2 x {p, u, v, w}
    const DevSensors ds = upload_sensors<T>(m, sens, s);
    const SensorList* dsens = ds.list;
    try {
        if (gK) {
            ws = pool_alloc(m->ctx, int64_t(every) * int64_t(field), s);
            st = pool_alloc(m->ctx, 8 * int64_t(field), s);
        }
        int64_t done = 0;
        // the trace gradients added after transposed step t (those of step t-1)
        auto src_of = [&](int64_t t) -> const T* {
            return (tgrad && t >= 2) ? (const T*)tgrad + (t - 2) * sens.n : nullptr;
        };
        auto adj_step = [&](int64_t t, const void* s_in) {
            void* const* in = (done & 1) ? lb : la;
            void* const* out = (done & 1) ? la : lb;
            const T* src = src_of(t);
            const row::RowAux<T> aux{dK, nullptr, nullptr, src, (const T*)s_in, s_in ? (T*)gK : nullptr, ds.tiles};
            launch_wave_row_aux<T>(m, 2, (const void* const*)in, out, K, nullptr, dt, dsens, aux, int(done & 1), s);
            ++done;
        };
        int64_t t = nsteps;
        while (t >= 1) {
            if (!gK) {
                adj_step(t, nullptr);
                --t;
                continue;
            }
            const int64_t seg = (t - 1) / every, t0 = seg * every, len = t - t0;
            const char* ck = (const char*)ckpt + size_t(seg) * 4 * field;
            for (int64_t k = 0; k < len; ++k) {  // state t0+k -> t0+k+1
                const void* in[4];
                void* out[4];
                for (int f = 0; f < 4; ++f) {
                    in[f] = k == 0 ? (const void*)(ck + f * field) : (const void*)((char*)st + (size_t(k & 1) * 4 + f) * field);
                    out[f] = (char*)st + (size_t((k + 1) & 1) * 4 + f) * field;
                }
                const row::RowAux<T> aux{T(0), nullptr, (T*)((char*)ws + size_t(k) * field), nullptr, nullptr,
                                         nullptr};
                launch_wave_row_aux<T>(m, 1, in, out, K, nullptr, dt, dsens, aux, int(k & 1), s);
            }
            for (int64_t tt = t; tt > t0; --tt) adj_step(tt, (char*)ws + size_t(tt - t0 - 1) * field);
            t = t0;
        }
        CFD_HIP(hipGetLastError());
    } catch (...) {
        pool_free(m->ctx, ws, s);
        pool_free(m->ctx, st, s);
        pool_free(m->ctx, ds.block, s);
        throw;
    }
    pool_free(m->ctx, ws, s);
    pool_free(m->ctx, st, s);
    pool_free(m->ctx, ds.block, s);
}

// Reverse loop.  adj_a holds the adjoint of the final state (without the last
// step's trace gradients); on return the adjoint of the initial state is in
// adj_a when nsteps is even, adj_b when odd.  grad_K (nullable) accumulates
// dL/dK per cell and needs the checkpoints: each segment of `every` steps is
// recomputed from its checkpoint.
template <class T>
void run_wave_adjoint(const cfd_mesh_s* m, void* const la[4], void* const lb[4], double K, const void* Kf,
                      double dt, int64_t nsteps, const SensorList& sens, const void* tgrad, const void* ckpt,
                      int64_t every, void* gK, hipStream_t s) {
    const int64_t N = m->N;
    const size_t field = size_t(N) * sizeof(T);
    if (tgrad && nsteps >= 1) launch_scatter_add<T>(la[0], sens, (const T*)tgrad + (nsteps - 1) * sens.n, s);
    {
        const void* fields[10] = {la[0], la[1], la[2], la[3], lb[0], lb[1], lb[2], lb[3], gK, ckpt};
        if (!Kf && adj_row_usable<T>(m, fields, 10, gK != nullptr)) {
            run_wave_adjoint_row<T>(m, la, lb, K, dt, nsteps, sens, tgrad, ckpt, every, gK, s);
            return;
        }
    }
    // With grad_K each segment is recomputed forward, keeping every step's
    // divergence S (one field per step); the state ping-pongs between two
    // buffers and the segment's last step stores S alone.
    const int states = every == 1 ? 0 : every == 2 ? 1 : 2;
    void* ws = nullptr;  // S of each step of one segment
    void* st = nullptr;  // recomputed states
    const star::SensorSet set = sensor_set(m, sens);
    try {
        if (gK) {
            ws = pool_alloc(m->ctx, every * int64_t(field), s);
            if (states) st = pool_alloc(m->ctx, states * 4 * int64_t(field), s);
        }
        int64_t done = 0;
        auto adj_step = [&](int64_t t, const void* s_in) {
            void* const* in = (done & 1) ? lb : la;
            void* const* out = (done & 1) ? la : lb;
            const T* src = (tgrad && t >= 2) ? (const T*)tgrad + (t - 2) * sens.n : nullptr;
            const star::WaveAux<T> aux{nullptr, nullptr, 1, src, (const T*)s_in, (T*)gK};
            launch_wave_star_aux<T>(m, 2, (const void* const*)in, out, K, Kf, dt, set, aux, s);
            ++done;
        };
        int64_t t = nsteps;
        while (t >= 1) {
            if (!gK) {
                adj_step(t, nullptr);
                --t;
                continue;
            }
            const int64_t seg = (t - 1) / every, t0 = seg * every, len = t - t0;
            const char* ck = (const char*)ckpt + size_t(seg) * 4 * field;
            for (int64_t k = 0; k < len; ++k) {  // state t0+k -> t0+k+1
                const bool last = k + 1 == len;
                const void* in[4];
                void* out[4];
                for (int f = 0; f < 4; ++f) {
                    in[f] = k == 0 ? (const void*)(ck + f * field)
                                   : (const void*)((char*)st + (size_t((k - 1) & 1) * 4 + f) * field);
                    out[f] = last ? nullptr : (void*)((char*)st + (size_t(k & 1) * 4 + f) * field);
                }
                const star::WaveAux<T> aux{nullptr, (T*)((char*)ws + size_t(k) * field), last ? 0 : 1,
                                           nullptr, nullptr, nullptr};
                launch_wave_star_aux<T>(m, 1, in, out, K, Kf, dt, set, aux, s);
            }
            for (int64_t tt = t; tt > t0; --tt) adj_step(tt, (char*)ws + size_t(tt - t0 - 1) * field);
            t = t0;
        }
        CFD_HIP(hipGetLastError());
    } catch (...) {
        pool_free(m->ctx, ws, s);
        pool_free(m->ctx, st, s);
        throw;
    }
    pool_free(m->ctx, ws, s);
    pool_free(m->ctx, st, s);
}

#define CFD_ADJ_INSTANTIATE(T)                                                                                  \
    template void launch_scatter_add<T>(void*, const SensorList&, const void*, hipStream_t);                   \
    template void run_wave_traces<T>(const cfd_mesh_s*, void* const[4], void* const[4], double, const void*,   \
                                     double, int64_t, const SensorList&, void*, void*, int64_t, hipStream_t);   \
    template void run_wave_adjoint<T>(const cfd_mesh_s*, void* const[4], void* const[4], double, const void*,  \
                                      double, int64_t, const SensorList&, const void*, const void*, int64_t,    \
                                      void*, hipStream_t);
CFD_ADJ_INSTANTIATE(float)
CFD_ADJ_INSTANTIATE(double)

}  // namespace cfd
