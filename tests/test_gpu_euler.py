"""GPU parity of the Rusanov Euler stepper (cfd_euler_run) against the oracle,
and the Sod workload's full-size properties.

The kernel and the oracle evaluate the same operation sequence with no FMA
contraction and correctly rounded division and square root, so the fields and
every step's dt are compared for exact equality in FP64 and FP32.  The FP32
run's error against the FP64 oracle is reported per field and must stay within
twice the FP32 oracle's own error."""
import numpy as np
import pytest

from cfdarcov2_amd import workloads
from tests import riemann_exact

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _gpu_run(hip_ctx, n, d, off, dtype, U0, gamma, cfl, steps, shape=None):
    from cfdarcov2_amd import capi
    gm = capi.HexMesh(hip_ctx, *n, *d, dtype=dtype, vertex_offsets=off)
    if shape is not None:
        gm.set_euler_shape(*shape)
    A = [torch.from_numpy(np.ascontiguousarray(U0[k], dtype=dtype)).cuda() for k in range(5)]
    B = [torch.empty_like(a) for a in A]
    hist = torch.empty(max(steps, 1), dtype=A[0].dtype, device="cuda")
    res = gm.euler_run(A, B, gamma, cfl, steps, hist)
    torch.cuda.synchronize()
    out = np.stack([t.cpu().numpy() for t in res])
    h = hist.cpu().numpy()[:steps]
    gm.close()
    return out, h


CASES = [
    # name, shape, perturbation seed (None = uniform), steps
    ("uniform-1d", (40, 1, 1), None, 30),
    ("uniform-3d", (20, 7, 9), None, 20),
    ("perturbed", (24, 10, 12), 3, 25),
    ("perturbed-wide", (70, 6, 5), 8, 15),
]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_euler_matches_oracle(hip_ctx, oracle_lib, case, dtype):
    name, n, seed, steps = case
    print(f"\n[case] euler {name} {np.dtype(dtype).name} n={n} steps={steps}", flush=True)
    d = (1.0 / n[0],) * 3
    off = None if seed is None else workloads.perturbed_vertex_offsets(*n, *d, seed=seed, frac=0.2)
    om = oracle_lib.OracleMesh(*n, *d, dtype=dtype, perturb=off)
    U0 = workloads.sod_state(om.table("ccx"), dtype=dtype)
    if name == "uniform-3d":  # add transverse motion so every flux term is live
        rng = np.random.default_rng(2)
        U0[1:4] = (0.1 * rng.standard_normal((3, om.N)) * U0[0]).astype(dtype)
    ref, ref_dt = om.euler_run(U0, 1.4, 0.3, steps)
    got, got_dt = _gpu_run(hip_ctx, n, d, off, dtype, U0, 1.4, 0.3, steps)
    assert np.all(np.isfinite(ref))
    assert np.array_equal(got_dt, ref_dt), np.max(np.abs(got_dt - ref_dt))
    for k in range(5):
        assert np.array_equal(got[k], ref[k]), (k, np.max(np.abs(got[k] - ref[k])))


SHAPES = [(0, 4, 16), (1, 2, 5), (1, 4, 16), (1, 8, 3), (1, 4, 64)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", SHAPES, ids=[f"v{a}-ty{b}-L{c}" for a, b, c in SHAPES])
def test_euler_kernel_shapes(hip_ctx, oracle_lib, shape, dtype):
    """Per-thread and 2.5D-march forms, partial tiles in y and z, two z tiles
    and chunks that do not divide x: the oracle's bits, fields and time steps."""
    n, steps = (23, 9, 70), 9
    print(f"\n[case] euler shape {shape} {np.dtype(dtype).name}", flush=True)
    if dtype == np.float64 and shape[0] == 1 and shape[1] == 8:
        # the FP64 8-row march build would spill registers: rejected
        from cfdarcov2_amd import capi
        gm = capi.HexMesh(hip_ctx, *n, *(1.0 / 23,) * 3, dtype=dtype)
        with pytest.raises(capi.CfdError):
            gm.set_euler_shape(*shape)
        gm.close()
        return
    d = (1.0 / 23,) * 3
    off = workloads.perturbed_vertex_offsets(*n, *d, seed=4, frac=0.2)
    om = oracle_lib.OracleMesh(*n, *d, dtype=dtype, perturb=off)
    U0 = workloads.sod_state(om.table("ccx"), dtype=dtype)
    rng = np.random.default_rng(6)
    U0[1:4] = (0.05 * rng.standard_normal((3, om.N)) * U0[0]).astype(dtype)
    ref, ref_dt = om.euler_run(U0, 1.4, 0.3, steps)
    got, got_dt = _gpu_run(hip_ctx, n, d, off, dtype, U0, 1.4, 0.3, steps, shape)
    assert np.array_equal(got_dt, ref_dt)
    for k in range(5):
        assert np.array_equal(got[k], ref[k]), k


def test_fp32_error_against_fp64_oracle(hip_ctx, oracle_lib):
    n, steps = (48, 8, 8), 40
    d = (1.0 / 48,) * 3
    off = workloads.perturbed_vertex_offsets(*n, *d, seed=1, frac=0.2)
    o64 = oracle_lib.OracleMesh(*n, *d, dtype=np.float64, perturb=off)
    o32 = oracle_lib.OracleMesh(*n, *d, dtype=np.float32, perturb=off)
    U64, _ = o64.euler_run(workloads.sod_state(o64.table("ccx")), 1.4, 0.3, steps)
    U32, _ = o32.euler_run(workloads.sod_state(o32.table("ccx"), dtype=np.float32), 1.4, 0.3, steps)
    got, _ = _gpu_run(hip_ctx, n, d, off, np.float32, workloads.sod_state(o32.table("ccx"), dtype=np.float32),
                      1.4, 0.3, steps)
    for k, name in zip((0, 1, 4), ("rho", "rho_u", "E")):
        err_cpu = np.sum(np.abs(U32[k] - U64[k])) / np.sum(np.abs(U64[k]))
        err_gpu = np.sum(np.abs(got[k] - U64[k])) / np.sum(np.abs(U64[k]))
        print(f"[fp32 vs fp64] {name}: gpu rel L1 {err_gpu:.3e}, cpu fp32 oracle {err_cpu:.3e}")
        assert err_gpu <= 2 * err_cpu + 1e-12


def test_sod_against_exact_riemann(hip_ctx, oracle_lib):
    """Uniform tube, 400 cells along x: the density profile is within the
    scheme's first-order L1 error of the exact solution."""
    n = (400, 2, 2)
    d = (1.0 / 400,) * 3
    om = oracle_lib.OracleMesh(*n, *d, dtype=np.float64)
    x = om.table("ccx")
    U0 = workloads.sod_state(x)
    got, dts = _gpu_run(hip_ctx, n, d, None, np.float64, U0, 1.4, 0.3, 240)
    t = float(np.sum(dts))
    rho_ex, u_ex, p_ex = riemann_exact.sod(x, t)
    assert np.mean(np.abs(got[0] - rho_ex)) < 0.005
    assert np.mean(np.abs(got[1] / got[0] - u_ex)) < 0.02


def test_sod_full_size_properties(hip_ctx):
    """512 x 64 x 64, interior vertices moved by up to 20% of dx, FP32, 500
    steps at CFL 0.3: finite, positive density and pressure, mass and energy
    conserved (reflective walls), positive time steps, the right-moving shock
    ahead of the contact."""
    from cfdarcov2_amd import capi
    cfg = workloads.sod_config()
    n, d = cfg.n, cfg.spacing
    print(f"\n[case] euler full size n={n} steps={cfg.steps}", flush=True)
    gm = capi.HexMesh(hip_ctx, *n, *d, dtype=np.float32, vertex_offsets=cfg.vertex_offsets)
    ccx = gm.table("ccx")
    vol = gm.table("fv_vol").astype(np.float64)
    assert np.all(vol > 0)
    U0 = workloads.sod_state(ccx, dtype=np.float32)
    A = [torch.from_numpy(U0[k].copy()).cuda() for k in range(5)]
    B = [torch.empty_like(a) for a in A]
    hist = torch.empty(cfg.steps, dtype=torch.float32, device="cuda")
    res = gm.euler_run(A, B, cfg.gamma, cfg.cfl, cfg.steps, hist)
    torch.cuda.synchronize()
    U = np.stack([t.cpu().numpy() for t in res]).astype(np.float64)
    dts = hist.cpu().numpy()
    assert np.all(np.isfinite(U)) and np.all(dts > 0)
    for k in (0, 4):
        before = np.sum(vol * U0[k].astype(np.float64))
        after = np.sum(vol * U[k])
        assert abs(after - before) <= 1e-5 * abs(before), (k, before, after)
    rho = U[0]
    p = 0.4 * (U[4] - 0.5 * (U[1] ** 2 + U[2] ** 2 + U[3] ** 2) / rho)
    assert rho.min() > 0.1 and p.min() > 0.09
    t = float(np.sum(dts.astype(np.float64)))
    # column-averaged density against the exact solution
    X = n[0]
    rho_x = rho.reshape(X, -1).mean(axis=1)
    x_c = ccx.reshape(X, -1).mean(axis=1)
    rho_ex, _, _ = riemann_exact.sod(x_c, t)
    assert np.mean(np.abs(rho_x - rho_ex)) < 0.01
    gm.close()


# Cells-in-a-row tiles of the march: planes that fill a tile, end inside one or
# need several, rows of one cell and of half a tile, chunks of one plane to
# more than the mesh; on perturbed (face arrays), decimal (layer widths) and
# dyadic (constants) meshes.
TILE_CASES = [((9, 16, 32), (1, 2, 1)), ((7, 13, 20), (1, 2, 3)), ((6, 1, 1), (1, 4, 2)), ((5, 130, 1), (1, 2, 4)),
              ((12, 9, 64), (1, 2, 16)), ((4, 11, 128), (1, 4, 2)), ((3, 9, 200), (1, 8, 5)), ((17, 24, 23), None),
              ((40, 12, 300), None)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["perturbed", "decimal", "dyadic"])
@pytest.mark.parametrize("n,shape", TILE_CASES, ids=lambda v: "x".join(map(str, v)) if v else "auto")
def test_euler_tiles(hip_ctx, oracle_lib, n, shape, kind, dtype):
    if dtype == np.float64 and shape and shape[1] == 8:
        shape = (1, 4, shape[2])
    d = (0.125, 0.25, 0.125) if kind == "dyadic" else (0.1, 0.07, 0.09)
    off = workloads.perturbed_vertex_offsets(*n, *d, seed=4, frac=0.2) if kind == "perturbed" else None
    om = oracle_lib.OracleMesh(*n, *d, dtype=dtype, perturb=off)
    rng = np.random.default_rng(9)
    U0 = np.empty((5, om.N), dtype=dtype)
    U0[0] = 1.0 + 0.5 * rng.random(om.N)
    U0[1:4] = 0.2 * rng.standard_normal((3, om.N))
    U0[4] = 3.0 + rng.random(om.N)
    ref, ref_dt = om.euler_run(U0, 1.4, 0.3, 5)
    got, got_dt = _gpu_run(hip_ctx, n, d, off, dtype, U0, 1.4, 0.3, 5, shape)
    assert np.all(np.isfinite(ref))
    assert np.array_equal(got_dt, ref_dt)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("kind", ["decimal", "dyadic"])
def test_euler_axis_aligned_equals_face_arrays(hip_ctx, kind):
    """Axis-aligned geometry against the face arrays of the same mesh (forced
    general), with infinite and NaN cells: the same values, NaN in the same
    places."""
    from cfdarcov2_amd import capi
    n, d = (14, 9, 12), (0.125,) * 3 if kind == "dyadic" else (0.1, 0.07, 0.09)
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(1)
    for special in (None, np.inf, -np.inf, np.nan):
        for field in range(5) if special is not None else (0,):
            U0 = np.stack([1.0 + 0.3 * rng.random(N), *(0.2 * rng.standard_normal((3, N))), 3.0 + rng.random(N)])
            if special is not None:
                U0[field, rng.integers(N, size=3)] = special
            res = []
            for force in (False, True):
                gm = capi.HexMesh(hip_ctx, *n, *d, dtype="f64", force_general=force)
                A = [torch.from_numpy(U0[k].copy()).cuda() for k in range(5)]
                B = [torch.empty_like(a) for a in A]
                hist = torch.empty(3, dtype=torch.float64, device="cuda")
                out = gm.euler_run(A, B, 1.4, 0.3, 3, hist)
                res.append([t.cpu().numpy() for t in out] + [hist.cpu().numpy()])
                gm.close()
            for k, (x, y) in enumerate(zip(*res)):
                assert np.array_equal(x, y, equal_nan=True), (special, field, k)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["decimal", "dyadic"])
@pytest.mark.parametrize("first,then", [((-1, 4, 16), (0, 4, 16)), ((1, 4, 2), (1, 2, 2)), ((0, 4, 16), (-1, 4, 16))],
                         ids=["auto-cell", "tile-march", "cell-auto"])
def test_euler_capture_after_a_change_of_shape(hip_ctx, first, then, kind, dtype):
    """A mesh that has run once can change its shape (and with it the geometry
    the kernels read) and have the next run captured: every replay, with eager
    work and synchronisations between, equals the eager run."""
    from cfdarcov2_amd import capi
    n, d = (6, 5, 100), (0.125,) * 3 if kind == "dyadic" else (0.1, 0.07, 0.09)
    gm = capi.HexMesh(hip_ctx, *n, *d, dtype=dtype)
    rng = np.random.default_rng(3)
    U0 = [1.0 + 0.3 * rng.random(gm.N), *(0.2 * rng.standard_normal((3, gm.N))), 3.0 + rng.random(gm.N)]
    U0 = [torch.from_numpy(u.astype(dtype)).cuda() for u in U0]
    A, B = [u.clone() for u in U0], [torch.empty_like(u) for u in U0]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        gm.set_euler_shape(*first)
        ref = [t.clone() for t in gm.euler_run(A, B, 1.4, 0.3, 4)]
        gm.set_euler_shape(*then)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            gm.euler_run(A, B, 1.4, 0.3, 4)
        for _ in range(3):
            for a, u in zip(A, U0):
                a.copy_(u)
            graph.replay()
            torch.randn(1 << 18, device="cuda").sum().item()
            assert all(torch.equal(a, r) for a, r in zip(A, ref))
    torch.cuda.synchronize()
    del graph
    gm.close()
