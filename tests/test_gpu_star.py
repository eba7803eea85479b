"""Star-form kernels (16 bytes of consecutive z-cells per thread, no march) on
rows that are not a multiple of the vector width, shorter than it, and on
one- to three-cell extents, with fields that start at any element: the
oracle's bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# z extents around the vector widths (4 in FP32, 2 in FP64) and the workgroup's
# units; x and y extents where a cell's two neighbours on each side are walls
EXTENTS = [(1, 1, 1), (2, 1, 2), (3, 2, 3), (1, 3, 4), (5, 4, 5), (4, 5, 7), (2, 3, 130), (3, 2, 1030), (6, 67, 9)]
# above the sizes that take one cell per thread: FP64, and both
VECTOR = [(24, 90, 67), (40, 121, 131)]


def _view(a, dtype, shift):
    """Device copy of `a` starting `shift` elements into a buffer."""
    buf = torch.zeros(a.size + shift, dtype=torch.float32 if dtype == np.float32 else torch.float64, device="cuda")
    buf[shift:].copy_(torch.from_numpy(np.ascontiguousarray(a, dtype=dtype)))
    return buf[shift:]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", EXTENTS + VECTOR, ids=lambda n: "x".join(map(str, n)))
def test_wave_star(hip_ctx, oracle_lib, n, shift, dtype):
    from cfdarcov2_amd import capi
    d = (0.125, 0.25, 0.5) if shift else (0.125, 0.125, 0.125)
    gm = capi.HexMesh(hip_ctx, *n, *d, dtype=dtype)
    gm.set_wave_shape(0, 4, 8, 0)
    om = oracle_lib.OracleMesh(*n, *d, dtype=dtype)
    rng = np.random.default_rng(11)
    f = [rng.standard_normal(om.N).astype(dtype) for _ in range(4)]
    K = (-(0.5 + rng.random(om.N)) ** 2).astype(dtype)
    for kf in (None, K):
        A = [_view(a, dtype, shift) for a in f]
        B = [_view(np.zeros_like(a), dtype, shift) for a in f]
        got = gm.wave_run(A, B, -1.0, 0.03, 5, K_field=None if kf is None else _view(kf, dtype, shift))
        ref = om.wave_run(*f, -1.0, 0.03, 5, K_field=kf)
        for name, g, r in zip("puvw", got, ref):
            assert np.array_equal(g.cpu().numpy(), r), f"field {name}, K field {kf is not None}"
    gm.close()


def _mesh(hip_ctx, oracle_lib, n, kind, dtype):
    """(star mesh, the same mesh in general form, oracle) of a uniform, decimal or graded lattice or a skewed mesh."""
    from cfdarcov2_amd import capi
    off, d = None, (0.125, 0.25, 0.5) if kind == "dyadic" else (0.1, 0.3, 0.7)
    if kind == "graded":  # vertex layers moved along their own axis
        g = np.meshgrid(*[0.05 * s * (np.arange(k + 1) % 3) for k, s in zip(n, d)], indexing="ij")
        off = np.stack([a.ravel() for a in g], axis=1)
    elif kind == "skewed":
        off = np.random.default_rng(8).uniform(-0.02, 0.02, ((n[0] + 1) * (n[1] + 1) * (n[2] + 1), 3))
    gm = capi.HexMesh(hip_ctx, *n, *d, dtype=dtype, vertex_offsets=off)
    gg = capi.HexMesh(hip_ctx, *n, *d, dtype=dtype, vertex_offsets=off, force_general=True)
    assert gg.info().uniform == 0
    if kind == "dyadic":
        assert gm.info().uniform == 1
    elif kind != "skewed" and min(n) > 3:  # (one or two layers can be exactly uniform) the lattice's tables are there
        assert gm.info().uniform == 0 and gm.info().device_bytes > gg.info().device_bytes
    return gm, gg, oracle_lib.OracleMesh(*n, *d, dtype=dtype, perturb=off)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["dyadic", "decimal", "graded", "skewed"])
@pytest.mark.parametrize("n", EXTENTS + VECTOR, ids=lambda n: "x".join(map(str, n)))
def test_operators_and_steps_star(hip_ctx, oracle_lib, n, kind, dtype):
    gm, gg, om = _mesh(hip_ctx, oracle_lib, n, kind, dtype)
    rng = np.random.default_rng(5)
    phi = rng.standard_normal(om.N).astype(dtype)
    af = (1e-3 * (1 + rng.random(om.N))).astype(dtype)
    for shift in (0, 1):
        t, out = _view(phi, dtype, shift), _view(phi, dtype, shift)
        for mask in (1, 2, 4, 7, 0):
            for wall in (-1, 0, 1, 2):
                assert np.array_equal(gm.grad(t, mask, wall, out=out).cpu().numpy(), om.grad(phi, mask, wall)), (mask, wall)
            assert np.array_equal(gm.lapl(t, mask, out=out).cpu().numpy(), om.lapl(phi, mask)), mask
            assert np.array_equal(gm.stab(t, mask, out=out).cpu().numpy(), om.stab(phi, mask)), mask
        for a in (None, af):
            A, B = _view(phi, dtype, shift), _view(phi, dtype, shift)
            got = gm.heat_run(A, B, 2e-3, 0.5, 5, alpha_field=None if a is None else _view(a, dtype, shift))
            assert np.array_equal(got.cpu().numpy(), om.heat_run(phi, 2e-3, 0.5, 5, alpha_field=a)), a is None
        f = [phi, *(rng.standard_normal(om.N).astype(dtype) for _ in range(3))]
        for k in (None, -af):
            A, B = [[_view(a, dtype, shift) for a in f] for _ in range(2)]
            got = gm.wave_run(A, B, -1.0, 0.02, 3, K_field=None if k is None else _view(k, dtype, shift))
            for g, r in zip(got, om.wave_run(*f, -1.0, 0.02, 3, K_field=k)):
                assert np.array_equal(g.cpu().numpy(), r), k is None


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["decimal", "graded"])
@pytest.mark.parametrize("n", EXTENTS + VECTOR, ids=lambda n: "x".join(map(str, n)))
def test_lattice_equals_general_form(hip_ctx, oracle_lib, n, kind, dtype):
    """Every operator and step on a lattice against the general form of the
    same mesh, with infinities, NaN and values near the ends of the range
    among the cells: the same bits, NaN in the same places."""
    gm, gg, om = _mesh(hip_ctx, oracle_lib, n, kind, dtype)
    if gm.info().uniform:
        pytest.skip("one or two layers per axis: exactly uniform, no lattice tables")
    rng = np.random.default_rng(6)
    tiny, big = np.finfo(dtype).smallest_subnormal, np.finfo(dtype).max
    fields = []
    for special in (None, (np.inf, np.nan, big, -big, tiny, -0.0)):
        f = [rng.standard_normal(om.N).astype(dtype) for _ in range(4)]
        if special:
            for a in f:
                a[rng.integers(om.N, size=max(1, om.N // 40))] = rng.choice(special)
        fields.append(f)
    K = (-(0.5 + rng.random(om.N))).astype(dtype)

    def same(a, b):
        return np.array_equal(a.cpu().numpy(), b.cpu().numpy(), equal_nan=True)

    for f in fields:
        t = _view(f[0], dtype, 0)
        for mask in (1, 6, 7):
            assert same(gm.grad(t, mask, -1), gg.grad(t, mask, -1)) and same(gm.grad(t, mask, 2), gg.grad(t, mask, 2))
            assert same(gm.lapl(t, mask), gg.lapl(t, mask))
            assert same(gm.stab(t, mask), gg.stab(t, mask))
        for m in (3, 4):
            x = [_view(f[0], dtype, 0) for _ in range(4)]
            assert same(gm.heat_run(x[0], x[1], 2e-3, 0.5, m), gg.heat_run(x[2], x[3], 2e-3, 0.5, m))
        for kf in (None, _view(K, dtype, 0)):
            A, C = [[_view(a, dtype, 0) for a in f] for _ in range(2)]
            B, D = [[torch.empty_like(a) for a in A] for _ in range(2)]
            for g, r in zip(gm.wave_run(A, B, -1.0, 0.02, 3, K_field=kf), gg.wave_run(C, D, -1.0, 0.02, 3, K_field=kf)):
                assert same(g, r)


def _uniform_ops(phi, h):
    """Gradient, Laplacian and stabilisation of (X, Y, Z) values on a uniform
    mesh of power-of-two spacings, in the scheme's operation order."""
    T = phi.dtype.type
    V = T(h[0] * h[1] * h[2])
    lo = lambda f, a: np.concatenate([f.take([0], a), f.take(range(f.shape[a] - 1), a)], a)
    hi = lambda f, a: np.concatenate([f.take(range(1, f.shape[a]), a), f.take([-1], a)], a)
    grad, lapl, stab = (np.zeros_like(phi) for _ in range(3))
    for a in range(3):
        A, al, L = T(h[0] * h[1] * h[2] / h[a]), T(1 / h[a]), T(h[a] / 2)
        g = (-((phi + lo(phi, a)) * T(0.5)) * A + (phi + hi(phi, a)) * T(0.5) * A) / V
        grad = grad + g
        lapl = lapl + ((-phi + lo(phi, a)) * al * A + (-phi + hi(phi, a)) * al * A) / V
        f_lo = T(0.5) * ((phi + L * g * T(-1)) - (lo(phi, a) + L * lo(g, a)))
        f_hi = T(0.5) * ((phi + L * g) - (hi(phi, a) + L * hi(g, a) * T(-1)))
        stab = stab + (f_lo * A + f_hi * A) / V
    return grad, lapl, stab


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [(3, 2, 3), (5, 4, 8), (16, 12, 32), (40, 121, 132)], ids=lambda n: "x".join(map(str, n)))
def test_uniform_nonfinite(hip_ctx, n, dtype):
    """Infinities, NaN and values near the ends of the range on a uniform mesh:
    the operators against their definition, the acoustic step against the
    march tiles, the heat step (one and two per launch) against the LDS boxes,
    the adjoint against the row form: the same bits, NaN in the same places."""
    from cfdarcov2_amd import adjoint, capi
    h = (0.125, 0.25, 0.5)
    gm = capi.HexMesh(hip_ctx, *n, *h, dtype=dtype)
    assert gm.info().uniform == 1
    N = gm.N
    rng = np.random.default_rng(7)
    special = np.array([np.inf, -np.inf, np.nan, np.finfo(dtype).max, -np.finfo(dtype).max,
                        np.finfo(dtype).smallest_subnormal, -0.0], dtype=dtype)

    def field():
        f = rng.standard_normal(N).astype(dtype)
        f[rng.integers(N, size=max(2, N // 60))] = rng.choice(special, size=max(2, N // 60))
        return f

    def same(a, b):
        a, b = (x.cpu().numpy() if torch.is_tensor(x) else x for x in (a, b))
        return np.array_equal(a, b, equal_nan=True)

    phi = field()
    with np.errstate(all="ignore"):
        ref = [r.reshape(-1) for r in _uniform_ops(phi.reshape(n), h)]
    t = _view(phi, dtype, 1)
    for name, r in zip(("grad", "lapl", "stab"), ref):
        assert same(getattr(gm, name)(t), r), name

    def heat(shape, steps, af=None):
        gm.set_heat_shape(*shape)
        return gm.heat_run(_view(phi, dtype, 0), _view(phi, dtype, 0), 2e-3, 0.5, steps, alpha_field=af)

    for steps in (1, 4, 6):
        assert same(heat((0, 8, 16), steps), heat((2, 4, 2), steps)), steps
    af = _view(np.abs(field()), dtype, 0)
    x = [_view(phi, dtype, 0), _view(phi, dtype, 0)]
    for k in range(4):  # single steps against two per launch, with an alpha field
        x.reverse() if k else None
        gm.heat_run(*x, 2e-3, 0.5, 1, alpha_field=af)
    assert same(heat((0, 8, 16), 4, af), x[1])

    f = [field() for _ in range(4)]
    for kf in (None, _view(-np.abs(field()), dtype, 0)):
        out = []
        for shape in ((0, 4, 8, 0), (1, 4, 8, 0)):
            gm.set_wave_shape(*shape)
            out.append(gm.wave_run([_view(a, dtype, 0) for a in f], [_view(a, dtype, 0) for a in f], -1.0, 0.02, 3,
                                   K_field=kf))
        assert all(same(a, b) for a, b in zip(*out)), kf is None
    if n[2] % 4 == 0:
        pr = adjoint.WaveProblem(gm, np.array([0, N // 2, N - 1]), 0.02, 5, K=-1.0, every=2)
        out, g = [], torch.from_numpy(rng.standard_normal((5, 3)).astype(dtype)).cuda()
        g[2, 1] = float("inf")
        for form in (0, 1):
            gm.set_adjoint_shape(form, 4, 8)
            tr, _, ck = adjoint.forward_traces(pr, _view(f[0], dtype, 0))
            out.append([tr, *adjoint.adjoint(pr, g, None, ck, want_K=True)])
        assert all(same(a, b) for a, b in zip(*out))
    gm.close()


def test_perturbed_mesh_is_no_lattice(hip_ctx):
    """One vertex moved by one unit in the last place of its coordinate (0.9),
    which reaches the face normals: the general form."""
    from cfdarcov2_amd import capi
    n, d = (5, 4, 6), (0.1, 0.3, 0.7)
    off = np.zeros(((n[0] + 1) * (n[1] + 1) * (n[2] + 1), 3))
    off[2 * 5 * 7 + 3 * 7 + 3, 1] = np.spacing(3 * d[1])
    gm = capi.HexMesh(hip_ctx, *n, *d, dtype="f64", vertex_offsets=off)
    gg = capi.HexMesh(hip_ctx, *n, *d, dtype="f64", vertex_offsets=off, force_general=True)
    assert gm.info().device_bytes == gg.info().device_bytes


# launch geometries: runs that divide y, three columns where a row is just over
# half a workgroup (in cells and in vectors), and the rows' ends of both
PLANS = [(22, 20, 300), (22, 20, 150), (9, 40, 130), (6, 24, 67), (2, 512, 140), (3, 13, 1030)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["dyadic", "decimal", "skewed"])
@pytest.mark.parametrize("n", PLANS, ids=lambda n: "x".join(map(str, n)))
def test_launch_geometries(hip_ctx, oracle_lib, n, kind, dtype):
    _check_against_oracle(*_mesh(hip_ctx, oracle_lib, n, kind, dtype), dtype)


@pytest.mark.parametrize("dtype,n", [(np.float64, (258, 257, 254)), (np.float32, (323, 322, 323))], ids=["f64", "f32"])
def test_some_axes_beyond_the_cache(hip_ctx, n, dtype):
    """Gradient and Laplacian over some axes on fields beyond the last-level
    cache, which load those axes' neighbours only, against their definition."""
    from cfdarcov2_amd import capi
    h = (0.125, 0.25, 0.5)
    assert 2 * np.prod(n) * np.dtype(dtype).itemsize > 256 << 20
    gm = capi.HexMesh(hip_ctx, *n, *h, dtype=dtype)
    phi = torch.from_numpy(np.random.default_rng(3).standard_normal(n).astype(dtype)).cuda()
    out = torch.empty(gm.N, dtype=phi.dtype, device="cuda")
    V = h[0] * h[1] * h[2]
    for mask in (0, 1, 2, 4, 3, 5, 6):
        grad, lapl = torch.zeros_like(phi), torch.zeros_like(phi)
        for a in range(3):
            if not mask & (1 << a):
                continue
            k, A = n[a], V / h[a]
            lo = torch.cat([phi.narrow(a, 0, 1), phi.narrow(a, 0, k - 1)], a)
            hi = torch.cat([phi.narrow(a, 1, k - 1), phi.narrow(a, k - 1, 1)], a)
            grad += (-((phi + lo) * 0.5) * A + (phi + hi) * 0.5 * A) / V
            lapl += ((-phi + lo) / h[a] * A + (-phi + hi) / h[a] * A) / V
            del lo, hi
        assert torch.equal(gm.grad(phi.reshape(-1), mask, -1, out=out), grad.reshape(-1)), mask
        assert torch.equal(gm.lapl(phi.reshape(-1), mask, out=out), lapl.reshape(-1)), mask
    gm.close()


@pytest.mark.parametrize("dtype,n", [(np.float64, (20, 21, 2400)), (np.float32, (24, 23, 3602))], ids=["f64", "f32"])
def test_launch_geometry_of_long_perturbed_meshes(hip_ctx, oracle_lib, n, dtype):
    """Runs of columns: face arrays beyond half the last-level cache, z at
    least eight times as long as x and y."""
    assert 34 * np.prod(n) * np.dtype(dtype).itemsize > 256 << 20
    _check_against_oracle(*_mesh(hip_ctx, oracle_lib, n, "skewed", dtype), dtype)


# either side of the sizes up to which an operator takes one cell per thread
# (2^15 and 2^16 cells in FP64; 2^18, 2^19, 2^21 and 2^22 in FP32)
@pytest.mark.parametrize("kind", ["decimal", "skewed"])
@pytest.mark.parametrize("dtype,n", [(np.float64, (32, 31, 33)), (np.float64, (32, 33, 33)), (np.float64, (41, 40, 41)),
                                     (np.float32, (63, 64, 65)), (np.float32, (64, 65, 65)), (np.float32, (81, 80, 82)),
                                     (np.float32, (130, 128, 127)), (np.float32, (163, 161, 161))],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else np.dtype(v).name)
def test_widths_of_face_geometry_kernels(hip_ctx, oracle_lib, n, kind, dtype):
    _check_against_oracle(*_mesh(hip_ctx, oracle_lib, n, kind, dtype), dtype)


def _check_against_oracle(gm, gg, om, dtype):
    """Every operator and step of the mesh against the oracle's."""
    gg.close()
    rng = np.random.default_rng(12)
    f = [rng.standard_normal(om.N).astype(dtype) for _ in range(4)]
    phi, (t, out) = f[0], (_view(f[0], dtype, 1), _view(f[0], dtype, 1))
    for mask in (7, 1, 2, 4, 5):
        assert np.array_equal(gm.grad(t, mask, mask % 3, out=out).cpu().numpy(), om.grad(phi, mask, mask % 3)), mask
        assert np.array_equal(gm.lapl(t, mask, out=out).cpu().numpy(), om.lapl(phi, mask)), mask
    assert np.array_equal(gm.stab(t, 7, out=out).cpu().numpy(), om.stab(phi, 7))
    A, B = [[_view(a, dtype, 0) for a in f] for _ in range(2)]
    for steps in (1, 4):
        A[0].copy_(_view(phi, dtype, 0))
        assert np.array_equal(gm.heat_run(A[0], B[0], 2e-3, 0.5, steps).cpu().numpy(), om.heat_run(phi, 2e-3, 0.5, steps))
    A[0].copy_(_view(phi, dtype, 0))
    if gm.info().uniform:
        gm.set_wave_shape(0, 4, 8, 0)
    for g, r in zip(gm.wave_run(A, B, -1.0, 0.02, 2), om.wave_run(*f, -1.0, 0.02, 2)):
        assert np.array_equal(g.cpu().numpy(), r)
    gm.close()


def test_lattice_without_room_for_its_tables(hip_ctx):
    """A pool limit that holds the face arrays and no more: the mesh is made
    without the tables, as before they existed, and gives the same results."""
    from cfdarcov2_amd import capi
    n, d = (7, 6, 9), (0.1, 0.3, 0.7)
    ctx = capi.Context(0)
    gm = capi.HexMesh(ctx, *n, *d, dtype="f64")
    gg = capi.HexMesh(ctx, *n, *d, dtype="f64", force_general=True)
    faces, both = gg.info().device_bytes, gm.info().device_bytes
    assert both > faces
    gg.close()
    ctx.pool_set_limit(both + faces)
    gl = capi.HexMesh(ctx, *n, *d, dtype="f64")
    assert gl.info().device_bytes == faces
    phi = torch.from_numpy(np.random.default_rng(1).standard_normal(gm.N)).cuda()
    for op in ("grad", "lapl"):
        assert torch.equal(getattr(gm, op)(phi), getattr(gl, op)(phi))
    ctx.pool_set_limit(both + 2 * faces - 1)
    with pytest.raises(capi.CfdError):
        capi.HexMesh(ctx, *n, *d, dtype="f64")
    torch.cuda.synchronize()
    gl.close()
    gm.close()
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("every", [1, 2, 3, 9])
@pytest.mark.parametrize("n", EXTENTS[1:] + [(600, 2, 5), VECTOR[1]], ids=lambda n: "x".join(map(str, n)))
def test_adjoint_star(hip_ctx, n, every, dtype):
    """Traces and gradients (K field and constant K, checkpoint segments of
    one to all steps, sensors in the first and last cells) against autograd
    through the plain FP64 stepper.  Bound: 7 steps forward and back of some
    30 roundings each, eps * 420 = 2.5e-5 in FP32 and 5e-14 in FP64."""
    from cfdarcov2_amd import adjoint, capi
    from tests import torch_wave
    d, steps, dt = (0.125, 0.125, 0.125), 7, 0.04
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(N)
    sens = np.unique(np.concatenate([[0, N - 1, N // 2], rng.integers(N, size=min(N, 20))]))
    p0 = rng.standard_normal(N).astype(dtype)
    Kf = (-(0.5 + rng.random(N))).astype(dtype)
    g = rng.standard_normal((steps, sens.size)).astype(dtype)
    gm = capi.HexMesh(hip_ctx, *n, *d, dtype=dtype)
    gm.set_adjoint_shape(0, 4, 8)
    for field in (True, False):
        pr = adjoint.WaveProblem(gm, sens, dt, steps, K=-0.75, every=every)
        tp = torch.from_numpy(p0).cuda().requires_grad_(True)
        tk = torch.from_numpy(Kf).cuda().requires_grad_(True) if field else None
        tr = adjoint.wave_traces(tp, tk, pr)
        got = [tr.detach(), *torch.autograd.grad(tr, [tp, tk] if field else [tp], torch.from_numpy(g).cuda())]
        if not field:  # the K gradient at a constant K
            _, _, ck = adjoint.forward_traces(pr, tp, checkpoints=True)
            got.append(adjoint.adjoint(pr, torch.from_numpy(g).cuda(), None, ck, want_K=True)[1])
        rp = torch.from_numpy(p0).double().requires_grad_(True)
        rk = (torch.from_numpy(Kf).double() if field else torch.full((N,), -0.75, dtype=torch.float64)).requires_grad_(True)
        rt = torch_wave.traces(rp, rk, dt, steps, torch.from_numpy(sens), n, d)
        ref = [rt.detach(), *torch.autograd.grad(rt, [rp, rk], torch.from_numpy(g).double())]
        for a, b in zip(got, ref):
            err = (a.cpu().double() - b).norm() / max(float(b.norm()), 1e-30)
            assert err < (2.5e-5 if dtype == np.float32 else 5e-14), (field, float(err))
    gm.close()


def test_batch_star_mixed_extents(hip_ctx):
    """One batch of cases of any extents (rows shorter than a vector, not a
    multiple of it, volumes that are no power of two): each equals its
    single-case run."""
    import ctypes

    from cfdarcov2_amd import capi
    rng = np.random.default_rng(2)
    meshes, states, keep = [], [], []
    for k, n in enumerate(EXTENTS + [(20, 12, 33), (16, 16, 16)]):
        d = (0.125, 0.375, 0.25) if k % 3 == 0 else (0.125,) * 3
        m = capi.HexMesh(hip_ctx, *n, *d, dtype="f32")
        assert m.info().uniform == 1
        heat = k % 2 == 0
        a = [torch.from_numpy(rng.standard_normal(m.N).astype(np.float32)).cuda() for _ in range(1 if heat else 4)]
        meshes.append(m)
        states.append((heat, a, [torch.empty_like(t) for t in a], [t.clone() for t in a]))
    arr = (capi.BatchCase * len(meshes))()
    for c, m, (heat, a, b, _) in zip(arr, meshes, states):
        c.mesh, c.kind, c.coef, c.dt = m.h, 0 if heat else 1, 1e-3 if heat else -0.8, 0.02
        for f, (x, y) in enumerate(zip(a, b)):
            c.state_a[f], c.state_b[f] = x.data_ptr(), y.data_ptr()
    h = ctypes.c_void_p()
    capi.check(hip_ctx.lib.cfd_batch_create(hip_ctx.h, arr, len(meshes), ctypes.byref(h)))
    for graph in (0, 1):
        for _, a, _, a0 in states:
            for x, y in zip(a, a0):
                x.copy_(y)
        for _ in range(2):
            capi.check(hip_ctx.lib.cfd_batch_run(h, 4, graph, capi._stream_ptr()))
        torch.cuda.synchronize()
        for k, (m, (heat, a, _, a0)) in enumerate(zip(meshes, states)):
            A, B = [t.clone() for t in a0], [torch.empty_like(t) for t in a0]
            ref = [m.heat_run(A[0], B[0], 1e-3, 0.02, 8)] if heat else m.wave_run(A, B, -0.8, 0.02, 8)
            for g, r in zip(a, ref):
                assert torch.equal(g, r), (k, graph)
    capi.check(hip_ctx.lib.cfd_batch_destroy(h))


def test_batch_with_a_case_beyond_the_cache(hip_ctx):
    """Form 0 of a batch whose acoustic case exceeds the last-level cache (march
    tiles, at each of their shapes) between cases that do not (star form), in
    every order of the descriptors: each equals its single-case run."""
    import ctypes
    import itertools

    from cfdarcov2_amd import capi
    rng = np.random.default_rng(4)
    cases = []
    for n, heat in (((191, 187, 250), False), ((9, 7, 33), False), ((16, 12, 20), True)):
        m = capi.HexMesh(hip_ctx, *n, 0.125, 0.125, 0.125, dtype="f32")
        a0 = [torch.from_numpy(rng.standard_normal(m.N, dtype=np.float32)).cuda() for _ in range(1 if heat else 4)]
        a, b = [t.clone() for t in a0], [torch.empty_like(t) for t in a0]
        ref = [m.heat_run(a[0], b[0], 1e-3, 0.02, 4)] if heat else m.wave_run(a, b, -0.8, 0.02, 4)
        cases.append((m, heat, a0, a, b, [t.clone() for t in ref]))
    assert 8 * 4 * cases[0][0].N > 256 << 20
    shapes = itertools.cycle([(4, 8), (8, 5), (16, 32)])
    for order in itertools.permutations(range(3)):
        arr = (capi.BatchCase * 3)()
        for c, i in zip(arr, order):
            m, heat, a0, a, b, _ = cases[i]
            c.mesh, c.kind, c.coef, c.dt = m.h, 0 if heat else 1, 1e-3 if heat else -0.8, 0.02
            for f in range(len(a0)):
                a[f].copy_(a0[f])
                c.state_a[f], c.state_b[f] = a[f].data_ptr(), b[f].data_ptr()
        h = ctypes.c_void_p()
        capi.check(hip_ctx.lib.cfd_batch_create(hip_ctx.h, arr, 3, ctypes.byref(h)))
        shape = next(shapes)
        capi.check(hip_ctx.lib.cfd_batch_set_shape(h, *shape))
        capi.check(hip_ctx.lib.cfd_batch_run(h, 4, order[0] % 2, capi._stream_ptr()))
        for i in order:
            for g, r in zip(cases[i][3], cases[i][5]):
                assert torch.equal(g, r), (order, shape, i)
        capi.check(hip_ctx.lib.cfd_batch_destroy(h))
