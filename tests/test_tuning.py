"""The tuners choose among the forms that an untuned mesh takes, so tuning a
mesh does not leave it slower than not tuning it."""
import numpy as np
import pytest

from cfdarcov2_amd import autotune, workloads

gpu = pytest.mark.gpu


def test_best_keeps_the_automatic_form_within_noise():
    rows = lambda *ms: [{"variant": v, "ms_per_step": t} for v, t in zip((-1, 0, 1), ms)]
    assert autotune._best(rows(1.02, 3.0, 1.0), "variant")["variant"] == -1
    assert autotune._best(rows(1.05, 3.0, 1.0), "variant")["variant"] == 1
    assert autotune._best(rows(1.05, 3.0, 1.0)[1:], "variant")["variant"] == 1


def test_batch_candidates_hold_no_launch_twice():
    """Form 0 is timed once per group size, unless a case takes its tiles."""
    from types import SimpleNamespace as S

    from cfdarcov2_amd.ensemble import tune_candidates
    small = [S(kind="wave", n=128), S(kind="heat", n=300)]
    form0 = [c for c in tune_candidates(small) if c[3] == 0]
    assert len(form0) == len({c[2] for c in form0}) == 3
    assert len([c for c in tune_candidates(small + [S(kind="wave", n=256)]) if c[3] == 0]) == 27


def _euler_state(torch, N, dtype):
    rng = np.random.default_rng(2)
    U = np.stack([1.0 + 0.3 * rng.random(N), *(0.1 * rng.standard_normal((3, N))), 3.0 + rng.random(N)])
    return [torch.from_numpy(u.astype(dtype)).cuda() for u in U]


@gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_euler_tuner_times_the_automatic_tile(hip_ctx, dtype):
    """The tile by the mesh's size (of one plane at these extents) is among the
    candidates, a tuned mesh is as fast by the tuner's own table, and -1
    returns a mesh to it with the same results."""
    torch = pytest.importorskip("torch")
    from cfdarcov2_amd import capi
    n, d = (80, 33, 27), (0.1, 0.07, 0.09)
    gm = capi.HexMesh(hip_ctx, *n, *d, dtype=dtype, vertex_offsets=workloads.perturbed_vertex_offsets(*n, *d, 4, 0.2))
    U = _euler_state(torch, gm.N, dtype)

    def run():
        A, B = [u.clone() for u in U], [torch.empty_like(u) for u in U]
        return [t.clone() for t in gm.euler_run(A, B, 1.4, 0.3, 3)]

    ref = run()
    best = autotune.tune_euler(gm, U, steps=4)
    auto = [r for r in best["table"] if r["variant"] == -1]
    assert len(auto) == 1 and best["ms_per_step"] <= auto[0]["ms_per_step"]
    assert {r["chunk"] for r in best["table"] if r["variant"] == 1} >= {1, 2, 4}
    for shape in ((best["variant"], best["tile_rows"], best["chunk"]), (0, 4, 16), (-1, 4, 16)):
        gm.set_euler_shape(*shape)
        assert all(torch.equal(a, b) for a, b in zip(run(), ref)), shape
    with pytest.raises(capi.CfdError):
        gm.set_euler_shape(-2, 4, 16)
    gm.close()


@gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_adjoint_tuner_times_the_form_by_size(hip_ctx, dtype):
    """The form by size is among the candidates, and -1 returns a mesh to it:
    the K gradient's path, which the tuner does not time, stays free to differ."""
    torch = pytest.importorskip("torch")
    from cfdarcov2_amd import adjoint, capi
    n = (16, 12, 32)
    gm = capi.HexMesh(hip_ctx, *n, 1 / 32, 1 / 32, 1 / 32, dtype=dtype)
    pr = adjoint.WaveProblem(gm, np.array([0, 7, gm.N - 1]), 0.01, 6, K=-0.8)
    p0 = torch.from_numpy(np.random.default_rng(0).standard_normal(gm.N).astype(dtype)).cuda()

    def run():
        tr, _, ck = adjoint.forward_traces(pr, p0)
        return [tr, *adjoint.adjoint(pr, tr, None, ck, want_K=True)]

    ref = run()
    best = autotune.tune_adjoint(pr, steps=4)
    auto = [r for r in best["table"] if r["form"] == -1]
    assert len(auto) == 1 and best["ms_per_step"] <= auto[0]["ms_per_step"]
    for shape in ((best["form"], best["tile_rows"], best["chunk"]), (1, 4, 2), (-1, 4, 8)):
        gm.set_adjoint_shape(*shape)
        assert all(torch.equal(a, b) for a, b in zip(run(), ref)), shape
    with pytest.raises(capi.CfdError):
        gm.set_adjoint_shape(-2, 4, 8)
    gm.close()
