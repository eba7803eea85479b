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


def _view(a, dtype, shift):
    """Device copy of `a` starting `shift` elements into a buffer."""
    buf = torch.zeros(a.size + shift, dtype=torch.float32 if dtype == np.float32 else torch.float64, device="cuda")
    buf[shift:].copy_(torch.from_numpy(np.ascontiguousarray(a, dtype=dtype)))
    return buf[shift:]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", EXTENTS, ids=lambda n: "x".join(map(str, n)))
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
