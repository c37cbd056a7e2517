"""Point location where the cooperative search of k_locate can go wrong: point counts around
the 8 lanes of a query and the 8 queries of a wave, and points at the edges of the midpoint
grid (on the axis, near the centre, at and beyond the surface, at element corners), against
the oracle.  Element ids and ties are exact; xi and eta come from the same FP64 operations."""
import numpy as np
import pytest

from mc_kernel_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(tiny):
    import mc_kernel_amd as mk
    k = mk.MCKernel(tiny.setup)
    yield k
    k.close()


def _edge_points(p, kind, n):
    rng = np.random.default_rng(17)
    v = rng.normal(size=(n, 3))
    v /= np.linalg.norm(v, axis=1)[:, None]
    src = synth.geo_xyz(p.src_lat, p.src_lon, 1.0)
    if kind == "axis":        # within 100 m of the source frame's axis, both sides
        return src[None] * rng.uniform(-1, 1, n)[:, None] * 6.3e6 + v * 100.0
    if kind == "centre":
        return v * (1e3 * 10.0 ** rng.uniform(0, 3, n))[:, None]
    if kind == "surface":     # the clamp to the surface included
        return v * (synth.R_EARTH + rng.uniform(-2e3, 20e3, n))[:, None]
    r = np.cbrt(rng.uniform(1e6 ** 3, 6.3e6 ** 3, n))
    return v * r[:, None]


@pytest.mark.parametrize("frame", [0, 2])
@pytest.mark.parametrize("kind,n", [("mantle", 1), ("mantle", 7), ("mantle", 8), ("mantle", 9), ("mantle", 65),
                                    ("axis", 200), ("centre", 200), ("surface", 200)])
def test_locate_edges(tiny, tiny_oracle, gpu, frame, kind, n):
    print("locate", frame, kind, n, flush=True)
    x = np.ascontiguousarray(_edge_points(tiny, kind, n))
    oe, oxi, oeta, otie = tiny_oracle.locate(frame, x)
    ge, gxi, geta, gtie = gpu.locate(frame, x)
    assert np.array_equal(gtie, otie)
    ok = otie == 0
    assert np.array_equal(ge[ok], oe[ok])
    assert np.max(np.abs(gxi[ok] - oxi[ok]), initial=0) < 1e-9
    assert np.max(np.abs(geta[ok] - oeta[ok]), initial=0) < 1e-9
