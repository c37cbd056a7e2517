"""Point location where the cooperative search of k_locate can go wrong: point counts around
the 8 lanes of a query and the 8 queries of a wave, points at the edges of the midpoint
grid (on the axis, near the centre, at and beyond the surface), points with two midpoints at
the same single-precision distance, and databases of fewer elements than the 13 nearest,
against the oracle.  Element ids and ties are exact; xi and eta come from the same FP64
operations."""
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


def _in_frame(p, frame, q, rng):
    """points of the frame's (s, z) at random azimuths"""
    lat, lon = (p.src_lat, p.src_lon) if frame == 0 else (p.rec_lat[frame - 1], p.rec_lon[frame - 1])
    pole = synth.geo_xyz(lat, lon, 1.0)
    u = rng.normal(size=(len(q), 3))
    u -= (u @ pole)[:, None] * pole
    u /= np.linalg.norm(u, axis=1)[:, None]
    return np.ascontiguousarray(q[:, 1:] * pole + q[:, :1] * u)


def _tie_points(p, frame, rank, n=40):
    """points whose rank-th and next nearest midpoints (counted from 1) are at the same
    single-precision distance, and no others of the 15 nearest"""
    rng = np.random.default_rng(23)
    mp = np.stack([p.mesh.mp_s, p.mesh.mp_z], 1).astype(np.float64)
    r, th = np.sqrt(rng.uniform(2e6 ** 2, 6.2e6 ** 2, 8 * n)), rng.uniform(0.1, np.pi - 0.1, 8 * n)
    q = np.stack([r * np.sin(th), r * np.cos(th)], 1)
    for _ in range(3):                       # onto the bisector of the two midpoints
        i = np.argsort(((q[:, None] - mp[None]) ** 2).sum(2), axis=1)
        a, b = mp[i[:, rank - 1]], mp[i[:, rank]]
        q = q - (((q - (a + b) / 2) * (b - a)).sum(1) / ((b - a) ** 2).sum(1))[:, None] * (b - a)
    d = mp[None].astype(np.float32) - q[:, None].astype(np.float32)
    d = np.sort(d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1], axis=1)
    eq = d[:, 1:15] == d[:, :14]
    return _in_frame(p, frame, q[eq[:, rank - 1] & (eq.sum(1) == 1)][:n], rng)


@pytest.mark.parametrize("frame", [0, 2])
@pytest.mark.parametrize("rank", [1, 2, 4, 8, 9, 11, 12, 13])
def test_locate_ties(tiny, tiny_oracle, gpu, frame, rank):
    """Ties anywhere among the 12 nearest and between the 12th and the 13th are reported (of
    equal distances the lower element comes first), one beyond them is not."""
    print("locate ties", frame, rank, flush=True)
    x = _tie_points(tiny, frame, rank)
    oe, oxi, oeta, otie = tiny_oracle.locate(frame, x)
    assert len(x) >= 10 and np.all(otie == (1 if rank <= 12 else 0))
    ge, gxi, geta, gtie = gpu.locate(frame, x)
    assert np.array_equal(gtie, otie)
    assert np.array_equal(ge, oe)
    assert np.max(np.abs(gxi - oxi)) < 1e-9
    assert np.max(np.abs(geta - oeta)) < 1e-9


@pytest.mark.parametrize("nelem", [1, 5, 12, 13, 14])
def test_locate_few_elements(nelem):
    """Databases of 1 to 14 elements: the search ends with the grid."""
    import mc_kernel_amd as mk
    from oracle import oracle
    p = synth.make_problem("tiny", ntet=1)
    for db in (p.setup.fwd, p.setup.bwd):
        db.nelem = nelem
    rng = np.random.default_rng(4)
    e = np.arange(nelem).repeat(3)
    q = np.stack([p.mesh.mp_s[e], p.mesh.mp_z[e]], 1) * (1 + 0.02 * rng.uniform(-1, 1, (len(e), 2)))
    x = _in_frame(p, 1, q, rng)
    oe, oxi, oeta, otie = oracle.Oracle(p.setup).locate(1, x)
    assert np.array_equal(oe, e + 1)
    print("locate few", nelem, flush=True)
    k = mk.MCKernel(p.setup)
    try:
        ge, gxi, geta, gtie = k.locate(1, x)
    finally:
        k.close()
    assert np.array_equal(gtie, otie)
    assert np.array_equal(ge, oe)
    assert np.max(np.abs(gxi - oxi)) < 1e-9
    assert np.max(np.abs(geta - oeta)) < 1e-9
