"""Window sums of the matrix-core backward path (MCK_BWD_PATH=1): its slots are taken in
groups of 4 class positions, an even number of groups up to 8 in registers and more in
LDS, each class (lambda, mu, their combination) padded to whole groups.  Receivers with
few, many and different numbers of slots against the FP64 oracle: a full pinned
slave_work, each kernel within 1e-5 relative to its L2 norm, the bar of the parity
tests; launch: a workgroup per group of pairs (1) or per element (4)."""
import numpy as np
import pytest

from mc_kernel_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5
K = synth._kernels
CASES = {
    "one": (1, K(1, 1, ["CC"], ["vp"])),
    "mu only": (3, K(2, 3, ["CC"], ["mu"])),
    "5 lambda": (5, K(2, 5, ["CC"], ["vp"])),
    "6 + 6": (3, K(2, 3, ["CC", "AM"], ["vp", "vs"])),
    "10 + 10": (5, K(2, 5, ["CC", "AM"], ["vp", "vs"])),
    "14 + 14, 1": (7, K(1, 7, ["CC", "AM"], ["vp", "vs"])
                   + [{"rec": 1, "filter": 0, "misfit": "CC", "param": "vp"}]),
    "20 + 20 + 20": (10, K(2, 10, ["CC", "AM"], ["vp", "vs", "mu"])),
}


@pytest.mark.parametrize("launch", ["1", "4"])
@pytest.mark.parametrize("name", CASES)
def test_slot_groups(monkeypatch, name, launch):
    import mc_kernel_amd as mk
    from oracle import oracle
    nfilter, kernels = CASES[name]
    monkeypatch.setenv("MCK_BWD_PATH", "1")
    monkeypatch.setenv("MCK_MFMA_WAVES", launch)
    nrec = 1 + max(d["rec"] for d in kernels)
    p = synth.make_problem("tiny", ntet=4, receivers_deg=[30.0, 60.0][:nrec], kernels=kernels,
                           filters=[("Gabor", (40.0 + 3.0 * i, 0.5, 0.0, 0.0)) for i in range(nfilter)])
    print("slot groups:", name, launch, flush=True)
    ref = oracle.Oracle(p.setup).slave_work(p.verts, p.conn)
    k = mk.MCKernel(p.setup)
    try:
        res = k.slave_work(p.verts, p.conn, halton_offsets=ref["offsets"])
        assert k.stats()["bwd_path"] == 1
    finally:
        k.close()
    assert np.array_equal(res["niterations"], ref["niterations"])
    for j in range(p.nkernel):
        r = ref["values"][:, j]
        n = np.linalg.norm(r)
        assert np.linalg.norm(res["values"][:, j] - r) <= TOL * n, j


# carried components (forward, backward) and backward variables of each set: source, receiver
# component, parameters of its kernels (vp alone: the trace of the strain)
DC = [0.3e20, 1.0e20, -1.3e20, 0.5e20, -0.4e20, 0.7e20]   # general moment tensor
FORMS = {
    "1, 1, 2": (None, "Z", ["vp"]),
    "1, 1, 3": (DC, "R", ["vp"]),
    "4, 4, 2": (None, "Z", ["vp", "vs"]),
    "6, 4, 2": (DC, "Z", ["vp", "vs"]),
    "4, 6, 3": (None, "R", ["vp", "vs"]),
    "6, 6, 3": (DC, "T", ["vp", "vs"]),
}


@pytest.mark.parametrize("launch", ["1", "4"])
@pytest.mark.parametrize("nfilter", [2, 3, 5, 7, 9])
@pytest.mark.parametrize("form", FORMS)
def test_component_forms(monkeypatch, form, nfilter, launch):
    """Every strain component form of the matrix-core evaluation at 2, 4, 6, 8 and more than
    8 groups of slots: base kernels of 24 points, each within 1e-5 relative to its L2 norm."""
    import mc_kernel_amd as mk
    from oracle import oracle
    mij, component, params = FORMS[form]
    monkeypatch.setenv("MCK_BWD_PATH", "1")
    monkeypatch.setenv("MCK_MFMA_WAVES", launch)
    # slots: 2 per filter and parameter (CC, AM); the trace-only sets have lambda alone
    nf = nfilter if len(params) == 2 else 2 * nfilter
    p = synth.make_problem("tiny", ntet=4, mij=mij, component=component, kernels=K(2, nf, ["CC", "AM"], params),
                           filters=[("Gabor", (40.0 + 3.0 * i, 0.5, 0.0, 0.0)) for i in range(nf)])
    print("component form:", form, nfilter, launch, flush=True)
    o = oracle.Oracle(p.setup)
    x = p.sample_points(24, seed=31)
    ref_b = o.base_kernels(x)
    k = mk.MCKernel(p.setup)
    try:
        g = k.base_kernels(x)
        st = k.stats()
        assert st["bwd_path"] == 1 and "%d, %d" % (st["nd_f"], st["nd_b"]) == form[:4]
    finally:
        k.close()
    assert np.abs(ref_b).max() > 0
    for j in range(p.nkernel):
        for b in range(6):
            r = ref_b[:, j, b]
            assert np.linalg.norm(g[:, j, b] - r) <= TOL * np.linalg.norm(r), (j, b)
