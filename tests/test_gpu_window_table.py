"""A window-spectrum table of more than 4 GiB (520 receivers x 256 windows at nt 4096,
133,120 rows of 4112 bins): the matrix-core evaluation of the last receivers' kernels
against the per-pair kernel on the same handle, each kernel within 1e-5 relative to its L2
norm, the bar of the parity tests (which hold the per-pair kernel to the oracle)."""
import numpy as np
import pytest

from mc_kernel_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5


def test_window_table_beyond_4_gib():
    import mc_kernel_amd as mk
    nrec, nwin, nt, dt = 520, 256, 4096, 0.25
    kernels = [{"rec": r, "filter": 0, "misfit": "CC", "param": "vp"} for r in range(nrec) for _ in range(nwin)]
    p = synth.make_problem("tiny", nelem_target=120, nt=nt, dt=dt, ntet=4, kernels=kernels,
                           receivers_deg=np.linspace(30.0, 80.0, nrec).tolist(),
                           filters=[("Gabor", (40.0, 0.5, 0.0, 0.0))])
    # every kernel its own window: shifted by one sample each
    p.kernel_window += (np.tile(np.arange(nwin), nrec) * dt)[:, None]
    assert nrec * nwin * 4112 * 8 > 2 ** 32
    print("window table", flush=True)
    x = p.sample_points(2, seed=5)
    out = {}
    k = mk.MCKernel(p.setup)
    try:
        for path in (0, 1):
            k.set_tuning({"bwd_path": path, "mfma_waves": 1, "mfma_xcd": 0})
            out[path] = k.base_kernels(x)
            assert k.stats()["bwd_path"] == path
    finally:
        k.close()
    for r in (0, 400, 511, 519):
        s = slice(r * nwin, (r + 1) * nwin)
        ref, got = out[0][:, s, 0], out[1][:, s, 0]
        n = np.linalg.norm(ref, axis=0)
        assert n.min() > 0 and len(np.unique(n)) > nwin // 2
        err = float((np.linalg.norm(got - ref, axis=0) / n).max())
        assert err <= TOL, (r, err)
