"""Element spectra (k_elem_spectra) at trace lengths where its register FFT can go wrong: one
sample beyond a transform size, odd lengths (sample pairs unaligned), one or several
traces per wave, on few elements (each element's traces spread over workgroups).  The
matrix-core backward path (MCK_BWD_PATH=1) against the FP64 oracle: base kernels within
1e-5 relative to each kernel's L2 norm, the bar of the parity tests."""
import numpy as np
import pytest

from mc_kernel_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5
# nt -> complex FFT length: 257, 511 -> 512, 777 -> 1024, 1025, 1999 -> 2048, 2050 -> 4096
LENGTHS = [257, 511, 777, 1025, 1999, 2050]


@pytest.mark.parametrize("nt", LENGTHS)
def test_matrix_core_path_trace_lengths(monkeypatch, nt):
    import mc_kernel_amd as mk
    from oracle import oracle
    monkeypatch.setenv("MCK_BWD_PATH", "1")
    p = synth.make_problem("tiny", nelem_target=120, nt=nt, dt=1024.0 / nt, ntet=4)
    print("element spectra: nt", nt, flush=True)
    x = p.sample_points(9, seed=5)
    ref = oracle.Oracle(p.setup).base_kernels(x)
    k = mk.MCKernel(p.setup)
    try:
        g = k.base_kernels(x)
        assert k.stats()["bwd_path"] == 1
    finally:
        k.close()
    for j in range(p.nkernel):
        for b in range(6):
            r = ref[:, j, b]
            if not np.any(r):
                assert not np.any(g[:, j, b]), (j, b)
                continue
            assert np.linalg.norm(g[:, j, b] - r) / np.linalg.norm(r) < TOL, (j, b)
