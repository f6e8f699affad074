"""Grouped analysis alpha launches with scales on the work length 1024 (band
limits 129..256), on both sides of the line between the radix-8 body and the
three-stage engine (256 workgroups: ceil(hi / 4) N over those scales), against
the generic kernels (S2DW_HIP_FFT=generic at plan creation), and their moments
form.

Tolerance 1e-12 max abs on red N(0,1)/(l+1) spectra, the suite's bound for
device plans on red input; moments 1e-9 (sums of the same values in another
order)."""
import numpy as np
import pytest

from conftest import seeded_flm
from s2dw_amd import core

pytestmark = pytest.mark.gpu

TOL = 1e-12

# 66, 128, 256 (the line), 198, 252, 258 workgroups; then scale 2 of a two-stream plan: 64, 128, 256
CASES = [(129, 1), (256, 1), (256, 2), (129, 3), (168, 3), (171, 3), (512, 1), (512, 2), (512, 4)]


@pytest.mark.parametrize("B,N", CASES)
def test_group_alpha(B, N, monkeypatch):
    import torch

    print(f"group B={B} N={N}", flush=True)
    J = core.s2dw_core_comp_Jmax(B, 2.0)
    K, Phi2, _ = core.s2dw_core_init_kernels(J, B, 2.0)
    S = core.s2dw_core_init_directionality(B, N)
    monkeypatch.delenv("S2DW_HIP_FFT", raising=False)
    p = core.Plan(B, N, J, 2.0, K, Phi2, S)
    monkeypatch.setenv("S2DW_HIP_FFT", "generic")
    q = core.Plan(B, N, J, 2.0, K, Phi2, S)
    d = torch.from_numpy(np.ascontiguousarray(seeded_flm(B, 21 + B + N, red=True).T)).cuda()
    w, sc = [p.empty_wav(), q.empty_wav()], p.empty_scoeff()
    p.analysis(d, w[0], sc)
    q.analysis(d, w[1], sc)
    assert p.moments_fusable
    a = p.stat_moments(w[0]).cpu().numpy()
    b = p.analysis_moments(d, sc).cpu().numpy()
    torch.cuda.synchronize()
    assert float((w[0] - w[1]).abs().max()) <= TOL
    np.testing.assert_allclose(b, a, rtol=1e-9, atol=1e-9)
