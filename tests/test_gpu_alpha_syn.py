"""The synthesis alpha stage with the gamma-DFT in it, and the three-stage FFT
engine, against the generic kernels (S2DW_HIP_FFT=generic at plan creation:
alpha transform of packed real rows, gamma-DFT in the beta kernels): both
parities of N, n = 0 packed over row pairs, every remainder of the gamma loop,
and lengths at the edges of the work lengths 2048 and 4096.

Tolerance 1e-12 max abs for N(0,1) coefficients falling as 1/(2 hi): f_lm is a
quadrature mean of O(1) terms over 4 hi^2 N samples, whose rounding through
O(log hi) stages and an O(L) contraction is below 1e-13."""
import os

import numpy as np
import pytest

from conftest import seeded_flm
from s2dw_amd import core

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _plan(B, N, J, alpha, K, Phi2, S, generic):
    old = os.environ.pop("S2DW_HIP_FFT", None)
    try:
        if generic:
            os.environ["S2DW_HIP_FFT"] = "generic"
        return core.Plan(B, N, J, alpha, K, Phi2, S)
    finally:
        os.environ.pop("S2DW_HIP_FFT", None)
        if old is not None:
            os.environ["S2DW_HIP_FFT"] = old


CASES = ([(40, N, 2.0) for N in range(1, 13)] + [(48, N, 3.0) for N in (16, 17, 31, 32)] +
         [(B, 3, 2.0) for B in (2, 3, 4, 5, 8, 9, 16, 17, 33, 64, 65, 128, 129, 256, 257)] +
         [(300, 4, 2.0), (512, 3, 2.0), (512, 8, 4.0), (511, 5, 2.0), (513, 2, 2.0), (640, 3, 3.0), (1023, 1, 2.0)])


@pytest.mark.parametrize("B,N,alpha", CASES)
def test_alpha_stage_vs_generic(B, N, alpha):
    import torch

    if N > B:
        pytest.skip("N <= B")
    print(f"alpha_syn B={B} N={N} alpha={alpha}", flush=True)
    J = min(3, core.s2dw_core_comp_Jmax(B, alpha))
    K, Phi2, _ = core.s2dw_core_init_kernels(J, B, alpha)
    S = core.s2dw_core_init_directionality(B, N)
    p, q = (_plan(B, N, J, alpha, K, Phi2, S, generic) for generic in (False, True))
    g = torch.Generator(device="cuda")
    g.manual_seed(3 * B + N)
    wav = torch.randn(p.empty_wav().shape, dtype=torch.float64, device="cuda", generator=g) / (2.0 * B)
    sc = torch.zeros_like(p.empty_scoeff())
    out = [x.empty_flm() for x in (p, q)]
    for x, o in zip((p, q), out):
        x.synthesis(wav, sc, o)
    torch.cuda.synchronize()
    assert torch.isfinite(out[0]).all() and torch.isfinite(out[1]).all()
    assert float((out[0] - out[1]).abs().max()) <= TOL
    # and the analysis alpha and beta stages of the same lengths
    d = torch.from_numpy(np.ascontiguousarray(seeded_flm(B, 5 + B + N, red=True).T)).cuda()
    w = [p.empty_wav(), q.empty_wav()]
    p.analysis(d, w[0], sc)
    q.analysis(d, w[1], sc)
    torch.cuda.synchronize()
    assert float((w[0] - w[1]).abs().max()) <= TOL
