"""Kernel paths that only a switch at plan creation selects, against the
default plan: two-FFT beta columns and the generic beta lengths beside the
alpha stage without the gamma-DFT (S2DW_HIP_BETA_ONE=0), and the synthesis
contraction with a shared V tile on its own work list
(S2DW_HIP_SYN_MFMA=staged) with chunk widths ceil(B / 16) that are no power of
two.

Tolerance 1e-12 max abs: the same transform by other FFT lengths and another
summation order, on red N(0,1)/(l+1) spectra (analysis) and on their
coefficients (synthesis, f_lm of the same scale)."""
import numpy as np
import pytest

from conftest import seeded_flm
from s2dw_amd import core

pytestmark = pytest.mark.gpu

TOL = 1e-12

CASES = ([("S2DW_HIP_BETA_ONE", "0", B, N) for B, N in ((8, 3), (65, 2), (128, 3), (300, 2), (512, 2), (513, 1), (600, 2))] +
         [("S2DW_HIP_SYN_MFMA", "staged", B, N) for B, N in ((17, 3), (65, 3), (130, 5), (256, 2), (397, 6))])


@pytest.mark.parametrize("name,value,B,N", CASES)
def test_switch(name, value, B, N, monkeypatch):
    import torch

    print(f"{name}={value} B={B} N={N}", flush=True)
    J = min(5, core.s2dw_core_comp_Jmax(B, 2.0))
    K, Phi2, _ = core.s2dw_core_init_kernels(J, B, 2.0)
    S = core.s2dw_core_init_directionality(B, N)
    monkeypatch.delenv(name, raising=False)
    p = core.Plan(B, N, J, 2.0, K, Phi2, S)
    monkeypatch.setenv(name, value)
    q = core.Plan(B, N, J, 2.0, K, Phi2, S)
    d = torch.from_numpy(np.ascontiguousarray(seeded_flm(B, 31 + B + N, red=True).T)).cuda()
    w, sc, out = [p.empty_wav(), q.empty_wav()], p.empty_scoeff(), [p.empty_flm(), q.empty_flm()]
    for x, wx in zip((p, q), w):
        x.analysis(d, wx, sc)
    for x, o in zip((p, q), out):
        x.synthesis(w[0], sc, o)
    torch.cuda.synchronize()
    assert float((w[0] - w[1]).abs().max()) <= TOL
    assert float((out[0] - out[1]).abs().max()) <= TOL
    assert float((out[1] - d).abs().max()) <= TOL


def test_smooth_length_above_1024():
    """B = 1200: 2400 points run directly and off the workgroup engine, beside
    alpha transforms of 8192 points without the gamma-DFT; analysis and back,
    tolerance as above."""
    import torch

    B, N = 1200, 2
    print(f"round trip B={B} N={N}", flush=True)
    K, Phi2, _ = core.s2dw_core_init_kernels(2, B, 2.0)
    S = core.s2dw_core_init_directionality(B, N)
    p = core.Plan(B, N, 2, 2.0, K, Phi2, S)
    d = torch.from_numpy(np.ascontiguousarray(seeded_flm(B, 77, red=True).T)).cuda()
    w, sc, out = p.empty_wav(), p.empty_scoeff(), p.empty_flm()
    p.analysis(d, w, sc)
    p.synthesis(w, sc, out)
    torch.cuda.synchronize()
    assert float((out - d).abs().max()) <= TOL
