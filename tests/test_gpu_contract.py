"""The analysis contraction by parity of l against the general contraction
kernels (selected through S2DW_HIP_ANA_KERNEL at plan creation): every number
of columns, sizes at the edges of its groups of 8 l, 4 m' and 64 m, and
directionality arrays outside its symmetry, which must take the general path.

Tolerance 1e-12 max abs on red N(0,1)/(l+1) spectra: both sum the same O(L)
products of O(1) values in another order (about L eps = 1e-13 at L = 260)."""
import os

import numpy as np
import pytest

from conftest import seeded_flm
from s2dw_amd import core

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _analysis(B, N, alpha, J, K, Phi2, S, f, kernel=None):
    import torch

    old = os.environ.get("S2DW_HIP_ANA_KERNEL")
    try:
        if kernel:
            os.environ["S2DW_HIP_ANA_KERNEL"] = kernel
        plan = core.Plan(B, N, J, alpha, K, Phi2, S)
    finally:
        os.environ.pop("S2DW_HIP_ANA_KERNEL", None)
        if old is not None:
            os.environ["S2DW_HIP_ANA_KERNEL"] = old
    d = torch.from_numpy(np.ascontiguousarray(f.T)).cuda()
    wav, sc = plan.empty_wav(), plan.empty_scoeff()
    plan.analysis(d, wav, sc)
    torch.cuda.synchronize()
    return wav.cpu().numpy(), sc.cpu().numpy()


CASES = ([(B, 3, 2.0) for B in (4, 7, 8, 9, 15, 16, 17, 63, 64, 65, 127, 129)] +
         [(40, N, 2.0) for N in range(1, 10)] + [(130, N, 3.0) for N in (1, 2, 5, 6, 8)] +
         [(100, 4, 1.5), (260, 8, 2.0), (257, 7, 3.0)])


@pytest.mark.parametrize("B,N,alpha", CASES)
def test_parity_contraction_vs_general(B, N, alpha):
    print(f"contraction B={B} N={N} alpha={alpha}", flush=True)
    J = core.s2dw_core_comp_Jmax(B, alpha)
    K, Phi2, _ = core.s2dw_core_init_kernels(J, B, alpha)
    S = core.s2dw_core_init_directionality(B, N)
    f = seeded_flm(B, 11 + B + N, red=True)
    w, sc = _analysis(B, N, alpha, J, K, Phi2, S, f)
    for kernel in ("mfma", "valu"):
        w0, sc0 = _analysis(B, N, alpha, J, K, Phi2, S, f, kernel)
        assert np.abs(w - w0).max() <= TOL
        np.testing.assert_array_equal(sc, sc0)


@pytest.mark.parametrize("N,turn", [(3, 1j), (4, 1.0 + 0.5j), (2, 1j), (5, -1.0)])
def test_other_directionalities(N, turn):
    """S times a constant: an imaginary S(l,0) and an S with both parts are
    outside the symmetry, the others inside."""
    print(f"directionality N={N} turn={turn}", flush=True)
    B, alpha = 48, 2.0
    J = core.s2dw_core_comp_Jmax(B, alpha)
    K, Phi2, _ = core.s2dw_core_init_kernels(J, B, alpha)
    S = core.s2dw_core_init_directionality(B, N) * turn
    f = seeded_flm(B, 5 + N, red=True)
    w, _ = _analysis(B, N, alpha, J, K, Phi2, S, f)
    w0, _ = _analysis(B, N, alpha, J, K, Phi2, S, f, "valu")
    assert np.abs(w - w0).max() <= TOL
