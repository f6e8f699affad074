"""Transform lengths of the workgroup FFT engine: every band limit up to 1024
runs its alpha (2hi - 1) and beta (2hi) stages on it, through Bluestein where
the length is no power of two.  Sizes at the edges of its work lengths
(M >= 2n - 1, a power of two up to 4096) against the CPU oracle.

Tolerance 1e-12 max abs on red N(0,1)/(l+1) spectra, the suite's bound for
device plans on red input (rounding of the O(log M) stages is ~1e-15 of the
coefficients' scale; the reference's own Wigner planes dominate)."""
import numpy as np
import pytest

import oracle as O
from conftest import seeded_flm
from s2dw_amd import core

pytestmark = pytest.mark.gpu

TOL = 1e-12

# (B, N, alpha, J): 5..9 lengths of a few points; 127, 129 around a work
# length; 257 and 511 the first and last of M = 2048 pairs that are no power
# of two, 300 a smooth length; 513 and 600 M = 4096 pairs; alpha = 1.2 puts
# scales j >= 2 on M = 4096 (584) and 2048 (487) launches of their own
LENGTHS = [(5, 2, 2.0, None), (9, 3, 2.0, None), (127, 2, 2.0, None), (129, 3, 3.0, None), (257, 2, 2.0, 4),
           (300, 3, 2.0, 3), (511, 2, 2.0, 3), (513, 2, 2.0, 2), (600, 1, 3.0, None), (700, 2, 1.2, 4)]


@pytest.mark.parametrize("B,N,alpha,J", LENGTHS)
def test_lengths_vs_oracle(B, N, alpha, J):
    import torch

    print(f"lengths B={B} N={N} alpha={alpha} J={J}", flush=True)
    st = O.Setup(B, N, alpha, J=J)
    f = seeded_flm(B, 7 + B, red=True)
    w_ref, sc_ref = st.analysis(f)
    plan = core.Plan(B, N, st.J, alpha, st.K, st.Phi2, st.S)
    d = torch.from_numpy(np.ascontiguousarray(f.T)).cuda()
    wav, sc, out = plan.empty_wav(), plan.empty_scoeff(), plan.empty_flm()
    plan.analysis(d, wav, sc)
    plan.synthesis(wav, sc, out)
    torch.cuda.synchronize()
    for j in range(st.J + 1):
        w = plan.scale_view(wav, j).cpu().numpy().transpose(2, 1, 0)
        assert np.abs(w - w_ref[j]).max() <= TOL, j
    np.testing.assert_array_equal(sc.cpu().numpy().T, sc_ref)
    assert np.abs(out.cpu().numpy().T - f).max() <= TOL
    if plan.moments_fusable:
        a = plan.stat_moments(wav).cpu().numpy()
        b = plan.analysis_moments(d, sc).cpu().numpy()
        # central sums of the same values in another grouping: O(n eps) of
        # sums of like terms (1e-9 leaves room for the cancelling odd moments)
        np.testing.assert_allclose(b, a, rtol=1e-9, atol=1e-9)
