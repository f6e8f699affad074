"""The synthesis gamma-DFT as a pass after the alpha transform (N from 16, from
20 where 2 hi > 512 is a power of two, on band limits from 200, N hi^2 outside
1.82 to 2.4 million), on both sides of the rule's lines, against the generic kernels (S2DW_HIP_FFT=generic at plan
creation): grouped launches of one stream and of two, the pair on the
three-stage and on the odd-length engine, and scales launched one by one.

Tolerance 1e-12 max abs for N(0,1) coefficients falling as 1/(2 hi): f_lm is a
quadrature mean of O(1) terms over 4 hi^2 N samples, whose rounding through
O(log hi + N) operations and an O(L) contraction is below 1e-13."""
import pytest

from s2dw_amd import core

pytestmark = pytest.mark.gpu

TOL = 1e-12

# dilation 1.2 puts several band limits of one plan on both sides of 200 and 256
CASES = [(199, 16, 2.0), (200, 15, 2.0), (200, 16, 2.0), (256, 17, 2.0), (256, 27, 2.0), (256, 28, 2.0), (246, 30, 2.0), (257, 16, 2.0), (300, 31, 2.0),
         (512, 19, 2.0), (512, 20, 2.0), (512, 21, 4.0), (513, 16, 2.0), (420, 18, 1.2)]


@pytest.mark.parametrize("B,N,alpha", CASES)
def test_gamma_pass(B, N, alpha, monkeypatch):
    import torch

    print(f"gamma pass B={B} N={N} alpha={alpha}", flush=True)
    J = min(4, core.s2dw_core_comp_Jmax(B, alpha))
    K, Phi2, _ = core.s2dw_core_init_kernels(J, B, alpha)
    S = core.s2dw_core_init_directionality(B, N)
    monkeypatch.delenv("S2DW_HIP_FFT", raising=False)
    p = core.Plan(B, N, J, alpha, K, Phi2, S)
    monkeypatch.setenv("S2DW_HIP_FFT", "generic")
    q = core.Plan(B, N, J, alpha, K, Phi2, S)
    g = torch.Generator(device="cuda")
    g.manual_seed(B + N)
    wav = torch.randn(p.empty_wav().shape, dtype=torch.float64, device="cuda", generator=g) / (2.0 * B)
    sc = torch.zeros_like(p.empty_scoeff())
    out = [x.empty_flm() for x in (p, q)]
    for x, o in zip((p, q), out):
        x.synthesis(wav, sc, o)
    torch.cuda.synchronize()
    assert torch.isfinite(out[0]).all() and torch.isfinite(out[1]).all()
    assert float((out[0] - out[1]).abs().max()) <= TOL


@pytest.mark.parametrize("B,N", [(256, 16), (512, 20)])
def test_gamma_pass_graph(B, N):
    """Replays of the captured synthesis (one stream, two streams), with other
    work between them, repeat the eager result bit for bit."""
    import torch

    print(f"gamma pass graph B={B} N={N}", flush=True)
    J = min(4, core.s2dw_core_comp_Jmax(B, 2.0))
    K, Phi2, _ = core.s2dw_core_init_kernels(J, B, 2.0)
    S = core.s2dw_core_init_directionality(B, N)
    p = core.Plan(B, N, J, 2.0, K, Phi2, S)
    g = torch.Generator(device="cuda")
    g.manual_seed(B)
    wav = torch.randn(p.empty_wav().shape, dtype=torch.float64, device="cuda", generator=g) / (2.0 * B)
    sc = torch.zeros_like(p.empty_scoeff())
    want, out = p.empty_flm(), p.empty_flm()
    p.synthesis(wav, sc, want)
    torch.cuda.synchronize()
    p.set_graphs(True)
    for _ in range(4):
        out.zero_()
        p.synthesis(wav, sc, out)
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(out), torch.view_as_real(want))
