"""Host-array entry points whose copies go through the ring of pinned slots:
totals below its minimum, within one slot, across slot and scale boundaries,
and beyond the ring (the static layout at B = 256, N = 8: 150 MB).  Whole
numbers of bytes move, so static, dynamic and device-plan results agree bit
for bit."""
import numpy as np
import pytest

from conftest import seeded_flm
from s2dw_amd import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N", [(16, 2), (96, 3), (150, 4), (256, 8)])
def test_host_copies(B, N, monkeypatch):
    import torch

    monkeypatch.setenv("S2DW_HIP_ROUNDING", "streamed")
    J = core.s2dw_core_comp_Jmax(B, 2.0)
    K, Phi2, bl = core.s2dw_core_init_kernels(J, B, 2.0)
    S = core.s2dw_core_init_directionality(B, N)
    f = np.asfortranarray(seeded_flm(B, 3 + B, red=True))
    wav, sc = core.s2dw_core_analysis_flm2wav_dynamic(f, K, S, J, B, N, bl, 2.0)
    stat, sc1 = core.s2dw_core_analysis_flm2wav(f, K, S, J, B, N, bl, 2.0)
    np.testing.assert_array_equal(sc, sc1)
    for j, w in enumerate(wav):
        np.testing.assert_array_equal(stat[j, :w.shape[0], :w.shape[1]], w)
    plan = core.Plan(B, N, J, 2.0, K, Phi2, S)
    d, dsc = plan.empty_wav(), plan.empty_scoeff()
    plan.analysis(torch.from_numpy(np.ascontiguousarray(f.T)).cuda(), d, dsc)
    torch.cuda.synchronize()
    for j, w in enumerate(wav):
        np.testing.assert_array_equal(plan.scale_view(d, j).cpu().numpy().transpose(2, 1, 0), w)
    g = core.s2dw_core_synthesis_wav2flm_dynamic(wav, sc, K, Phi2, S, J, B, N, bl, 2.0)
    g1 = core.s2dw_core_synthesis_wav2flm(stat, sc, K, Phi2, S, J, B, N, bl, 2.0)
    np.testing.assert_array_equal(g, g1)
