"""Host-array copies in every size of the staging ring's slots (totals up to
16, 64 and 256 MB and beyond), small and large ones in turn so that the ring
grows and its slots change size while earlier transfers may still use them,
into arrays that the caller has and has not touched before.  Whole numbers of
bytes move: every result equals the device plan's bit for bit."""
import numpy as np
import pytest

from conftest import seeded_flm
from s2dw_amd import core

pytestmark = pytest.mark.gpu


# (B, N): dynamic / static totals 2.3 / 13, 157 / 537, 0.6 / 2.6, 24 / 94, 5 / 29 MB
SIZES = [(128, 3), (512, 8), (64, 3), (256, 5), (190, 3)]


def test_slot_sizes(monkeypatch):
    import torch

    monkeypatch.setenv("S2DW_HIP_ROUNDING", "streamed")
    for B, N in SIZES:
        print(f"host copies B={B} N={N}", flush=True)
        J = core.s2dw_core_comp_Jmax(B, 2.0)
        K, Phi2, bl = core.s2dw_core_init_kernels(J, B, 2.0)
        S = core.s2dw_core_init_directionality(B, N)
        f = np.asfortranarray(seeded_flm(B, 9 + B, red=True))
        plan = core.Plan(B, N, J, 2.0, K, Phi2, S)
        d, dsc, dflm = plan.empty_wav(), plan.empty_scoeff(), plan.empty_flm()
        plan.analysis(torch.from_numpy(np.ascontiguousarray(f.T)).cuda(), d, dsc)
        plan.synthesis(d, dsc, dflm)
        torch.cuda.synchronize()
        want = [plan.scale_view(d, j).cpu().numpy().transpose(2, 1, 0) for j in range(J + 1)]
        wflm = dflm.cpu().numpy().T
        args = (K, S, J, B, N, bl, 2.0)
        wav, sc = core.s2dw_core_analysis_flm2wav_dynamic(f, *args)
        for a, b in zip(wav, want):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(core.s2dw_core_synthesis_wav2flm_dynamic(wav, sc, K, Phi2, *args[1:]), wflm)
        for w in wav:  # the same arrays again, through the C entry
            w.fill(np.nan)
        ptrs = (core._dp * (J + 1))(*[core._p(w) for w in wav])
        assert core.lib().s2dw_hip_analysis_flm2wav_dynamic(ptrs, core._p(sc), core._p(f), core._p(K), core._p(S), J, B,
                                                            N, bl, 2.0) == 0
        for a, b in zip(wav, want):
            np.testing.assert_array_equal(a, b)
        stat, sc1 = core.s2dw_core_analysis_flm2wav(f, *args)
        np.testing.assert_array_equal(sc, sc1)
        for j, w in enumerate(want):
            np.testing.assert_array_equal(stat[j, :w.shape[0], :w.shape[1]], w)
        np.testing.assert_array_equal(core.s2dw_core_synthesis_wav2flm(stat, sc, K, Phi2, *args[1:]), wflm)
