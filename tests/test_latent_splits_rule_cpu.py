"""Key splits of portions whose workgroups are four tokens (a grid's third side is sequences times splits)."""
import pytest

from k8s_llm_scheduler_amd.ops import seqmix as sm


@pytest.mark.parametrize("T,nseq", [(4, 60000), (2, 3000), (97, 1), (200, 2), (1, 65535), (512, 4)])
def test_grids_stay_within_their_bounds(T, nseq):
    for H in (1, 16, 32):
        ns = sm.latent_quad_splits(T, nseq, H, 4096)
        assert 1 <= ns <= 32 and ns * nseq <= 65535
        assert nseq > 1000 or ns == max(1, min(256 // (min(T, T // 4 + nseq) * ((H + 15) // 16)), 32))
