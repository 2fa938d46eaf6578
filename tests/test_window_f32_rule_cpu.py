"""Which fp32 portions of windowed attention stay on the plain-FMA kernel and its key splits: few tokens behind many keys."""
import pytest

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm


def plain(T, longest, H, G, D, keys, window=0):
    rows = ops.native().window_tile_rows(H, G, D, D)
    return sm.window_f32_plain(T, longest, H, G, D, min(keys, window or keys), sm.window_splits(T, G, window, 0, keys, rows), rows)


@pytest.mark.parametrize("T,longest,H,G,D,keys", [(2, 2, 16, 4, 128, 1000), (2, 2, 16, 4, 128, 30000), (8, 8, 16, 4, 128, 3000),
                                                  (8, 8, 32, 8, 128, 30000), (8, 5, 16, 4, 64, 1000), (16, 16, 16, 4, 64, 3000),
                                                  (4, 4, 8, 8, 128, 3000), (4, 4, 16, 1, 128, 8000), (16, 16, 8, 8, 64, 30)])
def test_few_tokens_behind_many_keys_stay(T, longest, H, G, D, keys):
    assert plain(T, longest, H, G, D, keys)


@pytest.mark.parametrize("T,longest,H,G,D,keys", [(2, 2, 16, 4, 128, 30), (24, 24, 16, 4, 128, 3000), (97, 97, 16, 4, 128, 30000), (8, 8, 32, 8, 128, 1000),
                                                  (48, 12, 16, 4, 64, 8000), (24, 24, 8, 8, 64, 8000), (16, 16, 16, 1, 128, 1000), (300, 300, 32, 8, 128, 300)])
def test_others_do_not(T, longest, H, G, D, keys):
    assert not plain(T, longest, H, G, D, keys)


def test_a_window_bounds_the_keys():
    assert plain(2, 2, 16, 4, 128, 30000, 1024) and not plain(24, 24, 16, 4, 128, 30000, 1024) and not plain(2, 2, 16, 4, 128, 30000, 64)


def test_every_form_of_the_kernel_has_its_figures():
    forms = [(H, G, D) for D in (32, 64, 96, 128, 256) for G in (1, 2, 3, 4, 8) for R in (1, 2, 3, 4, 8, 16, 32) for H in (R * G,)]
    for H, G, D in forms:
        if ops.native().window_f32_ok(H, G, D, D):
            assert (D, H // G) in sm._WINDOW_PLAIN_COST and D in sm._WINDOW_F32_COST
            assert all(plain(T, T, H, G, D, k) in (True, False) for T in (1, 100, 5000) for k in (1, 4096))
