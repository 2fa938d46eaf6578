"""Which workgroup form the paged prompt attention takes, by the tokens that a batch really brings, without a GPU."""
import pytest

from k8s_llm_scheduler_amd import ops


@pytest.mark.parametrize("nq,nkv,qlens,form", [
    (64, 8, [241], 5), (64, 8, [97], 5), (64, 8, [512], 4), (64, 8, [900], 4), (64, 8, [1500], 16), (64, 8, [3413], 16), (64, 8, [24], 5),
    (32, 8, [512], 5), (32, 8, [2048], 8), (32, 8, [2049], 16), (8, 1, [3413], 5), (64, 8, [50] * 8, 4), (32, 8, [50] * 8, 5),
    # unequal batches, which a bound by the longest sequence would take for 8 or 9 prompts of that length
    (64, 8, [241] + [1] * 8, 4), (64, 8, [97] + [1] * 8, 5), (64, 8, [512] + [1] * 8, 4), (8, 1, [900] + [1] * 8, 5), (8, 1, [3000] + [1] * 8, 5),
    (64, 8, [300, 40, 50, 60, 70], 4), (32, 8, [1200, 30, 60], 4), (32, 8, [1500] + [1] * 8, 4), (64, 8, [900] + [1] * 8, 16),
    (64, 8, [2000, 100, 100, 100], 16), (16, 16, [1], 5), (64, 4, [1], 5)])
def test_rule(nq, nkv, qlens, form):
    assert ops._prefill_form(sum(qlens), max(qlens), len(qlens), nq, nkv) == form


def test_bound_on_the_tokens_of_a_padded_batch():
    """Tokens beyond the sequences' (a captured step's padding) never ask for more than every sequence at its longest."""
    assert ops._prefill_form(1 << 20, 97, 1, 64, 8) == ops._prefill_form(97, 97, 1, 64, 8)
