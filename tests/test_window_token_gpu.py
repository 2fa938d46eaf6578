"""Single tokens over paged keys: what is loaded ahead of the tile before, and the keys past the last, at the edges of tiles, of a wave's
tiles and of the rule that chooses the form."""
import pytest
import torch

from k8s_llm_scheduler_amd.ops import reference as ref
from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,G,D,most", [(1, 1, 128, 1024), (16, 4, 128, 1024), (17, 4, 128, 1024), (32, 4, 96, 1024), (33, 4, 128, 1024), (20, 4, 64, 4096),
                                        (66, 4, 96, 1024)])
@pytest.mark.parametrize("window,chunk", [(0, 0), (256, 0), (0, 300)])
def test_edges_of_tiles(T, G, D, most, window, chunk):
    g = torch.Generator().manual_seed(T + D + window)
    H, bs = 4 * G, 16
    keys = torch.tensor([(1, 31, 32, 33, 255, 256, 257, 289, 512, 545, 700, 2)[i % 12] for i in range(T)])
    per = -(-700 // bs)
    tables = torch.randperm(T * per + 3, generator=g)[:T * per].view(T, per).to(torch.int32)
    kc, vc = (torch.randn((T * per + 3) * bs, G, D, generator=g).to(torch.bfloat16) for _ in range(2))
    for t in range(T):                                   # what lies behind a sequence's last key is not read as a value
        last = int(keys[t])
        for j in range(last, min(per * bs, last + 40)):
            vc[int(tables[t, j // bs]) * bs + j % bs] = float("nan")
    q, gate = torch.randn(T, H * D, generator=g).to(torch.bfloat16), torch.randn(T, H, generator=g).to(torch.bfloat16)
    sinks, slopes = torch.randn(H, generator=g), torch.rand(H, generator=g) / 50
    pos, seq = (keys - 1).to(torch.int32), torch.arange(T, dtype=torch.int32)
    pos[T // 2] = -1                                     # an idle row
    args = (q, gate, kc, vc, None, None, tables, seq, pos)
    tail = (window, 0, D ** -0.5, True, bs)
    want = ref.window_attention(*args, H, G, D, D, *tail, torch.float32, chunk, 0.0, sinks, True, slopes)
    cu = torch.arange(T + 1, dtype=torch.int32).cuda()
    got = sm.window_attention(*(t.cuda() if t is not None else None for t in args), H, *tail, cu, 1, most, chunk=chunk, sinks=sinks.cuda(),
                              gate_per_head=True, slopes=slopes.cuda())
    live = pos >= 0
    # a rounding to bf16 of the result, the gate's and the softmax's fp32; weights enter as two bf16 terms (2^-16 of values up to 5)
    assert ((got.cpu().float() - want.float()).abs()[live] <= 2.0 ** -8 * want.float().abs()[live] + 5 * 2.0 ** -14).all()
    assert (got.cpu()[~live] == 0).all()
