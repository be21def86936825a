"""The planner of the varlen call at the sizes where its forms change: segments ranked by counting up to 512 and by the
bitonic network past them, heads dealt to the eight queues by head (H a multiple of 8) or by unit, one block of items
or several. Every segment's rows against fp32 attention on the same inputs: an item that the planner lost, doubled or
gave the wrong ranges leaves wrong rows. Small calls that would run without the planner are kept on it: at head_dim 64 by a
grid of two blocks, at 128 by a max_k that is not a short one. Tolerance as tests/test_gpu_attention.py (bf16 probabilities
and outputs)."""
import pytest
import torch

from helpers import assert_close
from onereel_amd import _lib as L
from onereel_amd import scene

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason='needs the GPU')]
DEV = 'cuda'


@pytest.mark.parametrize('n_seg,H,D', [(1, 3, 64), (8, 16, 64), (9, 12, 128), (511, 1, 64), (512, 5, 64), (513, 5, 64),
                                       (513, 8, 128), (1500, 2, 64), (4096, 1, 128)])
def test_every_item_runs_once(monkeypatch, n_seg, H, D):
    if D == 64:
        monkeypatch.setenv('ONEREEL_ATTN_MAX_BLOCKS', '2')
    print(f'plan n_seg={n_seg} H={H} D={D}', flush=True)
    g = torch.Generator().manual_seed(n_seg + H)
    lq = torch.randint(0, 5 if n_seg > 9 else 300, (n_seg,), generator=g)
    lk = torch.randint(1, 40, (n_seg,), generator=g)
    lq[0] = max(int(lq[0]), 1)
    if n_seg > 100:
        lq[n_seg // 2] = 700     # one segment of several tiles among the short ones
    cq, ck = (torch.cat([torch.zeros(1, dtype=torch.long), x.cumsum(0)]) for x in (lq, lk))
    q, k, v = (torch.randn(int(c[-1]), H, D, generator=g).bfloat16() for c in (cq, ck, ck))
    # the planner leaves its queues in the workspace: the items it counted
    ws = torch.zeros(int(L.lib().or_varlen_workspace_size(n_seg, q.shape[0], H, D)), dtype=torch.uint8, device=DEV)
    o = scene.varlen(q.to(DEV), k.to(DEV), v.to(DEV), cq.int().to(DEV), ck.int().to(DEV), int(lq.max()),
                     max(int(lk.max()), 257), workspace=ws)
    rows = 256 if D == 128 else 128
    counted = ws[:1024].view(torch.int32)[1::32].sum().item()
    split = int(ws.view(torch.int32)[3])
    items = H * int(((lq + rows - 1) // rows).sum())
    assert counted == items if split == 0 else counted > items
    # every query row against all keys of its segment, padded to the longest
    seg = torch.repeat_interleave(torch.arange(n_seg), lq)
    idx = torch.arange(int(lk.max()))[None] + ck[:-1, None]
    live = torch.arange(int(lk.max()))[None] < lk[:, None]
    idx = idx.clamp(max=int(ck[-1]) - 1)
    rows = idx[seg]
    s = torch.einsum('nhd,nkhd->nhk', q.float(), k.float()[rows]) * D ** -0.5
    s = s.masked_fill(~live[seg][:, None], float('-inf'))
    ref = torch.einsum('nhk,nkhd->nhd', s.softmax(-1), v.float()[rows])
    assert_close(o.cpu(), ref, what='planned items')
