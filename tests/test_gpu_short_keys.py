"""Varlen calls of at most 256 keys per segment at head_dim 128 (keys and values held in LDS, queries streamed past
them): every count of key blocks and remainders around them, query counts around the tile and item sizes, empty
segments on either side, row strides wider than a row, and a segment longer than the call's max_k said. Outputs against fp32 attention (bf16 probabilities and outputs:
max-abs 2e-2, mean-abs 2e-3), lse against fp32 logsumexp (scores of 128 bf16 products summed in fp32: 2e-3 as in
tests/test_gpu_attention.py)."""
import pytest
import torch

from helpers import assert_close, rand_bf16
from onereel_amd import scene
from oracle import attention as OA

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason='needs the GPU')]
DEV = 'cuda'


def _cu(lens):
    return torch.tensor([0] + lens).cumsum(0).int()


def _check(o, lse, q, k, v, lq, lk):
    cq, ck = _cu(lq).tolist(), _cu(lk).tolist()
    for s in range(len(lq)):
        if lq[s] == 0:
            continue
        ref, lref = OA.attention_lse(q[cq[s]:cq[s + 1]].float(), k[ck[s]:ck[s + 1]].float(), v[ck[s]:ck[s + 1]].float())
        assert_close(o[cq[s]:cq[s + 1]], ref, what=f'segment {s}: {lq[s]} queries, {lk[s]} keys')
        got = lse[:, cq[s]:cq[s + 1]]
        assert torch.isneginf(got).all() if lk[s] == 0 else (got - lref).abs().max() < 2e-3, s


@pytest.mark.parametrize('lq,lk,H,max_k', [
    ([1, 31, 32, 33, 127, 128, 129, 513], [1, 31, 32, 33, 64, 65, 96, 128], 3, None),
    ([129, 0, 40, 300, 7], [127, 50, 0, 97, 2], 8, None),
    ([255, 256, 257, 33, 1, 64, 65, 32], [129, 160, 161, 192, 193, 224, 225, 256], 2, None),
    ([300, 5, 70], [256, 0, 30], 5, None),
    ([200, 90], [100, 300], 2, 128),       # more keys than max_k said, in either form
    ([200, 90], [100, 600], 2, 256),
    ([2] * 256, [9] * 256, 2, None),       # the most segments of this form
])
def test_short_keys_match_reference(lq, lk, H, max_k):
    print(f'short keys lq={lq[:9]} lk={lk[:9]} H={H} max_k={max_k}', flush=True)
    q, k, v = (rand_bf16((sum(n), H, 128), 7 + i) for i, n in enumerate((lq, lk, lk)))
    lse = torch.empty(H, sum(lq), device=DEV)
    o = scene.varlen(q.to(DEV), k.to(DEV), v.to(DEV), _cu(lq).to(DEV), _cu(lk).to(DEV), max(lq), max_k or max(lk),
                     lse=lse)
    _check(o.cpu(), lse.cpu(), q, k, v, lq, lk)


@pytest.mark.parametrize('n_keys', [77, 200])
def test_short_keys_rows_in_wider_rows(n_keys):
    """rows inside wider ones and overlapping key ranges; nothing but the query rows is written"""
    H, D, n = 2, 128, 300
    wide = rand_bf16((n + 1, H + 1, D), 3).to(DEV)[:, :H]
    kv = rand_bf16((400, 2 * H, D), 5).to(DEV)
    k, v = kv[:, :H], kv[:, H:]
    out = torch.full((n + 1, H + 2, D), 7.0, dtype=torch.bfloat16, device=DEV)
    t32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    scene.varlen(wide[:n], k, v, t32([0, 140, n]), None, 160, n_keys, k_off=t32([100, 130]), k_len=t32([n_keys, 33]),
                 out=out[:n, :H])
    ref = OA.packed_attention(wide[:n].cpu(), k.cpu(), v.cpu(), [0, 140, n], None, k_off=[100, 130], k_len=[n_keys, 33])
    assert_close(out[:n, :H].cpu(), ref, what='rows in wider rows')
    assert bool((out[:, H:] == 7).all()) and bool((out[n] == 7).all())
