"""head_dim 64 calls whose items are resident at once run without the planner: the same bits as the planner's queues give
(a grid of three blocks makes a call too large for the direct form), over empty segments, more than 64 of them, keys by
offset and count, per-head key counts, queries by source row, values and keys read in place, and the log-sum-exp."""
import pytest
import torch

from helpers import assert_close
from onereel_amd import attention as A
from onereel_amd import scene

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason='needs the GPU')]
DEV, D = 'cuda', 64


def both(monkeypatch, call):
    got = call()
    monkeypatch.setenv('ONEREEL_ATTN_MAX_BLOCKS', '3')
    ref = call()
    monkeypatch.delenv('ONEREEL_ATTN_MAX_BLOCKS')
    for x, y in zip(got, ref):
        assert torch.equal(x, y)
    return got


def randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV).to(torch.bfloat16)


@pytest.mark.parametrize('H,lq,lk', [
    (2, [1], [1]), (3, [128, 129, 0, 127], [31, 32, 33, 65]), (12, [300, 5, 1, 257], [96, 0, 700, 64]),
    (1, [(7 * i) % 130 for i in range(200)], [1 + (13 * i) % 90 for i in range(200)]),
    (16, [1500, 1524], [100, 333]),            # the most items of 16 heads that are direct
])
def test_direct_matches_queues(monkeypatch, H, lq, lk):
    print(f'direct H={H} segments={len(lq)}', flush=True)
    g = torch.Generator(device=DEV).manual_seed(sum(lq))
    q, k, v = randn(g, sum(lq), H, D), randn(g, sum(lk), H, D), randn(g, sum(lk), H, D)
    cu_q, cu_k = A.cu_seqlens(lq), A.cu_seqlens(lk)
    o, lse = both(monkeypatch, lambda: A.varlen_lse(q, k, v, cu_q, cu_k, max(lq), max(lk)))
    a = b = 0
    for n, m in zip(lq, lk):
        if n and m:
            s = torch.einsum('qhd,khd->hqk', q[a:a + n].float().cpu(), k[b:b + m].float().cpu()) * D ** -0.5
            ref = torch.einsum('hqk,khd->qhd', s.softmax(-1), v[b:b + m].float().cpu())
            assert_close(o[a:a + n].cpu(), ref, what=f'{n} x {m}')
        a, b = a + n, b + m


def test_direct_options_match_queues(monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(1)
    H, n = 4, 3
    lq, lk, lead = [70, 200, 129], [150, 64, 97], [96, 32, 64]
    q, k, v, kt, vt = (randn(g, 500, H, D) for _ in range(5))
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    head = torch.tensor([[max(0, m - 17 * h) for h in range(H)] for m in lk], dtype=torch.int32, device=DEV).flatten()
    opts = dict(k_off=ints([0, 160, 230]), k_len=ints(lk), seg_q_src=ints([300, 0, 371]), n_q_video=500, sum_q=sum(lq))
    place = dict(v_tok=vt, v_lead=ints(lead), v_row=ints([5, 300, 120]), k_tok=kt, k_lead=ints(lead))

    def call(**more):
        out = torch.zeros(500, H, D, dtype=torch.bfloat16, device=DEV)
        scene.varlen(q, k, v, A.cu_seqlens(lq), None, max(lq), max(lk), out=out, **opts, **more)
        return [out]

    plain = both(monkeypatch, call)[0]
    heads = both(monkeypatch, lambda: call(k_len_head=head))[0]
    placed = both(monkeypatch, lambda: call(**place))[0]
    every = both(monkeypatch, lambda: call(k_len_head=head, **place))[0]
    assert not torch.equal(plain, heads) and not torch.equal(plain, placed) and not torch.equal(heads, every)
