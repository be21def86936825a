"""Varlen calls of at most 256 keys per segment at head_dim 128 (keys and values held in LDS, queries streamed past
them): every count of key blocks and remainders around them, query counts around the tile and item sizes, empty
segments on either side, row strides wider than a row, and a segment longer than the call's max_k said. Outputs against
fp32 attention (bf16 probabilities and outputs: max-abs 2e-2, mean-abs 2e-3), lse against fp32 logsumexp (scores of 128
bf16 products summed in fp32: 2e-3 as in tests/test_gpu_attention.py), and both against the ring kernel's bits."""
import pytest
import torch

from helpers import assert_close, rand_bf16
from onereel_amd import scene
from onereel_amd.layout import SceneLayout
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


@pytest.mark.parametrize('lq,lk,H,max_k', [
    ([1, 31, 32, 33, 127, 128, 129, 513], [1, 31, 32, 33, 64, 65, 96, 128], 3, 128),
    ([255, 256, 257, 33, 1, 64, 65, 32], [129, 160, 161, 192, 193, 224, 225, 256], 3, 256),
    ([300, 40, 700, 5], [70, 0, 100, 128], 5, 256),    # short segments in the form of the long ones
    ([300, 40, 700], [70, 200, 330], 5, 128),          # a segment longer than max_k says
])
def test_bits_do_not_depend_on_max_k(monkeypatch, lq, lk, H, max_k):
    """the ring kernel takes the same call when max_k is larger: the same bits, as long as it does not split items by keys
    (a grid of three blocks makes these calls too long for that) and no probability passes 2^20 of the first block's
    maximum"""
    print(f'short keys against the ring kernel lq={lq} lk={lk} H={H} max_k={max_k}', flush=True)
    q, k, v = (rand_bf16((sum(n), H, 128), 11 + i).to(DEV) for i, n in enumerate((lq, lk, lk)))
    cq, ck = _cu(lq).to(DEV), _cu(lk).to(DEV)
    got, want = (torch.empty(H, sum(lq), device=DEV) for _ in range(2))
    o = scene.varlen(q, k, v, cq, ck, max(lq), max_k, lse=got)
    monkeypatch.setenv('ONEREEL_ATTN_MAX_BLOCKS', '3')
    ref = scene.varlen(q, k, v, cq, ck, max(lq), 1000, lse=want)
    assert torch.equal(o, ref) and torch.equal(got, want)


@pytest.mark.parametrize('n_keys', [64, 100, 128, 150, 192, 199, 256])
def test_short_keys_running_max_moves(n_keys):
    """keys that grow by jumps at a third and two thirds of the blocks, for queries of three sizes: the largest queries'
    scores pass the running max by far more than 2^20 there, the smaller ones' of the same tiles by a factor that leaves
    their earlier keys part of the result (O, l and the scores in flight are rescaled with them)"""
    H, n, nb = 2, 400, (n_keys + 31) // 32
    print(f'short keys, moving maximum: {n_keys} keys', flush=True)
    q, k, v = (rand_bf16((m, H, 128), 17 + i) for i, m in enumerate((n, n_keys, n_keys)))
    block = torch.arange(n_keys) // 32
    grow = torch.where(block >= max(2 * nb // 3, 1), 40.0, torch.where(block >= max(nb // 3, 1), 12.0, 1.0))
    size = torch.tensor([1.0, 0.06, 0.02])[torch.arange(n) % 3]
    k = (k.float() * grow[:, None, None]).bfloat16()
    q = (q.float() * size[:, None, None]).bfloat16()
    lse = torch.empty(H, n, device=DEV)
    o = scene.varlen(q.to(DEV), k.to(DEV), v.to(DEV), _cu([n]).to(DEV), _cu([n_keys]).to(DEV), n, n_keys, lse=lse)
    s = torch.einsum('qhd,khd->hqk', q.float(), k.float()) * 128 ** -0.5 * 1.4426950408889634
    first, last = (s[:, :, block == b].amax(-1) for b in (0, nb - 1))
    assert bool((last - first > 20).any()) and bool(((last - first > 0.5) & (last - first < 4)).any())
    _check(o.cpu(), lse.cpu(), q, k, v, [n], [n_keys])


def test_small_scopes_fused_and_packed_agree(monkeypatch):
    """a scene layer whose scopes have at most 256 keys: the packed flow's call takes the short form, the fused one's (queries
    by source row) the ring kernel, here without key splits: the same bits"""
    lengths, T, counts, H, D = [2, 1, 2], 50, [20, 33, 7], 6, 128
    S, Le = sum(lengths) * T, sum(counts)
    q, k, v = (rand_bf16((S, H, D), 31 + i).to(DEV) for i in range(3))
    eq, ek, ev = (rand_bf16((Le, H, D), 41 + i).to(DEV) for i in range(3))
    cos, sin = (x.to(DEV) for x in OA.rope_table_3d(8, 5, 10, D))
    plan = scene.ScopePlan(SceneLayout(lengths, halo=0, extra={0: [3], 1: [0, 4], 2: []}), T, counts, Le, True, None, True,
                           True, torch.device(DEV))
    assert 128 < plan.max_k <= 256
    monkeypatch.setenv('ONEREEL_ATTN_MAX_BLOCKS', '1')
    a, b = (scene.scene_attention(plan, q, k, v, eq, ek, ev, cos, sin, mode='raw', fused=fused) for fused in (True, False))
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
