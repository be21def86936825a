"""The k-means passes at the edges of their tiles: candidates of one 16-row tile and of odd counts, past one chunk of the
update's member lists, clusters for one, two and four wavefront groups and past one round of 128, bf16 keys named by row
and fp32 keys. Checked against a float64 restatement of the same passes on groups that no rounding moves between
clusters (more groups than clusters would leave ties)."""
import pytest
import torch

from onereel_amd import _lib as L
from onereel_amd.memory import BoundaryMemory

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason='needs the GPU')]
DEV = 'cuda'


@pytest.mark.parametrize('B,H,D,M,dtype', [
    (5, 1, 64, 1, torch.bfloat16), (17, 3, 128, 3, torch.float32), (160, 5, 128, 33, torch.bfloat16),
    (999, 2, 64, 65, torch.bfloat16), (640, 1, 128, 129, torch.float32), (3000, 16, 128, 128, torch.bfloat16),
    (9001, 2, 128, 40, torch.bfloat16), (17000, 1, 64, 16, torch.float32)])
def test_select_passes(B, H, D, M, dtype):
    print(f'select B={B} H={H} D={D} M={M} {dtype}', flush=True)
    g = torch.Generator().manual_seed(B + M)
    group = torch.arange(B) * M // B
    init = torch.linspace(0, B - 1, M).round().long()
    group[init] = torch.arange(M)          # the cold start takes one member of each group
    x = (torch.randn(M, H, D, generator=g)[group] + 0.1 * torch.randn(B, H, D, generator=g)).to(dtype)
    n = torch.nn.functional.normalize(x.double(), dim=-1).transpose(0, 1)
    for wide in (False, True):
        if wide:    # candidates scattered over more rows, as a call names them
            rows = torch.randperm(2 * B + 1, generator=g)[:B]
            keys = torch.zeros(2 * B + 1, H, D, dtype=dtype)
            keys[rows] = x
            mem = BoundaryMemory(M)
            rep, valid = mem._select('a', keys.to(DEV), rows.to(torch.int32).to(DEV), B, H, D)
        else:
            mem = BoundaryMemory(M)
            rep, valid = mem.select('a', x.to(DEV))
        c = mem.centroids['a'].cpu().double()
        assert bool(valid.all())
        for h in range(H):
            mean = torch.stack([n[h, group == i].mean(0) for i in range(M)])
            # a mean of at most B unit vectors' elements in fp32, and x itself rounded: a few eps of 1 each
            assert (c[h] - mean).abs().max() < 1e-5
            d = ((n[h] - mean[group]) ** 2).sum(-1)
            chosen = rep[h].cpu()
            assert torch.equal(group[chosen], torch.arange(M))
            for i in range(M):              # nearest up to the rounding of |x|^2 - 2 x.c + |c|^2 near 1
                assert d[chosen[i]] <= d[group == i].min() + 1e-6


@pytest.mark.parametrize('B,H,D,M,dtype', [(777, 3, 128, 40, torch.bfloat16), (33, 1, 64, 7, torch.bfloat16),
                                           (777, 3, 128, 40, torch.float32)])
def test_workspace_of_each_key_type(B, H, D, M, dtype):
    """a call within exactly the bytes that its key type needs: nothing past them is written"""
    print(f'select workspace B={B} H={H} D={D} M={M} {dtype}', flush=True)
    x = torch.randn(B, H, D, generator=torch.Generator().manual_seed(B)).to(dtype).to(DEV)
    mem, fp32 = BoundaryMemory(M), int(dtype == torch.float32)
    rep, valid = mem.select('a', x)
    n = int(L.lib().or_memory_select_workspace_bytes(B, H, D, M, 50, fp32))
    ws = torch.full((n + 4096,), 0x5a, dtype=torch.uint8, device=DEV)
    c = torch.empty(H, M, D, device=DEV)
    init = torch.linspace(0, B - 1, M).round().to(torch.int32).to(DEV)
    got, ok = torch.empty_like(rep), torch.empty_like(valid)
    L.check(L.lib().or_memory_select(x.data_ptr(), fp32, None, x.stride(0), B, H, D, M, c.data_ptr(), init.data_ptr(),
                                     50, got.data_ptr(), ok.data_ptr(), ws.data_ptr(), n, L.stream_handle(x.device)),
            'or_memory_select')
    assert torch.equal(got, rep) and torch.equal(ok, valid) and torch.equal(c, mem.centroids['a'])
    assert bool((ws[n:] == 0x5a).all())
