"""Frame memory's kernels at the edges of their tiles: column blocks, row batches, load steps, candidate pairs."""
import pytest
import torch

from onereel_amd.frame_memory import FrameMemory
from onereel_amd.layout import SceneLayout
from oracle import frame_memory as OF

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason='needs the GPU')]
DEV = 'cuda'


# columns below, at and past one wavefront's 128; rows per frame below, at and past one and two batches of 32
@pytest.mark.parametrize('N,C,row0,T', [(9, 8, 2, 3), (129, 128, 0, 64), (700, 136, 100, 65), (97, 72, 0, 33),
                                        (96, 2048, 7, 32)])
def test_frame_pool_edges(N, C, row0, T):
    print(f'pool N={N} C={C} row0={row0} T={T}', flush=True)
    hs = torch.randn(N, C + 8, generator=torch.Generator().manual_seed(N)).to(torch.bfloat16)
    frame = (torch.arange(N) + row0) // T
    n = int(frame.max()) + 2
    fm = FrameMemory(budget=2)
    fm.reset(SceneLayout([n], halo=0), 2)
    for _ in range(2):   # a second collect adds to the first
        fm.collect(frame.to(DEV), hs.to(DEV)[:, :C], layer=0)
    s_ref, c_ref = OF.pool(frame, hs[:, :C].contiguous(), n)
    assert torch.equal(fm.counts[0].cpu(), 2 * c_ref.float())
    # fp32 sums of at most 2 T terms of a few units: 2 T eps of the sum of magnitudes, a few times over
    assert (fm.sums[0].cpu().double() - 2 * s_ref).abs().max() <= 1e-5 * max(1.0, float(s_ref.abs().max()))


# either pool kernel and the sizes between them: wavefronts of 512 columns from a few to thousands, rows below, at and past
# 32, 96 and 128 a frame, row blocks that start and end inside a frame; the last: columns past a wavefront's 512
@pytest.mark.parametrize('n,T,C,row0', [(5000, 1, 64, 0), (700, 32, 512, 5), (700, 33, 504, 0), (700, 33, 512, 32),
                                        (700, 95, 512, 1), (1100, 96, 512, 0), (1200, 130, 512, 7), (30, 33, 512, 0),
                                        (401, 3, 520, 2)])
def test_frame_pool_adds_in_row_order(n, T, C, row0):
    """the bits of a plain loop over a frame's rows"""
    print(f'pool order n={n} T={T} C={C} row0={row0}', flush=True)
    N = n * T - row0 - T // 2            # the last frame is cut short too
    hs = torch.randn(N, C, generator=torch.Generator(device=DEV).manual_seed(T), device=DEV).to(torch.bfloat16)
    at = torch.arange(N, device=DEV) + row0
    fm = FrameMemory(budget=1)
    fm.reset(SceneLayout([n], halo=0), 2)
    fm.collect(at // T, hs, layer=0)
    full = torch.zeros(n * T, C, dtype=torch.bfloat16, device=DEV)
    full[row0:row0 + N] = hs             # + 0.0 for the rows that are not there changes no sum
    want = torch.zeros(n, C, device=DEV)
    for t in range(T):
        want += full.view(n, T, C)[:, t].float()
    assert torch.equal(fm.sums[0], want)
    assert torch.equal(fm.counts[0], torch.bincount(at // T, minlength=n).float())


# C below, at and past one round of 16 load steps (1024), odd candidate counts, more than 8 centres; no cluster of two
# (its members are equally near their mean)
@pytest.mark.parametrize('sizes,C', [([1], 5), ([3, 5], 33), ([4, 9, 3], 1024), ([3, 30, 8, 1], 2052), ([7] * 11, 1030)])
def test_frame_select_edges(sizes, C):
    print(f'select sizes={sizes} C={C}', flush=True)
    g = torch.Generator().manual_seed(C)
    base = torch.randn(len(sizes), C, generator=g).repeat_interleave(torch.tensor(sizes), 0)
    sums = 3 * (base + 0.05 * torch.randn(sum(sizes), C, generator=g))
    feats = torch.nn.functional.normalize(sums / 3, dim=-1)
    fm = FrameMemory(budget=len(sizes))
    fm.reset(SceneLayout([sum(sizes)], halo=0), 2)
    want = OF.select(feats, list(range(sum(sizes))), len(sizes))
    assert fm.select(feats.to(DEV)) == want
    fm.sums, fm.counts = {fm.layer: sums.to(DEV)}, {fm.layer: torch.full((sum(sizes),), 3.0, device=DEV)}
    fm.finish()
    assert fm.pending == want
