"""The bounded memory's call on video and text rows in their own tensors against the call on them copied end to end
(itself checked against the oracle): the same kernels over the same keys in the same order, so the same bits."""
import pytest
import torch

from onereel_amd.layout import SceneLayout
from onereel_amd.memory import BoundaryMemory, MemoryAttention, frame_plan

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason='needs the GPU')]
DEV = 'cuda'


# one scene (its text rows follow its video rows, so its run of rows must end with the first tensor); padding text rows;
# frames of no whole key block; a text row alone
@pytest.mark.parametrize('lengths,T,counts,pad,H,D,M', [
    ([3], 40, [20], 0, 4, 64, 8), ([2, 3], 17, [5, 9], 3, 2, 128, 6), ([1, 4, 2], 70, [33, 1, 64], 0, 16, 128, 32),
    ([2, 2], 31, [1, 0], 0, 3, 128, 4)])
def test_text_in_its_own_tensor_gives_the_same_bits(lengths, T, counts, pad, H, D, M):
    print(f'memory with text lengths={lengths} T={T} counts={counts}', flush=True)
    lay = SceneLayout(lengths, halo=0)
    N, Le = lay.n_frames * T, sum(counts) + pad
    tr, at = [], 0
    for c in counts:
        tr.append((at, at + c))
        at += c
    plan = frame_plan(lay, T, torch.arange(N), N, [(j, lo * T, hi * T) for j, (lo, hi) in enumerate(lay.ranges)], tr,
                      {j for j, c in enumerate(counts) if c}, N, DEV)
    g = torch.Generator(device=DEV).manual_seed(3)
    new = lambda n: torch.randn(n, H, D, generator=g, device=DEV).to(torch.bfloat16)
    q, k, v, eq, ek, ev = new(N), new(N), new(N), new(Le), new(Le), new(Le)
    one, two, three = (MemoryAttention(BoundaryMemory(M)) for _ in range(3))
    wide = torch.cat([k, v], 1)     # keys that are not contiguous rows: copied first
    for _ in range(2):              # from no centroids, then from the stored ones
        ref = one('x', torch.cat([q, eq]), torch.cat([k, ek]), torch.cat([v, ev]), plan)
        for ov, ot in (two.with_text('x', q, k, v, eq, ek, ev, plan),
                       three.with_text('x', q, wide[:, :H], v, eq, ek, ev, plan)):
            assert torch.equal(ov, ref[:N]) and torch.equal(ot, ref[N:])
        assert torch.equal(one.memory.centroids['x'], two.memory.centroids['x'])
        assert not ref[N + sum(counts):].any()
