"""Offsets that travel with a launch, and the concatenation of packed sequences, at the edges of what one launch holds
(896 values, 112 sequences) and of a block's chunks, with empty sequences among them: byte for byte what torch gives."""
import pytest
import torch

from onereel_amd import _lib as L
from onereel_amd import attention as A

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason='needs the GPU')]
DEV = 'cuda'


@pytest.mark.parametrize('sizes', [[1], [0, 3, 0], [895, 2], [896], [1000, 1, 2000]])
def test_device_ints(sizes):
    lists = [[(7919 * i + 13 * n) % 65537 - 30000 for i in range(n)] for n in sizes]
    for got, want in zip(L.device_ints(lists, DEV), lists):
        assert got.dtype == torch.int32 and got.cpu().tolist() == want


# up to 112 sequences, and long ones past them, in or_concat's launches; many short ones by torch
@pytest.mark.parametrize('n,H,D,most', [(1, 1, 64, 5), (3, 24, 128, 400), (112, 2, 64, 40), (113, 2, 128, 40),
                                        (250, 1, 64, 9), (113, 16, 128, 300), (250, 16, 128, 200)])
def test_concat(n, H, D, most):
    print(f'concat n={n} H={H} D={D}', flush=True)
    g = torch.Generator(device=DEV).manual_seed(n)
    size = lambda i, m: (i * 7919 + 3) % (m + 1)      # 0 .. most
    new = lambda r: torch.randn(r, H, D, generator=g, device=DEV).to(torch.bfloat16)
    seg = [(new(max(size(i, most), i == 0)), *(new(max(size(i + 5, most), i == 0)) for _ in range(2))) for i in range(n)]
    (q, k, v, cu_q, cu_k, max_q, max_k), nq = A._concat(seg)
    for got, parts in zip((q, k, v), zip(*seg)):
        assert torch.equal(got, torch.cat(parts))
    assert cu_q.cpu().tolist() == A._offsets(nq) and cu_k.cpu().tolist() == A._offsets([k.shape[0] for _, k, _ in seg])
    assert (max_q, max_k) == (max(nq), max(k.shape[0] for _, k, _ in seg))
    # what or_concat does not take is concatenated by torch: the same tensors
    wide = [(torch.cat([q, q], 2)[..., :D], k, v) for q, k, v in seg]
    assert torch.equal(A._concat(wide)[0][0], q) and torch.equal(A._concat(wide)[0][3], cu_q)


def test_cu_seqlens_are_there_on_return():
    """offsets handed out are read on other streams without an event between: they are filled when the call returns, also
    behind work that its own stream has still to do"""
    want = [3 * i for i in range(513)]
    junk = torch.full((513,), -1, dtype=torch.int32, device=DEV)   # what the offsets' allocation holds before
    torch.cuda.synchronize()
    del junk
    side = torch.cuda.Stream()
    torch.cuda._sleep(200_000_000)
    cu = A.cu_seqlens([3] * 512, DEV)
    with torch.cuda.stream(side):
        got = cu.cpu()
    torch.cuda.synchronize()
    assert got.tolist() == want


def test_device_ints_takes_what_torch_takes():
    """values that are no 32-bit integers convert or fail as torch's do; empty lists, numpy integers and tensors"""
    import numpy as np
    for lists in ([[1.9, -2.9]], [[True, 3]], [[np.int64(7), torch.tensor(5)]], [[], []], [[], [4], []], [[2 ** 31 - 1, -2 ** 31]]):
        for got, values in zip(L.device_ints(lists, DEV), lists):
            assert torch.equal(got.cpu(), torch.tensor(list(values), dtype=torch.int32)) and got.is_cuda
    for bad in (2 ** 31, -2 ** 31 - 1):
        with pytest.raises((RuntimeError, OverflowError)):
            L.device_ints([[bad]], DEV)
