"""Valid-row compaction around the edges of its workgroups (4096 labels)."""
import pytest
import torch

from mini_trainer_amd import _lib
from mini_trainer_amd.flce import _p, _stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("T", [1, 63, 4095, 4096, 4097, 12288, 70001])
@pytest.mark.parametrize("mask", [0.0, 0.4, 1.0])
def test_compaction_matches_torch(gpu, T, mask, shift):
    V = 1000
    g = torch.Generator().manual_seed(T)
    y = torch.randint(0, V, (T,), generator=g)
    y[torch.rand(T, generator=g) < mask] = -100
    bad = sorted({T // 3, T - 1}) if T > 64 and mask == 0.4 else []
    for i, t in enumerate(bad):
        y[t] = V + 5 if i else -7
    src = torch.cat([y[1:], torch.tensor([-100])]) if shift else y
    ok = (src >= 0) & (src < V)
    wrong = (src != -100) & ~ok
    want = torch.nonzero(ok).flatten().int()
    yd = y.to(gpu)
    ri, rl = (torch.full((T,), -1, dtype=torch.int32, device=gpu) for _ in range(2))
    counts = torch.empty(4, dtype=torch.int32, device=gpu)
    _lib.check(_lib.load().mt_flce_prepare(_p(yd), T, V, -100, shift, _p(ri), _p(rl), _p(counts),
                                           _stream(gpu)), "prepare")
    n = int(ok.sum())
    first = int(torch.nonzero(wrong)[0]) if wrong.any() else -1
    assert counts.tolist() == [n, int(wrong.sum()), first, 0]
    assert torch.equal(ri[:n].cpu(), want) and torch.equal(rl[:n].cpu(), src[ok].int())
    assert torch.equal(ri[n:].cpu(), torch.nonzero(~ok).flatten().int().flip(0))


@pytest.mark.parametrize("T,shift", [
    (1 << 20, 0),                # 256 workgroups of 4096 labels
    ((1 << 20) + 1, 1),          # two 4096s each, the last workgroup with one
    (3 * (1 << 20) - 4097, 0),   # three each, a last one that ends within its second
])
def test_compaction_of_several_chunks_per_workgroup(gpu, T, shift):
    test_compaction_matches_torch(gpu, T, 0.4, shift)
