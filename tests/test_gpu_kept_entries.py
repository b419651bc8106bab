"""The two C entries of the kept-logits path on buffers of exactly the sizes
they ask for."""
import pytest
import torch

from mini_trainer_amd import _lib, prepare_targets
from mini_trainer_amd.flce import _p, _stream, profile_enable, profile_report

from test_gpu_canary import Guarded, matrix, pad_intact

pytestmark = pytest.mark.gpu


def _al(b):
    return -(-b // 256) * 256


def _scratch(n, H, blocks, slices, acc):
    """Bytes of mt_flce_backward_logits' scratch: X^T, the work queue and dX's
    planes, or one slice's accumulator (tiles, rows with an accumulator)."""
    C = _al(n)
    planes = slices * C * H * 4 if slices > 1 or (blocks and acc) else \
        C // 256 * -(-H // 256) * 65536 * 4 if blocks else 0
    return _al(H * C * 2) + 256 + _al(planes)


def _call(gpu, T, H, V, cols, slices, acc):
    """Forward and backward through the entries; every buffer between guards,
    dX and the accumulator with wider rows.  Returns (dX, dW) after checking
    the guards."""
    lib, s = _lib.load(), _stream(gpu)
    g = torch.Generator(device=gpu).manual_seed(T + H)
    X = torch.randn(T, H, device=gpu, generator=g).bfloat16()
    W = (torch.randn(V, H, device=gpu, generator=g) * 0.05).bfloat16()
    y = torch.randint(0, V, (T,), device=gpu, generator=g)
    y[::7] = -100
    ri, rl, n = prepare_targets(y, V)
    lb, sb = _al(n) * cols * 2, _scratch(n, H, cols < V, slices, acc)
    wsb = lib.mt_flce_forward_workspace_bytes(T, n, H, V, _lib.MT_DTYPE_BF16)
    bufs = loss, lse, ws, kept, scratch = [Guarded(gpu, b) for b in (T * 4, n * 4, wsb, lb, sb)]
    _lib.check(lib.mt_flce_forward_logits(_p(X), _p(W), T, H, V, H, H, _lib.MT_DTYPE_BF16, 0.0,
                                          _p(ri), _p(rl), n, loss.ptr, lse.ptr, ws.ptr, wsb,
                                          kept.ptr, cols, lb, s), "forward_logits")
    torch.cuda.synchronize()
    assert all(b.intact() for b in bufs)
    grad = torch.rand(T, device=gpu, generator=g)
    gdx, dX = matrix(gpu, T, H, H + 8, torch.bfloat16)
    gdw, dW = matrix(gpu, V, H, H + (4 if acc else 0), torch.float32 if acc else torch.bfloat16)
    dW[:, :H] = 0
    _lib.check(lib.mt_flce_backward_logits(_p(X), _p(W), T, H, V, H, H, _lib.MT_DTYPE_BF16, 0.0,
                                           _p(ri), _p(rl), n, lse.ptr, _p(grad), 1, gdx.ptr, H + 8,
                                           None if acc else gdw.ptr, V * H * 2,
                                           gdw.ptr if acc else None, H + 4 if acc else 0, kept.ptr,
                                           cols, lb, scratch.ptr, sb, s), "backward_logits")
    torch.cuda.synchronize()
    assert all(b.intact() for b in bufs + [gdx, gdw])
    assert pad_intact(dX, H) and pad_intact(dW, H)
    # fp32 products of the same roundings, as in the torch path
    z = (X.double() @ W.double().t()).bfloat16().double()
    ok = y != -100
    G = torch.softmax(z, 1)
    G[torch.arange(T, device=gpu)[ok], y[ok]] -= 1
    G = (G * (grad * ok).double()[:, None])
    return dX[:, :H].double(), dW[:, :H].double(), G @ W.double(), G.t() @ X.double()


@pytest.mark.parametrize("H,slices", [(64, 1), (64, 8), (128, 1), (128, 4)])
def test_slices_are_those_of_the_scratch(gpu, monkeypatch, H, slices):
    """One slice keeps its accumulator as 256-column tiles, which at H = 64 is
    the size of four planes: the launch runs the one slice all the same."""
    monkeypatch.setenv("MT_FLCE_SPLIT_PHASE", "1")  # (names dX's launches)
    profile_enable(True)
    try:
        dX, dW, rdX, rdW = _call(gpu, 300, H, 5000, 2304, slices, False)
    finally:
        profile_enable(False)
    rep = profile_report()
    assert ("dx_bf16_kernel<store_tiles>" in rep) == (slices == 1)
    assert ("dx_bf16_kernel<split>" in rep) == (slices > 1)
    assert float((dX - rdX).norm()) <= 1e-2 * float(rdX.norm())
    assert float((dW - rdW).norm()) <= 1e-2 * float(rdW.norm())


@pytest.mark.parametrize("T,H,V,cols,slices,acc", [
    (3, 8, 1, 256, 1, False),           # the smallest: one row tile, one column
    (700, 200, 1300, 1536, 1, False),   # all kept, tails in every dimension
    (700, 200, 1300, 1536, 4, False),   # the same with dX slices
    (700, 200, 1300, 1536, 4, True),
    (300, 136, 5000, 1024, 1, False),   # blocks, a short last one
    (300, 136, 5000, 1024, 1, True),
    (520, 264, 12500, 6144, 8, False),  # a last block (212 columns) with fewer stages than slices
    (520, 264, 12500, 6144, 8, True),
    (511, 16, 5000, 2304, 8, False),    # slices' planes smaller than one slice's tiles
    (511, 16, 5000, 512, 2, False),
])
def test_guards_and_results(gpu, T, H, V, cols, slices, acc):
    """Against the same roundings of the logits in 64 bits: G is rounded to
    bf16 (2^-9 of each entry), so is a bf16 result."""
    dX, dW, rdX, rdW = _call(gpu, T, H, V, cols, slices, acc)
    assert float((dX - rdX).norm()) <= 2.0 ** -8 * float(rdX.norm())
    assert float((dW - rdW).norm()) <= 2.0 ** -8 * float(rdW.norm())
