"""A hidden size that is not whole K stages: the chunks past it come from
beyond the buffer's end as zeros, whatever lies behind a row."""
import pytest
import torch

from mini_trainer_amd import fused_linear_cross_entropy
from mini_trainer_amd.flce import FUSED_ENV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", ["auto", "0", "1"])
@pytest.mark.parametrize("H", [8, 56, 72, 136, 1000])
def test_nan_behind_the_rows(gpu, monkeypatch, H, fused):
    """Rows inside a wider buffer whose gaps hold NaN give the same bits as
    contiguous rows (the last row has nothing but the buffer's end behind it),
    and these match the torch path in fp32: logits of |z| <= 8 rounded to bf16
    are 2^-9 * 8 off, so is the loss, gradients carry three such roundings."""
    monkeypatch.setenv(FUSED_ENV, fused)
    T, V = 300, 1100
    g = torch.Generator().manual_seed(H)
    X = torch.randn(T, H, generator=g).bfloat16()
    W = (torch.randn(V, H, generator=g) / H ** 0.5).bfloat16()
    y = torch.randint(0, V, (T,), generator=g).to(gpu)

    def run(pad):
        def put(a):
            buf = torch.full((a.shape[0], H + pad), float("nan"), dtype=a.dtype, device=gpu)
            buf[:, :H] = a.to(gpu)
            return buf[:, :H].detach().requires_grad_(True)
        x, w = put(X), put(W)
        loss = fused_linear_cross_entropy(x, w, y)
        loss.sum().backward()
        return loss.detach(), x.grad, w.grad

    loss, dX, dW = run(0)
    for a, b in zip((loss, dX, dW), run(24)):
        assert torch.equal(a, b)
    x, w = X.float().to(gpu).requires_grad_(True), W.float().to(gpu).requires_grad_(True)
    ref = torch.nn.functional.cross_entropy(x @ w.T, y, reduction="none")
    ref.sum().backward()
    assert float((loss - ref.detach()).abs().max()) <= 2.0 ** -6
    for a, b in ((dX, x.grad), (dW, w.grad)):
        assert float((a.float() - b).norm() / b.norm()) <= 3 * 2.0 ** -8
