"""A bf16 weight that is a column slice of a wider matrix: its rows, gaps
included, lie beyond one buffer's reach (lowered by the test hook) while the
same rows without gaps would not."""
import pytest
import torch

from mini_trainer_amd import fused_linear_cross_entropy
from mini_trainer_amd.flce import FUSED_ENV

from test_gpu_parity import check_parity, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["unit", "accumulator", "promise", "frozen"])
@pytest.mark.parametrize("fused", ["auto", "1", "0"])
def test_strided_weight_beyond_one_buffer(gpu, monkeypatch, fused, how):
    """Parity bounds as for a contiguous weight (check_parity)."""
    T, H, V = 200, 136, 5000
    print(f"case weight pitch {fused} {how}", flush=True)
    monkeypatch.setenv(FUSED_ENV, fused)
    monkeypatch.setenv("MT_FLCE_MAX_BUFFER_BYTES", str(3 << 20))
    assert V * H * 2 < 3 << 20 < V * 4 * H * 2
    X, W, y = make_case(T, H, V, torch.bfloat16, seed=5)
    wide = torch.full((V, 4 * H), float("nan"), dtype=torch.bfloat16, device=gpu)
    wide[:, H:2 * H] = W.to(gpu)
    w = wide[:, H:2 * H].detach().requires_grad_(how != "frozen")
    x = X.to(gpu).requires_grad_(True)
    n = int((y != -100).sum())
    acc = torch.zeros(V, H, device=gpu) if how in ("accumulator", "promise") else None
    loss = fused_linear_cross_entropy(x, w, y.to(gpu), dw_accumulator=acc,
                                      grad_scale=1.0 / n if how == "promise" else None)
    (loss.sum() / n).backward()
    torch.cuda.synchronize()
    if how == "frozen":
        assert w.grad is None
        w2 = W.to(gpu).requires_grad_(True)
        loss2 = fused_linear_cross_entropy(X.to(gpu), w2, y.to(gpu))
        (loss2.sum() / n).backward()
        dW = w2.grad
    else:
        dW = w.grad if acc is None else acc
    check_parity(X, W, y, loss.detach().cpu(), x.grad.cpu(), dW.float().cpu(),
                 grad=torch.full((T,), 1.0 / n))
