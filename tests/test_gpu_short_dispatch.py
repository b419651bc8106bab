"""The paths of short calls and small vocabularies, which the least workspace
(flce.MIN_BUDGET) decides."""
import pytest
import torch

from mini_trainer_amd import fused_linear_cross_entropy, path_of
from mini_trainer_amd.flce import _general_pays, _kept_plan, fused_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grad_scale,path", [(None, "general"), (0.25, "fused")])
def test_small_vocabulary(gpu, grad_scale, path):
    """5% of these logits holds 256 rows of exponentials: without a promise
    the general path runs in the least workspace, with one the fused path runs
    in chunks that fit it.  Against torch in fp32 with the logits rounded to
    bf16: loss and gradients carry at most three roundings of 2^-9."""
    T, n, H, V = 11217, 10350, 760, 10337
    assert not _kept_plan(T, n, H, V)[3] and _general_pays(T, n, H, V)
    assert fused_plan(T, n, H, V)[0] == 256 and fused_plan(T, n, H, V, 192 << 20)[0] > 256
    g = torch.Generator(device=gpu).manual_seed(1)
    X = torch.randn(T, H, device=gpu, generator=g).bfloat16().requires_grad_(True)
    W = (torch.randn(V, H, device=gpu, generator=g) * 0.05).bfloat16().requires_grad_(True)
    y = torch.randint(0, V, (T,), device=gpu, generator=g)
    y[:T - n] = -100
    loss = fused_linear_cross_entropy(X, W, y, grad_scale=grad_scale)
    assert path_of(loss) == path
    (loss.sum() * 0.25).backward()
    x, w = X.detach().float().requires_grad_(True), W.detach().float().requires_grad_(True)
    z = x @ w.t()
    z = z + (z.detach().bfloat16().float() - z.detach())
    ref = torch.nn.functional.cross_entropy(z, y, reduction="none")
    (ref.sum() * 0.25).backward()
    assert float((loss - ref).detach().abs().max()) <= 1e-4
    for a, b in ((X.grad, x.grad), (W.grad, w.grad)):
        assert float((a.float() - b).norm()) <= 3 * 2.0 ** -9 * float(b.norm())
