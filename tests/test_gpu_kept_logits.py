"""The path that keeps logits from the forward to the backward, at the
sizes where a tile, a K stage or a dX slice ends: loss and gradients equal the
recomputing general path's (same roundings: the loss bit for bit, the
gradients up to the order of fp32 sums), also for a per-token gradient, a
second backward and logits far outside the exponentials' range."""
import pytest
import torch

from mini_trainer_amd import fused_linear_cross_entropy, path_of
from mini_trainer_amd.flce import FUSED_ENV, profile_enable, profile_report

pytestmark = pytest.mark.gpu


def _inputs(T, H, V, mask, shift=0.0):
    g = torch.Generator().manual_seed(T * 31 + H + V)
    X = torch.randn(T, H, generator=g)
    W = torch.randn(V, H, generator=g) * (1.3 / H ** 0.5)
    if shift:
        X[:, 0], W[:, 0] = shift, 1.0
    y = torch.randint(0, V, (T,), generator=g)
    y[torch.rand(T, generator=g) < mask] = -100
    return X.to(torch.bfloat16), W.to(torch.bfloat16), y, torch.rand(T, generator=g) + 0.5


def _chain(gpu, X, W, y, grad, cap):
    """Loss and the gradients of two backwards through it: the first from the
    kept logits, the second (they are G by then) by recomputing."""
    Xd, Wd = X.to(gpu).requires_grad_(True), W.to(gpu).requires_grad_(True)
    loss = fused_linear_cross_entropy(Xd, Wd, y.to(gpu), softcap=cap or None)
    out = []
    for k in range(2):
        Xd.grad = Wd.grad = None
        if grad is None:
            (loss.sum() * 0.37).backward(retain_graph=k == 0)
        else:
            loss.backward(grad.to(gpu), retain_graph=k == 0)
        out.append((Xd.grad, Wd.grad))
    return loss, out


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


def _budget(n, H, V, cols, slices):
    """Budget bytes under which the plan keeps `cols` columns with `slices`
    dX slices (1: the tiled accumulator)."""
    C, al = -(-n // 256) * 256, lambda b: -(-b // 256) * 256  # noqa: E731
    acc = slices * C * H * 4 if slices > 1 else C // 256 * -(-H // 256) * 65536 * 4
    return C * cols * 2 + al(H * C * 2) + 256 + al(acc)


@pytest.mark.parametrize("per_token", [False, True])
@pytest.mark.parametrize("T,H,V,mask,cap,shift,cols,slices", [
    (3, 64, 700, 0.0, 0.0, 0.0, 0, 0),          # one partial row tile, several dX slices
    (256, 256, 1024, 0.0, 0.0, 0.0, 0, 0),      # whole tiles
    (257, 264, 1025, 0.1, 0.0, 0.0, 0, 0),      # one row, one column, one K chunk over
    (300, 520, 40000, 0.2, 30.0, 0.0, 0, 0),    # more vocabulary tiles than CUs, softcap
    (700, 1024, 66000, 0.3, 0.0, 0.0, 0, 0),    # the dW work queue
    (130, 128, 600, 0.0, 0.0, 60.0, 0, 0),      # logits near 60: past the range of exp in bf16
    (300, 136, 5000, 0.1, 0.0, 0.0, 1024, 1),   # blocks after the kept one, a short last one
    (300, 136, 5000, 0.1, 0.0, 0.0, 2048, 8),   # the same with dX slices in planes
    (520, 264, 12500, 0.2, 20.0, 0.0, 6144, 8),  # a last block with fewer columns than its slices
])
def test_kept_logits_equal_recompute(gpu, monkeypatch, T, H, V, mask, cap, shift, cols, slices,
                                     per_token):
    """Bound, against the recomputing backward: a per-token gradient gives the
    same G on both, rounded to bf16 and summed in fp32 in another order
    (differences of sqrt(V) 2^-24), and the result is rounded to bf16 once: a
    value near a rounding boundary moves by one step, 2^-8 of itself at most,
    in well below one value in 64: 2^-11.  One scalar is applied after the
    sums here and before G's rounding there (2^-9 of each G at most, the
    scalar's own rounding alike in every G): 2^-8."""
    from mini_trainer_amd.flce import BACKWARD_BUDGET_ENV, _kept_plan

    X, W, y, grad = _inputs(T, H, V, mask, shift)
    grad = grad if per_token else None
    n = int((y != -100).sum())
    if cols:
        monkeypatch.setenv(BACKWARD_BUDGET_ENV, str(_budget(n, H, V, cols, slices)))
        kept = _kept_plan(T, n, H, V)
        assert 0 < kept[0] < V
        monkeypatch.setattr("mini_trainer_amd.flce._kept_plan", lambda *a: kept[:3] + (True,))
    profile_enable(True)
    try:
        loss, ((dX, dW), (dX0, dW0)) = _chain(gpu, X, W, y, grad, cap)
        torch.cuda.synchronize()
    finally:
        profile_enable(False)
    rep = profile_report()
    assert "fwd_bf16_kernel<store_logits>" in rep and path_of(loss) == "general"
    assert "recompute_bf16_kernel" in rep
    monkeypatch.setenv(FUSED_ENV, "0")
    assert torch.equal(loss, fused_linear_cross_entropy(X.to(gpu), W.to(gpu), y.to(gpu),
                                                        softcap=cap or None))
    assert dW.untyped_storage().nbytes() == V * H * 2
    bound = 2.0 ** (-11 if per_token else -8)
    assert _rel(dX, dX0) <= bound and _rel(dW, dW0) <= bound
    masked = (y == -100).to(gpu)
    assert torch.count_nonzero(dX[masked]) == 0


def test_kept_logits_host_checks():
    """The plan: 0 beyond the budget, and with the gradient's bytes counted
    the whole thing within 5% of the logits plus those bytes."""
    from mini_trainer_amd.flce import _kept_plan

    for T, n, H, V in ((16384, 6554, 8192, 128256), (4096, 2868, 4096, 128256), (192, 134, 128, 1000)):
        cols, lb, sb, pays = _kept_plan(T, n, H, V)
        Hp, vt = -(-H // 256) * 256, -(-V // 256)
        room = Hp * 512 + vt * 256 * Hp * 4 - V * H * 2
        assert pays and cols == vt * 256 and lb >= -(-n // 256) * 256 * cols * 2
        assert lb + sb <= max(0.05 * T * V * 2, 192 << 20) + room + 512
    cols, _, _, pays = _kept_plan(65536, 45875, 4096, 128256)
    assert cols < 128256 and not pays


@pytest.mark.parametrize("T,H,V,cols,slices", [
    (3, 64, 700, 0, 0),           # all kept, several dX slices
    (700, 520, 5000, 0, 0),
    (700, 1024, 66000, 0, 0),     # the dW work queue
    (300, 136, 5000, 1024, 1),    # blocks after the kept one, one dX accumulator
    (520, 264, 12500, 6144, 8),   # the same with dX slices in planes
])
def test_kept_logits_into_accumulator(gpu, monkeypatch, T, H, V, cols, slices):
    """dW added into an fp32 accumulator that holds other values already,
    against the recomputing backward into an empty one: the same G in both, so
    only the order of the fp32 sums differs (sqrt(V) 2^-24 of dX before its
    rounding, at most 2^-11 after; sqrt(T) 2^-24 of dW, 2^-18)."""
    import mini_trainer_amd.flce as flce

    X, W, y, grad = _inputs(T, H, V, 0.1)
    n = int((y != -100).sum())
    if cols:
        C, al = -(-n // 256) * 256, lambda b: -(-b // 256) * 256  # noqa: E731
        monkeypatch.setenv(flce.BACKWARD_BUDGET_ENV,
                           str(C * cols * 2 + al(H * C * 2) + 256 + al(slices * C * H * 4)))
    kept = flce._kept_plan(T, n, H, V, True)
    assert kept[0] >= V if not cols else 0 < kept[0] < V
    plan = flce._kept_plan
    start = torch.randn(V, H, generator=torch.Generator().manual_seed(1)).to(gpu)

    def run(keep, acc):
        monkeypatch.setattr(flce, "_kept_plan", lambda *a: plan(*a)[:3] + (keep,))
        Xd, Wd = X.to(gpu).requires_grad_(True), W.to(gpu).requires_grad_(True)
        loss = fused_linear_cross_entropy(Xd, Wd, y.to(gpu), dw_accumulator=acc)
        (loss * grad.to(gpu)).sum().backward()
        assert Wd.grad is None
        return loss, Xd.grad

    acc, acc0 = start.clone(), torch.zeros(V, H, device=gpu)
    profile_enable(True)
    try:
        loss, dX = run(True, acc)
        torch.cuda.synchronize()
    finally:
        profile_enable(False)
    rep = profile_report()
    assert "fwd_bf16_kernel<store_logits>" in rep
    assert ("recompute_bf16_kernel" in rep) == bool(cols)
    loss0, dX0 = run(False, acc0)
    assert torch.equal(loss, loss0)
    assert _rel(dX, dX0) <= 2.0 ** -11
    # acc - start loses 2^-24 of the start's size
    assert float(((acc.double() - start.double()) - acc0.double()).norm()) <= \
        2.0 ** -18 * float(acc0.double().norm()) + 2.0 ** -24 * float(start.double().norm())
