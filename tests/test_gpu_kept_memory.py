"""Memory of the path that keeps logits from the forward to the backward: the
logits are a saved tensor like any activation, released at the first backward,
and the call's peak is what the plan says."""
import pytest
import torch
from torch.utils.checkpoint import checkpoint

from mini_trainer_amd import fused_linear_cross_entropy
from mini_trainer_amd.flce import _kept_plan

pytestmark = pytest.mark.gpu

T, H, V = 1024, 512, 32000


@pytest.fixture
def case(gpu):
    g = torch.Generator(device=gpu).manual_seed(3)
    X = torch.randn(T, H, generator=g, device=gpu).bfloat16().requires_grad_(True)
    W = (torch.randn(V, H, generator=g, device=gpu) * 0.05).bfloat16().requires_grad_(True)
    y = torch.randint(0, V, (T,), generator=g, device=gpu)
    cols, logits, scratch, pays = _kept_plan(T, T, H, V)
    assert pays and cols == V and logits == T * V * 2
    loss = fused_linear_cross_entropy(X, W, y)  # (library and allocator set up)
    loss.sum().backward()
    want = X.grad, W.grad
    X.grad = W.grad = None
    return X, W, y, want, logits, scratch


def _held(f):
    """f()'s result and the bytes it left allocated."""
    before = torch.cuda.memory_allocated()
    out = f()
    return out, torch.cuda.memory_allocated() - before


@pytest.mark.parametrize("how", ["plain", "offload", "checkpoint"])
def test_saved_like_an_activation(gpu, case, how):
    """Offloading saved tensors, or recomputing them in the backward
    (checkpointing), leaves no logits on the GPU after the forward; the
    gradients are the same bits."""
    X, W, y, want, logits, _ = case

    def forward():
        if how == "offload":
            with torch.autograd.graph.save_on_cpu():
                return fused_linear_cross_entropy(X, W, y)
        if how == "checkpoint":
            return checkpoint(fused_linear_cross_entropy, X, W, y, use_reentrant=False)
        return fused_linear_cross_entropy(X, W, y)

    loss, held = _held(forward)
    assert held >= logits if how == "plain" else held < logits // 4
    loss.sum().backward()
    assert torch.equal(X.grad, want[0]) and torch.equal(W.grad, want[1])


def test_released_by_the_first_backward(gpu, case):
    X, W, y, want, logits, _ = case
    loss, held = _held(lambda: fused_linear_cross_entropy(X, W, y))
    assert held >= logits
    _, left = _held(lambda: loss.sum().backward(retain_graph=True))
    assert left <= (T + V) * H * 2 + (4 << 20) - logits
    X.grad = W.grad = None
    loss.sum().backward()  # recomputes: the kept logits are gone
    for a, b in ((X.grad, want[0]), (W.grad, want[1])):
        assert float((a.float() - b.float()).norm()) <= 2.0 ** -8 * float(b.float().norm())


def test_peak_is_the_plans(gpu, case):
    """Logits, the backward's scratch and the bf16 outputs; 1 MiB for loss,
    lse, row lists and the like, and up to 1 MiB with each of the three large
    blocks (the allocator does not split off less than that)."""
    X, W, y, _, logits, scratch = case
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    fused_linear_cross_entropy(X, W, y).sum().backward()
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - base <= \
        logits + scratch + (T + V) * H * 2 + (4 << 20)


@pytest.fixture
def memory_limit():
    """limit(slack): from now on the allocator has `slack` bytes left (what lies
    free between its blocks is taken up, to a MiB); limit(None) lifts that."""
    total = torch.cuda.get_device_properties(0).total_memory
    taken = []

    def limit(slack):
        taken.clear()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        if slack is None:
            torch.cuda.set_per_process_memory_fraction(1.0)
            return
        reserved = torch.cuda.memory_reserved()
        torch.cuda.set_per_process_memory_fraction(reserved / total)
        size = 1 << 30
        while size >= 1 << 20:
            try:
                taken.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:
                size //= 2
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + slack) / total)

    yield limit
    limit(None)


@pytest.mark.parametrize("short,accumulator,T,V", [
    ("forward", False, 4096, 64000),
    ("forward", True, 2048, 32000),
    ("backward", False, 4096, 64000),
])
def test_recomputes_where_the_room_is_short(gpu, memory_limit, short, accumulator, T, V):
    """No room for the logits at the forward, or for the backward's buffers
    beside them: the call recomputes instead of raising.  Bound: the roundings
    of the two backwards differ by 2^-8 at most (test_gpu_kept_logits)."""
    H = 4096
    g = torch.Generator(device=gpu).manual_seed(4)
    X = torch.randn(T, H, generator=g, device=gpu).bfloat16().requires_grad_(True)
    W = (torch.randn(V, H, generator=g, device=gpu) * 0.02).bfloat16().requires_grad_(True)
    y = torch.randint(0, V, (T,), generator=g, device=gpu)
    cols, logits, scratch, _ = _kept_plan(T, T, H, V, accumulator)
    accs = [torch.zeros(V, H, device=gpu) if accumulator else None for _ in range(2)]

    def run(acc, before_forward, before_backward):
        X.grad = W.grad = None
        before_forward()
        loss = fused_linear_cross_entropy(X, W, y, dw_accumulator=acc)
        kept = loss.grad_fn.logits is not None
        before_backward()
        loss.sum().backward()
        memory_limit(None)
        return kept, loss.detach(), X.grad, W.grad if acc is None else acc

    kept, *want = run(accs[0], lambda: None, lambda: None)
    assert kept and cols == V
    outputs = T * H * 2 + (0 if accumulator else V * H * 2)
    if short == "forward":
        kept, *got = run(accs[1], lambda: memory_limit(logits - (16 << 20)),
                         lambda: memory_limit(None))
        assert not kept
    else:
        kept, *got = run(accs[1], lambda: None,
                         lambda: memory_limit(outputs + scratch - (4 << 20)))
        assert kept
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:], want[1:]):
        assert float((a.float() - b.float()).norm()) <= 2.0 ** -8 * float(b.float().norm())
