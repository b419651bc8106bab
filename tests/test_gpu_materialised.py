"""Cross-entropy over materialised logits: the target check that runs ahead of
the pass over the logits, and that pass at the row lengths, alignments and
pitches where its vector loops end."""
import pytest
import torch

from mini_trainer_amd import _lib, cross_entropy_none

pytestmark = pytest.mark.gpu


def _case(T, V, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    z = (torch.randn(T, V, generator=g) * 2).to(dtype)
    y = torch.randint(0, V, (T,), generator=g)
    y[1::5] = -100
    return z, y


def _matches(z, y, gpu):
    """Loss and gradient of one call against torch's in fp32 on the CPU.  The
    kernel's lse is that of fp32 sums (2^-20 of a loss of about 10 at most);
    a bf16 result is rounded once (2^-9 of its size, halves of a step apart)."""
    src = z.to(gpu).requires_grad_(True)
    out = cross_entropy_none(src, y.to(gpu))
    out.float().sum().backward()
    ref = z.float().requires_grad_(True)
    want = torch.nn.functional.cross_entropy(ref, y, reduction="none")
    want.sum().backward()
    tol = 1e-5 if z.dtype == torch.float32 else 2.0 ** -8
    torch.testing.assert_close(out.float().cpu(), want.detach(), rtol=tol, atol=1e-5)
    diff = (src.grad.float().cpu() - ref.grad).norm()
    assert float(diff) <= tol * float(ref.grad.norm())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_default_device_is_the_gpu(gpu, dtype):
    """No allocation of the call depends on torch's default device."""
    z, y = _case(70, 1000, dtype)
    with torch.device(gpu):
        out = cross_entropy_none(z.to(gpu), y.to(gpu))
    assert torch.equal(out, cross_entropy_none(z.to(gpu), y.to(gpu)))


@pytest.mark.parametrize("T", [1, 257, 5000])
@pytest.mark.parametrize("where", ["first", "last"])
@pytest.mark.parametrize("value", [-1, -7, "V", 1 << 40])
def test_target_out_of_range(gpu, T, where, value):
    """A target outside [0, V) that is not ignore_index raises IndexError and
    names it; the next call is not affected."""
    V = 333
    z, y = _case(T, V, torch.bfloat16)
    bad = y.clone()
    bad[0 if where == "first" else -1] = V if value == "V" else value
    zd = z.to(gpu)
    with pytest.raises(IndexError, match=f"Target {V if value == 'V' else value} is out of bounds"):
        cross_entropy_none(zd, bad.to(gpu))
    _matches(z, y, gpu)


def test_failed_launch_after_the_check(gpu, monkeypatch):
    """The pass over the logits fails to launch while the check, which writes
    host memory, may still run: the call raises only once that is done."""
    z, y = _case(257, 333, torch.bfloat16)
    zd, yd = z.to(gpu), y.to(gpu)
    waited = []
    sync = torch.cuda.Event.synchronize
    monkeypatch.setattr(torch.cuda.Event, "synchronize", lambda e: (waited.append(1), sync(e))[1])
    monkeypatch.setenv("MT_FLCE_TEST_FAIL_LAUNCH", "ce_forward")
    with pytest.raises(_lib.FlceError, match="injected launch failure"):
        cross_entropy_none(zd, yd)
    assert waited
    monkeypatch.delenv("MT_FLCE_TEST_FAIL_LAUNCH")
    _matches(z, y, gpu)


@pytest.mark.parametrize("dtype,T,V", [
    (torch.float32, 24, 4099),        # one round of four vectors a thread and three columns
    (torch.float32, 24, 12291),       # three rounds and three columns
    (torch.float32, 24, 8192),        # whole rounds, rows aligned
    (torch.bfloat16, 24, 8191),       # every alignment of a row, one column short of a round
    (torch.bfloat16, 24, 8193),
    (torch.bfloat16, 24, 32003),
    (torch.bfloat16, 24, 16384),
    (torch.float32, 5, 1),            # rows shorter than a vector
    (torch.bfloat16, 24, 3),
    (torch.float32, 1000, 64003),     # 256,012,000 bytes: past the caches, odd rows
    (torch.bfloat16, 1000, 128001),   # 256,002,000 bytes: just past them
    (torch.bfloat16, 1000, 127999),   # 255,998,000 bytes: just short of that
])
def test_row_lengths(gpu, dtype, T, V):
    """Labels at a row's first and last columns and in between."""
    z, y = _case(T, V, dtype, seed=V)
    for t, c in enumerate((0, V - 1, min(1, V - 1), V // 2, max(0, V - 2))):
        y[t] = c
    _matches(z, y, gpu)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("ld,ldd", [(0, 0), (0, 1), (1, 0), (3, 2), (8, 16), (0, 5)])
def test_gradient_of_another_pitch(gpu, dtype, ld, ldd):
    """Logits and gradient rows of different pitches: those that start alike
    within 16 bytes, and those that do not; what lies between the gradient's
    rows is untouched."""
    T, V = 24, 8193
    z, y = _case(T, V, dtype, seed=1)
    es = z.element_size()
    code = {torch.float32: _lib.MT_DTYPE_F32, torch.bfloat16: _lib.MT_DTYPE_BF16}[dtype]
    lib, s = _lib.load(), torch.cuda.current_stream(gpu).cuda_stream
    src = torch.full((T, V + ld), float("nan"), dtype=dtype, device=gpu)
    src[:, :V] = z.to(gpu)
    out = torch.full((T, V + ldd), 7.0, dtype=dtype, device=gpu)
    yd, w = y.to(gpu), torch.rand(T, device=gpu)
    loss, lse = torch.empty(T, device=gpu), torch.empty(T, device=gpu)
    _lib.check(lib.mt_ce_forward_checked(src.data_ptr(), T, V, V + ld, code, yd.data_ptr(), -100,
                                         loss.data_ptr(), lse.data_ptr(), s), "ce_forward")
    _lib.check(lib.mt_ce_backward(src.data_ptr(), T, V, V + ld, code, yd.data_ptr(), -100,
                                  lse.data_ptr(), w.data_ptr(), 1, out.data_ptr(), V + ldd, s),
               "ce_backward")
    torch.cuda.synchronize()
    ref = z.double().requires_grad_(True)
    want = torch.nn.functional.cross_entropy(ref, y, reduction="none")
    (want * w.double().cpu()).sum().backward()
    torch.testing.assert_close(loss.double().cpu(), want.detach(), rtol=1e-5, atol=1e-5)
    diff = (out[:, :V].double().cpu() - ref.grad).norm()
    assert float(diff) <= (1e-5 if es == 4 else 2.0 ** -8) * float(ref.grad.norm())
    assert bool((out[:, V:] == 7.0).all())
