"""The two-pass loss forward and the backward at any vocabulary and row alignment (V % 8 != 0, rows
past the row walk's reach), against the fp64 oracle at the edges of their chunks and steps: fewer
logits than a chunk, a lone tail, exact multiples of a step (8 x 256 or 512 logits) and one more or
less, and the borders between 64, 256 and 512 threads and between the two backwards. Bars as in
tests/test_gpu_loss.py; the argmax exact."""

import numpy as np
import pytest
import torch

from aspec_amd.loss import ce_l1_from_logits, cross_entropy
from oracle import loss as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1, 7, 9, 257, 1017, 1024, 1025, 2047, 2049, 4095, 4097, 8191, 8193, 16383, 32769, 40960, 65537, 152063])
def test_any_vocabulary(gpu, vocab):
    rows, trows = 5, 3
    g = torch.Generator(device=gpu).manual_seed(vocab)
    x = (torch.randn(rows, vocab, device=gpu, generator=g) * 3).to(torch.bfloat16)
    y = (torch.randn(trows, vocab, device=gpu, generator=g) * 3).to(torch.bfloat16)
    x[0] += (torch.arange(vocab, device=gpu) * (60.0 / vocab)).to(torch.bfloat16)  # a rising maximum
    x[1] = y[2]                                                                       # identical rows
    x[2, vocab // 2:] = x[2].max()                                                    # tied maxima
    index = torch.tensor([0, 2, 1, 1, 0], device=gpu)
    t = torch.tensor([vocab - 1, 0, vocab // 2, -100, vocab // 3], device=gpu)
    gce, gl1 = torch.randn(rows, device=gpu, generator=g), torch.randn(rows, device=gpu, generator=g)
    xin = x.clone().requires_grad_()
    ce, l1, amax = ce_l1_from_logits(xin, t, y, teacher_indices=index, return_argmax=True)
    ((ce * gce).sum() + (l1 * gl1).sum()).backward()
    xd, yd, td = x.double().cpu().numpy(), y[index].double().cpu().numpy(), t.cpu().numpy()
    np.testing.assert_allclose(ce.detach().double().cpu().numpy(), L.cross_entropy(xd, td), atol=2e-5, rtol=2e-6)
    np.testing.assert_allclose(l1.detach().double().cpu().numpy(), L.l1(xd, yd), atol=2e-6, rtol=2e-6)
    assert l1[1].item() == 0.0
    assert torch.equal(amax.cpu(), torch.as_tensor(np.argmax(xd, axis=-1)))  # the first maximum
    ref = torch.as_tensor(L.cross_entropy_grad(xd, td, gce.double().cpu().numpy())
                          + L.l1_grad(xd, yd, gl1.double().cpu().numpy()))
    assert (xin.grad.double().cpu() - ref).norm() <= 0.01 * ref.norm() + 1e-6
    torch.testing.assert_close(xin.grad.cpu(), ref.to(torch.bfloat16), atol=1e-6, rtol=0.02)
    torch.testing.assert_close(cross_entropy(x, t), ce.detach(), atol=0, rtol=0)


def test_rows_off_alignment(gpu):
    """A 2-byte-aligned view of a vocabulary that is a multiple of eight: the same numbers as the
    aligned copy (which the row walk serves) within its rounding."""
    rows, vocab = 4, 4096
    g = torch.Generator(device=gpu).manual_seed(5)
    flat = torch.randn(1 + rows * vocab, device=gpu, generator=g).to(torch.bfloat16)
    off = flat[1:].view(rows, vocab)
    y = torch.randn(rows, vocab, device=gpu, generator=g).to(torch.bfloat16)
    t = torch.randint(0, vocab, (rows,), device=gpu, generator=g)
    grads = []
    for x in (off, off.clone()):
        xin = x.detach().requires_grad_()
        ce, l1 = ce_l1_from_logits(xin, t, y)
        grads.append((ce.detach(), l1.detach(), torch.autograd.grad(ce.sum() + l1.sum(), xin)[0]))
    assert off.data_ptr() % 16 == 2
    torch.testing.assert_close(grads[0][0], grads[1][0], atol=2e-5, rtol=2e-6)
    torch.testing.assert_close(grads[0][1], grads[1][1], atol=2e-6, rtol=2e-6)
    torch.testing.assert_close(grads[0][2], grads[1][2], atol=1e-6, rtol=0.02)


def _check_against_torch(x, y, t):
    """CE, L1, their gradient and the argmax of the kernels against the fp64 softmax on the CPU, NaN
    for NaN. Bars as above."""
    g = torch.Generator().manual_seed(17)
    w = torch.rand(2, x.shape[0], generator=g)
    xin = x.clone().requires_grad_()
    ce, l1, amax = ce_l1_from_logits(xin, t, y, return_argmax=True)
    (grad,) = torch.autograd.grad((ce, l1), xin, tuple(w.to(x.device)))
    ref = x.double().cpu().requires_grad_()
    ref_ce = torch.nn.functional.cross_entropy(ref, t.cpu(), reduction="none")
    ref_l1 = (ref.softmax(-1) - y.double().cpu().softmax(-1)).abs().sum(-1)
    (ref_grad,) = torch.autograd.grad((ref_ce, ref_l1), ref, tuple(w.double()))
    torch.testing.assert_close(ce.detach().double().cpu(), ref_ce.detach(), atol=2e-5, rtol=2e-6, equal_nan=True)
    torch.testing.assert_close(l1.detach().double().cpu(), ref_l1.detach(), atol=2e-6, rtol=2e-6, equal_nan=True)
    assert torch.equal(amax.cpu(), ref.detach().argmax(-1))
    torch.testing.assert_close(grad.double().cpu(), ref_grad, atol=1e-6, rtol=0.02, equal_nan=True)


@pytest.mark.parametrize("value", [-float("inf"), float("inf"), float("nan")])
@pytest.mark.parametrize("vocab", [2, 7, 9, 2047, 4103, 8193, 16383, 32769, 152063])
def test_nonfinite_tail(gpu, vocab, value):
    """Logits that are not finite among a row's last V % 8, in the draft, the teacher and both; at
    V < 8 that is the whole row but its first."""
    g = torch.Generator(device=gpu).manual_seed(vocab)
    x, y = (torch.randn(6, vocab, device=gpu, generator=g) * 3 for _ in range(2))
    tail = min(vocab % 8, vocab - 1)
    x[0, -1] = y[1, -1] = value
    x[2, -tail:] = y[2, -tail:] = value
    x[3, -tail:] = value
    y[4, -1] = value
    x[4, -tail] = value
    t = torch.zeros(6, dtype=torch.long, device=gpu)
    _check_against_torch(x.to(torch.bfloat16), y.to(torch.bfloat16), t)


@pytest.mark.parametrize("vocab", [7, 4096, 4103, 16000, 16001, 32000, 40960, 40963, 151936])
def test_saturated_rows(gpu, vocab):
    """One token holds all of p and of q to fp32's last digits, so p against q there is rounding: the
    forward's masses and the backward have to take the same side. p (sign(p - q) - E_p[sign]) is then
    at most twice the mass outside that token, V e^-30 (the logit's margin: 40 less six sigma of 1.5,
    rounded up)."""
    rows = 256
    g = torch.Generator(device=gpu).manual_seed(vocab)
    x, y = (torch.randn(rows, vocab, device=gpu, generator=g) * 1.5 for _ in range(2))
    at = torch.randint(0, vocab, (rows, 1), device=gpu, generator=g)
    for z in (x, y):
        z.scatter_(1, at, 40 + 30 * torch.rand(rows, 1, device=gpu, generator=g))
    xin = x.to(torch.bfloat16).requires_grad_()
    _, l1 = ce_l1_from_logits(xin, at[:, 0], y.to(torch.bfloat16))
    (grad,) = torch.autograd.grad(l1.sum(), xin)
    assert grad.abs().max() <= 2 * vocab * np.exp(-30.0)


@pytest.mark.parametrize("value", [-1e9, -1e10, -1e20, -1e30, torch.finfo(torch.bfloat16).min])
@pytest.mark.parametrize("vocab", [2048, 2055, 4096, 8191, 8192, 8193, 16000, 16383, 32000, 40960, 152063])
def test_large_finite_masks(gpu, vocab, value):
    """Runs of logits masked with a large finite value at the start, the middle and the end of a row,
    of a chunk's length and of most of the row, in the draft, the teacher and both."""
    g = torch.Generator(device=gpu).manual_seed(vocab)
    x, y = (torch.randn(9, vocab, device=gpu, generator=g) * 3 for _ in range(2))
    mid, most = vocab // 16 * 8, vocab // 64 * 56
    x[0, :8] = y[1, :8] = value
    x[2, mid:mid + 64] = y[3, mid:mid + 64] = value
    x[4, -9:] = y[5, -9:] = value
    x[6, :most] = y[6, :most] = value
    x[7, vocab - most:] = value
    y[8, 8:] = value
    t = torch.full((9,), vocab // 2, device=gpu)
    t[2], t[6], t[7], t[4] = 3, vocab - 1, 0, 1
    _check_against_torch(x.to(torch.bfloat16), y.to(torch.bfloat16), t)
