"""Batch normalisation (+ ReLU) kernels of include/phx_bn.h against torch's batch_norm evaluated in fp64 on
the CPU from the same (fp16- or fp32-rounded) inputs: output, saved and running statistics, input gradient
and parameter gradients.  Tolerance: 1e-4 (fp32 tensors) / 4e-3 (fp16 tensors, whose outputs are rounded to
fp16) of the largest reference magnitude."""
import numpy as np
import pytest
import torch

import phoenix_core_amd as phx

pytestmark = pytest.mark.gpu

SHAPES = [(8, 16, 14, 14), (12, 5, 7, 7), (3, 130, 1, 1), (64, 33, 9, 5), (1, 4, 3, 3), (256, 16, 28, 28), (40, 512, 7, 7)]


def close(got, want, tol, what):
    got = got.detach().double().cpu()
    err = (got - want).abs().max().item()
    assert torch.isfinite(got).all(), what
    assert err <= tol * max(want.abs().max().item(), 1e-6), "%s: abs err %.3e of max %.3e" % (what, err, want.abs().max().item())


@pytest.mark.parametrize("relu,residual", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_batch_norm_matches_torch(shape, dtype, relu, residual):
    print("shape", shape, dtype, relu, residual, flush=True)
    gen = torch.Generator().manual_seed(sum(shape))
    c = shape[1]
    x = (torch.randn(shape, generator=gen) * 1.5 + 0.3).to(dtype)
    dy = torch.randn(shape, generator=gen).to(dtype)
    gamma = torch.rand(c, generator=gen) + 0.5
    beta = torch.randn(c, generator=gen) * 0.3
    mod = phx.QBatchNorm2d(c, relu=relu).cuda().train()
    with torch.no_grad():
        mod.weight.copy_(gamma)
        mod.bias.copy_(beta)
    res = (torch.randn(shape, generator=gen) * 0.7).to(dtype) if residual else None
    if relu:
        # The gradient of the ReLU jumps at zero: an element whose pre-activation is zero to rounding error gets its
        # gradient in one precision and not in the other.  Those elements carry no output gradient here.
        with torch.no_grad():
            z = torch.nn.functional.batch_norm(x.double(), None, None, gamma.double(), beta.double(), True, 0.1, 1e-5)
            if residual:
                z = z + res.double()
            dy[z.abs() < (1e-4 if dtype == torch.float32 else 2e-2)] = 0
    xd = x.cuda().requires_grad_(True)
    rd = res.cuda().requires_grad_(True) if residual else None
    y = mod(xd, rd) if residual else mod(xd)
    y.backward(dy.cuda())

    x64 = x.double().requires_grad_(True)
    g64, b64 = gamma.double().requires_grad_(True), beta.double().requires_grad_(True)
    rm, rv = torch.zeros(c, dtype=torch.float64), torch.ones(c, dtype=torch.float64)
    ref = torch.nn.functional.batch_norm(x64, rm, rv, g64, b64, True, 0.1, 1e-5)
    r64 = res.double().requires_grad_(True) if residual else None
    if residual:
        ref = ref + r64
    if relu:
        ref = torch.relu(ref)
    ref.backward(dy.double())
    tol = 1e-4 if dtype == torch.float32 else 4e-3
    assert y.dtype == dtype and y.shape == tuple(shape)
    close(y, ref.detach(), tol, "y")
    close(xd.grad, x64.grad, tol, "dx")
    if residual:
        close(rd.grad, r64.grad, tol, "dresidual")
    close(mod.weight.grad, g64.grad, tol, "dgamma")
    close(mod.bias.grad, b64.grad, tol, "dbeta")
    close(mod.running_mean, rm, 1e-4, "running mean")
    close(mod.running_var, rv, 1e-4, "running var")


def test_eval_mode_uses_running_statistics():
    mod = phx.QBatchNorm2d(6, relu=True).cuda()
    x = torch.randn(8, 6, 5, 5, device="cuda")
    mod.train()
    mod(x)
    mod.eval()
    y = mod(x)
    want = torch.relu(torch.nn.functional.batch_norm(x, mod.running_mean, mod.running_var, mod.weight, mod.bias, False, 0.0,
                                                     mod.eps))
    assert torch.allclose(y, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_statistics_of_a_channel_with_a_large_mean(dtype):
    """Channels whose mean is ~1000 times their spread (fp32) / ~100 times (fp16): E[x^2] - E[x]^2 in fp32 would
    lose every significant bit of the variance; the kernels sum around a shift inside the data's range instead.
    Saved inverse standard deviation, running variance and the normalised output against fp64."""
    gen = torch.Generator().manual_seed(77)
    shape = (32, 6, 12, 12)
    big = 1000.0 if dtype == torch.float32 else 100.0
    offsets = torch.tensor([big, -big, 0.0, 3 * big, big, -2 * big]).view(1, 6, 1, 1)
    x = (torch.randn(shape, generator=gen) + offsets).to(dtype)
    mod = phx.QBatchNorm2d(6, relu=False).cuda().train()
    y = mod(x.cuda())
    x64 = x.double()
    var = x64.var(dim=(0, 2, 3), unbiased=False)
    want = (x64 - x64.mean(dim=(0, 2, 3), keepdim=True)) / (var.view(1, 6, 1, 1) + 1e-5).sqrt()
    n = shape[0] * shape[2] * shape[3]
    close(mod.running_var, 0.9 + 0.1 * var * n / (n - 1), 1e-3, "running var")
    close(y, want, 1e-3 if dtype == torch.float32 else 4e-3, "y")


@pytest.mark.parametrize("relu,residual", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (3, 130, 1, 1), (5, 7, 1, 3), (4, 6, 2, 3), (9, 33, 7, 1), (2, 3, 2, 4),
                                   (12, 65, 7, 7), (1, 2, 64, 32), (3, 5, 45, 91)], ids=lambda s: "x".join(map(str, s)))
def test_evaluation_pass(shape, dtype, relu, residual):
    """The one-pass evaluation kernel at the edges of its runs (planes smaller than a 16-byte chunk, of exactly one, of
    a whole run; a ragged end) against fp64.  Five fp32 operations: 8 * 2^-24 of the largest term, and half a unit in
    the last place of the result type."""
    gen = torch.Generator().manual_seed(sum(shape))
    c = shape[1]
    mod = phx.QBatchNorm2d(c, relu=relu).cuda().eval()
    x = (torch.randn(shape, generator=gen) * 1.5 + 20.0).to(dtype)
    res = torch.randn(shape, generator=gen).to(dtype) if residual else None
    with torch.no_grad():
        mod.weight.copy_(torch.rand(c, generator=gen) + 0.5)
        mod.bias.copy_(torch.randn(c, generator=gen))
        mod.running_mean.copy_(torch.randn(c, generator=gen) + 20.0)
        mod.running_var.copy_(torch.rand(c, generator=gen) + 0.5)
        y = mod(x.cuda(), res.cuda()) if residual else mod(x.cuda())
    d = [t.detach().double().cpu().view(1, c, 1, 1) for t in (mod.weight, mod.bias, mod.running_mean, mod.running_var)]
    term = d[0] * (x.double() - d[2]) / (d[3] + mod.eps).sqrt()
    want = term + d[1] + (res.double() if residual else 0.0)
    if relu:
        want = torch.relu(want)
    size = term.abs().max() + d[1].abs().max() + (res.double().abs().max() if residual else 0.0)
    bound = 8 * 2.0 ** -24 * size + (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -24) * want.abs()
    assert ((y.double().cpu() - want).abs() <= bound).all()
    if shape != (1, 1, 1, 1):  # a gradient through the evaluation mode takes torch's way and agrees
        xg = x.cuda().requires_grad_(True)
        yg = mod(xg, res.cuda()) if residual else mod(xg)
        yg.sum().backward()
        assert torch.isfinite(xg.grad).all()


def test_evaluation_under_transforms():
    """What batches, differentiates forward or traces through the evaluation mode sees torch's operators: the kernel,
    which reads memory, would drop tangents and freeze a trace."""
    gen = torch.Generator().manual_seed(5)
    mod = phx.QBatchNorm2d(3, relu=False).cuda().eval().requires_grad_(False)
    mod.running_mean.copy_(torch.randn(3, generator=gen))
    mod.running_var.copy_(torch.rand(3, generator=gen) + 0.5)
    x, t = (torch.randn((2, 5, 3, 4, 4), generator=gen).cuda() for _ in range(2))
    want = torch.stack([mod(v) for v in x])
    scale = (mod.weight / (mod.running_var + mod.eps).sqrt()).view(1, 3, 1, 1)
    assert torch.allclose(torch.func.vmap(mod)(x), want, rtol=1e-5, atol=1e-6)
    y, dy = torch.func.jvp(mod, (x[0],), (t[0],))
    assert torch.allclose(y, want[0], rtol=1e-5, atol=1e-6) and torch.allclose(dy, scale * t[0], rtol=1e-5, atol=1e-6)
    assert torch.allclose(torch.jit.trace(mod, x[0])(x[1]), want[1], rtol=1e-5, atol=1e-6)
    assert torch.allclose(torch.fx.symbolic_trace(mod, {"residual": None})(x[1]), want[1], rtol=1e-5, atol=1e-6)
