"""fp32 passes on bf16 instructions over the whole range of fp32: infinities and values that bf16 rounds to one, values whose second
and third part bf16 would not hold."""
import pytest
import torch

import phoenix_core_amd as phx
from phoenix_core_amd import capi, ops
from test_gpu_dense_gemm import _dense
from test_gpu_split_f32 import _hamilton

pytestmark = pytest.mark.gpu

# kind, n, inputs, outputs, h, w, taps, layout, kernels of the forward / input gradient and of the filter gradient (None: not on these
# instructions), more of a convolution
CASES = [
    ("conv", 3, 24, 40, 13, 9, 3, "NCHW", "f32mfmax3_p8", "f32mfmax3_p8"), ("conv", 2, 128, 96, 7, 7, 3, "NCHW", "kslices", "f32mfmax3_p8"),
    ("conv", 64, 64, 64, 28, 28, 3, "NCHW", "flat", "f32mfmax3_p8"), ("conv", 2, 40, 30, 15, 7, 1, "NCHW", "f32mfmax3pw", "f32mfmax3_p8"),
    ("conv", 3, 97, 100, 7, 5, 1, "NCHW", "f32mfmax3pw", "mfmagemm"), ("conv", 9, 128, 128, 14, 11, 1, "NHWC", "f32mfmax3pw", "mfmagemm"),
    ("conv", 2, 20, 40, 15, 17, 3, "NCHW", "f32mfmax3", None, dict(dilation=2)), ("conv", 2, 24, 40, 21, 18, 7, "NCHW", "f32mfmax3", None, dict(stride=2)),
    ("conv", 2, 80, 96, 13, 11, 3, "NCHW", "groups2", "groups2", dict(groups=2)),
    ("dense", 70, 130, 90, 1, 1, 1, "", "mfmagemm", "mfmagemm"), ("dense", 33, 1000, 24, 1, 1, 1, "", "mfmagemm", "mfmagemm"),
]


class _Layer:
    def __init__(self, case):
        self.kind, n, ci, co, h, w, k, self.layout, self.fwd_kernel, self.wgrad_kernel = case[:10]
        self.more = dict(case[10]) if len(case) > 10 else {}
        gen = torch.Generator(device="cuda").manual_seed(ci)

        def values(*shape):  # magnitudes from 1/8 to 7/8
            return (torch.rand(shape, generator=gen, device="cuda") * 0.75 + 0.125) * (torch.randint(0, 2, shape, generator=gen, device="cuda") * 2 - 1)

        if self.kind == "dense":
            self.x, self.w, self.g = values(4 * n, ci), values(4, ci, co), values(4 * n, co)
            self.desc = ops.DenseDescriptor(self.x.shape, self.w.shape, dtype=torch.float32, context=phx.Context({}))
        else:
            self.k = k
            stride = self.more.get("stride", 1)
            self.x, self.w = values(4 * n, ci, h, w), values(4, co, ci // self.more.get("groups", 1), k, k)
            self.g = values(4 * n, co, -(-h // stride), -(-w // stride))
            self.desc = ops.Conv2DDescriptor(self.last(self.x).shape, self.w.shape, padding="SAME", dtype=torch.float32, context=phx.Context({}),
                                             data_format=self.layout, **self.more)

    def last(self, t):
        return t.permute(0, 2, 3, 1).contiguous() if self.layout == "NHWC" else t

    def first(self, t):
        return t.permute(0, 3, 1, 2).contiguous() if self.layout == "NHWC" else t

    def reference(self, which):
        x, w, g = (t.double().requires_grad_() for t in (self.x, self.w, self.g))
        if self.kind == "dense":
            y = _dense(x, w)
        else:
            (pt, pl), (pb, pr) = self.desc.pad_before, self.desc.pad_after
            y = _hamilton(torch.nn.functional.pad(x, (pl, pr, pt, pb)), w, lambda a, b: torch.nn.functional.conv2d(a, b, **self.more))
        if which == "fwd":
            return y.detach()
        return torch.autograd.grad(y, x if which == "dgrad" else w, g)[0]

    def run(self, which):
        if self.kind == "dense":
            if which == "fwd":
                y = phx.dense_fwd(self.x, self.w, None, self.desc)
                assert self.fwd_kernel in capi.last_kernel_name()
                return y
            dw, dx = phx.dense_bwd(self.x, self.w, self.g, self.desc)
            assert self.fwd_kernel in capi.last_kernel_name()
            return dx if which == "dgrad" else dw
        if which == "wgrad":
            dw = ops.conv2d_bwd_weights(self.last(self.x), self.last(self.g), self.desc)
            assert self.wgrad_kernel in capi.last_kernel_name(), capi.last_kernel_name()
            return dw
        if which == "fwd":
            y = phx.conv2d_fwd(self.last(self.x), self.w, None, self.desc)
        else:
            y = ops.conv2d_bwd_data(self.w, self.last(self.g), self.desc)
        assert self.fwd_kernel in capi.last_kernel_name(), capi.last_kernel_name()
        return self.first(y)

    def operands(self, which):
        return {"fwd": (self.x, self.w), "dgrad": (self.g, self.w), "wgrad": (self.x, self.g)}[which]


def _layer(case, tune_env):
    tune_env(PHX_TUNE_DENSEGEMM="1")
    return _Layer(case)


_ids = lambda c: "%s_n%d_%dto%d_%dx%d_k%d%s" % c[:8] + "".join("_%s%d" % m for m in (c[10] if len(c) > 10 else {}).items())
_everywhere = pytest.mark.parametrize("case,which", [(c, w) for c in CASES for w in ("fwd", "dgrad", "wgrad") if w != "wgrad" or c[9]],
                                      ids=lambda v: v if isinstance(v, str) else _ids(v))


def _middle(t):
    """An element in the middle of a tensor, away from the border of its plane."""
    i = [s // 2 for s in t.shape]
    if t.dim() == 5:  # a filter: its middle tap
        i[0] = 2
    return tuple(i)


def _same(got, want):
    """Infinities where fp64 has them, elsewhere an error of fp32."""
    inf = torch.isinf(want)
    assert torch.equal(got.double()[inf], want[inf]) and bool(torch.isfinite(got[~inf]).all())
    # (sums of some hundred to some thousand terms on either path: half a dozen roundings of 2^-24 in the root mean square)
    assert float((got.double() - want)[~inf].norm()) <= 2e-6 * float(want[~inf].norm())


@pytest.mark.parametrize("operand", [0, 1])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), 3.4e38, -1e32])
@_everywhere
def test_one_extreme_value(case, which, value, operand, tune_env):
    layer = _layer(case, tune_env)
    t = layer.operands(which)[operand]
    t[_middle(t)] = value
    # (fp64's convolution multiplies the padding's zeros too: _middle keeps clear of them)
    want = layer.reference(which)
    assert bool(torch.isinf(want).any()) == (abs(value) == float("inf"))
    _same(layer.run(which), want)


@_everywhere
def test_not_a_number_reaches_what_it_reaches(case, which, tune_env):
    layer = _layer(case, tune_env)
    t = layer.operands(which)[0]
    t[_middle(t)] = float("nan")
    want, got = layer.reference(which), layer.run(which)
    nan = torch.isnan(want)
    assert bool(nan.any()) and torch.equal(torch.isnan(got), nan)


@pytest.mark.parametrize("powers", [(-118, 30), (30, -118), (-60, -40), (70, -10)], ids=str)
@_everywhere
def test_powers_of_two_change_no_bit(case, which, powers, tune_env):
    """From operands of 2^-121 on the three parts hold 24 bits, so every product and sum is the scaled one."""
    layer = _layer(case, tune_env)
    plain = layer.run(which)
    for t, power in zip(layer.operands(which), powers):
        t.mul_(2.0 ** power)
    assert torch.equal(layer.run(which).double(), plain.double() * 2.0 ** sum(powers))


@_everywhere
def test_subnormal_and_huge_operands(case, which, tune_env):
    for powers in ((-140, 60), (110, -40), (60, 50)):
        layer = _layer(case, tune_env)
        for t, power in zip(layer.operands(which), powers):
            t.mul_(2.0 ** (power / 2)).mul_(2.0 ** (power / 2))
        _same(layer.run(which), layer.reference(which))


@pytest.mark.parametrize("case", [c for c in CASES if c[0] == "conv" and c[7] == "NCHW"], ids=_ids)
def test_packed_filters_keep_an_infinity(case, tune_env):
    layer = _layer(case, tune_env)
    layer.w[_middle(layer.w)] = float("inf")
    layer.x[_middle(layer.x)] = -1e38
    packed = ops.conv2d_pack_filters(layer.w, layer.desc)
    zero = torch.zeros_like(layer.w)
    y, dx = phx.conv2d_fwd(layer.x, layer.w, None, layer.desc), ops.conv2d_bwd_data(layer.w, layer.g, layer.desc)
    assert bool(torch.isinf(y).any()) and bool(torch.isinf(dx).any()) and not bool(torch.isnan(dx).any())
    assert torch.equal(y, phx.conv2d_fwd(layer.x, zero, None, layer.desc, packed=packed))
    assert torch.equal(dx, ops.conv2d_bwd_data(zero, layer.g, layer.desc, packed=packed))
