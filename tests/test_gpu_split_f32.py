"""fp32 passes on bf16 instructions (phx_kernels_x3.h, phx_kernels_wgx3.h) against fp64, beside the fp32 instructions."""
import ctypes

import pytest
import torch

import phoenix_core_amd as phx
from phoenix_core_amd import capi, ops

pytestmark = pytest.mark.gpu


def _hamilton(x, w, f):
    xs, out = x.chunk(4), [0, 0, 0, 0]
    for p in range(4):
        for q in range(4):
            out[q] = out[q] + f(xs[p], w[p ^ q]) * (-1 if (0x3950 >> (p * 4 + q)) & 1 else 1)
    return torch.cat(out)


def _gap(a, b):
    return float((a.double() - b).norm() / b.norm())


# n, ci, co, h, w, k, stride, dilation, groups: sub-tiles of 32 and 64 output channels, wide and narrow tiles, flat and
# rectangular tilings, ragged channels, planes that are one partial group of four, tensors whose ends every load meets;
# pointwise: odd planes, a plane of one pair, tiles over several images, a remainder of a K step, slices, groups, a stride
CASES = [
    (3, 8, 40, 9, 13, 3, 1, 1, 1), (1, 9, 33, 3, 3, 3, 1, 1, 1), (1, 1, 1, 1, 2, 3, 1, 1, 1), (40, 16, 64, 14, 14, 3, 1, 1, 1),
    (2, 24, 20, 30, 7, 5, 1, 1, 1), (4, 130, 70, 21, 18, 3, 2, 1, 1), (2, 17, 65, 20, 20, 3, 1, 2, 1), (1, 64, 96, 7, 7, 3, 1, 1, 1),
    (2, 80, 96, 12, 10, 3, 1, 1, 2), (64, 72, 64, 16, 16, 3, 1, 1, 1), (1, 5, 7, 70, 3, 7, 1, 1, 1),
    (2, 20, 33, 5, 7, 1, 1, 1, 1), (1, 16, 16, 1, 2, 1, 1, 1, 1), (1, 3, 1, 3, 1, 1, 1, 1, 1), (13, 40, 24, 9, 9, 1, 1, 1, 1),
    (2, 512, 128, 7, 7, 1, 1, 1, 1), (3, 80, 96, 12, 10, 1, 1, 1, 2), (4, 40, 72, 15, 14, 1, 2, 1, 1),
]


def _rounds_less(channels, k):
    """Whether the bf16 instructions round a sum over these channels less often than the fp32 instructions: they take it then."""
    return channels > 2 if k == 1 else 3 * -(-channels // 8) <= 0.455 * channels


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_error_against_fp64(case, tune_env):
    n, ci, co, h, w, k, stride, dilation, groups = case
    on_bf16 = _rounds_less(ci // groups, k), _rounds_less(co // groups, k)
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(4 * n, ci, h, w, generator=gen, device="cuda")
    wt = torch.randn(4, co, ci // groups, k, k, generator=gen, device="cuda")
    bias = torch.randn(4, co, generator=gen, device="cuda")
    args = dict(stride=stride, dilation=dilation, padding="SAME", groups=groups, dtype=torch.float32, context=phx.Context({}))
    desc, back = ops.Conv2DDescriptor(x.shape, wt.shape, use_bias=True, **args), ops.Conv2DDescriptor(x.shape, wt.shape, **args)
    grad = torch.randn(desc.output_shape, generator=gen, device="cuda")
    (pt, pl), (pb, pr) = desc.pad_before, desc.pad_after
    xr = x.double().requires_grad_()
    yr = _hamilton(torch.nn.functional.pad(xr, (pl, pr, pt, pb)), wt.double(),
                   lambda a, b: torch.nn.functional.conv2d(a, b, stride=stride, dilation=dilation, groups=groups))
    dxr, = torch.autograd.grad(yr, xr, grad.double())
    yr = yr.detach() + bias.double().view(4, 1, co, 1, 1).expand(4, n, co, 1, 1).reshape(4 * n, co, 1, 1)
    gaps = {}
    for nox3 in (None, "1"):
        tune_env(PHX_TUNE_NOX3=nox3)
        y = phx.conv2d_fwd(x, wt, bias, desc)
        names = [capi.last_kernel_name()]
        dx = ops.conv2d_bwd_data(wt, grad, back)
        names.append(capi.last_kernel_name())
        assert ("f32mfmax3" in names[0]) == (nox3 is None and on_bf16[0]), names
        assert stride > 1 or ("f32mfmax3" in names[1]) == (nox3 is None and on_bf16[1]), names
        packed = ops.conv2d_pack_filters(wt, desc)
        if packed is not None:
            assert torch.equal(y, phx.conv2d_fwd(x, torch.zeros_like(wt), bias, desc, packed=packed))
            assert torch.equal(dx, ops.conv2d_bwd_data(torch.zeros_like(wt), grad, back, packed=packed))
        gaps[nox3] = _gap(y, yr), _gap(dx, dxr)
    # each error is a sum of many roundings of like size: their 2-norms over hundreds of results lie within a tenth of their
    # expectation; a dozen results, of a dozen roundings of 2^-25 in the mean each, are bounded by those
    few = min(yr.numel(), xr.numel()) < 500
    for ours, fp32 in zip(gaps[None], gaps["1"]):
        assert ours <= 1.1 * fp32 + (2.0 ** -23 if few else 0.0), gaps


@pytest.mark.parametrize("case", [(2, 512, 64, 14, 5), (1, 600, 40, 14, 7), (1, 1024, 30, 21, 5), (4, 8192, 64, 14, 1), (2, 9250, 30, 9, 1)],
                         ids=lambda c: "n%d_%dto%d_%dx_k%d" % c)
def test_long_reductions_do_not_drift(case, tune_env):
    """One chain of all products: the instructions drop low bits downwards, which would take 0.3 of the root mean square error
    and more off every result at 12800 products and 8192 single ones.  What remains is at most half a stretch of 2304 products'
    own, a sixth of the error there and less behind longer sums."""
    tune_env(PHX_TUNE_KSLICES="0")
    n, ci, co, h, k = case
    gen = torch.Generator(device="cuda").manual_seed(5)
    x, wt, grad = (torch.randn(s, generator=gen, device="cuda") for s in ((4 * n, ci, h, h), (4, co, ci, k, k), (4 * n, ci, h, h)))
    conv = lambda a, b: torch.nn.functional.conv2d(a, b, padding=k // 2)
    desc = ops.Conv2DDescriptor(x.shape, wt.shape, padding="SAME", dtype=torch.float32, context=phx.Context({}))
    y = phx.conv2d_fwd(x, wt, None, desc)
    assert "f32mfmax3" in capi.last_kernel_name() and "kslices" not in capi.last_kernel_name()
    # (the input gradient of the layer whose filter is the other way round)
    back = wt.transpose(1, 2).contiguous()
    desc = ops.Conv2DDescriptor((4 * n, co, h, h), back.shape, padding="SAME", dtype=torch.float32, context=phx.Context({}))
    dx = ops.conv2d_bwd_data(back, grad, desc)
    assert "f32mfmax3" in capi.last_kernel_name() and "kslices" not in capi.last_kernel_name()
    z = torch.zeros(4 * n, co, h, h, dtype=torch.float64, device="cuda", requires_grad=True)
    dxr, = torch.autograd.grad(_hamilton(z, back.double(), conv), z, grad.double())
    for got, want in ((y, _hamilton(x.double(), wt.double(), conv)), (dx, dxr)):
        error = got.double() - want
        assert abs(float(error.mean())) <= 0.15 * float(error.square().mean().sqrt())


@pytest.mark.parametrize("k", [1, 3, 5])
@pytest.mark.parametrize("ci", [1, 2, 3, 6, 7, 8, 9, 12, 13, 14, 17, 19, 20, 26, 27, 33, 41])
def test_sums_over_few_channels(ci, k, tune_env):
    """A chunk of eight channels is rounded as often for one of them as for all."""
    gen = torch.Generator(device="cuda").manual_seed(ci)
    x, wt = torch.randn(32, ci, 20, 20, generator=gen, device="cuda"), torch.randn(4, 32, ci, k, k, generator=gen, device="cuda")
    desc = ops.Conv2DDescriptor(x.shape, wt.shape, padding="SAME", dtype=torch.float32, context=phx.Context({}))
    want = _hamilton(x.double(), wt.double(), lambda a, b: torch.nn.functional.conv2d(a, b, padding=k // 2))
    gaps = []
    for nox3 in (None, "1"):
        tune_env(PHX_TUNE_NOX3=nox3)
        gaps.append(_gap(phx.conv2d_fwd(x, wt, None, desc), want))
        assert ("f32mfmax3" in capi.last_kernel_name()) == (nox3 is None and _rounds_less(ci, k))
    # (the 2-norms of the roundings of 400 thousand results, those of a filter row alike: within some per cent)
    assert gaps[0] <= 1.03 * gaps[1], gaps


@pytest.mark.parametrize("case,kernel", [((2, 24, 16, 9, 9, 3), "thin"), ((20, 16, 32, 14, 14, 3), "thin"), ((21, 24, 17, 14, 14, 3), "f32mfmax3"),
                                         ((64, 18, 18, 14, 14, 5), "thin"), ((1, 24, 24, 1, 3, 3), "f32mfmav"), ((1, 64, 24, 2, 2, 1), "f32mfmax3")],
                         ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_filter_gradients_of_few_channels_and_of_few_pixels(case, kernel):
    """Short sums run where they are rounded least."""
    x, grad, desc, ref = _wgrad(case + (1, 1))
    dw = ops.conv2d_bwd_weights(x, grad, desc)
    assert kernel in capi.last_kernel_name(), capi.last_kernel_name()
    assert _gap(dw, ref) <= 2e-7


SIGNS = ["mean_zero", "one_sign"]


def _values(signs, gen, *shape):
    """Normal values, or positive ones (activations behind a ReLU, say), whose sums grow with every product."""
    return torch.randn(shape, generator=gen, device="cuda") if signs == "mean_zero" else torch.rand(shape, generator=gen, device="cuda") + 0.05


@pytest.mark.parametrize("signs", SIGNS)
@pytest.mark.parametrize("case", [(8, 64, 64, 28, 3), (2, 512, 64, 14, 5), (16, 64, 64, 28, 1), (4, 2048, 64, 14, 1)], ids=lambda c: "n%d_%dto%d_%d_k%d" % c)
def test_error_of_either_kind_of_sums(case, signs, tune_env):
    n, ci, co, h, k = case
    gen = torch.Generator(device="cuda").manual_seed(5)
    x, wt = _values(signs, gen, 4 * n, ci, h, h), _values(signs, gen, 4, co, ci, k, k)
    if signs == "one_sign":
        wt[1:] *= -1  # (a component of four products of one sign)
    desc = ops.Conv2DDescriptor(x.shape, wt.shape, padding="SAME", dtype=torch.float32, context=phx.Context({}))
    want = _hamilton(x.double(), wt.double(), lambda a, b: torch.nn.functional.conv2d(a, b, padding=k // 2))
    gaps = []
    for nox3 in (None, "1"):
        tune_env(PHX_TUNE_NOX3=nox3)
        gaps.append(_gap(phx.conv2d_fwd(x, wt, None, desc), want))
        assert ("f32mfmax3" in capi.last_kernel_name()) == (nox3 is None)
    assert gaps[0] <= 1.1 * gaps[1], gaps  # (see test_error_against_fp64)


@pytest.mark.parametrize("signs", SIGNS)
@pytest.mark.parametrize("case", [(32, 96, 96, 56, 56, "NCHW"), (32, 96, 96, 56, 56, "NHWC"), (16, 256, 128, 28, 28, "NCHW"), (1, 475, 475, 28, 27, "NCHW"), (4096, 256, 256, 1, 1, ""),
                                  (20000, 64, 64, 1, 1, ""), (1000, 2048, 100, 1, 1, "")], ids=lambda c: "n%d_%dto%d_%dx%d%s" % c)
def test_filter_gradients_as_matrix_products_of_long_sums(case, signs, tune_env):
    """Reductions over thousands of pixels or rows, in up to a hundred slices, beside the fp32 instructions."""
    n, ci, co, h, w, layout = case
    gen = torch.Generator(device="cuda").manual_seed(5)
    x, grad = _values(signs, gen, 4 * n, h, w, ci), _values(signs, gen, 4 * n, h, w, co)
    rows = lambda t: t.reshape(4, -1, t.shape[-1]).double()
    xs, gs, want = rows(x), rows(grad), torch.zeros(4, ci, co, dtype=torch.float64, device="cuda")
    for p in range(4):
        for q in range(4):
            want[p ^ q] += (xs[p].t().contiguous() @ gs[q]) * (-1 if (0x3950 >> (p * 4 + q)) & 1 else 1)
    gaps = []
    for nox3 in (None, "1"):
        tune_env(PHX_TUNE_NOX3=nox3, PHX_TUNE_NOSMALLDENSE="1")
        if layout:
            last = (lambda t: t) if layout == "NHWC" else (lambda t: t.permute(0, 3, 1, 2).contiguous())
            desc = ops.Conv2DDescriptor(last(x).shape, (4, co, ci, 1, 1), dtype=torch.float32, context=phx.Context({}), data_format=layout)
            dw = ops.conv2d_bwd_weights(last(x), last(grad), desc).view(4, co, ci).transpose(1, 2)
            assert ("mfmagemm" in capi.last_kernel_name()) == (nox3 is None), capi.last_kernel_name()
        else:
            x2, g2 = x.view(4 * n, ci), grad.view(4 * n, co)
            wt = torch.zeros(4, ci, co, device="cuda")
            desc = ops.DenseDescriptor(x2.shape, wt.shape, dtype=torch.float32, context=phx.Context({}))
            dw, _ = phx.dense_bwd(x2, wt, g2, desc)
            assert ("mfmagemm" in capi.last_kernel_name()) == (nox3 is None), capi.last_kernel_name()
        gaps.append(_gap(dw, want))
    # (of one sign both are little above the last rounding, 2^-25 / sqrt(3) of each value in the mean: it counts for both)
    assert gaps[0] <= 1.1 * gaps[1], gaps


def test_whole_numbers_are_exact():
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randint(-300, 301, (8, 16, 12, 12), generator=gen, device="cuda").float()
    wt = torch.randint(-40, 41, (4, 40, 16, 3, 3), generator=gen, device="cuda").float()
    desc = ops.Conv2DDescriptor(x.shape, wt.shape, padding="VALID", dtype=torch.float32, context=phx.Context({}))
    y = phx.conv2d_fwd(x, wt, None, desc)
    assert "f32mfmax3" in capi.last_kernel_name()
    assert torch.equal(y.double(), _hamilton(x.double(), wt.double(), torch.nn.functional.conv2d))


def test_fixed_scratch_keeps_the_fp32_instructions_where_the_parts_do_not_fit(tune_env):
    """192 x 192 x 9 filter values: 10.6 MB packed for the fp32 instructions, twice that as three parts."""
    x, wt = torch.randn(4, 192, 6, 6, device="cuda"), torch.randn(4, 192, 192, 3, 3, device="cuda")
    desc = ops.Conv2DDescriptor(x.shape, wt.shape, padding="SAME", dtype=torch.float32, context=phx.Context({}))
    assert desc.workspace_bytes(capi.PHX_PASS_FWD) > capi.PHX_NOALLOC_SCRATCH_BYTES
    y = torch.empty(desc.output_shape, device="cuda")
    stream = ops.current_stream_handle(x.device)
    capi.check(capi.lib().phx_qconv2d_fwd_noalloc(ctypes.byref(desc.c), stream, x.data_ptr(), wt.data_ptr(), None, y.data_ptr()), "noalloc")
    assert "f32mfmax3" not in capi.last_kernel_name()
    phx.conv2d_fwd(x, wt, None, desc)
    assert "f32mfmax3" in capi.last_kernel_name()
    tune_env(PHX_TUNE_NOX3="1")
    assert torch.equal(y, phx.conv2d_fwd(x, wt, None, desc))


# n, ci, co, h, w, k, stride, groups: one, two and three taps of a filter row and their remainders (5, 7), rows shorter than a
# segment and with a remainder, an odd number of segments, channels past a tile of either side, one and many reduction slices,
# tensors whose ends every load meets, groups in one launch, strides by tap classes
WGRAD_CASES = [
    (1, 24, 24, 9, 9, 3, 1, 1), (4, 70, 130, 14, 14, 3, 1, 1), (2, 33, 31, 9, 17, 7, 1, 1), (16, 104, 40, 58, 7, 5, 1, 1),
    (64, 32, 32, 9, 9, 1, 1, 1), (64, 64, 64, 4, 4, 3, 1, 1), (20, 64, 64, 17, 17, 3, 1, 1), (128, 48, 40, 9, 9, 3, 1, 1),
    (16, 512, 256, 7, 7, 3, 1, 1), (4, 160, 192, 12, 10, 3, 1, 2), (32, 128, 128, 14, 14, 5, 2, 1),
]


def _wgrad(case, x=None, grad=None):
    n, ci, co, h, w, k, stride, groups = case
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(4 * n, ci, h, w, generator=gen, device="cuda") if x is None else x
    desc = ops.Conv2DDescriptor(x.shape, (4, co, ci // groups, k, k), stride=stride, padding="SAME", groups=groups,
                                dtype=torch.float32, context=phx.Context({}))
    grad = torch.randn(desc.output_shape, generator=gen, device="cuda") if grad is None else grad
    (pt, pl), (pb, pr) = desc.pad_before, desc.pad_after
    wr = torch.zeros(4, co, ci // groups, k, k, dtype=torch.float64, device="cuda", requires_grad=True)
    yr = _hamilton(torch.nn.functional.pad(x.double(), (pl, pr, pt, pb)), wr,
                   lambda a, b: torch.nn.functional.conv2d(a, b, stride=stride, groups=groups))
    return x, grad, desc, torch.autograd.grad(yr, wr, grad.double())[0]


@pytest.mark.parametrize("case", WGRAD_CASES, ids=lambda c: "x".join(map(str, c)))
def test_filter_gradient_error_against_fp64(case, tune_env):
    x, grad, desc, ref = _wgrad(case)
    gaps = {}
    for nox3 in (None, "1"):
        tune_env(PHX_TUNE_NOX3=nox3)
        dw = ops.conv2d_bwd_weights(x, grad, desc)
        assert ("f32mfmax3" in capi.last_kernel_name()) == (nox3 is None), capi.last_kernel_name()
        gaps[nox3] = _gap(dw, ref)
    assert gaps[None] <= 1.1 * gaps["1"], gaps  # (the norms of thousands of roundings: see above)


def test_filter_gradient_of_whole_numbers_is_exact():
    case = (6, 40, 70, 11, 13, 3, 1, 1)
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randint(-300, 301, (24, 40, 11, 13), generator=gen, device="cuda").float()
    grad = 2 * torch.randint(-20, 21, (24, 70, 11, 13), generator=gen, device="cuda").float()  # (four of the lanes are halved)
    x, grad, desc, ref = _wgrad(case, x, grad)
    dw = ops.conv2d_bwd_weights(x, grad, desc)
    assert "f32mfmax3" in capi.last_kernel_name()
    assert torch.equal(dw.double(), ref)
