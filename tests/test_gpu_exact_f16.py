"""fp16 tensors whose policy asks for fp32 arithmetic run on the fp16 matrix instructions in 16-product form: products
of fp16 values are exact in fp32 and the sums are fp32 sums, so the result is fp32 arithmetic's.  The bound is that of an
fp32 sum rounded once to fp16, which arithmetic on lanes rounded to fp16 would exceed."""
import numpy as np
import pytest
import torch

import oracle
import phoenix_core_amd as phx
from phoenix_core_amd import capi, ops

pytestmark = pytest.mark.gpu

# n, ci, co, h, w, k, stride, what runs it: pointwise streaming, odd plane, one column tile, flat tiling with ragged
# channels, zero-inserted / strided windows, few pixels and many channels, which fp16 arithmetic would slice (slices round
# their partial results to fp16; what fp32 instructions would slice too is left out)
CASES = [(2, 24, 40, 8, 8, 1, 1), (3, 17, 33, 7, 7, 1, 1), (2, 8, 16, 5, 9, 3, 1), (2, 70, 66, 14, 14, 3, 1),
         (1, 20, 36, 11, 13, 3, 2), (2, 3, 16, 16, 16, 5, 2),
         (16, 256, 256, 7, 7, 1, 1)]


class Ctx:
    memory_optimized = False

    def __init__(self, policy):
        self.product_mode = capi.PHX_PRODUCT_8
        self.fp16_policy = {"fp32": capi.PHX_FP16_FULL32, "backward32": capi.PHX_FP16_BACKWARD32}[policy]


def check(got, want, magnitude, terms, what):
    """|got - want| <= half an fp16 ulp of the result + fp32 rounding of a sum of `terms` exact products (every partial
    sum is at most `magnitude`, the sum of the products' absolute values) + half the spacing of fp16 subnormals."""
    bound = 2.0 ** -11 * np.abs(want) + terms * 2.0 ** -24 * magnitude + 2.0 ** -25
    worst = (np.abs(got.cpu().numpy().astype(np.float64) - want) / bound).max()
    assert worst <= 1.0, (what, worst, capi.last_kernel_name())


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -20], ids=["normal", "subnormal"])
@pytest.mark.parametrize("policy", ["fp32", "backward32"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "n%d_%dto%d_%dx%d_k%d_s%d" % c)
def test_fp32_arithmetic_on_fp16_matrix_instructions(case, policy, scale):
    n, ci, co, h, w, k, stride = case
    g = oracle.make_geom(n, ci, co, h, w, k, k, stride, 1, "SAME")
    r = np.random.default_rng(n * 1000 + ci)
    x = (scale * r.standard_normal((4 * n, ci, h, w))).astype(np.float16)
    wt = r.standard_normal((4, co, ci, k, k)).astype(np.float16)
    gr = (scale * r.standard_normal((4 * n, co, g.ho, g.wo))).astype(np.float16)
    gx = (gr / scale).astype(np.float16)  # (the filter gradient multiplies both: one of them at unit scale)
    desc = phx.Conv2DDescriptor(x.shape, wt.shape, stride, 1, "SAME", dtype=torch.float16, context=Ctx(policy))
    xd, wd, gd, gxd = (torch.from_numpy(a).cuda() for a in (x, wt, gr, gx))
    x64, w64, g64, gx64 = (a.astype(np.float64) for a in (x, wt, gr, gx))
    if policy == "fp32":
        y = phx.conv2d_fwd(xd, wd, None, desc)
        assert "exact16mfma" in capi.last_kernel_name()
        check(y, oracle.conv2d_fwd(g, x64, w64, None, "hamilton"), bound_fwd(g, x64, w64), 4 * ci * k * k, "fwd")
    dx = ops.conv2d_bwd_data(wd, gd, desc)
    assert "exact16mfma" in capi.last_kernel_name()
    _, want_dx = oracle.conv2d_bwd(g, x64, w64, g64, "hamilton")
    check(dx, want_dx, bound_dx(g, x64, w64, g64), 4 * co * k * k, "dgrad")
    dw = ops.conv2d_bwd_weights(xd, gxd, desc)
    assert "exact16mfma" in capi.last_kernel_name()
    want_dw, _ = oracle.conv2d_bwd(g, x64, w64, gx64, "hamilton")
    check(dw, want_dw, bound_dw(g, x64, w64, gx64), 4 * n * g.ho * g.wo, "wgrad")


def _components_summed(t, n):
    """The sum of the four components' absolute values, as the real part of a quaternion tensor: products of such
    tensors, component by component equal, bound every component's sum of absolute products."""
    a = np.abs(t).reshape(4, n, *t.shape[1:]).sum(0) if n else np.abs(t).sum(0, keepdims=True)
    z = np.zeros_like(a)
    return np.concatenate([a, z, z, z]) if n else np.concatenate([a, 0 * a, 0 * a, 0 * a])


def bound_fwd(g, x, w):
    y = oracle.conv2d_fwd(g, _components_summed(x, g.n), _components_summed(w, 0), None, "hamilton")
    return np.tile(y[: g.n], (4, 1, 1, 1))


def bound_dx(g, x, w, gr):
    _, dx = oracle.conv2d_bwd(g, x, _components_summed(w, 0), _components_summed(gr, g.n), "hamilton")
    return np.tile(dx[: g.n], (4, 1, 1, 1))


def bound_dw(g, x, w, gr):
    dw, _ = oracle.conv2d_bwd(g, _components_summed(x, g.n), w, _components_summed(gr, g.n), "hamilton")
    return np.tile(dw[:1], (4, 1, 1, 1, 1))
