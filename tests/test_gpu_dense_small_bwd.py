"""Both gradients of a small Dense layer in one launch (phx_qdense_bwd): the bits of the two passes behind each other, and the
oracle, where rows do not fill the slices of the filter gradient and quaternions not its workgroups."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
import phoenix_core_amd as phx
from phoenix_core_amd import capi, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("layout", ["IO", "OI"])
@pytest.mark.parametrize("n,ci,co", [(1, 1, 1), (3, 7, 9), (4, 64, 1), (5, 1, 65), (33, 17, 64), (32, 128, 128)])
def test_both_gradients_in_one_launch(n, ci, co, layout, dtype):
    r = np.random.default_rng(n + ci + co)
    x, w, g = r.standard_normal((4 * n, ci)), r.standard_normal((4, ci, co)) * ci ** -0.5, r.standard_normal((4 * n, co))
    w_mem = w.transpose(0, 2, 1) if layout == "OI" else w
    xd, wd, gd = (torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dtype) for a in (x, w_mem, g))
    desc = ops.DenseDescriptor(xd.shape, wd.shape, dtype=dtype, filter_layout=layout, context=phx.Context({}))
    dw, dx = phx.dense_bwd(xd, wd, gd, desc)
    assert "dgrad_wgrad_fma" in capi.last_kernel_name()
    L, dw2, dx2 = capi.lib(), torch.empty_like(dw), torch.empty_like(dx)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert L.phx_qdense_bwd_weights(ctypes.byref(desc.c), stream, xd.data_ptr(), gd.data_ptr(), dw2.data_ptr(), None, 0) == capi.PHX_OK
    assert L.phx_qdense_bwd_data(ctypes.byref(desc.c), stream, gd.data_ptr(), wd.data_ptr(), dx2.data_ptr(), None, 0) == capi.PHX_OK
    assert torch.equal(dw, dw2) and torch.equal(dx, dx2)
    x64, g64 = (a.double().cpu().numpy() for a in (xd, gd))
    w64 = wd.double().cpu().numpy()
    w64 = w64.transpose(0, 2, 1) if layout == "OI" else w64
    want_dw, want_dx = oracle.dense_bwd(x64, w64, g64, "generic")
    got_dw = dw.double().cpu().numpy()
    got_dw = got_dw.transpose(0, 2, 1) if layout == "OI" else got_dw
    # (fp32 sums: every addition rounds what it has so far by 2^-24; one rounding to the storage type)
    once = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -11
    comps = lambda t: np.abs(t).reshape((4, -1, t.shape[-1])).sum(0)
    for got, want, sums, terms in ((got_dw, want_dw, comps(x64).T @ comps(g64), 4 * n), (dx.double().cpu().numpy().reshape(4, n, ci), want_dx.reshape(4, n, ci), comps(g64) @ np.abs(w64).sum(0).T, 4 * co)):
        assert (np.abs(got - want) <= terms * 2.0 ** -24 * sums + once * np.abs(want) * 1.01 + 1e-7).all()


@pytest.mark.parametrize("place", ["x", "half of x", "w", "dw"])
def test_results_on_operands_are_those_of_the_two_passes(place):
    """What the two passes behind each other allow stays allowed, and is not run at once."""
    n, c = 24, 40
    size = 4 * n * c
    desc = ops.DenseDescriptor((4 * n, c), (4, c, c), dtype=torch.float32, context=phx.Context({}))
    L, stream = capi.lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    results = []
    for both in (False, True):
        gen = torch.Generator(device="cuda").manual_seed(3)
        memory = torch.randn(5 * size + 8 * c * c, generator=gen, device="cuda")
        at = lambda element: memory.data_ptr() + 4 * element
        x, g, w, dx, dw = at(0), at(2 * size), at(4 * size), at(4 * size + 4 * c * c), at(5 * size + 4 * c * c)
        if place == "x":
            dx = x
        elif place == "half of x":
            x, dx, g = at(0), at(size // 2), at(size + size // 2)  # (dx: the second half of x and what lies between the two)
        elif place == "w":
            dw = w
        else:
            dx = dw  # (the input gradient is left, and behind it what the filter gradient is longer by)
        if both:
            assert L.phx_qdense_bwd(ctypes.byref(desc.c), stream, x, w, g, dw, dx, None, 0) == capi.PHX_OK
            assert "dgrad_wgrad" not in capi.last_kernel_name()
        else:
            assert L.phx_qdense_bwd_weights(ctypes.byref(desc.c), stream, x, g, dw, None, 0) == capi.PHX_OK
            assert L.phx_qdense_bwd_data(ctypes.byref(desc.c), stream, g, w, dx, None, 0) == capi.PHX_OK
        results.append(memory)
    assert torch.equal(*results)


def test_refusals_are_those_of_the_two_passes():
    desc = ops.DenseDescriptor((8, 4), (4, 4, 4), dtype=torch.float32, context=phx.Context({}))
    x = torch.zeros(8, 4, device="cuda")
    p = x.data_ptr()
    L = capi.lib()
    assert L.phx_qdense_bwd(ctypes.byref(desc.c), None, p, p, p, None, p, None, 0) == capi.PHX_ERR_INVALID_ARGUMENT
    assert L.phx_qdense_bwd(ctypes.byref(desc.c), None, None, p, p, p, p, None, 0) == capi.PHX_ERR_INVALID_ARGUMENT
    assert L.phx_qdense_bwd(None, None, p, p, p, p, p, None, 0) == capi.PHX_ERR_INVALID_ARGUMENT
