"""The one-pass batch-norm kernels, whose workgroups hold their part of a channel in registers and wait for their neighbours'
sums, at the edges of their plan: planes of one 16-byte chunk and of one element more, a partial last chunk in every plane, one
workgroup a channel, as many as ask for 512 threads, and more than 64 of those, which stay on two launches.  Against fp64 with
test_gpu_bn's tolerances; with no wait allowed every workgroup forms the channel's sums itself, and the results are the same.
What ran is read from the kernels' names."""
import ctypes

import pytest
import torch

import test_gpu_bn
from phoenix_core_amd import capi, ops

pytestmark = pytest.mark.gpu

# threads of a workgroup, 0: two launches; (fp32, fp16), where they differ by the pass (forward, with a residual, backward)
SHAPES = {(8, 16, 14, 14): (256, 256), (12, 5, 7, 7): (256, 256), (64, 33, 9, 5): (256, 256), (2, 3, 2, 4): (256, 256), (5, 1100, 3, 3): (256, 256),
          (65, 2, 4, 8): (256, 256), (37, 6, 31, 17): (256, 256), (1, 1, 64, 96): (256, 256), (257, 1, 40, 41): (0, 0), (700, 2, 21, 20): (0, 0),
          (40, 512, 7, 7): (256, 256), (131, 17, 57, 55): ((256, 512, 512), 256)}
MANY = {(293, 17, 57, 55): (512, (256, 512, 512))}  # (61 and 60 workgroups a channel)


def _ran(shape, dtype, passes):
    """The start of the names of these passes of a shape."""
    threads = {**SHAPES, **MANY}[shape][dtype == torch.float16]
    threads = threads if isinstance(threads, tuple) else (threads,) * 3
    names = {"fwd": ("bn_fwd_%s", threads[0]), "fwd_res": ("bn_fwd_%s_res", threads[1]), "bwd": ("bn_bwd_%s", threads[2]), "bwd_res": ("bn_bwd_%s_res", threads[2])}
    of = lambda name, t: (name + ("_held%d_s" % t if t else "_two_s")) % ("f16" if dtype == torch.float16 else "f32")
    return [of(*names[p]) for p in passes]


@pytest.fixture(params=["4096", "0"], ids=["waits", "alone"])
def held(request, tune_env):
    tune_env(PHX_TUNE_BN_HELD="1", PHX_TUNE_BN_WAITS=request.param)


@pytest.fixture
def names(monkeypatch):
    """What the operators' batch-norm calls ran, in their order."""
    seen = []

    def watched(op):
        def call(*args):
            result = op(*args)
            seen.append(capi.bn_last_kernel_name())
            return result
        return call

    for op in ("batch_norm_fwd", "batch_norm_bwd"):
        monkeypatch.setattr(ops, op, watched(getattr(ops, op)))
    return seen


def _are(names, expected):
    assert len(names) == len(expected) and all(n.startswith(e) for n, e in zip(names, expected)), (names, expected)


@pytest.mark.parametrize("relu,residual", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_one_pass_matches_torch(held, names, shape, dtype, relu, residual):
    test_gpu_bn.test_batch_norm_matches_torch(shape, dtype, relu, residual)
    _are(names, _ran(shape, dtype, ("fwd_res", "bwd_res") if residual else ("fwd", "bwd")))


@pytest.mark.parametrize("shape,dtype,residual", [(s, d, r) for s in MANY for d, r in ((torch.float32, False), (torch.float16, True))],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_many_workgroups_a_channel_match_torch(shape, dtype, residual, names, tune_env):
    tune_env(PHX_TUNE_BN_HELD="1")
    test_gpu_bn.test_batch_norm_matches_torch(shape, dtype, True, residual)
    _are(names, _ran(shape, dtype, ("fwd_res", "bwd_res") if residual else ("fwd", "bwd")))


def test_calls_that_stay_on_two_launches():
    """By the rule's sizes, a workspace that does not hold the words, one that is not aligned for them, and results on operands."""
    rows, c, hw = 8, 64, 112 * 112
    gen = torch.Generator(device="cuda").manual_seed(7)
    x, dy = (torch.randn(rows, c, 112, 112, generator=gen, device="cuda").half() for _ in range(2))
    gamma, beta = torch.rand(c, device="cuda") + 0.5, torch.randn(c, device="cuda")
    mean, invstd, dgamma, dbeta = (torch.empty(c, device="cuda") for _ in range(4))
    desc = capi.BnDesc(capi.PHX_F16, rows, c, hw, 1e-5, 0.1, 1)
    L, stream, at = capi.lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), lambda t: t.data_ptr()
    size = L.phx_bn_workspace_bytes(ctypes.byref(desc))
    memory = torch.empty(size + 256, dtype=torch.uint8, device="cuda")

    def bwd(dx, offset=0, nbytes=size):
        x0 = x.clone()
        out = x0 if dx == "x" else dy.clone() if dx == "dy" else torch.empty_like(x)
        grad = out if dx == "dy" else dy
        assert L.phx_bn_bwd(ctypes.byref(desc), stream, at(x0), None, at(grad), at(gamma), at(beta), at(mean), at(invstd), at(out), None, at(dgamma),
                            at(dbeta), at(memory) + offset, nbytes) == capi.PHX_OK
        return capi.bn_last_kernel_name(), [out, dgamma.clone(), dbeta.clone()]

    y = torch.empty_like(x)
    fwd = lambda out: L.phx_bn_fwd_train(ctypes.byref(desc), stream, at(out), None, at(gamma), at(beta), at(y), at(mean), at(invstd), None, None, at(memory), size)
    assert fwd(x) == capi.PHX_OK and capi.bn_last_kernel_name().startswith("bn_fwd_f16_two_s")  # (12.8 MB)
    name, want = bwd("own")
    assert name == "bn_bwd_f16_held256_s16"
    words = 8 * c * 16  # (two launches ask for half of that)
    assert bwd("own", nbytes=words)[0] == name
    for args in (dict(dx="x"), dict(dx="dy"), dict(dx="own", offset=4), dict(dx="own", nbytes=words - 8)):
        name, got = bwd(**args)
        assert name == "bn_bwd_f16_two_s8", (args, name)
        # (fp32 sums of 100352 terms in another order, then one rounding to fp16)
        for a, e in zip(got, want):
            assert float((a.double() - e.double()).norm() / e.double().norm()) < 1e-3


def test_one_pass_under_capture_and_on_nonfinite_values():
    """A replayed graph waits for the sums of its own replay; a NaN or an infinity reaches its whole channel and no other."""
    shape = (512, 24, 41, 42)  # (42 MB: the rule's own choice)
    params = [torch.rand(24, device="cuda") + 0.5 for _ in range(4)]
    x = torch.randn(shape, device="cuda", dtype=torch.float16)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        run = lambda: ops.batch_norm_fwd(x, *params[:2], params[2].clone(), params[3].clone(), 1e-5, 0.1, True, None)
        run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        replayed = run()
    for seed in range(3):
        x.copy_(torch.randn(shape, generator=torch.Generator().manual_seed(seed)).half())
        eager = run()
        assert capi.bn_last_kernel_name().startswith("bn_fwd_f16_held256_s")
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(eager, replayed))
    x[3, 5, 2, 1] = float("nan")
    x[200, 7, 0, 0] = float("inf")
    y = run()[0]
    bad = [c for c in range(24) if not torch.isfinite(y[:, c]).all() or bool((y[:, c] == 0).all())]
    assert bad == [5, 7]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(64, 33, 9, 5), (37, 6, 31, 17), (131, 17, 57, 55)], ids=lambda s: "x".join(map(str, s)))
def test_results_do_not_depend_on_who_forms_the_sums(shape, dtype, names, tune_env):
    gen = torch.Generator(device="cuda").manual_seed(5)
    x, dy, res = (torch.randn(shape, generator=gen, device="cuda").to(dtype) for _ in range(3))
    gamma, beta = torch.rand(shape[1], device="cuda") + 0.5, torch.randn(shape[1], device="cuda")
    results = []
    for waits in ("4096", "0"):
        tune_env(PHX_TUNE_BN_HELD="1", PHX_TUNE_BN_WAITS=waits)
        for r in (None, res):
            run = [torch.zeros(shape[1], device="cuda") for _ in range(2)]
            y, mean, invstd = ops.batch_norm_fwd(x, gamma, beta, *run, 1e-5, 0.1, True, r)
            results += [y, mean, invstd, *run, *(t for t in ops.batch_norm_bwd(x, dy, gamma, beta, mean, invstd, 1e-5, True, r) if t is not None)]
    _are(names, _ran(shape, dtype, ("fwd", "bwd", "fwd_res", "bwd_res") * 2))
    half = len(results) // 2
    assert all(torch.equal(a, b) for a, b in zip(results[:half], results[half:]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_statistics_are_rounded_at_their_end(dtype):
    """Over 256 channels' root mean square: 1/deviation carries its own last roundings (the variance's, the root's, the quotient's: 0.3
    of 2^-23 each, the variance's halved) and next to nothing of the 401408 additions in front, the mean its last one at most.
    A thread's elements one behind the other and the channel's words added in fp32 gave two and three times as much."""
    errors = torch.zeros(2, dtype=torch.float64, device="cuda")
    for seed in range(4):
        x = (torch.randn(128, 64, 56, 56, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda") * 1.5 + 0.3).to(dtype)
        run = [torch.zeros(64, device="cuda"), torch.ones(64, device="cuda")]
        _, mean, invstd = ops.batch_norm_fwd(x, torch.ones(64, device="cuda"), torch.zeros(64, device="cuda"), *run, 1e-5, 0.1, False, None)
        assert "_held" in capi.bn_last_kernel_name()
        exact = x.double()
        m, i = exact.mean((0, 2, 3)), (exact.var((0, 2, 3), unbiased=False) + 1e-5).rsqrt()
        errors += torch.stack([((mean.double() - m) * i).square().mean(), (invstd.double() / i - 1).square().mean()])
    errors = (errors / 4).sqrt()
    assert float(errors[0]) < 2.0 ** -25 and float(errors[1]) < 2.0 ** -24, errors.tolist()
