"""The one-pass batch-norm kernels, whose workgroups hold their part of a channel in registers and wait for their neighbours'
sums, at the edges of their plan: planes of one 16-byte chunk and of one element more, a partial last chunk in every plane, one
workgroup a channel, as many as ask for 512 threads, and more than 64 of those, which stay on two launches.  Against fp64 with
test_gpu_bn's tolerances; with no wait allowed every workgroup forms the channel's sums itself, and the results are the same."""
import pytest
import torch

import test_gpu_bn
from phoenix_core_amd import ops

pytestmark = pytest.mark.gpu

SHAPES = [(8, 16, 14, 14), (12, 5, 7, 7), (64, 33, 9, 5), (2, 3, 2, 4), (5, 1100, 3, 3), (65, 2, 4, 8), (37, 6, 31, 17), (1, 1, 64, 96), (257, 1, 40, 41),
          (700, 2, 21, 20), (330, 1, 56, 57), (40, 512, 7, 7)]


@pytest.fixture(params=["4096", "0"], ids=["waits", "alone"])
def held(request, tune_env):
    tune_env(PHX_TUNE_BN_HELD="1", PHX_TUNE_BN_WAITS=request.param)


@pytest.mark.parametrize("relu,residual", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_one_pass_matches_torch(held, shape, dtype, relu, residual):
    test_gpu_bn.test_batch_norm_matches_torch(shape, dtype, relu, residual)


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
@pytest.mark.parametrize("shape", [(64, 33, 9, 5), (37, 6, 31, 17), (700, 2, 21, 20)], ids=lambda s: "x".join(map(str, s)))
def test_results_do_not_depend_on_who_forms_the_sums(shape, dtype, tune_env):
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
    half = len(results) // 2
    assert all(torch.equal(a, b) for a, b in zip(results[:half], results[half:]))
