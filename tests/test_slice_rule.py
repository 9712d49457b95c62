"""Which passes run in reduction slices, read from the workspace they ask for (no device): the partial tensors of a sliced
fp16 pass have the tensors' type, so slicing rounds a result twice.  A faster kernel or a wider tile must not cut a pass
that its tiles' area (fp16 arithmetic) or the plan for the fp32 matrix instructions (fp32 arithmetic) leaves whole."""
import pytest
import torch

import phoenix_core_amd as phx
from phoenix_core_amd import capi

FWD, DGRAD = capi.PHX_PASS_FWD, capi.PHX_PASS_BWD_DATA


class Ctx:
    memory_optimized = False
    product_mode = capi.PHX_PRODUCT_8

    def __init__(self, policy):
        self.fp16_policy = {"full16": capi.PHX_FP16_FULL16, "backward32": capi.PHX_FP16_BACKWARD32, "fp32": capi.PHX_FP16_FULL32}[policy]


def workspaces(case, which, tune_env):
    """(workspace as planned, workspace with slices off)"""
    n, ci, co, h, w, k, stride, policy = case
    desc = phx.Conv2DDescriptor((4 * n, ci, h, w), (4, co, ci, k, k), stride, 1, "SAME", dtype=torch.float16, context=Ctx(policy))
    tune_env(PHX_TUNE_KSLICES=None)
    planned = desc.workspace_bytes(which)
    tune_env(PHX_TUNE_KSLICES="0")
    whole = desc.workspace_bytes(which)
    tune_env(PHX_TUNE_KSLICES=None)
    return planned, whole


# n, ci, co, h, w, k, stride, policy, pass: wide tiles of dealt lanes on at most half of the CUs; the phases of a strided
# input gradient on them; strided input gradients in fp32 arithmetic, whose phases the fp32 instructions leave whole
WHOLE = [((16, 256, 256, 14, 14, 3, 1, "full16"), FWD), ((16, 256, 256, 14, 14, 3, 1, "full16"), DGRAD),
         ((16, 256, 256, 12, 12, 3, 1, "full16"), FWD), ((8, 192, 192, 20, 20, 5, 1, "full16"), FWD),
         ((11, 320, 512, 14, 14, 3, 1, "full16"), DGRAD), ((16, 192, 320, 12, 12, 3, 1, "backward32"), FWD),
         ((48, 64, 256, 28, 28, 5, 2, "full16"), DGRAD),
         ((2, 32, 128, 56, 43, 3, 3, "backward32"), DGRAD), ((3, 48, 256, 56, 30, 2, 3, "fp32"), DGRAD)]


@pytest.mark.parametrize("case,which", WHOLE, ids=lambda v: "_".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_passes_that_run_whole(case, which, tune_env):
    planned, whole = workspaces(case, which, tune_env)
    assert planned == whole


# few workgroups and a long reduction: these stay sliced, the last two because a tile of whole images is preferred to
# tiles of single rows that would occupy more CUs for as long
SLICED = [((1, 512, 512, 7, 7, 3, 1, "full16"), FWD, 2), ((1, 512, 512, 7, 7, 3, 1, "full16"), DGRAD, 2),
          ((4, 512, 512, 7, 7, 3, 1, "full16"), FWD, 2), ((8, 256, 256, 14, 14, 3, 1, "full16"), FWD, 2),
          ((1, 512, 512, 7, 7, 3, 1, "fp32"), FWD, 2),
          ((24, 256, 24, 4, 20, 2, 1, "full16"), FWD, 8),
          ((128, 128, 24, 7, 7, 3, 1, "full16"), FWD, 4)]


@pytest.mark.parametrize("case,which,slices", SLICED, ids=lambda v: "_".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_passes_that_run_in_slices(case, which, slices, tune_env):
    planned, whole = workspaces(case, which, tune_env)
    n, ci, co, h, w, k, stride = case[:7]
    outputs = 4 * n * co * -(-h // stride) * -(-w // stride) if which == FWD else 4 * n * ci * h * w
    assert planned >= slices * outputs * 2 and planned != whole  # (that many partial tensors at least)


@pytest.mark.parametrize("case,which", [(c, w) for c, w, _ in SLICED], ids=str)
def test_slices_keep_32_channels(case, which, tune_env):
    """A slice's sums are rounded to the tensors' type: one per 32 reduced channels at most, also where slices are asked for."""
    _, whole = workspaces(case, which, tune_env)
    n, ci, co, h, w, k, stride, policy = case
    desc = phx.Conv2DDescriptor((4 * n, ci, h, w), (4, co, ci, k, k), stride, 1, "SAME", dtype=torch.float16, context=Ctx(policy))
    red = ci if which == FWD else co
    tune_env(PHX_TUNE_KSLICES=str(red // 16))
    assert desc.workspace_bytes(which) == whole
    tune_env(PHX_TUNE_KSLICES=str(red // 32))
    assert desc.workspace_bytes(which) != whole
