"""Which passes run as matrix products (phx_launch_dense_gemm.hip), read from the workspace they ask for (no device)."""
import pytest
import torch

import phoenix_core_amd as phx
from phoenix_core_amd import capi
from test_slice_rule import Ctx

WGRAD = capi.PHX_PASS_BWD_WEIGHTS


def _dense(n, ci, co, dtype):
    return phx.DenseDescriptor((4 * n, ci), (4, ci, co), dtype=dtype, context=Ctx("full16"))


def _pointwise(n, ci, co, h, w, layout):
    shape = (4 * n, ci, h, w) if layout == "NCHW" else (4 * n, h, w, ci)
    return phx.Conv2DDescriptor(shape, (4, co, ci, 1, 1), dtype=torch.float32, context=Ctx("fp32"), data_format=layout)


@pytest.mark.parametrize("desc,which", [(_dense(300, 700, 500, torch.float32), capi.PHX_PASS_FWD), (_dense(768, 512, 512, torch.float32), capi.PHX_PASS_BWD_DATA),
                                        (_dense(768, 512, 512, torch.float32), WGRAD), (_pointwise(32, 96, 96, 56, 56, "NCHW"), WGRAD),
                                        (_pointwise(32, 96, 96, 56, 56, "NHWC"), WGRAD)], ids=["fwd", "dgrad", "wgrad", "planes", "channels_last"])
def test_the_fp32_instructions_on_request(desc, which, tune_env):
    """PHX_TUNE_NOX3 keeps everything in fp32 off the bf16 instructions, these products too."""
    sizes = []
    for variables in ({}, {"PHX_TUNE_NOX3": "1"}, {"PHX_TUNE_NOX3": "1", "PHX_TUNE_NODENSEGEMM": "1"}):
        tune_env(**{"PHX_TUNE_NOX3": None, "PHX_TUNE_NODENSEGEMM": None, **variables})
        sizes.append(desc.workspace_bytes(which))
    assert sizes[1] == sizes[2] != sizes[0]


def test_fp16_products_are_not_concerned(tune_env):
    desc = _dense(300, 700, 500, torch.float16)
    planned = desc.workspace_bytes(capi.PHX_PASS_FWD)
    tune_env(PHX_TUNE_NOX3="1")
    assert desc.workspace_bytes(capi.PHX_PASS_FWD) == planned


def _searched(rows, columns, reduced, images):
    """The slices of an fp32 filter gradient, by the planner's estimate over every slice count."""
    chunks, best, slices = -(-reduced // 16) * max(images, 1), float("inf"), 1
    tiles = -(-rows // 64) * -(-columns // 64)
    for z in range(1, min(chunks, 512 if images else 64) + 1):
        per = -(-chunks // z)
        if -(-chunks // per) != z:
            continue
        full, rest = divmod(-(-tiles * z // 256), 2)
        us = 4.0 + per * (full * 5.7 + (3.4 + (rest - 1) * 2.3 if rest else 0.0))
        us += 4.0 + (z + 0.5) * 32.0 * rows * columns / 3.0e6 if z > 1 else 0.0
        if us < best:
            best, slices = us, z
    return slices


@pytest.mark.parametrize("n,ci,co,h,w", [(32, 96, 96, 56, 56), (4, 256, 64, 56, 56), (1, 100, 97, 2, 2), (64, 256, 256, 14, 14), (7, 512, 130, 13, 9)])
def test_slices_are_those_of_the_whole_search(n, ci, co, h, w):
    z = _searched(ci, co, h * w, n)
    assert _pointwise(n, ci, co, h, w, "NCHW").workspace_bytes(WGRAD) == (z * 16 * ci * co if z > 1 else 0)
    z = _searched(ci, co, n * h * w, 0)
    assert _dense(n * h * w, ci, co, torch.float32).workspace_bytes(WGRAD) == (z * 16 * ci * co if z > 1 else 0)
