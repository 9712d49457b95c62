"""The factorized fp16 kernel whose waves own two product lanes each: at the edges of its tiles, windows and staging it
gives bit for bit what the kernel that forms all lanes in every wave gives (the same products in the same order), and
both agree with the oracle."""
import numpy as np
import pytest
import torch

import oracle
import phoenix_core_amd as phx
from phoenix_core_amd import capi, ops

from test_gpu_parity import Ctx, assert_close, make_inputs, name_seed

pytestmark = pytest.mark.gpu

# name, n, ci, co, h, w, kh, kw, stride, dilation, padding, channels-last
CASES = [
    ("window_of_256", 1, 48, 64, 6, 30, 3, 3, 1, 1, "SAME", False),        # 8 rows of 32: the window starts a column early, all of it used
    ("row_end_shared", 3, 40, 70, 14, 14, 3, 3, 1, 1, "SAME", False),      # 16 columns of window for 14 + 2: one more would not fit
    ("odd_width", 2, 34, 48, 9, 13, 3, 3, 1, 1, "SAME", False),            # 2-byte aligned loads
    ("one_chunk_many_images", 40, 8, 64, 7, 7, 3, 3, 1, 1, "SAME", False),  # 7x7 planes: tensor ends inside loads, runs of any length
    ("asym_pad_gap", 4, 33, 100, 11, 12, 3, 3, 1, 1, (0, 2, 2, 0), False),
    ("k5_dil2", 1, 48, 64, 20, 24, 5, 5, 1, 2, "SAME", False),             # nine groups of taps, two of them padding
    ("k4x2_stride2", 2, 64, 96, 19, 22, 4, 2, 2, 1, "SAME", False),        # eight taps: one of them padding
    ("tall_1px", 5, 32, 64, 1, 1, 3, 3, 1, 1, "SAME", False),
    ("cl_ragged", 3, 56, 72, 13, 11, 3, 3, 1, 1, "SAME", True),
    ("cl_wide", 1, 40, 64, 4, 60, 3, 3, 1, 1, "SAME", True),
]


@pytest.mark.parametrize("tile", ["2,2", "2,1"], ids=["px128", "px64"])
@pytest.mark.parametrize("flat", [False, True], ids=["tiles", "flat"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: c[0])
def test_lanes_dealt_over_the_waves(case, flat, tile, tune_env):
    name, n, ci, co, h, w, kh, kw, stride, dilation, padding, cl = case
    if flat and stride != 1:
        pytest.skip("flat tiling is for unit stride")
    dtype = torch.float16
    g, x, wt, b, gr = make_inputs(name_seed(name) + 5, n, ci, co, h, w, kh, kw, stride, dilation, padding, dtype, 0.5)
    to_dev = (lambda a: np.ascontiguousarray(a.transpose(0, 2, 3, 1))) if cl else (lambda a: a)
    back = (lambda a: a.transpose(0, 3, 1, 2)) if cl else (lambda a: a)
    desc = phx.Conv2DDescriptor(to_dev(x).shape, wt.shape, stride, dilation, padding, use_bias=True, dtype=dtype,
                                context=Ctx(8, "full16"), data_format="NHWC" if cl else "NCHW")
    xd, wd, bd, gd = (torch.from_numpy(a).cuda() for a in (to_dev(x), wt, b, to_dev(gr)))
    # (ZI8: problems of few channels stay in factorized form; dilation phases and reduction slices off)
    base = dict(PHX_TUNE_TILE=tile, PHX_TUNE_ZI8="1", PHX_TUNE_KSLICES="0", PHX_TUNE_NODILPHASE="1",
                PHX_TUNE_FLAT="1" if flat else None, PHX_TUNE_NOFLAT=None if flat else "1")
    dgrad = ci > 32 and stride == 1  # (at most 32 channels have no tile of two sub-tiles, zero-inserted windows none of this shape)
    got = {}
    for dealt in (True, False):
        tune_env(**base, PHX_TUNE_NOLANES=None if dealt else "1")
        y = phx.conv2d_fwd(xd, wd, bd, desc)
        names = [capi.last_kernel_name()]
        dx = ops.conv2d_bwd_data(wd, gd, desc) if dgrad else gd
        names.append(capi.last_kernel_name())
        packed = ops.conv2d_pack_filters(wd, desc, bwd_data=dgrad)
        assert torch.equal(phx.conv2d_fwd(xd, torch.zeros_like(wd), bd, desc, packed=packed), y)
        assert names[0].endswith("_lanes") == dealt and (not dgrad or names[1].endswith("_lanes") == dealt), names
        got[dealt] = (y, dx)
    assert torch.equal(got[True][0], got[False][0]), "fwd " + name
    assert torch.equal(got[True][1], got[False][1]), "dgrad " + name
    x64, w64, b64, g64 = (a.astype(np.float64) for a in (x, wt, b, gr))
    assert_close(back(got[True][0].cpu().numpy()), oracle.conv2d_fwd(g, x64, w64, b64, "hamilton"), dtype, "fwd " + name)
    if dgrad:
        assert_close(back(got[True][1].cpu().numpy()), oracle.conv2d_bwd(g, x64, w64, g64, "hamilton")[1], dtype, "dgrad " + name)
