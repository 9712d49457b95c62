"""Windows of unit stride that the models of both sides send to the fp16 kernel on registers (csrc/phx_kernels_reg16.h): few
channels in their chunks, ragged and odd extents, spans of six pixels, dilation; against the oracle, on the plan's own split."""
import pytest

import test_gpu_reg16

pytestmark = pytest.mark.gpu

# n, ci, co, h, w, kh, kw, stride, dilation, padding
CASES = [
    (3, 24, 24, 35, 13, 5, 5, 1, 1, "SAME"),         # 24 of 32 channels, wide spans
    (15, 39, 39, 8, 8, 3, 3, 1, 1, "SAME"),          # 39 of 64: seven in the last chunk
    (4, 17, 33, 13, 21, 5, 5, 1, 1, "SAME"),         # one channel beyond two and one beyond three tiles of 16
    (9, 40, 21, 9, 17, 3, 3, 1, 1, "SAME"),          # an odd plane
    (9, 24, 40, 10, 11, 3, 3, 1, 2, "SAME"),         # dilated rows
    (17, 36, 20, 12, 10, 5, 3, 1, 1, "VALID"),        # five rows of three taps
]


@pytest.mark.parametrize("layout", ["NCHW", "NHWC"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "n%d_%d-%d_%dx%d_%dx%d_s%s_d%s_%s" % c)
def test_the_plans_own_split(case, layout, tune_env):
    print(case, layout, flush=True)
    test_gpu_reg16.test_against_the_oracle(case, None, layout, tune_env)
