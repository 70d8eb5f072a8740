"""The GPU tests of the convolutions over the flattened batch reach every variant that is compiled: the library's plan for their
shapes, asked without a GPU, against the lists in the sources."""
import os
import re

import pytest

import test_gpu_conv_f32
import test_gpu_conv_few
from test_conv_plan import conv_plan

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tannic_amd", "csrc")


def test_fp32_variants_are_all_reached():
    source = open(os.path.join(CSRC, "conv2d_f32.hip")).read()
    compiled = set()
    for side, u, pt, nl, wo, wide in re.findall(r"\bF\((\d), (\d), (\d+), (\d+), (?:true|false), (\d), (WIDE|true|false)\)", source):
        for w in ((0, 1) if wide == "WIDE" else (int(wide == "true"),)):
            compiled.add((int(side), int(u), int(pt), int(nl), int(wo), w))
    assert len(compiled) > 40 and compiled == set(test_gpu_conv_f32.VARIANTS)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_variants_are_the_plan_of_their_shapes(dtype):
    for variant, (x, w, stride) in test_gpu_conv_few.VARIANTS.items():
        kernel, plan = conv_plan(dtype, x, w, (stride, stride), (w[2] // 2,) * 2)
        assert kernel == "few" and tuple(plan[n] for n in ("side", "mo", "np", "waves")) == variant
    for variant, (x, w, stride) in test_gpu_conv_f32.VARIANTS.items():
        kernel, plan = conv_plan("float32", x, w, (stride, stride), (w[2] // 2,) * 2)
        assert kernel == "f32" and tuple(plan[n] for n in ("side", "u", "pt", "nl", "wo", "wide")) == variant


def test_few_pixel_variants_are_all_reached():
    # one tile; two of pixels (1x1) or of channels (3x3, a stride); four, up to eight wavefronts
    shapes = {1: ((1, 1), (1, 2), (2, 1), (2, 2)), 3: ((1, 1), (2, 1), (2, 2))}
    compiled = {(side, *tiles, waves) for side in shapes for tiles in shapes[side] for waves in (2, 4, 8, 16) if waves <= 8 or tiles != (2, 2)}
    assert compiled == set(test_gpu_conv_few.VARIANTS)
