"""GPU: the flow update where one workgroup transforms a whole plane in x and y (itot, jtot >= 32, at
most 8192 cells), every plane shape, and the shapes and plane counts beside the rule.

The checks and the tolerance are those of tests/test_gpu_flow_lines.py: solver1d against numpy's
transforms and an elimination in 64 bits (1e-12 of the largest value), halos untouched, and the
step's pressure bit for bit fillps and solver1d.
"""
import pytest

import test_gpu_flow_lines as lines

pytestmark = pytest.mark.gpu

SHAPES = [(32, 32, 2), (32, 32, 33), (32, 64, 5), (64, 32, 5), (32, 128, 3), (128, 32, 3), (64, 64, 3),
          (32, 256, 32), (256, 32, 32), (64, 128, 32), (128, 64, 33), (128, 64, 31), (128, 128, 32),
          (16, 64, 32), (64, 16, 32)]


@pytest.mark.parametrize("shape", SHAPES)
def test_planes_match_reference(shape):
    lines.test_line_lengths_match_oracle(shape)
