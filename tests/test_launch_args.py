"""The argument block that a launch passes by value: past 112 bytes a launch takes the host twice
as long (see emit_launch).  Kernels with up to four arrays fit; Hydro's steps, with eight, do
not."""
import ctypes
import re

import pytest

from paraiso_amd import variants
from paraiso_amd.generator import _hip_sources
from test_batch_args import args_type


@pytest.mark.parametrize("name", ["life_i32", "wave3d_f32", "wave3d_f64", "hydro_f32", "hydro_f64"])
def test_small_argument_blocks(name):
    mk, _, precise = variants.VARIANTS[name]
    src = _hip_sources(variants.setup_of(name), mk(), precise)[1]
    seen = 0
    for fn in re.findall(r"struct Args_(\w+) \{", src):
        Args = args_type(src, fn)
        if sum(1 for f, _ in Args._fields_ if re.match(r"(ld|st)\d", f)) <= 4:
            assert ctypes.sizeof(Args) <= 112, fn
            seen += 1
    assert seen >= 2
