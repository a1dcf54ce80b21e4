"""csrc/midpoints.h, built with the host compiler: for which pre-scales no 16-bit value times the pre-scale comes near a midpoint
between two E2M1 values, against every value's product."""
import ctypes
import math
import os
import subprocess

import numpy as np
import pytest
import torch

from conftest import PKG


@pytest.fixture(scope="module")
def never(tmp_path_factory):
    d = tmp_path_factory.mktemp("midpoints")
    (d / "t.cpp").write_text('#include "%s"\nextern "C" int never(float pre, int digits) { return never_near_midpoint(pre, digits); }\n' % os.path.join(PKG, "csrc", "midpoints.h"))
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-shared", "-fPIC", "-o", str(d / "t.so"), str(d / "t.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "t.so"))
    lib.never.argtypes = [ctypes.c_float, ctypes.c_int]
    return lambda pre, dtype: bool(lib.never(pre, 8 if dtype is torch.bfloat16 else 11))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_no_product_has_the_pattern(never, dtype):
    values = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).float().numpy()
    values = values[np.isfinite(values) & (values != 0)]
    rng, seen = np.random.default_rng(2), set()
    pres = [math.log2(math.e) * d ** -0.5 for d in (32, 64, 72, 80, 96, 128, 256)] + [1.25 / (1 + 5 / 128), 0.1, -0.7, 3.0, 1e-30, 1e30]
    pres += list(np.exp2(rng.uniform(-20, 20, 300))) + list(1.25 / (1 + np.arange(0, 1024, 37) / 1024))
    for pre in np.asarray(pres, dtype=np.float32):
        with np.errstate(over="ignore", under="ignore"):
            x = values * pre
        x = x[(np.abs(x) >= 2.0 ** -126) & np.isfinite(x)]
        near = ((x.view(np.uint32) << np.uint32(11)) + np.uint32(128 << 11)) < np.uint32(256 << 11)
        assert never(float(pre), dtype) == (not near.any()), pre
        seen.add(bool(near.any()))
    assert seen == {True, False}


def test_what_is_no_normal_number_is_not_sure(never):
    for pre in (0.0, -0.0, 1e-40, float("inf"), float("nan")):
        assert not never(pre, torch.bfloat16) and not never(pre, torch.float16)
