"""Launch arithmetic (csrc/pxh_launch.h) at the ends of its range: the items are
capacities of buffers that grow on demand, so every int is a size that can occur."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "physx_amd", "csrc")
SOURCE = """
#include "pxh_launch.h"
extern "C" int stride_blocks(long long items, int per, int most) { return pxh::strideBlocks(items, per, most); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch")
    (d / "launch.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-ftrapv", "-I", CSRC, str(d / "launch.cpp"), "-o",
                    str(d / "liblaunch.so")], check=True)
    return ctypes.CDLL(str(d / "liblaunch.so"))


@pytest.mark.parametrize("per,most", [(4, 16384), (4, 8192), (64, 2048), (256, 1024)])
@pytest.mark.parametrize("items", [1, 3, 4, 5, 65, 2**27 - 1, 2**27, 2**27 + 1, 2**31 - 1])
def test_stride_blocks(lib, items, per, most):
    assert lib.stride_blocks(ctypes.c_longlong(items), per, most) == min(-(-items // per), most)


def test_convex_launches_use_it():
    """every launch over the convex pairs' capacity takes its blocks from there"""
    src = open(os.path.join(CSRC, "pxh_kernels.hip")).read()
    body = src[src.index("void launch_np_convex("):]
    body = body[:body.index("\n}\n")]
    assert body.count("strideBlocks(cap,") == 3 and "cap *" not in body
