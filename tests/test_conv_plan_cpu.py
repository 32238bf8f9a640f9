"""The rules that choose a convolution's kernel, tile and grid (csrc/conv_plan.h), compiled for
the host: the plans stay inside what the kernels and a launch can hold, and the cases of the GPU
tests run the code they name."""
import ctypes
import os
import subprocess

import pytest

from ogle_amd import hip as H
import test_kernels_gpu as K

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("plan") / "probe.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "ogle_amd", "csrc"),
                    os.path.join(ROOT, "tests", "conv_plan_probe.cc"), "-o", so], check=True)
    return ctypes.CDLL(so)


def conv(n, h, w, c, o, k=1, s=1, p=0, d=1, g=1, dtype=H.F32):
    """Plan arguments of a convolution; the pointers are only looked at for their alignment."""
    return H.conv_args(4096, 4096, None, 4096, n, h, w, c, o, k, s, p, d, g, H.ACT_NONE, 0.0, 0.0,
                       H.VARIANT_ANY4 if g > 1 else H.VARIANT_NHWC4, dtype)


PATCH_FIELDS = ("cols", "gp", "cc", "runs", "boxes", "box_blocks", "blocks", "vec_x", "vec_w", "lds_floats")


def patch_plan(probe, *shape, **kw):
    out = (ctypes.c_int64 * len(PATCH_FIELDS))()
    if not probe.probe_patch(ctypes.byref(conv(*shape, **kw)), out):
        return None
    return dict(zip(PATCH_FIELDS, out))


def test_infinite_filter_cases_walk_several_boxes(probe):
    """Of the cases with infinite filter values some give a workgroup one box, some several, one
    stages its channels in chunks."""
    plans = [patch_plan(probe, n, h, w, c, o, k, s, p, 1, g) for n, h, w, c, o, k, s, p, g in K.INFINITE_FILTER_CASES]
    assert [p["boxes"] > p["box_blocks"] for p in plans] == [False, False, True, True]
    assert plans[1]["cc"] < 130
    assert plans[2]["gp"] > 1
    assert plans[3]["runs"] == 1 and plans[3]["cols"] == 64
