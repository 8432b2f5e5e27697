"""The kernel names by which bench.py looks up measured traffic are names of
kernels in the library, and every stencil kernel of it is in a class."""
import os
import re
import subprocess

import pytest

import ddx
from conftest import PKG, ROOT

import sys

sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.fixture(scope="module")
def kernels():
    out = subprocess.run(["nm", "-C", os.path.join(PKG, "lib", "libddx.so")], capture_output=True, text=True, check=True)
    names = set(re.findall(r"ddx::__device_stub__(\w+(?:<[^(]*>)?)\(", out.stdout))
    assert names
    return names


class Bricks:
    def __init__(self, *shape):
        self.shape = shape

    def brick(self, kernel, mode):
        return self.shape


@pytest.mark.parametrize("storage,shape", [("fp32", (64, 4, 1, 8, 1)), ("fp32", (64, 4, 1, 2, 2)),
                                           ("fp32", (64, 8, 1, 4, 3)), ("fp32", (64, 8, 1, 2, 4)),
                                           ("bf16", (64, 4, 1, 4, 1)), ("fp16", (32, 8, 1, 4, 2))])
def test_brick_kernel_names_are_kernels(storage, shape, kernels):
    modes = [ddx.PURE_FORWARD, ddx.RTM_FORWARD, ddx.RTM_BACKWARD, ddx.RTM_REVERSE]
    for k in (0, 1):
        for name in bench.brick_kernel_names(Bricks(*shape), k, modes, storage):
            assert name.replace("ddx::", "", 1) in kernels, name
            assert bench.kernel_class(f"void {name}(ddx::PhyDesc const*)") == k


def test_every_stencil_kernel_has_a_class(kernels):
    """All but the copies, the receivers' and sources' kernels and those that
    run once per shot."""
    small = ("k_copy", "k_save", "k_inject", "k_ring", "k_recv", "k_source", "k_set_int", "k_advance", "k_nonfinite",
             "k_laplace", "k_compensate")
    for k in kernels:
        if not k.startswith(small):
            assert bench.kernel_class("void ddx::" + k) is not None, k
