"""What the products' rules and entries take and refuse, which needs no GPU."""
from __future__ import annotations

import ctypes
import shutil
import subprocess

import pytest
import torch

from llama_cu_amd.kernels import build, ops


def rows(m, k, device="cpu"):
    return torch.empty(m, k, dtype=torch.bfloat16, device=device)


def test_operands_that_are_not_on_one_gpu():
    """The kernel takes addresses, so operands in host memory, or on two devices, are left to the library, which refuses them."""
    for x, w in ((rows(300, 2048), rows(2048, 2048)), (rows(300, 2048, "meta"), rows(2048, 2048)), (rows(300, 2048), rows(2048, 2048, "meta"))):
        assert not ops.tiles_supported(x, w)


def test_products_over_nothing():
    """A sum of no terms is zeros, which the library gives; the kernel refuses it."""
    for swiglu in (False, True):
        assert ops.tiles_choice(1100, 2048, 0, swiglu) == -1 and ops.tiles_choice(1100, 0, 2048, swiglu) == -1


def test_the_kernel_asks_for_its_lds():
    """Its tiles take 128 to 160 KB of LDS, and a launch is promised 64 KB unless it asks: the library calls what asks (a runtime that does not hold launches to the
    promise runs the kernel either way)."""
    if not shutil.which("nm"):
        pytest.skip("no nm")
    names = subprocess.run(["nm", "-D", "--undefined-only", build.build("gemm_tiles")], check=True, capture_output=True, text=True).stdout
    assert "hipFuncSetAttribute" in names


def test_rows_that_span_more_than_a_load_reaches():
    """The product that shares rows through LDS refuses rows of 4 GiB and more from the first to the last before it launches anything (the addresses are none)."""
    lib, p, f = build.load("gemm_mid"), ctypes.c_void_p(4096), ctypes.c_float
    apart = (1 << 31) // 99 + 8 & ~7
    for packed, epilogue in ((1, 1), (0, 1), (1, 2), (1, 0)):
        assert lib.lcu_gemm_mid_bf16(p, apart, p, 128, p, 64, 100, 64, 128, epilogue, 1, packed, f(1), f(0), None) == -1
