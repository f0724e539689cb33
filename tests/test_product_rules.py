"""What kernels' rules and entries take and refuse, which needs no GPU."""
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


@pytest.mark.parametrize("name", ["attention_mfma", "attention_mfma_bias", "attention_mfma_cap"])
def test_waves_of_the_decode_attention(name):
    """Eight waves a workgroup where every workgroup has a compute unit of its own, four beyond (256 requests of some 129 keys took twice as long with eight), for sixteen
    rows, and for parts of heads of 128 that fill more than half of the chip."""
    waves = lambda *a, lengths=0: build.load(name).lcu_attention_decode_waves(*a, lengths)
    for dh in (32, 64, 96, 128):
        assert [waves(n, 16, 16, dh, 1, 256) for n in (1, 16, 17, 256)] == [8, 8, 4, 4]
        assert [waves(n, 32, 8, dh, 1, 256) for n in (32, 33)] == [8, 4] and waves(33, 32, 8, dh, 1, 304) == 8
        assert [waves(1, g, 1, dh, 1, 256) for g in (15, 16, 17, 32)] == [8, 4, 4, 4]
        assert [waves(n, 32, 8, dh, 4, 256) for n in (4, 5, 8, 9)] == [8, 8, 8, 4]
        assert [waves(n, 32, 8, dh, 4, 256, lengths=2) for n in (4, 5, 8, 9)] == [8, 4 if dh == 128 else 8, 4 if dh == 128 else 8, 4]
        assert waves(1, 32, 8, dh, 1, 0) == 4                  # (a device that does not say how many units it has)
        assert [waves(n, 32, 8, dh, 1, 256, lengths=2) for n in (32, 33, 64, 65)] == [8, 8, 8, 4] and waves(33, 32, 8, dh, 2, 256, lengths=2) == 4
        assert waves(1, 32, 8, dh, 1, 256, lengths=1) == 4 and waves(40, 16, 1, dh, 1, 256, lengths=2) == 4


def test_requests_whose_longest_has_many_keys():
    """Where the decode attention's workgroups are one to two a compute unit, and where parts of heads of 128 fill more than half of the chip; not for layers that see a window of fewer keys."""
    long = ops.decode_long
    if ops.TUNING.compute_units != 256:
        pytest.skip("the lines are those of 256 compute units")
    assert [long(n, 32, 8, 64, 1025) for n in (32, 33, 64, 65)] == [False, True, True, False] and not long(64, 32, 8, 64, 1024)
    assert not long(64, 32, 8, 128, 4000, 1024) and not long(64, 32, 8, 128, 4000, -128) and long(64, 32, 8, 128, 4000, 1025) and not long(300, 16, 1, 64, 4000) and long(300, 15, 1, 64, 4000)
    assert not long(8, 32, 8, 128, 3072) and long(8, 32, 8, 128, 3073) and not long(8, 32, 8, 96, 3073) and long(16, 32, 8, 128, 1537) and not long(16, 32, 8, 128, 1537, 1536)
    assert not long(4, 32, 8, 128, 3073) and long(4, 32, 8, 128, 6145) and not long(1, 32, 8, 128, 24576) and long(1, 32, 8, 128, 24577) and not long(8, 32, 8, 128, 1537, 0, 4) and long(8, 32, 8, 128, 1537, 0, 2) == False


def test_short_steps_do_not_ask_for_many_keys():
    """Up to the number of keys that a step looks at first no sizes count on many; behind it some do."""
    least = ops.decode_long_from()
    sizes = [(n, nh, nkv, dh) for n in (1, 7, 8, 33, 64, 300) for nh, nkv in ((32, 8), (16, 4), (40, 8), (15, 1)) for dh in (64, 128)]
    assert not any(ops.decode_long(*z, least) for z in sizes) and any(ops.decode_long(*z, least + 1) for z in sizes)


def test_parts_of_few_requests():
    """One part up to 512 keys, eight beyond as far as the chip has compute units for them, longer ones from 4,097 keys on."""
    splits = ops.decode_splits
    assert [splits(1, 16, 4, c) for c in (1, 512, 513, 1024, 1025, 4096, 4097)] == [1, 1, 8, 8, 8, 8, 16]
    assert [splits(n, 16, 4, 513) for n in (8, 9, 16, 32, 33)] == [8, 7, 4, 2, 1] and splits(32, 16, 4, 512) == 1


def test_experts_of_few_pairs():
    """Which products of a step's first pairs go to the kernel that holds the named experts' workgroups alone: at its edges (16 tokens, 64 pairs, 256 workgroups, or 384 where most experts
    have no pair, a dozen pairs an expert)."""
    takes = build.load("moe").lcu_moe_slots_take
    assert takes(1, 2, 16, 2048) and takes(16, 2, 40, 64) and not takes(17, 1, 40, 64) and takes(16, 4, 64, 64) and not takes(16, 5, 80, 64)
    assert takes(12, 1, 24, 1024) and not takes(12, 1, 24, 1025) and takes(12, 1, 23, 672) and not takes(12, 1, 23, 1024)
    assert takes(12, 4, 4, 1024) and not takes(13, 4, 4, 1024) and not takes(16, 4, 4, 1024) and takes(12, 1, 1, 1024) and not takes(13, 1, 1, 1024)


def test_what_the_recurrence_with_a_bonus_asks_for_in_front():
    """All of it, unless that takes another round of workgroups: heads of up to 64, of which a compute unit holds five then and six otherwise."""
    front = lambda *a: bool(build.load("wkv").lcu_wkv_front(*a))
    assert [front(n, 1, 64, 256) for n in (1, 1280, 1281, 1536, 1537, 2560, 2561, 3072, 3073)] == [True, True, False, False, True, True, False, False, True]
    assert not front(128, 12, 48, 256) and front(128, 12, 65, 256) and front(128, 12, 48, 0)


@pytest.mark.parametrize("m,n,k,swiglu,shape", [
    (341, 6144, 2048, False, -1), (342, 6144, 2048, False, 0), (300, 6144, 1024, False, 0), (363, 5632, 2048, True, 0), (297, 5632, 2048, True, -1), (299, 5632, 2048, True, 0),      # rows that fill half, or two fifths
    (3073, 768, 2112, False, -1), (3073, 768, 2048, False, 0), (1536, 1024, 2112, False, -1), (2304, 1536, 2048, False, 0), (2433, 1536, 2048, False, -1),                       # few features
    (1843, 2048, 4096, False, 0), (1844, 2048, 4160, False, -1), (1843, 2048, 4160, False, 0), (800, 4096, 4160, False, 0), (1117, 2048, 14336, False, -1), (513, 4096, 14336, False, 0), (1004, 2560, 11008, False, -1),     # long sums
    (2049, 2048, 1984, False, 1), (2049, 2048, 2048, False, -1), (2305, 2048, 2048, False, 1), (1400, 3072, 2048, False, -1), (1400, 3072, 1984, False, 1),                                                    # 128 x 256
    (1861, 5632, 2048, True, -1), (1862, 5632, 2048, True, 2), (1400, 5632, 960, True, 2), (1400, 5632, 1024, True, -1)])                                                        # 256 x 256
def test_where_the_library_s_tiles_fit_better(m, n, k, swiglu, shape):
    """On both sides of the lines behind which many rows in tiles stay with the library, on a card of 256 compute units."""
    if ops.TUNING.compute_units != 256:
        pytest.skip("the lines are those of 256 compute units")
    assert ops.tiles_choice(m, n, k, swiglu) == shape
