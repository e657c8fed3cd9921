"""The rule that sends an fp16 product of the block to the MFMA kernel or to
hipBLASLt, by its sizes, and the kernel's tile plans; nothing is launched.

The rule is held to the measurement it comes from: profiles/
inner_product_sweep.json has each of the model's four products at row counts
from 256 to 21658 on both, against the two hipBLASLt builds a process may map
(torch's and ROCm's)."""
from __future__ import annotations

import ctypes
import json
from pathlib import Path

import pytest

SWEEP = Path(__file__).resolve().parent.parent / "profiles" / "inner_product_sweep.json"
EPILOGUES = ("store", "residual", "swiglu")
PRODUCTS = json.loads(SWEEP.read_text())


@pytest.mark.parametrize("build", ["torch", "rocm"])
@pytest.mark.parametrize("product", PRODUCTS, ids=lambda p: f"{p['epilogue']}-{p['in']}-{p['out']}")
def test_rule_against_the_measured_products(hip, product, build):
    """Where the rule takes the kernel it is never more than 6% behind the
    library, which picks its own tile and now and then a good one where the
    kernel's plan leaves CUs idle, and it is ahead on average."""
    epilogue = EPILOGUES.index(product["epilogue"])
    gains = {}
    for rows, lib, ker in zip(product["rows"], product[f"{build}_library_us"], product[f"{build}_kernel_us"]):
        if hip.inner_product_f16_plan(rows, product["in"], product["out"], epilogue, block=True)[0] and lib is not None:
            gains[rows] = lib / ker
    assert len(gains) >= 10
    assert min(gains.values()) > 0.94, sorted(gains.items(), key=lambda kv: kv[1])[:5]
    assert sum(gains.values()) / len(gains) > 1.01


def test_few_rows_and_other_shapes_go_to_the_library(hip):
    for epilogue in range(3):
        assert not hip.inner_product_f16_plan(255, 2560, 7680, epilogue, block=True)[0]
    assert hip.inner_product_f16_plan(255, 2560, 7680)[0]  # the entry point itself has one kernel
    assert hip.inner_product_f16_plan(4096, 132, 2560, block=True) == (False, 0, None)  # in % 64
    assert hip.inner_product_f16_plan(4096, 2560, 64, block=True) == (False, 0, None)   # out % 256


def test_plans_of_the_entry_point(hip):
    """Products rounded to fp16 are summed in one order in every form: none
    of their plans splits K."""
    for rows in range(1, 4000, 37):
        for k, n in ((2560, 2560), (6912, 2560), (2560, 7680), (64, 256)):
            for epilogue in (hip.EPI_STORE, hip.EPI_RESIDUAL):
                kernel, first, form = hip.inner_product_f16_plan(rows, k, n, epilogue)
                assert kernel and first % 256 == 0 and 0 <= first < rows and form != "128x128-ksplit"


def test_plan_argument_checks(hip):
    lib = hip.load()
    plan = (ctypes.c_int * 3)()
    f = lib.sv2_inner_product_f16_plan
    assert f(4, 64, 256, hip.EPI_STORE, 0, None) == hip.SV2_EINVAL
    assert f(0, 64, 256, hip.EPI_STORE, 0, plan) == hip.SV2_EINVAL
    assert f(4, 64, 256, 3, 0, plan) == hip.SV2_EINVAL
    assert f(4, 48, 256, hip.EPI_STORE, 0, plan) == hip.SV2_EUNSUPPORTED
    assert f(1 << 24, 64, 256, hip.EPI_STORE, 0, plan) == hip.SV2_EUNSUPPORTED  # X of 2 GiB
    assert f(4, 48, 256, hip.EPI_STORE, 1, plan) == hip.SV2_OK and plan[0] == 0 and plan[2] == -1


def test_forms_of_the_residual_products(hip):
    """The forms the blocks' residual products reach: proj in one launch of
    K-split tiles, out in 256 x 256 tiles alone, with a K-split rest and with a
    256 x 128 one; and a count (16961) that is the library's, whose build in
    torch has no kernel for out there."""
    plan = lambda rows, k: hip.inner_product_f16_plan(rows, k, 2560, hip.EPI_RESIDUAL, block=True)
    assert plan(1224, 2560) == (True, 0, "128x128-ksplit")
    assert plan(18881, 6912) == (True, 0, "256x256")
    assert plan(20161, 6912) == (True, 19456, "128x128-ksplit")
    assert plan(21658, 6912) == (True, 19456, "256x128")
    assert plan(16961, 6912) == (False, 0, "256x256")
