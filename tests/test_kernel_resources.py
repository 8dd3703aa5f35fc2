"""Registers and scratch of every compiled kernel form, from the compiler's resource report of the build:
no form that a launch can select spills, and the register bound leaves a CU the workgroups that its LDS
holds.  (The 64-bit addressing form of the 256 x 256 work tile spills; launches route such problems to
the 128 x 128 work tile of the same macro-tile.)"""
import json

import pytest

from grouped_gemm_gpu_kernel_amd import build

LARGE = (0, 1, 2)  # GGK_VARIANT_64x64x16, 128x64x32, 64x128x32: 256 x 256 work tiles on the MFMA path
MFMA, FMA = 1, 0


def _forms():
    path = build.BUILD / build.FORMS_NAME
    if not path.exists():
        pytest.skip("no regular build in the tree (build first)")
    return json.loads(path.read_text())


def _key(f):
    return f["kind"], f["variant"], f["path"], f["traced"], f["wide"]


def test_report_covers_every_form():
    # grouped: 6 variants x 2 paths x traced x wide; single: 6 x 2 x wide
    forms = _forms()
    assert len(forms) == 6 * 2 * 4 + 6 * 2 * 2
    assert len({_key(f) for f in forms}) == len(forms)


def test_no_selectable_form_spills():
    spills = {}
    for f in _forms():
        if f["path"] == MFMA and f["wide"] and f["variant"] in LARGE:
            continue  # not launched
        if f["scratch"]:
            spills[_key(f)] = f["scratch"]
    assert not spills, f"(kind, variant, path, traced, wide): bytes of scratch a lane {spills}"


def test_fma_registers_allow_the_workgroups_that_lds_holds():
    """160 KB of LDS hold four 64 x 64 tiles or three larger ones; a workgroup is one wave per SIMD."""
    for f in _forms():
        if f["path"] == FMA and not f["wide"]:
            assert f["waves"] >= (4 if f["variant"] in (0, 5) else 3), f
