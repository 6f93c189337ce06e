"""CPU tests of the form that a linear's product takes (host arithmetic of the
library, 256 CUs where no GPU is visible) against measured times of the forms
(profiles/gemm_form_timings.txt)."""

import ctypes
import math
import os

import pytest

from conftest import ROOT


def _form(m, blocks, n, bits, out_f32=False):
    """The library's choice, named as in the table."""
    from polarengine_vllm import _lib
    form = (ctypes.c_int * 4)()
    fmt = (_lib.PE_PACK_NIBBLE if bits <= 4 else 0) | _lib.PE_LAYOUT_TILE16
    _lib.check(_lib.lib().pe_linear_xtf_form(m, 128 * blocks, n, bits, fmt, int(out_f32), form),
               "pe_linear_xtf_form")
    kernel, rows, cols, z = form
    return "s" if kernel == 0 else f"{4 if kernel == 2 else 8}:{rows}x{cols}/{z}"


@pytest.fixture(scope="module")
def timings():
    """[(shape, {form: (us repeated, us from HBM)}, form of the thresholds)]"""
    if not os.path.exists(os.path.join(ROOT, "polarengine-vllm_amd", "lib", "libpolarengine_amd.so")):
        pytest.skip("library not built")
    out = []
    with open(os.path.join(ROOT, "profiles", "gemm_form_timings.txt")) as f:
        for line in f:
            if line.startswith("#"):
                continue
            shape, *forms = line.split()
            times, before = {}, None
            for item in forms:
                name, us = item.split("=")
                if name.endswith("*"):
                    name = before = name[:-1]
                times[name] = tuple(float(v) for v in us.split("/"))
            out.append((tuple(int(v) for v in shape.split(",")), times, before))
    return out


@pytest.mark.parametrize("weights", ["repeated", "from HBM"])
def test_plan_is_near_the_fastest_form(timings, weights):
    i = ("repeated", "from HBM").index(weights)
    over, behind = [], []
    for (m, n, blocks, bits), times, before in timings:
        got = times.get(_form(m, blocks, n, bits))
        if got is None:  # a form that was not timed at this shape
            continue
        over.append(got[i] / min(t[i] for t in times.values()))
        behind.append(got[i] / times[before][i])
    assert len(over) >= 0.95 * len(timings)
    assert sum(over) / len(over) <= 1.018
    # calls that got slower than by the thresholds that the model replaced
    assert sum(b > 1.05 for b in behind) <= 0.03 * len(behind)
    assert sum(b > 1.10 for b in behind) <= 0.01 * len(behind)
    assert max(behind) < 1.4 and math.exp(sum(map(math.log, behind)) / len(behind)) < 0.82
