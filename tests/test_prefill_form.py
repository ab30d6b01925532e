"""The prefill attention's form by rows, heads and switches (csrc/prefill_form.hpp), on the CPU."""

from __future__ import annotations

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is not available")


@pytest.fixture(scope="module")
def form(tmp_path_factory):
    exe = tmp_path_factory.mktemp("form") / "prefill_form_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", str(ROOT / "fast-dllm-relax_amd" / "csrc"),
                    str(ROOT / "tests" / "prefill_form_check.cpp"), "-o", str(exe)], check=True)

    def get(rows, nq, nkv, pair, hpw, cus=256):
        out = subprocess.run([str(exe), *map(str, (rows, nq, nkv, cus, pair, hpw))], capture_output=True, text=True, check=True)
        whole, paired = out.stdout.split()
        return f"{'twelve' if whole == '1' else 'four'} {'paired' if paired == '1' else 'alone'}"

    return get


def test_forms_by_size(form):
    for rows, want in [(128, "four alone"), (1504, "four alone"), (1728, "four paired"), (2048, "four paired"),
                       (2880, "twelve alone"), (6000, "twelve alone"), (7168, "twelve paired"), (8192, "twelve paired")]:
        assert form(rows, 12, 2, 1, 0) == want, rows
        assert form(rows // 2, 12, 2, 1, 0, cus=128) == want, (rows // 2, "of 128 compute units")
    assert form(8192, 4, 2, 1, 0) == "four paired"  # no group of six heads


def test_forms_by_switch(form):
    """FDLLM_PREFILL_PAIR and FDLLM_PREFILL_HPW: two heads per workgroup are four tiles at any size."""
    for rows in (352, 8192):
        assert form(rows, 12, 2, 0, 0) == "four alone"
        assert form(rows, 12, 2, 0, 6) == "twelve alone"
        assert form(rows, 12, 2, 2, 0) == "twelve paired"
        assert form(rows, 12, 2, 3, 0) == "four paired"
        assert form(rows, 12, 2, 1, 6).startswith("twelve")
        assert form(rows, 12, 2, 1, 2).startswith("four") and form(rows, 12, 2, 2, 2) == "four paired"
        assert form(rows, 4, 2, 0, 6) == "four alone"
