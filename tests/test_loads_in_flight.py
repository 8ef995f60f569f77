"""Kernels whose speed rests on loads that are issued together, as compiled: in
the assembly of this repository's own sources, the loads in flight at some
wait of the kernel's main loop.  (A compiler that interleaves loads and uses
halves the speed of these kernels on large vectors without changing a result.)
"""
import functools
import os
import re
import subprocess

import pytest

from jadamilu_amd import build as B


@functools.lru_cache(maxsize=None)
def _assembly(source):
    if not os.path.exists(B.HIPCC):
        pytest.skip("no hipcc")
    cmd = [B.HIPCC, *B.HIPFLAGS, *B.COMMON, "--cuda-device-only", "-S",
           os.path.join(B.CSRC, source), "-o", "-"]
    return subprocess.run(cmd, capture_output=True, text=True, check=True).stdout


def _most_in_flight(source, kernel):
    """The most vector loads that the kernel (a pattern of its mangled name) has
    outstanding at a wait."""
    text = _assembly(source)
    start = re.search(r"\n(_Z\S*" + kernel + r"\S*):", text)
    assert start, kernel
    body = text[start.end():text.index(".Lfunc_end", start.end())]
    loads, most = 0, 0
    for line in body.splitlines():
        if "global_load_dword" in line:
            loads += 1
        wait = re.search(r"s_waitcnt.*vmcnt\((\d+)\)", line)
        if wait:
            most = max(most, loads)
            loads = min(loads, int(wait[1]))
    return most


@pytest.mark.parametrize("kernel,loads", [
    # the columns of a step (eight at most) and the vector
    ("k_multidotIdLi4E", 5), ("k_multidotIdLi8E", 9), ("k_multidotIdLi16E", 9),
    ("k_multidotIfLi4E", 5), ("k_multidotIfLi8E", 9),
    # the same and two vectors
    ("k_project_rhoIdLi4E", 6), ("k_project_rhoIdLi8E", 10), ("k_project_rhoIfLi8E", 10)])
def test_inner_step(kernel, loads):
    assert _most_in_flight("kernels_inner.hip", kernel) >= loads


@pytest.mark.parametrize("kernel,loads", [
    # a value and an x for every entry of a row, with one more x and u
    ("k_spmv_diaIddLi4ELb0ELb1E", 15), ("k_spmv_diaIddLi7ELb0ELb1E", 27),
    ("k_spmv_diaIffLi4ELb0ELb1E", 15), ("k_spmv_diaIfdLi4ELb0ELb1E", 15)])
def test_diagonal_product(kernel, loads):
    assert _most_in_flight("kernels_dia.hip", kernel) >= loads
