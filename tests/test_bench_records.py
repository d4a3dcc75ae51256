"""What bench.py's output line says about the kernels -- CPU only: the launches of a step, and
the sources whose hash decides whether a recorded traffic figure still holds."""
import os
import re

import pytest

import bench


def _included(rel):
    """A source and the repository headers it includes, transitively."""
    seen, todo = set(), [rel]
    while todo:
        cur = todo.pop()
        if cur in seen:
            continue
        seen.add(cur)
        with open(os.path.join(bench.ROOT, cur)) as fh:
            names = re.findall(r'^#include "([^"]+)"', fh.read(), re.M)
        for d in ("flagattention_amd/csrc", "include"):
            todo += [f"{d}/{n}" for n in names if os.path.exists(os.path.join(bench.ROOT, d, n))]
    return seen


@pytest.mark.parametrize("family", sorted(bench.KERNEL_SOURCES))
def test_hashed_sources_cover_the_translation_unit_and_its_headers(family):
    listed = bench.KERNEL_SOURCES[family]
    assert set(listed) >= _included(listed[0])


@pytest.mark.parametrize("workload,kernels", [
    ("dense", ["mla_metadata_kernel", "mla_decode_kernel", "mla_combine_kernel"]),
    ("sparse", ["mla_metadata_uniform_kernel", "mla_decode_kernel", "mla_combine_kernel"]),
    ("sparse_fp8", ["mla_metadata_uniform_kernel", "mla_decode_kernel", "mla_combine_kernel"]),
])
def test_step_kernels(workload, kernels):
    """As profiles/perf_cases_kernel_trace.md has them for the same calls."""
    assert bench.step_kernels(bench.workload_spec(workload)) == kernels
