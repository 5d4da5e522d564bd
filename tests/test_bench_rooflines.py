"""bench.py's rooflines, without a GPU: what is reported for each of the sub-step's kernels."""
from __future__ import annotations

import json

import bench

N = 256 * 256


def entry(kernel, substeps, sub, march=(0.0, 0), rows=0, listed=0, mixed=False):
    t = {"sub": sub, "march": march, "sweep": (1.0, 1)}
    r = bench.rooflines(mixed, 2, False, N, t, kernel, substeps, rows, 0, listed, None)
    json.dumps(r)
    return r


def test_tiles_have_no_bandwidth():
    # 12 sub-steps move the concentration once: no bytes per sub-step to divide by its time
    roof, sub = entry("diffuse_tile_kernel", 12, (0.26, 188), listed=900)
    assert roof["kernel"] == "diffuse_tile_kernel<FormF64, 2>"
    assert roof["achieved"] is None and roof["frac"] is None and roof["bytes_per_cell"] is None
    assert roof["substep_us"] == round(260 / 188, 2) and "launch_us" not in roof
    assert sub["achieved_gbs"] is None and sub["frac"] is None and sub["bytes"] is None


def test_nothing_timed_is_null():
    # all sub-steps in the batch's first launch, which is not timed
    for kernel, substeps in (("diffuse_tile_kernel", 8), ("diffuse_direct_kernel", 1)):
        roof, sub = entry(kernel, substeps, (0.0, 0))
        assert roof["achieved"] is None and roof["frac"] is None
        assert sub["us"] is None and sub["achieved_gbs"] is None


def test_one_launch_and_marching_kernels():
    us = 4.0
    roof, sub = entry("diffuse_direct_kernel", 1, (us * 100 / 1e3, 100), listed=900)
    assert roof["kernel"] == "diffuse_direct_kernel<FormF64, 2>"
    assert roof["achieved"] == round(N * 16 / us / 1e3, 1) == sub["achieved_gbs"]
    assert roof["launch_us"] == us and roof["launches_timed"] == 100
    # the marching kernel by its own launches, the sub-step with the listed pass
    roof, sub = entry("diffuse_bulk_march_kernel", 1, (us * 200 / 1e3, 200), (3.0 * 25 / 1e3, 25), rows=8,
                      listed=900, mixed=True)
    assert roof["kernel"] == bench.march_kernel_name(True, 2, False, 8)
    assert roof["achieved"] == round(N * 9 / 3.0 / 1e3, 1)
    assert sub["bytes"] == N * 9 + 900 * bench.listed_bytes_per_cell(True, 2)
    assert sub["achieved_gbs"] == round(sub["bytes"] / us / 1e3, 1)
    # a plane above the tiles' size: single sub-steps under their own name
    roof, _ = entry("diffuse_linear_kernel", 1, (us * 100 / 1e3, 100))
    assert roof["kernel"] == "diffuse_linear_kernel<FormF64, 2>"
