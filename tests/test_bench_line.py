"""The bench line's rooflines name the kernels that run with its options, and take counters only
from a profile of those kernels on that workload."""
import argparse
import json
import os

import pytest

import bench

KSTATS = {"likelihood": {"ms": 2.0, "launches": 10, "flops": 1e9, "bytes": 0.0},
          "extract": {"ms": 1.0, "launches": 2, "flops": 0.0, "bytes": 1e9},
          "step": {"ms": 0.0, "launches": 0, "flops": 0.0, "bytes": 0.0}}


def _args(**more):
    base = dict(config="197dish", batch=1, grid_variant=5, lik_block=0, lik_precision=0, fuse_step=1,
                tile_cells=0, tile_passes=0, tile_blocks=0, tile_streams=1)
    return argparse.Namespace(**{**base, **more})


def _recorded():
    with open(os.path.join(bench.ROOT, "profiles", "traffic.json")) as f:
        return json.load(f)


def test_the_default_workload_has_counters_of_its_own_kernels():
    _, lik, ext = bench.roofline(KSTATS, 78.6, _args())
    got = {tuple(e["kernels"]): e for e in _recorded()["measured"]}
    assert _recorded()["config"] == "197dish"
    e = got["lik_p0_group_kernel", "lik_fused_kernel", "lik_fused_wide_kernel"]
    assert lik["traffic"] == e["launch_bytes"] and lik["valu_busy"] == e["valu_busy"]
    assert ext["traffic"] == got["grid_cell_kernel",]["launch_bytes"]
    assert "grid_cell_kernel" in ext["kernel"] and "lik_fused_wide_kernel" in lik["kernel"]


@pytest.mark.parametrize("more,kernel", [
    (dict(config="64dish"), "lik_task_kernel"),
    (dict(fuse_step=0), "lik_tile_kernel"),
    (dict(fuse_step=2), "lik_persist_kernel"),
    (dict(lik_precision=2), "lik_tile_kernel"),
    (dict(lik_block=256), "likelihood_kernel"),
])
def test_other_kernels_take_no_counters(more, kernel):
    _, lik, _ = bench.roofline(KSTATS, 78.6, _args(**more))
    assert kernel in lik["kernel"] and lik["traffic"] is None and lik["valu_busy"] is None


@pytest.mark.parametrize("more,kernel", [
    (dict(config="64dish"), "grid_cell_kernel"),
    (dict(grid_variant=3), "grid_run_kernel"),
    (dict(batch=16), "grid_batch_kernel"),
])
def test_other_extractions_take_no_counters(more, kernel):
    _, _, ext = bench.roofline(KSTATS, 78.6, _args(**more))
    assert kernel in ext["kernel"] and ext["traffic"] is None
