"""Registers, LDS and scratch of the built kernels (from their metadata, no GPU): what a
kernel was designed to fit beside on a compute unit."""
import pytest

from tests import kernel_info as ki

STEP_THREADS, REDUCE_THREADS = 512, 256


@pytest.mark.parametrize("shape", ["Li0ELi1E", "Li1ELi0E", "Li2ELi1E", "Li3ELi0E"])
@pytest.mark.parametrize("comp", [0, 1])
def test_tracking_step_lds_does_not_limit_its_blocks(comp, shape):
    k = ki.find(f"icp_stepILb{comp}E{shape}")
    assert ki.blocks_by_lds(k) >= ki.blocks_by_registers(k, STEP_THREADS) >= 2
    if not comp:
        assert k[".group_segment_fixed_size"] <= 8192  # no rows for the matrix cores


@pytest.mark.parametrize("comp", [0, 1])
def test_reduce_lds_does_not_limit_its_blocks(comp):
    k = ki.find(f"icp_partialsILb{comp}E")
    assert ki.blocks_by_lds(k) >= ki.blocks_by_registers(k, REDUCE_THREADS)
    if not comp:
        assert k[".group_segment_fixed_size"] <= 4096


@pytest.mark.parametrize("comp", [0, 1])
def test_single_launch_tracking_has_no_scratch(comp):
    k = ki.find(f"icp_chainILb{comp}E")
    assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0
    assert ki.blocks_by_lds(k) >= 3


@pytest.mark.parametrize("zero_tail", [0, 1])
@pytest.mark.parametrize("radius", [0, 1, 2, 3, 4])
def test_depth_filter_waves(radius, zero_tail):
    k = ki.find(f"depth_levelsILi{radius}ELb{zero_tail}E")
    # the window's rows are unrolled where the weights end in the table, up to radius 3
    assert ki.waves_by_registers(k) >= (3 if zero_tail and radius <= 3 else ki.MAX_WAVES)
    assert ki.blocks_by_lds(k) * 256 >= ki.MAX_WAVES * ki.SIMDS * 64


@pytest.mark.parametrize("fmt", [0, 1])
def test_sweep_keeps_seven_waves(fmt):
    assert ki.waves_by_registers(ki.find(f"integrateILi{fmt}E")) >= 7


@pytest.mark.parametrize("latency", [0, 1])
def test_brick_classes_keep_three_waves(latency):
    assert ki.waves_by_registers(ki.find(f"brick_classifyILb{latency}E")) >= 3  # kLatencyBricks counts on them
