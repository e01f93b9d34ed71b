"""What the compiler made of kernels whose speed hangs on it: properties that a
change elsewhere can take away without any wrong result."""
import re

import pytest

import code_objects as co


@pytest.mark.skipif(not co.have_objdump(), reason="llvm-objdump of ROCm")
@pytest.mark.parametrize("N", [7, 9, 12])
@pytest.mark.parametrize("here", [0, 1])
def test_scatter_loads_from_scalar_bases(N, here):
    """k_uw_scatter's columns: the base in scalar registers, one lane offset for
    all of them (with addresses in vector registers the kernel's stores waited
    for whole batches of loads)."""
    (name,) = co.find(f"k_uw_scatterILi{N}ELb{here}E")
    loads = [i for i in co.instructions(name) if i.startswith("global_load_dwordx2")]
    scalar = [i for i in loads if re.search(r", s\[\d+:\d+\]", i)]
    assert len(loads) >= 4 * N * 4  # every column of the four groups
    assert len(scalar) >= 4 * N * 4


# Waves per SIMD of the kernels over stored events, which the columns bound, for
# 2 .. 12 bodies.
STORED = {
    "k_event_weight": [8, 7, 6, 5, 5, 4, 4, 4, 3, 3, 3],
    "k_max_weight": [8, 7, 6, 5, 5, 4, 4, 4, 3, 3, 3],
}


@pytest.mark.parametrize("kernel", STORED)
def test_stored_events_waves(kernel):
    for N, want in zip(range(2, 13), STORED[kernel]):
        (k,) = co.find(f"{kernel}ILi{N}E").values()
        assert co.waves(k) >= want, (kernel, N, k[".vgpr_count"])


# Bytes of a kernel's arguments: of calls on few events, the launch is the time.
ARGUMENTS = {
    "k_evaluate_f64ILi3ELi0ELb0E": 2208,
    "k_hist_fillILi3ELb0E": 2080,
    "k_average_f64ILi3ELi0ELb0E": 1088,
    "k_average_mixedILi3ELi0ELb0ELi4E": 960,
    "k_uw_flagsILi3E": 928,
    "k_range_histILi3E": 1824,
}


@pytest.mark.parametrize("kernel", ARGUMENTS)
def test_argument_bytes(kernel):
    for k in co.find(kernel).values():
        assert k[".kernarg_segment_size"] <= ARGUMENTS[kernel]


@pytest.mark.parametrize("engine", range(2, 6))
@pytest.mark.parametrize("kernel", ["k_generate_f64", "k_evaluate_f64", "k_generate_mixed"])
def test_single_blocks_stay_in_registers(kernel, engine):
    """2-body events of the Random123 engines need one block each: nothing of it is
    shared, so nothing goes through LDS."""
    for k in co.find(f"{kernel}ILi2ELi{engine}ELb0E").values():
        assert k[".group_segment_fixed_size"] == 0


@pytest.mark.parametrize("mothers", [0, 1])
@pytest.mark.parametrize("N", [2, 3, 4])
def test_average_spills_nothing(N, mothers):
    """AverageOn's form of four waves per chunk, every engine."""
    for engine in range(6):
        for name, k in co.find(f"k_average_f64ILi{N}ELi{engine}ELb{mothers}E").items():
            if k[".max_flat_workgroup_size"] == 256:
                assert k[".vgpr_spill_count"] == 0, name
