"""Host-side checks of the GEMM on 16 x 16 tiles (q8_gemm16.hip).  No device
is touched."""
import ctypes

import pytest


# offsets of stages past the last (4 KiB and 512 B per activation stage, a
# unit of 2176 B per weight stage) and lane offsets, up to the 4 GiB operands
OFFSETS = [0, 512, 4096, 2176, 20 * 4096, 18 * 2176, 0x7FFFFFFF, 0x80000000, 0xFFFFF000]
LANES = [0, 16, 1008, 4 * 5 * 2176, 0x7FFFFFF0, 0x80000000, 0xFFFFFFE0]


def stage(q8, t, stages, offset):
    extent, scalar = ctypes.c_uint32(), ctypes.c_uint32()
    q8.lib().llmcp_q8_test_dma_stage(t, stages, offset, ctypes.byref(extent), ctypes.byref(scalar))
    return extent.value, scalar.value


@pytest.mark.parametrize("offset", OFFSETS)
@pytest.mark.parametrize("t,stages", [(0, 0), (3, 0), (10, 10), (13, 10), (4 * 10**6, 10)])
def test_stage_past_the_last_reads_nothing(q8, t, stages, offset):
    """A raw buffer load is in range where its lane offset is below extent -
    scalar offset (mod 2^32); a stage that is not there must have no lane in
    range, whether the scalar offset takes part in the check or not."""
    extent, scalar = stage(q8, t, stages, offset)
    for lane in LANES:
        assert not lane < (extent - scalar) % 2**32, (offset, lane)
        assert not lane < extent and not lane + scalar < extent, (offset, lane)


@pytest.mark.parametrize("offset", OFFSETS)
@pytest.mark.parametrize("t,stages", [(0, 1), (9, 10), (0, 4 * 10**6)])
def test_stage_that_is_there_keeps_its_offset(q8, t, stages, offset):
    assert stage(q8, t, stages, offset) == (0xFFFFFFFF, offset)


# the shapes that tests/test_gpu_split.py names as splitting by their own choice
@pytest.mark.parametrize("m,n,k", [(2, 136, 1024), (33, 520, 2560), (97, 2560, 9216),
                                   (40, 264, 4096), (200, 2560, 2560), (48, 1024, 2560),
                                   (32, 2560, 2560), (16, 2560, 9216), (64, 256, 2560)])
def test_shapes_of_the_split_tests_split(q8, m, n, k):
    assert q8.gemm_plan(m, [n], k)[1] > 1
