"""Host-side rules of the region inserts (mutation.hpp, partition.hpp), as the
test libraries built from the headers evaluate them; no GPU."""
import ctypes
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent / "device_api"


def _lib(name):
    path = HERE / f"libwc_{name}.so"
    if not path.exists():
        from device_api.build import build
        build()
    return ctypes.CDLL(str(path))


@pytest.mark.parametrize("which,many", [(0, 1), (1, 1), (2, 0)])
def test_null_stream_of_a_per_thread_build_is_many(which, many):
    """The null and the per-thread handle name another stream in every host
    thread there; a created stream's handle does not."""
    assert _lib("per_thread").wcp_per_thread_stream(which) == many


@pytest.mark.parametrize("resident", [1, 7, 8, 9, 228, 252, 255, 256, 300, 304, 512, 516, 520])
def test_grids_are_multiples_of_the_xcds(resident):
    """part_refine's blocks stride by gridDim / 8 from blockIdx / 8, one of the
    8 XCDs each: every (unit, XCD) pair has exactly one block."""
    lib = _lib("per_thread")
    lib.wcp_part_blocks.restype = ctypes.c_uint
    lib.wcp_part_blocks.argtypes = [ctypes.c_uint64, ctypes.c_uint]
    for wanted in (0, 1, 7, 8, 9, 250, 255, 256, 257, 1 << 33):
        grid = lib.wcp_part_blocks(wanted, resident)
        assert grid % 8 == 0 and 8 <= grid <= max(8, resident)
        units = 100
        taken = sorted((v, b % 8) for b in range(grid) for v in range(b // 8, units, grid // 8))
        assert taken == [(v, x) for v in range(units) for x in range(8)]


def test_copies_of_a_table_keep_its_mutation_state():
    """A copy is copied after its table is gone: the state they share is
    deleted once, with the last of them."""
    assert _lib("host_memory").wch_tracker_lifetime() == 1
