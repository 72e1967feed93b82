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
