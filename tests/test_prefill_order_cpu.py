"""The order of a prompt's attention tiles (turn_of): each tile once, the first batch and those behind the second longest first."""
import re
import os
import subprocess

import pytest


@pytest.fixture(scope="module")
def turn_of(tmp_path_factory):
    import ctypes
    src = os.path.join(os.path.dirname(__file__), "..", "bitmtp_amd", "csrc", "prefill_attn.hip.h")
    body = re.search(r"__device__ __forceinline__ (int turn_of\(.*?\n\})", open(src).read(), re.S).group(1)
    out = tmp_path_factory.mktemp("order")
    (out / "t.c").write_text(body)
    subprocess.run(["gcc", "-shared", "-fPIC", str(out / "t.c"), "-o", str(out / "t.so")], check=True)
    return ctypes.CDLL(str(out / "t.so")).turn_of


@pytest.mark.parametrize("batch", [0, 1, 32, 256])
@pytest.mark.parametrize("tiles", [1, 2, 31, 32, 33, 63, 64, 65, 94, 513])
def test_every_tile_once(turn_of, tiles, batch):
    order = [turn_of(i, tiles, batch) for i in range(tiles)]
    assert sorted(order) == list(range(tiles))
    second = order[batch:2 * batch]
    assert second == sorted(second, reverse=True)
    assert order[:batch] + sorted(second) + order[2 * batch:] == list(range(tiles))
