"""What the compiler noted of the built kernels: the tile kernels keep everything in registers. A spilled one is a load from scratch memory in the
inner loop, and the waits of these kernels count the loads in flight."""
import os

import pytest

from dwarfstar_red_lite_amd._lib import LIB_PATH


def uint(b, at):
    """a msgpack number that is not negative"""
    return b[at] if b[at] < 0x80 else int.from_bytes(b[at + 1:at + 1 + (1 << (b[at] - 0xcc))], "big")


def spilled():
    """{kernel: vector registers spilled} from the metadata notes of the code objects; a kernel's entries are sorted by key"""
    with open(LIB_PATH, "rb") as f:
        b = f.read()
    key, out, at = b".vgpr_spill_count", {}, 0
    while (at := b.find(key, at)) >= 0:
        name = b.rfind(b".symbol", 0, at)
        start = b.find(b"_Z", name)
        out[b[start:b.find(b".kd", start)].decode()] = uint(b, at + len(key))
        at += len(key)
    return out


@pytest.mark.skipif(not os.path.exists(LIB_PATH), reason="nothing is built")
def test_tile_kernels_spill_nothing():
    tiles = {k: v for k, v in spilled().items() if "staged_tiles_kernel" in k}
    assert len(tiles) >= 70
    assert not {k: v for k, v in tiles.items() if v}
