"""The sizes where batches of large experts leave the slices for the tile kernels, on both sides of each line, against the CPU path; a token
gets the same from either, and each side is the one that it is said to be."""
import ctypes as C
import json
import os

import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import load
from dwarfstar_red_lite_amd import moe as moe_api
from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe
from gpu_common import REL_L2_TOL, rel_l2
from test_gpu_moe_layer import ids_match_up_to_ties

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def on_tiles(call):
    """the call's result, and whether the tile kernels made it"""
    lib = load()
    n = lib.redhip_profile_stage_count()
    ms, launches = (C.c_double * n)(), (C.c_uint32 * n)()
    lib.redhip_profile_begin()
    out = call().cpu().numpy()
    lib.redhip_profile_end(ms, launches, n)
    return out, launches[[lib.redhip_profile_stage_name(i) for i in range(n)].index(b"prefill_gateup")] > 0


# experts per layer, experts per token and size all move the lines (most tokens that are slices: behind the own router, with the routing given); layers of
# few experts per token have none below 32 and 24 tokens. With more than 64 distinct experts one more costs the tiles less: the shapes of the last two rows leave
# the slices two to ten tokens earlier than at the same cost for each
@pytest.mark.parametrize("layout,shape,own,given", [("iq2", (2048, 512, 64, 6), 24, 22), ("iq2", (2048, 768, 40, 4), 25, 22), ("m", (2048, 512, 48, 5), 21, 19),
                                                    ("f2", (2048, 512, 48, 5), 24, 22), ("xs", (2048, 512, 64, 6), 23, 21), ("m", (1024, 512, 24, 8), 19, 17),
                                                    ("f2", (1024, 512, 24, 8), 24, 24), ("xs", (1024, 512, 24, 8), 24, 24), ("iq2", (2048, 512, 40, 10), 16, 16),
                                                    ("iq2", (1024, 512, 24, 8), 32, 24), ("iq2", (2048, 512, 60, 2), 32, 24), ("f2", (2048, 512, 60, 2), 32, 24), ("m", (1024, 512, 60, 4), 28, 24),
                                                    ("iq2", (2048, 512, 128, 8), 20, 18), ("m", (2048, 512, 128, 8), 17, 16), ("f2", (2048, 512, 256, 6), 23, 22),
                                                    ("xs", (2048, 512, 512, 10), 17, 16), ("iq2", (2048, 512, 512, 6), 24, 21), ("m", (1024, 512, 256, 8), 21, 19)])
def test_both_sides_of_the_line(layout, shape, own, given, golden_dir):
    if layout in ("m", "xs"):
        g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
        grids = [np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m")]
        moe_api.set_codebooks(*grids)
        orc.set_codebooks(*grids)
    H, F, E, K = shape
    cfg = synth.layer_config(hidden=H, ffn=F, n_expert=E, top_k=K, layout=layout)
    lay = synth.make_layer(95, cfg)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=own + 1)
    m.load_layer(0, lay)
    x = synth.normed_x(np.random.default_rng(96), own + 1, H)
    x_dev = torch.from_numpy(x).cuda()
    want, cids, _, clog = orc.Layer(cfg, **lay).forward(x, threads=8)
    whole = []
    for n in (own, own + 1):
        out, tiles = on_tiles(lambda: m.forward(0, x_dev[:n]))
        assert tiles == (n > own)
        whole.append(out)
    gids, gw, _ = m.last_route(own + 1)
    same = [t for t in range(own) if np.array_equal(gids[t], cids[t])]
    assert all(ids_match_up_to_ties(gids[t], cids[t], clog[t]) for t in range(own + 1)) and len(same) >= own - 1
    ids_dev, w_dev = torch.from_numpy(gids.astype(np.int32)).cuda(), torch.from_numpy(gw).cuda()
    for n in (given, given + 1):
        out, tiles = on_tiles(lambda: m.experts(0, x_dev[:n], ids_dev[:n].contiguous(), w_dev[:n].contiguous()))
        assert tiles == (n > given)
        whole.append(out)
    for got in whole:
        assert max(rel_l2(got[t], want[t]) for t in same if t < len(got)) <= REL_L2_TOL
        assert max(rel_l2(got[t], whole[1][t]) for t in range(len(got))) <= 1e-6      # (either path is 2e-7 off from exact)
    m.close()
