"""The sizes where batches of large experts leave the slices for the tile kernels, on both sides of each line, against the CPU path; a token
gets the same from either."""
import json
import os

import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import moe as moe_api
from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe
from gpu_common import REL_L2_TOL, rel_l2
from test_gpu_moe_layer import ids_match_up_to_ties

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("layout,shape,own,given", [("iq2", (2048, 512, 40, 10), 22, 19), ("iq2", (2048, 768, 24, 8), 22, 19), ("m", (2048, 512, 40, 10), 16, 16),
                                                    ("f2", (2048, 512, 40, 10), 19, 19), ("xs", (2048, 512, 40, 10), 23, 22), ("m", (1024, 512, 24, 8), 25, 22),
                                                    ("f2", (1024, 512, 24, 8), 28, 24), ("xs", (1024, 512, 24, 8), 30, 24)])
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
    whole = [m.forward(0, x_dev[:n]).cpu().numpy() for n in (own, own + 1)]
    gids, gw, _ = m.last_route(own + 1)
    same = [t for t in range(own) if np.array_equal(gids[t], cids[t])]
    assert all(ids_match_up_to_ties(gids[t], cids[t], clog[t]) for t in range(own + 1)) and len(same) >= own - 1
    ids_dev, w_dev = torch.from_numpy(gids.astype(np.int32)).cuda(), torch.from_numpy(gw).cuda()
    for n in (given, given + 1):
        whole.append(m.experts(0, x_dev[:n], ids_dev[:n].contiguous(), w_dev[:n].contiguous()).cpu().numpy())
    for got in whole:
        assert max(rel_l2(got[t], want[t]) for t in same if t < len(got)) <= REL_L2_TOL
        assert max(rel_l2(got[t], whole[1][t]) for t in range(len(got))) <= 1e-6      # (either path is 2e-7 off from exact)
    m.close()
