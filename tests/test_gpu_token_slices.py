"""Two to eight tokens on the one-token slices of the mixed layouts, one grid layer per token: batches on both sides of the line (680
workgroups), tokens that share all of their experts, and the block form, against the CPU path."""
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


@pytest.mark.parametrize("layout", ["f2", "xs", "m"])
@pytest.mark.parametrize("shape,tokens", [((2048, 512, 48, 10), (3, 4)), ((1024, 256, 32, 8), (3, 7, 8)), ((512, 256, 16, 3), (5, 8)), ((1024, 512, 24, 15), (2, 3))])
def test_small_batches_behind_the_own_router(layout, shape, tokens, golden_dir):
    if layout in ("xs", "m"):
        g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
        grids = [np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m")]
        moe_api.set_codebooks(*grids)
        orc.set_codebooks(*grids)
    H, F, E, K = shape
    cfg = synth.layer_config(hidden=H, ffn=F, n_expert=E, top_k=K, layout=layout)
    lay = synth.make_layer(871, cfg)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=max(tokens))
    m.load_layer(0, lay)
    ref, rng = orc.Layer(cfg, **lay), np.random.default_rng(19)
    for n in tokens:
        x = synth.normed_x(rng, n, H)
        x[n - 1] = x[0] if n % 2 else x[n - 1] * np.float32(1e-3)      # (odd: the last token takes the first one's experts)
        x_dev = torch.from_numpy(x).cuda()
        got = m.forward(0, x_dev).cpu().numpy()
        gids, gw, _ = m.last_route(n)
        want, cids, cw, clog = ref.forward(x, threads=8)
        for t in range(n):
            assert ids_match_up_to_ties(gids[t], cids[t], clog[t]), (n, t)
            if np.array_equal(gids[t], cids[t]):
                assert rel_l2(got[t], want[t]) <= 1e-5 and np.abs(gw[t] - cw[t]).max() <= 1e-5, (n, t)
        if n % 2:
            assert np.array_equal(got[n - 1], got[0])
        one = torch.cat([m.forward(0, x_dev[t:t + 1]) for t in range(n)]).cpu().numpy()
        assert max(rel_l2(got[t], one[t]) for t in range(n)) <= 1e-6
        # x + branch with the branch zero and the norm's weights one: the norm is all that the layer adds
        out = m.forward_block(0, x_dev, torch.zeros_like(x_dev), torch.ones(H, device="cuda")).cpu().numpy() - x
        normed = x / np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=1, keepdims=True) + 1e-6)
        want = ref.forward(normed.astype(np.float32), threads=8)[0]
        assert max(rel_l2(out[t], want[t]) for t in range(n)) <= REL_L2_TOL
    m.close()
