"""The f32 products of a chunk (router, dense shared expert with its SwiGLU) in every tile size they are cut into, and two tokens on the
one-token slices of the mixed layouts, against the CPU path."""
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


def forward_and_check(m, ref, x, pick):
    got = m.forward(0, torch.from_numpy(x).cuda()).cpu().numpy()
    gids, _, _ = m.last_route(len(x))
    want, cids, _, clog = ref.forward(np.ascontiguousarray(x[pick]), threads=8)
    assert all(ids_match_up_to_ties(gids[t], cids[i], clog[i]) for i, t in enumerate(pick))
    agree = [(i, t) for i, t in enumerate(pick) if np.array_equal(gids[t], cids[i])]
    assert len(agree) >= len(pick) - 1
    assert max(rel_l2(got[t], want[i]) for i, t in agree) <= REL_L2_TOL


@pytest.mark.parametrize("ntok", [41, 77, 301, 1025, 2047])      # tiles of 32 x 16, 32 x 32 and 64 x 32, ragged
def test_dense_products_of_a_chunk(ntok):
    cfg = synth.layer_config(hidden=512, ffn=256, n_expert=512, top_k=4, layout="f2")
    lay = synth.make_layer(95, cfg)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=ntok)
    m.load_layer(0, lay)
    x = synth.normed_x(np.random.default_rng(96), ntok, 512)
    forward_and_check(m, orc.Layer(cfg, **lay), x, [0, 1, 15, 16, 31, 32, ntok // 2, ntok - 2, ntok - 1])
    m.close()


@pytest.mark.parametrize("layout", ["f2", "xs", "m"])
@pytest.mark.parametrize("shape", [(2048, 512, 48, 10), (1024, 256, 32, 8), (512, 512, 16, 2)])
def test_two_tokens_behind_the_own_router(layout, shape, golden_dir):
    if layout in ("xs", "m"):
        g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
        grids = [np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m")]
        moe_api.set_codebooks(*grids)
        orc.set_codebooks(*grids)
    H, F, E, K = shape
    cfg = synth.layer_config(hidden=H, ffn=F, n_expert=E, top_k=K, layout=layout)
    lay = synth.make_layer(97, cfg)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=2)
    m.load_layer(0, lay)
    ref, rng = orc.Layer(cfg, **lay), np.random.default_rng(98)
    for scale in (1.0, 1e-3):
        x = synth.normed_x(rng, 2, H)
        x[1] *= np.float32(scale)
        forward_and_check(m, ref, x, [0, 1])
    m.close()
