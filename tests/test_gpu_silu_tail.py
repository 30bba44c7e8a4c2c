"""SwiGLU of gates whose exponential is almost all that a float holds: beyond -87.3 the reciprocal of 1 + exp(-g) is no normal float any more, the product with g
still is. Chunks on the tile kernels, tiles of up to eight pairs, full and wider ones, against sums in double."""
import json
import os

import numpy as np
import pytest

from dwarfstar_red_lite_amd import moe as moe_api
from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe
from test_gpu_batch_lines import on_tiles
from test_gpu_batch_precision import routed_in_double
from test_gpu_staged_tiles import routing_with

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("layout,hidden,ffn", [("iq2", 512, 256), ("f2", 2048, 512), ("m", 1024, 512), ("xs", 2048, 768)])
def test_gates_down_to_the_last_exponent(layout, hidden, ffn, golden_dir):
    if layout in ("m", "xs"):
        g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
        moe_api.set_codebooks(*(np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m")))
    counts, top_k = [5, 12, 32, 1, 30], 2
    E, n = len(counts), sum(counts) // top_k
    cfg = synth.layer_config(hidden=hidden, ffn=ffn, n_expert=E, top_k=top_k, layout=layout)
    lay, rng = synth.make_layer(41, cfg), np.random.default_rng(42)
    lay["sh_down"] = np.zeros_like(lay["sh_down"])      # the routed experts alone
    # small gate weights (so large activations) and large others: the outputs are 1e-27 and not at the end of the range themselves
    one = synth.quant_rows(rng, cfg["gate_up_type"], 1, hidden, d_range=(1e-4, 1e-4))
    lay["gate"] = np.tile(one, (E, ffn))                 # every gate of a token is the same
    lay["up"] = synth.quant_rows(rng, cfg["gate_up_type"], E * ffn, hidden, d_range=(100.0, 100.0)).reshape(E, -1)
    lay["down"] = synth.quant_rows(rng, cfg["down_type"], E * hidden, ffn, d_range=(10.0, 10.0)).reshape(E, -1)
    row = moe_api.dequant_rows(cfg["gate_up_type"], torch.from_numpy(one).cuda(), hidden).cpu().numpy().astype(np.float64)[0]
    ids = routing_with(counts, n, top_k, rng).astype(np.int32)
    # an activation along the gate row: nothing cancels, the gate is as good as its terms
    gates = np.concatenate([np.linspace(-88.70, -87.36, n - 6), [-88.722, -87.2, -86.0, -60.0, -20.0, -1.0]])
    x = (row * (gates / np.square(row).sum())[:, None]).astype(np.float32)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=n)
    m.load_layer(0, lay)
    x_dev, ids_dev = torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda()
    w = torch.from_numpy((rng.random((n, top_k)) + 0.1).astype(np.float32)).cuda()
    got, tiles = on_tiles(lambda: m.experts(0, x_dev, ids_dev, w))
    assert tiles
    want = routed_in_double(lay, cfg, x_dev, ids_dev, w).cpu().numpy()
    off = np.linalg.norm(got.astype(np.float64) - want, axis=1) / np.linalg.norm(want, axis=1)
    assert off.max() <= 4e-5, list(zip(gates, off))      # a gate's relative error of 2e-7 is one of 88 times that in its exponential
    m.close()
