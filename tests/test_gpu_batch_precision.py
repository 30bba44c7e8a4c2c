"""A batch loses no precision where it leaves the slices for the tile kernels: the same tokens with the same routing, as a batch of slices and as
part of one on the tiles, against sums in double. The two differ in nothing but the kernels, so their errors are compared with each other."""
import json
import os

import numpy as np
import pytest

from dwarfstar_red_lite_amd import moe as moe_api
from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe
from test_gpu_batch_lines import on_tiles
from test_gpu_staged_tiles import routing_with

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def routed_in_double(lay, cfg, x, ids, w):
    """the routed experts' part of a layer's output"""
    H, F, d = cfg["hidden"], cfg["ffn"], torch.float64

    def rows(t, raw, n, cols):
        return moe_api.dequant_rows(t, torch.from_numpy(raw.reshape(n, -1)).cuda(), cols).to(d).T.contiguous()
    out, xd = torch.zeros((len(x), H), dtype=d, device="cuda"), x.to(d)
    for e in range(cfg["n_expert"]):
        tok, k = torch.nonzero(ids == e, as_tuple=True)
        if not len(tok):
            continue
        g, u = (xd[tok] @ rows(cfg["gate_up_type"], lay[m][e], F, H) for m in ("gate", "up"))
        y = (g / (1.0 + torch.exp(-g)) * u) @ rows(cfg["down_type"], lay["down"][e], H, F)
        out.index_add_(0, tok, y * w[tok, k].to(d)[:, None])
    return out


# 16 tokens are slices on all of these and 32 with the routing given never are. 96 tokens, whose errors' mean varies by 1 % from one draw to another
@pytest.mark.parametrize("layout,hidden,ffn", [("iq2", 2048, 512), ("f2", 2048, 512), ("xs", 2048, 512), ("m", 2048, 512), ("m", 1024, 512), ("iq2", 2048, 768)])
def test_tiles_against_slices(layout, hidden, ffn, golden_dir):
    if layout in ("m", "xs"):
        g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
        moe_api.set_codebooks(*(np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m")))
    cfg = synth.layer_config(hidden=hidden, ffn=ffn, n_expert=24, top_k=8, layout=layout)
    err, norm = np.zeros(2), 0.0
    for seed in range(6):
        lay = synth.make_layer(seed, cfg)
        lay["sh_down"] = np.zeros_like(lay["sh_down"])      # the routed experts alone
        m = ResidentMoe(cfg, n_layer=1, max_tokens=32)
        m.load_layer(0, lay)
        rng = np.random.default_rng(100 + seed)
        x = torch.from_numpy(synth.normed_x(rng, 32, hidden)).cuda()
        ids = torch.from_numpy(np.stack([rng.permutation(24)[:8] for _ in range(32)]).astype(np.int32)).cuda()
        w = torch.from_numpy((rng.random((32, 8)) + 0.1).astype(np.float32)).cuda()
        want = routed_in_double(lay, cfg, x[:16], ids[:16], w[:16])
        for i, n in enumerate((16, 32)):
            got = m.experts(0, x[:n].contiguous(), ids[:n].contiguous(), w[:n].contiguous())[:16]
            err[i] += float((got.to(torch.float64) - want).square().sum())
        norm += float(want.square().sum())
        m.close()
    slices, tiles = np.sqrt(err / norm)
    print("%s %d x %d: slices %.3e, tiles %.3e" % (layout, hidden, ffn, slices, tiles))
    assert slices <= 2.1e-7 and tiles <= slices, (slices, tiles)      # (2.1e-7: what f32 products of such a layer give)


# Where many experts are named nearly every tile has one to eight pairs, whose high and low halves are rows of one operand and are rounded apart. (16 tokens are
# slices with the routing given, ten a token of 128 experts.)
@pytest.mark.parametrize("layout,ffn", [("iq2", 512), ("f2", 512), ("xs", 512), ("m", 512), ("iq2", 768)])
def test_small_tiles_against_slices(layout, ffn, golden_dir):
    if layout in ("m", "xs"):
        g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
        moe_api.set_codebooks(*(np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m")))
    hidden, E, K = 2048, 128, 10
    cfg = synth.layer_config(hidden=hidden, ffn=ffn, n_expert=E, top_k=K, layout=layout)
    err, norm = np.zeros(2), 0.0
    lay = synth.make_layer(7, cfg)
    lay["sh_down"] = np.zeros_like(lay["sh_down"])      # the routed experts alone
    m = ResidentMoe(cfg, n_layer=1, max_tokens=32)
    m.load_layer(0, lay)
    for seed in range(6):
        rng = np.random.default_rng(200 + seed)
        x = torch.from_numpy(synth.normed_x(rng, 32, hidden)).cuda()
        ids = routing_with([8] * 8 + [7] * 8 + [6] * 8 + [2] * 48 + [1] * 56, 32, K, rng)
        ids = torch.from_numpy(ids.astype(np.int32)).cuda()
        w = torch.from_numpy((rng.random((32, K)) + 0.1).astype(np.float32)).cuda()
        want = routed_in_double(lay, cfg, x[:16], ids[:16], w[:16])
        for i, n in enumerate((16, 32)):
            got, tiles = on_tiles(lambda: m.experts(0, x[:n].contiguous(), ids[:n].contiguous(), w[:n].contiguous())[:16])
            assert tiles == (n == 32)
            err[i] += float((torch.from_numpy(got).cuda().to(torch.float64) - want).square().sum())
        norm += float(want.square().sum())
    m.close()
    slices, tiles = np.sqrt(err / norm)
    print("%s 2048 x %d, small tiles: slices %.3e, tiles %.3e" % (layout, ffn, slices, tiles))
    assert slices <= 2.1e-7 and tiles <= slices, (slices, tiles)


# where 32 tokens with the routing given would be further off on the tiles than as slices, 24 still are slices, however few the experts
@pytest.mark.parametrize("layout", ["iq2", "f2", "xs"])
def test_small_experts_stay_slices(layout, golden_dir):
    if layout == "xs":
        g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
        moe_api.set_codebooks(*(np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m")))
    cfg = synth.layer_config(hidden=1024, ffn=512, n_expert=24, top_k=8, layout=layout)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=32)
    m.load_layer(0, synth.make_layer(3, cfg))
    x = torch.from_numpy(synth.normed_x(np.random.default_rng(4), 32, 1024)).cuda()
    ids = torch.from_numpy(np.stack([np.random.default_rng(t).permutation(24)[:8] for t in range(32)]).astype(np.int32)).cuda()
    w = torch.full((32, 8), 0.125, device="cuda")
    for n in (17, 24, 25):
        assert on_tiles(lambda: m.experts(0, x[:n].contiguous(), ids[:n].contiguous(), w[:n].contiguous()))[1] == (n > 24)
    m.close()
