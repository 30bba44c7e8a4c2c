"""Down matrices of three and four blocks of 256 columns on raw rows: their tiles are cut into parts (a pass each, fours of 32-row items), as many as the
busiest workgroup has anyway, and tiles of up to 32 pairs have a launch of their own again. Numbers of tiles on both sides of what the device holds at
once, against sums in double."""
import ctypes as C
import json
import os

import numpy as np
import pytest

from dwarfstar_red_lite_amd import load
from dwarfstar_red_lite_amd import moe as moe_api
from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe
from test_gpu_batch_precision import routed_in_double
from test_gpu_precision import F32_CHUNK

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def layer(layout, hidden, ffn, n_expert, max_tokens, golden_dir):
    if layout in ("m", "xs"):
        g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
        moe_api.set_codebooks(*(np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m")))
    cfg = synth.layer_config(hidden=hidden, ffn=ffn, n_expert=n_expert, top_k=4, layout=layout)
    lay = synth.make_layer(71, cfg)
    lay["sh_down"] = np.zeros_like(lay["sh_down"])      # the routed experts alone
    m = ResidentMoe(cfg, n_layer=1, max_tokens=max_tokens)
    m.load_layer(0, lay)
    return cfg, lay, m


def evenly(n, used, seed):
    """n tokens, their pairs dealt to the first `used` experts in turn"""
    ids = ((torch.arange(n, device="cuda")[:, None] * 4 + torch.arange(4, device="cuda")) % used).to(torch.int32)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return ids.contiguous(), torch.softmax(torch.randn((n, 4), device="cuda", generator=gen), dim=1).contiguous()


def down_stage(call):
    """(us, launches) of the down tiles of a call"""
    lib = load()
    n = lib.redhip_profile_stage_count()
    ms, launches = (C.c_double * n)(), (C.c_uint32 * n)()
    at = [lib.redhip_profile_stage_name(i) for i in range(n)].index(b"prefill_down")
    torch.cuda.synchronize()
    lib.redhip_profile_begin()
    call()
    lib.redhip_profile_end(ms, launches, n)
    return ms[at] * 1e3, launches[at]


# (hidden: 4, 8 and 16 fours of items a tile; tiles: 5, 100, 129, 260 narrow ones of two experts' sizes)
@pytest.mark.parametrize("layout,ffn", [("f2", 768), ("f2", 1024), ("xs", 768), ("m", 1024), ("m", 768)])
@pytest.mark.parametrize("hidden,used,n", [(512, 5, 17), (1024, 100, 125), (2048, 129, 129), (512, 130, 565)])
def test_narrow_tiles(layout, ffn, hidden, used, n, golden_dir):
    cfg, lay, m = layer(layout, hidden, ffn, used, n, golden_dir)
    x = torch.from_numpy(synth.normed_x(np.random.default_rng(72), n, hidden)).cuda()
    ids, w = evenly(n, used, 73)
    got = m.experts(0, x, ids, w).to(torch.float64)
    want = routed_in_double(lay, cfg, x, ids, w)
    assert float((got - want).norm() / want.norm()) <= F32_CHUNK
    m.close()


# 30 pairs an expert beside some of 31 and 32; weights in wide tiles above the line of 200 million
@pytest.mark.parametrize("layout,hidden,ffn,used", [("f2", 2048, 768, 136), ("xs", 2048, 768, 136), ("m", 2048, 768, 136), ("f2", 2048, 1024, 104)])
def test_wide_tiles(layout, hidden, ffn, used, golden_dir):
    n = used * 30 // 4 + 11
    cfg, lay, m = layer(layout, hidden, ffn, used, n, golden_dir)
    x = torch.from_numpy(synth.normed_x(np.random.default_rng(74), n, hidden)).cuda()
    ids, w = evenly(n, used, 75)
    out = []
    assert down_stage(lambda: out.append(m.experts(0, x, ids, w)))[1] == 2      # a launch for wide and one for narrow tiles
    want = routed_in_double(lay, cfg, x, ids, w)
    assert float((out[0].to(torch.float64) - want).norm() / want.norm()) <= F32_CHUNK
    m.close()


def test_fewer_tiles_take_no_longer():
    """64 tiles of 32 items are a pass of eight for each of 256 workgroups; 60 were two for many of them, 1.35 times as long"""
    cfg, lay, m = layer("f2", 1024, 768, 64, 128, None)
    x = torch.from_numpy(synth.normed_x(np.random.default_rng(76), 128, 1024)).cuda()
    us = []
    for used in (64, 60):
        ids, w = evenly(2 * used, used, 77)
        us.append(min(down_stage(lambda: m.experts(0, x[:2 * used].contiguous(), ids, w))[0] for _ in range(12)))
    print("64 tiles %.1f us, 60 tiles %.1f us" % tuple(us))
    assert us[1] <= 1.15 * us[0], us
    m.close()
