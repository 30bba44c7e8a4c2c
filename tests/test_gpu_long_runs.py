"""Chunks of so many tiles that a workgroup of the tile kernels has more of them than it keeps notes of at a time (32): the run is cut into parts.
What a token gets does not depend on the chunk it is in, so the large call has to agree with calls of 3000 tokens."""
import json
import os

import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import synth
from gpu_common import rel_l2

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def grids(golden_dir):
    g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
    xs, m = (np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m"))
    orc.set_codebooks(xs, m)
    return xs, m


# 22000 pairs an expert: 688 tiles of 32, 8256 in all (and the shared expert's), 33 and more in a run of 256; 24 experts of 11000 pairs: 344 tiles of
# 32 each, a down matrix of three blocks (half as many: 17 a run)
@pytest.mark.parametrize("layout,ffn,n_expert,ntok", [("iq2", 256, 12, 66000), ("m", 768, 24, 33000), ("m", 768, 24, 66000)])
def test_more_tiles_than_infos(grids, layout, ffn, n_expert, ntok):
    from dwarfstar_red_lite_amd import moe as moe_api
    hidden, top_k = 512, 4
    moe_api.set_codebooks(*grids)
    cfg = synth.layer_config(hidden=hidden, ffn=ffn, n_expert=n_expert, top_k=top_k, layout=layout)
    m = moe_api.ResidentMoe(cfg, n_layer=1, max_tokens=ntok)
    m.load_layer(0, synth.make_layer(17, cfg))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    x = torch.randn((ntok, hidden), device="cuda", generator=gen)
    ids = ((torch.arange(ntok)[:, None] * top_k + torch.arange(top_k)[None]) % n_expert).to(torch.int32).cuda()      # every expert as often
    w = torch.softmax(torch.randn((ntok, top_k), device="cuda", generator=gen), dim=1)
    whole = m.experts(0, x, ids, w)
    for t0 in (0, 21000, ntok - 3000):
        rows = slice(t0, t0 + 3000)
        part = m.experts(0, x[rows].contiguous(), ids[rows].contiguous(), w[rows].contiguous())
        assert rel_l2(whole[rows].cpu().numpy(), part.cpu().numpy()) <= 5e-7      # (each is 2e-7 off from exact)
    m.close()
