"""The tile kernels (csrc/redhip_tiles.hip) on raw and packed rows: chunks on the pool's slots and on resident layers without tile-major
copies, against the CPU path. Experts with 1, 15, 16, 17, 31, 32, 33 and more pairs (edges of the 16- and 32-pair tiles), few and
many wide tiles (few of them run as tiles of 16), every row format, every split of K."""
import json
import os

import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import synth
from gpu_common import REL_L2_TOL, rel_l2
from test_gpu_topk_pool import Case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def grids(golden_dir):
    g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
    xs, m = (np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m"))
    orc.set_codebooks(xs, m)
    return xs, m


def routing_with(counts, ntok, top_k, rng):
    """[ntok][top_k] distinct experts per token in which expert e appears counts[e] times: the experts with most left go to each token"""
    left = np.array(counts)
    assert left.sum() == ntok * top_k and left.max() <= ntok
    ids = np.empty((ntok, top_k), np.uint32)
    for t in range(ntok):
        pick = np.argsort(-left + 1e-3 * rng.random(len(left)))[:top_k]
        left[pick] -= 1
        ids[t] = rng.permutation(pick)
    assert (left == 0).all()
    return ids[rng.permutation(ntok)]


# (hidden, ffn): K parts 2 / 4 / 8 of the gate/up kernel, 1 / 2 / 3 / 4 of the down kernel
SHAPES = [("iq2", 512, 256), ("f2", 1024, 512), ("xs", 2048, 768), ("m", 512, 1024), ("iq2", 1024, 768), ("f2", 512, 768), ("xs", 512, 512), ("m", 1024, 256),
          ("f2", 2048, 256), ("xs", 1024, 1024), ("m", 512, 768), ("iq2", 512, 1024), ("f2", 512, 1024)]
# 1008 wide tiles are above both kernels' lines for these (290 million weights in them for gate/up, 200 million for down)
WIDE = [("iq2", 512, 512), ("iq2", 1024, 256), ("f2", 1024, 512), ("f2", 512, 768), ("f2", 1024, 256), ("f2", 512, 1024), ("xs", 512, 512), ("xs", 1024, 1024), ("m", 1024, 256),
        ("m", 512, 768), ("m", 2048, 512)]


@pytest.mark.parametrize("layout,hidden,ffn,many_wide", [s + (False,) for s in SHAPES] + [s + (True,) for s in WIDE])
def test_pool_slots(tmp_path, grids, layout, hidden, ffn, many_wide):
    n_expert, top_k = 12, 4
    c = Case(tmp_path, grids, layout, hidden=hidden, ffn=ffn, n_expert=n_expert, seed=811)
    rng = np.random.default_rng(3)
    if many_wide:      # 12 experts with 2700 pairs (84 tiles of 32 each): enough for the wide launches, remainders of 12, one wide remainder
        ntok = 8100
        counts = [2700] * n_expert
        counts[0] += 15
        counts[1] -= 15
    else:
        counts, ntok = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 3, 0], 73
    ids = routing_with(counts, ntok, top_k, rng)
    w = (rng.random((ntok, top_k)).astype(np.float32) + 0.1)
    uid, start, ptok, pw, tp = orc.group_pairs(ids, w, n_expert)
    x = synth.normed_x(rng, ntok, hidden)
    x[7] *= 1e-6
    x[9] *= 1e5
    x_dev, out = torch.from_numpy(x).cuda(), torch.zeros((ntok, hidden), device="cuda")
    slots = [c.slot_of[int(e)] for e in uid]
    args = (slots, [c.layouts[int(e)] for e in uid], c.word, hidden, ffn, 0, ntok, top_k, ptok, pw, start, tp, x_dev.data_ptr(), out.data_ptr())
    c.pool.encode_batched(torch.cuda.current_stream().cuda_stream, *args)
    torch.cuda.synchronize()
    c.pool.release(slots)
    got = out.cpu().numpy()
    out.zero_()
    c.pool.encode_batched(torch.cuda.current_stream().cuda_stream, *args)
    torch.cuda.synchronize()
    c.pool.release(slots)
    assert np.array_equal(got, out.cpu().numpy())            # the same every time
    for t in sorted({7, 9} | set(rng.choice(ntok, 20, replace=False).tolist())):
        assert rel_l2(got[t], c.want(ids[t], w[t], x[t])) <= 1e-5, (layout, hidden, ffn, t)
    c.pool.close()


@pytest.mark.parametrize("layout,shape,ntok", [("iq2", (2048, 768, 24, 4), 41), ("iq2", (512, 1024, 12, 6), 130), ("f2", (1024, 768, 12, 6), 130), ("xs", (2048, 768, 16, 4), 33),
                                               ("m", (1024, 1024, 16, 4), 48), ("m", (512, 768, 24, 4), 17)])
def test_resident_layers(layout, shape, ntok, grids):
    """own router (shared expert's tiles on all-IQ2_XXS layers, its dense products beside the tiles on the others) and given routing"""
    from dwarfstar_red_lite_amd.moe import ResidentMoe
    from test_gpu_moe_batch import oracle_tokens
    from test_gpu_moe_layer import ids_match_up_to_ties
    orc.set_codebooks(*grids)
    H, F, E, K = shape
    cfg = synth.layer_config(hidden=H, ffn=F, n_expert=E, top_k=K, layout=layout)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=ntok)
    lay = synth.make_layer(31 + H + F, cfg)
    m.load_layer(0, lay)
    rng = np.random.default_rng(29)
    xs = synth.normed_x(rng, ntok, H)
    xs[3:9] = xs[2]
    x_dev = torch.from_numpy(xs).cuda()
    out = m.forward(0, x_dev).cpu().numpy()
    gids, _, _ = m.last_route(ntok)
    want, cids, _, clog = orc.Layer(cfg, **lay).forward(xs, threads=8)
    for i in range(ntok):
        assert ids_match_up_to_ties(gids[i], cids[i], clog[i])
        assert rel_l2(out[i], want[i]) <= REL_L2_TOL, (layout, shape, i)
    assert np.array_equal(out[6], out[2])
    ids = synth.zipf_topk(rng, ntok, E, K)
    w = rng.random((ntok, K)).astype(np.float32)
    w /= w.sum(axis=1, keepdims=True)
    got = m.experts(0, x_dev, torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w).cuda()).cpu().numpy()
    want = oracle_tokens(cfg, lay, xs, ids, w)
    assert max(rel_l2(got[t], want[t]) for t in range(ntok)) <= REL_L2_TOL
    m.close()


def test_resident_packed_rows_in_wide_tiles(grids):
    """all-IQ2_XXS layers with ffn 768 have no tile-major copies: more than 70 wide tiles of packed gate/up rows, the shared expert's among them"""
    from dwarfstar_red_lite_amd.moe import ResidentMoe
    from test_gpu_moe_batch import oracle_tokens
    H, F, E, K, ntok = 2048, 768, 8, 4, 500
    cfg = synth.layer_config(hidden=H, ffn=F, n_expert=E, top_k=K, layout="iq2")
    m = ResidentMoe(cfg, n_layer=1, max_tokens=ntok)
    lay = synth.make_layer(41, cfg)
    m.load_layer(0, lay)
    rng = np.random.default_rng(30)
    xs = synth.normed_x(rng, ntok, H)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(ntok)]).astype(np.uint32)
    w = rng.random((ntok, K)).astype(np.float32)
    w /= w.sum(axis=1, keepdims=True)
    n = np.append(np.bincount(ids.ravel(), minlength=E), ntok)
    assert (n // 32 + (n % 32 > 16)).sum() >= 70
    got = m.experts(0, torch.from_numpy(xs).cuda(), torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w).cuda()).cpu().numpy()
    pick = rng.choice(ntok, 12, replace=False)
    want = oracle_tokens(cfg, lay, xs[pick], ids[pick], w[pick])
    assert max(rel_l2(got[t], want[i]) for i, t in enumerate(pick)) <= 1e-5
    m.close()
