"""How far the matrix-instruction kernels on quantised experts are from the same sums in double precision.

Bounds. A rounding to f32 loses 2.4e-8 of a value (root mean square), n of them behind one another, while a sum of independent terms grows to
its full size, sqrt(n / 2) times that. Rows of 2048 x 512 multiplied in f32, a lane adding 32 products before the lanes' sums meet, come out
2.1e-7 off after gate, up, SwiGLU, down and the weighted sum. The kernels here split activations into fp16 halves (22 bits: 0.8e-7 of those
2.1e-7) and add on the matrix unit, which rounds four times per instruction: with 16 roundings behind one another per block (0.7e-7 in each of
the three products) they stay below that; with 64 they were at 2.9e-7."""
import json
import os

import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import moe as moe_api
from dwarfstar_red_lite_amd import synth
from test_gpu_staged_tiles import routing_with
from test_gpu_topk_pool import Case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
F32_CHUNK, F32_TOKEN = 2.3e-7, 2.1e-7


@pytest.fixture(scope="module")
def grids(golden_dir):
    g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
    xs, m = (np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m"))
    orc.set_codebooks(xs, m)
    moe_api.set_codebooks(xs, m)
    return xs, m


def rel(got, want):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


def pool_chunk(c, hidden, ffn, counts, ntok, top_k, x, rng, pick):
    ids = routing_with(counts, ntok, top_k, rng)
    w = rng.random((ntok, top_k)).astype(np.float32) + 0.1
    uid, start, ptok, pw, tp = orc.group_pairs(ids, w, len(counts))
    x_dev, out = torch.from_numpy(x).cuda(), torch.zeros((ntok, hidden), device="cuda")
    slots = [c.slot_of[int(e)] for e in uid]
    c.pool.encode_batched(torch.cuda.current_stream().cuda_stream, slots, [c.layouts[int(e)] for e in uid], c.word, hidden, ffn, 0, ntok, top_k, ptok, pw, start, tp,
                          x_dev.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    c.pool.release(slots)
    got = out.cpu().numpy()
    return rel(got[pick], np.stack([c.want(ids[t], w[t], x[t]) for t in pick]))


# raw rows and tile-major copies; tiles of 16 pairs (the first two sizes) and of 32
@pytest.mark.parametrize("layout", ["iq2", "f2", "xs", "m"])
@pytest.mark.parametrize("hidden,ffn,tiles,wide", [(2048, 512, False, False), (1024, 256, True, False), (512, 512, False, True), (1024, 256, True, True)])
def test_chunk_of_pairs(tmp_path, grids, layout, hidden, ffn, tiles, wide):
    c = Case(tmp_path, grids, layout, hidden=hidden, ffn=ffn, n_expert=12, seed=821, fast=tiles, tiles=tiles)
    rng = np.random.default_rng(4)
    ntok, counts = (8100, [2700] * 12) if wide else (24, [8] * 12)
    x = synth.normed_x(rng, ntok, hidden)
    pick = rng.choice(ntok, 24, replace=False)
    assert pool_chunk(c, hidden, ffn, counts, ntok, 4, x, rng, pick) <= F32_CHUNK
    c.pool.close()


@pytest.mark.parametrize("layout,wide", [("iq2", False), ("iq2", True), ("xs", False)])
def test_small_activations_beside_large_ones(tmp_path, grids, layout, wide, monkeypatch):
    """The block that holds a token's largest values meets weights of scale zero: the result hangs on values 2^-18 of the largest, and
    keeps their 22 bits."""
    hidden, ffn = 512, 256
    plain = synth.make_layer

    def first_block_zero(seed, cfg):
        lay = plain(seed, cfg)
        t = cfg["gate_up_type"]
        for k in ("gate", "up"):
            b = lay[k].reshape(cfg["n_expert"], cfg["ffn"], cfg["hidden"] // 256, synth.BLOCK_BYTES[t])
            b[:, :, 0, synth.D_OFFSET[t]:synth.D_OFFSET[t] + 2] = 0
        return lay
    monkeypatch.setattr(synth, "make_layer", first_block_zero)
    c = Case(tmp_path, grids, layout, hidden=hidden, ffn=ffn, n_expert=12, seed=823)
    rng = np.random.default_rng(6)
    ntok, counts = (8100, [2700] * 12) if wide else (24, [8] * 12)
    x = synth.normed_x(rng, ntok, hidden)
    x[:, :256] *= np.float32(2.0 ** 18)
    pick = rng.choice(ntok, 24, replace=False)
    assert pool_chunk(c, hidden, ffn, counts, ntok, 4, x, rng, pick) <= F32_CHUNK
    c.pool.close()


@pytest.mark.parametrize("layout", ["f2", "m"])
def test_wide_experts_of_a_mixed_layer(layout, grids):
    """ffn 768: routed experts on raw rows, the shared expert's dense f32 rows on the matrix unit's f32 products (on IQ1_M layers the larger part of the output)"""
    H, F, E, K, ntok = 2048, 768, 16, 4, 40
    cfg = synth.layer_config(hidden=H, ffn=F, n_expert=E, top_k=K, layout=layout)
    lay = synth.make_layer(61, cfg)
    m = moe_api.ResidentMoe(cfg, n_layer=1, max_tokens=ntok)
    m.load_layer(0, lay)
    rng = np.random.default_rng(62)
    x = synth.normed_x(rng, ntok, H)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(ntok)]).astype(np.uint32)
    w = rng.random((ntok, K)).astype(np.float32)
    w /= w.sum(axis=1, keepdims=True)
    got = m.experts(0, torch.from_numpy(x).cuda(), torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w).cuda()).cpu().numpy()
    pick = range(0, ntok, 4)
    want = []
    for t in pick:
        y = sum(float(w[t, k]) * orc.expert_ffn(cfg["gate_up_type"], cfg["down_type"], lay["gate"][e], lay["up"][e], lay["down"][e], H, F, x[t]) for k, e in enumerate(ids[t]))
        gate = 1.0 / (1.0 + np.exp(-float(np.dot(lay["sh_gate_inp"].astype(np.float64), x[t].astype(np.float64)))))
        want.append(y + gate * orc.expert_ffn(cfg["sh_gate_up_type"], cfg["sh_down_type"], lay["sh_gate"], lay["sh_up"], lay["sh_down"], H, F, x[t]))
    assert rel(got[list(pick)], np.stack(want)) <= F32_CHUNK
    m.close()


@pytest.mark.parametrize("layout", ["iq2", "f2", "xs", "m"])
def test_one_token(tmp_path, grids, layout):
    hidden, ffn = 2048, 512
    c = Case(tmp_path, grids, layout, hidden=hidden, ffn=ffn, n_expert=16, seed=825)
    rng = np.random.default_rng(12)
    got, want = [], []
    for _ in range(6):
        experts, w, x = rng.permutation(16)[:10], rng.random(10).astype(np.float32) + 0.05, synth.normed_x(rng, 1, hidden)[0]
        got.append(c.pool.execute([c.slot_of[int(e)] for e in experts], [c.layouts[e] for e in experts], w, c.word, hidden, ffn, 0, hidden, x)[0])
        want.append(c.want(experts, w, x))
    assert rel(np.stack(got), np.stack(want)) <= F32_TOKEN
    c.pool.close()
