"""Tiles of up to eight pairs, which multiply the high and the low halves of their activations in one instruction: experts with 1, 7, 8 and 9 pairs, and with
as many behind full tiles of 16 and 32, as the only tiles of a chunk and beside larger ones."""
import numpy as np
import pytest

from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe
from gpu_common import rel_l2
from test_gpu_moe_batch import oracle_tokens
from test_gpu_staged_tiles import grids, routing_with      # noqa: F401 (fixture)
from test_gpu_topk_pool import Case
import oracle_lib as orc

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

COUNTS = {"small": ([8, 7, 1, 8, 5, 2, 8, 1, 4, 8, 3, 1], 14), "edges": ([8, 9, 7, 1, 24, 25, 40, 41, 2, 16, 48, 59], 70), "none": ([9, 16, 12, 25, 9, 10, 9, 14, 9, 13, 9, 9], 36)}
# two matrices deep, each 1.8e-7 off: eight 32-bit roundings of a row's sum and the low half's 22 bits stay below it
TOL = 1e-6


# K parts 2 / 4 / 8 of the gate/up kernel, 1 .. 4 of the down kernel, every row format
@pytest.mark.parametrize("counts", sorted(COUNTS))
@pytest.mark.parametrize("layout,hidden,ffn", [("iq2", 2048, 512), ("f2", 512, 256), ("xs", 1024, 768), ("m", 2048, 1024), ("f2", 1024, 512)])
def test_small_tiles(tmp_path, grids, layout, hidden, ffn, counts):      # noqa: F811
    n_expert, top_k = 12, 4
    counts, ntok = COUNTS[counts]
    c = Case(tmp_path, grids, layout, hidden=hidden, ffn=ffn, n_expert=n_expert, seed=77)
    rng = np.random.default_rng(5)
    ids = routing_with(counts, ntok, top_k, rng)
    w = rng.random((ntok, top_k)).astype(np.float32) + 0.1
    uid, start, ptok, pw, tp = orc.group_pairs(ids, w, n_expert)
    x = synth.normed_x(rng, ntok, hidden)
    x[2] *= 1e-6                                             # (a pair's scale is its own)
    x[3] *= 1e5
    x_dev, out = torch.from_numpy(x).cuda(), torch.zeros((ntok, hidden), device="cuda")
    slots = [c.slot_of[int(e)] for e in uid]
    c.pool.encode_batched(torch.cuda.current_stream().cuda_stream, slots, [c.layouts[int(e)] for e in uid], c.word, hidden, ffn, 0, ntok, top_k, ptok, pw, start, tp,
                          x_dev.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    c.pool.release(slots)
    got = out.cpu().numpy()
    for t in range(ntok):
        assert rel_l2(got[t], c.want(ids[t], w[t], x[t])) <= TOL, (layout, hidden, ffn, t)
    c.pool.close()


# The same pairs on resident layers: tile-major copies (IQ3_S words of the down operand among them), packed rows (iq2 of 512 x 1024), raw rows beside a dense shared
# expert (768). On iq2 the shared expert's tiles stand in the same list; its last one has 1, 7, 8 and 9 pairs.
@pytest.mark.parametrize("ntok", [33, 39, 40, 41])
@pytest.mark.parametrize("layout,hidden,ffn", [("iq2", 2048, 512), ("iq2", 512, 1024), ("f2", 2048, 512), ("f2", 1024, 768), ("xs", 2048, 512), ("m", 1024, 256)])
def test_small_tiles_of_resident_layers(grids, layout, hidden, ffn, ntok):      # noqa: F811
    n_expert, top_k = 12, 4
    counts = [1, 7, 8, 9, 17, 23, 24, 25]
    rest = ntok * top_k - sum(counts)
    counts += [rest // 4 + (i < rest % 4) for i in range(4)]
    orc.set_codebooks(*grids)
    cfg = synth.layer_config(hidden=hidden, ffn=ffn, n_expert=n_expert, top_k=top_k, layout=layout)
    lay, rng = synth.make_layer(78, cfg), np.random.default_rng(6)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=ntok)
    m.load_layer(0, lay)
    ids = routing_with(counts, ntok, top_k, rng)
    w = rng.random((ntok, top_k)).astype(np.float32) + 0.1
    x = synth.normed_x(rng, ntok, hidden)
    x[2] *= 1e-6
    x[3] *= 1e5
    got = m.experts(0, torch.from_numpy(x).cuda(), torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w).cuda()).cpu().numpy()
    want = oracle_tokens(cfg, lay, x, ids, w)
    off = [rel_l2(got[t], want[t]) for t in range(ntok)]
    assert max(off) <= TOL, (layout, hidden, ffn, int(np.argmax(off)), max(off))
    m.close()


# Behind wide tiles: 84 of 32 pairs an expert are enough for the wide launches, and the narrow ones find the remainders alone
@pytest.mark.parametrize("layout,hidden,ffn", [("f2", 1024, 512), ("m", 2048, 512)])
def test_small_tiles_behind_wide_ones(tmp_path, grids, layout, hidden, ffn):      # noqa: F811
    n_expert, top_k, rest = 12, 4, [1, 7, 8, 9, 17, 24, 2, 16, 5, 3, 4, 0]
    counts = [84 * 32 + r for r in rest]
    ntok = sum(counts) // top_k
    c = Case(tmp_path, grids, layout, hidden=hidden, ffn=ffn, n_expert=n_expert, seed=79)
    rng = np.random.default_rng(7)
    ids = routing_with(counts, ntok, top_k, rng)
    w = rng.random((ntok, top_k)).astype(np.float32) + 0.1
    uid, start, ptok, pw, tp = orc.group_pairs(ids, w, n_expert)
    x = synth.normed_x(rng, ntok, hidden)
    x_dev, out = torch.from_numpy(x).cuda(), torch.zeros((ntok, hidden), device="cuda")
    slots = [c.slot_of[int(e)] for e in uid]
    c.pool.encode_batched(torch.cuda.current_stream().cuda_stream, slots, [c.layouts[int(e)] for e in uid], c.word, hidden, ffn, 0, ntok, top_k, ptok, pw, start, tp,
                          x_dev.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    c.pool.release(slots)
    got = out.cpu().numpy()
    last = {int(ptok[p]) for u, e in enumerate(uid) for p in range(int(start[u + 1]) - min(rest[int(e)], 9), int(start[u + 1]))}      # tokens of the remainders' last pairs
    assert len(last) >= 19                                   # (73 pairs, at most four a token)
    for t in sorted(last):
        assert rel_l2(got[t], c.want(ids[t], w[t], x[t])) <= TOL, (layout, hidden, ffn, t)
    c.pool.close()
