"""Pools whose IQ2_XS / IQ1_M codebooks hold any int8 value (the kernels on the matrix units hold weights of eleven bits and take only
codebooks of smaller entries) and codebooks at that limit: one token, a chunk, one expert, with and without the slots' copies."""
import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.redmetal_ffn import RedMetalFfnPool
from gpu_common import rel_l2
from test_gpu_topk_pool import Case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def codebooks(values):
    """any int8, the largest entries that fit eleven bits, or large ones that fit for their trailing zeros"""
    rng = np.random.default_rng(77)
    pick = {"any": (np.arange(-128, 128), np.arange(-128, 128)), "limit": (np.array([-66, -65, 65, 66]), np.array([-16, -15, 0, 16])),
            "zeros": (np.array([-128, -100, 96, 120]), np.array([-16, 16])), "beyond": (np.array([67, -67, 1]), np.array([17, -17, 1]))}[values]
    return rng.choice(pick[0].astype(np.int8), 512 * 8), rng.choice(pick[1].astype(np.int8), 2048 * 8)


@pytest.mark.parametrize("layout", ["xs", "m"])
@pytest.mark.parametrize("values,copies", [("any", False), ("any", True), ("limit", False), ("limit", True), ("zeros", False), ("beyond", False)])
def test_pools_decode_every_codebook(tmp_path, layout, values, copies):
    grids = codebooks(values)
    orc.set_codebooks(*grids)
    hidden, ffn, n_expert, ntok, top_k = 512, 256, 8, 20, 4
    c = Case(tmp_path, grids, layout, hidden=hidden, ffn=ffn, n_expert=n_expert, seed=831, fast=copies, tiles=copies)
    rng = np.random.default_rng(14)
    x = synth.normed_x(rng, ntok, hidden)
    ids = np.stack([rng.permutation(n_expert)[:top_k] for _ in range(ntok)]).astype(np.uint32)
    w = rng.random((ntok, top_k)).astype(np.float32) + 0.1
    want = [c.want(ids[t], w[t], x[t]) for t in range(ntok)]
    # f32 sums over weights that are exact
    got, _ = c.pool.execute([c.slot_of[int(e)] for e in ids[0]], [c.layouts[int(e)] for e in ids[0]], w[0], c.word, hidden, ffn, 0, hidden, x[0])
    assert rel_l2(got, want[0]) <= 1e-6
    uid, start, ptok, pw, tp = orc.group_pairs(ids, w, n_expert)
    slots = [c.slot_of[int(e)] for e in uid]
    x_dev, out = torch.from_numpy(x).cuda(), torch.zeros((ntok, hidden), device="cuda")
    c.pool.encode_batched(torch.cuda.current_stream().cuda_stream, slots, [c.layouts[int(e)] for e in uid], c.word, hidden, ffn, 0, ntok, top_k, ptok, pw, start, tp,
                          x_dev.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    c.pool.release(slots)
    assert max(rel_l2(g, v) for g, v in zip(out.cpu().numpy(), want)) <= 1e-6
    if not copies:
        one = RedMetalFfnPool(c.path, 4 * c.slot_bytes + 65536, c.slot_bytes, iq2_xs_grid=grids[0], iq1_m_grid=grids[1])
        one.load(0, c.layouts[3])
        got, _ = one.execute(0, c.layouts[3], c.word, hidden, ffn, 0, hidden, x[1])
        assert rel_l2(got, c.want([3], [1.0], x[1])) <= 1e-6
        one.close()
    c.pool.close()
