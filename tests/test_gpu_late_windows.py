"""Chunks whose tokens are a window of a longer sequence (tok_first > 0): only the rows that the pairs name are read of the input, which
may therefore be all there is."""
import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import synth
from gpu_common import rel_l2
from test_gpu_topk_pool import Case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("layout,copies", [("iq2", False), ("f2", True)])
@pytest.mark.parametrize("tok_first,named", [(0, 0), (1, 1), (2000, 2000), (2000, 1995)])      # (named: the first row that a pair names)
def test_rows_in_front_of_the_window(tmp_path, layout, copies, tok_first, named):
    zeros = np.zeros(512 * 8, np.int8), np.zeros(2048 * 8, np.int8)
    hidden, ffn, n_expert, ntok, top_k = 512, 256, 6, 21, 3
    c = Case(tmp_path, zeros, layout, hidden=hidden, ffn=ffn, n_expert=n_expert, seed=861, fast=copies, tiles=copies)
    rng = np.random.default_rng(18)
    rows = tok_first + ntok - named
    x = synth.normed_x(rng, rows, hidden)
    ids = np.stack([rng.permutation(n_expert)[:top_k] for _ in range(ntok)]).astype(np.uint32)
    w = rng.random((ntok, top_k)).astype(np.float32) + 0.1
    uid, start, ptok, pw, tp = orc.group_pairs(ids, w, n_expert)
    row_of = np.arange(ntok) + (tok_first - named)
    row_of[0] = 0                                        # (token 0's input is the first row named)
    ptok = (row_of[ptok] + named).astype(np.uint32)
    x_dev, out = torch.from_numpy(x).cuda(), torch.full((tok_first + ntok, hidden), 7.0, device="cuda")
    slots = [c.slot_of[int(e)] for e in uid]
    c.pool.encode_batched(torch.cuda.current_stream().cuda_stream, slots, [c.layouts[int(e)] for e in uid], c.word, hidden, ffn, tok_first, ntok, top_k, ptok, pw, start, tp,
                          x_dev.data_ptr() - named * hidden * 4, out.data_ptr())
    torch.cuda.synchronize()
    c.pool.release(slots)
    got = out.cpu().numpy()
    assert (got[:tok_first] == 7.0).all()
    for t in range(ntok):
        assert rel_l2(got[tok_first + t], c.want(ids[t], w[t], x[row_of[t]])) <= 1e-6, t
    c.pool.close()
