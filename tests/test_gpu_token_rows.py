"""One token on raw rows (csrc/redhip_token.hip) against the CPU path: every row format, numbers of 256-column blocks below, at and beyond
what the waves of a workgroup take at once, down products of one to many units, row windows that begin and end inside sixteen rows."""
import json
import os

import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import synth
from gpu_common import rel_l2
from test_gpu_topk_pool import Case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def grids(golden_dir):
    g = json.load(open(os.path.join(golden_dir, "iq_grids.json")))
    xs, m = (np.frombuffer(bytes.fromhex(g[k]), np.int8) for k in ("iq2_xs", "iq1_m"))
    orc.set_codebooks(xs, m)
    return xs, m


# gate/up: 1 .. 4 blocks (two groups of rows per workgroup), 5 .. 8, 9 (a second trip); down: blocks x experts = 1 .. 8 units on the small workgroups, 9 .. on the large
@pytest.mark.parametrize("layout,hidden,ffn", [("iq2", 256, 256), ("f2", 512, 512), ("xs", 1024, 768), ("m", 1280, 256), ("f2", 2048, 256), ("xs", 2304, 512), ("m", 512, 1280),
                                               ("iq2", 2304, 256)])
def test_rows_of_one_token(tmp_path, grids, layout, hidden, ffn):
    c = Case(tmp_path, grids, layout, hidden=hidden, ffn=ffn, n_expert=16, seed=907)
    rng = np.random.default_rng(11)
    for top_k, row_start, row_count in ((1, 0, hidden), (2, 5, 30), (3, 0, hidden), (5, hidden - 17, 17), (8, 0, hidden), (9, hidden - 1, 1), (16, 3, hidden - 3)):
        experts = rng.permutation(16)[:top_k]
        w = rng.random(top_k).astype(np.float32) + 0.05
        x = synth.normed_x(rng, 1, hidden)[0]
        x[::3] *= 1e-4                         # (small values beside large ones in every block)
        x *= np.float32(10.0 ** rng.integers(-3, 3))
        got, _ = c.pool.execute([c.slot_of[int(e)] for e in experts], [c.layouts[e] for e in experts], w, c.word, hidden, ffn, row_start, row_count, x)
        assert rel_l2(got, c.want(experts, w, x, row_start, row_count)) <= 2e-6, (top_k, row_start)
    c.pool.close()
