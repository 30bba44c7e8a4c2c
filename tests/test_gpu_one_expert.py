"""One expert per call (redmetal_ffn_*): synchronous calls that follow each other without a wait between, each with an input of its own, and
the enqueued form on an input that does not begin at a multiple of sixteen bytes."""
import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import expert_type_word, synth
from dwarfstar_red_lite_amd.gguf_writer import write_moe_gguf
from dwarfstar_red_lite_amd.moe import gguf_expert_layout
from dwarfstar_red_lite_amd.redmetal_ffn import ExpertLayout, RedMetalFfnPool
from gpu_common import rel_l2

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


class Experts:
    def __init__(self, tmp_path, layout, hidden, ffn, n):
        self.cfg = synth.layer_config(hidden=hidden, ffn=ffn, n_expert=n, top_k=1, layout=layout)
        self.lay = synth.make_layer(851, self.cfg)
        path = str(tmp_path / "one.gguf")
        write_moe_gguf(path, self.cfg, [self.lay])
        names = ("gate_offset", "gate_bytes", "up_offset", "up_bytes", "down_offset", "down_bytes")
        self.at = [ExpertLayout(*(gguf_expert_layout(path, n, 0, e)[k] for k in names)) for e in range(n)]
        size = 2 * self.at[0].gate_bytes + self.at[0].down_bytes
        self.pool = RedMetalFfnPool(path, (n + 1) * (size + 4096), size)
        for e in range(n):
            self.pool.load(e, self.at[e])
        self.word, self.shape = expert_type_word(self.cfg["gate_up_type"], self.cfg["down_type"]), (hidden, ffn)

    def want(self, e, x, row_start, row_count):
        c = self.cfg
        return orc.expert_ffn(c["gate_up_type"], c["down_type"], self.lay["gate"][e], self.lay["up"][e], self.lay["down"][e], *self.shape, x, row_start, row_count)


@pytest.mark.parametrize("layout,hidden,ffn", [("f2", 2048, 512), ("iq2", 256, 256)])
def test_calls_behind_one_another(tmp_path, layout, hidden, ffn):
    ex = Experts(tmp_path, layout, hidden, ffn, 4)
    rng = np.random.default_rng(16)
    x = synth.normed_x(rng, 50, hidden)
    calls = [(int(rng.integers(4)), i, *((0, hidden) if i % 3 else (int(rng.integers(hidden - 9)), 9))) for i in range(50)]
    out = [[ex.pool.execute(e, ex.at[e], ex.word, hidden, ffn, start, count, x[i])[0] for e, i, start, count in calls] for _ in range(4)]
    for k, (e, i, start, count) in enumerate(calls):
        assert rel_l2(out[0][k], ex.want(e, x[i], start, count)) <= 2e-6, k
        assert all(np.array_equal(out[0][k], o[k]) for o in out[1:]), k
    ex.pool.close()


@pytest.mark.parametrize("layout,hidden,ffn", [("f2", 2048, 512), ("iq2", 512, 256)])
def test_enqueued_call_with_an_input_at_any_float(tmp_path, layout, hidden, ffn):
    ex = Experts(tmp_path, layout, hidden, ffn, 2)
    x = synth.normed_x(np.random.default_rng(17), 1, hidden)[0]
    for off in (0, 1, 2, 3):
        buf, out = torch.full((hidden + 4,), float("nan"), device="cuda"), torch.full((hidden + 4,), float("nan"), device="cuda")
        buf[off:off + hidden] = torch.from_numpy(x).cuda()
        ex.pool.execute_noalloc(1, ex.at[1], ex.word, hidden, ffn, 3, hidden - 3, buf[off:].data_ptr(), out[off:].data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert rel_l2(got[off:off + hidden - 3], ex.want(1, x, 3, hidden - 3)) <= 2e-6, off
        assert np.isnan(got[:off]).all() and np.isnan(got[off + hidden - 3:]).all()
    ex.pool.close()
