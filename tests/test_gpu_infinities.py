"""Infinite activations, and finite ones whose SwiGLU product overflows, on raw rows, whose kernels split activations into fp16 terms: signed
infinities come out where sums of f32 products give them. Every weight is given one sign here, so that no sum holds infinities of both."""
import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.redmetal_ffn import RedMetalFfnPool
from gpu_common import rel_l2
from test_gpu_topk_pool import Case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def one_sign(matrix, negative):
    """IQ2_XXS rows with every sign field 0 (plus) or 127 (minus, the eighth sign by parity)"""
    words = matrix.reshape(matrix.shape[0], -1, 66)[:, :, 2:].reshape(matrix.shape[0], -1, 8, 8).copy()
    field = np.ascontiguousarray(words[..., 4:]).view(np.uint32)
    field[...] = (field & np.uint32(0xF0000000)) | np.uint32(0x0FFFFFFF if negative else 0)
    words[..., 4:] = field.view(np.uint8)
    matrix.reshape(matrix.shape[0], -1, 66)[:, :, 2:] = words.reshape(matrix.shape[0], -1, 64)


@pytest.mark.parametrize("negative", [False, True])
@pytest.mark.parametrize("what", ["infinite input", "overflowing product"])
def test_signed_infinities(tmp_path, monkeypatch, what, negative):
    plain = synth.make_layer

    def signed(seed, cfg):
        lay = plain(seed, cfg)
        one_sign(lay["gate"], False)
        one_sign(lay["up"], negative)
        one_sign(lay["down"], False)
        return lay
    monkeypatch.setattr(synth, "make_layer", signed)
    zeros = np.zeros(512 * 8, np.int8), np.zeros(2048 * 8, np.int8)
    hidden, ffn, n_expert, ntok, top_k = 512, 256, 8, 20, 4
    c = Case(tmp_path, zeros, "iq2", hidden=hidden, ffn=ffn, n_expert=n_expert, seed=841)
    rng = np.random.default_rng(15)
    x = np.abs(synth.normed_x(rng, ntok, hidden))
    bad = [0, 5, 19]
    for t in bad:
        if what == "infinite input":
            x[t, 100 + t] = np.inf
            x[t, 200] = 3e38
        else:
            x[t] *= np.float32(1e25)
    with np.errstate(all="ignore"):
        ids = np.stack([rng.permutation(n_expert)[:top_k] for _ in range(ntok)]).astype(np.uint32)
        w = rng.random((ntok, top_k)).astype(np.float32) + 0.1
        inf = np.full(hidden, -np.inf if negative else np.inf, np.float32)
        got, _ = c.pool.execute([c.slot_of[int(e)] for e in ids[5]], [c.layouts[int(e)] for e in ids[5]], w[5], c.word, hidden, ffn, 0, hidden, x[5])
        assert np.array_equal(got, inf)
        uid, start, ptok, pw, tp = orc.group_pairs(ids, w, n_expert)
        slots = [c.slot_of[int(e)] for e in uid]
        x_dev, out = torch.from_numpy(x).cuda(), torch.zeros((ntok, hidden), device="cuda")
        c.pool.encode_batched(torch.cuda.current_stream().cuda_stream, slots, [c.layouts[int(e)] for e in uid], c.word, hidden, ffn, 0, ntok, top_k, ptok, pw, start, tp,
                              x_dev.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        c.pool.release(slots)
        for t, row in enumerate(out.cpu().numpy()):
            assert np.array_equal(row, inf) if t in bad else rel_l2(row, c.want(ids[t], w[t], x[t])) <= 1e-6, t
        one = RedMetalFfnPool(c.path, 4 * c.slot_bytes + 65536, c.slot_bytes)
        one.load(0, c.layouts[3])
        got, _ = one.execute(0, c.layouts[3], c.word, hidden, ffn, 0, hidden, x[19])
        assert np.array_equal(got, inf)
        one.close()
    c.pool.close()
