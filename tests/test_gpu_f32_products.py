"""The f32 products of a chunk on the bf16 matrix units (three terms for each f32): every tile they are cut into, activations at any float of
memory and of any scale, and infinities, against sums in double."""
import numpy as np
import pytest

from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# of the rms of a token's outputs: 0.74e-7 was measured over 3000 outputs of 2048 columns (eight parts of two chains of four additions, each rounded to
# 2^-25 of a partial sum, the products left out at 2^-24 of the others, the result's own 2^-25); one token's outputs spread around that, and one product
# that outweighs the rest shows the last two undiluted: 2^-24 + 2^-25 = 0.9e-7 with the chains' roundings of it, each at most 2^-25, beside them
TOL = 2e-7


def layer(hidden, n_expert, **kw):
    cfg = synth.layer_config(hidden=hidden, ffn=256, n_expert=n_expert, top_k=2, layout="iq2", **kw)
    lay = synth.make_layer(41, cfg)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=2100)
    m.load_layer(0, lay)
    return m, np.frombuffer(np.ascontiguousarray(lay["router"]).tobytes(), np.float32).reshape(n_expert, hidden)


def check(logits, x, rows):
    want = x.astype(np.float64) @ rows.T.astype(np.float64)
    err = np.sqrt(((logits - want) ** 2).mean(axis=1) / (want ** 2).mean(axis=1))
    assert err.max() <= TOL, err.max()


# 16 rows of 32 x 16, 300 experts' rows (a ragged last block) and tiles of every size: up to 77, 512 and 2048 tokens
@pytest.mark.parametrize("hidden,n_expert,tokens", [(512, 16, (41, 47)), (1024, 300, (77, 513)), (2048, 512, (40, 77, 512, 2047)), (1536, 48, (49,))])
def test_logits(hidden, n_expert, tokens):
    m, rows = layer(hidden, n_expert)
    for n in tokens:
        x = synth.normed_x(np.random.default_rng(n), n, hidden)
        x *= np.float32(10.0) ** np.random.default_rng(1).integers(-28, 29, size=(n, 1)).astype(np.float32)      # a scale per token
        x[3, 11] *= np.float32(1e5)      # one product that outweighs the others: what its terms leave out (2^-24 of it) is seen undiluted
        check(m.route(0, torch.from_numpy(x).cuda())[2].cpu().numpy(), x, rows)
    m.close()


@pytest.mark.parametrize("hidden,outweigh", [(512, 1.0), (2048, 1.0), (512, 1e5), (2048, 1e5)])
def test_terms_are_rounded(hidden, outweigh):
    """Terms that are cut instead of rounded leave out products that all have the sign of the whole: sums come out 3e-8 .. 4e-8 too small in magnitude
    (the products left out, by themselves; rounded 1e-10), which a bound on the error itself does not see. Rounding errors of either sign, 1e-7 of each of
    513 x 256 outputs (a token's share one factor where a product outweighs the rest), leave less than 1e-8 of a mean."""
    m, rows = layer(hidden, 256)
    x = synth.normed_x(np.random.default_rng(9), 513, hidden)
    x[:, 11] *= np.float32(outweigh)
    logits, want = m.route(0, torch.from_numpy(x).cuda())[2].cpu().numpy(), x.astype(np.float64) @ rows.T.astype(np.float64)
    bias = ((logits - want) * np.sign(want)).mean() / np.abs(want).mean()
    print("%d columns, outweighed %g: %.1e" % (hidden, outweigh, bias))
    assert abs(bias) <= 1e-8
    m.close()


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_activations_at_any_float(shift):
    m, rows = layer(1024, 48)
    n = 45
    x = synth.normed_x(np.random.default_rng(3), n, 1024)
    room = torch.zeros(n * 1024 + 4, device="cuda")
    room[shift:shift + n * 1024] = torch.from_numpy(x).cuda().reshape(-1)
    aligned = m.route(0, torch.from_numpy(x).cuda())[2].cpu().numpy()
    got = m.route(0, room[shift:shift + n * 1024].reshape(n, 1024))[2].cpu().numpy()
    assert np.array_equal(got, aligned)
    check(got, x, rows)
    m.close()


def test_infinities_and_overflow():
    m, rows = layer(512, 64)
    n = 44
    x = synth.normed_x(np.random.default_rng(4), n, 512)
    plain = m.route(0, torch.from_numpy(x).cuda())[2].cpu().numpy()
    y = x.copy()
    y[3, 100], y[20, 7], y[20, 300], y[43, 11], y[30, 0] = np.inf, 3e38, -np.inf, np.nan, 3.4e38
    got = m.route(0, torch.from_numpy(y).cuda())[2].cpu().numpy()
    ok = [t for t in range(n) if t not in (3, 20, 43, 30)]
    assert np.array_equal(got[ok], plain[ok])
    assert np.array_equal(got[3], np.where(rows[:, 100] > 0, np.inf, -np.inf).astype(np.float32)) and (rows[:, 100] != 0).all()
    assert np.array_equal(got[20], np.where(rows[:, 300] > 0, -np.inf, np.inf).astype(np.float32)) and (rows[:, 300] != 0).all()
    assert np.isnan(got[43]).all()
    check(got[30:31], y[30:31], rows)
    m.close()


def test_shared_expert_in_front_and_beside(golden_dir):
    """gate and up products of the shared expert in the launch in front of the routing (up to 448 workgroups: 352 tokens here) or of a given routing
    (256: 224 tokens), and on a stream of their own beyond: a token gets the same from either"""
    import oracle_lib as orc
    from gpu_common import REL_L2_TOL, rel_l2
    cfg = synth.layer_config(hidden=512, ffn=256, n_expert=64, top_k=4, layout="f2")
    lay = synth.make_layer(43, cfg)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=400)
    m.load_layer(0, lay)
    x = synth.normed_x(np.random.default_rng(5), 400, 512)
    x_dev = torch.from_numpy(x).cuda()
    whole = m.forward(0, x_dev).cpu().numpy()
    ids, w, _ = m.last_route(400)
    pick = [0, 7, 32, 33, 39]
    want, cids, _, _ = orc.Layer(cfg, **lay).forward(np.ascontiguousarray(x[pick]), threads=8)
    same = [i for i, t in enumerate(pick) if np.array_equal(ids[t], cids[i])]
    assert len(same) >= len(pick) - 1 and max(rel_l2(whole[pick[i]], want[i]) for i in same) <= REL_L2_TOL
    ids_dev, w_dev = torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w).cuda()
    for n in (40, 225, 352, 353, 368, 384):
        got = m.forward(0, x_dev[:n]).cpu().numpy()
        assert max(rel_l2(got[t], whole[t]) for t in range(n)) <= 1e-6, n
    for n in (33, 208, 224, 225, 240):
        got = m.experts(0, x_dev[:n], ids_dev[:n].contiguous(), w_dev[:n].contiguous()).cpu().numpy()
        assert max(rel_l2(got[t], whole[t]) for t in range(n)) <= 1e-6, n
    m.close()
