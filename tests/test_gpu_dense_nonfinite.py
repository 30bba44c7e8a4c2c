"""The dense f32 products of a chunk (router, shared expert with its SwiGLU) where a product of three bf16 terms is not finite: activations just below
the largest float round to an infinite leading term. They meet weights of zero here, so the results are those of the other columns: outputs in double
say what they are, in every tile size, in the launch in front of the routing and beside it. Chunks of NaN cost a pass more, not a thread's loop."""
import numpy as np
import pytest

import oracle_lib as orc
from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
H, F, E, K, COL = 512, 256, 64, 4, 5
Q6K_SCALES, IQ2_D = 192, 0      # byte of a Q6_K block's sixteen scales (one per sixteen columns), of an IQ2_XXS block's d


def shared_only_layer(seed):
    """an F2 layer whose routed experts give nothing and on which no matrix sees columns 0 .. 15"""
    cfg = synth.layer_config(hidden=H, ffn=F, n_expert=E, top_k=K, layout="f2")
    lay = synth.make_layer(seed, cfg)
    lay["down"][:] = 0
    for k in ("gate", "up"):
        lay[k].reshape(-1, H // 256, synth.BLOCK_BYTES[cfg["gate_up_type"]])[:, 0, IQ2_D:IQ2_D + 2] = 0
    for k in ("router", "sh_gate", "sh_up"):
        lay[k].reshape(-1, H // 256, synth.BLOCK_BYTES[cfg["router_type"]])[:, 0, Q6K_SCALES] = 0
    lay["sh_gate_inp"][:16] = 0.0
    return cfg, lay


def shared_in_double(cfg, lay, x):
    g, u, d = (orc.dequant_rows(cfg["sh_gate_up_type"], lay[k], c).astype(np.float64) for k, c in (("sh_gate", H), ("sh_up", H), ("sh_down", F)))
    xd = x.astype(np.float64)
    xd[:, :16] = 0.0
    a = xd @ g.T
    y = (a / (1.0 + np.exp(-a)) * (xd @ u.T)) @ d.T
    return y / (1.0 + np.exp(-(xd @ lay["sh_gate_inp"].astype(np.float64))))[:, None]


# tiles of 32 x 16 in front of the routing and of the pair sort, of 32 x 32 and of 64 x 32 on a stream of their own
@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("n", [44, 512, 2047])
def test_leading_terms_that_overflow(n, given):
    cfg, lay = shared_only_layer(51)
    m = ResidentMoe(cfg, n_layer=1, max_tokens=n)
    m.load_layer(0, lay)
    x = synth.normed_x(np.random.default_rng(52), n, H)
    bad = [0, 3, 17, n - 1]

    def call(a):
        a = torch.from_numpy(a).cuda()
        if not given:
            return m.forward(0, a).cpu().numpy()
        ids = ((torch.arange(n, device="cuda")[:, None] * K + torch.arange(K, device="cuda")) % E).to(torch.int32)
        return m.experts(0, a, ids, torch.full((n, K), 0.25, device="cuda")).cpu().numpy()
    plain, want = call(x), shared_in_double(cfg, lay, x)
    # of the rms of a token's outputs: products of three terms 0.5e-7 at 512 columns, twice through SwiGLU, once more for the down rows, and f32 in between
    assert np.sqrt(((plain - want) ** 2).sum() / (want ** 2).sum()) <= 2.0e-7
    y = x.copy()
    y[bad, COL] = np.float32(3.4e38)
    got, rest = call(y), [t for t in range(n) if t not in bad]
    assert np.array_equal(got[rest], plain[rest])
    # the fp32 unit, 16 products behind one another in each of eight parts
    assert np.isfinite(got[bad]).all() and np.sqrt(((got[bad] - want[bad]) ** 2).sum() / (want[bad] ** 2).sum()) <= 4.0e-7
    m.close()


@pytest.mark.parametrize("shift", [0, 1])      # (activations at any float: fetched by another way)
def test_infinite_and_nan_tokens(shift):
    cfg, lay = shared_only_layer(53)
    n = 600
    m = ResidentMoe(cfg, n_layer=1, max_tokens=n)
    m.load_layer(0, lay)
    x = synth.normed_x(np.random.default_rng(54), n, H)
    plain = m.forward(0, torch.from_numpy(x).cuda()).cpu().numpy()
    y = x.copy()
    y[7, 300], y[41, 20], y[599, 511] = np.nan, np.inf, -np.inf
    room = torch.zeros(n * H + 1, device="cuda")
    at = room[shift:shift + n * H].reshape(n, H)
    at.copy_(torch.from_numpy(y))
    got = m.forward(0, at).cpu().numpy()
    rest = [t for t in range(n) if t not in (7, 41, 599)]
    assert np.array_equal(got[rest], plain[rest]) and not np.isfinite(got[[7, 41, 599]]).any()
    m.close()


def test_a_chunk_of_nan_takes_little_longer():
    """1.2 times a chunk of numbers; 23 times while a thread multiplied the columns of its outputs one after the other"""
    cfg = synth.layer_config(hidden=2048, ffn=512, n_expert=16, top_k=4, layout="f2")
    m = ResidentMoe(cfg, n_layer=1, max_tokens=512)
    m.load_layer(0, synth.make_layer(55, cfg))
    us = []
    for fill in (None, float("nan")):
        x = torch.from_numpy(synth.normed_x(np.random.default_rng(56), 512, 2048)).cuda()
        if fill is not None:
            x.fill_(fill)
        out = torch.empty_like(x)
        times = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            m.forward(0, x, out=out)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        us.append(min(times))
    print("numbers %.0f us, NaN %.0f us" % tuple(us))
    assert us[1] <= 3.0 * us[0], us
    m.close()
