"""The workspace of a resident handle grows per token by what chunks use of it, and by nothing that only small batches reach."""
import pytest

from dwarfstar_red_lite_amd import synth
from dwarfstar_red_lite_amd.moe import ResidentMoe

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("layout", ["iq2", "f2"])
def test_bytes_per_token(layout):
    H, F, E, K = 512, 512, 8, 8
    cfg = synth.layer_config(hidden=H, ffn=F, n_expert=E, top_k=K, layout=layout)
    free = []
    for tokens in (8192, 8192, 4096):      # (the first handle of a process also loads the kernels)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        m = ResidentMoe(cfg, n_layer=1, max_tokens=tokens)
        free.append(before - torch.cuda.mem_get_info()[0])
        m.close()
    per_token = (free[1] - free[2]) / 4096
    # f32: normalised x, logits, weights, scalar, routed and shared activations, routed and shared products; fp16 halves of x and its exponent;
    # five lists of pairs and their weights; the pair sort's scratch and the tile lists: less than 64 bytes a pair
    used = 4 * (H + E + 1 + K + 1 + K * F + F + K * H + H) + 4 * H + 4 + 4 * K + 6 * 4 * K + 64 * K
    assert 0.9 * used <= per_token <= used + 512, (per_token, used)      # (memory comes in pieces of 2 MB, 512 bytes a token here)
