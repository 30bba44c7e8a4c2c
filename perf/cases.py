"""The work this library does for a program that uses it, as cases that can be timed and compared.

Three kinds of program stand behind them:
* a decode engine with every expert resident (ResidentMoe): one token, a verify pair or a few requests, prefill chunks, each through a
  stack of layers. `op` is the entry point it calls per layer: "block" (residual add, RMS-norm, layer, residual add), "forward" (the layer
  alone, the engine norms itself) or "experts" (the engine brings the routing);
* an engine that drives the bounded slot pool itself (RedMetalTopKPool): one token through the pool's device-driven call per layer, or a
  chunk's pairs sorted by expert in one batched call. Slots hold raw GGUF bytes; `fast` opts into the re-laid copies;
* a tool that runs one expert from host arrays (RedMetalFfnPool), synchronously.

Weights are random-valid GGUF blocks of the layer's formats, activations RMS-normalised normal rows, as everywhere in this repository.
"""
import os
import random
import tempfile

import numpy as np
import torch

from dwarfstar_red_lite_amd import expert_type_word, synth
from dwarfstar_red_lite_amd import moe as moe_api
from dwarfstar_red_lite_amd.moe import ResidentMoe
from dwarfstar_red_lite_amd.redmetal_ffn import RedMetalFfnPool
from dwarfstar_red_lite_amd.redmetal_topk import ExpertLayout, RedMetalTopKPool


def _case(name, kind, layout, op="block", tokens=1, layers=1, hidden=2048, ffn=512, experts=512, top_k=10, routing="router", fast=False):
    c = dict(kind=kind, layout=layout, op=op, tokens=tokens, layers=layers, hidden=hidden, ffn=ffn, experts=experts, top_k=top_k,
             routing=routing, fast=fast)
    return dict(c, name=name) if name else c


def listed():
    return [
        # decode, one token through a stack of resident layers with the residual steps around each: what an engine does per token.
        # More layers than the last-level cache holds of what a token touches, as in a model
        _case("decode-iq2", "resident", "iq2", layers=12),
        _case("decode-f2", "resident", "f2", layers=12),
        # the draft-and-verify pair of speculative decoding on the all-IQ2_XS layers of the mixed model files
        _case("verify-pair-xs", "resident", "xs", tokens=2, layers=8),
        # eight parallel requests whose tokens favour 32 hot experts, the engine brings the routing; mixed-precision layout
        _case("batch8-hot-f2", "resident", "f2", op="experts", tokens=8, layers=6, routing="hot"),
        # a server's ordinary batch, the layer's own router
        _case("batch24-iq2", "resident", "iq2", op="forward", tokens=24, layers=3),
        # a short ragged prompt on all-IQ1_M layers
        _case("prompt77-m", "resident", "m", tokens=77, layers=2),
        # a prefill chunk with Zipf-popular experts, routing given, mixed precision
        _case("chunk512-zipf-f2", "resident", "f2", op="experts", tokens=512, layers=2, routing="zipf"),
        # the largest chunk an engine hands over
        _case("chunk2048-iq2", "resident", "iq2", op="forward", tokens=2048, layers=1),
        # a wider expert with fewer of them (ffn above 512), ragged chunk, mixed precision
        _case("chunk300-wide-f2", "resident", "f2", op="forward", tokens=300, layers=1, ffn=768, experts=128, top_k=8),
        # the slot pool: a token through 16 layers' device-driven calls, raw slots of IQ2_XS experts
        _case("pool-token-xs", "pool-token", "xs", op="into", layers=16, experts=16),
        # the slot pool: a 512-token chunk over 512 raw slots, one batched call
        _case("pool-chunk-iq2", "pool-chunk", "iq2", op="batched", tokens=512),
        # one expert from host arrays, synchronous: the smallest call
        _case("expert-f2", "expert", "f2", op="execute", experts=8, top_k=1),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """Another case of the same ranges: formats, shapes with ffn 256 .. 768, 1 .. 2048 tokens, both pool forms with and without the copies."""
    assert isinstance(rng, random.Random)
    kind = rng.choice(["resident"] * 7 + ["pool-token", "pool-chunk", "expert"])
    layout = rng.choice(["iq2", "f2", "xs", "m"])
    hidden, ffn, experts, top_k = rng.choice([(2048, 512, 512, 10)] * 3 + [(2048, 768, 128, 8), (1024, 512, rng.randint(60, 300), rng.randint(4, 10)),
                                                                          (1024, 256, rng.randint(48, 160), rng.randint(2, 8))])
    shape = dict(hidden=hidden, ffn=ffn, experts=experts, top_k=top_k)
    if kind == "resident":
        size = rng.choice(["one", "few", "batch", "chunk", "chunk"])
        tokens = dict(one=1, few=rng.randint(2, 8), batch=rng.randint(9, 32), chunk=_log_int(rng, 33, 300 if ffn > 512 else 2048))[size]
        layers = 1 if tokens > 300 else rng.randint(1, 3) if tokens > 8 else rng.randint(4, 12)
        op = rng.choice(["block", "forward", "experts"])
        routing = rng.choice(["hot", "zipf", "even"]) if op == "experts" else "router"
        return _case(None, "resident", layout, op=op, tokens=tokens, layers=layers, routing=routing, **shape)
    if kind == "pool-token":
        return _case(None, kind, layout, op="into", layers=rng.randint(4, 16), hidden=hidden, ffn=ffn, experts=top_k + rng.randint(0, 8), top_k=top_k,
                     fast=rng.random() < 0.5)
    if kind == "pool-chunk":
        fast = ffn <= 512 and rng.random() < 0.5
        return _case(None, kind, layout, op="batched", tokens=_log_int(rng, 16, 512), fast=fast, hidden=hidden, ffn=min(ffn, 512), experts=experts, top_k=top_k)
    return _case(None, kind, layout, op="execute", hidden=hidden, ffn=ffn, experts=rng.randint(4, 32), top_k=1)


# ---- inputs ----

def _codebooks():
    """One pair of tables of the values such codebooks hold; a process has one pair."""
    r = np.random.default_rng(12345)
    return (r.choice(np.array([8, 25, 43], np.int8), size=512 * 8), r.choice(np.array([-1, 0, 1], np.int8), size=2048 * 8))


def _config(case):
    return synth.layer_config(hidden=case["hidden"], ffn=case["ffn"], n_expert=case["experts"], top_k=case["top_k"], layout=case["layout"])


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rows(gen, n, hidden):
    x = torch.randn((n, hidden), device="cuda", generator=gen)
    return (x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + 1e-6)).contiguous()


def _routing(case, gen):
    """(ids [tokens][top_k] int32, weights [tokens][top_k] f32, renormalised) as an engine's own selection gives them"""
    T, E, K = case["tokens"], case["experts"], case["top_k"]
    logits = torch.randn((T, E), device="cuda", generator=gen)
    if case["routing"] == "hot":
        logits[:, (torch.arange(min(32, E), device="cuda") * 37) % E] += 2.0
    elif case["routing"] == "zipf":      # Gumbel top-k: draws without replacement from a Zipf(1.1) popularity
        u = torch.rand((T, E), device="cuda", generator=gen).clamp_(1e-20, 1.0 - 1e-7)
        rank = torch.randperm(E, device="cuda", generator=gen).float() + 1.0
        logits = -1.1 * torch.log(rank) - torch.log(-torch.log(u))
    top, ids = torch.topk(logits, K, dim=1)
    return ids.to(torch.int32).contiguous(), torch.softmax(top, dim=1).contiguous()


def _prepare_resident(case, seed):
    if case["layout"] in ("xs", "m"):
        moe_api.set_codebooks(*_codebooks())
    cfg, gen, T, H = _config(case), _generator(seed), case["tokens"], case["hidden"]
    m = ResidentMoe(cfg, n_layer=case["layers"], max_tokens=T)
    for l in range(case["layers"]):
        m.load_layer(l, synth.make_layer_gpu(torch, gen, cfg))
    st = dict(op=case["op"], moe=m, layers=case["layers"], x=_rows(gen, T, H))
    if case["op"] == "block":
        st["branch"] = [0.5 * torch.randn((T, H), device="cuda", generator=gen) for _ in range(case["layers"])]
        st["norm"] = [1.0 + 0.1 * torch.randn(H, device="cuda", generator=gen) for _ in range(case["layers"])]
    else:      # the rows every layer sees, normed by the engine
        st["xs"] = [_rows(gen, T, H) for _ in range(case["layers"])]
        st["outs"] = [torch.empty((T, H), device="cuda") for _ in range(case["layers"])]
        if case["op"] == "experts":
            st["routes"] = [_routing(case, gen) for _ in range(case["layers"])]
    return st


def _raw_experts(gen, cfg, n):
    """n experts as a file holds them (gate | up | down bytes of one after the other) and the byte ranges of each"""
    a = synth.make_layer_gpu(torch, gen, dict(cfg, n_expert=n))
    gb, db = a["gate"].shape[1], a["down"].shape[1]
    blob = torch.cat([a["gate"], a["up"], a["down"]], dim=1).cpu().numpy()
    per = 2 * gb + db
    return blob, [ExpertLayout(e * per, gb, e * per + gb, gb, e * per + 2 * gb, db) for e in range(n)], per


class _File:
    """the experts in a temporary file for as long as a pool is being filled from it"""

    def __init__(self, blob):
        fd, self.path = tempfile.mkstemp(prefix="experts_")
        with os.fdopen(fd, "wb") as f:
            f.write(blob.data)

    def __enter__(self):
        return self.path

    def __exit__(self, *_):
        os.unlink(self.path)


class _Owned:
    """a pool that is closed with the last reference to it"""

    def __init__(self, pool):
        self.pool = pool

    def __del__(self):
        try:
            self.pool.close()
        except Exception:
            pass


def _prepare_pool(case, seed):
    cfg, gen, H, F = _config(case), _generator(seed), case["hidden"], case["ffn"]
    chunk = case["kind"] == "pool-chunk"
    n = case["experts"] if chunk else case["experts"] * case["layers"]
    word = expert_type_word(cfg["gate_up_type"], cfg["down_type"])
    blob, lays, per = _raw_experts(gen, cfg, n)
    cb = _codebooks()
    with _File(blob) as path:
        pool = RedMetalTopKPool(path, (n + 2) * (5 * per + 8192), per, slots_per_slab=64, iq2_xs_grid=cb[0], iq1_m_grid=cb[1])
        if case["fast"]:
            pool.enable_fast_path(word, H, F, tiles=chunk)
        for e in range(n):
            pool.load(e, lays[e])
    st = dict(op=case["op"], owner=_Owned(pool), pool=pool, word=word, hidden=H, ffn=F, K=case["top_k"], gate_bytes=lays[0].gate_bytes)
    if chunk:
        T, K = case["tokens"], case["top_k"]
        ids, w = (t.cpu().numpy() for t in _routing(dict(case, routing="even"), gen))
        flat = ids.ravel()
        order = np.argsort(flat, kind="stable")
        uid, count = np.unique(flat, return_counts=True)
        place = np.empty(T * K, np.uint32)
        place[order] = np.arange(T * K, dtype=np.uint32)
        st.update(tokens=T, slots=[int(e) for e in uid], lays=[lays[int(e)] for e in uid], pair_token=(order // K).astype(np.uint32),
                  pair_weight=w.ravel()[order].astype(np.float32), start=np.concatenate([[0], np.cumsum(count)]).astype(np.uint32), tok_pair=place,
                  x=_rows(gen, T, H), out=torch.zeros((T, H), device="cuda"))
    else:
        L, E = case["layers"], case["experts"]
        addr = [pool.addresses(e, lays[e])[0] for e in range(n)]
        pick = [torch.randperm(E, device="cuda", generator=gen)[:case["top_k"]].tolist() for _ in range(L)]
        st["table"] = [torch.from_numpy(np.array([addr[l * E + e] for e in pick[l]], np.uint64).view(np.int64)).cuda() for l in range(L)]
        st["w"] = [torch.softmax(torch.randn(case["top_k"], device="cuda", generator=gen), dim=0).contiguous() for _ in range(L)]
        st["x"], st["out"] = _rows(gen, L, H), torch.zeros((L, H), device="cuda")
    return st


def _prepare_expert(case, seed):
    cfg, gen, H, F, n = _config(case), _generator(seed), case["hidden"], case["ffn"], case["experts"]
    blob, lays, per = _raw_experts(gen, cfg, n)
    cb = _codebooks()
    with _File(blob) as path:
        pool = RedMetalFfnPool(path, (n + 2) * (per + 4096), per, iq2_xs_grid=cb[0], iq1_m_grid=cb[1])
        for e in range(n):
            pool.load(e, lays[e])
    x = _rows(gen, n, H).cpu().numpy()
    return dict(op=case["op"], owner=_Owned(pool), pool=pool, word=expert_type_word(cfg["gate_up_type"], cfg["down_type"]), hidden=H, ffn=F, lays=lays, x=x)


def prepare(case, seed):
    if case["kind"] == "resident":
        return _prepare_resident(case, seed)
    return _prepare_expert(case, seed) if case["kind"] == "expert" else _prepare_pool(case, seed)


def run(state):
    op = state["op"]
    if op == "block":
        x, m = state["x"], state["moe"]
        for l in range(state["layers"]):
            x = m.forward_block(l, x, state["branch"][l], state["norm"][l])
        return x
    if op in ("forward", "experts"):
        m = state["moe"]
        for l in range(state["layers"]):
            if op == "forward":
                m.forward(l, state["xs"][l], out=state["outs"][l])
            else:
                m.experts(l, state["xs"][l], *state["routes"][l], out=state["outs"][l])
        return state["outs"]
    pool, H, F, word = state["pool"], state["hidden"], state["ffn"], state["word"]
    if op == "execute":      # every expert the tool holds, one after the other
        return [pool.execute(e, lay, word, H, F, 0, H, state["x"][e])[0] for e, lay in enumerate(state["lays"])]
    stream = torch.cuda.current_stream().cuda_stream
    if op == "into":
        for l, table in enumerate(state["table"]):
            pool.encode_device_into(stream, table.data_ptr(), state["w"][l].data_ptr(), state["K"], word, H, F, state["gate_bytes"], state["gate_bytes"],
                                    state["x"][l].data_ptr(), state["out"][l].data_ptr())
        return state["out"]
    pool.encode_batched(stream, state["slots"], state["lays"], word, H, F, 0, state["tokens"], state["K"], state["pair_token"], state["pair_weight"],
                        state["start"], state["tok_pair"], state["x"].data_ptr(), state["out"].data_ptr())
    pool.release(state["slots"])
    return state["out"]


# ---- what a pass cannot do without ----

def _distinct(case):
    """expected number of distinct experts of one layer's tokens"""
    T, E, K = case["tokens"], case["experts"], case["top_k"]
    if case["routing"] in ("router", "even") or T == 1:
        return E * (1.0 - (1.0 - K / E) ** T)
    r = np.random.default_rng(1)
    logits = r.standard_normal((T, E))
    if case["routing"] == "hot":
        logits[:, (np.arange(min(32, E)) * 37) % E] += 2.0
    else:
        logits = -1.1 * np.log(np.arange(1, E + 1)) + r.gumbel(size=(T, E))
    return float(len(np.unique(np.argpartition(-logits, K - 1, axis=1)[:, :K])))


def work(case):
    cfg, T, H, F, E, K = _config(case), case["tokens"], case["hidden"], case["ffn"], case["experts"], case["top_k"]
    expert = 2 * F * synth.row_bytes(cfg["gate_up_type"], H) + H * synth.row_bytes(cfg["down_type"], F)
    if case["kind"] == "expert":
        return {"bytes": E * (expert + 8 * H), "flops": E * 6 * H * F}
    if case["kind"] == "pool-token":
        return {"bytes": case["layers"] * (K * (expert + 12) + 8 * H), "flops": case["layers"] * K * 6 * H * F}
    if case["kind"] == "pool-chunk":
        return {"bytes": int(_distinct(case) * expert) + 8 * T * H + 12 * T * K, "flops": T * K * 6 * H * F}
    shared = 2 * F * synth.row_bytes(cfg["sh_gate_up_type"], H) + H * synth.row_bytes(cfg["sh_down_type"], F) + 4 * H
    own = case["op"] != "experts"
    layer = _distinct(case) * expert + shared + (E * synth.row_bytes(cfg["router_type"], H) if own else 8 * T * K)
    # activations in and out of a layer (the block form also takes the branch's rows)
    layer += T * H * 4 * (3 if case["op"] == "block" else 2)
    return {"bytes": int(case["layers"] * layer), "flops": case["layers"] * T * ((K + 1) * 6 * H * F + (2 * E * H if own else 0))}


def tolerance(case):
    """32-bit sums over weights that are exact and activations of at least 22 significant bits"""
    return {"rel": 1e-5}
