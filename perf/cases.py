"""The work that this engine is used for, as a list of cases that can be timed and checked.

A case is one call pattern of a serving engine on one GPU: a decode step of a batch (replayed from a
HIP graph, as serving does), a prompt or several that arrive together, a prompt portion beside decoded
tokens, or a short answer from its prompt to its last token.  Every case runs the engine's step
function (``GraphRunner.step`` over pages of a ``CacheManager``), the one function that generation,
trace replay and the benchmark call.  Weights are random (a generator per tensor), tokens uniform over
the vocabulary, token ids given and not taken from the step before, so that every pass does the same.

Designs: the dense Qwen2.5 decoder at its 0.5B, 1.5B and 7B layer sizes, and three of the other
decoders at the layer sizes the benchmark runs them at: ``samovik`` (latent attention, linear attention
with decay, time mixing, routed experts), ``kabulix`` (windowed, latent and chunked attention, experts
chosen within groups) and ``taluvik`` (delta rule, selective scan, capped attention).
"""
from __future__ import annotations

import math
import zlib

import torch
import torch.nn.functional as F

DEVICE = "cuda:0"
PAGE = 16

# ---- the designs ----------------------------------------------------------------------------------
QWEN2 = {
    "qwen2-0.5b": dict(vocab_size=151936, hidden_size=896, intermediate_size=4864, num_hidden_layers=24, num_attention_heads=14,
                       num_key_value_heads=2, head_dim=64, tie_word_embeddings=True),
    "qwen2-1.5b": dict(vocab_size=151936, hidden_size=1536, intermediate_size=8960, num_hidden_layers=28, num_attention_heads=12,
                       num_key_value_heads=2, head_dim=128, tie_word_embeddings=True),
    "qwen2-7b": dict(vocab_size=152064, hidden_size=3584, intermediate_size=18944, num_hidden_layers=28, num_attention_heads=28,
                     num_key_value_heads=4, head_dim=128, tie_word_embeddings=False),
}
# width: (heads, experts, experts per token, width of an expert)
WIDTHS = {1024: (8, 32, 6, 512), 2048: (16, 64, 6, 1408), 4096: (32, 64, 6, 2048)}
VOCAB = 32000
YARN = {"base": 10000.0, "dims": 64, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}


def config_of(case: dict) -> dict:
    """The case's model as the dictionary of a config.json."""
    if case["design"] in QWEN2:
        return dict(QWEN2[case["design"]], architectures=["Qwen2ForCausalLM"], num_hidden_layers=case["layers"],
                    rope_theta=1000000.0, rms_norm_eps=1e-6, max_position_embeddings=32768)
    W = case["width"]
    H, E, top, ff = WIDTHS[W]
    kv = max(1, H // 4)
    latent = {"heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "scale": 192 ** -0.5, "rot": YARN}
    grouped = {"heads": H, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
    if case["design"] == "samovik":
        mlp = {"kind": "moe", "router": {"experts": E, "top": top}, "expert": {"ff": ff, "limit": 7.0}, "shared": {"ff": 2 * ff, "limit": 7.0}}
        lightning = {"heads": H, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-5 - 3 * h / H) for h in range(H)]}
        wkv = {"heads": 2 * H, "dim": 64, "decay_rank": 64}
        layers = [{"type": t, "mixer": m, "mlp": mlp} for t, m in
                  (("latent_attention", latent), ("lightning", lightning), ("wkv", wkv), ("latent_attention", latent))]
        return {"architecture": "Samovik", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-6},
                "token_side": {"dim": 128 if W == 1024 else 256}, "layers": layers}
    if case["design"] == "kabulix":
        windowed = dict(grouped, mask={"size": 4096, "keep_first": 4}, rot={"dims": 64, "base": 10000.0})
        masked = dict(latent, mask={"size": 4096})
        moe = {"kind": "moe", "router": {"experts": E, "top": top, "groups": {"count": 8, "keep": 4}}, "expert": {"ff": ff},
               "shared": {"ff": ff}}
        layers = [{"type": "attention", "mixer": windowed, "mlp": {"kind": "dense", "ff": 3 * W}},
                  {"type": "latent_attention", "mixer": masked, "mlp": moe}, {"type": "attention", "mixer": windowed, "mlp": moe},
                  {"type": "attention_2", "mixer": dict(grouped, mask={"size": 4096}), "mlp": moe}]
        return {"architecture": "Kabulix", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-6}, "layers": layers}
    if case["design"] == "taluvik":
        delta = {"heads": H, "kv_heads": H // 2, "dim": 128, "vdim": 128, "conv": 4}
        scan = {"inner": 2 * W, "state": 16, "dt_rank": W // 16, "conv": 4}
        attention = dict(grouped, softcap=30.0, mask={"size": 4096},
                         rot={"dims": 128, "base": 500000.0, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}})
        ff = {"kind": "dense", "ff": 3 * W}
        layers = [{"type": t, "mixer": m, "mlp": ff} for t, m in
                  (("delta", delta), ("mamba1", scan), ("attention", attention), ("delta", delta))]
        return {"architecture": "Taluvik", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0},
                "residual_mult": 0.5, "layers": layers}
    raise ValueError(case["design"])


def vocab_of(case: dict) -> int:
    return QWEN2[case["design"]]["vocab_size"] if case["design"] in QWEN2 else VOCAB


# ---- weights ----------------------------------------------------------------------------------------
def spread_of(name: str, case: dict) -> tuple[float, float]:
    """(mean, standard deviation) of a tensor's values: matrices N(0, 0.02), those that end a branch smaller the deeper the
    model is (so that the stream keeps its size and a rounding is not blown up from layer to layer, as in trained models),
    norm weights around one, and so on."""
    last = name.rsplit(".", 1)[-1]
    ends_branch = 0.02 / math.sqrt(2 * case.get("layers", 4))
    if name in ("embed", "model.embed_tokens.weight"):
        return 0.0, 1.0
    if case["design"] in QWEN2:
        if "norm" in name:
            return 1.0, 0.1
        if name == "lm_head.weight":
            return 0.0, 0.05
        return 0.0, ends_branch if name.endswith(("o_proj.weight", "down_proj.weight")) else 0.02
    if last in ("o", "down"):
        return 0.0, ends_branch
    if name.endswith(("norm1", "norm2", "final.norm")):
        return (0.0 if case["design"] == "kabulix" else 1.0), 0.1
    if name.endswith(("norm1.b", "norm2.b", "final.norm.b", "conv.b")):
        return 0.0, 0.1
    if last == "norm":
        return 1.0, 0.1
    if last == "alpha":
        return 1.0, 0.2
    if last == "D":
        return 1.0, 0.3
    if last == "conv":
        return 0.0, 0.4
    if last in ("A_log", "dt_bias", "sink") or name.endswith("dt.b"):
        return 0.0, 1.0
    if ".mu." in name or last == "u":
        return 0.0, 0.3
    if name == "side.embed":
        return 0.0, 0.5
    if last in ("uk", "uv"):
        return 0.0, 0.05
    return 0.0, 0.02


def tensor(case: dict, seed: int, name: str, shape) -> torch.Tensor:
    """A weight in float32; in a bfloat16 case its values are those of bfloat16."""
    g = torch.Generator(device=DEVICE).manual_seed((seed << 32) ^ zlib.crc32(name.encode()))
    mean, std = spread_of(name, case)
    t = torch.randn(tuple(shape), generator=g, dtype=torch.float32, device=DEVICE).mul_(std)
    if mean:
        t.add_(mean)
    return t.to(torch.bfloat16).to(torch.float32) if case["dtype"] == "bfloat16" else t


# ---- what a case asks for -----------------------------------------------------------------------------
def spread(low: int, high: int, n: int) -> list[int]:
    """n lengths from low to high, evenly, in an order that is not sorted."""
    if n == 1:
        return [high]
    out = [low + (high - low) * i // (n - 1) for i in range(n)]
    step = next(s for s in (7, 5, 3, 1) if math.gcd(s, n) == 1)
    return [out[(i * step) % n] for i in range(n)]


def shape_of(case: dict) -> list[tuple[int, int, list[int]]]:
    """The step that is measured: (tokens already cached, tokens brought, places whose logits are wanted) per request.
    ``generate`` cases: the prompts' step; ``steps`` decode steps follow it."""
    b, low, high = case["batch"], case["low"], case["high"]
    if case["kind"] == "decode":
        return [(n, 1, [0]) for n in spread(low, high, b)]
    if case["kind"] in ("prompts", "generate"):
        return [(0, n, [n - 1]) for n in spread(low, high, b)]
    # a portion in the middle of a long prompt (no logits wanted) beside one-token requests
    return [(case["behind"], case["portion"], [])] + [(n, 1, [0]) for n in spread(low, high, b)]


def token_ids(case: dict, seed: int) -> list[list[int]]:
    """The tokens of each request, from its first one to the last that the case brings."""
    g = torch.Generator().manual_seed(seed)
    more = case.get("steps", 0)
    return [torch.randint(0, vocab_of(case), (start + n + more,), generator=g).tolist() for start, n, _ in shape_of(case)]


def listed() -> list[dict]:
    bf, f32 = "bfloat16", "float32"
    return [
        # one user of a small model, short conversation: the smallest step there is
        dict(name="decode-0.5b-b1", design="qwen2-0.5b", layers=24, dtype=bf, kind="decode", batch=1, low=300, high=300),
        # the benchmark's headline: eight sequences deep into a 4,096-token context, the whole 7B model
        dict(name="decode-7b-b8", design="qwen2-7b", layers=28, dtype=bf, kind="decode", batch=8, low=3900, high=4080),
        # a busy server: 48 requests of very different lengths, tokens sampled with temperature and top-p
        dict(name="decode-7b-b48-sampled", design="qwen2-7b", layers=8, dtype=bf, kind="decode", batch=48, low=150, high=2300,
             sample=True),
        # one long prompt: a full portion of the default token budget, the whole 7B model
        dict(name="prefill-7b-2048", design="qwen2-7b", layers=28, dtype=bf, kind="prompts", batch=1, low=2048, high=2048),
        # chat prompts that arrive together and fit one step
        dict(name="prompts-1.5b-9", design="qwen2-1.5b", layers=28, dtype=bf, kind="prompts", batch=9, low=21, high=157),
        # continuous batching: a portion of a long prompt beside decoding requests
        dict(name="mixed-1.5b", design="qwen2-1.5b", layers=28, dtype=bf, kind="mixed", batch=24, low=90, high=1900, behind=3072,
             portion=489),
        # the true 32-bit path, prompt and decode, at 4 of the 7B shape's layers as the benchmark runs it
        dict(name="float32-prefill-2048", design="qwen2-7b", layers=4, dtype=f32, kind="prompts", batch=1, low=2048, high=2048),
        dict(name="float32-decode-b8", design="qwen2-7b", layers=4, dtype=f32, kind="decode", batch=8, low=2200, high=2400),
        # routed experts and masked attention: a long prompt at the largest width, decoding at the middle one
        dict(name="kabulix-prefill-2048", design="kabulix", width=4096, dtype=bf, kind="prompts", batch=1, low=2048, high=2048),
        dict(name="kabulix-decode-b16", design="kabulix", width=2048, dtype=bf, kind="decode", batch=16, low=700, high=1500),
        # latent and linear attention, time mixing and experts: three prompts of odd lengths in one step
        dict(name="samovik-prompts-3", design="samovik", width=2048, dtype=bf, kind="prompts", batch=3, low=211, high=803),
        # recurrent layers: short prompts and the first tokens of their answers
        dict(name="taluvik-answer-b4", design="taluvik", width=2048, dtype=bf, kind="generate", batch=4, low=130, high=411, steps=12),
    ]


def draw(rng) -> dict:
    def log_between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "prompts", "prompts", "mixed", "generate"])
    if kind == "generate" or (kind != "mixed" and rng.random() < 0.4):
        c = dict(design=rng.choice(["samovik", "kabulix", "taluvik"]), width=rng.choice([1024, 2048, 4096]), dtype="bfloat16")
        if kind == "decode":
            c["design"] = "kabulix"            # a decode step that can be run again and again: no recurrent state
    else:
        design = rng.choice(list(QWEN2))
        dtype = "float32" if rng.random() < 0.3 else "bfloat16"
        c = dict(design=design, layers=rng.randint(2, 8 if dtype == "bfloat16" else 4), dtype=dtype)
    c["kind"] = kind
    if kind == "decode":
        c["batch"] = log_between(1, 64)
        high = log_between(40, min(4090, 65536 // c["batch"]))
        c.update(low=max(1, int(high * rng.uniform(0.1, 1.0))), high=high)
        if c["dtype"] == "bfloat16":
            c["sample"] = rng.random() < 0.3
    elif kind == "mixed":
        c.update(batch=log_between(1, 40), behind=log_between(1, 3500), portion=log_between(16, 1900))
        high = log_between(40, 1500)
        c.update(low=max(1, high // rng.randint(1, 9)), high=high)
    else:
        total = log_between(24, 2048 if kind == "prompts" else 900)
        c["batch"] = min(log_between(1, 16), max(1, total // 12))
        mean = total // c["batch"]
        off = int(mean * rng.uniform(0.0, 0.8)) if c["batch"] > 1 else 0
        c.update(low=max(1, mean - off), high=mean + off)
        if kind == "generate":
            c["steps"] = rng.randint(3, 12)
    return c


# ---- a pass -------------------------------------------------------------------------------------------
class State:
    pass


def prepare(case: dict, seed: int) -> State:
    """The model with its weights, its cache and step function; for steps that come in the middle of requests also those
    requests' earlier tokens in the cache."""
    from tensorline_amd.cache.manager import CacheManager
    from tensorline_amd.config.registry import get_architecture
    from tensorline_amd.engine.batch import StepEntry
    from tensorline_amd.engine.graphs import GraphRunner
    from tensorline_amd.models.decoder import DecoderModel
    from tensorline_amd.sampling.sampler import Sampler
    from tensorline_amd.weights.loader import load_from_getter

    raw = config_of(case)
    arch = get_architecture(raw["architectures"][0] if "architectures" in raw else raw["architecture"])
    st = State()
    st.model = DecoderModel(arch.build_spec(arch.config_cls.from_dict(raw)), getattr(torch, case["dtype"]), DEVICE)
    load_from_getter(st.model, lambda name, decl: tensor(case, seed, name, decl.shape), DEVICE)
    plan, ids = shape_of(case), token_ids(case, seed)
    longest = max(4096, max(len(t) for t in ids))
    st.cache = CacheManager(st.model.cache_needs(), st.model.schedule, st.model.state_needs(), page_size=PAGE,
                            num_blocks=sum(-(-len(t) // PAGE) for t in ids) + 8, max_requests=len(ids), dtype=st.model.dtype,
                            device=DEVICE, prefix_caching=False, input_state_need=st.model.input_state_need())
    st.runner = GraphRunner(st.model, st.cache, max_batch=len(ids), max_blocks_per_seq=-(-longest // PAGE))
    st.kind, st.sampler = case["kind"], None
    rids = list(range(len(ids)))
    st.entries = [StepEntry(r, ids[r][start:start + n], start, want) for r, (start, n, want) in zip(rids, plan)]
    st.later = [[StepEntry(r, [ids[r][n + s]], n + s, [0]) for r, (_, n, _) in zip(rids, plan)] for s in range(case.get("steps", 0))]
    st.lengths = [len(t) for t in ids]
    if case.get("sample"):
        st.sampler = Sampler(DEVICE)
        st.draws = ([0.7] * len(rids), [0.9] * len(rids), [seed * 1000 + r for r in rids], [1] * len(rids))
    if case["kind"] in ("decode", "mixed"):
        for r in rids:
            st.cache.add_request(r)
            assert st.cache.grow(r, len(ids[r]))
        todo = [(r, s, min(2048, plan[r][0] - s)) for r in rids for s in range(0, plan[r][0], 2048)]
        while todo:                                      # earlier tokens, in steps of at most 2,048 tokens
            step, room, seen = [], 2048, set()
            while todo and todo[0][2] <= room and todo[0][0] not in seen:
                r, s, n = todo.pop(0)
                step.append(StepEntry(r, ids[r][s:s + n], s, []))
                seen.add(r)
                room -= n
            st.runner.step(step)
    if case["kind"] in ("decode", "generate"):
        run(st)                                          # a serving engine's graphs are captured before it serves
    return st


def run(st: State):
    if st.kind in ("decode", "mixed"):
        logits = st.runner.step(st.entries)
        if st.sampler is None:
            return logits
        return {"logits": logits, "tokens": st.sampler.sample_device(logits, *st.draws)}
    for entry, n in zip(st.entries, st.lengths):         # requests come, are answered and go
        st.cache.add_request(entry.rid)
        st.cache.grow(entry.rid, n)
    logits = st.runner.step(st.entries)
    if st.later:
        logits = [logits] + [st.runner.step(step).clone() for step in st.later]      # a replay writes its logits in place
    for entry in st.entries:
        st.cache.release(entry.rid)
    return logits


# ---- what a pass cannot do without ----------------------------------------------------------------------
def work(case: dict) -> dict:
    elem = 2 if case["dtype"] == "bfloat16" else 4
    plan, V = shape_of(case), vocab_of(case)
    total = {"bytes": 0.0, "flops": 0.0}

    def add_step(step):
        T, B, R = sum(n for _, n, _ in step), len(step), sum(len(w) for _, _, w in step)
        pairs = float(sum(n * s + n * (n + 1) // 2 for s, n, _ in step))            # (token, key it sees)
        past, keys = float(sum(s for s, _, _ in step)), float(T)
        weights, flops, moved = 0.0, 0.0, 0.0

        def matrix(params, rows=T):
            nonlocal weights, flops
            weights += params
            flops += 2.0 * rows * params

        def attention(heads, score_dim, value_dim, cached):
            """``cached``: values a token keeps; the step reads the earlier tokens' and writes its own."""
            nonlocal flops, moved
            flops += 2.0 * heads * pairs * (score_dim + value_dim)
            moved += (past + keys) * cached * elem

        if case["design"] in QWEN2:
            z = QWEN2[case["design"]]
            W, H, G, d = z["hidden_size"], z["num_attention_heads"], z["num_key_value_heads"], z["head_dim"]
            for _ in range(case["layers"]):
                matrix((2 * H + 2 * G) * d * W + 3 * W * z["intermediate_size"])
                attention(H, d, d, 2 * G * d)
        else:
            W = case["width"]
            H, E, top, ff = WIDTHS[W]
            G = max(1, H // 4)

            def experts(shared):
                nonlocal weights, flops
                touched = E * (1.0 - (1.0 - top / E) ** T)
                weights += touched * 3 * W * ff
                flops += 2.0 * T * top * 3 * W * ff
                matrix(E * W + 3 * W * shared)

            def latent():
                matrix(H * 192 * W + 256 * W + 2 * H * 128 * 192 + H * 128 * W)
                attention(H, 192, 128, 256)

            def state(values):
                nonlocal moved
                moved += 2.0 * B * values * 4
            if case["design"] == "samovik":
                side = 128 if W == 1024 else 256
                for _ in range(2):
                    latent()
                matrix(5 * W * W)                        # linear attention
                flops += 4.0 * T * H * 128 * 128
                state(H * 128 * 128)
                matrix(5 * W * W + 128 * W)              # time mixing
                flops += 4.0 * T * 2 * H * 64 * 64
                state(2 * H * 64 * 64)
                for _ in range(4):
                    experts(2 * ff)
                    matrix(2 * W * side)
            elif case["design"] == "kabulix":
                latent()
                for n in (1, 1, 2):                      # windowed layers keep keys only: their values are the keys
                    matrix((2 * H + n * G) * 128 * W)
                    attention(H, 128, 128, n * G * 128)
                matrix(9 * W * W + W * W)
                for _ in range(3):
                    experts(ff)
            else:
                for _ in range(2):
                    matrix((3 * H + H) * 128 * W)
                    flops += 6.0 * T * H * 128 * 128
                    state(H * 128 * 128)
                matrix(6 * W * W + 2 * W * (W // 16 + 32) + W // 16 * 2 * W)
                flops += 6.0 * T * 2 * W * 16
                state(2 * W * 16)
                matrix((2 * H + 2 * G) * 128 * W)
                attention(H, 128, 128, 2 * G * 128)
                for _ in range(4):
                    matrix(9 * W * W)
        matrix(V * W, R) if R else None
        total["bytes"] += weights * elem + moved + T * W * elem + R * V * 4
        total["flops"] += flops

    add_step(plan)
    for s in range(case.get("steps", 0)):
        add_step([(n + s, 1, [0]) for _, n, _ in plan])
    return total


def tolerance(case: dict) -> dict:
    """About four times the distance from ``exact`` that these paths show: 0.002 to 0.0066 in bfloat16 (0.03 for a row of a
    design with experts where rounding turned a close choice between two of them), 4e-6 in float32."""
    if case["dtype"] == "float32":
        return {"rel": 1.5e-5}
    out = {"rel": 0.025 if case["design"] in QWEN2 or case["design"] == "taluvik" else 0.06}
    if case.get("sample"):
        out["differ"] = 0.1
    return out


# ---- the same in 64 bits ---------------------------------------------------------------------------------
class Plain:
    """A decoder over whole sequences in float64, one method per mechanism, no cache."""

    def __init__(self, case: dict, seed: int):
        self.case, self.seed, self.cfg = case, seed, config_of(case)

    def w(self, name: str, *shape) -> torch.Tensor:
        return tensor(self.case, self.seed, name, shape).double()

    def times(self, x, name: str, n: int) -> torch.Tensor:
        return x @ self.w(name, n, x.shape[1]).T

    # -- small pieces
    @staticmethod
    def over_rms(x, eps):
        return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)

    @staticmethod
    def gelu(z):
        return F.gelu(z, approximate="tanh")

    @staticmethod
    def frequencies(rot: dict):
        n, base = rot["dims"] // 2, rot["base"]
        i = torch.arange(n, dtype=torch.float64, device=DEVICE)
        f, sc = base ** (-i / n), rot.get("scaling")
        if not sc:
            return f, 1.0
        if "fast" in sc:                                 # by dimension, with a factor on cosine and sine
            dim = lambda turns: rot["dims"] * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
            lo, hi = max(math.floor(dim(sc["fast"])), 0), min(math.ceil(dim(sc["slow"])), rot["dims"] - 1)
            ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
            return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
        turns = sc["original"] * f / (2 * math.pi)       # by wavelength
        s = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
        return (1 - s) * f / sc["factor"] + s * f, 1.0

    def turn(self, x, pos, rot, pairs: bool = False):
        """x [T, heads, d]: the first rot["dims"] dimensions turned, i with i + n, or neighbours."""
        f, mag = self.frequencies(rot)
        a = pos[:, None, None].double() * f
        c, s, n = a.cos() * mag, a.sin() * mag, rot["dims"] // 2
        head, rest = x[..., :2 * n], x[..., 2 * n:]
        u, v = (head[..., 0::2], head[..., 1::2]) if pairs else (head[..., :n], head[..., n:])
        a, b = u * c - v * s, v * c + u * s
        return torch.cat((torch.stack((a, b), -1).flatten(-2) if pairs else torch.cat((a, b), -1), rest), -1)

    @staticmethod
    def softmax_attention(q, k, v, scale, sees=None, cap=None, sink=None):
        """q [n, H, d], k [m, G, d], v [m, G, dv] of one sequence, queries the last n of its m tokens."""
        n, H, _ = q.shape
        m, G, _ = k.shape
        i, j = torch.arange(m - n, m, device=DEVICE)[:, None], torch.arange(m, device=DEVICE)[None, :]
        mask = (j <= i) if sees is None else (j <= i) & sees(i, j)
        out = []
        for g in range(G):
            s = torch.matmul(q[:, g * (H // G):(g + 1) * (H // G)].transpose(0, 1), k[:, g].T.contiguous()) * scale
            s = cap * torch.tanh(s / cap) if cap else s
            s = s.masked_fill(~mask, float("-inf"))
            if sink is not None:
                extra = sink[g * (H // G):(g + 1) * (H // G), None, None].expand(-1, n, 1)
                p = torch.softmax(torch.cat((s, extra), -1), -1)[..., :-1]
            else:
                p = torch.softmax(s, -1)
            out.append(torch.matmul(p, v[:, g].contiguous()).transpose(0, 1))
        return torch.cat(out, 1).reshape(n, -1)

    def per_sequence(self, lens, fn, *xs):
        return torch.cat([fn(*part) for part in zip(*(x.split(lens) for x in xs))])

    def gated(self, h, p, ff, act):
        W = h.shape[1]
        g, u, d = self.w(p + "gate", ff, W), self.w(p + "up", ff, W), self.w(p + "down", W, ff)
        return torch.cat([act(x @ g.T, x @ u.T) @ d.T for x in h.split(8192)])

    # -- mixers
    def latent(self, h, p, m, lens, pos, pairs, gate_width):
        H, d, r, dv, rank, eps = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], self.cfg["norm"]["eps"]
        q = self.times(h, p + "q", H * (d + r)).view(-1, H, d + r)
        q = torch.cat((q[..., :d], self.turn(q[..., d:], pos, m["rot"], pairs)), -1)
        low = self.times(h, p + "dkv", rank + r)
        c = self.over_rms(low[:, :rank], eps) * self.w(p + "dkv.norm", rank)
        k_rot = self.turn(low[:, None, rank:], pos, m["rot"], pairs).expand(-1, H, -1)
        k = torch.cat((self.times(c, p + "uk", H * d).view(-1, H, d), k_rot), -1)
        v = self.times(c, p + "uv", H * dv).view(-1, H, dv)
        o = self.per_sequence(lens, lambda q, k, v: self.softmax_attention(q, k, v, m["scale"]), q, k, v)
        gate = torch.sigmoid(self.times(h, p + "g", gate_width))
        return self.times(o * gate.repeat_interleave(o.shape[1] // gate_width, 1), p + "o", h.shape[1])

    def lightning(self, h, p, m, lens, pos):
        H, d, dv, W, eps = m["heads"], m["dim"], m["vdim"], h.shape[1], self.cfg["norm"]["eps"]
        q, k = (F.silu(self.times(h, p + n, H * d)).view(-1, H, d) for n in "qk")
        v = F.silu(self.times(h, p + "v", H * dv)).view(-1, H, dv)
        decay = torch.tensor(m["decay"], dtype=torch.float32, device=DEVICE).double()[:, None, None]

        def walk(q, k, v):
            S, out = torch.zeros(H, d, dv, dtype=torch.float64, device=DEVICE), []
            for t in range(q.shape[0]):
                S = decay * S + k[t, :, :, None] * v[t, :, None, :]
                out.append((S * q[t, :, :, None]).sum(1))
            return torch.stack(out)
        o = self.per_sequence(lens, walk, q, k, v).reshape(-1, H * dv)
        o = self.over_rms(o, eps) * self.w(p + "norm", H * dv) * torch.sigmoid(self.times(h, p + "g", H * dv))
        return self.times(o, p + "o", W)

    def wkv(self, h, p, m, lens, pos):
        H, d, W, eps = m["heads"], m["dim"], h.shape[1], self.cfg["norm"]["eps"]
        before = self.per_sequence(lens, lambda x: F.pad(x, (0, 0, 1, 0))[:-1], h)
        mix = {s: h + (before - h) * self.w(p + "mu." + s, W) for s in "rkvgw"}
        r, k, v = (self.times(mix[s], p + s, H * d).view(-1, H, d) for s in "rkv")
        low = torch.tanh(self.times(mix["w"], p + "w1", m["decay_rank"]))
        decay = torch.exp(-torch.exp(self.times(low, p + "w2", H * d) + self.w(p + "w0", H * d))).view(-1, H, d)
        u = self.w(p + "u", H, d)[:, :, None]

        def walk(r, k, v, decay):
            S, out = torch.zeros(H, d, d, dtype=torch.float64, device=DEVICE), []
            for t in range(r.shape[0]):
                kv = k[t, :, :, None] * v[t, :, None, :]
                out.append(((S + u * kv) * r[t, :, :, None]).sum(1))
                S = decay[t, :, :, None] * S + kv
            return torch.stack(out)
        o = self.over_rms(self.per_sequence(lens, walk, r, k, v, decay), eps).reshape(-1, H * d)
        return self.times(o * self.w(p + "norm", H * d) * F.silu(self.times(mix["g"], p + "g", H * d)), p + "o", W)

    def windowed(self, h, p, m, lens, pos):
        H, G, d, eps = m["heads"], m["kv_heads"], m["dim"], self.cfg["norm"]["eps"]
        q = (self.times(h, p + "q", H * d) + self.w(p + "q.b", H * d)).view(-1, H, d)
        v = (self.times(h, p + "k", G * d) + self.w(p + "k.b", G * d)).view(-1, G, d)
        q = self.turn(self.over_rms(q, eps) * self.w(p + "q.norm", d), pos, m["rot"], pairs=True)
        k = self.turn(self.over_rms(v, eps) * self.w(p + "k.norm", d), pos, m["rot"], pairs=True)
        size, first = m["mask"]["size"], m["mask"]["keep_first"]
        sees = lambda i, j: (i - j < size) | (j < first)
        o = self.per_sequence(lens, lambda q, k, v: self.softmax_attention(q, k, v, m["scale"], sees), q, k, v)
        return self.times(o, p + "o", h.shape[1])

    def chunked(self, h, p, m, lens, pos):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (self.times(h, p + s, n * d).view(-1, n, d) for s, n in (("q", H), ("k", G), ("v", G)))
        sees = lambda i, j: i // m["mask"]["size"] == j // m["mask"]["size"]
        o = self.per_sequence(lens, lambda q, k, v: self.softmax_attention(q, k, v, m["scale"], sees), q, k, v)
        gate = torch.sigmoid(self.times(h, p + "g", H)).repeat_interleave(d, 1)
        return self.times(o * gate, p + "o", h.shape[1])

    def capped(self, h, p, m, lens, pos):
        H, G, d, eps = m["heads"], m["kv_heads"], m["dim"], self.cfg["norm"]["eps"]
        q, k, v = (self.times(h, p + s, n * d).view(-1, n, d) for s, n in (("q", H), ("k", G), ("v", G)))
        q, k = (self.over_rms(self.turn(x, pos, m["rot"]), eps) for x in (q, k))
        sink, size = self.w(p + "sink", H), m["mask"]["size"]
        one = lambda q, k, v: self.softmax_attention(q, k, v, m["scale"], lambda i, j: i // size == j // size, m["softcap"], sink)
        return self.times(self.per_sequence(lens, one, q, k, v), p + "o", h.shape[1])

    def conv(self, x, lens, name, bias=None):
        taps = self.w(name, x.shape[1], 4)

        def one(x):
            padded = F.pad(x, (0, 0, 3, 0))
            return sum(padded[j:j + x.shape[0]] * taps[:, j] for j in range(4))
        out = self.per_sequence(lens, one, x)
        return out if bias is None else out + self.w(bias, x.shape[1])

    def delta(self, h, p, m, lens, pos):
        H, G, d, dv, W, eps = m["heads"], m["kv_heads"], m["dim"], m["vdim"], h.shape[1], self.cfg["norm"]["eps"]
        q, k, v = (F.silu(self.conv(self.times(h, p + s, n), lens, p + s + ".conv")) for s, n in (("q", G * d), ("k", G * d), ("v", H * dv)))
        unit = lambda x: x / torch.sqrt(x.pow(2).sum(-1, keepdim=True) + 1e-6)
        q, k = unit(q.view(-1, G, d)) * d ** -0.5, unit(k.view(-1, G, d))
        q, k = (x.repeat_interleave(H // G, 1) for x in (q, k))
        beta = torch.sigmoid(self.times(h, p + "b", H))
        decay = torch.exp(-torch.exp(self.w(p + "A_log", H)) * F.softplus(self.times(h, p + "a", H) + self.w(p + "dt_bias", H)))

        def walk(q, k, v, beta, decay):
            S, out = torch.zeros(H, d, dv, dtype=torch.float64, device=DEVICE), []
            for t in range(q.shape[0]):
                S = decay[t, :, None, None] * S
                u = beta[t, :, None] * (v[t] - (S * k[t, :, :, None]).sum(1))
                S = S + k[t, :, :, None] * u[:, None, :]
                out.append((S * q[t, :, :, None]).sum(1))
            return torch.stack(out)
        o = self.per_sequence(lens, walk, q, k, v.view(-1, H, dv), beta, decay)
        o = (self.over_rms(o, eps) * self.w(p + "norm", dv)).reshape(-1, H * dv)
        return self.times(o * F.silu(self.times(h, p + "g", H * dv)), p + "o", W)

    def mamba1(self, h, p, m, lens, pos):
        inner, N, R = m["inner"], m["state"], m["dt_rank"]
        x, z = self.times(h, p + "in", 2 * inner).chunk(2, 1)
        x = F.silu(self.conv(x, lens, p + "conv", p + "conv.b"))
        low = self.times(x, p + "x", R + 2 * N)
        dt = F.softplus(self.times(low[:, :R], p + "dt", inner) + self.w(p + "dt.b", inner))
        A = -torch.exp(self.w(p + "A_log", inner, N))

        def walk(x, dt, B, C):
            S, out = torch.zeros(inner, N, dtype=torch.float64, device=DEVICE), []
            for t in range(x.shape[0]):
                S = torch.exp(dt[t, :, None] * A) * S + (dt[t] * x[t])[:, None] * B[t]
                out.append(S @ C[t])
            return torch.stack(out)
        y = self.per_sequence(lens, walk, x, dt, low[:, R:R + N], low[:, R + N:]) + self.w(p + "D", inner) * x
        return self.times(y * F.silu(z), p + "o", h.shape[1])

    # -- feed-forwards
    def experts(self, h, p, mlp, act, shared_act):
        r, W, ff = mlp["router"], h.shape[1], mlp["expert"]["ff"]
        E, top = r["experts"], r["top"]
        z = self.times(h, p + "router", E)
        if "groups" in r:
            s = torch.sigmoid(z)
            per = E // r["groups"]["count"]
            best = s.view(-1, r["groups"]["count"], per).topk(2, -1).values.sum(-1).topk(r["groups"]["keep"], -1).indices
            kept = torch.zeros(s.shape[0], r["groups"]["count"], dtype=torch.bool, device=DEVICE).scatter_(1, best, True)
            val, idx = s.masked_fill(~kept.repeat_interleave(per, 1), -1.0).topk(top, -1)
            weight = val / (val.sum(-1, keepdim=True) + 1e-20)
        else:
            val, idx = (z + self.w(p + "router.b", E)).topk(top, -1)
            weight = torch.softmax(val, -1)
        out = torch.zeros_like(h)
        for e in range(E):
            rows, place = (idx == e).nonzero(as_tuple=True)
            if rows.numel():
                out[rows] += weight[rows, place][:, None] * self.gated(h[rows], f"{p}e{e}.", ff, act)
        shared = self.gated(h, p + "shared.", mlp["shared"]["ff"], shared_act)
        return out + (shared * torch.sigmoid(self.times(h, p + "shared.sg", 1)) if "groups" in r else shared)

    # -- the models: the residual stream after the last layer, normed, and the head
    def qwen2(self, x, ids, lens, pos):
        z, eps = self.cfg, self.cfg["rms_norm_eps"]
        W, H, G, d, ff = z["hidden_size"], z["num_attention_heads"], z["num_key_value_heads"], z["head_dim"], z["intermediate_size"]
        rot = {"dims": d, "base": z["rope_theta"]}
        for i in range(z["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = self.over_rms(x, eps) * self.w(p + "input_layernorm.weight", W)
            q, k, v = ((self.times(h, f"{p}self_attn.{s}_proj.weight", n * d) + self.w(f"{p}self_attn.{s}_proj.bias", n * d)).view(-1, n, d)
                       for s, n in (("q", H), ("k", G), ("v", G)))
            q, k = self.turn(q, pos, rot), self.turn(k, pos, rot)
            o = self.per_sequence(lens, lambda q, k, v: self.softmax_attention(q, k, v, d ** -0.5), q, k, v)
            x = x + self.times(o, p + "self_attn.o_proj.weight", W)
            h = self.over_rms(x, eps) * self.w(p + "post_attention_layernorm.weight", W)
            g, u, down = (self.w(f"{p}mlp.{s}_proj.weight", *n) for s, n in (("gate", (ff, W)), ("up", (ff, W)), ("down", (W, ff))))
            x = x + torch.cat([(F.silu(y @ g.T) * (y @ u.T)) @ down.T for y in h.split(8192)])
        return lambda rows: self.over_rms(x[rows], eps) * self.w("model.norm.weight", W)

    def samovik(self, x, ids, lens, pos):
        W, eps = self.cfg["width"], self.cfg["norm"]["eps"]
        side = self.cfg["token_side"]["dim"]
        norm = lambda x, n: torch.tanh(self.w(n + ".alpha") * x) * self.w(n, W) + self.w(n + ".b", W)

        def act(limit):
            def clamped(g, u):
                g = g.clamp(max=limit)
                return g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1.0)
            return clamped
        for i, layer in enumerate(self.cfg["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            h = norm(x, p + "norm1")
            if layer["type"] == "latent_attention":
                x = x + self.latent(h, p + "mix.", m, lens, pos, False, m["heads"])
            else:
                x = x + getattr(self, layer["type"])(h, p + "mix.", m, lens, pos)
            x = x + self.experts(norm(x, p + "norm2"), p + "mlp.", mlp, act(mlp["expert"]["limit"]), act(mlp["shared"]["limit"]))
            e = self.w("side.embed", VOCAB, side * len(self.cfg["layers"]))[ids][:, i * side:(i + 1) * side]
            y = self.times(self.gelu(self.times(x, p + "side.gate", side)) * e, p + "side.proj", W)
            x = x + self.over_rms(y, eps) * self.w(p + "side.norm", W)
        return lambda rows: norm(x[rows], "final.norm")

    def kabulix(self, x, ids, lens, pos):
        W, eps = self.cfg["width"], self.cfg["norm"]["eps"]
        norm = lambda x, n: self.over_rms(x, eps) * (1.0 + self.w(n, W))
        silu = lambda g, u: F.silu(g) * u
        for i, layer in enumerate(self.cfg["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            h = norm(x, p + "norm1")
            if layer["type"] == "latent_attention":
                x = x + self.latent(h, p + "mix.", m, lens, pos, True, m["heads"] * m["vdim"])
            else:
                x = x + (self.windowed if layer["type"] == "attention" else self.chunked)(h, p + "mix.", m, lens, pos)
            h = norm(x, p + "norm2")
            x = x + (self.gated(h, p + "mlp.", mlp["ff"], lambda g, u: self.gelu(g) * u) if mlp["kind"] == "dense"
                     else self.experts(h, p + "mlp.", mlp, silu, silu))
        return lambda rows: norm(x[rows], "final.norm")

    def taluvik(self, x, ids, lens, pos):
        W, eps, mult = self.cfg["width"], self.cfg["norm"]["eps"], self.cfg["residual_mult"]
        norm = lambda x, n: F.layer_norm(x, (W,), self.w(n, W), self.w(n + ".b", W), eps)
        for i, layer in enumerate(self.cfg["layers"]):
            p = f"l{i}."
            h = norm(x, p + "norm1")
            mixer = self.capped if layer["type"] == "attention" else getattr(self, layer["type"])
            y = mixer(h, p + "mix.", layer["mixer"], lens, pos)
            x = x + mult * (y + self.gated(h, p + "mlp.", layer["mlp"]["ff"], lambda g, u: self.gelu(g) * u))
        return lambda rows: norm(x[rows], "final.norm")

    def forward(self, sequences: list[list[int]], rows: list[int]) -> torch.Tensor:
        ids = torch.tensor([t for s in sequences for t in s], device=DEVICE)
        lens = [len(s) for s in sequences]
        pos = torch.cat([torch.arange(n, device=DEVICE) for n in lens])
        dense = self.case["design"] in QWEN2
        W = self.cfg["hidden_size"] if dense else self.cfg["width"]
        embed, V = ("model.embed_tokens.weight" if dense else "embed"), vocab_of(self.case)
        tied = self.cfg["tie_word_embeddings"] if dense else self.case["design"] == "kabulix"
        x = self.w(embed, V, W)[ids]
        normed = (self.qwen2 if dense else getattr(self, self.case["design"]))(x, ids, lens, pos)
        return self.times(normed(torch.tensor(rows, device=DEVICE)), embed if tied else "lm_head.weight" if dense else "head", V)


@torch.no_grad()
def exact(case: dict, seed: int):
    plan, ids = shape_of(case), token_ids(case, seed)
    first, rows = 0, []
    steps = case.get("steps", 0)
    per_step = [[] for _ in range(steps + 1)]
    for (start, n, want), seq in zip(plan, ids):
        for s in range(steps + 1):
            per_step[s] += [first + start + w + s for w in want]
        first += len(seq)
    for r in per_step:
        rows += r
    logits = Plain(case, seed).forward(ids, rows)
    if steps:
        return list(logits.split([len(r) for r in per_step]))
    return {"logits": logits, "tokens": None} if case.get("sample") else logits
