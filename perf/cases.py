"""What this framework is measured on: generation and scoring through the engines' public calls.

The models are random, of the shapes that the benchmark and the tests use: a Llama shape of 8 billion weights and a Gemma shape of
one billion (Q4_0 blocks, fp16 cache), a two-layer Llama shape for the smallest calls, and the two layered-mixer designs in
bfloat16 and float32.  The library keeps one context per process, so one engine lives at a time; it is made with a model's first
case and kept, as a serving program keeps it.  Prompts come from the seed.

In all of them the head's rows are the embedding's, moved on by a few tokens, so that the best token stands as clear of the
others as a trained model's does and does not hang on a rounding.

Tasks
  answer   a short prompt in, a few greedy tokens out
  turn     a turn of a conversation whose earlier turns are in the cache already: a message in, a greedy answer out
  prompt   a long prompt in: the first token (quantised models), or the logits of its last 16 places (mixers, `score`)
  sample   a prompt in, tokens drawn with the usual chat settings (temperature 0.8, top-k 40, top-p 0.95, repeat penalty 1.1)
  batch    several prompts of equal length, answered in lockstep
  steps    a sequence continued token by token from outside, logits back at each (what a program with its own sampler does)
"""
import math

import numpy as np
import torch

GRAIN = 600011            # blocks of 32 weights in the pool that quantised matrices are cut from (a prime: no two rows are alike)
POOL = (1 << 24) + 43     # values in the mixers' pool (the same)
SHIFT = 7                 # head row t + SHIFT is embedding row t

LLM = {
    "llama3-8b": dict(arch="llama", V=128256, E=4096, H=32, G=8, D=128, L=32, FF=14336, eps=1e-5, base=5e5, sigma=0.02, embed=100.0,
                      kv_cap=4224, batch=8),
    "gemma3-1b": dict(arch="gemma3", V=262144, E=1152, H=4, G=1, D=256, L=26, FF=6912, eps=1e-6, base=1e4, sigma=0.05, embed=0.0,
                      kv_cap=4096, batch=1),
    "llama-tiny": dict(arch="llama", V=512, E=128, H=4, G=1, D=64, L=2, FF=256, eps=1e-5, base=5e5, sigma=0.1, embed=10.0, kv_cap=64,
                       batch=1),
}


def _vomotar(width, ff, heads, dtype, chunk, batch):
    """Three delta-rule layers to one of chunk attention beside retention, heads of 128."""
    delta = dict(type="channel_delta", mixer=dict(heads=heads, kv_heads=heads, dim=128, vdim=128, conv=4), mlp=dict(kind="dense", ff=ff))
    decay = [1.0 - 2.0 ** -(5 + 7 * h / (heads - 1)) for h in range(heads)]
    both = dict(type="parallel", mlp=dict(kind="dense", ff=ff), mixer=dict(
        left=dict(heads=heads, kv_heads=8, dim=128, vdim=128, scale=128 ** -0.5, mask=dict(size=8192)),
        right=dict(heads=heads, dim=128, vdim=128, decay=decay, rot=dict(base=1e4, dims=128))))
    return dict(cfg=dict(architecture="Vomotar", vocab=32768, width=width, norm=dict(groups=4, eps=1e-6), layers=[delta, delta, both, delta]),
                dtype=dtype, chunk=chunk, batch=batch)


def _zaparax(width, heads, dtype, chunk):
    """State-space and window-attention layers in turn, 6 of 32 experts beside 2 identities and a shared one."""
    mlp = dict(kind="moe", router=dict(experts=32, identity=2, top=6), expert=dict(ff=1024), shared=dict(ff=2048))
    space = dict(type="mamba2", mixer=dict(heads=2 * width // 64, groups=8, state=128, vdim=64, conv=4, norm_groups=8), mlp=mlp)
    attn = dict(type="attention", mlp=mlp, mixer=dict(heads=heads, kv_heads=8, dim=128, vdim=128, scale=128 ** -0.5, mask=dict(size=8192),
                                                      softcap=50.0, q_temp=dict(coef=0.1, every=8192)))
    return dict(cfg=dict(architecture="Zaparax", vocab=32768, width=width, norm=dict(groups=1, eps=1e-6), layers=[space, attn, space, attn],
                         embedding=dict(scale=1.0, bigram=dict(buckets=16384, mul_prev=8191, mul_cur=3))),
                dtype=dtype, chunk=chunk, batch=1)


MIXER = {
    "vomotar-4096": _vomotar(4096, 14336, 32, "bfloat16", 2048, 16),
    "vomotar-2048-f32": _vomotar(2048, 8192, 16, "float32", 512, 1),
    "zaparax-2048": _zaparax(2048, 16, "bfloat16", 2048),
}

# the range of each use: bounds of the sizes; the listed cases lie in them
RANGES = [
    ("llama-tiny", "answer", dict(prompt=(1, 24), answer=(2, 8))),
    ("gemma3-1b", "turn", dict(context=(16, 2000), prompt=(1, 48), answer=(4, 16))),
    ("gemma3-1b", "sample", dict(prompt=(17, 1000), answer=(2, 8))),
    ("llama3-8b", "turn", dict(context=(16, 4000), prompt=(1, 48), answer=(2, 8))),
    ("llama3-8b", "prompt", dict(prompt=(17, 2000))),
    ("llama3-8b", "batch", dict(sequences=(2, 8), prompt=(4, 64), answer=(2, 8))),
    ("vomotar-4096", "answer", dict(prompt=(1, 48), answer=(4, 16))),
    ("vomotar-4096", "prompt", dict(prompt=(32, 4032))),
    ("vomotar-4096", "batch", dict(sequences=(2, 16), prompt=(2, 24), answer=(2, 6))),
    ("vomotar-2048-f32", "prompt", dict(prompt=(32, 1024))),
    ("zaparax-2048", "prompt", dict(prompt=(32, 4032))),
    ("zaparax-2048", "steps", dict(prompt=(1, 300), answer=(4, 16))),
]


def listed():
    return [
        # the smallest call there is: a toy model's few tokens, all latency and launches
        dict(name="tiny-answer", model="llama-tiny", task="answer", prompt=9, answer=8),
        # a chat turn with a small model on a context of ordinary length
        dict(name="gemma1b-turn", model="gemma3-1b", task="turn", context=512, prompt=17, answer=16),
        # a document and a question, answered with the usual chat settings; not a whole number of chunks
        dict(name="gemma1b-sample", model="gemma3-1b", task="sample", prompt=701, answer=6),
        # a late turn of a long conversation with an 8B model: decode near the end of its context
        dict(name="llama8b-turn", model="llama3-8b", task="turn", context=4000, prompt=24, answer=8),
        # time to the first token behind a long prompt, ragged last chunk
        dict(name="llama8b-prompt", model="llama3-8b", task="prompt", prompt=1877),
        # a few users at once
        dict(name="llama8b-batch", model="llama3-8b", task="batch", sequences=8, prompt=48, answer=8),
        # the mixer design: a question, a long document, many users
        dict(name="vomotar-answer", model="vomotar-4096", task="answer", prompt=21, answer=16),
        dict(name="vomotar-prompt", model="vomotar-4096", task="prompt", prompt=4001),
        dict(name="vomotar-batch", model="vomotar-4096", task="batch", sequences=16, prompt=12, answer=6),
        # scoring in full float32, a short document
        dict(name="vomotar-f32-prompt", model="vomotar-2048-f32", task="prompt", prompt=600),
        # the mixture-of-experts design: scoring a document, and continuing one with a sampler of one's own
        dict(name="zaparax-prompt", model="zaparax-2048", task="prompt", prompt=3000),
        dict(name="zaparax-steps", model="zaparax-2048", task="steps", prompt=40, answer=16),
    ]


def draw(rng):
    model, task, bounds = RANGES[rng.randrange(len(RANGES))]
    case = dict(model=model, task=task)
    for k, (lo, hi) in bounds.items():
        case[k] = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) if hi > 10 * lo else rng.randint(lo, hi)
    return case


# ------------------------------------------------------------------ weights
class Embedding:
    """Float32 rows of an untied embedding, looked up on the host: the head's 8-bit rows moved by SHIFT, on the scale of a residual."""

    def __init__(self, d, codes, shape, scale):
        self.d, self.codes, self.shape, self.scale = d, codes, shape, scale

    def _of(self, rows):
        v, e = self.shape
        rows = (rows + SHIFT) % v
        c = self.codes.reshape(v, e // 32, 32)[rows].astype(np.float32) - np.float32(128.0)
        return (c * (self.d.reshape(v, e // 32, 1)[rows].astype(np.float32) * np.float32(self.scale))).reshape(len(rows), e)

    def row(self, tok):
        return self._of(np.array([int(tok)], np.int64))[0]

    def rows(self, lo, hi):
        return self._of(np.arange(lo, hi, dtype=np.int64))


def _cut(pool, at, n):
    """n values of the pool from place `at` on, round its end as often as need be."""
    out = np.empty((n,) + pool.shape[1:], pool.dtype)
    done = 0
    while done < n:
        take = min(n - done, len(pool) - at)
        out[done:done + take] = pool[at:at + take]
        done, at = done + take, 0
    return out


def _blocks(bits):
    """The pool of blocks: normal weights, quantised by each block's largest value."""
    x = np.random.default_rng(17).standard_normal((GRAIN, 32), dtype=np.float32)
    if bits == 4:
        d = np.abs(x).max(axis=1) / np.float32(8.0)
        c = np.clip(np.rint(x / d[:, None]) + 8.0, 0, 15).astype(np.uint8)
        return d, c[:, 0::2] | (c[:, 1::2] << 4)
    d = np.abs(x).max(axis=1) / np.float32(127.0)
    return d, (np.clip(np.rint(x / d[:, None]), -127, 127) + 128).astype(np.uint8)


def _llm_shapes(m):
    E, q, k = m["E"], m["H"] * m["D"], m["G"] * m["D"]
    t = {}
    for i in range(m["L"]):
        for n, s in (("attn_q", (q, E)), ("attn_k", (k, E)), ("attn_v", (k, E)), ("attn_output", (E, q)), ("ffn_gate", (m["FF"], E)),
                     ("ffn_up", (m["FF"], E)), ("ffn_down", (E, m["FF"]))):
            t[f"blk.{i}.{n}.weight"] = s
    t["token_embd.weight" if m["arch"] == "gemma3" else "output.weight"] = (m["V"], E)
    return t


def _llm_weights(m):
    """name -> (bits, shape, block scales, codes), and name -> norm weights."""
    rng = np.random.default_rng(29)
    four, eight = _blocks(4), _blocks(8) if m["arch"] == "llama" else None
    d4 = (four[0] * np.float32(m["sigma"])).astype(np.float16)
    mats = {}
    for n, (rows, k) in _llm_shapes(m).items():
        at, count = int(rng.integers(0, GRAIN)), rows * k // 32
        if n == "output.weight":
            mats[n] = (8, (rows, k), _cut((eight[0] * np.float32(m["sigma"])).astype(np.float16), at, count), _cut(eight[1], at, count).reshape(-1))
        else:
            mats[n] = (4, (rows, k), _cut(d4, at, count), _cut(four[1], at, count).reshape(-1))
    norms = {}
    for i in range(m["L"]):
        for n in ["attn_norm", "ffn_norm"] + (["post_attention_norm", "post_ffw_norm"] if m["arch"] == "gemma3" else []):
            norms[f"blk.{i}.{n}.weight"] = m["E"]
        if m["arch"] == "gemma3":
            norms[f"blk.{i}.attn_q_norm.weight"] = norms[f"blk.{i}.attn_k_norm.weight"] = m["D"]
    norms["output_norm.weight"] = m["E"]
    return mats, {n: (1.0 + 0.1 * rng.standard_normal(s)).astype(np.float32) for n, s in norms.items()}


def _mixer_tensors(cfg):
    """name -> shape."""
    E, V = cfg["width"], cfg["vocab"]
    t = {"embed": (V, E), "head": (V, E), "final.norm": (E,)}
    post = cfg["architecture"] == "Zaparax"
    if post:
        t["bigram"] = (cfg["embedding"]["bigram"]["buckets"] + 1, E)

    def attn(c, p):
        H, G, D, W = c["heads"], c["kv_heads"], c["dim"], c["vdim"]
        t.update({p + "q": (H * D, E), p + "k": (G * D, E), p + "v": (G * W, E), p + "o": (E, H * W)})

    for i, L in enumerate(cfg["layers"]):
        c, p, m = L["mixer"], f"l{i}.mix.", f"l{i}.mlp."
        for n in ["norm1", "norm2"] + (["norm1b", "norm2b"] if post else []):
            t[f"l{i}.{n}"] = (E,)
        if L["type"] == "channel_delta":
            H, K, D, W, T = c["heads"], c["kv_heads"], c["dim"], c["vdim"], c["conv"]
            t.update({p + "q": (K * D, E), p + "k": (K * D, E), p + "v": (H * W, E), p + "b": (H, E), p + "a1": (128, E), p + "a2": (H * D, 128),
                      p + "g1": (128, E), p + "g2": (H * W, 128), p + "o": (E, H * W), p + "q.conv": (K * D, T), p + "k.conv": (K * D, T),
                      p + "v.conv": (H * W, T), p + "A_log": (H,), p + "dt_bias": (H * D,), p + "norm": (W,)})
        elif L["type"] == "parallel":
            l, r = c["left"], c["right"]
            attn(l, p + "left.")
            t.update({p + "left.r1": (l["heads"],), p + "left.r2": (l["heads"],), p + "left.out": (E,), p + "right.out": (E,)})
            H, D, W = r["heads"], r["dim"], r["vdim"]
            t.update({p + "right.q": (H * D, E), p + "right.k": (H * D, E), p + "right.v": (H * W, E), p + "right.g": (H * W, E),
                      p + "right.o": (E, H * W)})
        elif L["type"] == "attention":
            attn(c, p)
            t.update({p + "q.b": (c["heads"] * c["dim"],), p + "k.b": (c["kv_heads"] * c["dim"],), p + "v.b": (c["kv_heads"] * c["vdim"],),
                      p + "sink": (c["heads"],)})
        else:
            H, G, N, W = c["heads"], c["groups"], c["state"], c["vdim"]
            wide = H * W + 2 * G * N
            t.update({p + "in": (H * W + wide + H, E), p + "conv": (wide, c["conv"]), p + "conv.b": (wide,), p + "dt_bias": (H,), p + "A_log": (H,),
                      p + "D": (H,), p + "norm": (H * W,), p + "o": (E, H * W)})
        f = L["mlp"]
        if f["kind"] == "dense":
            t.update({m + "gate": (f["ff"], E), m + "up": (f["ff"], E), m + "down": (E, f["ff"])})
        else:
            n, one, sh = f["router"]["experts"] + f["router"]["identity"], f["expert"]["ff"], f["shared"]["ff"]
            t.update({m + "router": (n, E), m + "correction": (n,), m + "shared.gate": (sh, E), m + "shared.up": (sh, E), m + "shared.down": (E, sh),
                      m + "shared.sg": (1, E)})
            for e in range(f["router"]["experts"]):
                t.update({m + f"e{e}.gate": (one, E), m + f"e{e}.up": (one, E), m + f"e{e}.down": (E, one)})
    return t


def _bf16(x):
    return torch.from_numpy(x).bfloat16().view(torch.int16).numpy().view(np.uint16)


def _mixer_weights(cfg):
    """name -> bfloat16 bit patterns (uint16)."""
    rng = np.random.default_rng(31)
    pool = rng.standard_normal(POOL, dtype=np.float32)
    scaled, out = {}, {}
    around = {"A_log": (-2.0, 0.5), "dt_bias": (-3.0, 0.5), "r1": (0.5, 0.1), "r2": (0.3, 0.05), "sink": (0.0, 1.0), "b": (0.0, 0.1),
              "correction": (0.0, 0.01)}
    zero = 1.0 if cfg["architecture"] == "Zaparax" else 0.0      # its residual norms are stored around zero
    for n, shape in _mixer_tensors(cfg).items():
        last, at, size = n.split(".")[-1], int(rng.integers(0, POOL)), int(np.prod(shape))
        if len(shape) == 1:
            centre, spread = around.get(last, (1.0, 0.1))
            centre -= zero if "norm" in n and ".mix." not in n else 0.0
            out[n] = _bf16(np.float32(centre) + np.float32(spread) * pool[:size])
        elif n != "head":
            k = 1.0 if last == "conv" or n in ("embed", "bigram") else shape[-1] ** -0.5
            if k not in scaled:
                scaled[k] = _bf16(pool * np.float32(k))
            out[n] = _cut(scaled[k], at, size).reshape(shape)
    e = torch.from_numpy(np.roll(out["embed"], SHIFT, axis=0).view(np.int16)).view(torch.bfloat16)
    out["head"] = (e.float() * cfg["width"] ** -0.5).bfloat16().view(torch.int16).numpy().view(np.uint16)
    return out


_kept = {}


def _weights(model):
    """The model's weights on the host; one model's are kept."""
    if _kept.get("weights", (None,))[0] != model:
        _kept.pop("weights", None)
        _kept["weights"] = (model, _llm_weights(LLM[model]) if model in LLM else _mixer_weights(MIXER[model]["cfg"]))
    return _kept["weights"][1]


# ------------------------------------------------------------------ engines
def _engine(model):
    """The serving program's engine for the model, loaded once; another model's is shut down first."""
    if _kept.get("engine", (None,))[0] == model:
        return _kept["engine"][1]
    from adam_amd import adamah
    if "engine" in _kept:
        _kept.pop("engine")[1].gpu.shutdown()
    w, gpu = _weights(model), adamah.init()
    if model in LLM:
        from adam_amd.engine import DecodeEngine, ModelConfig
        from adam_amd.quant import QTensor
        m = LLM[model]
        gemma = m["arch"] == "gemma3"
        cfg = ModelConfig(arch=m["arch"], n_vocab=m["V"], n_ctx=m["kv_cap"], n_embd=m["E"], n_head=m["H"], n_head_kv=m["G"], n_layer=m["L"],
                          n_ff=m["FF"], head_dim=m["D"], head_dim_kv=m["D"], norm_eps=m["eps"], rope_base_global=1e6 if gemma else m["base"],
                          rope_base_local=m["base"], ffn_act="gelu" if gemma else "silu", emb_scale=float(np.sqrt(m["E"])) if gemma else 1.0,
                          attn_softcap=50.0 if gemma else 0.0, final_softcap=30.0 if gemma else 0.0)
        tensors = {n: QTensor("q4_0" if bits == 4 else "q8_0", shape, d, codes) for n, (bits, shape, d, codes) in w[0].items()}
        tensors.update(w[1])
        if not gemma:
            _, shape, d, codes = w[0]["output.weight"]
            tensors["token_embd.weight"] = Embedding(d, codes, shape, m["embed"])
        eng = DecodeEngine(gpu, cfg, tensors, kv_cap=m["kv_cap"], kv_fp16=True, fusion_scheduler_mode="level_batched",
                           prefill_chunk=512 if m["L"] > 2 else 0, batch=m["batch"])
    else:
        from adam_amd.mixer_engine import MixerEngine
        from adam_amd.models import ARCHITECTURES
        m = MIXER[model]
        eng = MixerEngine(gpu, ARCHITECTURES[m["cfg"]["architecture"]](m["cfg"]), w, dtype=m["dtype"], prefill_chunk=m["chunk"], batch=m["batch"])
    _kept["engine"] = (model, eng)
    _kept["cached"] = 0
    return eng


def _vocab(model):
    return LLM[model]["V"] if model in LLM else MIXER[model]["cfg"]["vocab"]


def _context(case):
    """The earlier turns of a conversation: the same for every seed, so that they can stay in the cache."""
    return np.random.default_rng(101).integers(0, _vocab(case["model"]), 4096)[:case["context"]]


def _tokens(case, seed):
    """[sequences, prompt] token ids."""
    return np.random.default_rng([seed, 5]).integers(0, _vocab(case["model"]), (case.get("sequences", 1), case["prompt"]))


def prepare(case, seed):
    eng = _engine(case["model"])
    state = dict(case=case, engine=eng, seed=int(seed))
    toks = _tokens(case, seed)
    if case["task"] == "turn":
        context = [int(t) for t in _context(case)]
        if _kept["cached"] < len(context):
            eng.prefill(context)
            eng.gpu.sync()
            _kept["cached"] = len(context)
        state["prompt"] = context + [int(t) for t in toks[0]]
    else:
        _kept["cached"] = 0                       # the pass writes the cache from its first row on
        state["prompt"] = [int(t) for t in toks[0]]
        state["prompts"] = [[int(t) for t in row] for row in toks]
        if case["task"] == "steps":
            state["next"] = [int(t) for t in np.random.default_rng([seed, 6]).integers(0, _vocab(case["model"]), case["answer"])]
    return state


def _want(case):
    return list(range(max(0, case["prompt"] - 16), case["prompt"]))


def run(state):
    from adam_amd.engine import GenerationConfig
    case, eng = state["case"], state["engine"]
    task, llm = case["task"], case["model"] in LLM
    if task == "prompt" and not llm:
        logits = eng.score("document", state["prompt"], _want(case))
        eng.release("document")
        return dict(logits=logits)
    if task == "steps":
        logits = [eng.score("text", state["prompt"], [case["prompt"] - 1])]
        logits += [eng.score("text", [t], [0]) for t in state["next"]]
        eng.release("text")
        return dict(logits=np.concatenate(logits))
    if task == "batch":
        toks, _ = eng.generate_batch(state["prompts"], case["answer"])
        n = case["sequences"]
        if llm:
            width = LLM[case["model"]]["E"]
            at = eng._cp["normed"]
            last = eng.gpu.gather(0, np.arange(at, at + n * width, dtype=np.uint32)).view(np.float32).reshape(n, width)
        else:
            last = eng.read_rows("hidden", n)
        return dict(tokens=np.array(toks, np.int64), last=[row for row in last])
    if task == "sample":
        chat = GenerationConfig.reference_defaults(max_tokens=case["answer"], seed=state["seed"], eos_token_ids=())
        toks, _ = eng.generate(state["prompt"], chat)
        return dict(tokens=np.array(toks, np.int64), last=eng.read_slot("normed"), best=eng.read_slot("sample_topk_val")[:40])
    toks, _ = eng.generate(state["prompt"], GenerationConfig(max_tokens=case.get("answer", 1)), reuse_prefix=case.get("context", 0))
    return dict(tokens=np.array(toks, np.int64), last=eng.read_slot("normed" if llm else "hidden"))


# ------------------------------------------------------------------ what a pass cannot do without
def _active(model):
    """(bytes a one-token step reads of the weights, bytes all of them have, weights a token is multiplied by without the head, the head's)."""
    if model in LLM:
        m = LLM[model]
        body = head = moved = 0
        for n, (r, k) in _llm_shapes(m).items():
            moved += r * k * (34 if n == "output.weight" else 18) // 32
            if r == m["V"]:
                head = r * k
            else:
                body += r * k
        return moved, moved, body, head
    cfg = MIXER[model]["cfg"]
    total = used = 0
    for n, s in _mixer_tensors(cfg).items():
        if len(s) == 2 and n not in ("embed", "head", "bigram"):
            size = s[0] * s[1]
            total += size
            f = cfg["layers"][int(n[1:n.index(".")])]["mlp"]
            if f["kind"] == "moe" and ".mlp.e" in n:
                size *= f["router"]["top"] / (f["router"]["experts"] + f["router"]["identity"])
            used += size
    head = cfg["vocab"] * cfg["width"]
    return 2 * (used + head), 2 * (total + head), used, head


def _attention(model):
    """(bytes of cached keys and values per token, operations per query and key) over all layers."""
    if model in LLM:
        m = LLM[model]
        return 4 * m["L"] * m["G"] * m["D"], 4 * m["L"] * m["H"] * m["D"]
    mx, by, fl = MIXER[model], 0, 0
    for L in mx["cfg"]["layers"]:
        c = L["mixer"].get("left", L["mixer"])
        if "mask" in c:
            by += (2 if mx["dtype"] == "bfloat16" else 4) * 2 * c["kv_heads"] * c["dim"]
            fl += 4 * c["heads"] * c["dim"]
    return by, fl


def _state_bytes(model):
    """Recurrent state of a sequence, read and written by a step."""
    if model in LLM:
        return 0
    n = 0
    for L in MIXER[model]["cfg"]["layers"]:
        c = L["mixer"].get("right", L["mixer"])
        n += c["heads"] * (c["state"] if "state" in c else c["dim"]) * c["vdim"] if "mask" not in c else 0
    return 8 * n


def work(case):
    step, whole, body, head = _active(case["model"])
    kv, score = _attention(case["model"])
    B, P, C, N = case.get("sequences", 1), case["prompt"], case.get("context", 0), case.get("answer", 1)
    if case["task"] == "prompt" and case["model"] not in LLM:
        N = 0
    many = lambda rows: min(whole, step * max(1, rows))           # a mixture's experts: as many as its rows can choose
    keys = P * C + P * (P + 1) / 2
    rows = 16 if case["task"] == "prompt" and N == 0 else 1
    b = many(B * P) + B * kv * (C + P)
    f = B * (2.0 * body * P + score * keys + 2.0 * head * min(rows, P))
    for i in range(N):
        b += many(B) + B * (kv * (C + P + i) + _state_bytes(case["model"]))
        f += B * (2.0 * (body + head) + score * (C + P + i))
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Four times the largest distance from `exact` seen over the listed and some drawn cases: 7e-4 with a 16-bit cache and float16
    operand rows, 3e-6 in float32, 4e-3 with bfloat16 operand rows (0.8e-2 where they also decide which expert a row takes)."""
    if case["model"] in LLM:
        return {"rel": 3e-3}
    if MIXER[case["model"]]["dtype"] == "float32":
        return {"rel": 1.2e-5}
    return {"rel": 3e-2 if case["model"].startswith("zaparax") else 1.6e-2}


# ------------------------------------------------------------------ the same in 64 bits
def _f64(x):
    return x.to(torch.float64)


def _silu(z):
    return z / (1.0 + torch.exp(-z))


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, pos, base, dims):
    """x [T, H, D]: pairs (i, i + dims / 2) turned by p * base^(-2 i / dims)."""
    half = dims // 2
    ang = pos[:, None] * base ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / dims)
    cs, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    u, w = x[..., :half], x[..., half:dims]
    return torch.cat([u * cs - w * sn, w * cs + u * sn, x[..., dims:]], -1)


class _Llm:
    """The quantised models' forward pass over cached keys and values."""

    def __init__(self, model):
        self.m = LLM[model]
        mats, norms = _weights(model)
        self.mats = {n: (bits, s, torch.from_numpy(d).cuda(), torch.from_numpy(c).cuda()) for n, (bits, s, d, c) in mats.items()}
        self.norms = {n: _f64(torch.from_numpy(v).cuda()) for n, v in norms.items()}
        self.head = "token_embd.weight" if self.m["arch"] == "gemma3" else "output.weight"

    def mat(self, name, rows=None):
        bits, (n, k), d, c = self.mats[name]
        d, c = d.view(n, k // 32, 1), c.view(n, -1)
        if rows is not None:
            n, d, c = len(rows), d[rows], c[rows]
        c = torch.stack([c & 15, c >> 4], -1).view(n, k // 32, 32).double() - 8.0 if bits == 4 else c.view(n, k // 32, 32).double() - 128.0
        return (c * d.double()).view(n, k)

    def step(self, toks, cache):
        """Normed rows [T, E] of tokens behind `cache` (a list of (keys, values) per layer, extended here)."""
        m, w = self.m, self.norms
        H, G, D, eps, gemma = m["H"], m["G"], m["D"], m["eps"], m["arch"] == "gemma3"
        rows = torch.as_tensor(toks, device="cuda")
        x = self.mat(self.head, rows) * m["E"] ** 0.5 if gemma else self.mat(self.head, (rows + SHIFT) % m["V"]) * m["embed"]
        T, past = len(rows), cache[0][0].shape[0] if cache else 0
        pos = torch.arange(past, past + T, dtype=torch.float64, device="cuda")
        for i in range(m["L"]):
            p = f"blk.{i}."
            base = 1e6 if gemma and (i + 1) % 6 == 0 else m["base"]
            h = _rms(x, eps) * w[p + "attn_norm.weight"]
            q = (h @ self.mat(p + "attn_q.weight").T).view(T, H, D)
            k = (h @ self.mat(p + "attn_k.weight").T).view(T, G, D)
            v = (h @ self.mat(p + "attn_v.weight").T).view(T, G, D)
            if gemma:
                q, k = _rms(q, 1e-6) * w[p + "attn_q_norm.weight"], _rms(k, 1e-6) * w[p + "attn_k_norm.weight"]
            q, k = _turn(q, pos, base, D), _turn(k, pos, base, D)
            if len(cache) <= i:
                cache.append((k, v))
            else:
                cache[i] = (torch.cat([cache[i][0], k]), torch.cat([cache[i][1], v]))
            k, v = cache[i]
            seen = torch.arange(past + T, device="cuda")[None] <= torch.arange(past, past + T, device="cuda")[:, None]
            o = torch.empty(T, H, D, dtype=torch.float64, device="cuda")
            for n in range(H):
                s = q[:, n] @ k[:, n // (H // G)].T / D ** 0.5
                if gemma:
                    s = 50.0 * torch.tanh(s / 50.0)
                o[:, n] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[:, n // (H // G)]
            y = o.view(T, H * D) @ self.mat(p + "attn_output.weight").T
            x = x + (_rms(y, eps) * w[p + "post_attention_norm.weight"] if gemma else y)
            h = _rms(x, eps) * w[p + "ffn_norm.weight"]
            a = h @ self.mat(p + "ffn_gate.weight").T
            a = torch.nn.functional.gelu(a, approximate="tanh") if gemma else _silu(a)
            y = (a * (h @ self.mat(p + "ffn_up.weight").T)) @ self.mat(p + "ffn_down.weight").T
            x = x + (_rms(y, eps) * w[p + "post_ffw_norm.weight"] if gemma else y)
        return _rms(x, eps) * w["output_norm.weight"]

    def logits(self, row):
        return torch.cat([self.mat(self.head, torch.arange(lo, min(self.m["V"], lo + 32768), device="cuda")) @ row
                          for lo in range(0, self.m["V"], 32768)])


def _cap(z):
    return 30.0 * torch.tanh(z / 30.0)


def _best(z, past):
    """The 40 best logits (capped) and their tokens, the penalty on tokens that were drawn already."""
    if past:
        at = torch.tensor(sorted(set(past[-64:])), device=z.device)
        z[at] = torch.where(z[at] > 0, z[at] / 1.1, z[at] * 1.1)
    val, ids = torch.topk(z, 40)
    return _cap(val), ids


def _answer_llm(net, toks, case, seed):
    """(tokens, last normed row, best 40 logits behind it), the row None where a choice was too close for 16-bit operands to settle."""
    cache, out, sure, best = [], [], True, None
    rng = np.random.default_rng(seed)
    for lo in range(0, len(toks), 1024):
        row = net.step(toks[lo:lo + 1024], cache)[-1]
    for _ in range(case.get("answer", 1)):
        z = net.logits(row)
        if case["task"] == "sample":
            val, ids = _best(z, out)
            p = torch.softmax(val / 0.8, 0)
            keep = int((torch.cumsum(p, 0) < 0.95).sum()) + 1
            run = torch.cumsum(p[:keep] / p[:keep].sum(), 0)
            r = np.float32(rng.random())
            sure = sure and float((run - float(r)).abs().min()) > 0.01 and float((torch.cumsum(p, 0) - 0.95).abs().min()) > 1e-3
            out.append(int(ids[min(int((run <= float(r)).sum()), keep - 1)]))
        else:
            val, ids = torch.topk(z, 2)
            sure = sure and float(val[0] - val[1]) > 0.03 * float(z.std())
            out.append(int(ids[0]))
        row = net.step(out[-1:], cache)[-1]
    if case["task"] == "sample":
        best = _best(net.logits(row), out)[0].cpu().numpy()
    return out, row.cpu().numpy() if sure else None, best if sure else None


class _Mixer:
    """The mixers' forward pass over whole sequences, recurrences token by token."""

    def __init__(self, model):
        self.c = MIXER[model]["cfg"]
        self.w = {n: torch.from_numpy(a.view(np.int16)).cuda().view(torch.bfloat16) for n, a in _weights(model).items()}
        self.eps = self.c["norm"]["eps"]

    def g(self, n):
        return self.w[n].double()

    def mm(self, h, n):
        return h @ self.g(n).T

    def conv(self, x, n, bias=None):
        w = self.g(n)
        J = w.shape[1]
        xp = torch.cat([x.new_zeros(J - 1, x.shape[1]), x])
        y = sum(w[:, j] * xp[j:j + x.shape[0]] for j in range(J))
        return _silu(y if bias is None else y + self.g(bias))

    def delta(self, h, p, c):
        T, H, K, D, V = h.shape[0], c["heads"], c["kv_heads"], c["dim"], c["vdim"]
        unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        q = unit(self.conv(self.mm(h, p + "q"), p + "q.conv").view(T, K, D)) * D ** -0.5
        k = unit(self.conv(self.mm(h, p + "k"), p + "k.conv").view(T, K, D))
        q, k = q.repeat_interleave(H // K, 1), k.repeat_interleave(H // K, 1)
        v = self.conv(self.mm(h, p + "v"), p + "v.conv").view(T, H, V)
        beta = torch.sigmoid(self.mm(h, p + "b"))
        a = (self.mm(self.mm(h, p + "a1"), p + "a2") + self.g(p + "dt_bias")).view(T, H, D)
        g = torch.exp(-torch.exp(self.g(p + "A_log"))[:, None] * torch.nn.functional.softplus(a, threshold=1e9))
        S, o = h.new_zeros(H, D, V), torch.empty_like(v)
        for t in range(T):
            S = g[t][:, :, None] * S
            u = beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], S)[:, 0])
            S = torch.baddbmm(S, k[t][:, :, None], u[:, None])
            o[t] = torch.bmm(q[t][:, None], S)[:, 0]
        gate = torch.sigmoid(self.mm(self.mm(h, p + "g1"), p + "g2"))
        return self.mm((_rms(o, self.eps) * self.g(p + "norm")).view(T, H * V) * gate, p + "o")

    def attend(self, q, k, v, weigh):
        """Heads in turn: `weigh` makes softmax weights [T, T] of a head's raw scores."""
        T, H, G = q.shape[0], q.shape[1], k.shape[1]
        i = torch.arange(T, device="cuda")
        far = (i[:, None] - i[None]).double()
        o = torch.empty(T, H, v.shape[2], dtype=torch.float64, device="cuda")
        for n in range(H):
            o[:, n] = weigh(q[:, n] @ k[:, n // (H // G)].T, far, n) @ v[:, n // (H // G)]
        return o.view(T, -1)

    def chunk_attention(self, h, p, c):
        T, H, G, D, V = h.shape[0], c["heads"], c["kv_heads"], c["dim"], c["vdim"]
        r1, r2 = self.g(p + "r1"), self.g(p + "r2")
        at = torch.arange(T, device="cuda") // c["mask"]["size"]

        def weigh(s, far, n):
            s = s * c["scale"] - r1[n] * torch.log1p(r2[n] * far.clamp(min=0))
            return torch.softmax(s.masked_fill((far < 0) | (at[:, None] != at[None]), -math.inf), -1)
        v = _rms(self.mm(h, p + "v").view(T, G, V), self.eps)
        return self.mm(self.attend(self.mm(h, p + "q").view(T, H, D), self.mm(h, p + "k").view(T, G, D), v, weigh), p + "o")

    def retention(self, h, p, c):
        T, H, D, V = h.shape[0], c["heads"], c["dim"], c["vdim"]
        pos = torch.arange(T, dtype=torch.float64, device="cuda")
        q = _turn(self.mm(h, p + "q").view(T, H, D), pos, c["rot"]["base"], c["rot"]["dims"])
        k = _turn(self.mm(h, p + "k").view(T, H, D), pos, c["rot"]["base"], c["rot"]["dims"]) * D ** -0.5
        v = self.mm(h, p + "v").view(T, H, V)
        decay = torch.tensor(c["decay"], dtype=torch.float64, device="cuda")[:, None, None]
        S, o = h.new_zeros(H, D, V), torch.empty_like(v)
        for t in range(T):
            S = torch.baddbmm(decay * S, k[t][:, :, None], v[t][:, None])
            o[t] = torch.bmm(q[t][:, None], S)[:, 0]
        return self.mm(_rms(o, self.eps).view(T, -1) * _silu(self.mm(h, p + "g")), p + "o")

    def window_attention(self, h, p, c):
        T, H, G, D, V = h.shape[0], c["heads"], c["kv_heads"], c["dim"], c["vdim"]
        q = _rms((self.mm(h, p + "q") + self.g(p + "q.b")).view(T, H, D), self.eps)
        k = _rms((self.mm(h, p + "k") + self.g(p + "k.b")).view(T, G, D), self.eps)
        v = (self.mm(h, p + "v") + self.g(p + "v.b")).view(T, G, V)
        pos, temp, sink = torch.arange(T, dtype=torch.float64, device="cuda"), c["q_temp"], self.g(p + "sink")
        q = q * (1.0 + temp["coef"] * torch.log(torch.floor((pos + 1) / temp["every"]) + 1.0))[:, None, None]

        def weigh(s, far, n):
            s = c["softcap"] * torch.tanh(s * c["scale"] / c["softcap"]) - 2.0 ** (-8.0 * (n + 1) / H) * far
            s = s.masked_fill((far < 0) | (far >= c["mask"]["size"]), -math.inf)
            top = s.max(1, keepdim=True).values.clamp(min=float(sink[n]))
            e = torch.exp(s - top)
            return e / (e.sum(1, keepdim=True) + torch.exp(sink[n] - top))
        return self.mm(self.attend(q, k, v, weigh), p + "o")

    def space(self, h, p, c):
        T, H, V, N, G = h.shape[0], c["heads"], c["vdim"], c["state"], c["groups"]
        u = self.mm(h, p + "in")
        z, xbc, dt = u[:, :H * V], u[:, H * V:2 * H * V + 2 * G * N], u[:, 2 * H * V + 2 * G * N:]
        xbc = self.conv(xbc, p + "conv", p + "conv.b")
        x = xbc[:, :H * V].reshape(T, H, V)
        B = xbc[:, H * V:H * V + G * N].reshape(T, G, N).repeat_interleave(H // G, 1)
        C = xbc[:, H * V + G * N:].reshape(T, G, N).repeat_interleave(H // G, 1)
        dt = torch.nn.functional.softplus(dt + self.g(p + "dt_bias"), threshold=1e9)
        keep = torch.exp(-torch.exp(self.g(p + "A_log")) * dt)
        S, y = h.new_zeros(H, N, V), torch.empty_like(x)
        for t in range(T):
            S = torch.baddbmm(keep[t][:, None, None] * S, (dt[t][:, None] * B[t])[:, :, None], x[t][:, None])
            y[t] = torch.bmm(C[t][:, None], S)[:, 0]
        y = (y + self.g(p + "D")[:, None] * x).view(T, -1) * _silu(z)
        return self.mm(_rms(y.view(T, c["norm_groups"], -1), self.eps).view(T, -1) * self.g(p + "norm"), p + "o")

    def gated(self, h, p):
        return self.mm(_silu(self.mm(h, p + "gate")) * self.mm(h, p + "up"), p + "down")

    def experts(self, h, p, c):
        r = c["router"]
        s = torch.softmax(self.mm(h, p + "router"), -1)
        ids = torch.topk(s + self.g(p + "correction"), r["top"]).indices
        w = torch.zeros_like(s).scatter(1, ids, s.gather(1, ids))
        y = torch.sigmoid(self.mm(h, p + "shared.sg")) * self.gated(h, p + "shared.")
        for e in range(s.shape[1]):
            rows = torch.nonzero(w[:, e])[:, 0]
            if len(rows):
                y[rows] += w[rows, e:e + 1] * (self.gated(h[rows], p + f"e{e}.") if e < r["experts"] else h[rows])
        return y

    def rows(self, toks):
        """(hidden rows [T, E], normed rows)."""
        c, eps = self.c, self.eps
        toks = torch.as_tensor(toks, device="cuda")
        x = self.w["embed"][toks].double()
        post = c["architecture"] == "Zaparax"
        if post:
            b = c["embedding"]["bigram"]
            pair = (torch.roll(toks, 1) * b["mul_prev"] + toks * b["mul_cur"]) % b["buckets"]
            pair[0] = b["buckets"]
            x = x + self.w["bigram"][pair].double()
        groups = c["norm"]["groups"]
        norm = lambda x, n: _rms(x.view(x.shape[0], groups, -1), eps).view(x.shape) * (self.g(n) + (1.0 if post else 0.0))
        behind = (lambda y, n: norm(y, n)) if post else (lambda y, n: y)
        kinds = {"channel_delta": self.delta, "attention": self.window_attention, "mamba2": self.space}
        for i, L in enumerate(c["layers"]):
            h, p, m = norm(x, f"l{i}.norm1"), f"l{i}.mix.", L["mixer"]
            if L["type"] == "parallel":
                left, right = self.chunk_attention(h, p + "left.", m["left"]), self.retention(h, p + "right.", m["right"])
                y = 0.5 * (_rms(left, eps) * self.g(p + "left.out") + _rms(right, eps) * self.g(p + "right.out"))
            else:
                y = kinds[L["type"]](h, p, m)
            x = x + behind(y, f"l{i}.norm1b")
            h = norm(x, f"l{i}.norm2")
            x = x + behind(self.experts(h, f"l{i}.mlp.", L["mlp"]) if L["mlp"]["kind"] == "moe" else self.gated(h, f"l{i}.mlp."), f"l{i}.norm2b")
        return x, norm(x, "final.norm")


def _answer_mixer(net, toks, count):
    toks, out, sure = list(toks), [], True
    for _ in range(count):
        z = net.mm(net.rows(toks)[1][-1:], "head")[0]
        val, ids = torch.topk(z, 2)
        sure = sure and float(val[0] - val[1]) > 0.03 * float(z.std())
        out.append(int(ids[0]))
        toks.append(out[-1])
    return out, net.rows(toks)[0][-1].cpu().numpy() if sure else None


def exact(case, seed):
    model, task = case["model"], case["task"]
    if _kept.get("net", (None,))[0] != model:
        _kept.pop("net", None)
        torch.cuda.empty_cache()
        _kept["net"] = (model, (_Llm if model in LLM else _Mixer)(model))
    net, toks = _kept["net"][1], _tokens(case, seed)
    if model not in LLM and task in ("prompt", "steps"):
        whole, at = toks[0], _want(case)
        if task == "steps":
            whole = np.concatenate([whole, np.random.default_rng([seed, 6]).integers(0, _vocab(model), case["answer"])])
            at = list(range(case["prompt"] - 1, len(whole)))
        return dict(logits=net.mm(net.rows(whole)[1][at], "head").cpu().numpy())
    if model not in LLM:
        got = [_answer_mixer(net, t, case["answer"]) for t in toks]
    else:
        context = _context(case) if "context" in case else []
        got = [_answer_llm(net, [int(t) for t in [*context, *t]], case, seed) for t in toks]
    if task == "batch":
        return dict(tokens=None, last=[g[1] for g in got])
    if task == "sample":
        return dict(tokens=None, last=got[0][1], best=got[0][2])
    return dict(tokens=None, last=got[0][1])
