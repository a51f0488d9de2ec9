"""What a user has this engine do, as cases that can be timed and checked: prompts in, generated tokens out, through
``Engine.add_request`` / ``step`` / ``take_finished``, on models with random weights of the sizes that bench.py and the
command lines know.

A case is a plain dict:

  design    "llama" | "kasuvik" | "fisesun"
  sizes     llama: a name of NAMED_SIZES; the others: the width of the model (bench.py --design's sizes)
  layers    layers of the model
  dtype     "bfloat16" | "float32"
  requests  requests of one pass, all there at its beginning
  prompt    tokens of every prompt; with ``spread`` > 0 the median of prompts whose logarithms are spread by that much
  new       tokens that every request generates; with ``chunk`` > 0 all requests but the last generate between a
            quarter and half of that
  chunk     0: all prompts fit one step; > 0: prompts enter in portions of that many tokens beside the tokens of the
            requests that decode already, 1,024 tokens a step

A pass returns every request's tokens and the logits of the pass's last step (the last token of every request; with
``chunk`` > 0 of the last request alone).

The output head's rows are the embedding's in another order, so that a token's successor stands above the others as it
does in a trained model: what greedy decoding picks then does not hang on rounding.
"""
import math

import numpy as np
import torch

import kvcm_amd
from kvcm_amd.cli.common import NAMED_SIZES
from kvcm_amd.config.fisesun_config import FisesunConfig
from kvcm_amd.config.kasuvik_config import KasuvikConfig
from kvcm_amd.config.model_config import LlamaConfig
from kvcm_amd.weights.random_init import expected_tensors

STEP_TOKENS = 1024       # tokens a step when prompts enter in portions
WORK_CAP = 36864         # tokens of one pass at most, in drawn cases


def listed():
    def case(name, design, sizes, layers, requests, prompt, new, dtype="bfloat16", spread=0.0, chunk=0):
        return dict(name=name, design=design, sizes=sizes, layers=layers, dtype=dtype, requests=requests, prompt=prompt,
                    spread=spread, new=new, chunk=chunk)
    return [
        # a test run of three short requests on a model of two layers, in 32 bits: launches and host time
        case("tiny model in 32 bits", "llama", "tiny-a", 2, 3, 8, 8, dtype="float32", spread=0.4),
        # one user chats: single rows
        case("chat with one user", "llama", "tinyllama-1.1b", 22, 1, 512, 128),
        # the headline workload of bench.py: eight requests decode together
        case("decode eight requests", "llama", "tinyllama-1.1b", 22, 8, 512, 128),
        # an offline batch: 64 prompts of 512 tokens at once, then 64 rows a step
        case("offline batch of 64", "llama", "tinyllama-1.1b", 22, 64, 512, 64),
        # a document is read and one token comes back (a classification, or the wait for the first token)
        case("one prompt of 2048", "llama", "tinyllama-1.1b", 22, 1, 2048, 1),
        # serving: ragged prompts enter in portions beside requests that decode, which end one after the other
        case("served 24 ragged requests", "llama", "tinyllama-1.1b", 22, 24, 403, 64, spread=0.8, chunk=512),
        # the 32-bit path that answers are checked against
        case("checked in 32 bits", "llama", "tinyllama-1.1b", 22, 2, 301, 16, dtype="float32", spread=0.3),
        # a larger model with longer contexts of all lengths
        case("8B eight long contexts", "llama", "llama-3-8b", 32, 8, 1201, 32, spread=0.3),
        # the Kasuvik decoder: a prompt, and eight requests that decode
        case("Kasuvik one prompt of 2048", "kasuvik", 2048, 4, 1, 2048, 1),
        case("Kasuvik eight requests", "kasuvik", 2048, 4, 8, 509, 64),
        # the Fisesun decoder (experts): a prompt, and eight requests that decode
        case("Fisesun one prompt of 2048", "fisesun", 2048, 4, 1, 2048, 1),
        case("Fisesun eight requests", "fisesun", 2048, 4, 8, 509, 64),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["llama", "llama", "llama", "served", "llama 8b", "32 bits", "32 bits tiny", "kasuvik", "kasuvik", "fisesun", "fisesun"])
    c = dict(design="llama", sizes="tinyllama-1.1b", layers=22, dtype="bfloat16", requests=1, prompt=1, spread=0.0, new=1, chunk=0)
    if kind == "served":
        c.update(requests=rng.randint(9, 32), prompt=_log_int(rng, 100, 500), spread=round(rng.uniform(0.3, 0.8), 2),
                 new=rng.randint(24, 64), chunk=rng.choice([128, 256, 512]))
        return c
    if kind == "llama 8b":
        c.update(sizes="llama-3-8b", layers=32, requests=_log_int(rng, 1, 8), prompt=_log_int(rng, 64, 1200), spread=0.3, new=_log_int(rng, 1, 32))
    elif kind == "32 bits":
        c.update(dtype="float32", requests=_log_int(rng, 1, 3), prompt=_log_int(rng, 10, 300), spread=0.3, new=_log_int(rng, 1, 16))
    elif kind == "32 bits tiny":
        c.update(sizes=rng.choice(["tiny-a", "tiny-b"]), dtype="float32", requests=rng.randint(1, 6), prompt=rng.randint(3, 24),
                 spread=0.4, new=rng.randint(2, 16))
        c["layers"] = NAMED_SIZES[c["sizes"]]["num_hidden_layers"]
    else:
        if kind != "llama":
            c.update(design=kind, sizes=rng.choice([2048, 2048, 4096]), layers=4)
        most = 64 if kind == "llama" else 16
        c["requests"] = _log_int(rng, 1, most)
        c["prompt"] = _log_int(rng, 8, 2048 if kind == "llama" else 2304)
        c["new"] = rng.choice([1, _log_int(rng, 2, 128), _log_int(rng, 2, 128)])
        c["spread"] = rng.choice([0.0, 0.3])
        room = WORK_CAP if kind == "llama" else 6144 if c["sizes"] == 2048 else 2560
        c["prompt"] = max(1, min(c["prompt"], room // c["requests"] - c["new"]))
    return c


# --------------------------------------------------------------------------------- models
# per width: heads, kv heads, head size, feed-forward, window, pooled block, scan state, step-size rank, decay rank
DESIGN_SIZES = {2048: (32, 4, 64, 5632, 512, 64, 16, 128, 64), 4096: (32, 8, 128, 14336, 1024, 64, 16, 256, 64)}
VOCAB = 32000


def _raw(case):
    """The configuration as config.json holds it."""
    if case["design"] == "llama":
        return dict(NAMED_SIZES[case["sizes"]], num_hidden_layers=case["layers"])
    width = case["sizes"]
    nh, nkv, hd, ff, window, pool, state, dt_rank, rank = DESIGN_SIZES[width]
    layers = []
    if case["design"] == "kasuvik":
        left = {"heads": nh, "kv_heads": nkv, "dim": hd, "vdim": hd, "conv": 4, "rot": {"dims": hd, "base": 10000.0},
                "scale": hd ** -0.5, "mask": {"size": window, "pool": pool}}
        right = {"inner": 2 * width, "state": state, "dt_rank": dt_rank, "conv": 4}
        for i in range(case["layers"]):
            mixer = {"heads": nh, "dim": hd, "rank": rank} if i % 4 == 1 else {"left": left, "right": right}
            layers.append({"type": "general_delta" if i % 4 == 1 else "parallel", "mixer": mixer, "mlp": {"kind": "dense", "ff": ff}})
        return {"architecture": "Kasuvik", "vocab": VOCAB, "width": width, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-6}, "layers": layers}
    mlp = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 8, "top": 2}, "shared": {"ff": ff // 2}}
    attention = {"heads": nh, "kv_heads": nkv, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "softcap": 50.0, "v_mix": True,
                 "mask": {"size": window, "keep_first": 4},
                 "rot": {"dims": hd, "base": 500000.0, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    memory = {"heads": nh, "dim": hd, "vdim": hd, "gate_cap": 15.0}
    for i in range(case["layers"]):
        layers.append({"type": "mlstm" if i % 4 == 2 else "attention", "mixer": memory if i % 4 == 2 else attention, "mlp": mlp})
    return {"architecture": "Fisesun", "vocab": VOCAB, "width": width, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-6},
            "logit_softcap": 30.0, "layers": layers}


def _model(case):
    raw = _raw(case)
    name, kind = {"llama": ("LlamaForCausalLM", LlamaConfig), "kasuvik": ("Kasuvik", KasuvikConfig),
                  "fisesun": ("Fisesun", FisesunConfig)}[case["design"]]
    return raw, name, kind.from_dict(raw)


def _vocab(raw):
    return raw["vocab"] if "vocab" in raw else raw["vocab_size"]


def _successors(raw):
    """The order of the head's rows: the token that follows each token."""
    return np.random.RandomState(11).permutation(_vocab(raw))


_EMBED, _HEAD = ("embed", "model.embed_tokens.weight"), ("head", "lm_head.weight")
_EMBED_STD = {"llama-3-8b": 4.0}      # the layers of the wide model add more to the stream


def _weights(case, raw, arch, cfg):
    """Tensors by their checkpoint names, the same for every seed: a program's weights stay when its inputs change.
    Matrices N(0, 0.02) as in bench.py, norm weights around 1, the scans' and gates' own vectors as such layers start."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(5)
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    std = _EMBED_STD.get(case["sizes"], 1.0)
    tied = bool(raw.get("tie_word_embeddings"))
    out = {}

    def normal(shape, scale):
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32).mul_(scale)

    for name, (shape, role) in sorted(expected_tensors(arch, cfg).items()):
        last = name.split("mix.")[-1]
        if role == "index":                      # rows of two different experts
            n = 8
            one = torch.randint(0, n, (shape[0], 1), generator=gen, device=dev)
            more = torch.randint(1, n, (shape[0], 1), generator=gen, device=dev)
            out[name] = torch.cat([one, (one + more) % n], 1).to(torch.int32).contiguous()
            continue
        if name in _HEAD:
            continue
        if name in _EMBED:
            t = normal(shape, 0.02 if tied else std)
        elif name.endswith("A_log"):
            t = torch.log(torch.arange(1, shape[1] + 1, device=dev, dtype=torch.float32)).repeat(shape[0], 1)
        elif name.endswith("conv"):
            t = normal(shape, 0.4)
        elif name.endswith("dt.b"):
            t = normal(shape, 1.0) - 3.5
        elif last == "f.b":
            t = torch.linspace(3.0, 6.0, shape[0], device=dev)
        elif last == "i.b":
            t = normal(shape, 0.1) - 1.0
        elif last == "w0":
            t = normal(shape, 1.0) - 2.0
        elif name.endswith("vmix"):
            t = torch.full(shape, 0.5, device=dev)
        elif name.endswith(".b"):
            t = normal(shape, 0.1)
        elif role == "vector":
            t = normal(shape, 0.1) + 1.0
        else:
            t = normal(shape, 0.02)
        out[name] = t.to(dtype)
    if not tied:
        e, h = (_EMBED[0], _HEAD[0]) if _EMBED[0] in out else (_EMBED[1], _HEAD[1])
        head = torch.empty_like(out[e])
        head[torch.from_numpy(_successors(raw)).to(dev)] = (out[e].float() * (0.02 / std)).to(dtype)
        out[h] = head
    return out


def _requests(case, raw, seed):
    """-> ([prompt token ids], [tokens to generate]) of one pass."""
    rng = np.random.RandomState(seed % (1 << 31))
    n = case["requests"]
    sizes = np.random.RandomState(3 + n)      # lengths are the case's, ids the seed's
    lengths = [case["prompt"]] * n
    if case["spread"]:
        top = 2.5 * case["prompt"]
        lengths = [max(1, int(min(top, case["prompt"] * math.exp(case["spread"] * z)))) for z in sizes.standard_normal(n)]
        if not case["chunk"]:
            lengths[0] = case["prompt"]
    new = [case["new"]] * n
    if case["chunk"]:
        new = [max(1, int(case["new"] * u)) for u in sizes.uniform(0.25, 0.5, n)]
        new[-1] = case["new"]
    prompts = [rng.randint(0, _vocab(raw), size=k).tolist() for k in lengths]
    return prompts, new


class State:
    """What a user's program holds: an engine with its weights and pool, and the next requests."""

    def __init__(self, engine, prompts, new):
        self.engine, self.prompts, self.new = engine, prompts, new


def prepare(case, seed):
    raw, arch, cfg = _model(case)
    prompts, new = _requests(case, raw, seed)
    longest = max(len(p) + n for p, n in zip(prompts, new))
    limit = -(-(longest + 1) // 64) * 64
    blocks = sum(-(-(len(p) + n + 1) // 16) + 1 for p, n in zip(prompts, new)) + 16
    total = sum(len(p) for p in prompts)
    budget = STEP_TOKENS if case["chunk"] else max(total, 64)
    engine = kvcm_amd.Engine(
        config=kvcm_amd.EngineConfig(block_size=16, max_seq_len=limit, num_blocks=blocks, watermark_blocks=0,
                                     max_num_seqs=max(8, case["requests"]), max_batched_tokens=budget, prefill_chunk=case["chunk"],
                                     max_logit_rows=64, dtype=case["dtype"], beyond_max_position=True),
        architecture=arch, model_config=cfg, tensors=_weights(case, raw, arch, cfg))
    return State(engine, prompts, new)


def run(state):
    eng = state.engine
    ids = [eng.add_request(p, n) for p, n in zip(state.prompts, state.new)]
    done, last = {}, []
    while not eng.idle():
        eng.step()
        last = eng.take_finished()
        for f in last:
            done[f.id] = f.generated
    # the logits of the last step lie in the engine's own buffer
    logits = eng.runner.workspace.get("logits", (len(last), eng.model.spec.vocab_size), torch.float32)
    return {"tokens": [np.asarray(done[i], dtype=np.int64) for i in ids] if len(ids) <= 32
            else np.asarray([done[i] for i in ids], dtype=np.int64), "logits": logits}


# ------------------------------------------------------------------------------------ cost
def work(case):
    """Bytes and operations of one pass: every step that waits for the one before it reads the weights it uses once, every
    generated token reads its context's keys and values (or states) once; products, scores and recurrences."""
    raw, arch, cfg = _model(case)
    prompts, new = _requests(case, raw, 0)
    item = 2 if case["dtype"] == "bfloat16" else 4
    vocab = _vocab(raw)
    tokens = sum(len(p) + n - 1 for p, n in zip(prompts, new))
    steps = max(new)
    rows = sum(new) / steps                                     # of a decode step, in the mean
    width = raw.get("width") or raw["hidden_size"]
    total = active = 0.0
    for name, (shape, role) in expected_tensors(arch, cfg).items():
        n = float(np.prod(shape)) if len(shape) else 1.0
        if role in ("table", "index"):
            continue
        if ".mlp.e" in name:
            total += n * min(1.0, 1.0 - (1.0 - 0.25) ** rows)       # of the experts, those that some row uses
            active += n * 0.25
        else:
            total += n
            active += n if role == "matrix" else 0.0
    read = steps * (total + vocab * width) * item + tokens * width * item
    flops = 2.0 * active * tokens + 2.0 * vocab * width * sum(new)
    for p, n in zip(prompts, new):
        for kind, kv, heads, dims, window in _mixers(raw):
            if kind == "attention":
                seen = [min(t, window) if window else t for t in (len(p), len(p) + n)]
                pairs = len(p) * (seen[0] if window and len(p) > window else len(p) / 2.0) + (n - 1) * (seen[0] + seen[1]) / 2.0
                flops += 4.0 * heads * dims * pairs
                read += 2 * kv * dims * item * ((n - 1) * (seen[0] + seen[1]) / 2.0 + len(p) + n)
            else:                                               # a state of heads x dims x kv numbers per request, in 32 bits
                flops += 6.0 * heads * dims * kv * (len(p) + n - 1)
                read += 2 * 4 * heads * dims * kv * n
    return {"bytes": read + sum(new) * 4 + vocab * 4 * case["requests"], "flops": flops}


def _mixers(raw):
    """(kind, kv heads or state columns, heads, dims, window) of every mixer."""
    if "layers" not in raw:
        hd = raw["head_dim"]
        return [("attention", raw["num_key_value_heads"], raw["num_attention_heads"], hd, 0)] * raw["num_hidden_layers"]
    out = []
    for layer in raw["layers"]:
        m = layer["mixer"]
        if layer["type"] == "parallel":
            l, r = m["left"], m["right"]
            out += [("attention", l["kv_heads"], l["heads"], l["dim"], l["mask"]["size"]), ("state", r["state"], 1, r["inner"], 0)]
        elif layer["type"] == "attention":
            out.append(("attention", m["kv_heads"], m["heads"], m["dim"], m["mask"]["size"]))
        else:
            out.append(("state", m["dim"], m["heads"], m["dim"], 0))
    return out


def tolerance(case):
    # Logits against the 64-bit values, measured: 32-bit storage 2e-7 (two layers) to 6e-6 (22 layers); bfloat16 storage
    # 0.013 to 0.017 (22 and 32 layers), 0.006 to 0.008 (the designs of four layers).  Up to four times that between two
    # correct ways, and five standard deviations of it at a single logit; tokens are the same.
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.0}
    return {"rel": 0.03, "max": 0.3, "differ": 0.0}


# ------------------------------------------------------------------------- 64-bit reference
# Sequences of different lengths are padded at their ends: everything here looks back only, so no real token sees a
# padding token.
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


class _Tensors:
    """A checkpoint's tensors in 64 bits, widened one at a time as they are asked for."""

    def __init__(self, tensors):
        self.tensors = tensors

    def __getitem__(self, name):
        t = self.tensors[name]
        return t if t.dtype == torch.int32 else t.double()

    def mul(self, x, name):
        return x @ self[name].t()


def _turn(x, freqs, pairs):
    """x [B, T, heads, d]: pairs (2i, 2i + 1), or (i, i + d/2), turned by position * freqs[i]."""
    a = torch.arange(x.shape[1], device=x.device, dtype=torch.float64)[:, None] * freqs[None, :]
    c, s = a.cos()[None, :, None, :], a.sin()[None, :, None, :]
    half = x.shape[-1] // 2
    u, v = (x[..., 0::2], x[..., 1::2]) if pairs else (x[..., :half], x[..., half:])
    one, two = u * c - v * s, v * c + u * s
    return torch.stack([one, two], -1).flatten(-2) if pairs else torch.cat([one, two], -1)


def _attend(q, k, v, scale, mask, cap=0.0):
    """q [B, T, H, d], k, v [B, K, G, d], mask [T, K] -> [B, T, H * d]; one sequence at a time."""
    H, G = q.shape[2], k.shape[2]
    out = []
    for b in range(q.shape[0]):
        one = []
        for g in range(G):
            z = torch.matmul(q[b, :, g * (H // G):(g + 1) * (H // G)].transpose(0, 1), k[b, :, g].t().contiguous()) * scale
            if cap:
                z = cap * torch.tanh(z / cap)
            p = torch.softmax(z.masked_fill(~mask, -math.inf), -1)
            one.append(torch.matmul(p, v[b, :, g].contiguous()))
        out.append(torch.cat(one, 0).transpose(0, 1).flatten(1))
    return torch.stack(out)


def _causal(T, device):
    i = torch.arange(T, device=device)
    return i[:, None] - i[None, :]


def _llama(raw, w, x):
    B, T, _ = x.shape
    H, G, d, eps = raw["num_attention_heads"], raw["num_key_value_heads"], raw["head_dim"], raw["rms_norm_eps"]
    freqs = raw["rope_theta"] ** (-torch.arange(0, d, 2, device=x.device, dtype=torch.float64) / d)
    mask = _causal(T, x.device) >= 0
    for i in range(raw["num_hidden_layers"]):
        p = "model.layers.%d." % i
        h = _rms(x, eps) * w[p + "input_layernorm.weight"]
        q, k, v = (w.mul(h, p + "self_attn.%s_proj.weight" % n).view(B, T, -1, d) for n in "qkv")
        o = _attend(_turn(q, freqs, False), _turn(k, freqs, False), v, d ** -0.5, mask)
        x = x + w.mul(o, p + "self_attn.o_proj.weight")
        h = _rms(x, eps) * w[p + "post_attention_layernorm.weight"]
        x = x + w.mul(_silu(w.mul(h, p + "mlp.gate_proj.weight")) * w.mul(h, p + "mlp.up_proj.weight"), p + "mlp.down_proj.weight")
    return _rms(x, eps) * w["model.norm.weight"]


def _conv(u, weight):
    """Causal over time per channel: u [B, T, C], weight [C, taps], the last tap on the current token."""
    taps = weight.shape[1]
    padded = torch.cat([u.new_zeros(u.shape[0], taps - 1, u.shape[2]), u], 1)
    return sum(padded[:, j:j + u.shape[1]] * weight[:, j] for j in range(taps))


def _window_pool(h, w, p, m):
    B, T, _ = h.shape
    H, G, d, window, pool = m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"], m["mask"]["pool"]
    q, k, v = (_conv(w.mul(h, p + n) + w[p + n + ".b"], w[p + n + ".conv"]).view(B, T, -1, d) for n in "qkv")
    freqs = m["rot"]["base"] ** (-torch.arange(0, d, 2, device=h.device, dtype=torch.float64) / d)
    q, k = _turn(q, freqs, True) * w[p + "temp"][:, None], _turn(k, freqs, True)
    n = T // pool
    far = _causal(T, h.device)
    mask = (far >= 0) & (far < window)
    if n:
        blocks = [t[:, :n * pool].reshape(B, n, pool, G, d).mean(2) for t in (k, v)]
        k, v = torch.cat([blocks[0], k], 1), torch.cat([blocks[1], v], 1)
        ends = torch.arange(n, device=h.device) * pool + pool - 1
        mask = torch.cat([ends[None, :] <= torch.arange(T, device=h.device)[:, None] - window, mask], 1)
    return w.mul(_attend(q, k, v, m["scale"], mask), p + "o")


def _scan(h, w, p, m):
    inner, n, r = m["inner"], m["state"], m["dt_rank"]
    x, z = w.mul(h, p + "in").split(inner, -1)
    x = _silu(_conv(x, w[p + "conv"]) + w[p + "conv.b"])
    dt, Bm, Cm = w.mul(x, p + "x").split([r, n, n], -1)
    dt = torch.nn.functional.softplus(w.mul(dt, p + "dt") + w[p + "dt.b"], threshold=1e9)
    A, D = -torch.exp(w[p + "A_log"]), w[p + "D"]
    S, y = h.new_zeros(h.shape[0], inner, n), torch.empty_like(x)
    for t in range(h.shape[1]):
        S = torch.exp(dt[:, t, :, None] * A) * S + (dt[:, t] * x[:, t])[..., None] * Bm[:, t, None, :]
        y[:, t] = (S * Cm[:, t, None, :]).sum(-1) + D * x[:, t]
    return w.mul(y * _silu(z), p + "o")


def _delta(h, w, p, m, eps):
    B, T, _ = h.shape
    H, d = m["heads"], m["dim"]
    r, k, v = (w.mul(h, p + n).view(B, T, H, d) for n in "rkv")
    decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(w.mul(torch.tanh(w.mul(h, p + "w1")), p + "w2") + w[p + "w0"])).view(B, T, H, d)
    a = torch.sigmoid(w.mul(h, p + "a") + w[p + "a.b"]).view(B, T, H, d)
    u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    S, o = h.new_zeros(B, H, d, d), torch.empty_like(v)
    for t in range(T):
        S = decay[:, t, :, :, None] * S - (a[:, t] * u[:, t])[..., None] * (u[:, t, :, :, None] * S).sum(2, keepdim=True) \
            + k[:, t, :, :, None] * v[:, t, :, None, :]
        o[:, t] = (S * r[:, t, :, :, None]).sum(2)
    return w.mul(_rms(o, eps).flatten(2) * w[p + "norm"] * torch.sigmoid(w.mul(h, p + "g")), p + "o")


def _kasuvik(raw, w, x):
    eps = raw["norm"]["eps"]
    for i, layer in enumerate(raw["layers"]):
        p, m = "l%d." % i, layer["mixer"]
        h = _rms(x, eps) * w[p + "norm1"]
        if layer["type"] == "parallel":
            y = 0.5 * (_rms(_window_pool(h, w, p + "mix.left.", m["left"]), eps) * w[p + "mix.left.out"]
                       + _rms(_scan(h, w, p + "mix.right.", m["right"]), eps) * w[p + "mix.right.out"])
        else:
            y = _delta(h, w, p + "mix.", m, eps)
        x = x + _rms(y, eps) * w[p + "norm1b"]
        h = _rms(x, eps) * w[p + "norm2"]
        f = w.mul(torch.relu(w.mul(h, p + "mlp.gate")) * w.mul(h, p + "mlp.up"), p + "mlp.down")
        x = x + _rms(f, eps) * w[p + "norm2b"]
    return _rms(x, eps) * w["final.norm"]


def _capped_attention(h, w, p, m, eps, first):
    B, T, _ = h.shape
    d, rot = m["dim"], m["rot"]
    q, k = ((_rms(w.mul(h, p + n), eps) * w[p + n + ".norm"]).view(B, T, -1, d) for n in "qk")
    own = w.mul(h, p + "v")
    mix = w[p + "vmix"] if first is not None else 0.0
    v = own if first is None else (1.0 - mix) * own + mix * first
    f = rot["base"] ** (-torch.arange(0, d, 2, device=h.device, dtype=torch.float64) / d)
    s = rot["scaling"]
    length = 2 * math.pi / f
    share = ((s["original"] / length - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
    f = (1.0 - share) * f / s["factor"] + share * f
    far = _causal(T, h.device)
    mask = (far >= 0) & ((far < m["mask"]["size"]) | (torch.arange(T, device=h.device)[None, :] < m["mask"]["keep_first"]))
    o = _attend(_turn(q, f, False), _turn(k, f, False), v.view(B, T, -1, d), m["scale"], mask, m["softcap"])
    return w.mul(o, p + "o"), own


def _memory(h, w, p, m, eps):
    B, T, _ = h.shape
    H, d, cap = m["heads"], m["dim"], m["gate_cap"]
    q, k, v = (w.mul(h, p + n).view(B, T, H, d) for n in "qkv")
    q = q * d ** -0.5
    take_log = cap * torch.tanh((w.mul(h, p + "i") + w[p + "i.b"]) / cap)
    keep_log = torch.nn.functional.logsigmoid(cap * torch.tanh((w.mul(h, p + "f") + w[p + "f.b"]) / cap))
    S, n, top, o = h.new_zeros(B, H, d, d), h.new_zeros(B, H, d), h.new_zeros(B, H), torch.empty_like(v)
    for t in range(T):
        high = torch.maximum(keep_log[:, t] + top, take_log[:, t])
        keep, take = torch.exp(keep_log[:, t] + top - high), torch.exp(take_log[:, t] - high)
        S = keep[..., None, None] * S + take[..., None, None] * k[:, t, :, :, None] * v[:, t, :, None, :]
        n = keep[..., None] * n + take[..., None] * k[:, t]
        top = high
        under = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
        o[:, t] = (S * q[:, t, :, :, None]).sum(2) / under[..., None]
    return w.mul(_rms(o, eps).flatten(2) * w[p + "norm"] * torch.sigmoid(w.mul(h, p + "g")), p + "o")


def _fisesun(raw, w, x, tokens):
    eps, first = raw["norm"]["eps"], None

    def gated(h, p):
        return w.mul(_silu(w.mul(h, p + "gate")) * w.mul(h, p + "up"), p + "down")

    for i, layer in enumerate(raw["layers"]):
        p, m = "l%d." % i, layer["mixer"]
        if layer["type"] == "attention":
            y, own = _capped_attention(x, w, p + "mix.", m, eps, first)
            first = own if first is None else first
        else:
            y = _memory(x, w, p + "mix.", m, eps)
        x = x + _rms(y, eps) * w[p + "norm1"]
        chosen = w[p + "mlp.table"][tokens].long()              # [B, T, top]
        f = gated(x, p + "mlp.shared.")
        for e in range(layer["mlp"]["router"]["experts"]):
            at = (chosen == e).any(-1)
            f[at] += gated(x[at], p + "mlp.e%d." % e) / chosen.shape[-1]
        x = x + _rms(f, eps) * w[p + "norm2"]
    return _rms(x, eps) * w["final.norm"]


def _hidden(case, raw, w, tokens):
    """Rows before the output head [B, T, width] of tokens [B, T]."""
    tokens = tokens.to("cuda:0")
    x = w.tensors[_EMBED[0] if _EMBED[0] in w.tensors else _EMBED[1]][tokens].double()
    if case["design"] == "llama":
        return _llama(raw, w, x)
    return _kasuvik(raw, w, x) if case["design"] == "kasuvik" else _fisesun(raw, w, x, tokens)


def exact(case, seed):
    """Greedy decoding in 64 bits: the whole sequences are run with the tokens that follow by the head's order, and again
    with what they gave where that was another, until they agree."""
    raw, arch, cfg = _model(case)
    prompts, new = _requests(case, raw, seed)
    w = _Tensors(_weights(case, raw, arch, cfg))
    after = _successors(raw)
    tied = bool(raw.get("tie_word_embeddings"))
    head = w[next(n for n in ((_EMBED if tied else _HEAD)) if n in w.tensors)].t()
    generated = []
    for p, n in zip(prompts, new):
        g = [p[-1]]
        for _ in range(n):
            g.append(g[-1] if tied else int(after[g[-1]]))
        generated.append(g[1:])
    logits = None
    group = max(1, 24576 // max(len(p) + n for p, n in zip(prompts, new)))
    for lo in range(0, len(prompts), group):
        at = range(lo, min(len(prompts), lo + group))
        longest = max(len(prompts[i]) + new[i] - 1 for i in at)
        for _ in range(1 + max(new)):
            seqs = torch.zeros(len(at), longest, dtype=torch.long)
            for r, i in enumerate(at):
                s = prompts[i] + generated[i][:-1]
                seqs[r, :len(s)] = torch.tensor(s)
            x = _hidden(case, raw, w, seqs)
            agreed, ends = True, []
            for r, i in enumerate(at):
                z = x[r, len(prompts[i]) - 1:len(prompts[i]) + new[i] - 1] @ head
                if raw.get("logit_softcap"):
                    z = raw["logit_softcap"] * torch.tanh(z / raw["logit_softcap"])
                got = z.argmax(-1).tolist()
                agreed, generated[i] = agreed and got == generated[i], got
                ends.append(z[-1])
            if agreed:
                break
        ends = torch.stack(ends)
        logits = ends if logits is None else torch.cat([logits, ends])
    if case["chunk"]:
        logits = logits[-1:]
    tokens = [np.asarray(g, dtype=np.int64) for g in generated]
    return {"tokens": tokens if len(tokens) <= 32 else np.asarray(tokens), "logits": logits}
