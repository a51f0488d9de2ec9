"""The parts a Llama-style decoder is made of: RMS norm, rotary positions, grouped-query attention
over the paged cache, SwiGLU feed-forward, token embedding, output head, and the pre-norm residual
arrangement.  Formulas and rounding points follow the reference step (src/model/llama.cpp:84-128)
and its kernels (src/cuda/kernels.cu, src/cuda/paged_attention.cu); every size and constant is a
parameter.
"""
import math

import torch

from ..registry import BLOCKS, EMBEDDINGS, FEED_FORWARDS, HEADS, MIXERS, NORMS, POSITIONS
from . import paged_attention
from .base import (Block, Embedding, FeedForward, Head, KVCacheNeed, Mixer, Norm, ParamSpec, PositionEncoding, as_tensor, said_with)


def _linear(ctx, step, x, w, name, keep_partial=False, dtype=None):
    """x @ w^T into the work buffer ``name``.  With ``keep_partial`` the result may come back as
    un-added split-K sums (ops.PartialSums) for a consumer that adds them up itself."""
    out = step.ws(name, (x.shape[0], w.shape[0]), dtype)
    scratch = step.scratch(name, x.shape[0], w.shape[0], w.shape[1])
    return ctx.ops.gemm(x, w, out, scratch=scratch, keep_partial=keep_partial and scratch is not None,
                        tuning=step.tune_products, unsplit=True)


def linear_pair(ctx, step, first, second):
    """Two products that do not wait for one another, each (x, w, name, dtype) of ``_linear``: in one launch where they are of few rows."""
    ops = ctx.ops
    if step.rows <= ops.FUSED_NORM_MAX_ROWS:
        outs = [step.ws(name, (x.shape[0], w.shape[0]), dtype) for x, w, name, dtype in (first, second)]
        splits = [step.scratch(name, x.shape[0], *w.shape) is not None for x, w, name, _ in (first, second)]
        if ops.gemm_pair(*first[:2], outs[0], *second[:2], outs[1], *splits):
            return outs
    return [_linear(ctx, step, x, w, name, dtype=dtype) for x, w, name, dtype in (first, second)]


# A mixer that has ``stages(step, h)`` runs as a generator: it yields its larger products, (x, w, name, dtype) of ``_linear``, takes their results
# and returns its output, so that two mixers on one input can run in step.  ``buffers``: what its work buffers' names begin with; in step
# only with a mixer of other names.
def run_stages(ctx, step, stages):
    try:
        product = next(stages)
        while True:
            x, w, name, dtype = product
            product = stages.send(_linear(ctx, step, x, w, name, dtype=dtype))
    except StopIteration as end:
        return end.value


def side_by_side(ctx, step, left, right):
    """Two mixers' stages in step: the first products of both together, then what follows each, and so on.  -> both outputs.  Steps of more rows than
    share launches run one after the other: what a product leaves is then read before the other mixer's rows push it out of the caches (a prompt of
    2,048 rows 2.91 / 2.86 ms)."""
    if step.rows > ctx.ops.FUSED_NORM_MAX_ROWS:
        return [run_stages(ctx, step, left), run_stages(ctx, step, right)]
    both, asked, outputs = [left, right], [None, None], [None, None]

    def go(i, result):
        try:
            asked[i] = both[i].send(result)
        except StopIteration as end:
            asked[i], outputs[i] = None, end.value

    go(0, None)
    go(1, None)
    while asked[0] is not None or asked[1] is not None:
        if asked[0] is not None and asked[1] is not None:
            results = linear_pair(ctx, step, *asked)
        else:
            results = [q and _linear(ctx, step, *q[:3], dtype=q[3]) for q in asked]
        waits = [q is not None for q in asked]
        for i in (0, 1):
            if waits[i]:
                go(i, results[i])
    return outputs


def _to_residual(ctx, step, x, w, name, defer=False):
    """A part's last product, whose result goes to the residual stream.  For decode steps of a few
    rows it is handed on unrun (ops.PendingProduct): the norm that follows runs it with the addition
    and its own preparation in the epilogue.  Otherwise it runs here, split sums left un-added.  ``defer``: the
    caller takes it unrun in 32 bits too."""
    ops = ctx.ops
    if (step.fold_norms and x.dtype == torch.bfloat16 and x.shape[0] <= min(ops.FUSED_NORM_MAX_ROWS, step.fold_rows)
            and ops.gemm8_supported(x.shape[0], w.shape[0], w.shape[1])):
        out = step.ws(name, (x.shape[0], w.shape[0]))
        return ops.PendingProduct(x, w, out, step.scratch(name, x.shape[0], w.shape[0], w.shape[1]))
    if defer and step.fold_norms and x.dtype == torch.float32 and ops.f32_few_takes(x.shape[0], w.shape[1]):
        return ops.PendingProduct(x, w, step.ws(name, (x.shape[0], w.shape[0])))
    return _linear(ctx, step, x, w, name, keep_partial=True)


@NORMS.register("rmsnorm")
class RMSNorm(Norm):
    """out = weight * round(x / sqrt(mean(x^2) + eps)); eps inside the root, no mean removed, the
    weight a plain multiplier (src/cuda/kernels.cu:34-49).  params: size, eps."""

    capturable = True
    accepts_partial_sums = True
    defers = True

    def param_specs(self):
        return [ParamSpec("weight", ((self.prefix + "weight", (self.params["size"],)),), role="vector")]

    def bind(self, tensors):
        super().bind(tensors)
        # where the folded form of this norm leaves its rows (ops.NormedRows), kept for good: recorded
        # steps hold the addresses
        H, ops = self.params["size"], self.ctx.ops
        self._folded = None
        if ops is not None and self.ctx.dtype == torch.bfloat16 and H % 8 == 0 and self.ctx.device.type == "cuda":
            self._folded = (torch.empty(ops.FUSED_NORM_MAX_ROWS, H, dtype=torch.bfloat16, device=self.ctx.device),
                            torch.empty(ops.FUSED_NORM_MAX_ROWS, H // 8, dtype=torch.float32, device=self.ctx.device))

    def forward(self, x, out, add=None, rows=None, defer=False):
        ops = self.ctx.ops
        if defer == "rows" and rows is None and (add is None or isinstance(add, ops.PendingProduct)) and ops.can_norm_rows(x, self.w["weight"], out):
            if add is not None:
                ops.gemm_residual(add, x)
            return ops.RowsToNorm(x, self.w["weight"], self.params["eps"], out)
        if isinstance(add, ops.PendingProduct):
            if (defer and rows is None and self._folded is not None and add.x.shape[0] == x.shape[0] <= ops.FUSED_NORM_MAX_ROWS
                    and add.dtype == torch.bfloat16):
                return ops.gemm_residual_norm(add, x, self.w["weight"], self.params["eps"], *self._folded, out)
            add = add.run(keep_partial=True)
        ops.rmsnorm(x, self.w["weight"], out, self.params["eps"], add=add, rows=rows)
        return out


@POSITIONS.register("rotary")
class Rotary(PositionEncoding):
    """Rotate-half rotary positions over the first ``dim`` (= head_dim) entries of every q and k
    head: pairs (j, j + dim/2), inv_freq_j = theta^(-2j/dim), angle = position * inv_freq_j in
    32-bit (src/cuda/kernels.cu:51-70).  params: theta, dim."""

    capturable = True
    accepts_partial_sums = True

    def __init__(self, params, prefix, ctx):
        super().__init__(params, prefix, ctx)
        dim = params["dim"]
        j = torch.arange(0, dim, 2, dtype=torch.float32)
        self.inv_freq = (1.0 / torch.pow(torch.tensor(float(params["theta"]), dtype=torch.float32), j / dim)).to(ctx.device)

    def ignorable_tensors(self):
        return (self.prefix + "rotary_emb.inv_freq",)

    def rotation_table(self, step, head_dim):
        """(cos, sin) of every row's angles [rows, head_dim/2, 2].  The angles depend on the row
        only: the first layer of a step computes them, the others with the same theta and dim read
        them.  Each (theta, dim) has a table and a work buffer of its own, so layers that alternate
        between two thetas do not overwrite each other's angles."""
        if head_dim != self.params["dim"]:
            return None
        theta = float(self.params["theta"])
        key = ("rotary", theta, head_dim)
        table = step.shared.get(key)
        if table is None:
            name = "rotary_cos_sin_%d_%s" % (head_dim, theta.hex())
            table = step.ws(name, (step.rows, head_dim), torch.float32).view(step.rows, head_dim // 2, 2)
            self.ctx.ops.rope_table(step.positions, self.inv_freq, table, rows=step.rows)
            step.shared[key] = table
        return table

    def apply(self, step, qkv, num_heads, num_kv_heads, head_dim, cache=None, slots=None, source=None):
        if head_dim != self.params["dim"]:
            raise ValueError("rotary: this kernel rotates the whole head (dim must equal head_dim)")
        k, v = cache if cache is not None else (None, None)
        table = self.rotation_table(step, head_dim)
        self.ctx.ops.rope_cache(qkv, num_heads, num_kv_heads, head_dim, positions=step.positions,
                                inv_freq=self.inv_freq, slots=slots, kcache=k, vcache=v,
                                block_size=self.ctx.block_size, rows=step.rows, source=source, cos_sin=table)
        return cache is not None


@POSITIONS.register("none")
class NoPosition(PositionEncoding):
    capturable = True
    rotates = False

    def apply(self, step, qkv, num_heads, num_kv_heads, head_dim, cache=None, slots=None):
        return False


@MIXERS.register("gqa_attention")
class GQAAttention(Mixer):
    """Grouped-query attention over the paged cache.  One fused projection [q | k | v]
    (src/model/llama.cpp:108), positions applied to q and k, k and v stored to the pages of this
    step's rows before attention reads them (llama.cpp:111-115), so a portion of a prompt attends
    to itself through the cache; causality is context length = position + 1.
    params: num_heads, num_kv_heads, head_dim, scale, window (0 = all keys), position (PartSpec)."""

    capturable = True
    accepts_normed_rows = accepts_rows_to_norm = True
    defers = True

    def sub_parts(self):
        return (self.position,)

    def __init__(self, params, prefix, ctx):
        super().__init__(params, prefix, ctx)
        p = params
        self.nh, self.nkv, self.hd = p["num_heads"], p["num_kv_heads"], p["head_dim"]
        # refused where the model is built, not at the first step's launch
        if self.hd <= 0 or self.hd % 8 or self.hd > 256:
            raise ValueError(f"gqa_attention {prefix!r}: head_dim {self.hd} is not supported (the attention kernels take "
                             f"multiples of 8 up to 256; num_heads {self.nh}, num_kv_heads {self.nkv})")
        if self.nkv <= 0 or self.nh % self.nkv:
            raise ValueError(f"gqa_attention {prefix!r}: num_heads {self.nh} is not a multiple of num_kv_heads {self.nkv}")
        self.scale = p.get("scale", 1.0 / math.sqrt(self.hd))
        self.window = p.get("window", 0)
        pos = p["position"]
        self.position = POSITIONS.get(pos.kind)(pos.params, prefix, ctx)
        self.q_dim, self.kv_dim = self.nh * self.hd, self.nkv * self.hd

    def param_specs(self):
        H, pre = self.ctx.hidden_size, self.prefix
        return [ParamSpec("wqkv", ((pre + "q_proj.weight", (self.q_dim, H)), (pre + "k_proj.weight", (self.kv_dim, H)),
                                   (pre + "v_proj.weight", (self.kv_dim, H)))),
                ParamSpec("wo", ((pre + "o_proj.weight", (H, self.q_dim)),))]

    def ignorable_tensors(self):
        return self.position.ignorable_tensors()

    def cache_need(self):
        return KVCacheNeed(self.nkv, self.hd, self.window)

    def flops(self, rows, attended=0):
        # the two projections, and q.k and p.v over every (row, key) pair of every query head
        return super().flops(rows) + 4.0 * attended * self.hd * self.nh

    def forward(self, step, h, defer=False):
        wo = self.w["wo"]
        parts = self._one_launch_parts(step, h) if defer else 0
        if not parts:
            return _to_residual(self.ctx, step, self._attention(step, h), wo, "mixer_out", defer)
        ops, g = self.ctx.ops, self.cache.group
        table = self.position.rotation_table(step, self.hd) if self.position.rotates else None
        return ops.PendingAttention(
            lambda: self._attention(step, h), h, self.w["wqkv"], step.ws("attn", (step.rows, self.q_dim)), wo,
            step.ws("mixer_out", (step.rows, wo.shape[0])), step.scratch("mixer_out", step.rows, wo.shape[0], wo.shape[1]),
            (self.cache.k(self.cache_index), self.cache.v(self.cache_index)), step.tables(g), step.table_stride(g), step.row_seq, step.ctx_lens,
            step.slots(g), table, (self.nh, self.nkv, self.hd), self.scale, parts,
            lambda: ops.decode_front_buffers(step, step.rows, self.nh, self.nkv, self.hd, parts))

    def _one_launch_parts(self, step, h):
        """How the step's attention half is cut where it can be one launch with the norm that follows (ops.PendingAttention), else 0."""
        ops = self.ctx.ops
        if not (step.fold_norms and step.max_run == 1 and step.attention_mode == "auto" and self.window == 0 and self.cache_owner
                and h.dtype == torch.bfloat16 and step.rows <= min(ops.FUSED_NORM_MAX_ROWS, step.fold_rows)):
            return 0
        if self.position.rotates and self.position.rotation_table(step, self.hd) is None:
            return 0
        return ops.decode_front_parts(step.rows, self.ctx.hidden_size, self.nh, self.nkv, self.hd, self.ctx.block_size, step.max_context_bound)

    def _attention(self, step, h):
        """The attention's rows, in the work buffer ``attn``."""
        ops = self.ctx.ops
        g = self.cache.group
        kc, vc = self.cache.k(self.cache_index), self.cache.v(self.cache_index)
        pos = self.position
        # (the rotation of many rows reads whole rows, eight entries a lane; that of slices a head at a time)
        res = _linear(self.ctx, step, h, self.w["wqkv"], "qkv", keep_partial=pos.accepts_partial_sums and not ops.many_rows(step.rows))
        qkv = step.ws("qkv", (step.rows, self.q_dim + 2 * self.kv_dim))
        slots = step.slots(g) if self.cache_owner else None
        attn = step.ws("attn", (step.rows, self.q_dim))
        # decode-shaped steps: rotation, page write and attention in one launch, where the position
        # encoding is a rotation by pairs (or none) and the step's shape has that kernel
        table = pos.rotation_table(step, self.hd) if pos.rotates else None
        if (table is not None or not pos.rotates) and paged_attention.attend_from_projection(
                step, ops, res, attn, kc, vc, g, self.nh, self.nkv, self.hd, self.scale, self.window, table, slots):
            return attn
        # 32-bit rows of different sequences: rotation, page write and attention in one launch, the same bits
        if (slots is not None and step.max_run == 1 and qkv.dtype == torch.float32
                and (table is not None and said_with(pos, "rotation_table", "apply") or not pos.rotates)
                and ops.attention_f32_decode_supported(self.nh, self.nkv, self.hd, self.ctx.block_size)):
            ops.attention_f32_decode(res, attn, kc, vc, step.tables(g), step.table_stride(g), step.row_seq, step.ctx_lens, self.nh, self.nkv, self.hd,
                                     self.scale, slots, cos_sin=table, window=self.window, rows=step.rows)
            return attn
        extra = {"source": res} if hasattr(res, "materialize") else {}
        stored = pos.apply(step, qkv, self.nh, self.nkv, self.hd,
                           cache=(kc, vc) if self.cache_owner else None, slots=slots, **extra)
        if self.cache_owner and not stored:
            ops.rope_cache(qkv, self.nh, self.nkv, self.hd, slots=slots, kcache=kc, vcache=vc,
                           block_size=self.ctx.block_size, rows=step.rows)
        paged_attention.attend(step, ops, qkv, attn, kc, vc, g, self.nh, self.nkv, self.hd, self.scale, self.window)
        return attn


@FEED_FORWARDS.register("swiglu")
class SwiGLU(FeedForward):
    """down( round(silu(gate(h))) * up(h) ) with gate and up as one fused projection
    (src/model/llama.cpp:119-122, src/cuda/kernels.cu:72-82).  params: intermediate_size."""

    capturable = True
    accepts_normed_rows = accepts_rows_to_norm = True
    defers = True

    def param_specs(self):
        H, I, pre = self.ctx.hidden_size, self.params["intermediate_size"], self.prefix
        return [ParamSpec("w_gate_up", ((pre + "gate_proj.weight", (I, H)), (pre + "up_proj.weight", (I, H)))),
                ParamSpec("w_down", ((pre + "down_proj.weight", (H, I)),))]

    def forward(self, step, h, defer=False):
        I = self.params["intermediate_size"]
        act = step.ws("act", (step.rows, I))
        if not self.ctx.ops.gemm_swiglu(h, self.w["w_gate_up"], act, tuning=step.tune_products):      # few rows: one launch
            h = as_tensor(h)
            if not self.ctx.ops.gemm_swiglu(h, self.w["w_gate_up"], act, tuning=step.tune_products):
                gu = _linear(self.ctx, step, h, self.w["w_gate_up"], "gate_up")
                self.ctx.ops.swiglu(gu, act)
        return _to_residual(self.ctx, step, act, self.w["w_down"], "ffn_out", defer)


@EMBEDDINGS.register("token_embedding")
class TokenEmbedding(Embedding):
    """x = float(table[token]); nothing scaled or added (src/cuda/kernels.cu:27-32).
    params: vocab_size."""

    capturable = True

    def param_specs(self):
        return [ParamSpec("table", ((self.prefix + "weight", (self.params["vocab_size"], self.ctx.hidden_size)),),
                          role="table")]

    def forward(self, step, out):
        self.ctx.ops.embed(step.tokens, self.w["table"], out)
        return out

    def bytes_read(self, rows):
        table = self.w["table"]
        return rows * table.shape[1] * table.element_size()      # only the rows of the step's tokens

    def flops(self, rows, attended=0):
        return 0.0


@HEADS.register("linear_head")
class LinearHead(Head):
    """logits = h @ table^T in 32-bit, only for the rows that are asked for
    (src/model/llama.cpp:126-128).  params: vocab_size, tied (use the embedding's table), scale (a factor on the
    logits, default 1: applied to the 32-bit logits), softcap (c > 0: logits <- c tanh(logits / c) after the factor;
    default none)."""

    capturable = True

    def _name(self):
        return self.params.get("name", self.prefix + "weight")      # name: the table's checkpoint name

    def param_specs(self):
        if self.params.get("tied"):
            return []
        return [ParamSpec("table", ((self._name(), (self.params["vocab_size"], self.ctx.hidden_size)),), role="table")]

    def ignorable_tensors(self):
        # a tied checkpoint may still carry a copy of the shared table
        return (self._name(),) if self.params.get("tied") else ()

    def forward(self, step, h, out):
        self.ctx.ops.gemm(h, self.w["table"], out, tuning=step.tune_products, unsplit=True)
        if float(self.params.get("scale", 1.0)) != 1.0:
            self.ctx.ops.scale_rows(out, self.params["scale"])
        if float(self.params.get("softcap") or 0.0) > 0.0:
            self.ctx.ops.softcap_rows(out, self.params["softcap"])
        return out


@BLOCKS.register("prenorm_residual")
class PreNormResidual(Block):
    """x += mixer(norm_mixer(x)); x += ffn(norm_ffn(x))  (src/model/llama.cpp:104-124).  Each
    addition is done by the norm that follows it."""

    capturable = True

    def forward(self, step, x, pending):
        buf = step.ws("normed", (step.rows, x.shape[1]))
        n1, n2 = self.parts["norm_mixer"], self.parts["norm_ffn"]
        mixer, ffn = self.parts["mixer"], self.parts["ffn"]
        # a norm may leave its scale to the product that follows (Norm.defers) where that part takes it
        fold1, fold2 = ({"defer": "rows" if part.accepts_rows_to_norm and said_with(part, "accepts_rows_to_norm", "forward") else True}
                        if (step.fold_norms and norm.defers and part.accepts_normed_rows) else {} for norm, part in ((n1, mixer), (n2, ffn)))
        h = n1.forward(x, buf, add=pending if n1.accepts_partial_sums else as_tensor(pending), **fold1)
        # a mixer may leave all of its launches to the norm behind it (Mixer.defers), which runs at once
        late = {"defer": True} if (n2.defers and n2.accepts_partial_sums and mixer.defers and fold2 and said_with(mixer, "defers", "forward")) else {}
        a = mixer.forward(step, buf if h is None else h, **late)
        h = n2.forward(x, buf, add=a if n2.accepts_partial_sums else as_tensor(a), **fold2)
        return ffn.forward(step, buf if h is None else h, **({"defer": True} if fold2 and ffn.defers and said_with(ffn, "defers", "forward") else {}))
