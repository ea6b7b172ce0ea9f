"""Runs of plain decoder layers whose few-row steps are launched by one native call, or are one launch."""
import torch

from ..ops import attention_bf16 as A
from ..ops import few_row_layers as F
from ..ops import resident_layers as R
from ..ops.linear import HalfNormed
from .attention import Attention
from .block import PreNormBlock
from .feed_forward import GatedFeedForward
from .norm import RMSNorm, ScalarRMSNorm
from .position import RotaryPosition


def _plain_layer(block) -> bool:
    """Pre-norm attention with interleaved rotation, then a gated feed-forward, root-mean-square norms before
    both: the layers whose few-row steps ops.few_row_layers launches.  Exactly these classes: the call takes their
    weights and never asks their ``forward``, which a class derived from one may have replaced."""
    if type(block) is not PreNormBlock or type(block.mixer) is not Attention \
            or type(block.feed_forward) is not GatedFeedForward:
        return False
    f, p = block.feed_forward.spec, block.mixer.position
    norms = (RMSNorm, ScalarRMSNorm)                     # both hold a float32 weight per column
    return (type(block.mixer_norm) in norms and type(block.feed_forward_norm) in norms and not _own_forward(block)
            and type(p) is RotaryPosition and p.spec.layout == "interleaved"
            and f.activation in F.GATE_MODES and f.limit is None)


def _own_forward(block) -> bool:
    """A ``forward`` put on the object itself, over its class's."""
    return ("forward" in block.__dict__ or "forward" in block.mixer.__dict__ or "forward" in block.feed_forward.__dict__
            or "forward" in block.mixer_norm.__dict__ or "forward" in block.feed_forward_norm.__dict__)


def _parts(block):
    return (block, block.mixer, block.mixer.position, block.feed_forward, block.mixer_norm, block.feed_forward_norm)


def _alike(a, b) -> bool:
    return (a.mixer.spec == b.mixer.spec and a.feed_forward.spec == b.feed_forward.spec
            and a.mixer_norm.spec.eps == b.mixer_norm.spec.eps
            and a.feed_forward_norm.spec.eps == b.feed_forward_norm.spec.eps)


class FewRowRuns:
    """For every run of a plan's order, where the plain layers of one shape that begin with it end.  None
    (bfloat16) where the layer behind them would take its norm in halves from their last product
    (``ops.linear.HalfNormed``): the native call ends in plain sums, and a norm kernel more per
    run of layers costs a recorded step what the call saves an eager one."""

    def __init__(self, plan, blocks, runtime):
        self.plan, self.dtype = plan, runtime.dtype
        self._find(blocks)

    def _find(self, blocks):
        order, is_float32 = self.plan.order, self.dtype == torch.float32
        self.blocks = [blocks[run.layer] for run in order]
        self.ends = [0] * len(order)
        self.parts = [None] * len(order)
        if self.plan.streams is not None:
            return
        for n in reversed(range(len(order))):
            if not _plain_layer(self.blocks[n]) or order[n].cache_from is not None:
                continue
            self.parts[n] = _parts(self.blocks[n])
            behind = n + 1
            if behind == len(order) or getattr(order[behind], "enter", None) is not None \
                    or is_float32 and not self._joins(n, behind) or not getattr(self.blocks[behind], "takes_prepared", False):
                self.ends[n] = behind
                continue
            if self._joins(n, behind):
                self.ends[n] = self.ends[behind]

    def _as_found(self, n: int, blocks) -> bool:
        """Whether run n's layer still has the parts that were looked at: a program may put one of its own, or a
        ``forward`` of its own, in a part's place at any time."""
        block = blocks[self.plan.order[n].layer]
        was, mixer, position, feed_forward, mixer_norm, ff_norm = self.parts[n]
        return (block is was and block.mixer is mixer and mixer.position is position and block.feed_forward is feed_forward
                and block.mixer_norm is mixer_norm and block.feed_forward_norm is ff_norm and not _own_forward(block))

    def _joins(self, n: int, behind: int) -> bool:
        return bool(self.ends[behind]) and _alike(self.blocks[n], self.blocks[behind])

    def take(self, n: int, stream, batch, cache, blocks) -> int:
        """Run the plain layers from run ``n`` on over the stream, if this step's rows are few enough;
        the number of runs taken (0: none).  ``blocks``: the model's, by layer."""
        if not 0 < batch.n_tokens <= F.MAX_ROWS or not self.ends[n]:
            return 0
        if not all(self._as_found(i, blocks) for i in range(n, self.ends[n])):
            self._find(blocks)
        end = self.ends[n]
        if not end:
            return 0
        first = self.blocks[n]
        m, f = first.mixer.spec, first.feed_forward.spec
        entries = cache.entries[n:end]
        if not F.takes(batch.n_tokens, m.dim, f.hidden, m.n_heads, m.n_kv_heads, m.head_dim, m.position.rotary_dim,
                       self.dtype) \
                or any(not e.writes for e in entries) \
                or len({batch.table(e.group_id).shape for e in entries}) != 1:
            return 0
        layers = [F.Layer(b.mixer.wqkv, b.mixer.wo, b.feed_forward.w13, b.feed_forward.w2, b.mixer_norm.weight,
                          b.feed_forward_norm.weight, e.k_pages, e.v_pages, batch.table(e.group_id))
                  for b, e in zip(self.blocks[n:end], entries)]
        p, sizes = m.position, (m.dim, f.hidden, m.n_heads, m.n_kv_heads, m.head_dim)
        if self.dtype == torch.bfloat16 and R.takes(batch.n_tokens, *sizes, p.rotary_dim) \
                and R.pays(end - n, batch.n_tokens, batch.n_seqs, layers[0].table.shape[1], *sizes,
                           A.compute_units(layers[0].w2.device), first.mixer.window) \
                and R.aligned(layers, stream.tensor):
            R.run(layers, stream.tensor, first.mixer.position.freqs, p.rotary_dim, batch, m.n_heads, m.n_kv_heads, m.head_dim,
                  first.mixer.window, first.mixer_norm.spec.eps, first.feed_forward_norm.spec.eps, first.mixer.scale,
                  f.activation)
            return end - n
        x = None                                         # in float32 the first product makes its norm itself
        if self.dtype == torch.bfloat16:
            x = stream.normed(first.mixer_norm, reader=first.mixer)
            x = (x.xg, x.ssq) if isinstance(x, HalfNormed) else x
        elif not F.aligned(layers):
            return 0
        F.run_layers(layers, x, stream.tensor,
                     first.mixer.position.freqs, m.position.rotary_dim, batch, m.n_heads, m.n_kv_heads, m.head_dim,
                     first.mixer.window, first.mixer_norm.spec.eps, first.feed_forward_norm.spec.eps, first.mixer.scale,
                     f.activation)
        return end - n
