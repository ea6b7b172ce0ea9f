"""Python face of the entry that launches whole decoder layers over a few rows
(csrc/gemm_bf16.hip: gfa_few_row_layers_bf16)."""
import ctypes

import torch

from . import attention_bf16 as A
from .gemm_bf16 import GATE_MODES, ChunkedRows, share_rows
from .kernels import PAGE
from .library import KernelError, check, library, require_contiguous, require_device, stream_handle

MAX_ROWS = 16

_p, _i, _f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


class _Step(ctypes.Structure):
    _fields_ = ([(n, _p) for n in ("x0", "ssq0", "residual", "freqs", "tok_seq", "tok_pos", "q_start", "start_pos", "work",
                                   "attend", "attend_tiled")]
                + [(n, _i) for n in ("t0", "M", "D", "I", "H", "Hkv", "hd", "rot", "table_stride", "n_seqs", "window",
                                     "gate_mode", "rows_tiled", "row_tiles", "n_waves", "max_tiles", "n_splits",
                                     "one_token_each")]
                + [(n, _f) for n in ("eps_mixer", "eps_ffn", "scale")])


def takes(n_rows: int, dim: int, hidden: int, n_heads: int, n_kv_heads: int, head_dim: int, rotary_dim: int) -> bool:
    """Whether the step's products and attention are the kernels that the entry launches."""
    return (0 < n_rows <= MAX_ROWS and dim % 8 == 0 and hidden % 8 == 0 and head_dim % 16 == 0 and head_dim <= 256
            and n_heads % n_kv_heads == 0 and rotary_dim % 2 == 0 and 0 < rotary_dim <= head_dim)


class Layer:
    """What one layer reads: its four matrices, the float32 weights of the norm before its feed-forward
    and of the norm before the layer behind it (None: the last of a run), its pages and their table."""

    __slots__ = ("wqkv", "wo", "w13", "w2", "norm_ffn", "norm_next", "k_pages", "v_pages", "table")

    def __init__(self, wqkv, wo, w13, w2, norm_ffn, norm_next, k_pages, v_pages, table):
        self.wqkv, self.wo, self.w13, self.w2 = wqkv, wo, w13, w2
        self.norm_ffn, self.norm_next = norm_ffn, norm_next
        self.k_pages, self.v_pages, self.table = k_pages, v_pages, table

    def pointers(self):
        return [0 if t is None else t.data_ptr() for t in (getattr(self, n) for n in self.__slots__)]


def _check_layer(L: Layer, D: int, inner: int, H: int, G: int, hd: int, n_seqs: int, width: int):
    tensors = {n: getattr(L, n) for n in Layer.__slots__}
    require_device(*tensors.values())
    require_contiguous(**tensors)
    for name, shape in (("wqkv", ((H + 2 * G) * hd, D)), ("wo", (D, H * hd)), ("w13", (2 * inner, D)), ("w2", (D, inner))):
        w = tensors[name]
        if tuple(w.shape) != shape or w.dtype != torch.bfloat16:
            raise KernelError(f"few_row_layers: {name} is {tuple(w.shape)} {w.dtype}, expected {shape} bfloat16")
    for g in (L.norm_ffn, L.norm_next):
        if g is not None and (g.dtype != torch.float32 or g.numel() != D):
            raise KernelError("few_row_layers: one float32 norm weight per column")
    if tuple(L.k_pages.shape[1:]) != (G, PAGE, hd) or tuple(L.v_pages.shape[1:]) != (G, hd, PAGE) \
            or L.k_pages.dtype != torch.bfloat16 or L.v_pages.dtype != torch.bfloat16:
        raise KernelError("few_row_layers: pages have the wrong shape or dtype")
    if L.table.dtype != torch.int32 or tuple(L.table.shape) != (n_seqs, width):
        raise KernelError("few_row_layers: tables must be int32 and of one shape")


def run_layers(layers, x, residual, freqs, rotary_dim: int, batch, n_heads: int, n_kv_heads: int, head_dim: int,
               window: int, eps_mixer: float, eps_ffn: float, scale: float, activation: str) -> None:
    """residual (float32 [M <= 16, D]) through ``layers`` (:class:`Layer` each), in place.  ``x``: the rows of the
    first layer's norm over it, bfloat16 [M, D] or a pair (``ChunkedRows``, ssq) as
    ``gemm_bf16.skinny_into_chain`` leaves them.  The tokens are those of ``batch``."""
    M, D = residual.shape
    inner, width = layers[0].w2.shape[1], layers[0].table.shape[1]
    H, G, hd = n_heads, n_kv_heads, head_dim
    if not takes(M, D, inner, H, G, hd, rotary_dim) or activation not in GATE_MODES:
        raise KernelError(f"few_row_layers: {M} rows of {D}, {inner} inner, {H}/{G} heads of {hd}, {activation}")
    halves = isinstance(x, tuple)
    rows, ssq = x if halves else (x, None)
    data = rows.data if halves else rows
    maps = dict(tok_seq=batch.tok_seq, tok_pos=batch.tok_pos, q_start=batch.q_start, start_pos=batch.start_pos)
    require_device(residual, data, ssq, freqs, *maps.values())
    require_contiguous(residual=residual, x=data, ssq=ssq, freqs=freqs, **maps)
    if halves and (not isinstance(rows, ChunkedRows) or rows.shape != (M, D) or ssq.dtype != torch.float32
                   or ssq.dim() != 2 or ssq.shape[1] != share_rows(M)):
        raise KernelError("few_row_layers: the halves of the first norm do not fit the rows")
    if not halves and (tuple(rows.shape) != (M, D) or rows.dtype != torch.bfloat16):
        raise KernelError("few_row_layers: x must be bfloat16 [M, D]")
    if residual.dtype != torch.float32 or freqs.dtype != torch.float32 or freqs.numel() != rotary_dim // 2:
        raise KernelError("few_row_layers: float32 residual and one float32 frequency per pair")
    n_seqs = batch.n_seqs
    if any(t.dtype != torch.int32 for t in maps.values()) or batch.tok_seq.numel() < M or batch.tok_pos.numel() < M \
            or batch.q_start.numel() != n_seqs + 1 or batch.start_pos.numel() != n_seqs:
        raise KernelError("few_row_layers: the batch description does not fit its tokens")
    for L in layers:
        _check_layer(L, D, inner, H, G, hd, n_seqs, width)
        if (L.norm_next is None) != (L is layers[-1]):
            raise KernelError("few_row_layers: every layer but the last needs the norm of the one behind it")
    R = H // G
    tiled = batch.max_q_len * R if batch.max_q_len * R >= A.TILED_MIN_ROWS and hd <= 128 else 0
    rt, nw, tiles, splits = (1, 1, 1, 1) if tiled else A.plan(n_seqs, batch.max_q_len, H, G, hd, width)
    lib, attention = library("gemm_bf16"), library("attention_bf16")
    lib.gfa_few_row_work_bytes.restype = ctypes.c_long
    work = torch.empty(lib.gfa_few_row_work_bytes(_i(M), _i(D), _i(inner), _i(H), _i(hd), _i(splits)),
                       dtype=torch.uint8, device=residual.device)
    pointers = (_p * (9 * len(layers)))(*[q for L in layers for q in L.pointers()])

    def entry(fn):
        return ctypes.cast(fn, _p).value
    step = _Step(data.data_ptr(), None if ssq is None else ssq.data_ptr(), residual.data_ptr(), freqs.data_ptr(),
                 batch.tok_seq.data_ptr(), batch.tok_pos.data_ptr(), batch.q_start.data_ptr(), batch.start_pos.data_ptr(),
                 work.data_ptr(), entry(attention.gfa_attention_bf16), entry(attention.gfa_attention_tiled_bf16),
                 0 if ssq is None else ssq.shape[0], M, D, inner, H, G, hd, rotary_dim, width, n_seqs, window,
                 GATE_MODES[activation], tiled, rt, nw, tiles, splits,
                 int(batch.max_q_len == 1 and M == n_seqs), eps_mixer, eps_ffn, scale)
    check(lib.gfa_few_row_layers_bf16(pointers, _i(len(layers)), ctypes.byref(step), stream_handle()), "few_row_layers")
