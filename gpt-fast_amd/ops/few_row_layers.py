"""Python face of the entries that launch whole decoder layers over a few rows
(csrc/gemm_bf16.hip: gfa_few_row_layers_bf16, csrc/core.hip: gfa_few_row_layers_f32)."""
import ctypes

import torch

from . import attention_bf16 as A
from .gemm_bf16 import GATE_MODES, ChunkedRows, share_rows
from .kernels import GATE_ACTIVATIONS, PAGE
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


def takes(n_rows: int, dim: int, hidden: int, n_heads: int, n_kv_heads: int, head_dim: int, rotary_dim: int,
          dtype=torch.bfloat16) -> bool:
    """Whether the step's products and attention are the kernels that the entry of this type launches.  The float32 one
    may work the norms out inside the products: rows that the norm's own kernel keeps one float4 a thread of."""
    if dtype == torch.float32 and dim > 4096:
        return False
    return (0 < n_rows <= MAX_ROWS and dim % 8 == 0 and hidden % 8 == 0 and head_dim % 16 == 0 and head_dim <= 256
            and n_heads % n_kv_heads == 0 and rotary_dim % 2 == 0 and 0 < rotary_dim <= head_dim)


class Layer:
    """What one layer reads: its four matrices, the float32 weights of the norms before its attention
    and before its feed-forward, its pages and their table."""

    __slots__ = ("wqkv", "wo", "w13", "w2", "norm_mixer", "norm_ffn", "k_pages", "v_pages", "table")

    def __init__(self, wqkv, wo, w13, w2, norm_mixer, norm_ffn, k_pages, v_pages, table):
        self.wqkv, self.wo, self.w13, self.w2 = wqkv, wo, w13, w2
        self.norm_mixer, self.norm_ffn = norm_mixer, norm_ffn
        self.k_pages, self.v_pages, self.table = k_pages, v_pages, table

    def pointers(self):
        return [getattr(self, n).data_ptr() for n in self.__slots__]


def aligned(layers) -> bool:
    """Whether what the float32 entry reads in 16-byte loads begins at such addresses."""
    return all(t.data_ptr() % 16 == 0 for L in layers for t in (L.wqkv, L.w13, L.norm_mixer, L.norm_ffn))


def _check_layer(L: Layer, D: int, inner: int, H: int, G: int, hd: int, n_seqs: int, width: int, dtype):
    tensors = {n: getattr(L, n) for n in Layer.__slots__}
    require_device(*tensors.values())
    require_contiguous(**tensors)
    for name, shape in (("wqkv", ((H + 2 * G) * hd, D)), ("wo", (D, H * hd)), ("w13", (2 * inner, D)), ("w2", (D, inner))):
        w = tensors[name]
        if tuple(w.shape) != shape or w.dtype != dtype:
            raise KernelError(f"few_row_layers: {name} is {tuple(w.shape)} {w.dtype}, expected {shape} {dtype}")
    for g in (L.norm_mixer, L.norm_ffn):
        if g.dtype != torch.float32 or g.numel() != D:
            raise KernelError("few_row_layers: one float32 norm weight per column")
    if tuple(L.k_pages.shape[1:]) != (G, PAGE, hd) or tuple(L.v_pages.shape[1:]) != (G, hd, PAGE) \
            or L.k_pages.dtype != dtype or L.v_pages.dtype != dtype:
        raise KernelError("few_row_layers: pages have the wrong shape or dtype")
    if L.table.dtype != torch.int32 or tuple(L.table.shape) != (n_seqs, width):
        raise KernelError("few_row_layers: tables must be int32 and of one shape")


def run_layers(layers, x, residual, freqs, rotary_dim: int, batch, n_heads: int, n_kv_heads: int, head_dim: int,
               window: int, eps_mixer: float, eps_ffn: float, scale: float, activation: str) -> None:
    """residual (float32 [M <= 16, D]) through ``layers`` (:class:`Layer` each), in place; the tokens are those
    of ``batch``.  ``x`` None: float32 layers.  Else bfloat16 ones, and the rows of the first layer's norm over the
    stream: [M, D] or a pair (``ChunkedRows``, ssq) as ``gemm_bf16.skinny_into_chain`` leaves them."""
    M, D = residual.shape
    inner, width = layers[0].w2.shape[1], layers[0].table.shape[1]
    H, G, hd = n_heads, n_kv_heads, head_dim
    dtype = torch.float32 if x is None else torch.bfloat16
    if not takes(M, D, inner, H, G, hd, rotary_dim, dtype) or activation not in GATE_MODES:
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
    if not halves and x is not None and (tuple(rows.shape) != (M, D) or rows.dtype != torch.bfloat16):
        raise KernelError("few_row_layers: x must be bfloat16 [M, D]")
    if residual.dtype != torch.float32 or freqs.dtype != torch.float32 or freqs.numel() != rotary_dim // 2:
        raise KernelError("few_row_layers: float32 residual and one float32 frequency per pair")
    n_seqs = batch.n_seqs
    if any(t.dtype != torch.int32 for t in maps.values()) or batch.tok_seq.numel() < M or batch.tok_pos.numel() < M \
            or batch.q_start.numel() != n_seqs + 1 or batch.start_pos.numel() != n_seqs:
        raise KernelError("few_row_layers: the batch description does not fit its tokens")
    for L in layers:
        _check_layer(L, D, inner, H, G, hd, n_seqs, width, dtype)
    step = _Step(residual=residual.data_ptr(), freqs=freqs.data_ptr(), M=M, D=D, I=inner, H=H, Hkv=G, hd=hd,
                 rot=rotary_dim, table_stride=width, n_seqs=n_seqs, window=window, eps_mixer=eps_mixer, eps_ffn=eps_ffn,
                 scale=scale, **{n: t.data_ptr() for n, t in maps.items()})
    pointers = (_p * (9 * len(layers)))(*[q for L in layers for q in L.pointers()])
    if x is None:
        lib = library("core")
        lib.gfa_few_row_work_bytes_f32.restype = ctypes.c_long
        size = lib.gfa_few_row_work_bytes_f32(_i(M), _i(D), _i(inner), _i(H), _i(G), _i(hd))
        step.gate_mode = GATE_ACTIVATIONS[activation]
        launch = lib.gfa_few_row_layers_f32
    else:
        R = H // G
        step.rows_tiled = batch.max_q_len * R if batch.max_q_len * R >= A.TILED_MIN_ROWS and hd <= 128 else 0
        step.row_tiles, step.n_waves, step.max_tiles, step.n_splits = \
            (1, 1, 1, 1) if step.rows_tiled else A.plan(n_seqs, batch.max_q_len, H, G, hd, width)
        lib, attention = library("gemm_bf16"), library("attention_bf16")
        lib.gfa_few_row_work_bytes.restype = ctypes.c_long
        size = lib.gfa_few_row_work_bytes(_i(M), _i(D), _i(inner), _i(H), _i(hd), _i(step.n_splits))
        step.x0 = data.data_ptr()
        if halves:
            step.ssq0, step.t0 = ssq.data_ptr(), ssq.shape[0]
        step.attend = ctypes.cast(attention.gfa_attention_bf16, _p).value
        step.attend_tiled = ctypes.cast(attention.gfa_attention_tiled_bf16, _p).value
        step.gate_mode = GATE_MODES[activation]
        step.one_token_each = int(batch.max_q_len == 1 and M == n_seqs)
        launch = lib.gfa_few_row_layers_bf16
    work = torch.empty(size, dtype=torch.uint8, device=residual.device)
    step.work = work.data_ptr()
    check(launch(pointers, _i(len(layers)), ctypes.byref(step), stream_handle()), "few_row_layers")
