"""Python face of the kernel that takes few rows through whole plain layers in one launch
(csrc/resident_layers.hip)."""
import ctypes

import torch

from .few_row_layers import _Step, _check_layer
from .gemm_bf16 import GATE_MODES
from .kernels import PAGE
from .library import KernelError, check, library, require_contiguous, require_device, stream_handle

MAX_ROWS = 16
X_BYTES = 88 * 1024          # of shared memory for the rows that a product multiplies (RL_X_BYTES)
MOST_BYTES = 0xffff0000      # of one matrix: offsets into it are 32-bit
MOST_COLUMNS = 1 << 23       # of a row of x: so are those into a layer's rows

_p, _i = ctypes.c_void_p, ctypes.c_int


def takes(n_rows: int, dim: int, hidden: int, n_heads: int, n_kv_heads: int, head_dim: int, rotary_dim: int) -> bool:
    """Whether the kernel computes such layers at all."""
    return (0 < n_rows <= MAX_ROWS and dim % 8 == 0 and hidden % 8 == 0 and head_dim % 16 == 0 and head_dim <= 128
            and n_heads % n_kv_heads == 0 and n_heads // n_kv_heads <= 16 and rotary_dim % 2 == 0
            and 0 < rotary_dim <= head_dim and max(dim, hidden, n_heads * head_dim) < MOST_COLUMNS and 4 * dim * hidden < MOST_BYTES
            and 2 * dim * (n_heads + 2 * n_kv_heads) * head_dim < MOST_BYTES)


def pays(n_layers: int, n_rows: int, n_seqs: int, table_pages: int, dim: int, hidden: int, n_heads: int, n_kv_heads: int,
         head_dim: int, units: int) -> bool:
    """Whether one launch that stays on its ``units`` compute units takes less time than five launches a layer
    (ops.few_row_layers), both measured on 256 units, in us a step (this side when its phases met through 16 counters, not 128:
    2 to 9 % longer than now):

    - From 8 layers on: meeting at the start costs what some layers give.  768 wide, 1 row: 3 layers 118 -> 130, 6 layers
      190 -> 190, 12 layers 333 -> 306; 288 wide, 8 layers 215 -> 204; 4096 wide (8B) 2 layers 373 -> 380, 4 layers 554 -> 542,
      8 layers 895 -> 851, 32 layers 2990 -> 2740.
    - More than 8 rows only where those of the widest product fit the two halves of their shared memory one after
      the other.  12 rows: 768 wide 400 -> 370, 2048 wide (5632 inner) 577 -> 558, 3072 (8192) 828 -> 873, 8B 3365 -> 3646.
    - As many pairs of a row and a key/value head as units at most: 6656 wide, 52 heads, 12 layers: 4 rows 2366 -> 2329, 8 rows
      2506 -> 2696.
    - One or two sequences with one new token each, up to 12288 keys: attention that has the chip to itself then
      reads the cache at 5.1 TB/s, beside waves that hold weights at 3.6.  8B, 1 row: 6000 keys 3240 -> 3149, 12000 keys
      3359 -> 3347, 30000 keys 3755 -> 3827.  Several new tokens of a sequence pay at any length: 8 behind 6000 keys
      10300 -> 3710; so do more sequences: 4 of 15000 keys 4470 -> 4343, 8 of which one has 16000 4310 -> 3740."""
    widest = max(dim, hidden, n_heads * head_dim)
    return (n_layers >= 8 and n_rows * n_kv_heads <= units
            and (n_rows <= 8 or 2 * MAX_ROWS * widest <= 2 * X_BYTES)
            and (n_rows > 2 or n_rows > n_seqs or table_pages * PAGE <= 12288))


def aligned(layers, residual) -> bool:
    """Whether what is read in 16-byte loads begins at such addresses."""
    return residual.data_ptr() % 16 == 0 and all(
        t.data_ptr() % 16 == 0 for L in layers
        for t in (L.wqkv, L.wo, L.w13, L.w2, L.norm_mixer, L.norm_ffn, L.k_pages, L.v_pages))


def run(layers, residual, freqs, rotary_dim: int, batch, n_heads: int, n_kv_heads: int, head_dim: int, window: int,
        eps_mixer: float, eps_ffn: float, scale: float, activation: str, *, workgroups: int = 0,
        start_polls: int = 0) -> None:
    """residual (float32 [M <= 16, D]) through bfloat16 ``layers`` (few_row_layers.Layer each), in place; the tokens
    are those of ``batch``.  ``workgroups``, ``start_polls``: fewer of either than usual (0: the usual number)."""
    M, D = residual.shape
    inner, width = layers[0].w2.shape[1], layers[0].table.shape[1]
    H, G, hd = n_heads, n_kv_heads, head_dim
    if not takes(M, D, inner, H, G, hd, rotary_dim) or activation not in GATE_MODES:
        raise KernelError(f"resident_layers: {M} rows of {D}, {inner} inner, {H}/{G} heads of {hd}, {activation}")
    maps = dict(tok_seq=batch.tok_seq, tok_pos=batch.tok_pos, start_pos=batch.start_pos)
    require_device(residual, freqs, *maps.values())
    require_contiguous(residual=residual, freqs=freqs, **maps)
    if residual.dtype != torch.float32 or freqs.dtype != torch.float32 or freqs.numel() != rotary_dim // 2:
        raise KernelError("resident_layers: float32 residual and one float32 frequency per pair")
    if any(t.dtype != torch.int32 for t in maps.values()) or batch.tok_seq.numel() < M or batch.tok_pos.numel() < M \
            or batch.start_pos.numel() != batch.n_seqs:
        raise KernelError("resident_layers: the batch description does not fit its tokens")
    for L in layers:
        _check_layer(L, D, inner, H, G, hd, batch.n_seqs, width, torch.bfloat16)
    if not aligned(layers, residual):
        raise KernelError("resident_layers: weights, pages and the residual must begin at multiples of 16 bytes")
    step = _Step(residual=residual.data_ptr(), freqs=freqs.data_ptr(), M=M, D=D, I=inner, H=H, Hkv=G, hd=hd,
                 rot=rotary_dim, table_stride=width, n_seqs=batch.n_seqs, window=window, eps_mixer=eps_mixer, eps_ffn=eps_ffn,
                 scale=scale, gate_mode=GATE_MODES[activation], **{n: t.data_ptr() for n, t in maps.items()})
    lib = library("resident_layers")
    lib.gfa_resident_work_bytes.restype = ctypes.c_long
    launches = -(-len(layers) // lib.gfa_resident_layers_max())
    each = -(-len(layers) // launches)
    for at in range(0, len(layers), each):
        some = layers[at:at + each]
        size = lib.gfa_resident_work_bytes(_i(len(some)), _i(M), _i(D), _i(inner), _i(H), _i(G), _i(hd), _i(width))
        work = torch.empty(size, dtype=torch.uint8, device=residual.device)
        step.work = work.data_ptr()
        pointers = (_p * (9 * len(some)))(*[q for L in some for q in L.pointers()])
        check(lib.gfa_resident_layers_bf16(pointers, _i(len(some)), ctypes.byref(step), _i(workgroups),
                                           _i(start_polls), stream_handle()), "resident_layers")
