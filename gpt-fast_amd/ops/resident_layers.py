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
         head_dim: int, units: int, window: int = 0) -> bool:
    """Whether one launch that stays on its ``units`` compute units takes less time than five launches a layer
    (ops.few_row_layers), both measured on 256 units, in us for the layers alone, 200 keys a row where nothing else is said
    (some 1,800 steps of 31 shapes):

    - From 8 layers on: meeting at the start costs what some layers give.  1 row and 8 rows: 288 wide, 2 layers 51 -> 66, 54 -> 65;
      5 layers 118 -> 119, 122 -> 118; 8 layers 184 -> 169, 192 -> 172; 768 wide 4 layers 106 -> 108, 112 -> 112; 8 layers 205 -> 185,
      225 -> 194; 8B 3 layers 266 -> 258, 276 -> 282; 8 layers 701 -> 642, 718 -> 699; 70B 10 layers 3051 -> 2772, 3044 -> 2960.
      Five to seven layers of most shapes would gain 1 to 8 % too.
    - More than 8 rows only where those of the widest product fit the two halves of their shared memory one after
      the other.  12 layers of 12 rows: 768 wide 358 -> 290, 2048 wide (5632 inner) 514 -> 466, 3072 (8192) 754 -> 778,
      8B 1199 -> 1288, 5120 (13824) 1836 -> 2210.
    - As many pairs of a row and a key/value head as units at most.  12 layers 5120 wide, 40 such heads: 6 rows 1638 -> 1594, 8 rows
      1692 -> 1674; 10 layers 6656 wide, 52 heads: 4 rows 1963 -> 1858, 5 rows 2063 -> 2195.
    - One or two sequences with one new token each, up to 12288 keys.  12 layers of 8B, 1 row: 12000 keys 1210 -> 1169, 30000
      keys 1381 -> 1367, 1 %, which is less than two machines differ by.
    - One new token for each sequence: up to 4608 keys, and of all rows' and heads' blocks of 32 keys no more than 24 a unit.  Attention by three
      waves of a workgroup has fewer keys under way than a launch of its own, and from some length on that costs more
      than the meetings save.  12 layers, 4000, 6000 and 12000 keys: 1024 wide, 4 kv heads of 128, 1 row 387 -> 354, 396 -> 380, 437 -> 459; heads of 32,
      1 row, 3500 and 5000 keys 346 -> 322, 341 -> 354.  768 wide, heads of 64 (12 blocks a unit with 8 rows of 1000 keys): 8 rows of 1000, 2000, 6000 keys
      420 -> 357, 504 -> 447, 724 -> 749; 16 rows of 500, 1500 and 5000 keys 388 -> 352, 494 -> 523, 831 -> 1180; 512 wide, heads of 32, 16 rows
      of 1500 keys 411 -> 485.  All contexts are taken to be as long as the table: which are shorter is known on the device
      only, and may change from replay to replay.  (One long context among short ones gains: 768 wide, 8 rows, one of 6000 keys 450 -> 376.)
      With a window the keys are the window's: 768 wide, 8 rows of 10000 keys, window 1024 420 -> 357, 4096 619 -> 623.
    - But for heads of 128, eight or more of keys and values: at any length: 8B, 8 rows of 20000 keys 2438 -> 2329; a 7B shape, 8 rows of 16000
      5403 -> 5160, 4 rows of 30000 4988 -> 4825.  Blocks of such heads are large enough.  Four of them: 1 row of 30000 keys
      10 to 16 % slower.
    - Several new tokens of a sequence pay at any length, since the attention of prompts has too few workgroups there: 2048 wide, 8 behind 6000
      keys 1211 -> 511; 768 wide, 15 rows of 5000 keys and one more for one of them 2249 -> 1164."""
    widest = max(dim, hidden, n_heads * head_dim)
    keys = table_pages * PAGE
    if window > 0:
        keys = min(keys, window)
    one_each = n_rows <= n_seqs
    few_keys = keys <= 4608 and n_rows * n_kv_heads * -(-keys // 32) <= 24 * units
    large_blocks = head_dim == 128 and n_kv_heads >= 8 and (n_rows > 2 or keys <= 12288)
    return (n_layers >= 8 and n_rows * n_kv_heads <= units
            and (n_rows <= 8 or 2 * MAX_ROWS * widest <= 2 * X_BYTES)
            and (not one_each or few_keys or large_blocks))


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
