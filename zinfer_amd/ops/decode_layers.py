"""All layers of a decoder in one launch (csrc/decode_layers.hip): which shapes the kernel takes, its
buffers, its launch."""
from __future__ import annotations

import ctypes
import functools

import torch

from ..errors import KernelUnavailable
from . import _check, _i32, _launches, _need_gpu, _stream, build

HEAD_DIM = 128               # DL_HD in decode_layers.hip
SPLIT_KEYS = 128             # DL_SPLIT
MAX_SPLITS = 32              # of a context
MAX_CONTEXT = MAX_SPLITS * SPLIT_KEYS
MAX_UNITS = 16               # DL_UNITS
MAX_FF_UNITS = 32            # DL_FF_UNITS
MAX_ATTENTION = 8            # DL_ATT
MAX_TOKENS = 4               # DL_TOKENS
MEETING = 512                # bytes of DecodeMeet
# Of 10 ns: how long the workgroups that have come wait for the others, and while they are fewer than hold a
# phase's sums (longer than most kernels keep a CU; the 0.6B shape on 16 workgroups, which do, 1.3 ms a step, on
# 15 4.9, on all 256 0.47; eight layers of the 8B shape on 24 2.4, on 16 6.0, on all 0.60)
MEET_TICKS, MEET_MOST = 5000, 100000
SPIN_FROM = 0                # looks that a wait between workgroups begins with (of DL_SPINS)

_vp, _i, _f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


class Layer(ctypes.Structure):
    """``DecodeLayer``."""
    _fields_ = [("w", _vp * 4), ("q_gain", _vp), ("k_gain", _vp), ("ff_gain", _vp),
                ("next_gain", _vp), ("k_pool", _vp), ("v_pool", _vp)]


class _Layers(ctypes.Structure):
    """``DecodeLayers``."""
    _fields_ = [("layers", _vp)] \
        + [(n, _i) for n in ("tokens", "n_layers", "hidden", "ff", "n_heads", "n_kv_heads", "page_size",
                             "max_pages", "max_splits")] \
        + [(n, _f) for n in ("eps_in", "eps_ff", "eps_head", "scale_log2e")] \
        + [("cos", _vp), ("sin", _vp), ("table_rows", _i), ("positions", _vp), ("slot_mapping", _vp),
           ("block_table", _vp), ("ctx_len", _vp), ("x", _vp), ("xg", _vp), ("sq", _vp),
           ("words", _vp), ("meet", _vp)] \
        + [(n, _i) for n in ("need", "meet_ticks", "meet_most", "spin_from")] + [("status", _vp)]


@functools.lru_cache(maxsize=None)
def compute_units(device_index: int) -> int:
    return torch.cuda.get_device_properties(device_index).multi_processor_count


def workgroups(device_index: int) -> int:
    """A workgroup a CU."""
    return compute_units(device_index)


def sizes_covered(tokens: int, hidden: int, ff: int, n_heads: int, n_kv_heads: int, head_dim: int,
                  page_size: int, wgs: int) -> bool:
    """Whether the kernel takes a step of so many tokens of such layers on ``wgs`` workgroups."""
    if not (1 <= tokens <= MAX_TOKENS and head_dim == HEAD_DIM and n_kv_heads >= 1
            and n_heads % n_kv_heads == 0 and n_heads // n_kv_heads <= 15 and page_size % 16 == 0
            and hidden % 64 == 0 and ff % 64 == 0
            and min(hidden, ff, n_heads * head_dim) >= 512):
        return False
    units = (hidden // 16, (n_heads + 2 * n_kv_heads) * head_dim // 16)
    row = 2 * max(hidden, ff, n_heads * head_dim) + 16
    most = wgs // 2                # (the half of a launch that meets another one runs as it is meant to)
    return max(units) <= MAX_UNITS // tokens * most and ff // 16 <= MAX_FF_UNITS // tokens * most \
        and tokens * n_kv_heads * MAX_SPLITS <= MAX_ATTENTION * most \
        and 80 * 1024 + tokens * (row + hidden // 4 + 512) <= 160 * 1024


def uneven_bytes(hidden: int, ff: int, n_heads: int, n_kv_heads: int, cus: int) -> int:
    """What all workgroups would read of a layer's weights if each read as much as the busiest one of
    each phase, beyond what there is."""
    q = n_heads * HEAD_DIM
    phases = (((q + 2 * n_kv_heads * HEAD_DIM) // 16, 32 * hidden), (hidden // 16, 32 * (q + ff)),
              (ff // 16, 64 * hidden))
    return sum((-(-units // cus) * cus - units) * unit for units, unit in phases)


def pays(tokens: int, hidden: int, ff: int, n_heads: int, n_kv_heads: int, keys: int, cus: int) -> bool:
    """Whether a step of so many tokens under tables of ``keys`` keys is faster in one launch than with a
    launch a product.  Measured in us a layer gained, head and draw in both.  A phase ends with its busiest
    workgroup: by ``uneven_bytes``, one token behind 100 to 3900 keys 17 MB (8B shape) +8.6 to 10.1, 79
    (4B) +5.4 to 7.3, 183 (5120 wide, 32 heads, 13824) +1.2 to 3.9, 197 (4608, 36, 14336) -1.8 to +0.8,
    211 (14B) -1.9 to +1.2, 291 (32B) -4.9 to -2.0; two tokens 71 (3584, 28, 18944) -0.1 to +2.6, 183 -2.8 to
    +1.2, 211 -8.4 to -0.7.  The rows that splits of contexts hand on grow with tokens, heads and keys: behind 2400 and
    3900 keys three tokens of 32 heads gain +4.0 and -0.4 (2048 wide), +1.0 and -3.0 (4B), of 24 +2.2 and
    -1.8, of 16 (1.7B) +2.4 at 3900; four tokens of 16 heads +1.0 and -1.3, of 24 (2560 wide) behind 700, 1400 and
    2400 +3.3, -0.8 and -2.2."""
    narrow = n_heads <= 16
    most_keys = MAX_CONTEXT if tokens <= 2 else \
        (4096 if narrow else 3072) if tokens == 3 else (3072 if narrow else 1024)
    return keys <= most_keys and \
        uneven_bytes(hidden, ff, n_heads, n_kv_heads, cus) <= (185e6 if tokens == 1 else 130e6)


def words(tokens: int, hidden: int, ff: int, n_heads: int, n_kv_heads: int, device) -> torch.Tensor:
    """The words the workgroups hand rows on with, and behind them where they meet; zero at first."""
    lib = build.load("decode_layers")
    lib.zf_decode_layers_words.restype = ctypes.c_longlong
    n = lib.zf_decode_layers_words(tokens, hidden, ff, n_heads, n_kv_heads, MAX_SPLITS)
    n = (n + MEETING - 1) // MEETING * MEETING
    return torch.zeros((n + MEETING,), dtype=torch.uint8, device=device)


@_launches("products")
def decode_layers(table: torch.Tensor, n_layers: int, x: torch.Tensor, xg: torch.Tensor,
                  sq: torch.Tensor, ff: int, n_heads: int, n_kv_heads: int, page_size: int,
                  eps_in: float, eps_ff: float, eps_head: float, scale: float, cos, sin,
                  positions: torch.Tensor, slot_mapping: torch.Tensor, block_table: torch.Tensor,
                  ctx_len: torch.Tensor, word_buffer: torch.Tensor, status: torch.Tensor) -> None:
    """The layers of ``table`` (``Layer`` records on the device) over the stream x [M, hidden], in
    place, a sequence a token; xg and sq are what ``ops.gemm_emit`` leaves of it, before the first
    layer's norm and behind the last layer for the norm that reads the stream next.  ``status``
    (pinned host memory) becomes 1 if a wait between workgroups came to its end, with rows of NaN."""
    _need_gpu(table, x, xg, sq, cos, sin, positions, slot_mapping, block_table, ctx_len, word_buffer)
    M, H = x.shape
    wgs = workgroups(x.device.index or 0)
    if not sizes_covered(M, H, ff, n_heads, n_kv_heads, HEAD_DIM, page_size, wgs) \
            or x.dtype != torch.float32 or xg.dtype != torch.bfloat16 or xg.shape != (M, H) \
            or sq.dtype != torch.float32 or sq.shape != (H // 16, 16) or ctx_len.shape[0] != M \
            or block_table.shape[0] != M or positions.shape[0] != M or slot_mapping.shape[0] != M \
            or table.numel() != n_layers * ctypes.sizeof(Layer) \
            or block_table.shape[1] * page_size > MAX_CONTEXT or (cos is None) != (sin is None) \
            or any(t is not None and (t.dtype != torch.float32 or t.shape != cos.shape
                                      or t.shape[1] != HEAD_DIM // 2 or not t.is_contiguous())
                   for t in (cos, sin)) \
            or not all(t.is_contiguous() for t in (x, xg, sq, block_table)):
        raise KernelUnavailable(f"decode_layers: x {tuple(x.shape)}, ff {ff}, {n_heads} heads on "
                                f"{n_kv_heads}, tables {tuple(block_table.shape)} of {page_size} rows")
    for t, name in ((positions, "positions"), (slot_mapping, "slot_mapping"),
                    (block_table, "block_table"), (ctx_len, "ctx_len")):
        _i32(t, name)
    ptr = lambda t: None if t is None else t.data_ptr()
    p = _Layers(ptr(table), M, n_layers, H, ff, n_heads, n_kv_heads, page_size, block_table.shape[1],
                MAX_SPLITS, eps_in, eps_ff, eps_head, scale * 1.4426950408889634, ptr(cos), ptr(sin),
                0 if cos is None else cos.shape[0], ptr(positions), ptr(slot_mapping),
                ptr(block_table), ptr(ctx_len), ptr(x), ptr(xg), ptr(sq), ptr(word_buffer),
                word_buffer.data_ptr() + word_buffer.numel() - MEETING, 0, MEET_TICKS, MEET_MOST, SPIN_FROM,
                ptr(status))
    lib = build.load("decode_layers")
    _check(lib.zf_decode_layers(ctypes.byref(p), wgs, _stream()), "decode_layers")
