"""Library matrix products whose result goes straight into a residual add."""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from zipage_amd import _lib

_TENSORS, _FEW_TYPES = (torch.Tensor, torch.nn.Parameter), (torch.bfloat16, torch.float16)
_is_compiling, _is_autocast_enabled, _is_tracing = torch.compiler.is_compiling, torch.is_autocast_enabled, torch._C._is_tracing
_transforms, _current_device = torch._C._functorch.peek_interpreter_stack, torch._C._cuda_getDevice
_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack


def pad_to_multiple(n: int, to: int) -> int:
    return -(-n // to) * to


def fit(t: torch.Tensor, *shape: int) -> torch.Tensor:
    """`t` in the corner of a zero tensor of `shape`."""
    out = torch.zeros(shape, dtype=t.dtype, device=t.device)
    out[tuple(slice(0, n) for n in t.shape)] = t
    return out


def _few_rows(n: int, k: int, m: int) -> bool:
    """Whether a product of n rows of k elements and (m, k) weights goes to the kernel for few rows: where that is no slower on the GPU, with
    weights from memory (us of both, the library second; a call of the library costs 18 us of host time, of the kernel 7).

    Up to 16 rows: nearly everywhere (8 rows, 1024 -> 4096 4.3 and 7.7, 4096 -> 4096 9.1 and 15.8, 2048 -> 151 936 121 and 212).
    Long contractions need outputs that fill one round of workgroups (12 288 -> 4096 21.6 and 22.5, but -> 1024 18.6 and 17.0,
    -> 9216 59 and 50), and rows that are not a multiple of 16 KB apart (8192 -> 4096 17.2 and 16.2); many outputs a
    contraction that is worth a workgroup's beginning (128 -> 32 768 6.6 and 6.2, 1024 -> 65 536 29 and 27.5).
    Up to 32: as far as one round of workgroups goes (24 rows, 1024 -> 16 384 9.5 and 13.0, -> 20 480 15.1 and 14.4; 2048
    -> 8192 11.2 and 14.6, -> 9216 17.0 and 14.1; 4096 -> 4096 10.4 and 13.6, -> 6144 16.5 and 15.4).
    Up to 64, since each workgroup reads all rows: 48 rows, 1024 -> 4096 6.6 and 11.3, 3072 -> 1024 11.3 and 11.7 (which parts of the
    contraction take first, unless rows lie more than 2^22 elements apart), but -> 2048 11.4 and 10.3, -> 256 10.6 and 9.3; 64 -> 8192
    4.0 and 3.8."""
    if n <= 0 or k <= 0 or m <= 0 or k % 32 or m % 4 or k > 1 << 23:
        return False
    if n <= 16:
        if k > 4096:
            return (1024 if k <= 6144 else 4096) <= m <= 8192 and k % 8192 != 0
        return m <= 16384 or k >= (192 if m <= 32768 else 2048)
    if n <= 32:
        return k <= 4608 if m <= 4096 else 128 <= k and (k <= 2048 and m <= 8192 or k < 2048 and m <= 16384)
    return n <= 64 and m * k <= 1 << 23 and m <= 8192 and (96 <= k <= 1024 or 512 <= m and 1024 < k <= 2048 or 512 <= m <= 1280 and 2048 < k <= 4096)


def _row_tiles(n: int, k: int, m: int) -> bool:
    """The same for 65 to 256 rows, in tiles of up to 64 x 64: what makes one round of workgroups, over contractions that are not much
    longer than their beginning and end (us of both: 65 to 128 rows, 1024 -> 4096 7.7 and 12.0, 2048 -> 1024 6.5 and 8.3, 2048 -> 4096
    11.4 and 12.8, 128 -> 2048 4.1 and 4.0; 129 to 256, 1024 -> 4096 9.8 and 12.4, 2048 -> 2048 10.5 and 11.8).  The largest tiles,
    of which a CU has one workgroup, neither for long contractions (256 rows, 1536 -> 4096 12.7 and 11.2, 2048 -> 4096 18.1 and 13.2; 69
    rows, 2048 -> 7620 15.3 and 14.6) nor for so short ones that writing decides (95 rows, 160 -> 5188 5.6 and 4.8).  Longer
    contractions up to 128 rows, where the library's tiles leave most of the chip idle (128 rows, 3072 -> 4096 14.9 and 20.2; 100 rows 13.6
    and 16.5; 113 to 128 rows, up to 4064 -> 1024 to 4096 1.3 to 1.6 times as fast), but not of 4096, whose rows the library reads better
    (120 rows, -> 1776 14.2 and 12.8; 128, -> 2560 1.4 times as fast again).  Of these sizes 96 % of random ones are no more than 2 %
    slower, on average they are 1.29 times as fast (13 700 of them)."""
    if not 64 < n <= 256 or m <= 0 or k % 32 or m % 4 or k < 96:
        return False
    tiles = lambda outs: -(-n // 64) * -(-m // outs)
    if tiles(32) > 256 and (tiles(64) > 256 or not 320 <= k <= (1024 if n > 128 else 2048 if n > 112 else 2016)):
        return False
    if k == 4096 and 1024 < m <= (2176 if n == 128 else 3964):
        return False
    return k <= 2048 or n <= 128 and (n > 96 and k <= 3072 or n > 112 and k <= 4096)


def _split_rows(n: int, k: int, m: int) -> bool:
    """The same for 17 to 256 rows, in parts of the contraction, before the two above: where the library's tiles leave most of the chip
    idle (us of both: 64 rows, 12 288 -> 4096 25.5 and 36.3, 4096 -> 6144 17.2 and 17.6; 128 rows 31.1 and 66.0, 21.1 and 25.0; 192 rows 37
    and 89, 25.0 and 33.3; 256 rows 41 and 53, 28 and 39.5; 4096 -> 4096 17.3 and 23.5 for 128 rows, 21.6 and 31.5 for 192), and up to 64
    rows outputs of many rounds of workgroups (64 rows, 4096 -> 151 936 227 and 262; 48 rows, 1024 -> 151 936 66 and 77; 96 rows 259 and 273).
    Outputs that make one full round of them, in one part: up to 128 rows, 4096 -> 32 768 54 and 61 (64 rows), 51 and 67 (24), 58 and 64 (128),
    2560 -> 32 512 33 and 44; longer contractions stream weights as fast in the library (96 rows, 9728 -> 29 952 138 and 118; 128 rows,
    11 776 -> 32 256 189 and 152).
    The library's choices are uneven, so the lines are drawn where nearly all random sizes are no slower: it is good at 6144 and 8192 -> 1280
    and fewer (32 to 128 rows, 10.9 and 9.7; 144 to 184 rows to 1664, 20 and 17), at contractions of 4096 of some rows (80 rows,
    -> 3392 17.0 and 16.2; 256 rows, -> 4096 24.1 and 22.0; 255, -> 6144 28.0 and 26.3, but 224 26.6 and 36.2), of 80 and 112 rows to many outputs
    (80 rows, 2432 -> 132 352 182 and 144), at fewer than 2560 to 4096 (160 rows, 2560 -> 1216 14.3 and 9.6) and wherever
    its tiles fill the chip (256 rows, 4096 -> 24 576 64 and 62; but 128 rows 45.3 and 48.3).  Of these sizes 98 % of random ones are no
    more than 2 % slower, on average they are 1.44 times as fast (17 300 of them)."""
    if not 16 < n <= 256 or k % 32 or m % 4 or m < 512:
        return False
    if m >= 73728:
        return 1024 <= k and (n <= 32 or n <= 64 and k <= 5088) or k >= 2048 and 80 < n <= (112 if m >= 147456 else 96) and m >= 131072
    if n <= 128 and 26880 <= m <= 32768:
        return 2048 <= k <= (8192 if n <= 48 else 4608)
    if k < 2560 or m < (1664 if 64 < n <= 80 and k == 8192 else 1280) and 6144 <= k <= 8192:
        return False
    if n <= 32:
        return k <= 5120 and 21504 <= m <= 25600 or k > 4608 and (1984 if k <= 8192 else 1280) <= m <= 4864
    if n <= 64:
        return m <= 10240 if k >= 4096 else m <= 1280 or 2816 <= m <= 8192
    if n <= 128:
        if 21120 <= m <= 24576:
            return 3072 <= k <= 8192
        least = 1024 if k >= 5376 else 2432 if k >= 4480 else 3968 if n > 88 else 5632
        return k >= 4096 and least <= m <= 12288
    if k < 4096 or not 1024 <= m <= 12288:
        return False
    if n <= 192:
        return k >= 6656 or k >= 5888 and m >= 1792 or 2816 <= m <= (6656 if k < 4608 else 12288)
    return k >= 7168 or m >= 5888 and (k > 4608 or n % 32 == 0)


def _seen_by_others(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether something beside the product looks at the call, which only the library's passes through torch's dispatcher:
    gradients of either mode, vmap and its like, autocast, modes, subclasses, tracing and compilation; or another device than the current
    one is meant."""
    return (_is_compiling() or type(x) not in _TENSORS or type(w) not in _TENSORS or forward_ad._current_level >= 0
            or _transforms() is not None or _is_autocast_enabled() or _dispatch_modes() > 0 or _function_modes() > 0 or _is_tracing()
            or (x.requires_grad or w.requires_grad) and torch.is_grad_enabled() or x.device.index != _current_device())


def _linear(x: torch.Tensor, w: torch.Tensor, parts: bool) -> torch.Tensor:
    if x.is_cuda and not _seen_by_others(x, w) and x.dim() == 2 == w.dim() and x.layout == w.layout == torch.strided:
        (n, k), (m, wk), (stride, one) = x.shape, w.shape, x.stride()
        if k == wk and x.dtype == w.dtype in _FEW_TYPES and one == 1 and k <= stride <= 1 << 23 and stride % 8 == 0 and w.is_contiguous() and \
                w.device == x.device:
            at, w_at = x.data_ptr(), w.data_ptr()
            split = _split_rows(n, k, m) and stride <= 1 << 22
            if (at | w_at) % 16 == 0 and (split or _few_rows(n, k, m) or _row_tiles(n, k, m)):
                tag, stream = _lib.dtype_tag(x), _lib.stream_ptr(x)
                size = _lib.size("zp_split_rows_workspace", n, k, m) if split else 0
                parts = parts and size > 0
                out = None if parts else x.new_empty(n, m)
                if split:
                    room = x.new_empty(size // (4 * n * m), n, m, dtype=torch.float32) if size else None
                    _lib.call_models("zp_split_rows_linear", at, w_at, None if parts else out.data_ptr(), n, k, m, stride, m, tag,
                                     room.data_ptr() if size else None, size, stream)
                    if parts:
                        return room
                else:
                    _lib.call_models("zp_few_rows_linear" if n <= 64 else "zp_row_tiles_linear", at, w_at, out.data_ptr(), n, k, m, stride, m,
                                     tag, stream)
                return out
    return F.linear(x, w)


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear(x, w) without a bias."""
    return _linear(x, w, False)


def linear_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """`linear`, but a product that is made in parts of the contraction stays in them, (parts, n, m) fp32, for what adds them up itself: their
    sum in this order, rounded, is the product."""
    return _linear(x, w, True)


def step_product(ctx):
    """What a step's layers multiply with: `linear` where every sequence has one token.  What a step holds of a prompt may be few rows as
    well, and keeps the library's products, as the same rows of a whole prompt do, so that both round alike.  (All but the low-rank
    products of the delta rule: a step of runs alone makes them in the blocked kernels, whose order of fp32 sums is their own.)"""
    segments = getattr(ctx, "segments", None)
    prompts = getattr(ctx, "is_prefill", False) or getattr(ctx, "runs", None) or getattr(ctx, "run_segments", None) is not None or \
        segments is not None and segments.max_count != 1
    return F.linear if prompts else linear


class ResidualLinear:
    """y = W x, returned as planes of partial sums (planes, N, out) that `residual_norm` adds up in
    fp32.

    A product with few rows, few outputs and a long contraction leaves most of the chip idle unless
    the contraction is split; the library does not do that by itself here (4096 x 18432 at 64 rows:
    130 us whole, 37 us in four parts).  So a long bfloat16 contraction is kept in a second layout,
    one contiguous (in / 4, out) matrix per part, and steps of up to `SPLIT_ROWS` rows run the four
    parts as one batched product.  Rounding the parts to 16 bits costs no accuracy: each is half as
    large, in the root mean square, as the whole."""

    PARTS, MIN_CONTRACTION, SPLIT_ROWS = 4, 4096, 1024

    def __init__(self, w: torch.Tensor):
        self.w = w
        out, inn = w.shape
        self.parts = None
        if w.dtype == torch.bfloat16 and inn >= self.MIN_CONTRACTION and inn % (8 * self.PARTS) == 0:
            self.parts = w.t().contiguous().view(self.PARTS, inn // self.PARTS, out)

    def forward(self, x: torch.Tensor, product=linear) -> torch.Tensor:
        """`product`: see `step_product`."""
        N = x.shape[0]
        if self.parts is None or N > self.SPLIT_ROWS:
            return product(x, self.w).unsqueeze(0)
        P, k, _ = self.parts.shape
        return torch.bmm(x.view(N, P, k).transpose(0, 1), self.parts)
