"""Entry points of the routing kernels and the grouped product (`csrc/routed.hip`): routed experts, and products
in which every head has a weight matrix of its own."""

from __future__ import annotations

import ctypes
import functools
from dataclasses import dataclass
from typing import Optional, Tuple

import torch

from . import build as _build

MAX_ROUTE_TOP = 16  # csrc/routed.hip: ROUTE_MAX_TOP
MAX_EXPERTS = 256  # csrc/routed.hip: ROUTE_MAX_EXPERTS
TILE_ROWS = 16  # rows of a tile of the grouped product
# From MEDIUM_ROWS rows an expert (on average) a block of the grouped product takes 4 row tiles instead of 2, and from
# WIDE_ROWS, 8: at 16 experts of 2,048 x 1,024 gate, up and down together take 49 us with 2 and 4 tiles at 16 rows, 71 and
# 50 us at 24; 76 us with 4 and 57 us with 8 at 48, where the busier experts have more than 64.
MEDIUM_ROWS = 16
WIDE_ROWS = 48
STREAM_ROWS = 3  # up to so many rows an expert, gate and up go to the kernel that splits K: 28 instead of 30 us at 2 rows (weights
# of 2,048 x 1,024), 102 instead of 115 us (3,072 x 1,536, 32 experts); at 4 rows 35 and 33 us, 134 and 124 us


@functools.cache  # an import statement costs a launch-bound step a microsecond and more a call
def _base():
    from . import KernelError, _check, _code, _i32, _need_gpu, _ptr, _stream

    return KernelError, _check, _code, _i32, _need_gpu, _ptr, _stream


def _check_scores(scores: str, correction: Optional[torch.Tensor], scale: float, renormalize: bool, n_experts: int) -> None:
    KernelError = _base()[0]
    if scores not in ("softmax_chosen", "softmax_all"):
        raise KernelError(f"router scores {scores!r}: 'softmax_chosen' and 'softmax_all' are known")
    if scores == "softmax_chosen" and (correction is not None or scale != 1.0 or renormalize):
        raise KernelError("a correction, a scale and renormalised weights belong to router scores over all experts")
    if correction is not None and (correction.dtype != torch.float32 or correction.shape != (n_experts,) or not correction.is_contiguous()):
        raise KernelError("the router's correction must be a contiguous float32 tensor, one value an expert")


def _open_groups(groups: Optional[Tuple[int, int]], n_experts: int, top: int) -> Tuple[int, int]:
    count, keep = groups if groups is not None else (1, 1)
    if count < 1 or n_experts % count != 0 or not 1 <= keep <= count or top > keep * (n_experts // count):
        raise _base()[0](f"{keep} of {count} groups of {n_experts} experts do not hold {top} choices")
    return count, keep


def route_top(
    logits: torch.Tensor, top: int, scores: str = "softmax_chosen", correction: Optional[torch.Tensor] = None, scale: float = 1.0,
    renormalize: bool = False, groups: Optional[Tuple[int, int]] = None,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """float32 router logits [T, E] -> (chosen int32 [T, top], weights float32 [T, top]), the chosen in falling order
    of what they were chosen by (the lower index first among equals).
    `scores` "softmax_chosen": the `top` largest logits, weighted by the softmax over those alone.
    `scores` "softmax_all": s = softmax over all experts; the `top` largest of s + `correction` (float32 [E], None for
    none) are chosen; their weights are `scale` * s (the correction is no part of a weight), divided by the sum of
    the chosen s first if `renormalize`.  `groups` (count, keep): the experts form `count` equal groups of neighbours, and
    only those of the `keep` groups with the best members can be chosen."""
    KernelError, _check, _code, _i32, _need_gpu, _ptr, _stream = _base()
    _need_gpu(logits, correction)
    _check_scores(scores, correction, scale, renormalize, logits.shape[-1])
    if logits.dtype != torch.float32 or logits.dim() != 2 or not logits.is_contiguous():
        raise KernelError("router logits must be a contiguous float32 [T, E] tensor")
    n, e = logits.shape
    if not 1 <= top <= min(e, MAX_ROUTE_TOP):
        raise KernelError(f"{top} of {e} experts: the kernel takes 1..{min(e, MAX_ROUTE_TOP)}")
    count, keep = _open_groups(groups, e, top)
    chosen = torch.empty((n, top), dtype=torch.int32, device=logits.device)
    weights = torch.empty((n, top), dtype=torch.float32, device=logits.device)
    lib = _build.load("routed")
    _check(
        lib,
        lib.cwm_route_top(
            _ptr(logits), _ptr(chosen), _ptr(weights), ctypes.c_int(n), ctypes.c_int(e), ctypes.c_int(top),
            ctypes.c_int(int(scores == "softmax_all")), _ptr(correction), ctypes.c_float(scale), ctypes.c_int(int(renormalize)),
            ctypes.c_int(count), ctypes.c_int(keep), _stream(),
        ),
    )
    return chosen, weights


@dataclass
class ExpertGroups:
    """The step's (token, choice) pairs grouped by expert in tiles of 16 rows."""

    row_token: torch.Tensor  # int32 [tiles * 16]: the token of each row, -1 in the padding
    pair_row: torch.Tensor  # int32 [T * top]: the row of each pair
    tile_expert: torch.Tensor  # int32 [tiles]: the expert of each tile, -1 for tiles not in use
    n_tiles: int
    tiles_a_block: int  # an expert's tiles start at a multiple of so many: the most row tiles that a block of the grouped product takes
    top: int
    used: Optional[torch.Tensor] = None  # int32 [1]: the tiles up to the last one in use, where they have been counted


def _tiles_a_block(rows: float) -> int:
    return 8 if rows >= WIDE_ROWS else 4 if rows >= MEDIUM_ROWS else 2


def _product_tiles(dtype: torch.dtype, k: int, rows: float, gated: bool) -> int:
    """Row tiles that a block of the product takes: a divisor of the list's own multiple (`_tiles_a_block`)."""
    if dtype != torch.bfloat16 or k % 64 != 0:  # the kernels whose operands do not go through LDS
        return 8 if rows >= 256 else 4 if rows >= 64 else 1
    return 1 if gated and rows < STREAM_ROWS else _tiles_a_block(rows)


LOOP_BLOCKS = 256  # csrc/routed.hip: GROUPED_BLOCKS


def _loop_pays(pairs: int, n_experts: int, columns: int, k: int, gated: bool) -> bool:
    """Whether a product of many rows an expert goes to the persistent blocks, which take tiles of 128 rows and 256 columns of
    weights in rounds, and what is left below half a round in quarters.  The rounds are those that the rows and half a tile of padding an
    expert make expect.  One round of quarters is always ahead (the other kernel / this, us, weights not in a cache: 4 experts of
    2,048 x 2,048, 203 tokens, gates and ups then without, 34 / 22 and 29 / 19).  Two of them are ahead with gates and ups, and not without (16 of
    2,048 x 1,024, 262 tokens, evenly spread 36 / 36 and 20 / 24, unevenly 48 / 41 and 27 / 26; 8 of 1,024 x 1,024, 0.4 rounds, 18.2 / 19.6).  Whole
    tiles take a round to its end: ahead from two thirds of one up to 1.25 and from 1.9 on, in between or not (4 of 2,048 x 2,048, 1.4
    rounds 59 / 66, 1.6 68 / 67).  A short K has too little to do between a tile's sums (8 of 512 x 320, 1.1 rounds 18 / 24), and
    after four rounds the other kernel's last one weighs no more (64 of 2,048 x 768 with gates and ups, 2,600 tokens 168 / 169, 8,195 408 / 435).  Of 1,300 products of 13 shapes and 48 to 4,096 rows an expert, evenly and unevenly spread, this
    takes 556, 1.12 times as fast in the mean and 33 slower by more than 3% (evenly spread rows that end with their tiles, mostly)."""
    rounds = (pairs / 128 + n_experts / 2) * -(-columns // (128 if gated else 256)) / LOOP_BLOCKS
    if rounds <= 0.25:
        return True
    return k >= (1536 if gated else 640) and ((gated or rounds > 0.65) and rounds <= 1.25 or 1.9 < rounds <= 4.2)


def _empty_groups(n: int, top: int, n_experts: int, device: torch.device) -> ExpertGroups:
    pairs = n * top
    align = _tiles_a_block(pairs / n_experts)
    n_tiles = -(-pairs // TILE_ROWS) + n_experts * align
    lists = torch.empty(n_tiles * TILE_ROWS + pairs + n_tiles + 1, dtype=torch.int32, device=device)
    row_token, pair_row, tile_expert, used = lists.split_with_sizes((n_tiles * TILE_ROWS, pairs, n_tiles, 1))
    return ExpertGroups(row_token, pair_row, tile_expert, n_tiles, align, top, used)


_ROUTE_GROUP_LIMITS: Optional[Tuple[int, int, int]] = None


def route_group_limits() -> Tuple[int, int, int]:
    """(tokens, experts, K) up to which `route_and_group` goes, asked of the library."""
    global _ROUTE_GROUP_LIMITS
    if _ROUTE_GROUP_LIMITS is None:
        lib = _build.load("routed")
        _ROUTE_GROUP_LIMITS = int(lib.cwm_route_group_tokens()), int(lib.cwm_route_group_experts()), int(lib.cwm_route_group_max_k())
    return _ROUTE_GROUP_LIMITS


# The one block of `route_and_group` reads the router 16 experts after the other, so it is ahead of the three launches for so many and a K of up to
# 4,096 only.  One launch / three, us, weights not in a cache, at 1, 8 and 16 tokens: 16 experts, K = 1,024 7.8 / 9.5, 8.5 / 10.3, 9.1 / 10.1;
# 2,048 8.7 / 10.9, 9.5 / 11.7, 10.7 / 12.6; 4,096 10.3 / 13.2, 11.8 / 14.9, 13.7 / 16.0; 8,192 13.1 / 14.6, 16.5 / 16.2, 20.7 / 17.8; 8 experts, 4,096 9.6 /
# 11.5, 10.9 / 12.9, 13.4 / 14.4; 32 experts, 1,024 10.3 / 10.5, 11.5 / 11.3, 14.1 / 11.3; 2,048 11.3 / 11.6, 13.6 / 12.1, 15.5 / 13.4; 4,096 14.8 /
# 14.0, 17.4 / 15.3, 21.9 / 17.0; 64 experts, 2,048 18.0 / 13.0, 20.7 / 13.6, 24.9 / 14.7; 8,192 35 / 17, 48 / 19, 61 / 20.
ROUTE_GROUP_PAYS_EXPERTS, ROUTE_GROUP_PAYS_K = 16, 4096


def route_group_pays(n_experts: int, k: int) -> bool:
    """Whether a step of few tokens makes logits, choices and lists of such a router faster in one launch than in three."""
    return n_experts <= ROUTE_GROUP_PAYS_EXPERTS and k % 32 == 0 and k <= ROUTE_GROUP_PAYS_K


def _route_checks(x, router_copy, bias, n_experts, top, scores, correction, scale, renormalize, groups) -> Tuple[int, int, int, int]:
    """(tokens, K, groups of experts, groups that stay open) of a router's launch after checking its arguments."""
    KernelError, _, _, _, _need_gpu, *_ = _base()
    _need_gpu(x, router_copy, bias, correction)
    _check_scores(scores, correction, scale, renormalize, n_experts)
    _, most_experts, most_k = route_group_limits()
    if x.dim() != 2 or x.dtype != torch.bfloat16 or x.stride(1) != 1:
        raise KernelError("x must be bfloat16 [T, K] with contiguous rows")
    n, k = x.shape
    if not 1 <= n_experts <= most_experts or k % 32 != 0 or k > most_k:
        raise KernelError(f"{n_experts} experts of rows of {k}: the kernel takes up to {most_experts}, rows of a multiple of 32 up to {most_k}")
    if router_copy.dtype != torch.bfloat16 or tuple(router_copy.shape) != (-(-n_experts // 16), k // 32, 64, 8) or not router_copy.is_contiguous():
        raise KernelError(f"the router's streaming copy {tuple(router_copy.shape)} does not fit {n_experts} experts of rows of {k}")
    if bias is not None and (bias.dtype != torch.float32 or bias.shape != (n_experts,) or not bias.is_contiguous()):
        raise KernelError("the router's bias must be a contiguous float32 tensor, one value an expert")
    if not 1 <= top <= min(n_experts, MAX_ROUTE_TOP):
        raise KernelError(f"{top} of {n_experts} experts: the kernel takes 1..{min(n_experts, MAX_ROUTE_TOP)}")
    count, keep = _open_groups(groups, n_experts, top)
    return n, k, count, keep


def route_rows_pays(n_tokens: int, k: int) -> bool:
    """Whether so many tokens' logits and choices are made faster in one launch than as a product and its choice.  The product reads x once
    whatever the number of tokens; the one launch is ahead by what a launch costs, for 2 to 16 experts up to 4,096 tokens (us, product / one launch, 16
    experts of 2,048: 17 tokens 8.6 / 6.0, 2,048 8.3 / 6.4) and with rows of up to 1,536 to 8,192; of 2,048 and more 6,000 tokens take 9.2 / 9.9 (2
    experts) to 13.0 / 13.6 (16 of 3,072), 16,384 17 to 18.5 / 19 to 20 and 65,536 of 3,072 84 to 98 / 115 to 119."""
    return n_tokens <= (8192 if k <= 1536 else 4096)


def route_rows(
    x: torch.Tensor, router_copy: torch.Tensor, bias: Optional[torch.Tensor], n_experts: int, top: int, scores: str = "softmax_chosen",
    correction: Optional[torch.Tensor] = None, scale: float = 1.0, renormalize: bool = False, groups: Optional[Tuple[int, int]] = None,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """A router's logits (bfloat16 x [T, K], its streaming copy, `bias` float32 [E] or None) and the choice of `route_top` in one launch, a
    block for every 16 tokens: (chosen, weights).  The logits' sums are those of `route_and_group`."""
    KernelError, _check, _code, _i32, _need_gpu, _ptr, _stream = _base()
    n, k, count, keep = _route_checks(x, router_copy, bias, n_experts, top, scores, correction, scale, renormalize, groups)
    chosen = torch.empty((n, top), dtype=torch.int32, device=x.device)
    weights = torch.empty((n, top), dtype=torch.float32, device=x.device)
    lib = _build.load("routed")
    _check(
        lib,
        lib.cwm_route_rows(
            _ptr(x), ctypes.c_long(x.stride(0) if n > 1 else k), _ptr(router_copy), _ptr(bias), ctypes.c_int(k), ctypes.c_int(n), ctypes.c_int(n_experts),
            ctypes.c_int(top), ctypes.c_int(int(scores == "softmax_all")), _ptr(correction), ctypes.c_float(scale), ctypes.c_int(int(renormalize)),
            ctypes.c_int(count), ctypes.c_int(keep), _ptr(chosen), _ptr(weights), _stream(),
        ),
    )
    return chosen, weights


def route_and_group(
    x: torch.Tensor, router_copy: torch.Tensor, bias: Optional[torch.Tensor], n_experts: int, top: int, scores: str = "softmax_chosen",
    correction: Optional[torch.Tensor] = None, scale: float = 1.0, renormalize: bool = False, groups: Optional[Tuple[int, int]] = None,
) -> Tuple[torch.Tensor, torch.Tensor, ExpertGroups]:
    """(chosen, weights, lists): what `route_top` and `group_by_expert` make of the logits W x + bias, in one launch; the logits are added in the
    streaming product's order, so the bits are the same where that does not split K (up to 6,144).
    `x` bfloat16 [T <= 16, K] (K a multiple of 32, up to 8,192), `router_copy` the streaming copy (`stream_layout`) of the
    bfloat16 router [E <= 64, K], `bias` float32 [E] or None; the rest as in `route_top`."""
    KernelError, _check, _code, _i32, _need_gpu, _ptr, _stream = _base()
    if x.dim() == 2 and x.shape[0] > route_group_limits()[0]:
        raise KernelError(f"x must be bfloat16 [T <= {route_group_limits()[0]}, K] with contiguous rows")
    n, k, count, keep = _route_checks(x, router_copy, bias, n_experts, top, scores, correction, scale, renormalize, groups)
    chosen = torch.empty((n, top), dtype=torch.int32, device=x.device)
    weights = torch.empty((n, top), dtype=torch.float32, device=x.device)
    lists = _empty_groups(n, top, n_experts, x.device)
    lib = _build.load("routed")
    _check(
        lib,
        lib.cwm_route_group(
            _ptr(x), ctypes.c_long(x.stride(0) if n > 1 else k), _ptr(router_copy), _ptr(bias), ctypes.c_int(k), ctypes.c_int(n), ctypes.c_int(n_experts),
            ctypes.c_int(top), ctypes.c_int(int(scores == "softmax_all")), _ptr(correction), ctypes.c_float(scale), ctypes.c_int(int(renormalize)),
            ctypes.c_int(count), ctypes.c_int(keep), _ptr(chosen), _ptr(weights), _ptr(lists.row_token), _ptr(lists.pair_row), _ptr(lists.tile_expert),
            _ptr(lists.used), ctypes.c_int(lists.n_tiles), ctypes.c_int(lists.tiles_a_block), _stream(),
        ),
    )
    return chosen, weights, lists


def group_by_expert(chosen: torch.Tensor, n_experts: int) -> ExpertGroups:
    """Group the pairs of `chosen` (int32 [T, top]) by expert.  The lists have a size that depends on T, top and
    the number of experts alone, so no count has to come to the host."""
    KernelError, _check, _code, _i32, _need_gpu, _ptr, _stream = _base()
    _need_gpu(chosen)
    _i32(chosen, "chosen")
    if chosen.dim() != 2:
        raise KernelError("chosen must be [T, top]")
    if not 1 <= n_experts <= MAX_EXPERTS:
        raise KernelError(f"{n_experts} experts: the kernel takes up to {MAX_EXPERTS}")
    n, top = chosen.shape
    groups = _empty_groups(n, top, n_experts, chosen.device)
    n_tiles, align = groups.n_tiles, groups.tiles_a_block
    lib = _build.load("routed")
    _check(
        lib,
        lib.cwm_group_by_expert(
            _ptr(chosen), ctypes.c_int(n), ctypes.c_int(top), ctypes.c_int(n_experts), _ptr(groups.row_token), _ptr(groups.pair_row),
            _ptr(groups.tile_expert), _ptr(groups.used), ctypes.c_int(n_tiles), ctypes.c_int(align), _stream(),
        ),
    )
    return groups


def expert_tiles(weights: torch.Tensor) -> torch.Tensor:
    """The experts' matrices [E, N, K] (bfloat16, N a multiple of 16, K of 64) in operand tiles [E, N / 16, K / 32, 64, 8]: lane
    16 j + r of a step of 32 columns holds row r's columns 8 j .. 8 j + 7, as in `stream_layout`, so that a wavefront's load of an
    operand is 1 KB of consecutive memory instead of 16 rows' pieces of 64 bytes.  The grouped products take either form and
    give the same bits."""
    from . import stream_layout

    KernelError = _base()[0]
    if weights.dim() != 3 or weights.dtype != torch.bfloat16 or not weights.is_contiguous() or weights.shape[1] % 16 or weights.shape[2] % 64:
        raise KernelError(f"operand tiles are made of contiguous bfloat16 [E, N, K] with N a multiple of 16 and K of 64, not {tuple(weights.shape)} {weights.dtype}")
    e, n, k = weights.shape
    return stream_layout(weights.view(e * n, k)).view(e, n // 16, k // 32, 64, 8)


def _weight_shape(w: torch.Tensor) -> Tuple[int, int, int]:
    """(experts, N, K) of grouped weights in either form."""
    return (w.shape[0], 16 * w.shape[1], 32 * w.shape[2]) if w.dim() == 5 else tuple(w.shape)


def _grouped(
    a: torch.Tensor, a_ld: int, a_batch: int, groups: Optional[ExpertGroups], w0: torch.Tensor, w1: Optional[torch.Tensor],
    out: torch.Tensor, out_ld: int, out_batch: int, n_rows: int, n_batch: int,
    activation: Optional["GatedActivation"] = None, gather: bool = True,
) -> None:
    """`gather`: `a` has the tokens' rows, which the list picks; else it has the list's own rows."""
    KernelError, _check, _code, _i32, _need_gpu, _ptr, _stream = _base()
    _need_gpu(a, w0, w1, out)
    tiled = w0.dim() == 5
    if (
        not (w0.dim() == 3 or (tiled and tuple(w0.shape[3:]) == (64, 8) and w0.shape[2] % 2 == 0 and w0.dtype == torch.bfloat16))
        or not w0.is_contiguous() or w0.dtype != a.dtype or (w1 is not None and (w1.shape != w0.shape or not w1.is_contiguous() or w1.dtype != a.dtype))
    ):
        raise KernelError("grouped weights must be contiguous [experts, N, K] tensors of the rows' type, or bfloat16 in operand tiles (`expert_tiles`)")
    e, n, k = _weight_shape(w0)
    if tiled and a.data_ptr() % 16 != 0:
        a = a.clone()  # the kernels that read operand tiles take rows at multiples of 16 bytes
    if groups is not None:
        if groups.tile_expert.numel() < groups.n_tiles or groups.row_token.numel() < groups.n_tiles * TILE_ROWS:
            raise KernelError(f"lists of {groups.tile_expert.numel()} tiles and {groups.row_token.numel()} rows do not hold {groups.n_tiles} tiles")
        tiles_a_block = min(groups.tiles_a_block, _product_tiles(a.dtype, k, groups.pair_row.numel() / e, w1 is not None))
    else:  # a product a head: few rows go through the weights' stream
        tiles_a_block = _product_tiles(a.dtype, k, n_rows, False) if n_rows >= MEDIUM_ROWS else 1
    lib = _build.load("routed")
    _check(
        lib,
        lib.cwm_grouped_product(
            _ptr(a), ctypes.c_long(a_ld), ctypes.c_long(a_batch), ctypes.c_int(_code(a.dtype)),
            _ptr(groups.row_token if groups is not None and gather else None), _ptr(w0), _ptr(w1), ctypes.c_long(n * k),
            _ptr(groups.tile_expert if groups is not None else None), _ptr(groups.used if groups is not None else None), ctypes.c_int(groups.n_tiles if groups is not None else 0),
            ctypes.c_int(n_batch), _ptr(out), ctypes.c_int(_code(out.dtype)), ctypes.c_long(out_ld), ctypes.c_long(out_batch),
            ctypes.c_int(n_rows), ctypes.c_int(n), ctypes.c_int(k), ctypes.c_int(tiles_a_block),
            ctypes.c_int(groups.tiles_a_block if groups is not None else 1),
            ctypes.c_int(activation.code() if activation is not None else 0), ctypes.c_float(activation.alpha if activation is not None else 1.0),
            ctypes.c_float(activation.limit if activation is not None else 0.0), ctypes.c_int(int(tiled)),
            ctypes.c_int(int(groups is not None and _loop_pays(groups.pair_row.numel(), e, n, k, w1 is not None))), _stream(),
        ),
    )


@dataclass(frozen=True)
class GatedActivation:
    """What a gated feed-forward makes of g = W_gate x and u = W_up x.
    "silu": silu(g) * u.
    "clamped_swish": g' * sigmoid(alpha * g') * (u' + 1) with g' = min(g, limit) and u' = clamp(u, -limit, limit).
    "gelu_tanh": gelu(g) * u with the tanh form of gelu."""

    kind: str = "silu"
    alpha: float = 1.0
    limit: float = 0.0

    def code(self) -> int:
        kinds = {"silu": 0, "clamped_swish": 1, "gelu_tanh": 2}
        if self.kind not in kinds:
            raise ValueError(f"gated activation {self.kind!r}: known are {', '.join(kinds)}")
        return kinds[self.kind]


def grouped_gate_up(
    x: torch.Tensor, groups: ExpertGroups, gate: torch.Tensor, up: torch.Tensor, activation: Optional[GatedActivation] = None
) -> torch.Tensor:
    """act(W_gate,e x_t, W_up,e x_t) for every pair's row, act = silu(g) * u unless `activation` says otherwise:
    `x` [T, D] contiguous, weights [E, F, D]; returns [rows, F] in the type of `x` (rows of the padding are not
    written)."""
    KernelError = _base()[0]
    _, hidden, dim = _weight_shape(gate)
    if x.dim() != 2 or not x.is_contiguous() or dim != x.shape[1]:
        raise KernelError("x must be a contiguous [T, D] tensor that fits the experts' weights")
    out = torch.empty((groups.n_tiles * TILE_ROWS, hidden), dtype=x.dtype, device=x.device)
    _grouped(x, x.shape[1], 0, groups, gate, up, out, hidden, 0, groups.n_tiles * TILE_ROWS, 1, activation)
    return out


def grouped_linear(rows: torch.Tensor, groups: ExpertGroups, weight: torch.Tensor) -> torch.Tensor:
    """W_e row for every row of the list (`rows` [rows, F] as `grouped_gate_up` leaves them, `weight` [E, D, F]):
    float32 [rows, D]."""
    KernelError = _base()[0]
    _, dim, hidden = _weight_shape(weight)
    if rows.dim() != 2 or not rows.is_contiguous() or hidden != rows.shape[1] or rows.shape[0] != groups.n_tiles * TILE_ROWS:
        raise KernelError("the rows do not fit the list or the experts' weights")
    out = torch.empty((rows.shape[0], dim), dtype=torch.float32, device=rows.device)
    _grouped(rows, rows.shape[1], 0, groups, weight, None, out, dim, 0, rows.shape[0], 1, gather=False)
    return out


def combine_routed(rows: torch.Tensor, groups: ExpertGroups, weights: torch.Tensor) -> torch.Tensor:
    """out[t] = sum_k weights[t, k] * rows[row of pair (t, k)], added in the order of k: float32 [T, D]."""
    KernelError, _check, _code, _i32, _need_gpu, _ptr, _stream = _base()
    _need_gpu(rows, weights)
    if rows.dtype != torch.float32 or rows.dim() != 2 or not rows.is_contiguous():
        raise KernelError("the experts' rows must be a contiguous float32 tensor")
    if weights.dtype != torch.float32 or weights.dim() != 2 or not weights.is_contiguous() or weights.shape[1] != groups.top:
        raise KernelError("weights must be float32 [T, top]")
    n, top = weights.shape
    out = torch.empty((n, rows.shape[1]), dtype=torch.float32, device=rows.device)
    lib = _build.load("routed")
    _check(
        lib,
        lib.cwm_combine_routed(_ptr(rows), ctypes.c_long(rows.shape[1]), _ptr(groups.pair_row), _ptr(weights), _ptr(out), ctypes.c_int(n), ctypes.c_int(top), ctypes.c_int(rows.shape[1]), _stream()),
    )
    return out


def absorb_queries(rest: torch.Tensor, ask: torch.Tensor, lead: int, weight: torch.Tensor) -> torch.Tensor:
    """Per head h: ask[t, h, lead + j] = sum_d weight[h, j, d] * rest[t, h, d]; the leading elements of `ask` stay as they are.
    `rest` [T, H, d] (heads and tokens may lie apart), `ask` [T, H, lead + n] contiguous, `weight` [H, n, d]; returns `ask`."""
    KernelError = _base()[0]
    n_tokens, heads, width = ask.shape
    if not ask.is_contiguous() or weight.dim() != 3 or weight.shape[0] != heads or weight.shape[1] != width - lead or ask.dtype != rest.dtype:
        raise KernelError(f"the heads' weights {tuple(weight.shape)} do not fill rows {tuple(ask.shape)} from element {lead} on")
    if rest.dim() != 3 or tuple(rest.shape) != (n_tokens, heads, weight.shape[2]) or rest.stride(2) != 1:
        raise KernelError(f"unrotated parts {tuple(rest.shape)} do not fit the heads' weights {tuple(weight.shape)}")
    if n_tokens:
        _grouped(rest, max(rest.stride(0), heads * rest.shape[2]), rest.stride(1), None, weight, None, ask.view(-1)[lead:], heads * width, width, n_tokens, heads)
    return ask


def expand_values(mixed: torch.Tensor, lead: int, weight: torch.Tensor) -> torch.Tensor:
    """Per head h: out[t, h, :] = weight[h] applied to mixed[t, h, lead:], i.e. out[t, h, v] = sum_j weight[h, v, j] * mixed[t, h, lead + j].
    `mixed` [T, H, lead + n] contiguous, `weight` [H, v, n]; returns [T, H * v]."""
    KernelError = _base()[0]
    if mixed.dim() != 3 or not mixed.is_contiguous() or weight.dim() != 3 or weight.shape[0] != mixed.shape[1] or weight.shape[2] != mixed.shape[2] - lead:
        raise KernelError(f"rows {tuple(mixed.shape)} do not fit the heads' weights {tuple(weight.shape)} after {lead} leading elements")
    n_tokens, heads, width = mixed.shape
    v = weight.shape[1]
    out = torch.empty((n_tokens, heads * v), dtype=mixed.dtype, device=mixed.device)
    if n_tokens:
        _grouped(mixed.view(-1)[lead:], heads * width, width, None, weight, None, out, heads * v, v, n_tokens, heads)
    return out
