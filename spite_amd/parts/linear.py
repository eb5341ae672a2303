"""Matrix products of the parts: picks the kernel for the dtypes and shapes at hand.

``Y = X . W^T`` with W ``[out, in]``; the grouped form walks a row list (see
``gemm_generic.hip``).  A weight that stayed in 32-bit inside a bfloat16 run is multiplied in
32-bit: the activations are widened for that product.
"""
from __future__ import annotations

import functools
import math
from typing import List

import torch

from ..csrc import hipops


def _scratch(ws, shape, dtype, device):
    """From the step's workspace when the caller has one (a warmed-up engine then allocates
    nothing inside a step), else a fresh tensor."""
    return ws.take(tuple(shape), dtype) if ws is not None else torch.empty(tuple(shape), dtype=dtype, device=device)


def _widen(x, ws=None):
    y = _scratch(ws, x.shape, torch.float32, x.device)
    hipops.convert(x, y)
    return y


SKINNY_MAX_ROWS = 64


class Weight:
    """A weight as the product kernels want it.  bfloat16 matrices whose rows are a multiple of
    16 and whose columns a multiple of 64 are kept in MFMA operand order (``hipops.operand_order``:
    a wave's operand load is then one run of whole cache lines, which the prefill products are
    bound by); everything else stays row-major.  ``shape`` is the logical ``[..., out, in]``."""

    __slots__ = ("data", "tiled", "shape", "dtype")

    def __init__(self, w: torch.Tensor, allow_tiled: bool = True):
        w = w.contiguous()
        self.shape, self.dtype = tuple(w.shape), w.dtype
        self.tiled = bool(allow_tiled and w.dtype == torch.bfloat16 and w.dim() >= 2 and w.is_cuda
                          and w.shape[-2] % 16 == 0 and w.shape[-1] % 64 == 0)
        self.data = hipops.operand_order(w) if self.tiled else w

    def slow_reason(self, name: str) -> List[str]:
        """Why products with this weight will not run on the matrix units in a bfloat16 run."""
        if self.dtype == torch.bfloat16 and self.shape[-1] % 8:
            return [f"{name} {self.shape}: rows of {self.shape[-1]} are no multiple of 8, its products run on plain FMAs"]
        if self.dtype == torch.float32:
            return [f"{name} {self.shape}: kept in 32-bit by the checkpoint, and so are its products"]
        return []

    def group(self, g: int) -> "Weight":
        """Group ``g`` of a stack of matrices ``[groups, out, in]`` as a weight of its own (the same
        memory)."""
        one = object.__new__(Weight)
        one.data, one.tiled, one.shape, one.dtype = self.data[g], self.tiled, self.shape[1:], self.dtype
        return one


# what a tile of 160 rows costs against one of 128 (a tile's time is a fixed part and a part per
# 16 rows, 38 and 8.5 us at K = 5,120 on an MI355X: (38 + 85) / (38 + 68))
TILE_160_COST = 1.16


def grouped_tile_shape(tokens: int, groups: int, whole_groups: int = 0, col_tiles: int = 0, cus: int = 0) -> int:
    """Which tile of ``gemm_tiled`` suits ``tokens`` rows that spread evenly over ``groups``
    groups (experts that a router picks), beside ``whole_groups`` groups that take every row.
    A group costs whole row tiles, each of which streams the group's weights once.  (The product
    then takes that tile only where ``linear`` estimates no other kernel to be the faster one:
    ``hipops.gemm_groups_choice`` weighs the tiles of several heights against it.)

    * Few rows a group and few groups (a short prompt over a few experts): the time is the stream
      of the weights from memory and there are too few workgroups to keep it busy; the 64-row
      tile with its deeper run of loads (shape 4) streams faster, as long as the groups that take
      every row do not need many of those small tiles.  (With 128 experts there are workgroups
      enough: measured no gain.)
    * Else 128 rows a tile (shape 1), or 160 (shape 3, about a sixth dearer per tile) where that
      saves time: with groups of about 128 rows half of them need a second tile of 128, almost
      none a second one of 160.  The expected number of row tiles of each shape, group sizes
      taken as normal around tokens/groups, times ``col_tiles`` column tiles, runs on ``cus``
      compute units in whole rounds (a workgroup a unit): the fewer rounds, each at its tile's
      cost, win.  (Measured at widths of 4,096 to 6,144, 8 and 16 experts of 8,192 and 14,336:
      the choice by rounds was the faster tile in all eight products.)  Without ``col_tiles`` the
      row tiles alone are compared."""
    if groups <= 0 or tokens <= 0:
        return 1
    mean, sd = _group_size(tokens, groups)
    if groups <= 32 and mean + 4.0 * sd <= 64.0 and whole_groups * -(-tokens // 64) <= 0.25 * groups:
        return 4
    if col_tiles > 0:
        return _rounds(tokens, groups, whole_groups, col_tiles, cus or hipops.cu_count())[0]
    tiles = lambda rows: _row_tiles(tokens, groups, whole_groups, rows)
    return 3 if 1.17 * tiles(160) < tiles(128) else 1


def _group_size(tokens, groups):
    """Mean and standard deviation of a group's rows."""
    return tokens / groups, max(math.sqrt(tokens * (1.0 / groups) * (1.0 - 1.0 / groups)), 1e-6)


def _row_tiles(tokens, groups, whole_groups, rows_per_tile, deviations=0.0):
    """The row tiles to expect, and so many standard deviations more (each further tile of a group comes or does not)."""
    mean, sd = _group_size(tokens, groups)
    extra, spread, k = 0.0, 0.0, 1
    while k * rows_per_tile < mean + 6 * sd:
        p = 0.5 * math.erfc((k * rows_per_tile + 0.5 - mean) / (sd * math.sqrt(2.0)))
        extra, spread, k = extra + p, spread + p * (1.0 - p), k + 1
    return groups * (1.0 + extra) + deviations * math.sqrt(groups * spread) + whole_groups * -(-tokens // rows_per_tile)


def _rounds(tokens, groups, whole_groups, col_tiles, cus, deviations=0.0, full=1.0):
    """(tile shape, its rounds over the chip times its tile's cost); ``full``: how much of a round may be counted on."""
    rounds = lambda rows: math.ceil(_row_tiles(tokens, groups, whole_groups, rows, deviations) * col_tiles / (full * cus) - 1e-9)
    wide, narrow = TILE_160_COST * rounds(160), float(rounds(128))
    return (3, wide) if wide < narrow else (1, narrow)


@functools.lru_cache(maxsize=4096)
def whole_group_apart(tokens: int, groups: int, N: int, K: int) -> int:
    """Whether a plain product over ``groups`` groups that ``tokens`` rows spread over and one group that takes every row
    is better done as two: the groups (the result is the tile shape that they then take, 0: together), and the one as a
    product of its own.  Together the tiles of the second kind fill the first one's last round; apart it may need one round
    fewer, and each has the kernel that suits it.  The price is ``gemm_tiled``'s: a round takes 146 us at K = 5,120 and the groups no
    less than their weights at 5.6 TB/s; the tiles of several heights that the products may take instead (``gemm_groups``) move both sides
    by less than the margins.  Routers do not spread their rows quite evenly, and a round that the groups miss by a tile costs more
    than is to be gained: with a standard deviation of tiles more they have to fit 85 % of their rounds, and the two to be 6 % faster
    than all tiles together with a deviation fewer.
    (Measured with whichever kernel each product then takes, at 420 sizes, 4 to 32 experts, 130 to 6,000 tokens: of the 30 that this takes
    in 7 are 2 % and more slower apart, most of them by 7, on average they are 4 % faster; never apart loses 46 of the 420 to what
    they took with gemm_tiled alone, this 30, and the estimates of those kernels, tried in its place, 36 to 49.  5,120 x 8,192 over 16
    experts, together / apart: 1,547 tokens 428 / 360 us, 1,685 408 / 371, 2,048 462 / 433; over 8: 1,629 367 / 322, 1,743 360 / 339; 3,072
    x 8,192 over 16: 3,192 401 / 378, over 32: 1,865 406 / 379.)  A gated product's rounds are many and its stream of weights long: there
    it never paid (2,048 tokens 719 / 759)."""
    cus, round_us, cols = hipops.cu_count(), 146.0 * K / 5120.0, -(-N // 512)
    together = round_us * _rounds(tokens, groups, 1, cols, cus, deviations=-1.0)[1]
    shape, cost = _rounds(tokens, groups, 0, cols, cus, deviations=1.0, full=0.85)
    routed = max(round_us * cost, groups * N * K * 2 / 5.6e6)
    return shape if routed + hipops.lds_us(tokens, N, K, False) < 0.94 * together else 0


def _routed_and_whole(M, n_groups, most, group_rows):
    """A routed group's rows on average and how many groups take every row: what the rows of the call leave over the routed
    ones' (arguments as ``linear``'s)."""
    mean = M / n_groups if group_rows is None else group_rows
    return mean, min(max(round((M - n_groups * mean) / (most - mean)), 0), n_groups - 1) if most > mean else 0


def _group_tiles(M, n_groups, most, group_rows, N, glu):
    """The tiles of ``gemm_tiled`` and of ``gemm_lds`` to expect of a product over groups (arguments as ``linear``'s)."""
    mean, whole = _routed_and_whole(M, n_groups, most, group_rows)
    tiles = lambda rows, cols: ((n_groups - whole) * math.ceil(mean / rows) + whole * -(-most // rows)) * -(-N // cols)
    return tiles(128, 256 if glu else 512), tiles(256, 128 if glu else 256)


def linear(x, w, y, *, glu=False, offsets=None, n_groups=1, a_rows=None, a_scale=None, y_rows=None, rows=None,
           max_rows=None, tile_shape=0, live_groups=0, group_rows=None, ws=None, act=None):
    """y[r] = W . x[r] for ``rows`` rows (default: all of x; for a row list: its length).

    With ``glu`` the weight holds gate rows then up rows and y = act(gate) * up: ``True`` or
    ``"silu"``, ``"gelu_tanh"``, ``"relu"`` or ``("clamped", limit)`` (``hipops.gate_code``).
    ``max_rows``: the most rows that one group can bring (default: ``rows``).
    ``tile_shape``: the prefill product's tile (``grouped_tile_shape``), 0 = the library's choice.
    ``live_groups``: a promise that at most this many groups hold rows (0: none).
    ``group_rows``: the rows of a routed group on average, beside which other groups may take every row
    (default: all groups alike).
    ``ws``: the workspace that temporaries (partial sums, widened rows) are taken from.
    ``act``: an activation on a plain product's result (``gelu``, ``gelu_tanh``, ``silu``; not beside
    ``glu``): in the epilogue of the bfloat16 weight-stream and tiled products, a pass of its own after
    the others."""
    tiled = False
    if isinstance(w, Weight):
        w, tiled = w.data, w.tiled
    glu, limit = hipops.gate_code(glu)   # the gate's activation and its bound
    K = x.shape[-1]
    N = y.shape[-1]
    M = rows if rows is not None else x.shape[0]
    most = max_rows if max_rows is not None else M
    if x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and K % 8 == 0 and x.stride(0) % 8 == 0 \
            and x.data_ptr() % 16 == 0:
        if tiled and M > 32 and tile_shape == 0 and offsets is None and a_rows is None and a_scale is None and y_rows is None and act is None \
                and not glu and hipops.gemm_groups_ok(x, y, M, N, K, glu):
            choice = hipops.gemm_runs_choice(M, N, K)
            if choice is not None:
                runs, nb = choice
                part = _scratch(ws, (runs, M, N), torch.float32, x.device) if runs > 1 else None
                hipops.gemm_runs(x, w, y, M, N, K, runs=runs, nb=nb, part=part)
                return
        # few rows: the time is the weights' stream (a very tall matrix, the output table, is
        # streamed faster by the tiled kernel from 33 rows on)
        if most <= SKINNY_MAX_ROWS and not (tiled and most > 32 and offsets is None and N >= 65536):
            hipops.gemm_skinny(x, w, y, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows,
                               a_scale=a_scale, y_rows=y_rows, glu=glu, max_rows=most, tiled=tiled,
                               live_groups=live_groups, act=act, act_limit=limit)
            return
        if tiled:
            splits = offsets is None and a_rows is None and a_scale is None and y_rows is None and not glu and act is None
            runs = hipops.tiled_k_runs(M, N, K) if splits and tile_shape == 0 and M > 0 else 1
            lds = M > 0 and hipops.gemm_lds_ok(x, w, M, N, K, glu) and (
                hipops.lds_suits(M, N, K, bool(glu), runs) if offsets is None
                else hipops.lds_suits_groups(M / n_groups if group_rows is None else group_rows, K,
                                             *_group_tiles(M, n_groups, most, group_rows, N, bool(glu))))
            if offsets is not None and M > 0 and act is None and hipops.gemm_groups_ok(x, y, M, N, K, glu):
                mean, whole = _routed_and_whole(M, n_groups, most, group_rows)
                sizes = (most, n_groups - whole, float(mean), whole, N, K)
                wide, rounds = (None, 0) if glu else hipops.gemm_groups_wide_estimate(*sizes, tile_shape, lds)
                if wide is not None:         # (where the groups are not as even as hoped for, they go to the product that follows)
                    others = _scratch(ws, (n_groups + 1,), torch.int32, x.device)
                    hipops.gemm_groups(x, w, y, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows, a_scale=a_scale,
                                       y_rows=y_rows, waves=wide[0], cap=wide[1], rounds=rounds, others=others)
                    offsets = others
                choice = hipops.gemm_groups_choice(*sizes, bool(glu), tile_shape, lds)
                if choice is not None:
                    hipops.gemm_groups(x, w, y, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows, a_scale=a_scale,
                                       y_rows=y_rows, glu=bool(glu), waves=choice[0], cap=choice[1])
                    return
            if lds:
                hipops.gemm_lds(x, w, y, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows, a_scale=a_scale,
                                y_rows=y_rows, glu=glu, act=act, act_limit=limit)
                return
            part = _scratch(ws, (runs, M, N), torch.float32, x.device) if runs > 1 else None
            hipops.gemm_tiled(x, w, y, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows, a_scale=a_scale,
                              y_rows=y_rows, glu=glu, shape=tile_shape, part=part, act=act, act_limit=limit)
            return
        hipops.gemm_mfma(x, w, y, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows, a_scale=a_scale,
                         y_rows=y_rows, glu=glu, act_limit=limit)
        _act_after(y, M, y_rows, act)
        return
    if tiled:
        raise hipops.KernelError("linear: a weight in operand order met an input that the MFMA products do not take")
    if w.dtype == torch.float32 and x.dtype != torch.float32:
        x32 = _widen(x, ws)
        if y.dtype == torch.float32:
            hipops.gemm_generic(x32, w, y, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows,
                                a_scale=a_scale, y_rows=y_rows, glu=glu, act_limit=limit)
            _act_after(y, M, y_rows, act)
        else:
            y32 = _scratch(ws, y.shape, torch.float32, y.device)
            hipops.gemm_generic(x32, w, y32, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows,
                                a_scale=a_scale, y_rows=y_rows, glu=glu, act_limit=limit)
            _act_after(y32, M, y_rows, act)
            hipops.convert(y32, y)
        return
    hipops.gemm_generic(x, w, y, M, N, K, offsets=offsets, n_groups=n_groups, a_rows=a_rows, a_scale=a_scale,
                        y_rows=y_rows, glu=glu, act_limit=limit)
    _act_after(y, M, y_rows, act)


def _act_after(y, M, y_rows, act):
    """The activation as a pass of its own over the product's rows (the kernels that have no epilogue for it)."""
    if act is None:
        return
    if y_rows is not None or not y.is_contiguous():
        raise hipops.KernelError("linear: an activation after a product wants its rows in a row")
    hipops.act_rows(y[:M], act)
