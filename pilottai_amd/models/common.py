"""What the model families beside Llama share: packed projections, checkpoint access, looped stacks."""
from __future__ import annotations

import os
from typing import Callable, List, Optional, Tuple

import torch
import torch.nn.functional as F

from pilottai_amd import ops
from pilottai_amd.ops.latent import pad_to


class PackedLinear:
    """y = x W^T with W [N, K] padded to [128 n, 64 k] by zeros: the packed projections in bf16
    (decode kernels up to 64 rows and where rows_gemm_pays, prefill kernel above), the library's fp32 GEMM in fp32."""

    def __init__(self, w: torch.Tensor, dtype, device):
        N, K = w.shape
        full = torch.zeros(pad_to(N, 128), pad_to(K, 64), dtype=dtype, device=device)
        full[:N, :K] = w.to(device=device, dtype=dtype)
        self.N, self.K = full.shape
        self.w = ops.pack_decode_weight(full) if dtype == torch.bfloat16 else full

    def __call__(self, x: torch.Tensor, live: Optional[torch.Tensor] = None) -> torch.Tensor:
        """`live`: see ops.prefill_gemm."""
        if self.w.dim() == 2:
            return F.linear(x, self.w)
        if x.shape[0] <= 64:
            return ops.decode_gemm(x, self.w)
        y = ops.rows_gemm(x, self.w) if ops.rows_gemm_pays(x.shape[0], self.w.shape[0] * 16, x.shape[1]) else None
        return ops.prefill_gemm(x, self.w, live=live) if y is None else y

    def parts(self, x: torch.Tensor, live: Optional[torch.Tensor] = None):
        """(y, n) for a reader that adds up n rows of y a row: unrounded parts (fp32) where they are the faster form, else y itself."""
        n = ops.rows_sums_slices(x.shape[0], self.N, self.K) if self.w.dim() == 4 and x.is_cuda else 1
        return (self(x, live), 1) if n == 1 else (ops.rows_sums(x, self.w, n), n)


def pad_heads(w: torch.Tensor, padded: int) -> torch.Tensor:
    """[heads, size, k] -> [heads, padded, k], zeros behind every head."""
    out = w.new_zeros(w.shape[0], padded, w.shape[2])
    out[:, :w.shape[1]] = w
    return out


def checkpoint_reader(path: str) -> Callable:
    """get(name, shape) over a folder's *.safetensors, checking that the tensor is there and has the shape; get.shape(name)
    for a size that no configuration gives."""
    from safetensors import safe_open

    where = {}
    for f in sorted(os.listdir(path)):
        if f.endswith(".safetensors"):
            fh = safe_open(os.path.join(path, f), framework="pt")
            where.update({k: fh for k in fh.keys()})

    def file(name):
        if name not in where:
            raise ValueError(f"{path}: tensor {name!r} is missing")
        return where[name]

    def get(name, shape):
        t = file(name).get_tensor(name)
        if tuple(t.shape) != tuple(shape):
            raise ValueError(f"{path}: {name} has shape {tuple(t.shape)}, the configuration gives {tuple(shape)}")
        return t
    get.shape = lambda name: tuple(file(name).get_slice(name).get_shape())
    return get


def parse_loop(loop: Optional[dict], layers: int) -> Optional[Tuple[int, int, int]]:
    """(start, stop, times) of a config's loop entry."""
    if not loop:
        return None
    out = (int(loop["start"]), int(loop["stop"]), int(loop["times"]))
    if not (0 <= out[0] < out[1] <= layers and out[2] >= 1):
        raise ValueError(f"loop {out} does not fit {layers} layers")
    return out


def layer_runs(layers: int, loop: Optional[Tuple[int, int, int]]) -> List[Tuple[int, bool]]:
    """(layer, whether a repeated pass starts here) for every layer run of a step, in order."""
    start, stop, times = loop or (0, 0, 1)
    out = []
    for again in range(times):
        lo = start if again else 0
        out += [(i, again > 0 and i == start) for i in range(lo, stop)]
    return out + [(i, False) for i in range(stop, layers)]


# (most rows a group has on average, rows per sorted tile) of the grouped projections: the fewest that hold a group's rows,
# with room for uneven groups, so that its weights are read once; above, 256 (the ping-pong kernels, whose MFMAs end with a
# tile's last 64 rows). us of both products, weights cold: 64 experts of 3 x 1408 x 2048, 6 rows an expert 16: 180, 32: 189;
# 14 rows 16: 203, 32: 194, 256: 201; 28 rows 32: 223, 64: 211, 256: 203; 94 rows 64: 289, 128: 253, 256: 225; 8 of 3 x 14336
# x 4096, 16 rows 16: 579, 32: 460, 256: 513; 37 rows 32: 744, 64: 519, 256: 529; 75 rows 64: 713, 128: 727, 256: 556. Of few
# inputs 16 rows go further (64 of 3 x 192 x 512, 14 rows 16: 16.1, 32: 17.8, 256: 18.6; 28 rows 32: 19.6, 64: 22.9, 256: 19.0).
GROUP_TILES, SHORT_GROUP_TILES = ((10, 16), (24, 32)), ((16, 16), (24, 32))
# of one group (gate and up of a dense unit): 64 rows share the weights through the caches of an XCD up to 448 rows (2 x 8192
# x 2048: 44 us at 400 rows, 256-row tiles 47), with weights above 128 MB up to 128 (2 x 14336 x 4096: 66 us at 100 rows, 81;
# 256 rows 89, 88); weights below 32 MB, whose 64-row tiles are few workgroups, take 32 up to 64 rows (2 x 4096 x 1024: 8.9 us
# at 64 rows, 64-row tiles 10.9; 2 x 8192 x 2048 23, 21)
ONE_SMALL_GROUP_TILES, ONE_GROUP_TILES = ((16, 16), (64, 32), (448, 64)), ((16, 16), (32, 32), (448, 64))
ONE_LARGE_GROUP_TILES = ((16, 16), (32, 32), (128, 64))


def expert_tile_rows(rows: float, dtype, min_k: int, steps=None) -> int:
    """Rows per sorted tile by the rows a group gets on average (fp32: 16; the 256-row kernels take every K of 128 on)."""
    if dtype != torch.bfloat16:
        return 16
    if steps is None:
        steps = GROUP_TILES if min_k > 256 else SHORT_GROUP_TILES
    return next((tm for most, tm in steps if rows <= most), 256 if min_k >= 128 else 64)
