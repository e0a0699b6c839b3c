"""fp16 GEMM on MI355X (gfx950): the reference's `mma.py` surface over a hand-written HIP kernel.

  * ``_matmul_contiguous_kernel[grid](a, b, c, M, N, K, BLOCK_M=, BLOCK_N=, BLOCK_K=, GROUP_M=,
    USE_CACHE_EVICTION_HINTS=, num_warps=, num_stages=)`` writes C = A @ B (fp32 accumulation,
    fp16 result) into the caller's ``c``, as mma.py:8-52 does. The BLOCK_* values are hints: a
    built gfx950 tile with those sizes that divides the problem is used, otherwise the tuned tile
    for (M, N, K). The grid argument is accepted (and may be a callable) but the launch computes
    its own grid for the chosen tile.
  * ``_select_2d_contiguous_config(m, n, k)`` returns (BLOCK_M, BLOCK_N, BLOCK_K, GROUP_M,
    num_warps, num_stages) for gfx950 (num_warps = wavefronts per workgroup, num_stages = LDS
    buffers) and raises ValueError for exactly the shapes the reference rejects (mma.py:63-81).
  * ``_supports_contiguous_cache_eviction_hints(device)`` keeps the reference contract
    (mma.py:55-60): True when a GPU with compute capability major >= 8 is present (gfx950 reports
    9.5). The hint is accepted by the launcher; the gfx950 kernel's loads already stream through
    L2 with the XCD-grouped tile order.
"""
from __future__ import annotations

import functools
import logging

import torch

import gfx950_configs as cfgs
import hip_lib
from tuner import get_architecture

logger = logging.getLogger(__name__)


@functools.lru_cache(maxsize=1024)
def _gemm_tile(M: int, N: int, K: int, hint: tuple[int, int, int] | None,
               group_m: int | None) -> tuple[hip_lib.GemmTile, int]:
    """Tile and K splits of a launch with BLOCK_* hints; hints that name another tile than the one the
    selector gives are kept (no split). Nor is a product with N % 8 == 4 split: the launch refuses it, as
    its B rows are not 16-byte aligned, while the split-K entry would take them."""
    try:
        bm, bn, bk, waves, gm = cfgs.choose_gemm_tile(M, N, K, hint)
        default = hint is None or cfgs.choose_gemm_tile(M, N, K)[:4] == (bm, bn, bk, waves)
    except ValueError:
        # no built tile divides the shape: the kernel masks partial tiles (K % 8, N % 4 suffice)
        bm, bn, bk, waves, gm = cfgs.choose_gemm_tile_any(M, N, K)
        default = True
    tile, splits = (bm, bn, bk, waves), 1
    if default and N % 8 == 0:
        tile, splits = cfgs.choose_gemm_splits(M, N, K, tile)
    return hip_lib.GemmTile(*tile, int(group_m) if group_m else gm), splits


# choose_gemm_tile_any asks the library for every built tile and sorts the table: 30 us a call, three
# times the product itself at 1000x1004x1000
@functools.lru_cache(maxsize=1024)
def _gemm_tile_any(M: int, N: int, K: int) -> tuple[hip_lib.GemmTile, int]:
    bm, bn, bk, waves, gm = cfgs.choose_gemm_tile_any(M, N, K)
    tile, splits = cfgs.choose_gemm_splits(M, N, K, (bm, bn, bk, waves))
    return hip_lib.GemmTile(*tile, gm), splits


class _HipMatmulKernel:
    """``kernel[grid](a, b, c, M, N, K, **meta)`` launcher (mma.py:8-21 layout)."""

    __name__ = "_matmul_contiguous_kernel"
    _META = {"BLOCK_M", "BLOCK_N", "BLOCK_K", "GROUP_M", "USE_CACHE_EVICTION_HINTS", "num_warps", "num_stages",
             "debug"}

    def __repr__(self) -> str:
        return "<gfx950 HIP kernel _matmul_contiguous_kernel>"

    def __getitem__(self, grid):
        def launch(*args, **kwargs):
            return self._launch(grid, args, kwargs)

        return launch

    def _launch(self, grid, args, kwargs):
        if len(args) != 6:
            raise TypeError(f"_matmul_contiguous_kernel takes (a, b, c, M, N, K), got {len(args)} arguments")
        unknown = set(kwargs) - self._META
        if unknown:
            raise TypeError(f"_matmul_contiguous_kernel got unexpected keyword arguments {sorted(unknown)}")
        a, b, c = args[0:3]
        M, N, K = (int(x) for x in args[3:6])
        if callable(grid):
            grid(kwargs)
        for name, t, shape in (("a", a, (M, K)), ("b", b, (K, N)), ("c", c, (M, N))):
            if not isinstance(t, torch.Tensor) or t.shape != shape:
                raise ValueError(f"{name} must have shape {shape}")
            if t.dtype != torch.float16:
                raise ValueError(f"{name} must be float16 (got {t.dtype})")
            if not t.is_contiguous():
                raise ValueError(f"{name} must be contiguous row-major (mma.py indexes it as such)")
        hint = None
        if all(kwargs.get(key) is not None for key in ("BLOCK_M", "BLOCK_N", "BLOCK_K")):
            hint = (int(kwargs["BLOCK_M"]), int(kwargs["BLOCK_N"]), int(kwargs["BLOCK_K"]))
            if kwargs.get("num_warps") is not None:
                hint = (*hint, int(kwargs["num_warps"]))
        tile, splits = _gemm_tile(M, N, K, hint, kwargs.get("GROUP_M"))
        hip_lib.gemm_f16(a, b, c, tile, ksplits=splits)


_matmul_contiguous_kernel = _HipMatmulKernel()


def _supports_contiguous_cache_eviction_hints(device=None) -> bool:
    if not torch.cuda.is_available():
        return False
    major, _ = torch.cuda.get_device_capability(device)
    return major >= 8


def _select_2d_contiguous_config(m: int, n: int, k: int) -> tuple[int, int, int, int, int, int]:
    get_architecture()
    bm, bn, bk, waves, group_m = cfgs.choose_gemm_tile(int(m), int(n), int(k))
    return bm, bn, bk, group_m, waves, 2


def matmul(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """C = A @ B through the gfx950 kernel (convenience entry). Unlike the reference selector it
    accepts shapes no tile divides (K % 8 == 0 and N % 4 == 0; partial tiles are masked). When
    N % 8 == 4 the rows of B start on 8-byte boundaries: the kernel reads them in place (ldb4). Only a B
    whose first row is not 16-byte aligned is copied, into rows of N + 4 elements (its last 4 columns
    are never stored to C)."""
    a = a.contiguous()
    b = b.contiguous()
    M, K = a.shape
    _, N = b.shape
    c = torch.empty((M, N), device=a.device, dtype=torch.float16) if out is None else out
    tile, splits = _gemm_tile_any(M, N, K)
    if N % 8:
        if b.data_ptr() % 16:
            b_rows = torch.zeros((K, N + 4), device=b.device, dtype=b.dtype)
            b_rows[:, :N].copy_(b)
            b = b_rows[:, :N]
        hip_lib.gemm_f16(a, b, c, tile, ldb4=True, ksplits=splits)
        return c
    if not c.is_contiguous():
        raise ValueError("out must be contiguous row-major")
    hip_lib.gemm_f16(a, b, c, tile, ksplits=splits)
    return c


__all__ = [
    "_select_2d_contiguous_config",
    "_supports_contiguous_cache_eviction_hints",
    "_matmul_contiguous_kernel",
]
