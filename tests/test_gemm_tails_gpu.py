"""GEMM shapes no tile divides (tails): the gfx950 kernel masks partial tiles in M, N
and K (K % 8 == 0, N % 4 == 0). Checked against the exact oracle, with NaN in the row padding of A
(past K) and B (past N) to show those elements never reach valid outputs, and a sentinel in C's
padding to show nothing is stored outside [M, N)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import gfx950_configs as cfgs
import hip_lib
import mma
import oracle
from helpers import to_device

pytestmark = pytest.mark.gpu

# every built tile (16x16 and 32x32 MFMAs; compiler-scheduled and pipelined loops)
TILES = [(256, 256, 64, 8), (256, 256, 32, 8), (256, 128, 64, 8), (128, 256, 64, 8), (256, 256, 64, 4),
         (256, 256, 32, 4), (128, 128, 64, 4), (128, 128, 32, 4), (128, 64, 32, 4), (64, 256, 32, 4),
         (128, 128, 32, 8), (128, 64, 32, 8), (128, 64, 32, 16), (64, 64, 32, 8)]
# K from 1 to 32 slabs: up to 8 slabs the 128x128, 128x64 and 64x256 tiles launch their
# shallow-ring kernels (K=256 is the last such for BK=32, K=264 the first deep one).
SHAPES = [(100, 200, 72), (257, 260, 520), (33, 4, 8), (1000, 1004, 1000), (300, 512, 136), (260, 392, 256),
          (260, 392, 264)]


def _padded(x: np.ndarray, cols: int, fill: float) -> torch.Tensor:
    rows, n = x.shape
    buf = np.full((rows, cols), fill, dtype=np.float32)
    buf[:, :n] = x
    t = to_device(buf, torch.float16, "cuda:0")
    return t[:, :n]  # row-major view with leading dimension `cols`


@pytest.mark.parametrize("shape", SHAPES, ids=[f"{m}x{n}x{k}" for m, n, k in SHAPES])
def test_gemm_tails_all_tiles(gpu, shape):
    M, N, K = shape
    print(f"[gemm_tails] M={M} N={N} K={K}", flush=True)
    a = oracle.round_to(oracle.portable_uniform(21, (M, K), -1, 1), 0)
    b = oracle.round_to(oracle.portable_uniform(22, (K, N), -1, 1), 0)
    ref = oracle.gemm(a, b)
    ad = _padded(a, K + 24, np.nan)                 # NaN past K in every A row (lda % 8 == 0)
    bd = _padded(b, -(-N // 8) * 8 + 8, np.nan)     # NaN past N in every B row (ldb % 8 == 0)
    sentinel = 1234.0
    cbuf = torch.full((M, N + 8), sentinel, dtype=torch.float16, device="cuda:0")
    cd = cbuf[:, :N]
    for tile in TILES:
        cbuf.fill_(sentinel)
        hip_lib.gemm_f16(ad, bd, cd, hip_lib.GemmTile(*tile, 4))
        torch.cuda.synchronize()
        c = cd.float().cpu().numpy()
        assert np.isfinite(c).all(), tile
        rel = float(np.linalg.norm(c - ref) / np.linalg.norm(ref))
        assert rel <= 1e-3, (tile, rel)
        assert bool((cbuf[:, N:] == sentinel).all()), tile


@pytest.mark.parametrize("shape", [(777, 1032, 264), (300, 100, 64), (65, 1028, 520)],
                         ids=["n_mod8_0", "n_mod8_4", "n_mod8_4_deep"])
def test_gemm_tails_convenience_entry(gpu, shape):
    """mma.matmul takes tail shapes (the reference selector still raises for them), N % 8 == 4
    included (B is read in place, its rows on 8-byte boundaries)."""
    M, N, K = shape
    print(f"[gemm_tails] mma.matmul {M}x{N}x{K}", flush=True)
    with pytest.raises(ValueError):
        mma._select_2d_contiguous_config(M, N, K)
    a = oracle.round_to(oracle.portable_uniform(31, (M, K), -1, 1), 0)
    b = oracle.round_to(oracle.portable_uniform(32, (K, N), -1, 1), 0)
    c = mma.matmul(to_device(a, torch.float16, "cuda:0"), to_device(b, torch.float16, "cuda:0"))
    torch.cuda.synchronize()
    assert c.is_contiguous() and tuple(c.shape) == (M, N)
    ref = oracle.gemm(a, b)
    assert float(np.linalg.norm(c.float().cpu().numpy() - ref) / np.linalg.norm(ref)) <= 1e-3
    assert cfgs.choose_gemm_tile_any(M, N, K)[:3] != ()


@pytest.mark.parametrize("pad", [0, 8], ids=["tight", "padded"])
@pytest.mark.parametrize("shape", [(33, 4, 8), (65, 60, 520), (260, 396, 264), (1000, 1004, 1000)],
                         ids=["33x4x8", "65x60x520", "260x396x264", "1000x1004x1000"])
def test_gemm_rows_of_b_on_8_byte_boundaries(gpu, shape, pad):
    """B rows whose pitch is 4 mod 8 elements, read in place: every other row starts 8 bytes past a
    16-byte boundary and the last row's last 16-byte piece crosses the end of the buffer range. NaN past
    N (padded) or in the next row's place after the last row must not reach C."""
    M, N, K = shape
    print(f"[gemm_tails] ldb4 M={M} N={N} K={K} pad={pad}", flush=True)
    a = oracle.round_to(oracle.portable_uniform(41, (M, K), -1, 1), 0)
    b = oracle.round_to(oracle.portable_uniform(42, (K, N), -1, 1), 0)
    ref = oracle.gemm(a, b)
    ad = to_device(a, torch.float16, "cuda:0")
    ldb = N + pad
    bbuf = torch.full((K + 1, ldb), float("nan"), dtype=torch.float16, device="cuda:0")
    bd = bbuf[:K, :N]
    bd.copy_(to_device(b, torch.float16, "cuda:0"))
    for tile in TILES:
        cd = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda:0")
        hip_lib.gemm_f16(ad, bd, cd, hip_lib.GemmTile(*tile, 4), ldb4=True)
        torch.cuda.synchronize()
        c = cd.float().cpu().numpy()
        assert np.isfinite(c).all(), tile
        # fp32 sums and one rounding to binary16: 2^-12 relative per element, the bound of the other tests
        assert float(np.linalg.norm(c - ref) / np.linalg.norm(ref)) <= 1e-3, tile
    with pytest.raises(ValueError, match="leading dimensions"):
        hip_lib.gemm_f16(ad, bd, cd, hip_lib.GemmTile(*TILES[0], 4))  # gemm_f16 keeps its 16-byte rows
    if pad == 0:  # a B whose base is not 16-byte aligned is restaged
        flat = torch.empty(K * N + 4, dtype=torch.float16, device="cuda:0")
        shifted = flat[4:].view(K, N)
        shifted.copy_(bd)
        torch.testing.assert_close(mma.matmul(ad, shifted), mma.matmul(ad, bd.contiguous()), rtol=0, atol=0)


@pytest.mark.parametrize("shape,ksplits", [((33, 4, 8), 4), ((64, 64, 64), 2), ((65, 60, 520), 3), ((130, 396, 1000), 7),
                                           ((100, 200, 2056), 16), ((257, 1004, 4000), 5)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else f"s{v}")
def test_gemm_splitk(gpu, shape, ksplits):
    """K split over the grid: one slab and more splits than slabs, a last split that is shorter, a ragged
    K, odd slab shares of the two K groups, ragged M and N; NaN past K in A and past N in B must not
    reach C, nothing is stored outside [M, N), and a repeat gives the same bits."""
    M, N, K = shape
    print(f"[gemm_tails] split-K M={M} N={N} K={K} ksplits={ksplits}", flush=True)
    a = oracle.round_to(oracle.portable_uniform(51, (M, K), -1, 1), 0)
    b = oracle.round_to(oracle.portable_uniform(52, (K, N), -1, 1), 0)
    ref = oracle.gemm(a, b)
    ad = _padded(a, K + 24, np.nan)
    bd = _padded(b, N + 8, np.nan)
    for tile in ((64, 64, 32, 8), (128, 64, 32, 8)):
        first = None
        for _ in range(2):
            cbuf = torch.full((M, N + 8), 1234.0, dtype=torch.float16, device="cuda:0")
            hip_lib.gemm_f16(ad, bd, cbuf[:, :N], hip_lib.GemmTile(*tile, 4), ksplits=ksplits)
            torch.cuda.synchronize()
            c = cbuf[:, :N].float().cpu().numpy()
            assert np.isfinite(c).all() and bool((cbuf[:, N:] == 1234.0).all()), tile
            assert float(np.linalg.norm(c - ref) / np.linalg.norm(ref)) <= 1e-3, tile
            assert first is None or torch.equal(first, cbuf)
            first = cbuf
    with pytest.raises(ValueError, match="no split-K kernel"):
        hip_lib.gemm_f16(ad, bd, cbuf[:, :N], hip_lib.GemmTile(128, 128, 32, 4, 4), ksplits=2)


@pytest.mark.parametrize("shape", [(74, 608, 6216), (64, 4096, 4096), (128, 1024, 4096)], ids=lambda v: "x".join(map(str, v)))
def test_gemm_few_tiles_long_k_takes_splits(gpu, shape):
    """mma.matmul and the launcher split K where the time model says so; the results are those of the
    unsplit kernel to fp32 summation order, before the one rounding to binary16."""
    M, N, K = shape
    g = torch.Generator(device="cuda:0").manual_seed(5)
    a = (torch.rand(M, K, device="cuda:0", generator=g) * 2 - 1).half()
    b = (torch.rand(K, N, device="cuda:0", generator=g) * 2 - 1).half()
    assert mma._gemm_tile_any(M, N, K)[1] > 1
    plain = torch.empty(M, N, device="cuda:0", dtype=torch.float16)
    hip_lib.gemm_f16(a, b, plain, hip_lib.GemmTile(64, 64, 32, 8, 8))
    outs = [mma.matmul(a, b)]
    if M % 128 == 0:
        c = torch.empty(M, N, device="cuda:0", dtype=torch.float16)
        mma._matmul_contiguous_kernel[(1,)](a, b, c, M, N, K)
        outs.append(c)
    ref = a.double() @ b.double()
    for out in outs:
        assert float((out.double() - ref).norm() / ref.norm()) <= 1.02 * float((plain.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("shape", [(256, 1004, 1000), (74, 612, 6216), (64, 4100, 4096), (128, 1028, 4096)],
                         ids=lambda v: "x".join(map(str, v)))
def test_launcher_refuses_rows_of_b_on_8_byte_boundaries(gpu, shape):
    """The launcher's B rows start on 16-byte boundaries whatever the time model would split."""
    M, N, K = shape
    a, b, c = (torch.zeros(s, dtype=torch.float16, device="cuda:0") for s in ((M, K), (K, N), (M, N)))
    with pytest.raises(ValueError, match="leading dimensions"):
        mma._matmul_contiguous_kernel[(1,)](a, b, c, M, N, K)
    with pytest.raises(ValueError, match="leading dimensions"):
        mma._matmul_contiguous_kernel[(1,)](a, b, c, M, N, K, BLOCK_M=64, BLOCK_N=64, BLOCK_K=32, num_warps=8)
    assert mma.matmul(a, b).shape == (M, N)  # mma.matmul takes them


def test_gemm_rejects_unaligned_tails(gpu):
    a = torch.zeros(64, 12, dtype=torch.float16, device="cuda:0")
    b = torch.zeros(12, 64, dtype=torch.float16, device="cuda:0")
    c = torch.zeros(64, 64, dtype=torch.float16, device="cuda:0")
    with pytest.raises(ValueError, match="multiple of 8"):
        hip_lib.gemm_f16(a, b, c, hip_lib.GemmTile(128, 128, 32, 4, 4))
