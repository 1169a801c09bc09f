"""The W8A16 block-tile kernel (w8a16_tile.h) on the GPU: every tile size the planner can pick, at
shapes that leave a remainder in both directions of the tile, with fewer, as many and more K steps
than the LDS ring has stages (the plan takes 128 x 64 with four K groups from 12 steps on only; with
RoPE in place of 64 x 96 from fewer), and through each epilogue (plain, fp32 logits rows, gated MLP,
RoPE with the cache write). Every case asserts that the plan takes the tile it is there for.

The product is held to the W8A16 bars of test_kernels_gpu.py (relative Frobenius 1e-3; 1 fp16 ulp
of the exact product plus fp32 accumulation noise, 1e-4 of the RMS); the fused epilogues equal the
separate calls bit for bit, since both take the same K order."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import quant as OQ
from turingserve_amd import _native
from turingserve_amd import hip_ops as K
from turingserve_amd.qwen2 import rope_tables

pytestmark = pytest.mark.gpu
DEV = "cuda"

# M, N, the plan's tile on 256 CUs (rows, cols, K groups), LDS stages: partial tiles in M and N
TILES = [(1000, 15988, (256, 256, 1), 3), (575, 17884, (256, 192, 1), 3), (1790, 2004, (128, 128, 2), 3),
         (1855, 1500, (128, 96, 4), 3), (1000, 2004, (128, 64, 4), 4), (750, 2004, (64, 96, 4), 4),
         (67, 17884, (128, 96, 2), 3), (195, 17884, (128, 96, 2), 3), (131, 17884, (128, 64, 2), 3),
         (9, 17884, (128, 32, 4), 4), (31, 17884, (128, 32, 4), 4), (17, 9724, (64, 32, 4), 4),
         (63, 9724, (64, 32, 4), 4)]
# 64 x 32 tiles: products that the wide kernel would split over K (from K = 768 on), and one of many
# columns at long K
SMALL = [(47, 2004, (64, 32, 4), 768), (64, 1500, (64, 32, 4), 896), (20, 32996, (64, 32, 4), 3072),
         (47, 2004, (64, 32, 4), 1152)]


def _with_steps(steps):
    """(M, N, tile, K) of each tile with K = that many of its steps; steps(S) lists them."""
    out = []
    for M, N, tile, S in TILES:
        bk = 128 if tile[2] == 4 or tile == (128, 128, 2) else 64
        counts = [12, 13] if tile == (128, 64, 4) else steps(S)
        out += [(M, N, tile, bk * c) for c in counts]
    return out


def _assert_plan(M, N, K, tile):
    t = _native.lib().ts_w8a16_plan_tile(M, N, K, _native.cu_count(0))
    assert (t >> 16, t >> 4 & 0xfff, t & 15) == tile


def _problem(M, N, Kd, fp16_scale=False):
    g = torch.Generator().manual_seed(M * 7 + N + Kd)
    wq = torch.randint(-127, 128, (N, Kd), generator=g, dtype=torch.int32).to(torch.int8)
    scale = torch.rand(N, generator=g) * 0.01 + 0.001
    scale = scale.half() if fp16_scale else scale
    x = torch.randn(M, Kd, generator=g).half()
    bias = (torch.randn(N, generator=g) * 0.5).half()
    return x, wq, scale, bias


@pytest.mark.parametrize("M,N,tile,Kd", _with_steps(lambda S: [1, S - 1, S, S + 1, 2 * S + 1]) + SMALL)
def test_every_tile_against_the_oracle(M, N, tile, Kd):
    _assert_plan(M, N, Kd, tile)
    x, wq, sc, bias = _problem(M, N, Kd, fp16_scale=Kd == 384)
    y = K.w8a16_linear(x.cuda(), wq.cuda(), sc.cuda(), bias.cuda()).float().cpu().numpy()
    ref = OQ.w8a16(x.numpy(), wq.numpy(), sc.numpy().astype(np.float64), bias.numpy(), np.float64)
    assert np.linalg.norm(y - ref) / np.linalg.norm(ref) < 1e-3
    rms = float(np.sqrt((ref ** 2).mean()))
    ulp = np.spacing(np.abs(ref).astype(np.float16)).astype(np.float64)
    assert (np.abs(y - ref.astype(np.float16).astype(np.float64)) <= ulp + 1e-4 * rms).all()


@pytest.mark.parametrize("M,N,tile,Kd", _with_steps(lambda S: [1, S]) + SMALL)
def test_gated_epilogue_equals_the_pair(M, N, tile, Kd):
    """The gated-MLP epilogue against the product then SiLU.up."""
    inter = N // 16 * 8                                       # the separate kernel needs I % 8 == 0
    _assert_plan(M, 2 * inter, Kd, tile)
    x, wq, sc, bias = (t.cuda() for t in _problem(M, 2 * inter, Kd))
    fused = K.w8a16_glu(x, wq, sc, bias)
    assert torch.equal(fused, K.silu_mul(K.w8a16_linear(x, wq, sc, bias)))


@pytest.mark.parametrize("M,N,tile,Kd", _with_steps(lambda S: [S]) + SMALL)
def test_logits_epilogue_equals_the_gathered_product(M, N, tile, Kd):
    _assert_plan(M, N, Kd, tile)
    x, wq, sc, _ = (t.cuda() for t in _problem(M, N, Kd))
    rows = torch.randint(0, M, (M,), generator=torch.Generator().manual_seed(N)).cuda()
    got = K.logits_int8(x, rows, wq, sc)
    assert torch.equal(got, K.w8a16_linear(x[rows], wq, sc, None).float())


@pytest.mark.parametrize("M,H,KVH,Kd,tile", [
    (700, 12, 2, 256, (64, 96, 4)), (700, 12, 2, 640, (64, 96, 4)), (1000, 12, 2, 1536, (128, 64, 4)),
    (1390, 12, 2, 256, (128, 96, 4)), (1801, 12, 2, 256, (128, 128, 2)), (555, 100, 20, 256, (256, 192, 1)),
    (1003, 84, 20, 256, (256, 256, 1)), (20, 100, 20, 1152, (128, 32, 4)), (45, 12, 2, 1152, (64, 32, 4)),
    (64, 12, 2, 1152, (64, 32, 4))])
def test_rope_epilogue_equals_the_separate_calls(M, H, KVH, Kd, tile):
    """Heads of 128 in tiles of 128 and 256 columns (700 rows: the plan's 64-column tile holds half
    a head, so the fused call takes 128 columns, as it does at 45 and 64 rows; at 20 the 128 x 32
    tiles), slots and positions out of range."""
    from turingserve_amd.quant import LinearWeight

    N, NB = (H + 2 * KVH) * 128, 8 + M // 16
    _assert_plan(M, N, Kd, tile)
    x, wq, sc, bias = (t.cuda() for t in _problem(M, N, Kd))
    g = torch.Generator().manual_seed(M)
    pos = torch.randint(-3, 600, (M,), generator=g).cuda()
    slots = torch.randperm(NB * 16, generator=g)[:M].long()
    slots[::5], slots[2] = -1, NB * 16 + 3
    slots = slots.cuda()
    cos, sin = rope_tables(128, 1e6, 512, DEV)
    kv = torch.randn(2, NB, KVH, 16, 128, generator=g).half().cuda()
    kv1, kv2 = kv.clone(), kv.clone()
    qkv1 = K.linear_rope_kv_write(x, LinearWeight(wq, bias, sc), pos, cos, sin, H, KVH, 128,
                                  kv1[0], kv1[1], slots)
    qkv2 = K.w8a16_linear(x, wq, sc, bias)
    assert K.rope_kv_write_(qkv2, pos, cos, sin, H, KVH, 128, kv2[0], kv2[1], slots)
    assert torch.equal(qkv1, qkv2) and torch.equal(kv1, kv2)


def test_weights_off_16_bytes_take_the_general_kernels():
    """The block tiles' weight DMA wants 16-byte rows; 8-byte aligned weights are served by the wide
    kernel, or, where that would split K (and the plan's workspace is none), by the skinny one."""
    for M, N, Kd in ((47, 2048, 1536), (20, 17920, 256), (700, 2048, 256)):
        x, wq, sc, bias = (t.cuda() for t in _problem(M, N, Kd))
        off = torch.empty(N * Kd + 8, dtype=torch.int8, device=DEV)[8:].view(N, Kd).copy_(wq)
        assert off.data_ptr() % 16 == 8
        y = K.w8a16_linear(x, off, sc, bias).float().cpu().numpy()
        ref = OQ.w8a16(x.cpu().numpy(), wq.cpu().numpy(), sc.cpu().numpy().astype(np.float64),
                       bias.cpu().numpy(), np.float64)
        assert np.linalg.norm(y - ref) / np.linalg.norm(ref) < 1e-3
