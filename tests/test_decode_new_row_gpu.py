"""The new row's way through the fused decode launch on the GPU: the workgroup that writes a sequence's
K/V row attends to it from LDS, not from the cache, and q's RoPE row is read ahead of positions[s].
Covered here: every place of the new token in its block and in the block pair (and in a split's last
pair), a cache whose slot held NaN, positions other than seq_len - 1, head dims of both pipelines,
with and without the split map. The launch must equal rope_kv_write (or kv_write), then attention,
bit for bit."""

from __future__ import annotations

import pytest
import torch

from turingserve_amd import hip_ops as K
from turingserve_amd.qwen2 import rope_tables

from .test_kernels_gpu import DEV, make_paged, meta_of

pytestmark = pytest.mark.gpu

# one token, both ends of a block and of a pair, 384-token (24-block) split ends, many splits
LENGTHS = [1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 384, 385, 399, 400, 416, 769, 1000, 5000]


def _case(H, KVH, D, seed):
    S = len(LENGTHS)
    q, kc, vc, qsl, sl, bt = make_paged(LENGTHS, H, KVH, D, [1] * S, seed=seed)
    meta = meta_of(qsl, sl, bt, S, [1] * S, S)
    g = torch.Generator().manual_seed(seed)
    qkv = torch.randn(S, (H + 2 * KVH) * D, generator=g).half().to(DEV)
    last = torch.tensor([int(bt[b, (n - 1) // 16]) for b, n in enumerate(LENGTHS)])
    slots = last * 16 + (torch.tensor(LENGTHS) - 1) % 16
    kc, vc = kc.to(DEV), vc.to(DEV)
    for c in (kc, vc):                                 # what the slot held before must not matter
        c[last.to(DEV), :, ((torch.tensor(LENGTHS) - 1) % 16).to(DEV)] = float("nan")
    meta.slot_mapping = slots.to(DEV)
    return qkv, kc, vc, meta


@pytest.mark.parametrize("version", [None, "v2"])
@pytest.mark.parametrize("with_map", [False, True])
@pytest.mark.parametrize("H,KVH,D", [(12, 2, 128), (14, 2, 64), (4, 2, 256)])
@pytest.mark.parametrize("shift", [0, -1, 7])
def test_rope_launch_equals_the_separate_calls(H, KVH, D, with_map, version, shift):
    qkv, kc, vc, meta = _case(H, KVH, D, seed=H + D)
    S, scale = len(LENGTHS), D ** -0.5
    pos = (torch.tensor(LENGTHS) - 1 + shift).to(DEV)   # -1 clamps to row 0, past the table to its end
    cos, sin = rope_tables(D, 1e6, 5003, DEV)
    ref_qkv, ref_k, ref_v = qkv.clone(), kc.clone(), vc.clone()
    assert K.rope_kv_write_(ref_qkv, pos, cos, sin, H, KVH, D, ref_k, ref_v, meta.slot_mapping)
    want = K.paged_attention(ref_qkv[:, :H * D].view(S, H, D), ref_k, ref_v, meta, scale,
                             decode_version=version)
    split = (K.decode_split_map(meta, H, KVH, D, kc.shape[0], kc.device, version)
             if with_map else None)
    got = K.decode_rope_kv_write_attention(qkv, pos, cos, sin, H, KVH, D, kc, vc, meta, scale,
                                           decode_version=version, split_map=split)
    assert torch.isfinite(got).all()
    assert torch.equal(got, want) and torch.equal(kc, ref_k) and torch.equal(vc, ref_v)


@pytest.mark.parametrize("H,KVH,D", [(12, 2, 128), (14, 2, 64), (4, 2, 16), (4, 2, 32)])
@pytest.mark.parametrize("with_map", [False, True])
def test_write_launch_equals_the_separate_calls(H, KVH, D, with_map):
    qkv, kc, vc, meta = _case(H, KVH, D, seed=2 * H + D)
    S, scale = len(LENGTHS), D ** -0.5
    rows = qkv.view(S, H + 2 * KVH, D)
    q, k, v = rows[:, :H], rows[:, H:H + KVH], rows[:, H + KVH:]
    ref_k, ref_v = kc.clone(), vc.clone()
    K.kv_write(k, v, ref_k, ref_v, meta.slot_mapping)
    want = K.paged_attention(q, ref_k, ref_v, meta, scale)
    split = K.decode_split_map(meta, H, KVH, D, kc.shape[0], kc.device) if with_map else None
    got = K.decode_kv_write_attention(q, k, v, kc, vc, meta, scale, split_map=split)
    assert torch.isfinite(got).all()
    assert torch.equal(got, want) and torch.equal(kc, ref_k) and torch.equal(vc, ref_v)
