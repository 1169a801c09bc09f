"""head_dim 64 prefill on the GPU (ts_prefill_attention[_ws]): the stream kernel and the tile kernel
with one and two key groups, split and unsplit, against the oracle to the attention bar of
test_kernels_gpu.py. The shapes put chunk ends, the diagonal and the key tail around the 32, 64 and
128-row tiles and the 64-key steps, with an even and an odd GQA group and KV heads that divide the
XCDs or do not; cache rows past seq_len are NaN."""

from __future__ import annotations

import pytest
import torch

from turingserve_amd import _native as N

from .test_kernels_gpu import DEV, assert_attn, make_paged, meta_of, oracle_attn

pytestmark = pytest.mark.gpu
D = 64

SHAPES = [((1,), (0,)), ((33,), (607,)), ((65, 2), (40, 575)),            # stream (short contexts)
          ((257,), (1000,)),
          ((64,), (1600,)), ((63, 129), (1700, 0)), ((700, 600), (0, 65)),  # two key groups, unsplit
          ((700, 30, 128), (0, 1500, 65)), ((260,), (2000,)),             # ... and split
          ((16,), (2003,)), ((31,), (610,)), ((5, 16), (900, 2100)),
          ((128,), (4100,)), ((130, 1), (4096, 3000)), ((900,), (4200,))]  # one key group, split


def _run(dev, meta, H, KVH, ws_bytes, max_seq=None, max_query=None):
    q, kc, vc, qsl, sl, bt = dev
    out = torch.full((q.shape[0], H * D), float("nan"), dtype=torch.float16, device=DEV)
    ws = torch.full((max(ws_bytes, 16) // 4,), float("nan"), device=DEV)
    mq = max_query or int(meta.max_query_len)
    N.check(N.lib().ts_prefill_attention_ws(
        q.data_ptr(), q.stride(0), q.stride(1), out.data_ptr(), out.stride(0), q.shape[0],
        kc.data_ptr(), vc.data_ptr(), kc.shape[0], bt.data_ptr(), bt.stride(0), bt.shape[1],
        sl.data_ptr(), qsl.data_ptr(), sl.shape[0], 0, mq, max_seq or int(meta.max_seq_len), H,
        KVH, D, D ** -0.5, ws.data_ptr() if ws_bytes else None, ws_bytes,
        torch.cuda.current_stream().cuda_stream), "prefill")
    torch.cuda.synchronize()
    return out


def _setup(q_lens, prefixes, H, KVH):
    seq = [p + n for p, n in zip(prefixes, q_lens)]
    q, kc, vc, qsl, sl, bt = make_paged(seq, H, KVH, D, list(q_lens), seed=sum(q_lens))
    ref = oracle_attn(q, kc, vc, qsl, sl, bt, D ** -0.5)
    for b, n in enumerate(seq):                       # a reused block's tail may hold anything
        if n % 16:
            blk = int(bt[b, n // 16])
            kc[blk, :, n % 16:] = float("nan")
            vc[blk, :, n % 16:] = float("nan")
    return [t.to(DEV) for t in (q, kc, vc, qsl, sl, bt)], meta_of(qsl, sl, bt, 0, list(q_lens),
                                                                  q.shape[0]), ref


@pytest.mark.parametrize("H,KVH", [(14, 2), (8, 8), (6, 3)])
@pytest.mark.parametrize("q_lens,prefixes", SHAPES)
def test_every_route_against_the_oracle(q_lens, prefixes, H, KVH):
    dev, meta, ref = _setup(q_lens, prefixes, H, KVH)
    nb = N.lib().ts_prefill_workspace_bytes(len(q_lens), H, D, int(meta.max_query_len),
                                            int(meta.max_seq_len), N.cu_count(0))
    assert_attn(_run(dev, meta, H, KVH, nb), ref, f"plan ({nb} bytes of partials)")
    assert_attn(_run(dev, meta, H, KVH, 0), ref, "no workspace")
    if nb:
        assert_attn(_run(dev, meta, H, KVH, nb - 4), ref, "workspace too small: unsplit")


def test_many_tiles_take_one_key_group():
    """Six chunks of 150 on 28 heads: 2 x 6 x 28 128-row tiles, more than 7 per 4 of 256 CUs are
    reached with 24 chunks; both sides of that line."""
    for P in (6, 24):
        q_lens, prefixes = [150 - i for i in range(P)], [(50 * i) % 300 for i in range(P)]
        dev, meta, ref = _setup(q_lens, prefixes, 28, 4)
        assert_attn(_run(dev, meta, 28, 4, 0), ref, f"{P} chunks")


@pytest.mark.parametrize("q_len,prefix", [(16, 2003), (900, 4200)])
def test_understated_seq_bound_is_still_computed(q_len, prefix):
    """max_seq_len below the real seq_len (a caller bug): the splits would not fit the plan's slots,
    so the tiles run unsplit and every row is right."""
    dev, meta, ref = _setup((q_len,), (prefix,), 14, 2)
    bound = prefix // 2 if q_len == 16 else 4100
    nb = N.lib().ts_prefill_workspace_bytes(1, 14, D, q_len, bound, N.cu_count(0))
    assert nb > 0
    assert_attn(_run(dev, meta, 14, 2, nb, max_seq=bound), ref, "understated max_seq_len")
