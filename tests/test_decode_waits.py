"""The waits that the compiler puts into the decode launches (no GPU needed: the sources are compiled to
gfx950 assembly). Each wavefront keeps two pairs of K/V blocks in flight; a wait for fewer
outstanding loads than a pair's V rows (8) inside the loop, or for the V rows requested ahead of it
(16) before the first MFMA, gives that up without changing a result, and so does a workgroup barrier
there. Both came from control flow around the requests: paths with and without loads that met."""

from __future__ import annotations

import concurrent.futures
import re
import subprocess

import pytest

from turingserve_amd.csrc import build as B

KERNELS = [("decode.hip", "decode_mfma_kernelILi%dELi4ELb%dELb%dEE" % k)
           for k in [(64, 1, 1), (64, 1, 0), (64, 0, 0), (128, 1, 1), (128, 1, 0), (128, 0, 0)]]
KERNELS += [("ragged.hip", "ragged_split_kernel")]


def _assembly(src: str) -> str:
    cmd = [B.hipcc(), *B.COMMON_FLAGS, *B.SOURCE_FLAGS[src], "--offload-device-only", "-S", "-o", "-",
           f"{B.HERE}/{src}"]
    return subprocess.run(cmd, capture_output=True, text=True, check=True).stdout


@pytest.fixture(scope="module")
def assembly():
    srcs = sorted({s for s, _ in KERNELS})
    with concurrent.futures.ThreadPoolExecutor() as ex:
        return dict(zip(srcs, ex.map(_assembly, srcs)))


def _events(text: str, name: str) -> list[list]:
    """The kernel's blocks: [in a loop, [events]]; an event is 'load', 'dma', 'store', 'mfma', 'bar' or the
    count of a wait on vector memory."""
    body = re.search(r"^_Z\S*%s\S*:.*?^\.Lfunc_end" % name, text, re.M | re.S).group(0)
    blocks = [[False, []]]
    for line in body.splitlines():
        s = line.strip()
        if s.startswith(".LBB"):
            blocks.append(["Loop" in s, []])
        elif m := re.match(r"s_waitcnt.*vmcnt\((\d+)\)", s):
            blocks[-1][1].append(int(m.group(1)))
        elif m := re.match(r"(global_load_lds|(?:global|buffer)_load|(?:global|buffer)_store|v_mfma|s_barrier)", s):
            kind = m.group(1).split("_")
            blocks[-1][1].append("dma" if "lds" in kind else {"v": "mfma", "s": "bar"}.get(
                kind[0], kind[1]))
    return blocks


@pytest.mark.parametrize("src,name", KERNELS, ids=[n for _, n in KERNELS])
def test_two_pairs_stay_in_flight(assembly, src, name):
    blocks = _events(assembly[src], name)
    if src == "ragged.hip":                       # its decode splits: from the first K DMA on
        first = next(i for i, b in enumerate(blocks) if "dma" in b[1])
        after = next(i for i, b in enumerate(blocks) if i > first and "bar" in b[1])
        blocks = blocks[first:after]
    # the requests: the last block before the first MFMA that issues a pair's V rows or more
    mfma = next(i for i, b in enumerate(blocks) if "mfma" in b[1])
    ask = max(i for i in range(mfma) if blocks[i][1].count("load") >= 16)
    events = blocks[ask][1][len(blocks[ask][1]) - blocks[ask][1][::-1].index("load"):]
    if events[:1] == [0]:                         # the tables again, for a position not expected
        events = events[1:]
    events += sum((ev for _, ev in blocks[ask + 1:mfma]), [])
    assert "bar" not in events
    assert all(e >= 16 for e in events if isinstance(e, int)), events
    # the written-out waits for the K ring count on this order: two pairs' K by DMA, then (the tables,
    # the new row and) both pairs' V; at each refill a pair's K by eight DMAs, then its V
    order = [e for _, ev in blocks[:mfma] for e in ev if e in ("dma", "load")]
    if "dma" in order:
        first = order.index("dma")
        assert order[first:first + 16] == ["dma"] * 16 and order.count("dma") == 16
        assert order[first + 16:].count("load") >= 16
        for _, ev in blocks[mfma:]:
            refill = [e for e in ev if e in ("dma", "load")]
            if "dma" in refill:
                assert refill == (["dma"] * 8 + ["load"] * 8) * (len(refill) // 16)
    loops = [ev for loop, ev in blocks if loop and "mfma" in ev]
    assert loops
    for ev in loops:
        assert all(e >= 8 for e in ev if isinstance(e, int)), ev
