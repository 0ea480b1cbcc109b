"""aegkv_copy_blocks_noalloc against aegkv_copy_blocks on the GPU.

Both entry points run the same copies on two identical caches, two calls in
a row on one stream (the second with fewer pairs) with no synchronization in
between, so a descriptor that was not taken from the fixed host area before
the next call overwrote it would show up as a difference. Byte equality
between the two caches, and the closed form seg[dst] == old seg[src].
"""

import ctypes
import sys

import numpy as np
import pytest
import torch

from aegaeon_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, file=sys.stderr, flush=True)


def _caches(n_seg, n_blocks, page, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    a = [torch.randint(0, 256, (n_blocks, page), dtype=torch.uint8, device=dev, generator=g)
         for _ in range(n_seg)]
    return a, [t.clone() for t in a]


def _pairs(rng, n_blocks, n):
    perm = rng.permutation(n_blocks)
    return perm[:n], perm[n:2 * n]


@pytest.mark.parametrize("n_seg,n_blocks,page,n1,n2", [
    (24, 512, 64 * 1024, 200, 37),        # 64 KiB tiles, one workgroup per tile
    (40, 256, 160 * 1024, 100, 1),        # 160 KiB tiles (10 loads per lane)
    (8, 1024, 16 * 1024, 500, 499),       # 16 KiB tiles
    (5, 64, 4000, 30, 7),                 # 16 B path with a tail chunk
    (3, 64, 1001, 20, 3),                 # byte path (odd page)
    (1, 2 * 65536 + 5, 256, 65536, 1000),  # the largest pair table
    (1024, 16, 64, 8, 5),                 # the largest segment table
])
def test_copy_blocks_noalloc_matches_copy_blocks(gpu, n_seg, n_blocks, page, n1, n2):
    _say("copy_blocks_noalloc vs copy_blocks", n_seg, n_blocks, page, n1, n2)
    rng = np.random.default_rng(n_seg * 1000 + n1)
    a, b = _caches(n_seg, n_blocks, page, n_seg + n1, gpu)
    before = [t.clone() for t in a]
    s1, d1 = _pairs(rng, n_blocks, n1)
    s2, d2 = _pairs(rng, n_blocks, n2)
    torch.cuda.synchronize()
    ops.copy_blocks(a, s1, d1)
    ops.copy_blocks(a, s2, d2)
    ops.copy_blocks_noalloc(b, s1, d1)
    ops.copy_blocks_noalloc(b, s2, d2)
    torch.cuda.synchronize()
    want = [t.clone() for t in before]
    for s_, d_ in ((s1, d1), (s2, d2)):
        si, di = torch.from_numpy(s_).to(gpu), torch.from_numpy(d_).to(gpu)
        for w in want:
            w[di] = w[si]
    for i in range(n_seg):
        assert torch.equal(a[i], b[i]), i
        assert torch.equal(b[i], want[i]), i


def test_copy_blocks_noalloc_after_rejection_and_on_a_second_stream(gpu):
    """A rejected call enqueues nothing and leaves the next call intact; the
    entry point runs on the stream it is given."""
    rng = np.random.default_rng(5)
    a, b = _caches(6, 128, 32 * 1024, 6, gpu)
    s1, d1 = _pairs(rng, 128, 40)
    with pytest.raises(ValueError, match="twice"):
        ops.copy_blocks_noalloc(b, s1[:2], [d1[0], d1[0]])
    with pytest.raises(ValueError, match="exceed"):
        ops.copy_blocks_noalloc(b, np.arange(ops.NOALLOC_MAX_PAIRS + 1),
                                np.arange(ops.NOALLOC_MAX_PAIRS + 1))
    st = torch.cuda.Stream(gpu)
    st.wait_stream(torch.cuda.current_stream(gpu))
    ops.copy_blocks(a, s1, d1)
    ops.copy_blocks_noalloc(b, s1, d1, stream=st)
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    assert ctypes.sizeof(ctypes.c_int64) == 8 and _lib.load().aegkv_copy_blocks_noalloc


def test_copy_blocks_noalloc_under_graph_capture(gpu):
    """A graph that captures the call replays its own descriptor. Between
    replays the test rewrites the captured targets and makes other
    allocation-free calls (which rewrite the library's packing area and the
    device array), then synchronizes; each of three replays must copy the
    captured pairs, and only those. The captured descriptor (250 pairs over
    12 segments, 4512 bytes) spans three fill launches."""
    _say("copy_blocks_noalloc under graph capture")
    rng = np.random.default_rng(11)
    n_seg, n_blocks, page = 12, 1024, 32 * 1024
    a, _ = _caches(n_seg, n_blocks, page, 11, gpu)
    perm = rng.permutation(n_blocks)
    sa, da = perm[:250], perm[250:500]          # captured pairs
    sb, db = perm[500:600], perm[600:700]       # eager pairs between replays
    ops.copy_blocks_noalloc(a, sb[:1], db[:1])  # first call on the device outside the capture
    torch.cuda.synchronize()
    before = [t.clone() for t in a]
    graph = torch.cuda.CUDAGraph()
    st = torch.cuda.Stream(gpu)
    with torch.cuda.graph(graph, stream=st):
        ops.copy_blocks_noalloc(a, sa, da)
    torch.cuda.synchronize()
    for x, y in zip(a, before):
        assert torch.equal(x, y)  # capturing ran nothing
    ia, ja = torch.from_numpy(sa).to(gpu), torch.from_numpy(da).to(gpu)
    for r in range(3):
        for t in a:
            t[ja] = r + 1
        k = 30 * r
        ops.copy_blocks_noalloc(a, sb[k:k + 30], db[k:k + 30])
        torch.cuda.synchronize()
        want = [t.clone() for t in a]
        for w in want:
            w[ja] = w[ia]
        graph.replay()
        torch.cuda.synchronize()
        for i in range(n_seg):
            assert torch.equal(a[i], want[i]), (r, i)
    del graph


# Descriptors around what one launch's arguments hold: the copy's own 3808
# bytes (32 a segment, 16 a pair) and a fill's 3776 (16 a segment, 8 a pair).
@pytest.mark.parametrize("page", [32, 33])
@pytest.mark.parametrize("n_seg,n", [
    (1, 235), (1, 236), (1, 237), (72, 94), (72, 95), (118, 2), (118, 3), (119, 1),
    (1, 470), (1, 471), (1, 942), (1, 943), (236, 5), (237, 5), (237, 471),
])
def test_copies_with_descriptors_around_a_launch_s_arguments(gpu, n_seg, n, page):
    _say("descriptors around a launch's arguments", n_seg, n, page)
    rng = np.random.default_rng(n_seg * 1000 + n)
    n_blocks = 2 * n + 3
    a, _ = _caches(n_seg, n_blocks, page, n, gpu)
    src, dst = _pairs(rng, n_blocks, n)
    s, d = torch.from_numpy(src.copy()).to(gpu), torch.from_numpy(dst.copy()).to(gpu)
    want = [t.clone().index_copy_(0, d, t[s]) for t in a]
    for entry in (ops.copy_blocks, ops.copy_blocks_noalloc):
        got = [t.clone() for t in a]
        entry(got, src, dst)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, want)), entry.__name__
    other = [torch.zeros_like(t) for t in a]
    ops.migrate_blocks(a, other, src, dst)
    torch.cuda.synchronize()
    for t, o, w in zip(a, other, want):
        assert torch.equal(o[d], w[d]) and int((o != 0).any(1).sum()) <= n


@pytest.mark.parametrize("n", [3, 250, 400])
def test_block_ids_beyond_32_bits(gpu, n):
    """A cache of more blocks than 32-bit ids name (1-byte pages): the copy
    with its descriptor in the launch, and one and two fill launches of
    whole 16-byte pairs."""
    _say("block ids beyond 32 bits", n)
    n_blocks = (1 << 32) + 1000
    a = torch.zeros(n_blocks, 1, dtype=torch.uint8, device=gpu)
    rng = np.random.default_rng(n)
    ids = rng.permutation(1000)
    src, dst = ids[:n] + (1 << 32) - 500, ids[n:2 * n] + (1 << 32) - 500
    s, d = torch.from_numpy(src).to(gpu), torch.from_numpy(dst).to(gpu)
    a[s] = torch.randint(1, 256, (n, 1), dtype=torch.uint8, device=gpu)
    ops.copy_blocks_noalloc([a], src, dst)
    torch.cuda.synchronize()
    assert torch.equal(a[d], a[s])
    assert not a[:4096].any() and int((a[-2000:] != 0).sum()) == 2 * n


@pytest.mark.parametrize("n", [20, 600])
def test_short_and_long_captured_copies_replay_their_own_pairs(gpu, n):
    """As above for a descriptor inside the copy's own launch and for one of
    two fill launches, with both kinds of eager call between the replays."""
    _say("captured copies", n)
    rng = np.random.default_rng(n)
    a, _ = _caches(6, 2048, 4096, n, gpu)
    perm = rng.permutation(2048)
    sa, da, rest = perm[:n], perm[n:2 * n], perm[2 * n:]
    ia, ja = torch.from_numpy(sa.copy()).to(gpu), torch.from_numpy(da.copy()).to(gpu)
    ops.copy_blocks_noalloc(a, rest[:1], rest[1:2])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(gpu)):
        ops.copy_blocks_noalloc(a, sa, da)
    for r in range(4):
        for t in a:
            t[ja] = r + 1
        ops.copy_blocks_noalloc(a, rest[:5 + r], rest[10:15 + r])
        ops.copy_blocks_noalloc(a, rest[20:420], rest[420:820])
        torch.cuda.synchronize()
        want = [t.clone().index_copy_(0, ja, t[ia]) for t in a]
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(a, want)), r
    del graph
