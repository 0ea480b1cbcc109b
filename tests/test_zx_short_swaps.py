"""DIRECT swaps with descriptors around what one launch's arguments hold, with
and without a move guard: the same bytes land, and a set guard stops them all.
"""

import sys

import numpy as np
import pytest
import torch

from aegaeon_amd import ops

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, file=sys.stderr, flush=True)


# the arguments hold 3776 bytes: 32 a segment, 8 a cache group, 32 an entry
@pytest.mark.parametrize("guarded", [False, True])
@pytest.mark.parametrize("page,segs,groups,n", [
    (4096, 1, 1, 1), (4096, 1, 1, 116), (4096, 1, 1, 117), (2048, 72, 1, 45), (2048, 72, 1, 46),
    (512, 116, 1, 1), (512, 116, 3, 2), (512, 117, 1, 1), (512, 118, 1, 1), (9232, 3, 2, 30),
    (9232, 3, 3, 113), (9232, 3, 3, 114), (16, 5, 64, 9), (4099, 2, 1, 20), (33, 2, 2, 115),
    (12800, 40, 1, 300),
])
def test_swaps_with_descriptors_around_a_launch_s_arguments(gpu, page, segs, groups, n, guarded):
    _say("short swaps", page, segs, groups, n, guarded)
    rng = np.random.default_rng(page + segs + n)
    g = torch.Generator(device=gpu).manual_seed(n)
    blocks = 2 * n + 1
    cache = [torch.randint(0, 256, (blocks, page), dtype=torch.uint8, device=gpu, generator=g)
             for _ in range(segs)]
    start = [t.clone() for t in cache]
    pool = ops.PinnedHostPool((n + 2) * segs * page)
    host = pool.tensor.view(n + 2, segs, page)
    host.random_()
    kept = host.clone()
    owners = [1 << (s % groups) for s in range(segs)]
    lay = ops.SegmentLayout(cache, [page] * segs, [s * page for s in range(segs)], owners,
                            blocks, [1] * groups, pool.tensor, segs * page, 0)
    ids, slots = rng.permutation(blocks), rng.permutation(n + 2)[:n]
    grp = rng.integers(0, groups, n)
    f, o = np.zeros(n, np.int64), np.ones(n, np.int64)
    words = ops.GuardWords(2)
    words.tensor[1] = 1
    kw = dict(guard=words.tensor) if guarded else {}

    def moved(into, rows, frm, out_rows):
        """into[rows, s] <- frm[out_rows, s] of the segments each entry's group owns."""
        for k in range(n):
            for s in range(segs):
                if s % groups == grp[k]:
                    into(s, rows[k], frm(s, out_rows[k]))

    try:
        torch.cuda.synchronize()
        if guarded:
            lay.swap(ids[:n], slots, grp, f, o, False, guard=words.tensor, guard_index=1)
            lay.swap(slots, ids[n:2 * n], grp, f, o, True, guard=words.tensor, guard_index=1)
            torch.cuda.synchronize()
            assert torch.equal(host, kept), "a set guard let a swap-out through"
            assert all(torch.equal(a, b) for a, b in zip(cache, start)), "a set guard, swap-in"
        lay.swap(ids[:n], slots, grp, f, o, False, **kw)
        torch.cuda.synchronize()
        want = kept.clone()
        cpu = torch.stack([t.cpu() for t in start], 1)
        moved(lambda s, r, v: want[r, s].copy_(v), slots, lambda s, r: cpu[r, s], ids[:n])
        assert torch.equal(host, want)
        lay.swap(slots, ids[n:2 * n], grp, f, o, True, **kw)
        torch.cuda.synchronize()
        now = cpu.clone()
        moved(lambda s, r, v: now[r, s].copy_(v), ids[n:2 * n], lambda s, r: want[r, s], slots)
        assert torch.equal(torch.stack([t.cpu() for t in cache], 1), now)
    finally:
        torch.cuda.synchronize()
        del lay, host
        pool.free()
