"""STAGED swaps by the runs of host bytes they leave: calls of short runs, few
bytes in all, move as DIRECT, calls of a few runs copy on the caller's stream,
the others fork over the library's streams. All give the same bytes.
"""

import sys

import numpy as np
import pytest
import torch

import test_gpu
import test_gpu_guards
from aegaeon_amd import _lib, ops

pytestmark = pytest.mark.gpu

restore_tuning = test_gpu.restore_tuning


def _say(*a):
    print(*a, file=sys.stderr, flush=True)


def test_the_rule_is_on_and_takes_0_or_1():
    assert _lib.tune(_lib.TUNE_STAGED_SHORT_RUNS) == 1
    with pytest.raises(ValueError):
        _lib.tune(_lib.TUNE_STAGED_SHORT_RUNS, 2)


# page, entries, host ids, staging bytes: runs of one page each (no two host
# pages adjacent), around 128 KiB, around four of them and around 2 MiB + 16 KiB
# a run; adjacent pages that merge; and more than one chunk
@pytest.mark.parametrize("page,n,step,staging", [
    (128 << 10, 4, 2, None), (128 << 10, 5, 2, None), ((128 << 10) - 16, 4, 2, None),
    ((128 << 10) - 16, 5, 2, None), ((128 << 10) + 16, 5, 2, None), (4096, 1, 1, None),
    (4096, 40, 1, None), (4099, 7, 2, None), (256 << 10, 9, 2, 1 << 20), (256 << 10, 9, 1, 1 << 20),
    (20 << 10, 120, 2, 1 << 20), (300 << 10, 4, 1, 1 << 20),
    (32 << 10, 128, 2, None), (32 << 10, 129, 2, None), (32 << 10, 128, 2, 1 << 20),
])
@pytest.mark.parametrize("rule", [1, 0])
@pytest.mark.parametrize("uncached", [False, True])
def test_staged_swaps_by_run_length(gpu, page, n, step, staging, rule, uncached):
    _say("staged by run length", page, n, step, staging, rule, uncached)
    prev = _lib.tune(_lib.TUNE_STAGED_SHORT_RUNS, rule)
    prev_bytes = _lib.tune(_lib.TUNE_STAGING_BYTES, staging if staging else -1)
    pool = ops.PinnedHostPool(n * step * page, uncached=uncached)
    try:
        g = torch.Generator(device=gpu).manual_seed(page + n)
        cache = torch.randint(0, 256, (2 * n + 1, page), dtype=torch.uint8, device=gpu, generator=g)
        before = cache.clone()
        host = pool.tensor.view(n * step, page)
        host.random_()
        kept = host.clone()
        rng = np.random.default_rng(n)
        ids = rng.permutation(2 * n + 1)
        out, back = ids[:n], ids[n:2 * n]
        slots = rng.permutation(np.arange(n) * step)
        ops.swap(out, slots, False, cache, pool.tensor, mode="staged")
        torch.cuda.synchronize()
        want = kept.clone()
        want[torch.from_numpy(slots.copy())] = before[torch.from_numpy(out.copy()).to(gpu)].cpu()
        assert torch.equal(host, want)
        ops.swap(slots, back, True, cache, pool.tensor, mode="staged")
        torch.cuda.synchronize()
        want = before.clone()
        want[torch.from_numpy(back.copy()).to(gpu)] = before[torch.from_numpy(out.copy()).to(gpu)]
        assert torch.equal(cache, want)
    finally:
        torch.cuda.synchronize()
        pool.free()
        _lib.tune(_lib.TUNE_STAGING_BYTES, prev_bytes)
        _lib.tune(_lib.TUNE_STAGED_SHORT_RUNS, prev)


# What the staging path is tested for elsewhere with short runs, kept staged.

@pytest.mark.parametrize("dma_streams", [0, 1, 2, 3, 4])
def test_fanout_of_short_runs(gpu, oracle, restore_tuning, always_staged, dma_streams):
    test_gpu.test_staged_dma_fanout_vs_oracle(gpu, oracle, restore_tuning, dma_streams)


def test_guarded_staging(gpu, always_staged):
    test_gpu_guards.test_guarded_swaps_in_both_modes(gpu, "staged")


@pytest.mark.parametrize("shift", [0, 7])
@pytest.mark.parametrize("page", [33, 4099, 16388])
def test_staging_at_any_alignment(gpu, always_staged, page, shift):
    test_gpu.test_moves_at_any_alignment(gpu, page, shift)
