"""The norm passes read the first 2^28 bytes of the grads with plain loads
and the rest nontemporally (kKeepBytes in dsx_step.hip). Both loops and the
trip on which they meet, flat and over a list, in every norm kind. The grads
are small integers, so every sum of squares and of magnitudes is an integer
below 2^53: exact in fp64 in any order, and compared exactly."""
from __future__ import annotations

import math
import sys

import pytest

pytestmark = pytest.mark.gpu

KEEP = 1 << 28  # bytes


def _say(msg):
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


def _grads(n, dtype, gpu):
    import torch
    g = torch.arange(n, dtype=torch.int32, device=gpu).remainder_(61)  # exact in bf16
    g[-1] = 100  # the maximum, in the last element
    return g.to(dtype)


def _expected(g):
    import torch
    x = g.to(torch.float64)
    return {2.0: float((x * x).sum()), 1.0: float(x.sum()), math.inf: 100.0}


@pytest.mark.parametrize("dtype,extra", [("float32", -5), ("float32", 0), ("float32", 3 * 8192 + 7),
                                         ("bfloat16", 3 * 8192 + 7)])
def test_flat_norms_across_the_kept_bytes(gpu, dtype, extra):
    import torch
    from distributedspeed_amd import ops
    dt = getattr(torch, dtype)
    n = KEEP // torch.empty(0, dtype=dt).element_size() + extra
    _say(f"flat norms n={n} {dtype}")
    g = _grads(n, dt, gpu)
    state = ops.new_state(gpu, 1.0, 1)
    nparts = ops.suggest_partials(n)
    s = ops.stream_of(gpu)
    want = _expected(g)
    partials = torch.full((nparts,), float("nan"), dtype=torch.float64, device=gpu)
    ops.plan_unscale_norm(g, state, partials)(s)
    assert float(partials.sum()) == want[2.0]
    for p, ref in want.items():
        partials.fill_(float("nan"))
        ops.plan_norm_partials(g, state, p, partials, nparts)(s)
        assert float(partials.max() if math.isinf(p) else partials.sum()) == ref, p


@pytest.mark.parametrize("chunk", [16384, 65536])  # one chunk per wave, one per block
def test_list_norms_across_the_kept_bytes(gpu, chunk):
    import torch
    from distributedspeed_amd import ops
    n = KEEP // 2 + 40_000_001
    _say(f"list norms n={n} chunk={chunk}")
    g = _grads(n, torch.bfloat16, gpu)
    cuts = [0, 24, 70_000_008, KEEP // 2 - 8, KEEP // 2 + 100_000, n]
    grads = [g[a:b] for a, b in zip(cuts, cuts[1:])]
    want = _expected(g)
    masters = [torch.zeros(t.numel(), device=gpu) for t in grads]  # the norm reads only the grads
    table = ops.ChunkTable(masters, masters, masters, None, grads, chunk_elems=chunk)
    state = ops.new_state(gpu, 1.0, 1)
    s = ops.stream_of(gpu)
    for nparts in (512, 97) if chunk == 65536 else (table.nchunks // 16 + 1,):
        partials = torch.full((nparts,), float("nan"), dtype=torch.float64, device=gpu)
        ops.plan_unscale_norm_multi(table, state, partials, nparts)(s)
        assert float(partials.sum()) == want[2.0], nparts
        for p, ref in want.items():
            partials.fill_(float("nan"))
            ops.plan_norm_partials_multi(table, state, p, partials, nparts)(s)
            assert float(partials.max() if math.isinf(p) else partials.sum()) == ref, (p, nparts)
