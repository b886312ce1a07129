"""The terms of the integer-power norms (p = 3 to 8) against exact rationals: one
grad per block, so that each of dsx_norm_partials' fp64 sums is one term."""
from __future__ import annotations

import sys
from fractions import Fraction

import pytest

pytestmark = pytest.mark.gpu

BLOCK_ELEMS = 256 * 4 * 4  # fp32 elements that a block takes in its first trip


@pytest.mark.parametrize("form", ["flat", "list"])
@pytest.mark.parametrize("p", [3, 4, 5, 6, 7, 8])
def test_terms_are_rounded_once(gpu, p, form):
    """Rounded once, a term is within 2**-53 of itself; 1e-6 of that is left for
    the rounding of the small part, some 2**-50 of it. pow promises 2**-52."""
    import torch
    from distributedspeed_amd import ops
    print(f"[gpu-test] terms of the {p}-norm, {form}", file=sys.stderr, flush=True)
    parts = 1024
    gen = torch.Generator(device=gpu).manual_seed(p)
    x = torch.empty(parts, device=gpu).normal_(0.0, 1e-3, generator=gen)
    x[:4] = torch.tensor([0.0, 3.4028234663852886e38, -1.0000001192092896, 1.9999998807907104], device=gpu)
    g = torch.zeros(parts * BLOCK_ELEMS, device=gpu)
    g[::BLOCK_ELEMS] = x
    state = ops.new_state(gpu, 1.0, 1)
    partials = torch.full((parts,), -1.0, dtype=torch.float64, device=gpu)
    if form == "flat":
        ops.plan_norm_partials(g, state, p, partials, parts)(ops.stream_of(gpu))
    else:
        spare = torch.zeros_like(g)  # the table's other columns, which a norm does not read
        table = ops.ChunkTable([spare], [spare], [spare], None, [g], chunk_elems=BLOCK_ELEMS)
        ops.plan_norm_partials_multi(table, state, p, partials, parts)(ops.stream_of(gpu))
    torch.cuda.synchronize()
    for a, term in zip(x.tolist(), partials.tolist()):
        exact = abs(Fraction(a)) ** p
        assert abs(Fraction(term) - exact) <= exact * Fraction(1 + 1e-6) / 2 ** 53, (a, term)


@pytest.mark.parametrize("p", [3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_a_grad_that_is_not_finite_shows(gpu, p, bad):
    import math
    import torch
    from distributedspeed_amd import ops
    g = torch.ones(10_001, device=gpu)
    g[77] = bad
    partials = torch.zeros(1, dtype=torch.float64, device=gpu)
    ops.plan_norm_partials(g, ops.new_state(gpu, 1.0, 1), p, partials, 1)(ops.stream_of(gpu))
    torch.cuda.synchronize()
    total = float(partials)
    assert math.isnan(total) if math.isnan(bad) else total == float("inf")
