"""clip_grad_norm_ in one call (dsx_clip_grad_norm / _multi): the norms whose
powers are products (p = 3 to 8) and those around them, against fp64 torch;
the same state as dsx_norm_partials + dsx_clip_prepare; a result of its own
for every call."""
from __future__ import annotations

import sys

import pytest

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


@pytest.mark.parametrize("form", ["flat", "ragged"])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
def test_norms_by_power(gpu, form, dtype):
    import torch
    from distributedspeed_amd import ops
    from distributedspeed_amd.optimizers import AdamWOptimizer, MultiTensorAdamWOptimizer
    dt = getattr(torch, dtype)
    sizes = (70_001, 24, 131_072 + 5)
    gen = torch.Generator(device=gpu).manual_seed(9)
    grads = [torch.empty(k, device=gpu).normal_(0.0, 1.0, generator=gen).to(dt) for k in sizes]
    ps = [torch.nn.Parameter(torch.zeros(k, device=gpu)) for k in sizes]
    cls = AdamWOptimizer if form == "flat" else MultiTensorAdamWOptimizer
    opt = cls(ps, param_dtype=None if dt == torch.float32 else dt, device=gpu)
    for p, g in zip(ps, grads):
        p.grad = g.clone()
    flat64 = torch.cat(grads).double().abs()
    results = []
    for p in (3, 4.0, 5, 7, 8, 2.5, 7.5, 8.5, 9, 1, 2, float("inf")):
        _say(f"norm p={p} {form} {dtype}")
        ref = float(flat64.max()) if p == float("inf") else float(flat64.pow(p).sum()) ** (1.0 / p)
        got = opt.clip_grad_norm_(0.5, p)
        torch.cuda.synchronize()
        assert got.shape == () and got.dtype == torch.float32 and got.is_cuda
        # fp64 sums of 2e5 terms of a few roundings each: 1e-11 at most; then fp32
        assert float(got) == pytest.approx(ref, rel=1.0e-7)
        one = opt.read_state()
        assert one.clip_once == 1
        # the same norm in two calls, in fp64
        norm = torch.zeros(1, dtype=torch.float64, device=gpu)
        ops.clip_prepare(opt.partials, opt.nparts, p, 0.5, opt.clip_eps, opt.dstate, norm)
        torch.cuda.synchronize()
        assert float(norm) == pytest.approx(ref, rel=1e-11)
        assert bytes(opt.read_state()) == bytes(one)
        results.append((got, float(got)))
    assert len({r.data_ptr() for r, _ in results}) == len(results)
    assert all(float(r) == v for r, v in results)  # no later call wrote an earlier result
