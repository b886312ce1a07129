"""dsx_zero_step_segments: the one-call step whose norm comes from the hooks'
hand-over copies, against dsx_reduce_segments, dsx_finalize_groups and
dsx_adamw_flat as separate launches (what the step issues with track_skips on).
The same bits over steps with an overflow and an explicit clip, folded in whole,
into the first part only, and not at all (more than 512 parameters)."""
from __future__ import annotations

import sys

import pytest

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


def _bits(a, b):
    import torch
    return torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("sizes", [(5,), (1000, 3, 70_001), (20_000_003, 9_000_001), (9,) * 512, (9,) * 513])
@pytest.mark.parametrize("groups", [1, 2])
def test_one_call_matches_separate_launches(gpu, sizes, groups):
    import torch
    from distributedspeed_amd.flat_step import ScalerConfig
    from distributedspeed_amd.optimizers import AdamWOptimizer
    if len(sizes) < groups:
        pytest.skip("fewer parameters than groups")
    _say(f"segments {len(sizes)} tensors, {sum(sizes)} elements, {groups} groups")
    gen = torch.Generator(device=gpu).manual_seed(3)
    init = [torch.empty(k, device=gpu).normal_(0.0, 0.02, generator=gen) for k in sizes]
    coef = [torch.empty(k, device=gpu).normal_(0.0, 1.0, generator=gen).half() for k in sizes]

    def make(separate):
        ps = [torch.nn.Parameter(t.clone()) for t in init]
        cut = len(ps) // 2
        gs = [{"params": ps}] if groups == 1 else [{"params": ps[:cut]}, {"params": ps[cut:], "weight_decay": 0.0}]
        opt = AdamWOptimizer(gs, lr=1e-3, param_dtype=torch.float16, device=gpu, max_grad_norm=1.0,
                             loss_scaler=ScalerConfig(mode="dynamic", init_scale=1024.0, hysteresis=1))
        opt.track_skips(separate)
        return ps, opt

    (pa, a), (pb, b) = make(False), make(True)
    for step in range(4):
        for ps, opt in ((pa, a), (pb, b)):
            opt.zero_grad()
            loss = sum((p * c).sum() for p, c in zip(ps, coef)) * (float("inf") if step == 2 else 1.0 + step)
            loss.backward()
            assert opt.flat.hook_norm_ready()
            if step in (1, 2):
                opt.clip_grad_norm_(0.01)
                assert opt.flat.hook_norm_ready()  # the clip reads the grads, it does not write them
            opt.step()
        torch.cuda.synchronize()
        assert bytes(a.read_state()) == bytes(b.read_state())
        assert bytes(a.last_scalars(groups - 1)) == bytes(b.last_scalars(groups - 1))
        for key in ("master", "exp_avg", "exp_avg_sq", "param16"):
            assert _bits(getattr(a.flat, key), getattr(b.flat, key)), (step, key)
    assert a.read_state().overflow_count == 1
