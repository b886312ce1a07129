"""K3's launch shapes by chunk count (one chunk per block, one block per CU in
one launch and in several, many blocks) and the tables the ragged store builds
for mid-size lists: the same bits as K2 over the same elements."""
from __future__ import annotations

import sys

import pytest

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


def _bits(a, b):
    import torch
    return torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


# chunks per CU around each change of shape, and chunks past a multiple of 256
@pytest.mark.parametrize("per_cu,extra", [(1, -1), (20, 0), (20, 1), (64, 0), (64, 1), (129, 77), (256, -1), (256, 3)])
@pytest.mark.parametrize("gdt", ["bfloat16", "float32"])
def test_every_k3_shape_gives_k2s_bits(gpu, per_cu, extra, gdt):
    import torch
    from distributedspeed_amd import ops
    from distributedspeed_amd._lib import DsxStepScalars
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    nchunks, chunk = per_cu * cus + extra, 24
    gdt = getattr(torch, gdt)
    pdt = torch.bfloat16 if gdt == torch.bfloat16 else None
    n = nchunks * chunk - 8  # the last chunk of the last tensor is short
    _say(f"K3 shape chunks={nchunks} {gdt}")
    gen = torch.Generator(device=gpu).manual_seed(per_cu)
    p, m = (torch.empty(n, device=gpu).normal_(0.0, 0.02, generator=gen) for _ in range(2))
    v = torch.empty(n, device=gpu).uniform_(0.0, 1e-6, generator=gen)
    g = torch.empty(n, device=gpu).normal_(0.0, 1e-3, generator=gen).to(gdt)
    p16 = p.to(pdt) if pdt else None
    cuts = [0, chunk, (nchunks // 2) * chunk, n]

    def split(t):
        return [t[a:b].clone() for a, b in zip(cuts, cuts[1:])] if t is not None else None

    sp, sm, sv, s16, sg = (split(t) for t in (p, m, v, p16, g))
    table = ops.ChunkTable(sp, sm, sv, s16, sg, chunk_elems=chunk)
    assert table.nchunks == nchunks
    sc = DsxStepScalars()
    sc.inv_scale, sc.clip_coef, sc.decay, sc.w1, sc.w1c = 1.0, 0.5, 0.9999, 0.1, 0.9
    sc.b2, sc.val2, sc.eps, sc.bc2s, sc.nss = 0.999, 0.001, 1e-8, 0.3, -1e-3
    scal = ops.scalars_from_host(sc, gpu)
    ops.adamw_multi(table, scal)
    ops.adamw_flat(p, m, v, p16, g, scal)
    for name, got, ref in (("master", sp, p), ("exp_avg", sm, m), ("exp_avg_sq", sv, v), ("param16", s16, p16)):
        assert got is None or _bits(torch.cat(got), ref), name


# chunks of 8192 (16-20 and 20-32 per CU) without and with tensors of K2's
# size, and a list of K2's tensors alone
@pytest.mark.parametrize("sizes,big", [((13_000_008, 9_000_001, 14_000_000), 0), ((15_000_000, 16_500_000, 16_000_003), 0),
                                       ((17_000_000, 20_000_000, 77), 2), ((18_000_000, 17_000_000), 2)])
def test_mid_size_lists_match_the_flat_form(gpu, sizes, big):
    import torch
    from distributedspeed_amd.optimizers import AdamWOptimizer, MultiTensorAdamWOptimizer
    _say(f"mid-size list {sizes}")
    gen = torch.Generator(device=gpu).manual_seed(5)
    init = [torch.empty(k, device=gpu).normal_(0.0, 0.02, generator=gen) for k in sizes]
    grads = [torch.empty(k, device=gpu).normal_(0.0, 1e-3, generator=gen).to(torch.bfloat16) for k in sizes]
    opts = []
    for cls in (AdamWOptimizer, MultiTensorAdamWOptimizer):
        ps = [torch.nn.Parameter(t.clone()) for t in init]
        opt = cls(ps, lr=1e-3, param_dtype=torch.bfloat16, device=gpu, max_grad_norm=1.0)
        for _ in range(2):
            for p, g in zip(ps, grads):
                p.grad = g.clone()
            opt.step()
        opts.append((ps, opt))
    store = opts[1][1].store
    assert store.chunk_elems == 8192 and len(store.k2_tensors) == big
    assert (store.small_table is None) == (big == len(sizes))
    for pf, pr in zip(opts[0][0], opts[1][0]):
        assert _bits(pf.data, pr.data)
        for key in ("master", "exp_avg", "exp_avg_sq"):
            assert _bits(opts[0][1].state[pf][key], opts[1][1].state[pr][key]), key


# Chunks in 1, 2, 8 and more than 8 spans of a trip with short last spans, and
# the element counts around the folded kernels' change of cache policy (2**26
# bytes of state: 5592405 elements; the flat form pads each parameter to 8).
@pytest.mark.parametrize("sizes,chunk", [((5000, 3, 2049), 2048), ((9000, 4097, 1), 4096), ((70_000, 16_385), 16384),
                                         ((300_001, 65_537), 65536), ((2_592_405, 3_000_000), 4096),
                                         ((2_592_406, 3_000_000), 4096), ((2_592_400, 3_000_000), 4096)])
@pytest.mark.parametrize("dtype", ["float16", None])
@pytest.mark.parametrize("form", ["ragged", "flat"])
def test_folded_steps_match_three_launches(gpu, sizes, chunk, dtype, form):
    import torch
    from distributedspeed_amd import _lib
    from distributedspeed_amd.optimizers import AdamWOptimizer, MultiTensorAdamWOptimizer
    _say(f"folded {form} {sizes} chunk={chunk} {dtype}")
    dt = getattr(torch, dtype) if dtype else None
    gen = torch.Generator(device=gpu).manual_seed(len(sizes))
    init = [torch.empty(k, device=gpu).normal_(0.0, 0.02, generator=gen) for k in sizes]
    grads = [torch.empty(k, device=gpu).normal_(0.0, 1e-3, generator=gen).to(dt or torch.float32) for k in sizes]

    def steps(bound):
        ps = [torch.nn.Parameter(t.clone()) for t in init]
        kw = {"chunk_elems": chunk} if form == "ragged" else {}
        cls = MultiTensorAdamWOptimizer if form == "ragged" else AdamWOptimizer
        opt = cls(ps, lr=1e-3, param_dtype=dt, device=gpu, max_grad_norm=1.0, **kw)
        _lib.call("dsx_set_tuning_fold", bound)
        try:
            for _ in range(3):
                for p, g in zip(ps, grads):
                    p.grad = g.clone()
                opt.step()
            torch.cuda.synchronize()
        finally:
            _lib.call("dsx_set_tuning_fold", 3 << 23)
        return ps, opt

    (pa, a), (pb, b) = steps(3 << 23), steps(0)
    if form == "flat" and sum(sizes) > 5_000_000:  # the largest step with its state kept, and the next
        assert a.flat.numel == (5_592_400 if sizes[0] == 2_592_400 else 5_592_408)
    assert bytes(a.read_state()) == bytes(b.read_state())
    for x, y in zip(pa, pb):
        assert _bits(x.data, y.data)
        for key in ("master", "exp_avg", "exp_avg_sq"):
            assert _bits(a.state[x][key], b.state[y][key]), key


@pytest.mark.parametrize("k", [1, 64, 65, 256, 257, 700])  # the launches' edges: 64 and 256 pointers
def test_set_grads_points_every_record_at_its_grad(gpu, k):
    import torch
    from distributedspeed_amd import ops
    from distributedspeed_amd._lib import DsxTensorRef
    _say(f"set_grads k={k}")
    ms = [torch.zeros(8, device=gpu) for _ in range(k)]
    old = [torch.zeros(8, device=gpu) for _ in range(k)]
    new = [torch.full((8,), float(i), device=gpu) for i in range(k)]
    table = ops.ChunkTable(ms, ms, ms, None, old, chunk_elems=8)
    before = table.tensors.cpu().numpy().tobytes()
    table.update_grads(new)
    torch.cuda.synchronize()
    after = table.tensors.cpu().numpy().tobytes()
    want = bytearray()
    size = len(before) // k
    for i in range(k):
        ref = DsxTensorRef.from_buffer_copy(before, i * size)
        ref.grad = new[i].data_ptr()
        want += bytes(ref)
    assert after == bytes(want)
    with pytest.raises(ValueError):
        table.update_grads(new[:-1] + [torch.zeros(9, device=gpu)])


def test_a_grad_of_another_size_is_refused(gpu):
    import torch
    from distributedspeed_amd.optimizers import MultiTensorAdamWOptimizer
    p = torch.nn.Parameter(torch.zeros(64, device=gpu))
    opt = MultiTensorAdamWOptimizer([p], param_dtype=torch.bfloat16, device=gpu)
    p.grad = torch.ones(64, device=gpu, dtype=torch.bfloat16)
    opt.step()
    p.data = p.data[:32]  # the same address, half the elements
    p.grad = torch.ones(32, device=gpu, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        opt.step()


# Lists above the fold's bound: K0 folded into K3's first chunks (one table; its
# own table; before K2's tensors) or into the first K2 tensor's first part,
# against K0 as a launch of its own.
@pytest.mark.parametrize("sizes,chunk", [((3000, 70_001, 5), 8), ((13_000_008, 9_000_001, 14_000_000), None),
                                         ((77, 17_000_000, 20_000_000), None), ((18_000_000, 17_000_000), None)])
def test_lists_fold_k0_into_a_first_part(gpu, sizes, chunk):
    import torch
    from distributedspeed_amd import _lib
    from distributedspeed_amd.flat_step import ScalerConfig
    from distributedspeed_amd.optimizers import MultiTensorAdamWOptimizer
    _say(f"list fold {sizes}")
    gen = torch.Generator(device=gpu).manual_seed(8)
    init = [torch.empty(k, device=gpu).normal_(0.0, 0.02, generator=gen) for k in sizes]
    grads = [torch.empty(k, device=gpu).normal_(0.0, 1.0, generator=gen).half() for k in sizes]

    def steps(bound):
        ps = [torch.nn.Parameter(t.clone()) for t in init]
        gs = [{"params": ps[:1]}, {"params": ps[1:], "lr": 3e-4, "weight_decay": 0.0}]
        opt = MultiTensorAdamWOptimizer(gs, lr=1e-3, param_dtype=torch.float16, device=gpu, max_grad_norm=1.0,
                                        loss_scaler=ScalerConfig(mode="dynamic", init_scale=1024.0, hysteresis=1),
                                        chunk_elems=chunk)
        _lib.call("dsx_set_tuning_fold", bound)
        try:
            for step in range(4):
                for p, g in zip(ps, grads):
                    p.grad = g.clone()
                if step == 1:
                    ps[-1].grad[3] = float("inf")
                if step == 2:
                    opt.clip_grad_norm_(0.01)
                opt.step()
            torch.cuda.synchronize()
        finally:
            _lib.call("dsx_set_tuning_fold", 3 << 23)
        return ps, opt

    # a bound of 1000 elements sends the small list past it as well
    (pa, a), (pb, b) = steps(1000 if chunk else 3 << 23), steps(0)
    assert bytes(a.read_state()) == bytes(b.read_state()) and a.read_state().overflow_count == 1
    for g in range(2):
        assert bytes(a.last_scalars(g)) == bytes(b.last_scalars(g))
    for x, y in zip(pa, pb):
        assert _bits(x.data, y.data)
        for key in ("master", "exp_avg", "exp_avg_sq"):
            assert _bits(a.state[x][key], b.state[y][key]), key


# Lists whose grads move at every step, at the most pointers that a step's
# first launch carries and one more, with the norm asked for in between.
@pytest.mark.parametrize("k", [1, 64, 65])
@pytest.mark.parametrize("size", [40, 3000])
def test_moving_grads_reach_every_launch(gpu, k, size):
    import torch
    from distributedspeed_amd.optimizers import AdamWOptimizer, MultiTensorAdamWOptimizer
    _say(f"moving grads k={k} size={size}")
    gen = torch.Generator(device=gpu).manual_seed(k)
    init = [torch.empty(size + i % 5, device=gpu).normal_(0.0, 0.02, generator=gen) for i in range(k)]
    opts = []
    for cls in (AdamWOptimizer, MultiTensorAdamWOptimizer):
        ps = [torch.nn.Parameter(t.clone()) for t in init]
        opts.append((ps, cls(ps, lr=1e-3, param_dtype=torch.bfloat16, device=gpu)))
    held = []  # every step's grads stay alive, so each step's are elsewhere
    for step in range(6):
        grads = [torch.empty(t.numel(), device=gpu).normal_(0.0, 1.0, generator=gen).bfloat16() for t in init]
        held.append(grads)
        for ps, opt in opts:
            for p, g in zip(ps, grads):
                p.grad = g if step % 2 else g.clone()
            if step == 3:
                opt.clip_grad_norm_(1e9)  # reads the grads, clips nothing
            if step == 4:
                opt.track_skips(True)
            if step == 5:
                opt.track_skips(False)
            opt.step()
    torch.cuda.synchronize()
    for pf, pr in zip(opts[0][0], opts[1][0]):
        assert _bits(pf.data, pr.data)
        for key in ("master", "exp_avg", "exp_avg_sq"):
            assert _bits(opts[0][1].state[pf][key], opts[1][1].state[pr][key]), key


@pytest.mark.parametrize("count", [1, 3, 5])
def test_moved_grads_of_the_first_tensors(gpu, count):
    """dsx_zero_step_multi_moved with the new addresses of the list's first
    tensors: the others' grads stay where the table has them."""
    import ctypes
    import torch
    from distributedspeed_amd import _lib, ops
    from distributedspeed_amd.optimizers import MultiTensorAdamWOptimizer
    _say(f"moved grads of the first {count} of 5")
    sizes = (5000, 3, 8193, 70_001, 16)
    gen = torch.Generator(device=gpu).manual_seed(4)
    init = [torch.empty(k, device=gpu).normal_(0.0, 0.02, generator=gen) for k in sizes]
    grads = [[torch.empty(k, device=gpu).normal_(0.0, 1e-3, generator=gen).half() for k in sizes] for _ in range(2)]
    taken = grads[1][:count] + grads[0][count:]

    def make(gs):
        ps = [torch.nn.Parameter(t.clone()) for t in init]
        opt = MultiTensorAdamWOptimizer(ps, lr=1e-3, param_dtype=torch.float16, device=gpu, max_grad_norm=1.0)
        for p, g in zip(ps, gs):
            p.grad = g
        return ps, opt

    (pa, a), (pb, b) = make(grads[0]), make(taken)
    b.step()
    a._plans()  # the table over grads[0]
    a.steps_issued += 1
    a._refresh_group_block()
    table = a.store.table()
    assert table.nchunks > 0 and a.store.small_table is None
    _lib.call("dsx_zero_step_multi_moved", table.tensors.data_ptr(), table.chunks.data_ptr(), table.nchunks, table.numel,
              table.pdt, table.gdt, a.dstate.data_ptr(), a.scaler.to_c(), ctypes.byref(a._gblock),
              a.partials.data_ptr(), a.nparts, a.scalars.data_ptr(),
              (ctypes.c_void_p * count)(*[g.data_ptr() for g in grads[1][:count]]), count, ops.stream_of(gpu))
    torch.cuda.synchronize()
    assert bytes(a.read_state()) == bytes(b.read_state())
    for x, y in zip(pa, pb):
        assert _bits(x.data, y.data)
        for key in ("master", "exp_avg", "exp_avg_sq"):
            assert _bits(a.state[x][key], b.state[y][key]), key
    refs = (_lib.DsxTensorRef * len(sizes)).from_buffer_copy(bytes(table.tensors.cpu().numpy()))
    assert [r.grad for r in refs] == [g.data_ptr() for g in taken]
