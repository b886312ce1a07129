"""K2 on fp32 state in pinned host memory (dsx_adamw_host_state): the same bits
as K2 on the same state in HBM, at the edges of its slots, trips and grid, and
through the offloaded step; host memory that is not pinned is refused by the
entry point and staged by the streamer, as is pinned memory off K2's alignment."""
from __future__ import annotations

import sys

import pytest

pytestmark = pytest.mark.gpu

TRIP = 256 * 2 * 4  # elements of a block's trip


def _say(msg):
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


def _inputs(n, gdt, pdt, gpu, seed):
    import torch
    gen = torch.Generator(device=gpu).manual_seed(seed)
    p, m = (torch.empty(n, device=gpu).normal_(0.0, 0.02, generator=gen) for _ in range(2))
    v = torch.empty(n, device=gpu).uniform_(0.0, 1e-6, generator=gen)
    g = torch.empty(n, device=gpu).normal_(0.0, 1e-3, generator=gen).to(gdt)
    return p, m, v, (p.to(pdt) if pdt is not None else None), g


def _scalars(gpu, skip=0):
    from distributedspeed_amd import ops
    from distributedspeed_amd._lib import DsxStepScalars
    sc = DsxStepScalars()
    sc.inv_scale, sc.clip_coef, sc.decay, sc.w1, sc.w1c = 1.0, 0.5, 0.9999, 0.1, 0.9
    sc.b2, sc.val2, sc.eps, sc.bc2s, sc.nss, sc.skip = 0.999, 0.001, 1e-8, 0.3, -1e-3, skip
    return ops.scalars_from_host(sc, gpu)


def _pinned(t):
    import torch
    from distributedspeed_amd.offload import pinned_empty
    h = pinned_empty(t.numel())
    h.copy_(t)
    torch.cuda.synchronize()
    return h


def _bits(a, b):
    import torch
    return torch.equal(a.cpu().view(torch.uint8), b.cpu().view(torch.uint8))


@pytest.mark.parametrize("n", [1, 3, 4, 1023, TRIP + 5, 32 * TRIP, 32 * TRIP + 1, 70 * TRIP + 1031])
@pytest.mark.parametrize("gdt,pdt", [("bfloat16", "bfloat16"), ("float16", "float16"), ("float32", None)])
def test_pinned_state_gives_the_bits_of_device_state(gpu, n, gdt, pdt):
    import torch
    from distributedspeed_amd import ops
    _say(f"host state n={n} {gdt}")
    gdt, pdt = getattr(torch, gdt), getattr(torch, pdt) if pdt else None
    p, m, v, p16, g = _inputs(n, gdt, pdt, gpu, n)
    host = [_pinned(t) for t in (p, m, v)]
    o16 = p16.clone() if p16 is not None else None
    ops.adamw_host_state(*host, o16, g, _scalars(gpu, skip=1))  # moves nothing
    torch.cuda.synchronize()
    assert all(_bits(h, t) for h, t in zip(host, (p, m, v)))
    ops.adamw_host_state(*host, o16, g, _scalars(gpu))
    ops.adamw_flat(p, m, v, p16, g, _scalars(gpu))
    torch.cuda.synchronize()
    for name, h, t in zip(("master", "exp_avg", "exp_avg_sq"), host, (p, m, v)):
        assert _bits(h, t), name
    assert p16 is None or _bits(o16, p16)


@pytest.mark.parametrize("pinned", [True, False])
def test_the_streamer_takes_pinned_and_pageable_state(gpu, pinned):
    import torch
    from distributedspeed_amd import _lib, ops
    from distributedspeed_amd.offload import HostStateStreamer
    n, cut = 100_040, 40_008
    p, m, v, p16, g = _inputs(n, torch.bfloat16, torch.bfloat16, gpu, 3)
    host = [_pinned(t) if pinned else t.cpu() for t in (p, m, v)]
    o16 = p16.clone()
    if not pinned:
        with pytest.raises(_lib.DsxError, match="not pinned"):
            ops.adamw_host_state(*host, o16, g, _scalars(gpu))
    st = HostStateStreamer(gpu, 8192)
    first, second = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    for s in (first, second):  # two steps on two streams, in order
        s.wait_stream(torch.cuda.current_stream(gpu))
        s.wait_stream(first)
        with torch.cuda.stream(s):
            st.run(tuple(host), o16, g, [(0, cut, _scalars(gpu)), (cut, n, _scalars(gpu))])
    for _ in range(2):
        ops.adamw_flat(p, m, v, p16, g, _scalars(gpu))
    torch.cuda.synchronize()
    assert st.last_bytes == 24 * n
    for name, h, t in zip(("master", "exp_avg", "exp_avg_sq"), host, (p, m, v)):
        assert _bits(h, t), name
    assert _bits(o16, p16)


@pytest.mark.parametrize("n,cut,nbuf", [(9_001, 0, 3), (10 * 4096 + 41, 5 * 4096 + 24, 3),
                                        (10 * 4096 + 41, 5 * 4096 + 24, 2)])
def test_pinned_state_off_k2s_alignment_is_staged(gpu, n, cut, nbuf):
    """Views that start 4 bytes into a pinned array: K2 reads 16 bytes at a
    time, so they take the staged path, as all pinned state once did. The larger
    ones are two pieces of 6 chunks each, two steps on end: every staging slot is
    filled, stepped and emptied four times a step or more, with copies that the
    host does not wait for."""
    import torch
    from distributedspeed_amd.offload import HostStateStreamer
    p, m, v, p16, g = _inputs(n, torch.bfloat16, torch.bfloat16, gpu, 5)
    host = [_pinned(torch.cat([t[:1], t]))[1:] for t in (p, m, v)]
    o16 = p16.clone()
    st = HostStateStreamer(gpu, 4096, nbuf)
    pieces = [(a, b, _scalars(gpu)) for a, b in ((0, cut), (cut, n)) if b > a]
    for _ in range(2):
        st.run(tuple(host), o16, g, pieces)
    assert st._stage is not None and st.last_bytes == 24 * n
    from distributedspeed_amd import ops
    for _ in range(2):
        ops.adamw_flat(p, m, v, p16, g, _scalars(gpu))
    torch.cuda.synchronize()
    for name, h, t in zip(("master", "exp_avg", "exp_avg_sq"), host, (p, m, v)):
        assert _bits(h, t), name
    assert _bits(o16, p16)


def _busy(gpu):
    """Work for the current stream that outlasts a few host calls by far."""
    import torch
    a = torch.ones(8192, 8192, device=gpu)
    for _ in range(60):
        a = (a @ a) * 0.0
    done = torch.cuda.Event()
    done.record()
    return done


def test_states_in_turn_do_not_block_the_host(gpu):
    """Two states in turn, and fresh views of one, through one streamer: run()
    returns while earlier work on the stream is still going on."""
    import torch
    from distributedspeed_amd import ops
    from distributedspeed_amd.offload import HostStateStreamer
    n = 10_008
    p, m, v, p16, g = _inputs(n, torch.bfloat16, torch.bfloat16, gpu, 11)
    states = [[_pinned(t) for t in (p, m, v)] for _ in range(2)]
    outs = [p16.clone() for _ in states]
    st = HostStateStreamer(gpu, 4096)
    sc = _scalars(gpu)
    _say("states in turn")
    st.run(tuple(states[0]), outs[0], g, [(0, n, sc)])
    torch.cuda.synchronize()
    done = _busy(gpu)
    st.run(tuple(states[1]), outs[1], g, [(0, n, sc)])
    st.run(tuple(t[:] for t in states[0]), outs[0], g, [(0, n, sc)])
    st.run(tuple(states[1]), outs[1], g, [(0, n, sc)])
    assert not done.query()
    torch.cuda.synchronize()
    for _ in range(2):
        ops.adamw_flat(p, m, v, p16, g, sc)
    torch.cuda.synchronize()
    for host, o16 in zip(states, outs):
        assert all(_bits(h, t) for h, t in zip(host, (p, m, v))) and _bits(o16, p16)


@pytest.mark.parametrize("torchs", [True, False])
def test_state_dropped_behind_a_step_outlives_it(gpu, torchs):
    """The streamer keeps no state, and a caller may drop it while the step is
    still to come: torch's pinned allocator does not hand out its memory before,
    and pinned_empty's is freed only then."""
    import torch
    import weakref
    from distributedspeed_amd import ops
    from distributedspeed_amd.offload import HostStateStreamer
    n = 1 << 16
    p, m, v, p16, g = _inputs(n, torch.bfloat16, torch.bfloat16, gpu, 12)
    o16 = p16.clone()
    host = [t.cpu().pin_memory() if torchs else _pinned(t) for t in (p, m, v)]
    gone, homes = [weakref.ref(t) for t in host], [t.data_ptr() for t in host]
    st = HostStateStreamer(gpu, 4096)
    sc = _scalars(gpu)
    spare = torch.full((n,), 7.0).pin_memory()  # written over whatever a too early reuse would give
    torch.cuda.synchronize()
    _say(f"dropped state, torch's allocator: {torchs}")
    done = _busy(gpu)
    st.run(tuple(host), o16, g, [(0, n, sc)])
    del host
    assert all(r() is None for r in gone)
    if torchs:
        new = [torch.empty(n, pin_memory=True) for _ in homes]
        for t in new:
            t.copy_(spare)
        assert not done.query()
        assert not {t.data_ptr() for t in new} & set(homes)
    else:
        assert done.query() and not set(homes) & set(ops.host_blocks)
    ops.adamw_flat(p, m, v, p16, g, sc)
    torch.cuda.synchronize()
    assert _bits(o16, p16)
    assert not torchs or all(torch.equal(t, spare) for t in new)


@pytest.mark.parametrize("start", [1, 2, 3, 4, 7])
def test_a_piece_off_k2s_alignment_is_staged(gpu, start):
    """A piece that starts where the 16-bit buffers are aligned and the fp32
    state is not (4 elements in, both are): staged, as every piece once was."""
    import torch
    from distributedspeed_amd import ops
    from distributedspeed_amd.offload import HostStateStreamer
    n = 9_001
    p, m, v, p16, g = _inputs(n, torch.bfloat16, torch.bfloat16, gpu, 13)
    host = [_pinned(t) for t in (p, m, v)]
    pad = 8 - start

    def at(t):  # t's values with element `start` on a 16-byte boundary
        return torch.cat([t[:1].expand(pad), t])[pad:]

    o16, og = at(p16), at(g)
    _say(f"piece from {start}")
    HostStateStreamer(gpu, 4096).run(tuple(host), o16, og, [(start, n, _scalars(gpu))])
    rest = [t[start:].clone() for t in (p, m, v, p16, g)]
    ops.adamw_flat(*rest, _scalars(gpu))
    torch.cuda.synchronize()
    for h, t, new in zip(host + [o16], (p, m, v, p16), rest):
        assert _bits(h[:start], t[:start]) and _bits(h[start:], new)
