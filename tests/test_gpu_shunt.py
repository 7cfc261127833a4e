"""sg_hip_shunt_batch -- one pass of the shunter's loop, gather and scatter in
ONE launch where the two calls can share one -- against the CPU oracle's
gather followed by its scatter, bit for bit, through the C ABI: arenas, TX
ring, offsets and both bump-ring cursors, over calls in a row and over graph
replays.  Pairs of calls that cannot share a launch (sizes that differ, an
echo answered in place) must come out the same through the two-call path the
entry point then takes; the launches are counted."""
import numpy as np
import pytest
import torch

from splitrpc_amd import capi, synth
from splitrpc_amd.engine import AppRef, DeviceWorkload, SgContext

from helpers import expected_gather, expected_scatter, first_diff

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _args(ctx, dw, w, req_arena, req_cap, req_offs, resp_offs, flags=0, rule=True):
    """Argument blocks of a gather into `req_arena` and the workload's scatter."""
    fx = int(w.req_sizes[0])
    ga = ctx.gather_args(dw.rx, dw.frag_slot, dw.frag_len if w.profile else None, dw.req_first, dw.n_req, dw.n_frags,
                         AppRef(arena=req_arena, cap=req_cap) if req_arena is not None else dw.req_app, req_offs,
                         flags=flags | (capi.F_RULE_FRAGS if rule else 0), fixed_req_size=fx if rule else 0, mtu=w.mtu)
    rs = w.resp_sizes
    one = bool((rs == rs[0]).all())
    sa = ctx.scatter_args(dw.rx, dw.tx, dw.tx_slot, dw.hdr_src_slot, dw.resp_first, None if one else dw.resp_size,
                          int(rs[0]) if one else 0, dw.n_req, dw.n_frames, w.mtu, dw.resp_app, resp_offs,
                          w.flags | flags)
    return ga, sa


SHARED = {
    "resnet50-2": lambda p: synth.make_workload(2, 2, profile=p),
    "three-frames": lambda p: synth.make_custom([4200] * 40, [3000] * 40, seed=71, profile=p,
                                                flags=synth.F_UDP_CSUM_PSEUDO | synth.F_IPV4_CSUM),
    "full-udp-checksum": lambda p: synth.make_custom([2800] * 33, [2799] * 33, seed=72, profile=p,
                                                     flags=synth.F_UDP_CSUM_FULL | synth.F_IPV4_CSUM),
    "one-request": lambda p: synth.make_custom([1400 * 9 + 1], [1400], seed=73, profile=p),
    # short last fragments riding in the gather's half, eight short frames to a wavefront in the scatter's
    "lenet-9": lambda p: synth.make_workload(1, 9, profile=p),
    "lenet-1500": lambda p: synth.make_workload(1, 1500, profile=p),   # 6128 wavefronts
}


@pytest.mark.parametrize("profile", [synth.HDR_BL58, synth.HDR_REF64], ids=["bl58", "ref64"])
@pytest.mark.parametrize("name", list(SHARED))
def test_one_launch_moves_what_two_calls_move(name, profile):
    w = SHARED[name](profile)
    print(f"case shunt shared {name} profile={profile} n_req={w.n_req} frags={w.n_frags} frames={w.n_resp_frames}",
          flush=True)
    ctx = SgContext(0, max_reqs=8192, max_frames=1 << 17)
    dw = DeviceWorkload(w)
    total = int(w.req_sizes.sum())
    cap = 2 * total + 4096 + 10  # no whole number of batches fills the arena: the third call wraps
    arena = torch.zeros(cap, dtype=torch.uint8, device=DEV)
    offs = torch.zeros(w.n_req + 1, dtype=torch.int64, device=DEV)
    ga, sa = _args(ctx, dw, w, arena, cap, offs, dw.resp_offsets)
    rcur, tcur = 77 * 16 + 6, 0
    ctx.set_cursor(0, rcur)
    ctx.set_cursor(1, tcur)
    ctx.set_profiling(True)
    for call in range(3):
        arena.zero_()
        dw.tx_ring.copy_(torch.from_numpy(w.tx_ring_init).to(DEV))
        torch.cuda.synchronize()
        ctx.shunt_batch_raw(ga, sa)
        exp, eoffs, ecur = expected_gather(w, arena_cap=cap, cursor=rcur)
        got = arena.cpu().numpy()
        assert np.array_equal(got, exp), f"call {call}: " + first_diff(got, exp)
        assert np.array_equal(offs.cpu().numpy().view(np.uint64), eoffs)
        assert ctx.get_cursor(0) == ecur
        exp_tx, toffs, tnext = expected_scatter(w, None, resp_cap=dw.resp_app.cap, cursor=tcur)
        got = dw.tx_ring.cpu().numpy()
        assert np.array_equal(got, exp_tx), f"call {call}: " + first_diff(got, exp_tx)
        assert np.array_equal(dw.resp_offsets.cpu().numpy().view(np.uint64), toffs)
        assert ctx.get_cursor(1) == tnext
        rcur, tcur = ecur, tnext
    # one launch per call carried both directions
    assert ctx.kernel_time(1)[1] == 3 and ctx.kernel_time(2)[1] == 0 and ctx.kernel_time(0)[1] == 0
    ctx.close()


# (workload, whether its two calls share a launch; if not, how many descriptor passes they make)
PAIRS = {
    "jumbo": (lambda: synth.make_workload(5, 1), True),                     # frames of several wavefronts
    "short-frames-16-lanes": (lambda: synth.make_custom([300] * 50, [300] * 50, seed=78), True),
    "bert": (lambda: synth.make_workload(3, 20), True),                     # tensors; short last fragments
    "tensors-in": (lambda: synth.make_custom([4200] * 40, [3000] * 40, seed=82, in_tensor_sizes=[1500, 2700]), True),
    "tensors-out": (lambda: synth.make_custom([4200] * 40, [3000] * 40, seed=83, out_tensor_sizes=[2000, 1000]), True),
    # more wavefronts than the chip holds at once
    "lenet-4096": (lambda: synth.make_workload(1, 4096), True),
    "two-frames-3000": (lambda: synth.make_custom([4200] * 3000, [2800] * 3000, seed=77, flags=synth.F_UDP_CSUM_PSEUDO), True),
    # more than advance their cursor themselves: both halves, the gather's alone, the scatter's alone
    "wavefronts-70000": (lambda: synth.make_custom([1000] * 70000, [1000] * 70000, slot_size=1536, seed=84), True),
    "gather-of-75000": (lambda: synth.make_custom([4200] * 25000, [40] * 25000, slot_size=1536, seed=85), True),
    "scatter-of-75000": (lambda: synth.make_custom([40] * 25000, [4200] * 25000, slot_size=1536, seed=86), True),
    "mixed-echo": (lambda: synth.make_workload(4, 50), 2),                  # variable sizes, answered in place
    "sizes-differ": (lambda: synth.make_custom([4200] * 12, [100 + 333 * k for k in range(12)], seed=74), 1),
}


@pytest.mark.parametrize("name", list(PAIRS))
def test_pairs_come_out_the_same_in_one_launch_or_two(name):
    w, shares = PAIRS[name][0](), PAIRS[name][1]
    print(f"case shunt pair {name} n_req={w.n_req} frags={w.n_frags} frames={w.n_resp_frames}", flush=True)
    ctx = SgContext(0, max_reqs=1 << 17, max_frames=1 << 17)
    dw = DeviceWorkload(w, arena_slack=0 if w.tx_in_place else 72)
    one_size = bool((w.req_sizes == w.req_sizes[0]).all())
    ga, sa = _args(ctx, dw, w, None, 0, dw.req_offsets, dw.resp_offsets, rule=one_size)
    rcap = 0 if w.out_tensor_sizes else dw.resp_app.cap
    if rcap and w.n_req > 1 and not w.tx_in_place:
        rcap = sa.app.arena_cap = rcap - 8  # a pass does not end where it began
    ctx.set_cursor(0, 0)
    ctx.set_cursor(1, 0)
    ctx.set_profiling(True)
    ctx.shunt_batch_raw(ga, sa)
    if shares is True:
        assert [ctx.kernel_time(k)[1] for k in range(3)] == [0, 1, 0]
    else:
        assert [ctx.kernel_time(k)[1] for k in range(3)] == [shares, 1, 1]
    if w.in_tensor_sizes:
        exp, _, _ = expected_gather(w)
        for t, e in zip(dw.in_tensors, exp):
            assert np.array_equal(t.cpu().numpy(), e)
        gathered, ecur = None, 0
    else:
        exp, eoffs, ecur = expected_gather(w, arena_cap=dw.req_app.cap)
        got = dw.req_arena.cpu().numpy()
        assert np.array_equal(got, exp), first_diff(got, exp)
        assert np.array_equal(dw.req_offsets.cpu().numpy().view(np.uint64), eoffs)
        gathered = exp
    assert ctx.get_cursor(0) == ecur
    exp_tx, toffs, tcur = expected_scatter(w, gathered, resp_cap=rcap or None)
    got = dw.tx_ring.cpu().numpy()
    assert np.array_equal(got, exp_tx), first_diff(got, exp_tx)
    if w.out_tensor_sizes:
        tcur = 0
    else:
        assert np.array_equal(dw.resp_offsets.cpu().numpy().view(np.uint64), toffs)
    assert ctx.get_cursor(1) == tcur
    ctx.close()


# (request bytes, response bytes, mtu, slot size): every shape of either half at least once, beside different shapes of
# the other -- short fragments 8, 16 and 32 lanes each, whole and long fragments with and without short last ones;
# short frames, whole and long frames with and without short last ones
ANY_SHAPE = [
    (100, 100, 1400, 2048), (300, 300, 1400, 2048), (900, 900, 1400, 2048),
    (2800, 1400 + 100, 1400, 2048), (2 * 1400 + 336, 1400 + 272, 1400, 2048), (1400 + 648, 2800 + 900, 1400, 2048),
    (1399, 128, 1400, 2048), (128, 2800, 1400, 2048), (17, 16, 1400, 2048),
    (17600, 17600, 8800, 9216), (8800 + 300, 8800 + 272, 8800, 9216), (8800 + 901, 8801, 8800, 9216), (17599, 129, 8800, 9216),
]


@pytest.mark.parametrize("n_req", [1, 37, 1100])
@pytest.mark.parametrize("sizes", ANY_SHAPE, ids=lambda s: f"{s[0]}-{s[1]}")
def test_every_shape_shares_a_launch(sizes, n_req):
    """Shapes beside each other in one launch, with the cursors advanced by the kernel (small calls) and by the one
    behind it (SG_F_TAIL_KERNEL on either half), the full UDP checksum on every second call."""
    size, resp, mtu, slot = sizes
    if n_req * (size + resp) > 6 << 20:
        n_req = 160
    profile = n_req & 1
    w = synth.make_custom([size] * n_req, [resp] * n_req, mtu=mtu, slot_size=slot, seed=size + resp, profile=profile)
    print(f"case shunt any {sizes} n_req={n_req}", flush=True)
    ctx = SgContext(0, max_reqs=8192, max_frames=1 << 14)
    dw = DeviceWorkload(w)
    total = int(w.req_sizes.sum())
    cap = 2 * total + 4096 + 10
    arena = torch.zeros(cap, dtype=torch.uint8, device=DEV)
    offs = torch.zeros(w.n_req + 1, dtype=torch.int64, device=DEV)
    ga, sa = _args(ctx, dw, w, arena, cap, offs, dw.resp_offsets, flags=capi.F_FORCE_SMALL)
    rcur, tcur = 6, 0
    ctx.set_cursor(0, rcur)
    ctx.set_cursor(1, tcur)
    ctx.set_profiling(True)
    g_flags, s_flags = ga.flags, sa.flags
    calls = [(0, 0), (0, capi.F_UDP_CSUM_FULL), (capi.F_TAIL_KERNEL, capi.F_IPV4_CSUM),
             (capi.F_TAIL_KERNEL, capi.F_UDP_CSUM_FULL), (0, capi.F_TAIL_KERNEL | capi.F_UDP_CSUM_PSEUDO)]
    for call, (gf, sf) in enumerate(calls):
        arena.zero_()
        dw.tx_ring.copy_(torch.from_numpy(w.tx_ring_init).to(DEV))
        torch.cuda.synchronize()
        ga.flags, sa.flags = g_flags | gf, s_flags | sf
        ctx.shunt_batch_raw(ga, sa)
        exp, eoffs, ecur = expected_gather(w, arena_cap=cap, cursor=rcur)
        got = arena.cpu().numpy()
        assert np.array_equal(got, exp), f"call {call}: " + first_diff(got, exp)
        assert np.array_equal(offs.cpu().numpy().view(np.uint64), eoffs)
        assert ctx.get_cursor(0) == ecur
        exp_tx, toffs, tnext = expected_scatter(w, None, resp_cap=dw.resp_app.cap, cursor=tcur, flags=sf & 0xf)
        got = dw.tx_ring.cpu().numpy()
        assert np.array_equal(got, exp_tx), f"call {call}: " + first_diff(got, exp_tx)
        assert np.array_equal(dw.resp_offsets.cpu().numpy().view(np.uint64), toffs)
        assert ctx.get_cursor(1) == tnext
        rcur, tcur = ecur, tnext
    assert ctx.kernel_time(1)[1] == len(calls) and ctx.kernel_time(2)[1] == 0 and ctx.kernel_time(0)[1] == 0
    ctx.close()


def test_halves_that_write_the_same_table_run_in_order():
    """One offsets table for both halves: the scatter's offsets are what it holds afterwards."""
    w = synth.make_custom([4200] * 300, [3000] * 300, seed=79)
    ctx = SgContext(0)
    dw = DeviceWorkload(w)
    ga, sa = _args(ctx, dw, w, None, 0, dw.req_offsets, dw.req_offsets)
    ctx.set_cursor(0, 0)
    ctx.set_cursor(1, 0)
    ctx.set_profiling(True)
    ctx.shunt_batch_raw(ga, sa)
    _, toffs, _ = expected_scatter(w, None, resp_cap=dw.resp_app.cap)
    assert np.array_equal(dw.req_offsets.cpu().numpy().view(np.uint64), toffs)
    assert ctx.kernel_time(1)[1] == 1 and ctx.kernel_time(2)[1] == 1
    ctx.close()


def test_refusals_come_through_either_half():
    w = synth.make_custom([4200] * 6, [3000] * 6, seed=75)
    ctx = SgContext(0)
    dw = DeviceWorkload(w)
    ga, sa = _args(ctx, dw, w, None, 0, dw.req_offsets, dw.resp_offsets)
    # refused by the host before anything is launched: cursors stay
    ctx.set_cursor(0, 64)
    ctx.set_cursor(1, 0)
    keep = sa.mtu
    sa.mtu = 0
    with pytest.raises(Exception) as e:
        ctx.shunt_batch_raw(ga, sa)
    assert e.value.code == capi.SG_E_INVAL
    sa.mtu = keep
    assert ctx.get_cursor(0) == 64 and ctx.get_cursor(1) == 0
    assert ctx.lib.sg_hip_shunt_batch(ctx.h, None, None) == capi.SG_E_INVAL
    # refused by the device: a bad slot index on the gather's side is reported, the scatter's frames are out
    from splitrpc_amd.engine import to_dev
    bad = w.frag_slot.copy()
    bad[4] = w.n_slots + 3
    bad_dev = to_dev(bad, DEV)
    ga.frag_slot = bad_dev.data_ptr()
    with pytest.raises(Exception) as e:
        ctx.shunt_batch_raw(ga, sa)
    assert e.value.code == capi.SG_E_DATA
    exp_tx, _, _ = expected_scatter(w, None, resp_cap=dw.resp_app.cap)
    assert np.array_equal(dw.tx_ring.cpu().numpy(), exp_tx)
    ctx.close()


@pytest.mark.parametrize("n_req", [6, 3000], ids=["small", "large"])
@pytest.mark.parametrize("shared", [True, False], ids=["one-launch", "two-calls"])
def test_what_a_refused_gather_leaves_of_the_scatter(shared, n_req):
    """In a shared launch of any size the scatter has run and both cursors are on; a pair made as two synchronous calls
    ends with the gather."""
    from splitrpc_amd.engine import to_dev
    w = synth.make_custom([4200] * n_req, [3000] * n_req, seed=80)
    ctx = SgContext(0)
    dw = DeviceWorkload(w, arena_slack=64)
    # (one offsets table for both halves keeps them apart)
    ga, sa = _args(ctx, dw, w, None, 0, dw.req_offsets, dw.resp_offsets if shared else dw.req_offsets)
    rcap = sa.app.arena_cap = dw.resp_app.cap - 100  # the responses do not fill it evenly
    bad = w.frag_slot.copy()
    bad[4] = w.n_slots + 3
    bad_dev = to_dev(bad, DEV)
    ga.frag_slot = bad_dev.data_ptr()
    ctx.set_cursor(0, 0)
    ctx.set_cursor(1, 0)
    torch.cuda.synchronize()
    with pytest.raises(Exception) as e:
        ctx.shunt_batch_raw(ga, sa)
    assert e.value.code == capi.SG_E_DATA
    exp, _, ecur = expected_gather(w, arena_cap=dw.req_app.cap)
    exp = exp.copy()
    exp[4 * 1400:5 * 1400] = 0  # the fragment that is not there (4200 = 3 * 1400)
    assert np.array_equal(dw.req_arena.cpu().numpy(), exp) and ctx.get_cursor(0) == ecur
    exp_tx, _, tcur = expected_scatter(w, None, resp_cap=rcap)
    assert ecur and tcur
    assert np.array_equal(dw.tx_ring.cpu().numpy(), exp_tx if shared else w.tx_ring_init)
    assert ctx.get_cursor(1) == (tcur if shared else 0)
    ctx.close()


@pytest.mark.parametrize("n_req", [500, 1150000], ids=["one-launch", "two-launches"])
def test_more_wavefronts_than_a_launch_takes(n_req):
    """Either half within what a launch takes (30 wavefronts per fragment by its mtu), both together not: two launches.
    Every request comes from one slot, every response goes to one."""
    mtu, slot, size = 60000, 60064, 16
    w = synth.make_custom([size], [size], mtu=mtu, slot_size=slot, seed=81)
    print(f"case shunt many wavefronts n_req={n_req}", flush=True)
    ctx = SgContext(0, max_reqs=n_req, max_frames=n_req)
    dw = DeviceWorkload(w)
    i32 = lambda t: t.to(torch.int32).to(DEV)
    zero, one = i32(torch.zeros(n_req)), i32(torch.arange(n_req + 1))
    frag, tx = zero + int(w.frag_slot[0]), zero + int(w.tx_slot[0])
    cap = n_req * size + 100
    arena = torch.zeros(cap, dtype=torch.uint8, device=DEV)
    resp = dw.resp_arena[:size].repeat(n_req + 1)
    flags = capi.F_NO_SMALL
    ga = ctx.gather_args(dw.rx, frag, None, one, n_req, n_req, AppRef(arena=arena, cap=cap), None,
                         flags=flags | capi.F_RULE_FRAGS, fixed_req_size=size, mtu=mtu)
    sa = ctx.scatter_args(dw.rx, dw.tx, tx, zero + int(w.hdr_src_slot[0]), one, None, size, n_req, n_req, mtu,
                          AppRef(arena=resp, cap=(n_req + 1) * size), None, w.flags | flags)
    ctx.set_cursor(0, 0)
    ctx.set_cursor(1, 0)
    ctx.set_profiling(True)
    torch.cuda.synchronize()
    ctx.shunt_batch_raw(ga, sa)
    assert bool((arena[:n_req * size].view(n_req, size) == torch.from_numpy(w.req_payload).to(DEV)).all())
    assert not bool(arena[n_req * size:].any())
    exp_tx, _, _ = expected_scatter(w, None, resp_cap=dw.resp_app.cap)
    assert np.array_equal(dw.tx_ring.cpu().numpy(), exp_tx)
    assert ctx.get_cursor(0) == n_req * size and ctx.get_cursor(1) == n_req * size
    assert ctx.kernel_time(1)[1] == 1 and ctx.kernel_time(2)[1] == (0 if n_req < 1000 else 1)
    ctx.close()


def test_shunt_calls_recorded_into_a_graph_continue_both_rings():
    """Three calls of one launch each in one graph; every replay continues both
    bump rings where the last one stopped, with eager work in between."""
    w = synth.make_custom([4200] * 10, [3000] * 10, seed=76, flags=synth.F_UDP_CSUM_PSEUDO)
    s = torch.cuda.Stream()
    ctx = SgContext(0, stream=s.cuda_stream)
    dw = DeviceWorkload(w)
    total = int(w.req_sizes.sum())
    cap = 3 * total + 1234
    arena = torch.zeros(cap, dtype=torch.uint8, device=DEV)
    offs = torch.zeros(w.n_req + 1, dtype=torch.int64, device=DEV)
    ga, sa = _args(ctx, dw, w, arena, cap, offs, dw.resp_offsets, flags=capi.F_ASYNC)
    ctx.set_cursor(0, 0)
    ctx.set_cursor(1, 0)
    ctx.shunt_batch_raw(ga, sa)  # warm
    ctx.sync()
    ctx.set_cursor(0, 0)
    ctx.set_cursor(1, 0)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        for _ in range(3):
            ctx.shunt_batch_raw(ga, sa)
    rcur = 0
    for rep in range(4):
        arena.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for _ in range(3):
            _, eoffs, rcur = expected_gather(w, arena_cap=cap, cursor=rcur)
        got = arena.cpu().numpy()
        # the three calls of a replay lay the batch down three times, one behind the other
        c = (rcur - 3 * total) % cap
        idx = np.zeros(cap, bool)
        idx[(c + np.arange(3 * total)) % cap] = True
        lin = np.concatenate([w.req_payload] * 3)
        assert np.array_equal(got[(c + np.arange(3 * total)) % cap], lin), f"replay {rep}"
        assert not got[~idx].any()
        assert np.array_equal(offs.cpu().numpy().view(np.uint64), eoffs)
        ctx.sync()
        assert ctx.get_cursor(0) == rcur
        assert ctx.get_cursor(1) == 0  # three whole passes over the responses
        exp_tx, _, _ = expected_scatter(w, None, resp_cap=dw.resp_app.cap)
        assert np.array_equal(dw.tx_ring.cpu().numpy(), exp_tx)
        junk = torch.full((1 << 18,), rep, dtype=torch.uint8, device=DEV)
        assert int(junk[7]) == rep
    ctx.close()
