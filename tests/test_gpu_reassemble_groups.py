"""The reassembly sorts each workgroup's arrivals by token before it goes to the
request table: streams at the sizes where that can go wrong -- one token per
workgroup or a token per arrival, groups on either side of the size that goes in
with one addition, records of one and of many steps, bursts on either side of
what the one-workgroup kernels take, more workgroups than a wavefront adds up at
a time -- against the oracle's table."""
import numpy as np
import pytest
import torch

import oracle
from splitrpc_amd import capi, synth
from splitrpc_amd.engine import RingRef, SgContext, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _stream(per_req, n_req, order, profile, seed=0):
    """n_req requests of per_req fragments of up to 16 bytes each."""
    return synth.make_custom([16 * per_req - 5] * n_req, [1] * n_req, mtu=16, slot_size=96, order=order,
                             seed=seed, profile=profile)


def _replay(w, bursts, max_reqs, max_frames):
    """The stream in calls of the given sizes: the calls' outputs laid end to end."""
    ctx = SgContext(0, max_reqs=max_reqs, max_frames=max_frames)
    ctx.reassemble_reset()
    rx = RingRef(torch.from_numpy(w.ring).to(DEV), w.n_slots, w.slot_size, w.profile)
    arr = to_dev(w.arrivals, DEV)
    ln = None
    if w.profile:
        nic = np.zeros(w.n_slots, np.uint32)
        nic[w.frag_slot] = w.frag_len
        ln = to_dev(nic, DEV)
    i32 = lambda n: torch.zeros(n, dtype=torch.int32, device=DEV)
    fs, fl, rf, hdr = i32(max_frames), i32(max_frames), i32(max_reqs + 1), i32(max_reqs)
    tok = torch.zeros(max_reqs, dtype=torch.int64, device=DEV)
    out, first, at = [[], [], [], []], [0], 0
    for n in bursts:
        n = min(n, len(w.arrivals) - at)
        n_req, n_frag, left = ctx.reassemble(rx, arr[at:at + n], n, fs, fl, rf, tok, ln,
                                             int(w.req_sizes[0]) if w.profile else 0, req_hdr_slot=hdr)
        at += n
        u = lambda t, k: t[:k].cpu().numpy().view(np.uint32)
        for o, g in zip(out, (u(fs, n_frag), u(fl, n_frag), tok[:n_req].cpu().numpy().view(np.uint64), u(hdr, n_req))):
            o.append(g)
        first.extend(int(x) + first[-1] for x in np.diff(u(rf, n_req + 1).astype(np.int64)))
    assert at == len(w.arrivals) and left == 0
    ctx.close()
    return [np.concatenate(o) for o in out] + [np.array(first, np.uint32)]


def _check(w, got):
    efs, efl, erf, etok = oracle.reassemble(w, req_size=int(w.req_sizes[0]) if w.profile else 0,
                                            frag_len_nic=_nic(w) if w.profile else None)
    for g, e, name in zip(got, (efs, efl, etok, efs[erf[:-1]], erf), ("slots", "lengths", "tokens", "headers", "first")):
        assert np.array_equal(g, e), name


def _nic(w):
    nic = np.zeros(w.n_slots, np.uint32)
    nic[w.frag_slot] = w.frag_len
    return nic


@pytest.mark.parametrize("profile", [synth.HDR_BL58, synth.HDR_REF64], ids=["bl58", "ref64"])
@pytest.mark.parametrize("order", ["in_order", "interleave_keep_order", "shuffle_all"])
@pytest.mark.parametrize("per_req", [1, 2, 7, 8, 9, 64, 256, 512, 513, 1023])
def test_tokens_per_workgroup_and_fragments_per_request(per_req, order, profile):
    n_req = max(2, -(-2600 // per_req))
    w = _stream(per_req, n_req, order, profile, seed=per_req)
    n = len(w.arrivals)
    print(f"case groups per_req={per_req} {order} profile={profile} arrivals={n}", flush=True)
    for bursts in ([n], [255, 256, 257, 1023, 1024, 1025] * (1 + n // 3840), [1] * 3 + [n]):
        _check(w, _replay(w, bursts, max_reqs=4096, max_frames=8192))


def test_more_workgroups_than_a_wavefront_adds_up_at_once():
    w = _stream(360, 400, "interleave_keep_order", synth.HDR_BL58)  # 144000 arrivals in one call: 563 workgroups
    print(f"case groups many workgroups arrivals={len(w.arrivals)}", flush=True)
    _check(w, _replay(w, [len(w.arrivals)], max_reqs=512, max_frames=1 << 18))


def test_output_tables_too_small_for_what_completes():
    """More requests complete in a call than the context's tables take: refused, nothing is handed
    over, the requests stay parked; the context goes on after a reset."""
    from splitrpc_amd.engine import SgError
    for n_req in (40, 400):                      # one workgroup; three kernels
        w = _stream(3, n_req, "in_order", synth.HDR_BL58)
        ctx = SgContext(0, max_reqs=32, max_frames=2048)
        rx = RingRef(torch.from_numpy(w.ring).to(DEV), w.n_slots, w.slot_size, w.profile)
        i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device=DEV)
        fs, fl, rf = i32(2048), i32(2048), i32(33)
        arr = to_dev(w.arrivals, DEV)
        with pytest.raises(SgError) as e:
            ctx.reassemble(rx, arr, len(w.arrivals), fs, fl, rf)
        assert e.value.code == capi.SG_E_DATA
        assert bool((fs == -7).all()) and int(rf[0]) == 0
        ctx.reassemble_reset()
        assert ctx.reassemble(rx, arr, 30, fs, fl, rf) == (10, 30, 0)
        assert np.array_equal(fs[:30].cpu().numpy().view(np.uint32), w.frag_slot[:30])
        ctx.close()
