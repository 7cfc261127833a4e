"""A fragment that crosses the end of an arena mapped once, in an arena that
holds no more than its request: the request starts anywhere in it, also at its
last byte, so that a byte's place reaches almost twice the capacity before it is
folded.  Gather and scatter, frames of one wavefront and of several, the
descriptor pass and the declared rule, the checksum over the split payload."""
import numpy as np
import pytest
import torch

import oracle
from splitrpc_amd import capi, synth
from splitrpc_amd.engine import AppRef, DeviceWorkload, to_dev

from helpers import first_diff

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("mode", ["scan", "rule"])
@pytest.mark.parametrize("mtu,slot,size", [(1400, 2048, 1001), (1400, 2048, 1400), (1400, 2048, 1401), (8800, 9216, 8800), (8800, 9216, 12345)])
def test_a_request_as_large_as_its_arena(ctx, mtu, slot, size, mode):
    rule = mode == "rule"
    w = synth.make_custom([size], [size], mtu=mtu, slot_size=slot, seed=size, flags=synth.F_IPV4_CSUM | synth.F_UDP_CSUM_FULL)
    dw = DeviceWorkload(w)
    offs = torch.zeros(2, dtype=torch.int64, device=DEV)
    for start in sorted({0, 1, 63, 64, 65, size // 2, size - 65, size - 2, size - 1}):
        print(f"case size {size} {mode} start {start}", flush=True)
        arena = torch.zeros(size, dtype=torch.uint8, device=DEV)
        ctx.set_cursor(0, start)
        ctx.gather_batch(dw.rx, dw.frag_slot, None, dw.req_first, 1, dw.n_frags, AppRef(arena=arena, cap=size), offs,
                         flags=capi.F_RULE_FRAGS if rule else 0, fixed_req_size=size if rule else 0, mtu=mtu)
        want, _, cur = oracle.gather(w, arena_cap=size, cursor=start, out=np.zeros(size, np.uint8))
        got = arena.cpu().numpy()
        assert np.array_equal(got, want), f"gather at {start}: " + first_diff(got, want)
        assert ctx.get_cursor(0) == cur == start
        # the response out of an arena like it
        src = np.roll(w.resp_payload, start)
        dw.tx_ring.copy_(to_dev(w.tx_ring_init, DEV))
        ctx.set_cursor(1, start)
        ctx.scatter_batch(dw.rx, dw.tx, dw.tx_slot, dw.hdr_src_slot, dw.resp_first, None, size, 1, dw.n_frames, mtu,
                          AppRef(arena=to_dev(src, DEV), cap=size), flags=w.flags | (0 if rule else capi.F_NO_FUSE))
        tx = w.tx_ring_init.copy()
        oracle.scatter(w, w.ring, tx, src, arena_cap=size, cursor=start)
        got = dw.tx_ring.cpu().numpy()
        assert np.array_equal(got, tx), f"scatter at {start}: " + first_diff(got, tx)
        assert ctx.get_cursor(1) == start
