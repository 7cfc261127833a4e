"""The size of a ring changes nothing in what a call moves: the same small batch
in a ring of its own size and at the head of a ring of more than 128 MB, by
every route -- separate calls and one launch, declared rule and descriptor pass,
arena and tensors, short, full and long fragments -- against the oracle."""
import numpy as np
import pytest
import torch

from splitrpc_amd import capi, synth
from splitrpc_amd.engine import DeviceWorkload, RingRef, SgContext

from helpers import expected_gather, expected_scatter, first_diff

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FULL = synth.F_UDP_CSUM_FULL | synth.F_IPV4_CSUM
BATCHES = {
    "full-and-remainder": dict(sizes=[3136] * 70, resp_sizes=[3000] * 70, flags=FULL),
    "short": dict(sizes=[300] * 90, resp_sizes=[40] * 90, flags=synth.F_UDP_CSUM_PSEUDO),
    "tensors": dict(sizes=[2048] * 40, resp_sizes=[3072] * 40, in_tensor_sizes=[1024, 1024], out_tensor_sizes=[3072], flags=0),
    "jumbo": dict(sizes=[20001] * 9, resp_sizes=[17000] * 9, mtu=8800, slot_size=9216, flags=FULL),
}


@pytest.mark.parametrize("beyond", [False, True], ids=["own-size", "beyond-128MB"])
@pytest.mark.parametrize("route", ["shunt", "rule", "scan"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_same_bytes_whatever_the_ring(name, route, beyond):
    w = synth.make_custom(seed=310, **BATCHES[name])
    dw = DeviceWorkload(w)
    slots = (128 << 20) // w.slot_size + 1

    def ring(t, n):
        if not beyond:
            return t, RingRef(t, n, w.slot_size, w.profile)
        big = torch.zeros(slots * w.slot_size, dtype=torch.uint8, device=DEV)
        big[:t.numel()].copy_(t)
        return big, RingRef(big, slots, w.slot_size, w.profile)

    rx_t, dw.rx = ring(dw.ring, w.n_slots)
    tx_t, dw.tx = ring(dw.tx_ring, w.tx_n_slots)
    ctx = SgContext(0, max_reqs=256, max_frames=4096)
    torch.cuda.synchronize()
    if route == "shunt":
        dw.shunt(ctx)
    else:
        dw.gather(ctx, rule=route == "rule", fixed=route == "rule")
        dw.scatter(ctx, fuse=route == "rule", fixed=route == "rule")
    exp, _, _ = expected_gather(w, arena_cap=None if w.in_tensor_sizes else dw.req_app.cap)
    got = [t.cpu().numpy() for t in dw.in_tensors] if w.in_tensor_sizes else [dw.req_arena.cpu().numpy()]
    for g, e in zip(got, exp if w.in_tensor_sizes else [exp]):
        assert np.array_equal(g, e), first_diff(g, e)
    exp_tx, _, _ = expected_scatter(w, None)
    got = tx_t.cpu().numpy()
    assert np.array_equal(got[:exp_tx.size], exp_tx), first_diff(got[:exp_tx.size], exp_tx)
    assert not got[exp_tx.size:].any()
    ctx.close()
