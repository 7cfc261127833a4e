"""Records whose first entries lie apart from the others (sg_hip_reassemble):
requests around that size, filed over two calls, dropped half filed and sent
again -- nothing of the dropped ones may show."""
import numpy as np
import pytest
import torch

import oracle
from splitrpc_amd import synth
from splitrpc_amd.engine import RingRef, SgContext, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FRAGMENTS = (1, 3, 4, 5, 8, 9, 64, 73, 431, 520, 1023)


@pytest.mark.parametrize("n_each", [1, 40], ids=["one-launch-and-more", "three-kernels"])
def test_requests_around_the_split_after_eviction(n_each):
    sizes = [n * 1400 - 3 for n in FRAGMENTS[:8 if n_each > 1 else None] for _ in range(n_each)]
    w = synth.make_custom(sizes, [64] * len(sizes), seed=320)
    ctx = SgContext(0, max_reqs=1024, max_frames=1 << 15)
    rx = RingRef(torch.from_numpy(w.ring).to(DEV), w.n_slots, w.slot_size, w.profile)
    n = len(w.arrivals)
    fs, fl = (torch.zeros(n, dtype=torch.int32, device=DEV) for _ in range(2))
    rf = torch.zeros(1025, dtype=torch.int32, device=DEV)
    tok = torch.zeros(1024, dtype=torch.int64, device=DEV)

    def call(arrivals):
        return ctx.reassemble(rx, to_dev(np.ascontiguousarray(arrivals, np.uint32), DEV), len(arrivals), fs, fl, rf, tok)

    ctx.reassemble_reset()
    # every second arrival: half filed requests, dropped
    call(w.arrivals[::2])
    ctx.reassemble_evict(0)
    # then all of them, in two calls: what the second completes comes in its order
    half = n // 2
    done = []
    for part in (w.arrivals[:half], w.arrivals[half:]):
        n_req, n_frag, left = call(part)
        first = rf[:n_req + 1].cpu().numpy().view(np.uint32)
        assert first[n_req] == n_frag
        slots, lens = fs[:n_frag].cpu().numpy().view(np.uint32), fl[:n_frag].cpu().numpy().view(np.uint32)
        for r in range(n_req):
            done.append((int(tok[r].item()), slots[first[r]:first[r + 1]].copy(), lens[first[r]:first[r + 1]].copy()))
    assert left == 0
    es, el, ef, et = oracle.reassemble(w, arrivals=w.arrivals)[:4]
    assert [t for t, _, _ in done] == [int(np.int64(np.uint64(t))) for t in et]
    assert np.array_equal(np.concatenate([s for _, s, _ in done]), es)
    assert np.array_equal(np.concatenate([x for _, _, x in done]), el)
    ctx.close()
