"""The descriptor pass whose workgroups add up the sizes before their own (few
requests, sizes or lengths in a table) on both sides of the sizes where it
gives way to a scan kernel, in every shape of the descriptor kernel, against
the CPU oracle: bytes, offsets and cursors, with a cursor that starts anywhere
and an arena that the batch wraps around."""
import numpy as np
import pytest
import torch

from splitrpc_amd import synth
from splitrpc_amd.engine import DeviceWorkload, SgContext

from helpers import expected_gather, expected_scatter, first_diff

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _sizes(n, frags, seed):
    """n sizes of about `frags` fragments of 64 bytes each, an empty request now and then."""
    rng = np.random.default_rng(seed)
    s = rng.integers(1, 128 * frags, size=n)
    s[rng.random(n) < 0.02] = 0
    s[0] = 64 * frags
    return s


# (requests, fragments of each on average): 16, 32 and 64 lanes per request, workgroups of 256 and 1024; one request;
# 16384 fragments (gather) and one more
SHAPES = [(1, 3), (15, 2), (17, 2), (130, 6), (61, 12), (9, 24), (5, 60), (7, 400), (16384, 1), (16385, 1), (700, 23), (1000, 17)]


@pytest.mark.parametrize("n_req,frags", SHAPES)
def test_offsets_of_a_batch_with_tables(n_req, frags):
    if n_req >= 16384:
        sizes = np.full(n_req, 33)
        sizes[::3] = 17
        resp = sizes[::-1].copy()
    else:
        sizes, resp = _sizes(n_req, frags, n_req), _sizes(n_req, frags, n_req + 1)
    w = synth.make_custom(sizes, resp, mtu=64, slot_size=128, seed=n_req, order="perm_within_request")
    print(f"case offsets n_req={n_req} frags={w.n_frags} frames={w.n_resp_frames}", flush=True)
    ctx = SgContext(0, max_reqs=n_req + 1, max_frames=max(w.n_frags, w.n_resp_frames) + 1)
    dw = DeviceWorkload(w, arena_slack=1001)
    cap, rcap = dw.req_app.cap, dw.resp_app.cap
    rcur, tcur = cap - 700, rcap - 5
    ctx.set_cursor(0, rcur)
    ctx.set_cursor(1, tcur)
    for _ in range(2):
        dw.req_arena.zero_()
        torch.cuda.synchronize()
        dw.gather(ctx, use_frag_len=True, fixed=False)
        exp, offs, rcur = expected_gather(w, arena_cap=cap, cursor=rcur)
        got = dw.req_arena.cpu().numpy()
        assert np.array_equal(got, exp), first_diff(got, exp)
        assert np.array_equal(dw.req_offsets.cpu().numpy().view(np.uint64), offs)
        assert ctx.get_cursor(0) == rcur
        dw.scatter(ctx, fixed=False)
        exp_tx, toffs, tcur = expected_scatter(w, None, resp_cap=rcap, cursor=tcur)
        got = dw.tx_ring.cpu().numpy()
        assert np.array_equal(got, exp_tx), first_diff(got, exp_tx)
        assert np.array_equal(dw.resp_offsets.cpu().numpy().view(np.uint64), toffs)
        assert ctx.get_cursor(1) == tcur
    ctx.close()


# frames of each response, and how many of those are still added up (the descriptor kernels of 16, 32 and 64 lanes per
# request, workgroups of 256 and of 1024 threads)
LINES = [(1, 12288), (8, 12288), (9, 10240), (16, 10240), (17, 12288), (32, 12288), (33, 6144), (40, 6144), (257, 640)]


@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("frames,line", LINES)
def test_responses_on_both_sides_of_the_line(frames, line, over):
    n = line + over
    resp = np.full(n, 16 * frames - 3)
    resp[::2] -= 5
    w = synth.make_custom(np.full(n, 8), resp, mtu=16, slot_size=96, seed=frames)
    print(f"case offsets frames={frames} n={n}", flush=True)
    ctx = SgContext(0, max_reqs=n, max_frames=w.n_resp_frames)
    dw = DeviceWorkload(w, arena_slack=1001)
    rcap = dw.resp_app.cap
    tcur = rcap - 5
    ctx.set_cursor(1, tcur)
    dw.scatter(ctx, fixed=False)
    exp_tx, toffs, tcur = expected_scatter(w, None, resp_cap=rcap, cursor=tcur)
    got = dw.tx_ring.cpu().numpy()
    assert np.array_equal(got, exp_tx), first_diff(got, exp_tx)
    assert np.array_equal(dw.resp_offsets.cpu().numpy().view(np.uint64), toffs)
    assert ctx.get_cursor(1) == tcur
    ctx.close()
