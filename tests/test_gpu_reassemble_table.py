"""The request table of the reassembly at its limits: as many requests in flight
as the context was made for, a table of a cell per request, tokens that share a
bucket, how much of the device it takes -- against requests collected in a dict."""
import ctypes as C

import numpy as np
import pytest
import torch

from splitrpc_amd import capi
from splitrpc_amd.engine import RingRef, SgContext, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SLOT, LEN = 64, 6


def _tokens(n, seed, buckets=1, bucket=0):
    """n tokens whose hash in the kernels (k ^= k >> 33; k *= M; k ^= k >> 33; the low bits) names one of `buckets`."""
    v = np.unique(np.random.default_rng(seed).integers(1, 1 << 62, 2 * n, dtype=np.uint64) // np.uint64(buckets) * np.uint64(buckets))
    v = np.random.default_rng(seed).permutation(v)[:n] + np.uint64(bucket)
    assert len(v) == n
    v ^= v >> np.uint64(33)
    with np.errstate(over="ignore"):
        v *= np.uint64(pow(0xff51afd7ed558ccd, -1, 1 << 64))
    return v ^ (v >> np.uint64(33))


class Stream:
    """One slot per fragment: slot r * per + i holds fragment i of request r."""

    def __init__(self, tokens, per, max_reqs, max_frames):
        n = len(tokens) * per
        ring = np.zeros((n, SLOT), np.uint8)
        at = lambda lo, a: ring.__setitem__((slice(None), slice(lo, lo + a.itemsize)), a.view(np.uint8).reshape(n, -1))
        at(42, np.repeat(tokens.astype(np.uint64), per))
        at(50, np.tile(np.arange(per, dtype=np.uint16), len(tokens)))
        at(52, np.full(n, per, np.uint16))
        at(54, np.full(n, LEN, np.uint32))
        self.tokens, self.per = tokens, per
        self.rx = RingRef(torch.from_numpy(ring).to(DEV), n, SLOT, 0)
        i32 = lambda k: torch.zeros(k, dtype=torch.int32, device=DEV)
        self.fs, self.fl, self.rf = i32(max_frames), i32(max_frames), i32(max_reqs + 1)
        self.tok = torch.zeros(max_reqs, dtype=torch.int64, device=DEV)
        self.counts = i32(4)
        self.parked = {}

    def call(self, ctx, slots):
        """One burst; what it must leave, and what it left."""
        done = []
        last = {}
        for i, s in enumerate(slots):
            r = int(s) // self.per
            self.parked.setdefault(r, set()).add(int(s))
            last[r] = i
        for r, _ in sorted(last.items(), key=lambda x: x[1]):
            if len(self.parked[r]) == self.per:
                done.append(r)
                del self.parked[r]
        n_req, n_frag, left = ctx.reassemble(self.rx, to_dev(np.ascontiguousarray(slots, np.uint32), DEV), len(slots), self.fs,
                                             self.fl, self.rf, self.tok, counts_out=self.counts)
        assert (n_req, n_frag, left, ctx.last_dropped) == (len(done), len(done) * self.per, len(self.parked), 0)
        want = (np.array(done, np.int64)[:, None] * self.per + np.arange(self.per)).reshape(-1)
        assert np.array_equal(self.fs[:n_frag].cpu().numpy(), want)
        assert bool((self.fl[:n_frag] == LEN).all())
        assert np.array_equal(self.rf[:n_req + 1].cpu().numpy(), np.arange(n_req + 1) * self.per)
        assert np.array_equal(self.tok[:n_req].cpu().numpy().view(np.uint64), self.tokens[done].astype(np.uint64))


# bursts that one workgroup of 256 threads takes, one of 1024, and three kernels
@pytest.mark.parametrize("burst", [200, 1000, 1 << 20], ids=["256", "1024", "kernels"])
@pytest.mark.parametrize("max_reqs", [4, 64, 100, 2048])
def test_all_the_requests_a_context_was_made_for(max_reqs, burst):
    """max_reqs requests in flight at once, three times over one table."""
    per = 3
    print(f"case table max_reqs={max_reqs} burst={burst}", flush=True)
    ctx = SgContext(0, max_reqs=max_reqs, max_frames=8192)
    for rep in range(3):
        st = Stream(_tokens(max_reqs, 10 * max_reqs + rep), per, max_reqs, 8192)
        rng = np.random.default_rng(5 + rep)
        # all but the last fragment of every request, then the last ones
        early = rng.permutation(np.concatenate([np.arange(max_reqs) * per + i for i in range(per - 1)]))
        late = rng.permutation(max_reqs) * per + per - 1
        for order in (early, late):
            for lo in range(0, len(order), burst):
                st.call(ctx, order[lo:lo + burst])
        assert not st.parked
    ctx.close()


BIG = 1 << 20  # requests: the table then has a cell each


def _took(max_reqs):
    ctx = SgContext(0, max_reqs=max_reqs, max_frames=1 << 21)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    ctx.reassemble_reset()
    return ctx, before - torch.cuda.mem_get_info()[0], before


@pytest.mark.parametrize("max_reqs", [1 << 10, 1 << 16, BIG])
def test_room_the_table_takes(max_reqs):
    """A record of 8 KiB for every request that may be in flight, and beyond that at most a 64th of what is free."""
    ctx, took, free = _took(max_reqs)
    assert took <= max_reqs * (8192 + 64) + free / 64 + (64 << 20), took
    ctx.close()


@pytest.mark.parametrize("share", [0.5, 0.99])
def test_a_table_of_a_cell_per_request(share):
    """Half and nearly all of the cells taken, six hundred tokens of one first bucket (of 32 cells) among the rest;
    then bursts of a few hundred over what that left of the table."""
    ctx, took, free = _took(BIG)
    if took > BIG * 2 * 8192:
        pytest.skip("so much memory that the table has more cells than requests")
    n = int(share * BIG)
    t = _tokens(n, 7)
    one = _tokens(600, 8, BIG // 32, 12345) if share < 0.9 else t[:0]
    t = np.unique(np.concatenate([t, one]))
    np.random.default_rng(9).shuffle(t)
    n = len(t)
    print(f"case table of {BIG} cells, {n} requests", flush=True)
    st = Stream(t, 2, BIG, 2 * n)
    rng = np.random.default_rng(10)
    early, late = rng.permutation(n), rng.permutation(n)
    call = lambda slots: ctx.reassemble(st.rx, to_dev(slots.astype(np.uint32), DEV), len(slots), st.fs, st.fl, st.rf, st.tok)
    assert call(2 * early) == (0, 0, n) and ctx.last_dropped == 0
    for lo, hi in ((0, 200), (200, 1100), (1100, n)):
        k = hi - lo
        assert call(2 * late[lo:hi] + 1) == (k, 2 * k, n - hi) and ctx.last_dropped == 0
        assert np.array_equal(st.fs[:2 * k].cpu().numpy().reshape(-1, 2), 2 * late[lo:hi, None] + np.arange(2))
        assert np.array_equal(st.tok[:k].cpu().numpy().view(np.uint64), t[late[lo:hi]])
    # the first bucket's tokens again, in the two kinds of bursts one workgroup takes
    few = np.flatnonzero(np.isin(t, one)) if len(one) else rng.permutation(n)[:600]
    for lo, hi in ((0, 250), (250, 600)):
        assert call(2 * few[lo:hi])[:2] == (0, 0)
    assert call(2 * few[::-1] + 1) == (600, 1200, 0)
    assert np.array_equal(st.fs[:1200].cpu().numpy().reshape(-1, 2), 2 * few[::-1, None] + np.arange(2))
    # launches sized for all of the arrivals, with fewer of them there
    arr = to_dev((2 * early).astype(np.uint32), DEV)
    for k in (0, 700, n - 5):
        dev = torch.tensor([k], dtype=torch.int32, device=DEV)
        assert ctx.reassemble(st.rx, arr, n, st.fs, st.fl, st.rf, st.tok, n_arrivals_dev=dev) == (0, 0, k)
        assert int(st.rf[0]) == 0 and ctx.reassemble_evict(0) == k
    ctx.close()


def test_a_table_of_more_records_than_a_launch_has_threads():
    """Eight million requests: 2^32 pairs of entries to empty."""
    max_reqs = 1 << 23
    if torch.cuda.mem_get_info()[0] < 90 << 30:
        pytest.skip("the table takes 64 GiB")
    print("case table of 2^23 cells", flush=True)
    ctx = SgContext(0, max_reqs=max_reqs, max_frames=4096)
    t = _tokens(2000, 11)
    st = Stream(t, 2, 4096, 4096)
    slots = np.random.default_rng(12).permutation(4000)
    for _ in range(2):
        st.call(ctx, slots[:3000])
        st.parked.clear()
        ctx.reassemble_reset()
    st.call(ctx, slots[:3100])
    st.call(ctx, slots[3100:])
    assert not st.parked
    ctx.close()


@pytest.mark.parametrize("max_reqs", [64, 1024], ids=["one-launch", "three-kernels"])
def test_requests_beyond_those_a_context_was_made_for(max_reqs):
    """A call may bring more requests than may be in flight if it completes enough of them; one that leaves more is
    refused, reports what it has handed over, and keeps the others."""
    full, part = max_reqs - 4, max_reqs // 2
    print(f"case table beyond max_reqs={max_reqs}", flush=True)
    ctx = SgContext(0, max_reqs=max_reqs, max_frames=8192)
    st = Stream(_tokens(full + part, 13), 2, max_reqs, 8192)
    rng = np.random.default_rng(14)
    st.call(ctx, rng.permutation(np.concatenate([np.arange(2 * full), 2 * np.arange(full, full + part)])))
    st.call(ctx, 2 * rng.permutation(np.arange(full, full + part)) + 1)
    assert not st.parked
    # twenty complete, one more than fit stays
    st = Stream(_tokens(20 + max_reqs + 1, 15), 2, max_reqs, 8192)
    slots = np.concatenate([np.arange(40), 2 * np.arange(20, 21 + max_reqs)]).astype(np.uint32)
    arr = to_dev(slots, DEV)
    counts = (C.c_uint32 * 4)()
    torch.cuda.synchronize()
    a = ctx.reassemble_args(st.rx, arr, len(slots), st.fs, st.fl, st.rf, st.tok, counts_out=st.counts)
    assert ctx.lib.sg_hip_reassemble(ctx.h, C.byref(a), C.byref(counts)) == capi.SG_E_DATA
    assert list(counts) == st.counts.cpu().tolist() == [20, 40, 0, max_reqs + 1]
    assert np.array_equal(st.fs[:40].cpu().numpy(), np.arange(40))
    st.parked = {r: {2 * r} for r in range(20, 21 + max_reqs)}
    late = 2 * rng.permutation(np.arange(20, 21 + max_reqs)) + 1
    st.call(ctx, late[:30])
    st.call(ctx, late[30:])
    assert not st.parked
    ctx.close()
