"""How a per-request call learns that its launch is through: the launch writes
the call's number into pinned host memory, and the calling thread looks there
for a while before it waits through the runtime.  Calls that find it there,
calls behind work that outlasts the looking, calls with profiling on (which
wait for events), calls after a refusal, tables flushed half way; one workgroup
and many, tables that travel with the launch and tables in host memory.  The
destination is pinned host memory read on return, with nothing else waited for."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from splitrpc_amd import capi, synth
from splitrpc_amd.engine import DeviceWorkload, SgError, to_dev

from helpers import first_diff

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
RUN = 700


class Runs:
    """A table of n runs from device memory into pinned host memory."""

    def __init__(self, n, seed):
        self.n, self.h = n, np.random.default_rng(seed).integers(0, 256, n * RUN, dtype=np.uint8)
        self.src = torch.from_numpy(self.h).to(DEV)
        self.dst = torch.zeros(n * RUN, dtype=torch.uint8, pin_memory=True)

    def call(self, ctx):
        s, d = self.src.data_ptr(), self.dst.data_ptr()
        ctx.copy_runs([s + i * RUN for i in range(self.n)], [d + i * RUN for i in range(self.n)], [RUN] * self.n)

    def check(self, what):
        got = self.dst.numpy()
        assert np.array_equal(got, self.h), f"{what}: " + first_diff(got, self.h)


class Hdrs:
    """n headers in pinned host memory, filled from a template."""

    HL, MTU, TOKEN = synth.hdr_len(synth.HDR_BL58), 1400, 0x0102030405060708

    def __init__(self, n, seed):
        rng = np.random.default_rng(seed)
        self.n, self.size = n, n * self.MTU - 9
        self.tmpl = rng.integers(0, 256, 64, dtype=np.uint8)
        self.tmpl[14] = 0x45
        self.dst = torch.zeros(n * 64, dtype=torch.uint8, pin_memory=True)

    def call(self, ctx):
        ctx.set_hdrs([self.dst.data_ptr() + i * 64 for i in range(self.n)], self.tmpl.tobytes(), self.TOKEN,
                     synth.HDR_BL58, self.size, self.MTU, synth.F_IPV4_CSUM)

    def check(self, what):
        want = np.zeros((self.n, 64), np.uint8)
        for i in range(self.n):
            h = np.zeros(64, np.uint8)
            oracle.lib().sgo_template_resp_hdr(h.ctypes.data_as(C.c_void_p), self.tmpl.ctypes.data_as(C.c_void_p),
                                               synth.HDR_BL58, synth.F_IPV4_CSUM, self.TOKEN, i, self.n,
                                               oracle.lib().sgo_frame_len(self.size, self.MTU, i))
            want[i, :self.HL] = h[:self.HL]
        got = self.dst.numpy()
        assert np.array_equal(got, want.reshape(-1)), f"{what}: " + first_diff(got, want.reshape(-1))


TABLES = [(Runs, 1), (Runs, 32), (Runs, 300), (Hdrs, 1), (Hdrs, 64), (Hdrs, 300)]
IDS = [f"{k.__name__}-{n}" for k, n in TABLES]


def _refused_before(ctx):
    """An asynchronous batch with a slot index beyond its ring, left on the context's stream."""
    w = synth.make_workload(1, 4)
    dw = DeviceWorkload(w)
    bad = w.frag_slot.copy()
    bad[5] = w.n_slots + 3
    bad = to_dev(bad, DEV)
    ctx.gather_batch(dw.rx, bad, None, dw.req_first, dw.n_req, dw.n_frags, dw.req_app, dw.req_offsets, flags=capi.F_ASYNC)
    return dw, bad  # kept until the call is through


@pytest.mark.parametrize("kind,n", TABLES, ids=IDS)
def test_an_earlier_refusal_is_reported_once(ctx, kind, n):
    held = _refused_before(ctx)
    t = kind(n, 11)
    with pytest.raises(SgError) as e:
        t.call(ctx)
    assert e.value.code == capi.SG_E_DATA and "slot index" in str(e.value)
    t.check("the call that reports it")
    t = kind(n, 12)
    t.call(ctx)
    t.check("the call behind it")
    ctx.sync()
    del held


@pytest.mark.parametrize("kind,n", TABLES, ids=IDS)
def test_behind_work_that_outlasts_the_looking(ctx, kind, n):
    x = torch.zeros(64 << 20, dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    late = torch.cuda.ExternalStream(ctx.stream, device=DEV)
    for turn in range(2):
        with torch.cuda.stream(late):
            for _ in range(200):  # 200 passes over 64 MB: some milliseconds
                x.add_(1)
        t = kind(n, 20 + turn)
        if kind is Runs:
            t.src, t.h = x[:n * RUN], np.full(n * RUN, (200 * (turn + 1)) & 255, np.uint8)
        t.call(ctx)
        t.check(f"behind other work, turn {turn}")
        t = kind(n, 30 + turn)
        t.call(ctx)
        t.check(f"straight after it, turn {turn}")


@pytest.mark.parametrize("kind,n", TABLES, ids=IDS)
def test_profiling_between_calls(ctx, kind, n):
    which = 3 if kind is Runs else 4
    for turn, on in enumerate((False, True, True, False, True, False)):
        ctx.set_profiling(on)
        t = kind(n, 40 + turn)
        t.call(ctx)
        t.check(f"turn {turn}, profiling {on}")
        assert ctx.kernel_time(which)[1] == (1 if on else 0)
    ctx.set_profiling(False)


def test_a_table_of_more_pieces_than_the_staging_holds(ctx):
    """Long runs are cut into pieces of 16 KB; 8192 of them are launched by themselves, and only the
    last launch tells."""
    n, each = 40, 3500001  # 214 pieces a run, 8560 in all
    src = torch.randint(0, 256, (each + n,), dtype=torch.uint8, device=DEV)
    dst = torch.zeros(n * each, dtype=torch.uint8, device=DEV)
    ctx.copy_runs([src.data_ptr() + i for i in range(n)], [dst.data_ptr() + i * each for i in range(n)], [each] * n)
    for i in range(n):
        assert torch.equal(dst[i * each:(i + 1) * each], src[i:i + each]), f"run {i}"
    t = Runs(5, 50)
    t.call(ctx)
    t.check("a short table behind it")
