"""The per-request entry points on both sides of the table sizes up to which a
table travels with the launch (32 runs, 64 headers), short and long tables in
turns, against plain copies and the CPU oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from splitrpc_amd import synth

from helpers import first_diff

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_run_tables_short_and_long_in_turns(ctx):
    rng = np.random.default_rng(500)
    src_h = rng.integers(0, 256, 1 << 19, dtype=np.uint8)
    src = torch.from_numpy(src_h).to(DEV)
    dst = torch.zeros(1 << 19, dtype=torch.uint8, device=DEV)
    want = np.zeros(1 << 19, np.uint8)
    at = 5
    for n in (1, 32, 33, 2, 4, 5, 31, 100, 32):
        print(f"case run table of {n}", flush=True)
        lens = rng.integers(0, 1500, size=n)
        lens[0] = 20000 if n == 31 else lens[0]  # two pieces: 32 runs
        d = at + np.concatenate([[0], np.cumsum(lens + 3)[:-1]])
        s = rng.integers(0, (1 << 19) - 20001, size=n)
        ctx.copy_runs([src.data_ptr() + int(x) for x in s], [dst.data_ptr() + int(x) for x in d], [int(x) for x in lens])
        for a, b, k in zip(s, d, lens):
            want[b:b + k] = src_h[a:a + k]
        at = int(d[-1] + lens[-1]) + 7
        got = dst.cpu().numpy()
        assert np.array_equal(got, want), f"{n} runs: " + first_diff(got, want)


@pytest.mark.parametrize("profile", [synth.HDR_BL58, synth.HDR_REF64])
@pytest.mark.parametrize("template", [False, True])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 200])
def test_header_tables(ctx, n, template, profile):
    rng = np.random.default_rng(n)
    slot, hl, mtu, token = 128, synth.hdr_len(profile), 1400, 0x1122334455667788
    flags = synth.F_IPV4_CSUM | synth.F_UDP_CSUM_PSEUDO
    buf = rng.integers(0, 256, n * slot, dtype=np.uint8)
    buf.reshape(n, slot)[:, 14] = 0x45
    tmpl = rng.integers(0, 256, 64, dtype=np.uint8)
    tmpl[14] = 0x45
    dev = torch.from_numpy(buf).to(DEV)
    size = (n - 1) * mtu + 77
    ptrs = [dev.data_ptr() + i * slot for i in range(n)]
    if template:
        ctx.set_hdrs(ptrs, tmpl.tobytes(), token, profile, size, mtu, flags)
    else:
        ctx.swap_hdrs(ptrs, profile, size, mtu, flags)
    want = buf.copy().reshape(n, slot)
    L = oracle.lib()
    for i in range(n):
        length = L.sgo_frame_len(size, mtu, i)
        h = want[i, :64].copy()
        p = h.ctypes.data_as(C.c_void_p)
        if template:
            L.sgo_template_resp_hdr(p, tmpl.ctypes.data_as(C.c_void_p), profile, flags, token, i, n, length)
        else:
            L.sgo_rewrite_resp_hdr(p, profile, flags, i, n, length)
        want[i, :hl] = h[:hl]
    got = dev.cpu().numpy().reshape(n, slot)
    assert np.array_equal(got, want), first_diff(got.reshape(-1), want.reshape(-1))
