"""What the gather/scatter path is timed on: calls a server makes, through the
library's public entry points, from the smallest batch to the largest.

A case says what a server does per pass (``kind``) and at which sizes:

step      one pass of the shunter's loop on a batch of equal requests: the
          requests that became ready are gathered, the responses that are done
          are scattered (``sg_hip_shunt_batch``), offsets derived from the size
echo      requests of all sizes answered in place, from the same slots: a
          descriptor pass, the gather, the scatter over its descriptors
tables    the batched calls over fragment tables that the receive thread keeps
          in pinned host memory: pulled over the bus with tokens, response
          sizes and header templates, then requests and responses of all sizes
request   one request at a time, synchronously: gather its run table, fill the
          response headers, scatter the response
receive   the receive path: bursts of arrivals sorted into requests on the
          device, what a burst completed gathered and answered, nothing known
          to the host in between

Bytes come out the same whatever moves them, so every output is exact.
"""
import ctypes as C
import math

import numpy as np
import torch

from splitrpc_amd import capi, synth
from splitrpc_amd.engine import AppRef, DeviceWorkload, RingRef, SgContext, to_dev

ASYNC = capi.F_ASYNC
ORDERS = ("in_order", "perm_within_request", "interleave_keep_order", "shuffle_all")
# one served batch (requests) of the five workloads, the frame limits, and the sizes of a request and its response
WORKLOADS = {1: (32, 1400, 2048, 3136, 40),         # lenet: 28x28 fp32 -> 10 fp32
             2: (16, 1400, 2048, 602112, 4000),     # resnet50: 3x224x224 fp32 -> 1000 fp32
             3: (256, 1400, 2048, 2048, 3072),      # bert: ids + mask of 128 int64 -> 768 fp32
             4: (4096, 1400, 2048, 0, 0),           # mixed: 64 B .. 64 KiB, echoed
             5: (16, 8800, 9216, 1572864, 1048576)}  # segmentation in jumbo frames: fp16 image -> int32 classes


def _case(name, kind, workload, n_req, profile=0, burst=0, **more):
    base, mtu, slot, size, resp = WORKLOADS[workload] if workload else (0, 1400, 2048, 0, 0)
    c = {"name": name, "kind": kind, "workload": workload, "n_req": n_req, "profile": profile, "mtu": mtu, "slot": slot,
         "size": size, "resp": resp, "flags": 0, "order": "", "split": 0, "burst": burst}
    c.update(more)
    return c


def listed():
    return [
        # a lightly loaded server: one batch of the smallest model, all launch and latency
        _case("step_lenet_32", "step", 1, 32),
        # the batch a vision server forms: 16 images, 6896 frames, again mostly latency
        _case("step_resnet50_16", "step", 2, 16),
        # small requests of many clients in one call
        _case("step_lenet_8192", "step", 1, 8192),
        # 32 such vision batches in one call: what a loaded server moves at a time
        _case("step_resnet50_512", "step", 2, 512),
        # a text server: requests in two tensors, interleaved on the wire, three response frames each
        _case("step_bert_131072", "step", 3, 131072),
        # large images in jumbo frames, the UDP checksum over header and payload finished in software
        _case("step_jumbo_256", "step", 5, 256),
        # requests of all sizes, answered from the buffers they came in
        _case("echo_mixed_32768", "echo", 4, 32768, flags=synth.F_UDP_CSUM_PSEUDO),
        # the reference's header, ragged sizes, tables and templates kept by host threads
        _case("tables_ragged_1000", "tables", 0, 1000, profile=1, size=60000, resp=20000,
              flags=synth.F_IPV4_CSUM | synth.F_UDP_CSUM_PSEUDO),
        # the literal drop-in: a server that handles one request per call
        _case("request_resnet50", "request", 2, 1),
        # a NIC's bursts of 64, requests straddling them
        _case("receive_resnet50_4_by_64", "receive", 2, 4, burst=64),
        # many small requests, interleaved, in large bursts
        _case("receive_bert_131072_by_65536", "receive", 3, 131072, burst=65536),
        # a whole call's arrivals at once, lengths from the NIC as the reference's header needs them
        _case("receive_resnet50_ref64_512", "receive", 2, 512, profile=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "step", "step", "echo", "tables", "request", "receive", "receive"))
    profile = rng.randrange(2)
    flags = rng.choice((0, synth.F_UDP_CSUM_PSEUDO, synth.F_IPV4_CSUM | synth.F_UDP_CSUM_PSEUDO, synth.F_UDP_CSUM_FULL,
                        synth.F_IPV4_CSUM | synth.F_UDP_CSUM_FULL))
    mtu, slot = rng.choice(((1400, 2048), (1400, 2048), (1436, 1536), (8800, 9216)))
    order = rng.choice(ORDERS)
    split = 0
    burst = 0
    if kind in ("echo", "tables"):
        # sizes inside the call are spread from a few bytes to these
        size, resp = _log(rng, 4096, 65536), _log(rng, 1024, 65536)
        n_req = _log(rng, 16, 32768 if kind == "echo" else 4096)
    elif kind == "request":
        size, resp, n_req = _log(rng, 100, 1000000), _log(rng, 40, 100000), 1
    else:
        size, resp = _log(rng, 40, 1000000), _log(rng, 40, 200000)
        most = min(131072, 200000000 // (size + resp), 262144 // (-(-size // mtu) + -(-resp // mtu)))
        n_req = _log(rng, 1, max(2, most))
        if kind == "step" and size > 64 and rng.random() < 0.25:
            split = rng.randrange(16, size - 16)  # a request goes to two tensors
        if kind == "receive":
            arrivals = n_req * -(-size // mtu)
            burst = rng.choice((0, _log(rng, max(16, arrivals // 32), max(64, arrivals))))
    return _case("", kind, 0, n_req, profile=profile, burst=burst, mtu=mtu, slot=slot, size=size, resp=resp,
                 flags=flags, order=order, split=split)


# ---- inputs -----------------------------------------------------------------

def _ragged(seed, n, top, low):
    """n sizes spread evenly over the logarithm of low .. top, in an order of the seed's."""
    q = (np.arange(n) + 0.5) / n
    s = np.rint(np.exp(math.log(low) + q * (math.log(top) - math.log(low)))).astype(np.int64)
    return np.random.default_rng(seed).permutation(s)


def _sizes(case, seed):
    """Request and response sizes of one call, in bytes."""
    n = case["n_req"]
    if case["kind"] == "tables":
        # at most 1023 fragments make a request
        return _ragged(seed, n, case["size"], 8), _ragged(seed + 1, n, case["resp"], 8)
    if case["kind"] == "echo":
        s = _ragged(seed, n, case["size"] or 65536, 64)
        return s, s
    return np.full(n, case["size"], np.int64), np.full(n, case["resp"], np.int64)


def _copies(case):
    """A call is laid out as this many like batches side by side, each with slots of its own."""
    n = case["n_req"]
    if case["workload"]:
        base = min(n, WORKLOADS[case["workload"]][0])
    elif case["kind"] in ("tables", "request"):
        base = n
    else:
        base = min(n, 4096, max(1, 24000000 // max(case["size"], case["resp"])))
    return base, -(-n // base)


def _workload(case, seed):
    base, copies = _copies(case)
    if case["workload"] and case["kind"] != "echo":
        return synth.make_workload(case["workload"], base, seed=seed, profile=case["profile"]), copies
    req, resp = _sizes(dict(case, n_req=base), seed)
    # the mixed workload's ring is twice as large as what is in it, and starts anywhere
    slots = 65536 if case["workload"] else None
    return synth.make_custom(req, resp, n_slots=slots, head=(seed * 7919) % slots if slots else 0, mtu=case["mtu"], slot_size=case["slot"], seed=seed, profile=case["profile"],
                             order=case["order"] or "shuffle_all", flags=case["flags"], in_place=case["kind"] == "echo",
                             in_tensor_sizes=[case["split"], case["size"] - case["split"]] if case["split"] else ()), copies


_stream = None


def _context(n_req, n_frames):
    """One stream for everything the server's shunter thread queues."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return SgContext(torch.cuda.current_device(), max_reqs=max(n_req, 64), max_frames=max(n_frames, 1024),
                     stream=_stream.cuda_stream)


def prepare(case, seed):
    w, copies = _workload(case, seed)
    slack = 4099 if case["kind"] == "tables" else 0  # a ring that batches do not fill evenly: requests wrap
    dw = DeviceWorkload(w, copies=copies, unique_tokens=True, arena_slack=slack)
    ctx = _context(dw.n_req, max(dw.n_frags, dw.n_frames))
    state = {"kind": case["kind"], "dw": dw, "ctx": ctx, "w": w}
    if case["kind"] == "tables":
        _prepare_tables(state, w, dw, ctx, seed)
    elif case["kind"] == "request":
        _prepare_request(state, w, dw)
    elif case["kind"] == "receive":
        _prepare_receive(state, case, w, dw, ctx, copies)
    torch.cuda.synchronize()
    return state


def _prepare_tables(state, w, dw, ctx, seed):
    n, hl = w.n_req, synth.hdr_len(w.profile)
    ring = dw.ring.data_ptr()
    tables = torch.empty((n, 2, capi.MAX_BI_SIZE), dtype=torch.int32, pin_memory=True)
    tab = tables.numpy()
    tab[:] = -1
    half = ((w.frag_slot.astype(np.int64) * w.slot_size + hl) >> 1).astype(np.int32)
    for r in range(n):
        a, b = int(w.req_first[r]), int(w.req_first[r + 1])
        tab[r, 0, :b - a] = half[a:b]
        tab[r, 1, :b - a] = w.frag_len[a:b]
    # per request: token, response size, header template; then the response frame tables
    rng = np.random.default_rng(seed + 2)
    templates = synth.build_headers(rng, 1, np.arange(n), np.zeros(n, np.uint32), np.ones(n, np.uint32),
                                    np.zeros(n, np.uint32), w.req_ids)
    parts = [w.req_ids.astype(np.uint64).view(np.uint32), w.resp_sizes.astype(np.uint64).view(np.uint32),
             np.ascontiguousarray(templates).view(np.uint32).reshape(-1), w.resp_first, w.tx_slot]
    words = np.concatenate([np.ascontiguousarray(p, dtype=np.uint32) for p in parts])
    at = np.concatenate([[0], np.cumsum([len(p) for p in parts])])
    pin = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int32).copy()).pin_memory()
    blob, idx, first = pin(words), pin(np.arange(n, dtype=np.uint32)), pin(w.req_first.astype(np.uint32))
    i32 = lambda k: torch.zeros(k, dtype=torch.int32, device=dw.dev)
    fs, fl, rf, dst = i32(w.n_frags), i32(w.n_frags), i32(n + 1), i32(len(words))
    p = capi.PackArgs()
    p.tables, p.n_tables, p.n_req, p.table_idx = tables.data_ptr(), n, n, idx.data_ptr()
    p.req_first, p.n_frags, p.pkt_base, p.ring = first.data_ptr(), w.n_frags, ring, dw.rx.desc()
    p.frag_slot, p.frag_len, p.req_first_out = fs.data_ptr(), fl.data_ptr(), rf.data_ptr()
    p.blob_src, p.blob_dst, p.blob_words = blob.data_ptr(), dst.data_ptr(), len(words)
    token, size, tmpl, rfirst, tslot = (dst[int(at[i]):int(at[i + 1])] for i in range(5))
    g = ctx.gather_args(dw.rx, fs, fl, rf, n, w.n_frags, dw.req_app, dw.req_offsets, ASYNC, mtu=w.mtu)
    s = ctx.scatter_args(dw.rx, dw.tx, tslot, None, rfirst, size, 0, n, w.n_resp_frames, w.mtu, dw.resp_app,
                         dw.resp_offsets, w.flags | ASYNC, hdr_templates=tmpl, req_token=token)
    state.update(pack=p, g=g, s=s, keep=(tables, blob, idx, first, fs, fl, rf, dst),
                 out=[dw.req_arena, dw.tx_ring, dw.req_offsets, dw.resp_offsets, fs, fl, rf])


def _prepare_request(state, w, dw):
    hl = synth.hdr_len(w.profile)
    rx, tx = dw.ring.data_ptr(), dw.tx_ring.data_ptr()
    gather, scatter, hdrs = capi.SkBuf(), capi.SkBuf(), capi.HBufs()
    at = dw.req_arena.data_ptr()
    for i in range(w.n_frags):
        gather.i_buf[i] = rx + int(w.frag_slot[i]) * w.slot_size + hl
        gather.o_buf[i] = at
        gather.len[i] = int(w.frag_len[i])
        at += int(w.frag_len[i])
    gather.num_items = w.n_frags
    at, left = dw.resp_arena.data_ptr(), int(w.resp_sizes[0])
    for i in range(w.n_resp_frames):
        slot = tx + int(w.tx_slot[i]) * w.slot_size
        n = min(left, w.mtu)
        scatter.i_buf[i], scatter.o_buf[i], scatter.len[i] = at, slot + hl, n
        hdrs.burst_items[i] = slot
        at, left = at + n, left - n
    scatter.num_items = hdrs.num_items = w.n_resp_frames
    first = int(w.frag_slot[0]) * w.slot_size
    template = (C.c_uint8 * 64).from_buffer_copy(w.ring[first:first + 64].tobytes())
    state.update(gather=gather, scatter=scatter, hdrs=hdrs, template=template, token=int(w.req_ids[0]),
                 flags=w.flags & (synth.F_IPV4_CSUM | synth.F_UDP_CSUM_PSEUDO), out=[dw.req_arena, dw.tx_ring])


def _prepare_receive(state, case, w, dw, ctx, copies):
    n, size, rsize = dw.n_req, int(w.req_sizes[0]), int(w.resp_sizes[0])
    per, per_resp = synth.num_frames(size, w.mtu), synth.num_frames(rsize, w.mtu)
    arrivals = dw.n_frags
    burst = min(case["burst"] or arrivals, arrivals)
    # requests a burst can complete: those whose last fragment is in it
    pos = np.empty(w.n_slots, np.int64)
    pos[w.arrivals] = np.arange(w.n_frags)
    last = np.array([pos[w.frag_slot[int(w.req_first[r]):int(w.req_first[r + 1])]].max() for r in range(w.n_req)])
    done = np.concatenate([last + i * w.n_frags for i in range(copies)]) // burst
    n_bursts = -(-arrivals // burst)
    completes = np.bincount(done, minlength=n_bursts)
    bound = int(completes.max())
    i32 = lambda k: torch.zeros(k, dtype=torch.int32, device=dw.dev)
    fs, fl, rf, hdr, counts = i32(_max_frames(dw)), i32(_max_frames(dw)), i32(max(n, 64) + 1), i32(max(n, 64)), i32(4)
    len_nic = None
    if w.profile:
        one = np.zeros(w.n_slots, np.uint32)
        one[w.frag_slot] = w.frag_len
        len_nic = to_dev(np.tile(one, copies), dw.dev)
    req = torch.zeros(n * size, dtype=torch.uint8, device=dw.dev)
    resp = dw.out_tensors[0] if w.out_tensor_sizes else dw.resp_arena
    # every burst's responses go to TX slots of their own
    tx_slot = to_dev(np.concatenate([np.arange(n * per_resp, dtype=np.uint32), np.zeros(bound * per_resp, np.uint32)]), dw.dev)
    tx_ring = torch.zeros(n * per_resp * w.slot_size, dtype=torch.uint8, device=dw.dev)
    tx = RingRef(tx_ring, n * per_resp, w.slot_size, w.profile)
    resp_first = to_dev((np.arange(bound + 1) * per_resp).astype(np.uint32), dw.dev)
    req_app, resp_app = AppRef(arena=req, cap=n * size), AppRef(arena=resp, cap=n * rsize)
    g = ctx.gather_args(dw.rx, fs, fl if w.profile else None, rf, bound, bound * per, req_app, None,
                        ASYNC | capi.F_RULE_FRAGS, fixed_req_size=size, mtu=w.mtu, counts=counts)
    calls, served = [], 0
    for b in range(n_bursts):
        lo = b * burst
        k = min(burst, arrivals - lo)
        ra = ctx.reassemble_args(dw.rx, dw.arrivals[lo:lo + k], k, fs, fl, rf, None, len_nic, size if w.profile else 0,
                                 req_hdr_slot=hdr, counts_out=counts, flags=ASYNC)
        s = ctx.scatter_args(dw.rx, tx, tx_slot[served * per_resp:], None, resp_first, None, rsize, bound,
                             bound * per_resp, w.mtu, resp_app, None, w.flags | ASYNC, hdr_src_req=hdr, counts=counts)
        calls.append((ra, s))
        served += int(completes[b])
    ctx.reassemble_reset()
    state.update(calls=calls, g=g, keep=(fs, fl, rf, hdr, len_nic, tx_slot, resp_first),
                 out=[req, tx_ring, counts])


def _max_frames(dw):
    return max(dw.n_frags, dw.n_frames, 1024)


# ---- one pass ---------------------------------------------------------------

def run(state):
    kind, dw, ctx = state["kind"], state["dw"], state["ctx"]
    if kind == "step":
        dw.shunt(ctx, ASYNC)
        req = list(dw.in_tensors) if dw.w.in_tensor_sizes else [dw.req_arena, dw.req_offsets]
        return req + [dw.tx_ring]
    if kind == "echo":
        dw.gather(ctx, ASYNC)
        dw.scatter(ctx, ASYNC, reuse=True)
        return [dw.req_arena, dw.ring, dw.req_offsets, dw.resp_offsets]
    if kind == "tables":
        ctx._check(ctx.lib.sg_hip_pack_tables(ctx.h, C.byref(state["pack"])))
        ctx.gather_batch_raw(state["g"])
        ctx.scatter_batch_raw(state["s"])
        return state["out"]
    if kind == "request":
        w, lib, h = state["w"], ctx.lib, ctx.h
        ctx._check(lib.sg_hip_gather(h, C.byref(state["gather"])))
        ctx._check(lib.sg_hip_set_hdrs(h, C.byref(state["hdrs"]), state["template"], state["token"], w.profile,
                                       int(w.resp_sizes[0]), w.mtu, state["flags"]))
        ctx._check(lib.sg_hip_scatter(h, C.byref(state["scatter"])))
        return state["out"]
    g = state["g"]
    for ra, s in state["calls"]:
        ctx.reassemble_raw(ra)
        ctx.shunt_batch_raw(g, s)
    return state["out"]


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    base, copies = _copies(case)
    req, resp = _sizes(dict(case, n_req=base), 1)
    frames = lambda s: int(((s + case["mtu"] - 1) // case["mtu"]).sum()) * copies
    hl = synth.hdr_len(case["profile"])
    f_in, f_out = frames(req), frames(resp)
    # payloads in and out, the RPC header of every fragment, a header in and out per response frame
    b = 2 * int(req.sum() + resp.sum()) * copies + 16 * f_in + 2 * hl * f_out
    b += 4 * f_in + 4 * f_out  # the slot tables
    if case["kind"] == "tables":
        b += 8 * f_in + 4 * f_out + 84 * base  # tables across the bus; token, size, template per request
    if case["kind"] == "receive":
        b += 24 * f_in  # an arrival's header words, slot and filed entry
    return {"bytes": b, "flops": 0}


def tolerance(case):
    return "exact"
