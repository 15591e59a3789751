"""Timed workloads of the silent-OT engine: what a program that uses
``cuot_amd`` has it do, through the package's public entry points.

    listed()            the workloads, each a dict of plain values
    draw(rng)           one more of the same kinds and ranges
    prepare(case, seed) contexts, plans, workspaces and inputs (on the GPU)
    run(state)          one pass; returns every output whole
    work(case)          bytes one pass has to read and write at least
    exact(case, seed)   nothing: every output is whole numbers (blocks, bits)

Kinds:
    sot      one plain SOT instance, both roles, from a 128-bit seed
             (2n GGM leaves, scaler-2 quasi-cyclic code, n COTs)
    ferret   one Ferret instance, both roles (MPCOT, then the 10-local LPN)
    extend   one extend of an iterating Ferret session, semi-honest or malicious
    ot       chosen-message OTs from a session's COTs (extend, online step, hash)
    rot      random OTs the same way
    batch    a list of uneven instances as one launch sequence
    qc       the quasi-cyclic encode alone, on a code prepared once
    mpcot    emp-ot's dev_layer calls, host arrays in and out
"""
import math

import numpy as np
import torch

import cuot_amd
from cuot_amd import dev_layer, workloads
from cuot_amd.ferret import FerretCOT

BLOCK = 16
SIZES = (1 << 14, 1 << 24)  # COTs of an instance: the serving mix's range
_ctx = None


def _context():
    """A program has one context per GPU."""
    global _ctx
    if _ctx is None:
        _ctx = cuot_amd.Context(0)
    return _ctx


def listed():
    return [
        # the headline workload: n = 2^24, t = 1024 trees of depth 15
        {"name": "sot 2^24", "kind": "sot", "n": 1 << 24},
        # the reference's own configuration size (t = 256, depth 13)
        {"name": "sot 2^20", "kind": "sot", "n": 1 << 20},
        # a request of the batched / served mixes: any n, rounded up inside
        {"name": "sot 190731", "kind": "sot", "n": 190731},
        # the smallest request, where launches and latency count
        {"name": "sot 2^14", "kind": "sot", "n": 1 << 14},
        # emp-ot's Ferret parameters (k = 452160, t = 1270 trees of 8192)
        {"name": "ferret 10168320", "kind": "ferret", "n": 10168320, "k": 452160, "t": 1270, "h": 13, "ntasks": 1},
        # an ordinary request, with the rows split as emp-ot's threads split them
        {"name": "ferret 300007", "kind": "ferret", "n": 300007, "k": 13637, "t": 37, "h": 13, "ntasks": 4},
        # the smallest request
        {"name": "ferret 20000", "kind": "ferret", "n": 20000, "k": 910, "t": 3, "h": 13, "ntasks": 1},
        # a long-lived client in malicious mode, one extend a pass
        {"name": "extend malicious 10168320", "kind": "extend", "n": 10168320, "k": 452160, "t": 1270, "h": 13,
         "malicious": True},
        # a million oblivious transfers of chosen messages
        {"name": "ot 1048576", "kind": "ot", "n": 1 << 20, "k": 47663, "t": 128, "h": 13},
        # many uneven requests together, replayed as a graph
        {"name": "batch 16", "kind": "batch", "count": 16, "mix": 5, "lo": 16, "hi": 22},
        # one party's encode on a prepared code of ragged length
        {"name": "qc 2500001", "kind": "qc", "n": 2500001},
        # emp-ot calling the drop-in GPU layer (blocking, host sums)
        {"name": "mpcot 1270x2^13", "kind": "mpcot", "t": 1270, "h": 13},
    ]


def _log_uniform(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["sot", "sot", "sot", "ferret", "ferret", "extend", "ot", "rot", "batch", "qc", "qc", "mpcot"])
    if kind == "sot" or kind == "qc":
        n = _log_uniform(rng, SIZES[0], SIZES[1] // 2)
        if rng.random() < 0.3:
            n = 1 << (n.bit_length() - 1)
        elif rng.random() < 0.5:
            n |= 1
        if kind == "qc" and n == 2500001:
            n += 1
        return {"kind": kind, "n": n}
    if kind == "ferret":
        n = _log_uniform(rng, SIZES[0], 10168320)
        t, h, k = workloads.ferret_shape(n)
        return {"kind": kind, "n": n, "k": k, "t": t, "h": h, "ntasks": rng.choice([1, 1, 4, 7])}
    if kind == "extend":
        n = _log_uniform(rng, 1 << 16, 10168320)
        t, h, k = workloads.ferret_shape(n)
        return {"kind": kind, "n": n, "k": k, "t": t, "h": h, "malicious": rng.random() < 0.5}
    if kind == "ot" or kind == "rot":
        n = _log_uniform(rng, 1 << 16, 1 << 22)
        t, h, k = workloads.ferret_shape(n)
        return {"kind": kind, "n": n, "k": k, "t": t, "h": h}
    if kind == "batch":
        return {"kind": kind, "count": rng.choice([4, 8, 16]), "mix": rng.randrange(1, 1 << 20), "lo": 14, "hi": 21}
    return {"kind": kind, "t": rng.randrange(1, 1271), "h": rng.choice([8, 10, 11, 12, 13])}


def _block(gen):
    return gen.integers(0, 1 << 63, size=2, dtype=np.int64).view(np.uint64) * np.uint64(2) + np.uint64(1)


def _rand(shape, seed, high=None, dtype=torch.int64):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if high is None:
        return torch.randint(-(1 << 63), (1 << 63) - 1, shape, dtype=dtype, device="cuda", generator=g)
    return torch.randint(0, high, shape, dtype=dtype, device="cuda", generator=g)


def _blocks(n):
    return torch.empty((n, 2), dtype=torch.int64, device="cuda")


def _mix(case):
    return workloads.batch_mix(case["count"], master=(case["mix"], 0), lo_log=case["lo"], hi_log=case["hi"])


def prepare(case, seed):
    ctx = _context()
    gen = np.random.default_rng(seed)
    kind = case["kind"]
    st = {"kind": kind, "ctx": ctx}
    if kind == "sot":
        n = case["n"]
        t, h = workloads.sot_shape(n)
        cfg = cuot_amd.SotConfig(n=n, t=t, h=h, reserved=0, k0=cuot_amd.to_block(np.array(workloads.SOT_K0)),
                                 k1=cuot_amd.to_block(np.array(workloads.SOT_K1)), seed=cuot_amd.to_block(_block(gen)))
        st.update(cfg=cfg, ws=torch.empty(ctx.sot_workspace_bytes(cfg), dtype=torch.uint8, device="cuda"),
                  v=_blocks(n), w=_blocks(n), delta=_blocks(1),
                  bits=torch.empty((n + 31) // 32, dtype=torch.int32, device="cuda"))
    elif kind == "ferret":
        cfg = cuot_amd.FerretConfig(n=case["n"], k=case["k"], t=case["t"], h=case["h"], ntasks=case["ntasks"],
                                    seed=cuot_amd.to_block(_block(gen)))
        st.update(cfg=cfg, ws=torch.empty(ctx.ferret_workspace_bytes(cfg), dtype=torch.uint8, device="cuda"),
                  s=_blocks(case["n"]), r=_blocks(case["n"]), delta=_blocks(1))
    elif kind in ("extend", "ot", "rot"):
        fc = FerretCOT(ctx, n=case["n"], k=case["k"], t=case["t"], h=case["h"], seed=_block(gen))
        st["fc"] = fc
        if kind == "extend":
            st["malicious"] = case["malicious"]
            fc.set_malicious(case["malicious"])
        else:
            num = fc.ot_limit  # each pass uses up one extend
            st.update(choice=_rand((num,), seed + 1, 2, torch.uint8), tweak=_block(gen))
            if kind == "ot":
                st.update(m0=_rand((num, 2), seed + 2), m1=_rand((num, 2), seed + 3))
    elif kind == "batch":
        ins = [cuot_amd.make_instance_struct(i.kind, i.n, i.t, i.h, i.k, _block(gen)) for i in _mix(case)]
        st["batch"] = cuot_amd.Batch(ctx, ins)
        st["stream"] = torch.cuda.Stream()  # graph replay takes a stream of the caller's
    elif kind == "qc":
        n = case["n"]
        a = _rand(((n + 7) // 8 + 16,), seed + 1, 256, torch.uint8)
        ahat = torch.empty(ctx.qc_ahat_len(n), dtype=torch.int32, device="cuda")
        scratch = torch.empty(ctx.qc_scratch_bytes(n), dtype=torch.uint8, device="cuda")
        ctx.qc_prepare(n, a, ahat, scratch)
        st.update(n=n, a=a, ahat=ahat, scratch=scratch, x=_rand((2 * n, 2), seed + 2), y=_blocks(n))
    else:
        t, h = case["t"], case["h"]
        alpha = gen.integers(0, 1 << h, size=t)
        bit = (alpha[:, None] >> np.arange(h - 1, -1, -1)[None, :]) & 1
        st.update(t=t, h=h, roots=_rand((t, 2), seed + 1), delta=_block(gen),
                  choice=np.ascontiguousarray(1 - bit, dtype=np.uint8).reshape(-1),
                  exp_s=_blocks(t << h), exp_r=_blocks(t << h), buf=_blocks(t << h), sep=_blocks(t << h),
                  lsum=np.zeros((t * h, 2), np.uint64), rsum=np.zeros((t * h, 2), np.uint64),
                  ssum=np.zeros((t, 2), np.uint64))
    return st


def run(st):
    ctx, kind = st["ctx"], st["kind"]
    if kind == "sot":
        ctx.sot_run(st["cfg"], st["ws"], st["v"], st["w"], st["bits"], st["delta"])
        return st["v"], st["w"], st["bits"], st["delta"]
    if kind == "ferret":
        ctx.ferret_run(st["cfg"], st["ws"], st["s"], st["r"], st["delta"])
        return st["s"], st["r"], st["delta"]
    if kind == "extend":
        fc = st["fc"]
        fc.extend_f2k()
        if not st["malicious"]:
            return fc.out_s, fc.out_r
        ok, xp, da, db = fc.check_result()  # a malicious-mode client looks at the verdict
        return fc.out_s, fc.out_r, ok, np.frombuffer(xp + da + db, dtype=np.uint8)
    if kind == "ot":
        return st["fc"].send_recv_ot(st["m0"], st["m1"], st["choice"], st["tweak"])
    if kind == "rot":
        return st["fc"].send_recv_rot(st["choice"], st["tweak"])
    if kind == "batch":
        b = st["batch"]
        b.run(graph=True, overlap=True, stream=st["stream"])
        return b.out0, b.out1, b.bits, b.delta
    if kind == "qc":
        ctx.qc_encode(st["n"], st["ahat"], st["x"], st["y"], st["scratch"])
        return st["y"]
    t, h = st["t"], st["h"]
    st["exp_s"][:t] = st["roots"]
    torch.cuda.current_stream().synchronize()  # the drop-in calls run on the context's own stream
    dev_layer.cuda_mpcot_sender(ctx, [st["exp_s"]], [st["buf"]], [st["sep"]], st["lsum"], st["rsum"], st["ssum"], [t],
                                h, st["delta"])
    csum = np.where(st["choice"][:, None] == 1, st["rsum"], st["lsum"])  # what the level OTs deliver
    dev_layer.cuda_mpcot_recver(ctx, [st["exp_r"]], [st["buf"]], [st["sep"]], csum, st["ssum"], [t], h, st["choice"])
    return st["exp_s"], st["exp_r"], st["lsum"], st["rsum"], st["ssum"]


def work(case):
    """Each input read once and each output written once (seeds count as nothing)."""
    kind = case["kind"]
    if kind == "sot":
        return {"bytes": case["n"] * (2 * BLOCK + 0.125), "flops": 0}
    if kind == "ferret":
        return {"bytes": case["n"] * 2 * BLOCK, "flops": 0}
    if kind == "extend":
        m = case["k"] + case["h"] * case["t"] + 128  # bootstrap COTs carried over
        return {"bytes": (case["n"] + 2 * m) * 2 * BLOCK, "flops": 0}
    if kind in ("ot", "rot"):
        m = case["k"] + case["h"] * case["t"] + 128
        num = case["n"] - m
        io = (2 + 3) * BLOCK + 1 if kind == "ot" else 3 * BLOCK + 1
        return {"bytes": (case["n"] + 2 * m) * 2 * BLOCK + num * io, "flops": 0}
    if kind == "batch":
        return {"bytes": sum(i.n * (2 * BLOCK + (0.125 if i.kind == workloads.SOT else 0)) for i in _mix(case)),
                "flops": 0}
    if kind == "qc":
        return {"bytes": case["n"] * (3 * BLOCK + 0.125), "flops": 0}
    return {"bytes": (case["t"] << case["h"]) * 2 * BLOCK, "flops": 0}


def exact(case, seed):
    """Blocks, bits and digests are whole numbers: there is no rounding to measure."""
    return None
