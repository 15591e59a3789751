"""Knobs never change outputs: stages run under another setting than the one
that left the workspace."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K0, K1 = (3242342, 0), (8993849, 0)
SEED = (0x0706050403020100, 0x0F0E0D0C0B0A0908)


def _shape(n):
    h = 9 if n > 512 else 3
    return -(-2 * n >> h), h


# the matrix cores' encodes read a's bits, the transforms' A^: a whole run leaves both
@pytest.mark.parametrize("n", [17, 4000, 9001, 16384, 36000])
def test_encode_stage_after_whole_run(ctx, n):
    import torch

    import cuot_amd
    from cuot_amd import tune

    t, h = _shape(n)
    print(f"encode stage n={n} t={t} h={h}", flush=True)
    B = cuot_amd.to_block
    cfg = cuot_amd.SotConfig(n=n, t=t, h=h, reserved=0, k0=B(K0), k1=B(K1), seed=B(SEED))
    ws = torch.full((ctx.sot_workspace_bytes(cfg),), 0xA5, dtype=torch.uint8, device="cuda")
    v, w, d = (torch.empty((m, 2), dtype=torch.int64, device="cuda") for m in (n, n, 1))
    b = torch.empty((n + 31) // 32, dtype=torch.int32, device="cuda")
    ctx.sot_run(cfg, ws, v, w, b, d)
    want = v.clone(), w.clone()
    ins = cuot_amd.make_instance_struct(cuot_amd.MODE_SOT, n, t, h, 0, SEED)
    bt = cuot_amd.Batch(ctx, [ins, ins])
    bt.ws.fill_(0xA5)
    torch.cuda.synchronize()
    _rebind(bt)
    bt.run()
    assert torch.equal(bt.out0[1], want[0]) and torch.equal(bt.out1[0], want[1])
    try:
        tune.set_knobs(qc_mfma_max=-1)
        ctx.sot_run_stages(cfg, ws, v.zero_(), w.zero_(), b, d, 16 | 32)
        for o in (*bt.out0, *bt.out1):
            o.zero_()
        bt.run(stages=16)
        torch.cuda.synchronize()
    finally:
        tune.set_knobs()
    assert torch.equal(v, want[0]) and torch.equal(w, want[1])
    for i in range(2):
        assert torch.equal(bt.out0[i], want[0]) and torch.equal(bt.out1[i], want[1])


def _rebind(bt):
    """upload the launch tables into the overwritten workspace"""
    import ctypes as C

    from cuot_amd._lib import check

    n = len(bt.instances)
    o0 = (C.c_void_p * n)(*[t.data_ptr() for t in bt.out0])
    o1 = (C.c_void_p * n)(*[t.data_ptr() for t in bt.out1])
    bb = (C.c_void_p * n)(*[(t.data_ptr() if t is not None else None) for t in bt.bits])
    check(bt.lib.cuot_batch_bind(bt.handle, bt.ws.data_ptr(), bt.ws_bytes, o0, o1, bb, bt.delta.data_ptr()),
          "cuot_batch_bind")


# every split of whole trees that ggm_dfs can ask for: tops of 2^8, 2^9 and 2^10
# nodes, with a truncated last tree, in single runs and in a batch, whose forms are
# chosen when it is made
@pytest.mark.parametrize("h", range(9, 17))
def test_ggm_splits_match_oracle(ctx, h):
    import torch

    import cuot_amd
    from cuot_amd import tune
    from oracle import pyoracle as po
    from tests.helpers import to_np

    B = cuot_amd.to_block
    t = 3 if h < 14 else 2
    nf = (t << h) - 77  # Ferret's outputs
    ns = ((t << h) - 40) // 2  # SOT: 2 ns leaves
    k0, k1, seed = (np.array(x, dtype=np.uint64) for x in (K0, K1, SEED))
    fs, fr, _ = po.ferret_run(nf, 60, t, h, seed, nthreads=4)
    sv, sw, sb, _ = po.sot_run(ns, t, h, k0, k1, seed, nthreads=4)
    fcfg = cuot_amd.FerretConfig(n=nf, k=60, t=t, h=h, ntasks=1, seed=B(SEED))
    scfg = cuot_amd.SotConfig(n=ns, t=t, h=h, reserved=0, k0=B(K0), k1=B(K1), seed=B(SEED))
    fws = torch.full((ctx.ferret_workspace_bytes(fcfg),), 0xA5, dtype=torch.uint8, device="cuda")
    sws = torch.full((ctx.sot_workspace_bytes(scfg),), 0xA5, dtype=torch.uint8, device="cuda")
    out = [torch.empty((n, 2), dtype=torch.int64, device="cuda") for n in (nf, nf, ns, ns, 1)]
    bits = torch.empty((ns + 31) // 32, dtype=torch.int32, device="cuda")
    ins = [cuot_amd.make_instance_struct(cuot_amd.MODE_FERRET, nf, t, h, 60, SEED),
           cuot_amd.make_instance_struct(cuot_amd.MODE_SOT, ns, t, h, 0, SEED)]
    splits = [L for L in range(1, 7) if h - 10 <= L <= h - 8]
    try:
        for L in splits:
            print(f"ggm split h={h} L={L}", flush=True)
            tune.set_knobs(ggm_dfs=L)
            for o in out:
                o.zero_()
            ctx.ferret_run(fcfg, fws, out[0], out[1])
            ctx.sot_run(scfg, sws, out[2], out[3], bits, out[4])
            bt = cuot_amd.Batch(ctx, ins)
            bt.run()
            torch.cuda.synchronize()
            got = out[:4] + [bt.out0[0], bt.out1[0], bt.out0[1], bt.out1[1]]
            for g, want in zip(got, (fs, fr, sv, sw) * 2):
                assert np.array_equal(to_np(g), want), (h, L)
    finally:
        tune.set_knobs()
    assert splits
