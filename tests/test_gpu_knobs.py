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
    v, w = (torch.empty((n, 2), dtype=torch.int64, device="cuda") for _ in range(2))
    b, d = torch.empty((n + 31) // 32, dtype=torch.int32, device="cuda"), torch.empty((1, 2), dtype=torch.int64, device="cuda")
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
