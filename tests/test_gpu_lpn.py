"""GPU parity: fused Ferret LPN against the oracle, bit-exact."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import dev_blocks, rand_blocks, rng, to_dev, to_np

pytestmark = pytest.mark.gpu


def _p(n, k, seed, ntasks=1):
    import cuot_amd

    return cuot_amd.LpnParams(n=n, k=k, d=10, ntasks=ntasks, seed=cuot_amd.to_block(seed))


@pytest.mark.parametrize("n,k,ntasks", [(1, 5, 1), (7, 11, 1), (1000, 452, 1), (12345, 999, 1), (4099, 3000, 3),
                                        (100000, 4523, 1), (100003, 4523, 7)])
def test_lpn_single_and_dual(ctx, n, k, ntasks):
    print(f"lpn n={n} k={k} ntasks={ntasks}", flush=True)
    r = rng(n + k)
    seed = rand_blocks(r, 1)[0]
    noise, kk = rand_blocks(r, n), rand_blocks(r, k)
    ref = po.ferret_lpn(noise, kk, seed, ntasks=ntasks, nthreads=4)
    out = dev_blocks(n)
    ctx.lpn(_p(n, k, seed, ntasks), to_dev(noise), to_dev(kk), out)
    assert np.array_equal(to_np(out)[:n], ref)
    # in place, dual role
    noise2, kk2 = rand_blocks(r, n), rand_blocks(r, k)
    ref2 = po.ferret_lpn(noise2, kk2, seed, ntasks=ntasks, nthreads=4)
    a, b = to_dev(noise), to_dev(noise2)
    ctx.lpn_dual(_p(n, k, seed, ntasks), a, to_dev(kk), a, b, to_dev(kk2), b)
    assert np.array_equal(to_np(a)[:n], ref)
    assert np.array_equal(to_np(b)[:n], ref2)


# tables above 11 MB are gathered in two slices (rows of the other slice read as
# zero): one role at the limit and past it, both roles interleaved past it
@pytest.mark.parametrize("n,k", [(4099, 720896), (4099, 720897), (3, 720897)])
def test_lpn_table_slices_one_role(ctx, n, k):
    print(f"lpn slices n={n} k={k}", flush=True)
    r = rng(n + k)
    seed = rand_blocks(r, 1)[0]
    noise, kk = rand_blocks(r, n), rand_blocks(r, k)
    ref = po.ferret_lpn(noise, kk, seed, ntasks=1, nthreads=4)
    a = to_dev(noise)
    ctx.lpn(_p(n, k, seed), a, to_dev(kk), a)
    assert np.array_equal(to_np(a)[:n], ref)


def test_lpn_table_slices_both_roles(ctx):
    import torch

    import cuot_amd

    n, k, t, h = 380003, 370003, 47, 13
    seed = np.array([77, 78], dtype=np.uint64)
    cfg = cuot_amd.FerretConfig(n=n, k=k, t=t, h=h, ntasks=3, seed=cuot_amd.to_block(seed))
    ws = torch.empty(ctx.ferret_workspace_bytes(cfg), dtype=torch.uint8, device="cuda")
    s, w = dev_blocks(n), dev_blocks(n)
    ctx.ferret_run(cfg, ws, s, w)
    os_, or_, _ = po.ferret_run(n, k, t, h, seed, ntasks=3, nthreads=4)
    assert np.array_equal(to_np(s), os_)
    assert np.array_equal(to_np(w), or_)


# two slices need rows enough as well as a table above 11 MB: at the least rows
# that take them, and one short of it
@pytest.mark.parametrize("n", [2 * 720897 - 1, 2 * 720897])
def test_lpn_table_slices_many_rows(ctx, n):
    k = 720897
    print(f"lpn slices n={n} k={k}", flush=True)
    r = rng(n + k)
    seed = rand_blocks(r, 1)[0]
    noise, kk = rand_blocks(r, n), rand_blocks(r, k)
    ref = po.ferret_lpn(noise, kk, seed, ntasks=3, nthreads=8)
    a = to_dev(noise)
    ctx.lpn(_p(n, k, seed, 3), a, to_dev(kk), a)
    assert np.array_equal(to_np(a)[:n], ref)


@pytest.mark.parametrize("n", [4 * 360449 - 1, 4 * 360449])
def test_lpn_table_slices_many_rows_both_roles(ctx, n):
    import torch

    import cuot_amd

    k, h = 360449, 13
    t = -(-n >> h)
    print(f"lpn slices both roles n={n} k={k}", flush=True)
    seed = np.array([79, 80], dtype=np.uint64)
    cfg = cuot_amd.FerretConfig(n=n, k=k, t=t, h=h, ntasks=1, seed=cuot_amd.to_block(seed))
    ws = torch.empty(ctx.ferret_workspace_bytes(cfg), dtype=torch.uint8, device="cuda")
    s, w = dev_blocks(n), dev_blocks(n)
    ctx.ferret_run(cfg, ws, s, w)
    os_, or_, _ = po.ferret_run(n, k, t, h, seed, nthreads=8)
    assert np.array_equal(to_np(s), os_)
    assert np.array_equal(to_np(w), or_)
