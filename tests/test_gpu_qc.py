"""GPU parity: exact QC encoder (additive FFT and, for small codes, the int8
matrix-core product), sparse encoder and the bit transpose against the CPU
oracle, bit-exact."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import dev_blocks, rand_blocks, rng, to_dev, to_np

pytestmark = pytest.mark.gpu


def rand_bits(r, n):
    a = r.integers(0, 256, size=(n + 7) // 8, dtype=np.uint8)
    if n % 8:
        a[-1] &= (1 << (n % 8)) - 1
    return a


def dev_bits(a, n):
    import torch

    words = (n + 31) // 32 + 2
    buf = np.zeros(words * 4, dtype=np.uint8)
    buf[: a.shape[0]] = a
    return torch.from_numpy(buf).cuda()


def qc_gpu(ctx, x, a, n):
    import torch

    ahat = torch.zeros(ctx.qc_ahat_len(n), dtype=torch.int32, device="cuda")
    scratch = torch.zeros(ctx.qc_scratch_bytes(n), dtype=torch.uint8, device="cuda")
    ctx.qc_prepare(n, dev_bits(a, n), ahat, scratch)
    y = dev_blocks(n)
    ctx.qc_encode(n, ahat, to_dev(x), y, scratch)
    return to_np(y)[:n]


@pytest.mark.parametrize("n", [1, 5, 16, 17, 100, 1000, 4096, 4099])
def test_qc_small_vs_brute(ctx, n):
    print(f"qc brute n={n}", flush=True)
    r = rng(n)
    a, x = rand_bits(r, n), rand_blocks(r, 2 * n)
    assert np.array_equal(qc_gpu(ctx, x, a, n), po.qc_encode_brute(x, a, n))


# 2^20 and 2^22 + 7 also cover the row conversion with several strings per
# workgroup at 2^17 .. 2^19-bit strings (folded and general output)
@pytest.mark.parametrize("n", [1 << 14, 65537, 1 << 18, 1 << 20, (1 << 22) + 7])
def test_qc_vs_karatsuba(ctx, n):
    print(f"qc karatsuba n={n}", flush=True)
    r = rng(n + 1)
    a, x = rand_bits(r, n), rand_blocks(r, 2 * n)
    assert np.array_equal(qc_gpu(ctx, x, a, n), po.qc_encode_fast(x, a, n, nthreads=8))


def test_qc_special_cases(ctx):
    n = 1 << 12
    r = rng(3)
    x = rand_blocks(r, 2 * n)
    one = np.zeros(n // 8, dtype=np.uint8)
    one[0] = 1
    assert np.array_equal(qc_gpu(ctx, x, one, n), x[:n] ^ x[n:])
    s = 1234
    xs = np.zeros(n // 8, dtype=np.uint8)
    xs[s >> 3] |= 1 << (s & 7)
    assert np.array_equal(qc_gpu(ctx, x, xs, n), x[:n] ^ x[n + (np.arange(n) - s) % n])


@pytest.fixture
def knob_mfma():
    """Sets the matrix-core crossover for one test and restores the rule after."""
    from cuot_amd import tune

    def set_(v):
        tune.set_knobs(qc_mfma_max=v)

    yield set_
    tune.set_knobs()


# small codes on the int8 matrix cores: one slice (n <= 256, direct write) and
# several (atomic XOR), n around the 32-row and 16-k tile edges
@pytest.mark.parametrize("n", [17, 31, 32, 33, 255, 256, 257, 1000, 4099, 10007])
def test_qc_mfma_vs_brute(ctx, knob_mfma, n):
    print(f"qc mfma brute n={n}", flush=True)
    knob_mfma(1 << 16)
    r = rng(n + 11)
    a, x = rand_bits(r, n), rand_blocks(r, 2 * n)
    assert np.array_equal(qc_gpu(ctx, x, a, n), po.qc_encode_brute(x, a, n))


# the two encoders on one prepared code (prepare keeps both forms), against
# the oracle's Karatsuba product, up to the largest matrix-core size
@pytest.mark.parametrize("n", [12345, 1 << 15, 40000, 1 << 16])
def test_qc_mfma_and_fft_agree(ctx, knob_mfma, n):
    import torch

    print(f"qc mfma/fft n={n}", flush=True)
    r = rng(n + 13)
    a, x = rand_bits(r, n), rand_blocks(r, 2 * n)
    want = po.qc_encode_fast(x, a, n, nthreads=8)
    ahat = torch.zeros(ctx.qc_ahat_len(n), dtype=torch.int32, device="cuda")
    scratch = torch.zeros(ctx.qc_scratch_bytes(n), dtype=torch.uint8, device="cuda")
    ctx.qc_prepare(n, dev_bits(a, n), ahat, scratch)
    xd = to_dev(x)
    for lim in (1 << 16, -1):
        knob_mfma(lim)
        y = dev_blocks(n)
        ctx.qc_encode(n, ahat, xd, y, scratch)
        assert np.array_equal(to_np(y)[:n], want), lim


# y over the first half of x (the C ABI allows the alias), both output modes
@pytest.mark.parametrize("n", [200, 5000])
def test_qc_mfma_in_place(ctx, knob_mfma, n):
    import torch

    knob_mfma(1 << 16)
    r = rng(n + 17)
    a, x = rand_bits(r, n), rand_blocks(r, 2 * n)
    ahat = torch.zeros(ctx.qc_ahat_len(n), dtype=torch.int32, device="cuda")
    scratch = torch.zeros(ctx.qc_scratch_bytes(n), dtype=torch.uint8, device="cuda")
    ctx.qc_prepare(n, dev_bits(a, n), ahat, scratch)
    xd = to_dev(x)
    ctx.qc_encode(n, ahat, xd, xd, scratch)
    assert np.array_equal(to_np(xd)[:n], po.qc_encode_brute(x, a, n))


def test_qc_mfma_special_cases(ctx, knob_mfma):
    knob_mfma(1 << 16)
    n = 3000
    r = rng(5)
    x = rand_blocks(r, 2 * n)
    one = np.zeros((n + 7) // 8, dtype=np.uint8)
    one[0] = 1
    assert np.array_equal(qc_gpu(ctx, x, one, n), x[:n] ^ x[n:])
    s = 2999
    xs = np.zeros((n + 7) // 8, dtype=np.uint8)
    xs[s >> 3] |= 1 << (s & 7)
    assert np.array_equal(qc_gpu(ctx, x, xs, n), x[:n] ^ x[n + (np.arange(n) - s) % n])
    ones = rand_bits(r, n)
    ones[:] = 0xFF
    ones[-1] &= (1 << (n % 8)) - 1 if n % 8 else 0xFF
    # all ones: y_i = x_i ^ XOR of the whole second half
    tot = np.bitwise_xor.reduce(x[n:], axis=0)
    assert np.array_equal(qc_gpu(ctx, x, ones, n), x[:n] ^ tot)


# 4096 and 2^16 take the word-aligned path (n a multiple of 32, >= 64 words)
@pytest.mark.parametrize("n", [1, 33, 1000, 4096, 100003, 1 << 16])
def test_sparse_vs_oracle(ctx, n):
    import torch

    r = rng(n + 7)
    a = rand_bits(r, n)
    w = 37
    pos = np.sort(r.choice(2 * n, size=min(w, 2 * n), replace=False)).astype(np.int64)
    out = torch.zeros(((n + 31) // 32) * 4, dtype=torch.uint8, device="cuda")
    ctx.qc_sparse(n, dev_bits(a, n), torch.from_numpy(pos).cuda(), out)
    got = out.cpu().numpy()[: (n + 7) // 8]
    assert np.array_equal(got, po.qc_sparse(pos, a, n))


# tiles of 128 words, chunks of 512 positions, four in flight per wavefront
@pytest.mark.parametrize("n, w", [(63, 5), (64, 1), (4095, 600), (4097, 512), (8192, 513), (100003, 1027), (1 << 17, 17)])
def test_sparse_tiles_and_chunks(ctx, n, w):
    import torch

    r = rng(n + 5)
    a = rand_bits(r, n)
    pos = np.sort(r.choice(2 * n, size=w, replace=False)).astype(np.int64)
    out = torch.full((((n + 31) // 32) * 4,), 0xA5, dtype=torch.uint8, device="cuda")
    ctx.qc_sparse(n, dev_bits(a, n), torch.from_numpy(pos).cuda(), out)
    assert np.array_equal(out.cpu().numpy()[: (n + 7) // 8], po.qc_sparse(pos, a, n))


@pytest.mark.parametrize("N", [32, 1024, 32 * 1000, 1 << 16])
def test_transpose(ctx, N):
    import torch

    r = rng(N)
    x = rand_blocks(r, N)
    rows = torch.zeros(128 * N // 8, dtype=torch.uint8, device="cuda")
    ctx.bit_transpose(to_dev(x), rows)
    assert np.array_equal(rows.cpu().numpy().reshape(128, N // 8), po.bit_transpose(x))
    back = dev_blocks(N)
    ctx.bit_untranspose(rows, N, back)
    assert np.array_equal(to_np(back), x)


# the product on Frobenius orbits (2^12 < n <= 2^24): both ends of every padded
# length and the neighbours outside its range.  A circulant with a few ones is a
# XOR of rotations at any length; random ones against Karatsuba at small ends.
@pytest.mark.parametrize("n", [4096, 4097, 8192, 8193, 65536, 131073, (1 << 18) + 1, 1 << 19, (1 << 19) + 1,
                               (1 << 20) + 1, (1 << 21) + 1, (1 << 22) + 1, (1 << 23) + 1, 1 << 24])
def test_qc_orbit_product_rotations(ctx, knob_mfma, n):
    import torch

    print(f"qc orbits rotations n={n}", flush=True)
    knob_mfma(-1)
    r = rng(n + 21)
    pos = sorted({0, 1, n - 1, n // 2, int(r.integers(0, n)), int(r.integers(0, n))})
    a = np.zeros((n + 7) // 8, dtype=np.uint8)
    for s in pos:
        a[s >> 3] |= 1 << (s & 7)
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randint(-(1 << 63), (1 << 63) - 1, (2 * n, 2), dtype=torch.int64, device="cuda", generator=g)
    ahat = torch.zeros(ctx.qc_ahat_len(n), dtype=torch.int32, device="cuda")
    scratch = torch.full((ctx.qc_scratch_bytes(n),), 0xA5, dtype=torch.uint8, device="cuda")
    ctx.qc_prepare(n, dev_bits(a, n), ahat, scratch)
    y = dev_blocks(n)
    ctx.qc_encode(n, ahat, x, y, scratch)
    want = x[:n].clone()
    for s in pos:
        want ^= torch.roll(x[n:], s, 0)
    assert torch.equal(y, want)


# conversion and output in columns of 2^16 - 1 (n <= 2^20) or 2^20 - 16 rows: i + n
# near a column's ends, whole and ragged last rows, with and without a wrap
@pytest.mark.parametrize("n", [32769, 65535, 99991, 131072, (1 << 18) - 5, (1 << 20) - 17, 1 << 20,
                               (1 << 21) - 1, (1 << 22) - 100, 3 * (1 << 20) + 513, (1 << 22) + (1 << 20),
                               (1 << 23) - (1 << 18) + 3, (1 << 24) - 1040])
def test_qc_columns_rotations(ctx, knob_mfma, n):
    test_qc_orbit_product_rotations(ctx, knob_mfma, n)


# n a power of two from 2^21 on: folded before the upper levels, one form of the
# output each (2^20: the general one)
@pytest.mark.parametrize("lg", [20, 21, 22, 23, 24])
def test_qc_cyclic_fold_rotations(ctx, knob_mfma, lg):
    test_qc_orbit_product_rotations(ctx, knob_mfma, 1 << lg)


# fewer layers per upper pass: several passes, tiles of 2^2 .. 2^5 rows
@pytest.mark.parametrize("radix", [2, 3, 5])
@pytest.mark.parametrize("n", [70001, (1 << 20) + 1])
def test_qc_orbit_layers_per_pass(ctx, knob_mfma, n, radix):
    from cuot_amd import tune

    tune.set_knobs(qc_radix=radix, qc_mfma_max=-1)
    try:
        test_qc_orbit_product_rotations(ctx, lambda v: None, n)
    finally:
        tune.set_knobs()


@pytest.mark.parametrize("n", [4097, 8193, 20000, 131073, (1 << 19) + 1])
def test_qc_orbit_product_vs_karatsuba(ctx, knob_mfma, n):
    print(f"qc orbits karatsuba n={n}", flush=True)
    knob_mfma(-1)
    r = rng(n + 23)
    a, x = rand_bits(r, n), rand_blocks(r, 2 * n)
    assert np.array_equal(qc_gpu(ctx, x, a, n), po.qc_encode_fast(x, a, n, nthreads=8))


# n > 2^24 stays with the transform on packed chunks: one more upper pass than
# 2^24 took (2^22 elements), an upper pass in full mode (2^24 elements), the
# conversion level by level, A^ in tiles, and other pass shapes by the knobs
@pytest.mark.parametrize("n, radix, cols", [((1 << 24) + 1, 0, 0), ((1 << 24) + 1, 3, 4), ((1 << 25) - 17, 8, 8),
                                            ((1 << 25) + 1, 5, 1), ((1 << 26) + 1, 0, 0)])
def test_qc_long_product_rotations(ctx, n, radix, cols):
    from cuot_amd import tune

    tune.set_knobs(qc_radix=radix, qc_cols=cols, qc_mfma_max=-1)
    try:
        test_qc_orbit_product_rotations(ctx, lambda v: None, n)
    finally:
        tune.set_knobs()


# y over x, on every form of the output: matrix cores, rows (by the knob), whole
# and half blocks a lane, folded
@pytest.mark.parametrize("n, mfma", [(1000, -1), (1000, 0), (9001, -1), (36000, 0), (50001, 0), (70000, 0), (400001, 0),
                                     ((1 << 20) - 3, 0), (1 << 21, 0), (2500001, 0), (1 << 22, 0), (1 << 23, 0)])
def test_qc_encode_in_place(ctx, knob_mfma, n, mfma):
    import torch

    print(f"qc in place n={n}", flush=True)
    knob_mfma(mfma)
    g = torch.Generator(device="cuda").manual_seed(n)
    a = torch.randint(0, 256, ((n + 7) // 8,), dtype=torch.uint8, device="cuda", generator=g)
    x = torch.randint(-(1 << 63), (1 << 63) - 1, (2 * n, 2), dtype=torch.int64, device="cuda", generator=g)
    ahat = torch.zeros(ctx.qc_ahat_len(n), dtype=torch.int32, device="cuda")
    scratch = torch.full((ctx.qc_scratch_bytes(n),), 0xA5, dtype=torch.uint8, device="cuda")
    ctx.qc_prepare(n, a, ahat, scratch)
    y = dev_blocks(n)
    ctx.qc_encode(n, ahat, x, y, scratch)
    upper = x[n:].clone()
    ctx.qc_encode(n, ahat, x, x, scratch)
    assert torch.equal(x[:n], y) and torch.equal(x[n:], upper)


# whole words of 2^25 bits and more take all positions in one lane, others share
# them out; positions at the ends, and ones to be ignored
@pytest.mark.parametrize("n", [(1 << 25) - 32, (1 << 25) - 1, 1 << 25, (1 << 25) + 1, (1 << 25) + 32])
def test_sparse_wide(ctx, n):
    import torch

    print(f"sparse wide n={n}", flush=True)
    r = rng(n)
    a = rand_bits(r, n)
    pos = np.array([-1, 0, 77, n - 1, n, n + 1, n + 63, 2 * n - 1, 2 * n, 2 * n + 5], dtype=np.int64)
    out = torch.full((((n + 31) // 32) * 4,), 0xA5, dtype=torch.uint8, device="cuda")
    ctx.qc_sparse(n, dev_bits(a, n), torch.from_numpy(pos).cuda(), out)
    assert np.array_equal(out.cpu().numpy()[: (n + 7) // 8], po.qc_sparse(pos, a, n))


# 2^26 elements: butterflies with more than 24 bits above them (about 95 GB in all)
def test_qc_longest_product_rotations(ctx):
    import torch

    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 110e9:
        pytest.skip("needs 110 GB of device memory")
    test_qc_orbit_product_rotations(ctx, lambda v: None, (1 << 28) + 1)
    torch.cuda.empty_cache()
