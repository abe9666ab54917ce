"""matmul_q8_0_direct and the W4A8 product below the LDS-tiled GEMM, bit for
bit against the oracle (block dots and outputs): row counts at the edges of
the 16-row groups, with one and two groups a wave, on few and many channels;
and the entry point's own rows against the no-allocation one, whose staging
holds whole groups of rows only up to its limit."""
import numpy as np
import pytest

import closed_form as CF
import oracle_lib as O
from gpu_util import F32, assert_bits_equal, dev, empty, host, synth_q4_0, synth_q8_0, torch

pytestmark = pytest.mark.gpu


def mri():
    import mri_qmatmul
    return mri_qmatmul


@pytest.mark.parametrize("m,n,k", [
    (5, 33, 96), (16, 40, 288), (17, 100, 544), (32, 16, 1056),   # one group a wave
    (17, 8210, 64), (32, 8200, 256),                              # two, many channels
    (33, 17, 320), (49, 1000, 96), (100, 300, 512),
    (64, 5200, 64), (81, 4500, 96),
    (16, 16392, 64), (40, 8200, 96), (100, 10000, 64),            # two tiles; one and two groups
    (70, 33000, 64), (77, 50008, 32)])                            # two tiles of two and four
@pytest.mark.parametrize("fmt", ["q8_0", "w4a8"])
def test_rows_bit_exact(m, n, k, fmt):
    t = torch()
    rng = np.random.default_rng(m + 5 * n + k)
    x = (rng.standard_normal((m, k)) * np.exp(rng.standard_normal(k))).astype(F32)
    if fmt == "q8_0":
        raw = synth_q8_0(rng, n, k, with_min=True)
        ref, bd, sa = O.matmul_q8_0_direct(x, raw, n, k, want_block_dots=True)
        w, f = mri().Q8Matrix.from_raw_bytes(raw, n, k), mri().matmul_q8_0_direct
    else:
        raw = synth_q4_0(rng, n, k)
        ref, bd, sa = O.matmul_q8_0_direct(x, CF.q4_0_to_q8_0(raw, n, k), n, k,
                                           want_block_dots=True)
        w, f = mri().Q4Matrix.from_raw_bytes(raw, n, k), mri().matmul_q4_0_w4a8
    out = t.full((m + 1, n), 7.0, device="cuda")
    f(dev(x), w, out[:m])
    got = host(out)
    assert_bits_equal(got[:m], ref, "outputs")
    assert np.all(got[m] == 7.0)
    dots, scales = empty((m, n, k // 32), t.int32), empty(m, t.float32)
    f(dev(x), w, out[:m], dots, scales)
    assert_bits_equal(host(out)[:m], ref, "outputs beside block dots")
    assert np.array_equal(host(dots), bd)
    assert_bits_equal(host(scales), sa, "scales")


def test_noalloc_at_its_staging_limit():
    """The most rows that the fixed staging holds, not a whole number of
    groups of 16: accepted, with the allocating entry point's bits."""
    t = torch()
    n, k = 40, 4096
    m = mri().NOALLOC_SCRATCH_BYTES // (k + 4)
    while (m * k + 255) // 256 * 256 + m * 4 > mri().NOALLOC_SCRATCH_BYTES:
        m -= 1
    if m % 16 == 0:
        m -= 1
    rng = np.random.default_rng(4)
    w = mri().Q8Matrix.from_raw_bytes(synth_q8_0(rng, n, k), n, k)
    x = dev(rng.standard_normal((m, k)).astype(F32))
    a, b = empty((m, n), t.float32), empty((m, n), t.float32)
    mri().matmul_q8_0_direct(x, w, a)
    mri().matmul_q8_0_direct_noalloc(x, w, b)
    assert_bits_equal(host(b), host(a), "no-allocation staging limit")


@pytest.mark.parametrize("m,n,k", [(130, 9000, 64), (300, 12008, 96), (523, 250, 1056)])
def test_block_order_at_many_rows(m, n, k):
    """matmul_q8_0_direct_exact where the rows and channels fill waves of two
    and four groups of rows and two tiles, and not quite."""
    t = torch()
    rng = np.random.default_rng(m + n)
    x = (rng.standard_normal((m, k)) * np.exp(rng.standard_normal(k))).astype(F32)
    raw = synth_q8_0(rng, n, k, with_min=True)
    ref, _, _ = O.matmul_q8_0_direct(x, raw, n, k, want_block_dots=True)
    out = t.full((m + 1, n), 7.0, device="cuda")
    mri().matmul_q8_0_direct_exact(dev(x), mri().Q8Matrix.from_raw_bytes(raw, n, k), out[:m])
    got = host(out)
    assert_bits_equal(got[:m], ref, "outputs")
    assert np.all(got[m] == 7.0)


def test_noalloc_gemm_at_its_staging_limit():
    """As above with enough channels for the LDS-tiled kernel, on rows instead
    of row groups: its own order of sums, within the entry point's contract."""
    t = torch()
    m, n, k = 1022, 1100, 4096
    assert m * (k + 4) <= mri().NOALLOC_SCRATCH_BYTES < 1024 * (k + 4)
    rng = np.random.default_rng(6)
    raw = synth_q8_0(rng, n, k)
    x = rng.standard_normal((m, k)).astype(F32)
    w = mri().Q8Matrix.from_raw_bytes(raw, n, k)
    out = empty((m, n), t.float32)
    mri().matmul_q8_0_direct_noalloc(dev(x), w, out)
    got, rows = host(out), [0, 17, 511, 1008, 1021]
    ref, bd, sa = O.matmul_q8_0_direct(x[rows], raw, n, k, want_block_dots=True)
    d, _ = CF.q8_0_split(raw, n, k)
    terms = np.abs(bd.astype(np.float64) * d[None]).sum(axis=2) * np.asarray(sa)[:, None]
    assert np.all(np.abs(got[rows] - ref.astype(np.float64)) <= 1e-5 * np.maximum(np.abs(ref), terms))
