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
    (64, 5200, 64), (81, 4500, 96)])                              # two, four waves a tile
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
