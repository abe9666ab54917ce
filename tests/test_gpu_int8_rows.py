"""matmul_int8_from_f32 at 2-63 rows, bit for bit against the oracle: rows
that the decode kernel quantizes itself, at every tile count it splits by;
the channel counts and K at which the kernel's tiles, waves and
K runs change (1 or 4 tiles of 16 channels, 4 or 16 waves, runs of no, one
and uneven chunks), rows in one to four tiles of 16, K with and without whole
float4s, and the sizes on both sides of the one-pass quantization."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_util import F32, assert_bits_equal, dev, empty, host, synth_int8_weights, torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (2, 33, 4), (3, 777, 1000), (4, 70, 3072), (4, 16, 3076), (3, 41, 1001),  # decode
    (2, 100, 6000), (3, 8200, 512), (4, 16400, 132), (2, 16390, 8192),
    (5, 1, 1), (16, 17, 63), (17, 40, 130), (33, 33, 1000), (63, 16, 3009),
    (20, 70, 3072), (49, 50, 4111),                      # 16 waves
    (6, 8192, 64), (31, 8177, 200), (40, 8200, 72), (63, 8193, 1028),  # four tiles
    (16, 24, 4096), (17, 24, 4096),                      # one pass, two launches
    (5, 4200, 1000), (30, 8000, 320), (63, 4113, 3000),  # two tiles a workgroup
    (7, 40, 8256), (40, 20, 8300),                       # one tile, long K
])
def test_rows_bit_exact(m, n, k):
    import mri_qmatmul as M
    t = torch()
    rng = np.random.default_rng(m + 3 * n + k)
    q, s = synth_int8_weights(rng, n, k)
    x = (rng.standard_normal((m, k)) * np.exp(rng.standard_normal(k))).astype(F32)
    ref, q0, s0, acc0 = O.matmul_int8_from_f32(x, q, s)
    w = M.QMatrix.from_host(q, s)
    out = t.full((m + 1, n), 7.0, device="cuda")
    qx, sx = empty((m, k), t.int8), empty(1, t.float32)
    acc = empty((m, n), t.int32)
    M.matmul_int8_from_f32(dev(x), w, out[:m], act_q_out=qx, act_scale_out=sx, acc_out=acc)
    got = host(out)
    assert_bits_equal(got[:m], ref, "from f32")
    assert np.all(got[m] == 7.0)
    assert np.array_equal(host(acc), acc0)
    assert np.array_equal(host(qx).ravel(), np.asarray(q0).ravel())
    assert_bits_equal(host(sx), np.asarray([s0], F32), "scale")
    out2 = empty((m, n), t.float32)  # without the optional outputs
    M.matmul_int8_from_f32(dev(x), w, out2)
    assert_bits_equal(host(out2), ref, "from f32, plain")


def test_no_rows_leave_a_scale():
    import mri_qmatmul as M
    t = torch()
    rng = np.random.default_rng(2)
    q, s = synth_int8_weights(rng, 16, 64)
    w = M.QMatrix.from_host(q, s)
    sx = t.zeros(1, device="cuda")
    M.matmul_int8_from_f32(empty((0, 64), t.float32), w, empty((0, 16), t.float32),
                           act_scale_out=sx)
    assert host(sx)[0] == 1.0


@pytest.mark.parametrize("n", [1, 2, 3, 5, 7, 4093, 9001, 65535, 65536, 65537, 600001, 1048577])
def test_tensor_of_any_length_and_alignment(n):
    """The maximum and the rounding of one tensor at every float alignment of
    the input and byte alignment of the output, with the largest value at either
    end; element by element, four at a time, one pass and two launches."""
    import mri_qmatmul as M
    t = torch()
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(F32)
    buf, sx = t.zeros(n + 4, device="cuda"), empty(1, t.float32)
    q = t.full((n + 8,), 77, dtype=t.int8, device="cuda")
    for off in range(4):
        x[(off % 2) * (n - 1)] = -7.5 - off
        q0, s0 = O.quantize_symmetric(x)
        buf[off:off + n] = dev(x)
        q.fill_(77)
        M.quantize_symmetric(buf[off:off + n], q[off + 1:off + 1 + n], sx)
        got = host(q)
        assert_bits_equal(host(sx), np.asarray([s0], F32), "scale")
        assert np.array_equal(got[off + 1:off + 1 + n], q0)
        assert np.all(got[:off + 1] == 77) and np.all(got[off + 1 + n:] == 77)
