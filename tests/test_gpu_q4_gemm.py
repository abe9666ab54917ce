"""matmul_q4_0_dequant on the matrix cores: the per-block kernel of up to 4
rows and every tile size and K split of the tiled one, at the edges of their
ranges, in both nibble orders, from weights at 2-byte alignment, against the
product in 64 bits.

Tolerance: the activations are split exactly and every product is exact, so
the f32 sums alone round: the entry point's contract (1e-5 of
max(|result|, sum of |terms|)) per element, and 1e-6 in the 2-norm (about 1e-7
per rounding of a sum, the roundings of a block's and a row's sums being
independent)."""
import numpy as np
import pytest

import closed_form as CF
from gpu_util import (F32, assert_bits_equal, dev, empty, host, synth_q4_0, synth_q8_0,
                      torch)

pytestmark = pytest.mark.gpu


def mri():
    import mri_qmatmul
    return mri_qmatmul


def at_two_bytes(raw):
    buf = torch().zeros(raw.size + 2, dtype=torch().uint8, device="cuda")
    buf[2:] = dev(raw)
    return buf[2:]


def exact(x, raw, n, k):
    d, q = CF.q4_0_split(raw, n, k)
    w = np.repeat(d.astype(np.float64), 32, axis=1) * q
    return x.astype(np.float64) @ w.T


def check(got, x, raw, n, k):
    ref = exact(x, raw, n, k)
    err = np.abs(got.astype(np.float64) - ref)
    scale = np.maximum(np.abs(ref), CF.q4_0_terms_abs_sum(x, raw, n, k))
    assert np.all(err <= 1e-5 * scale), float(np.max(err / scale))
    assert np.linalg.norm(err) <= 1e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("m,n,k", [
    (1, 33, 96), (2, 16, 32), (2, 40, 1056), (3, 50, 544), (4, 25, 4128),  # per block
    (1, 70, 8224), (3, 31, 8192), (1, 20, 32768),      # 16 waves; past its LDS
    (2, 33, 14336), (4, 20, 11008), (3, 17, 30016), (2, 40, 27488),  # LDS in parts
    (1, 2500, 8192), (1, 2500, 8448), (1, 3300, 12288),  # staged or per block
    (2, 4100, 2048), (2, 4150, 4096), (2, 40, 8192), (2, 1030, 14336),  # two rows staged
    (3, 6200, 64),                                     # tiled from 3 rows on
    (5, 1, 32), (16, 17, 288), (7, 6200, 544),          # 16-row tiles, narrow and wide
    (17, 33, 32), (32, 31, 288), (18, 8300, 320),       # 32-row tiles
    (33, 129, 96), (64, 127, 1056), (65, 300, 2048),    # 64 x 128 and its K split
    (130, 1000, 4096), (200, 515, 11008),               # 128-row tiles in K parts
    (513, 4100, 256), (1100, 777, 64)])
@pytest.mark.parametrize("ggml", [False, True])
def test_rows_and_tile_edges(m, n, k, ggml):
    rng = np.random.default_rng(m * 7 + n + k)
    raw = synth_q4_0(rng, n, k)
    x = (rng.standard_normal((m, k)) * np.exp(rng.standard_normal(k))).astype(F32)
    out = torch().full((m + 1, n), 7.0, device="cuda")
    disk = CF.q4_0_interleaved_to_ggml(raw) if ggml else raw
    order = mri().Q4_ORDER_GGML if ggml else mri().Q4_ORDER_INTERLEAVED
    for w in (dev(disk), at_two_bytes(disk)):
        mri().matmul_q4_0_dequant_ordered(dev(x), w, n, k, order, out[:m])
        got = host(out)
        check(got[:m], x, raw, n, k)
        assert np.all(got[m] == 7.0)


@pytest.mark.parametrize("scale", [1e-30, 1e30])
def test_wide_range_of_activations(scale):
    """Rows whose values span 2^24 at both ends of the f32 range: the three
    planes carry all of them (for the small ones, down to the last plane's
    2^-133, far below the bound)."""
    rng = np.random.default_rng(5)
    m, n, k = 40, 64, 512
    raw = synth_q4_0(rng, n, k)
    x = (rng.standard_normal((m, k)) * np.exp2(rng.integers(-12, 13, (m, k))) * scale).astype(F32)
    out = empty((m, n), torch().float32)
    mri().matmul_q4_0_dequant(dev(x), dev(raw), n, k, out)
    check(host(out), x, raw, n, k)


def test_nonfinite_activations_stay_in_their_rows():
    rng = np.random.default_rng(6)
    m, n, k = 9, 40, 96
    raw = synth_q4_0(rng, n, k)
    x = rng.standard_normal((m, k)).astype(F32)
    x[2, 5], x[4, 40], x[7, 95] = np.inf, -np.inf, np.nan
    out = empty((m, n), torch().float32)
    mri().matmul_q4_0_dequant(dev(x), dev(raw), n, k, out)
    got = host(out)
    bad = np.array([2, 4, 7])
    assert not np.isfinite(got[bad]).any()
    good = np.setdiff1d(np.arange(m), bad)
    check(got[good], x[good], raw, n, k)


def test_captured_call_needs_no_workspace():
    """A shape that splits K in an eager call is captured on a stream the
    library has not seen, and its replays match."""
    t = torch()
    rng = np.random.default_rng(8)
    m, n, k = 128, 512, 4096
    raw = synth_q4_0(rng, n, k)
    x = rng.standard_normal((m, k)).astype(F32)
    xd, w, out = dev(x), dev(raw), empty((m, n), t.float32)
    mri().matmul_q4_0_dequant(xd, w, n, k, out)
    check(host(out), x, raw, n, k)
    t.cuda.synchronize()
    s = t.cuda.Stream()
    g = t.cuda.CUDAGraph()
    with t.cuda.graph(g, stream=s):
        mri().matmul_q4_0_dequant(xd, w, n, k, out)
    for _ in range(3):
        out.fill_(0)
        g.replay()
        check(host(out), x, raw, n, k)
        xd.copy_(xd * 1.0)


def test_recorded_graph_outlives_a_larger_call():
    """The Q8_0 GEMM's K split recorded on a stream, then a Q4_0 call on that
    stream whose parts need more memory than it: replays and eager Q4_0 calls
    in turn give their own results."""
    t = torch()
    rng = np.random.default_rng(9)
    m, n, k = 200, 6000, 4096
    w8 = mri().Q8Matrix.from_raw_bytes(synth_q8_0(rng, n, k), n, k)
    x8, out8 = dev(rng.standard_normal((m, k)).astype(F32)), empty((m, n), t.float32)
    m4, n4, k4 = 256, 11008, 4096
    raw = synth_q4_0(rng, n4, k4)
    x4, w4 = dev(rng.standard_normal((m4, k4)).astype(F32)), dev(raw)
    out4 = empty((m4, n4), t.float32)
    s = t.cuda.Stream()
    s.wait_stream(t.cuda.current_stream())
    with t.cuda.stream(s):
        mri().matmul_q8_0_direct(x8, w8, out8)
    t.cuda.synchronize()
    want8 = host(out8)
    g = t.cuda.CUDAGraph()
    with t.cuda.graph(g, stream=s):
        mri().matmul_q8_0_direct(x8, w8, out8)
    want4 = None
    for _ in range(3):
        out8.zero_()
        s.wait_stream(t.cuda.current_stream())
        with t.cuda.stream(s):
            mri().matmul_q4_0_dequant(x4, w4, n4, k4, out4)
            g.replay()
        t.cuda.synchronize()
        assert_bits_equal(host(out8), want8, "replay")
        if want4 is None:
            want4 = host(out4)
            check(want4, host(x4), raw, n4, k4)
        assert_bits_equal(host(out4), want4, "Q4_0 beside the graph")


@pytest.mark.parametrize("m,n,k", [
    (128, 512, 4096), (256, 11008, 4096), (512, 4096, 4096), (65, 300, 2080),
    (33, 129, 1056), (200, 515, 11008), (64, 4100, 544)])
def test_captured_call_has_the_eager_bits(m, n, k):
    """A captured call, which has no workspace, adds the K parts of the eager
    one in the same order (the last sizes: stages of two blocks, odd block
    counts), on rows and channels that fill no tile."""
    t = torch()
    rng = np.random.default_rng(m + n + k)
    raw = synth_q4_0(rng, n, k)
    xd, w = dev((rng.standard_normal((m, k)) * np.exp(rng.standard_normal(k))).astype(F32)), dev(raw)
    out, cap = empty((m, n), t.float32), t.full((m + 1, n), 7.0, device="cuda")
    mri().matmul_q4_0_dequant(xd, w, n, k, out)
    t.cuda.synchronize()
    g = t.cuda.CUDAGraph()
    with t.cuda.graph(g, stream=t.cuda.Stream()):
        mri().matmul_q4_0_dequant(xd, w, n, k, cap[:m])
    for _ in range(2):
        cap[:m].fill_(float("nan"))
        g.replay()
        got = host(cap)
        assert_bits_equal(got[:m], host(out), "captured")
        assert np.all(got[m] == 7.0)


def test_eager_call_beside_a_capture():
    """An eager call whose workspace must grow while another stream of the
    thread is being captured: the bits are the same, and the capture ends well."""
    t = torch()
    rng = np.random.default_rng(10)
    n, k = 11008, 4096
    raw = synth_q4_0(rng, n, k)
    w, out, want = dev(raw), empty((256, n), t.float32), empty((256, n), t.float32)
    x = dev(rng.standard_normal((256, k)).astype(F32))
    mri().matmul_q4_0_dequant(x, w, n, k, want)
    y = t.ones(8, device="cuda")
    t.cuda.synchronize()
    a, b = t.cuda.Stream(), t.cuda.Stream()
    g = t.cuda.CUDAGraph()
    with t.cuda.graph(g, stream=a):
        y.add_(1)
        with t.cuda.stream(b):
            mri().matmul_q4_0_dequant(x, w, n, k, out)
    t.cuda.synchronize()
    assert_bits_equal(host(out), host(want), "beside a capture")
    g.replay()
    assert host(y).tolist() == [2.0] * 8


@pytest.mark.parametrize("m,n", [(1, 2**27 + 40), (3, 2**28 + 40)])
def test_channels_past_one_launch(m, n):
    """More channels than one launch has threads for: the first, the last and
    those around the second launch's first are what a call on them alone gives."""
    t = torch()
    k, g = 32, t.Generator(device="cuda")
    g.manual_seed(m)
    raw = t.randint(0, 2**31 - 1, (n * 18 // 4,), dtype=t.int32, device="cuda", generator=g)
    raw = raw.view(t.uint8).view(n, 18)
    raw[:, 1] = 0x1C    # scales of 2^-8 to 2^-7
    x = t.randn(m, k, device="cuda", generator=g)
    out = t.empty(m, n, device="cuda")
    mri().matmul_q4_0_dequant(x, raw.view(-1), n, k, out)
    per = 16 * ((2**32 - 1) // 512 // 8 * 8) if m == 1 else 64 * ((2**32 - 1) // 1024 // 8 * 8)
    part = t.empty(m, 136, device="cuda")
    for a in (0, n // 2, min(per - 64, n - 136), n - 136):
        mri().matmul_q4_0_dequant(x, raw[a:a + 136].reshape(-1), 136, k, part)
        check(host(part), host(x), host(raw[a:a + 136]).ravel(), 136, k)
        got = host(out[:, a:a + 136].contiguous())
        assert np.linalg.norm(got - host(part)) <= 1e-6 * np.linalg.norm(host(part)), a


@pytest.mark.parametrize("m,n,k", [
    (1, 40, 1056), (2, 33, 96), (4, 25, 4128), (3, 31, 8192),        # per block, 8 and 16 waves
    (5, 17, 288), (7, 6200, 544), (17, 33, 288), (18, 8300, 320),    # 16 and 32 rows
    (64, 127, 1056), (130, 1000, 4096), (256, 11008, 4096)])         # 64- and 128-row tiles, parts
@pytest.mark.parametrize("ggml", [False, True])
def test_activations_below_the_planes(m, n, k, ggml):
    """Activations down to 2^-149, whose last bits bf16 does not hold, in every
    row or in one block of one row, eager and captured.  Scales of 1 to 2 keep
    the results' own f32 steps (2^-150 a rounding) below the bound: sums of
    terms of 2^-126 and more, at most 344 roundings."""
    t = torch()
    rng = np.random.default_rng(m * 7 + n + k)
    raw = synth_q4_0(rng, n, k).reshape(-1, 18)
    raw[:, 1] = 0x3C
    raw = raw.ravel()
    order = mri().Q4_ORDER_GGML if ggml else mri().Q4_ORDER_INTERLEAVED
    w = dev(CF.q4_0_interleaved_to_ggml(raw) if ggml else raw)
    out, cap = empty((m, n), t.float32), empty((m, n), t.float32)
    one = rng.standard_normal((m, k))
    for e in (-118, -131):
        x = np.ldexp(one, e).astype(F32)
        part = rng.standard_normal((m, k)).astype(F32)
        part[m // 2, :-32] = 0
        part[m // 2, -32:] = x[m // 2, -32:]
        for v in (x, part):
            xd = dev(v)
            mri().matmul_q4_0_dequant_ordered(xd, w, n, k, order, out)
            check(host(out), v, raw, n, k)
            g = t.cuda.CUDAGraph()
            with t.cuda.graph(g, stream=t.cuda.Stream()):
                mri().matmul_q4_0_dequant_ordered(xd, w, n, k, order, cap)
            for _ in range(2):
                g.replay()
                assert_bits_equal(host(cap), host(out), "captured")
    x = np.ldexp(one[0], -131).astype(F32)   # and beside a scale that is not finite
    raw = raw.copy().reshape(n, -1, 18)
    raw[0, 0, :2] = 0, 0x7C
    raw[0, 0, 2:] = 0xFF
    x[:32] = np.abs(x[:32])
    xd = dev(np.broadcast_to(x, (m, k)).copy())
    w = dev(CF.q4_0_interleaved_to_ggml(raw.ravel()) if ggml else raw.ravel())
    mri().matmul_q4_0_dequant_ordered(xd, w, n, k, order, out)
    assert np.all(host(out)[:, 0] == np.inf)
