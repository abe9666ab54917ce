"""What calls do on the host, under a stand-in for the HIP runtime
(fake_hip.c): the device memory they take and give back.  Each check runs in a
process of its own, which loads the stand-in before the library."""
import ctypes as C
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
X, W, OUT = 0x100000, 0x200000, 0x300000   # operands: 16-byte aligned addresses
STREAM = 0x5000


class Host:
    def __init__(self, fake):
        self.f = C.CDLL(fake, mode=C.RTLD_GLOBAL)
        self.f.fake_launch.restype = C.c_char_p
        self.f.fake_alloc_bytes.restype = C.c_size_t
        sys.modules["torch"] = None   # its HIP runtime stays out of this process
        sys.path.insert(0, os.path.join(os.path.dirname(HERE), "mini-rust-inference_amd"))
        import mri_qmatmul
        self.m, self.lib = mri_qmatmul, mri_qmatmul.lib()

    def set(self, name, value):
        C.c_int.in_dll(self.f, name).value = value

    def live(self):
        return {i for i in range(self.f.fake_allocs()) if self.f.fake_live(i)}

    def launches(self, start=0):
        out = []
        for i in range(start, self.f.fake_launches()):
            v = (C.c_uint * 6)()
            name = self.f.fake_launch(i, v).decode()
            out.append((name, list(v)))
        return out

    def q8_0(self, m, k, n):
        h = C.c_void_p()
        self.m.check(self.lib.mri_q8_0_matrix_from_raw_device(W, n * k // 32 * 34, n, k, STREAM,
                                                              C.byref(h)))
        return lambda: self.lib.mri_matmul_q8_0_direct(X, (C.c_size_t * 2)(m, k), 2, h, OUT,
                                                       None, None, STREAM)

    def w4a8(self, m, k, n):
        """The launches of one matmul_q4_0_w4a8."""
        h = C.c_void_p()
        self.m.check(self.lib.mri_q4_0_matrix_from_raw_device(W, n * k // 32 * 18, n, k, 0,
                                                              STREAM, C.byref(h)))
        at = self.f.fake_launches()
        self.m.check(self.lib.mri_matmul_q4_0_w4a8(X, (C.c_size_t * 2)(m, k), 2, h, OUT, None,
                                                   None, STREAM))
        return self.launches(at)

    def q4_0(self, m, k, n, order=0):
        """The launches of one matmul_q4_0_dequant_ordered."""
        at = self.f.fake_launches()
        self.m.check(self.lib.mri_matmul_q4_0_dequant_ordered(
            X, (C.c_size_t * 2)(m, k), 2, W, n * k // 32 * 18, n, k, order, OUT, STREAM))
        return self.launches(at)


def check_q4_0_releases_no_workspace(h):
    """A recorded graph of the Q8_0 GEMM's K split replays with the stream's
    workspace: a later Q4_0 call on the stream, whose parts need more, leaves it."""
    call = h.q8_0(200, 4096, 6000)
    h.m.check(call())
    held = h.live()
    assert "k_gemm_q8_0" in h.launches()[-1][0]
    launched = h.q4_0(256, 4096, 11008)
    assert any("k_q4_0_gemm" in name for name, _ in launched)
    assert held <= h.live()
    for m in (512, 700):
        h.q4_0(m, 11008, 4096)
        assert held <= h.live()


def check_q4_0_without_memory(h):
    """A Q4_0 call whose K parts' memory is refused runs without the split, and
    a workspace that is too small for it stays."""
    h.q4_0(64, 1024, 1024)
    held = h.live()
    h.set("fake_refuse_malloc", 1)
    (whole, _), = h.q4_0(256, 4096, 11008)
    assert "k_q4_0_gemm" in whole and held == h.live()
    small, = h.q4_0(64, 1024, 1024)      # what is there is used
    h.set("fake_refuse_malloc", 0)
    split = h.q4_0(256, 4096, 11008)[-1][0]
    assert split != whole and len(h.live()) == 1
    assert h.q4_0(64, 1024, 1024) == [small]
    h.set("fake_capturing", 1)           # a captured call: the unsplit form too
    assert h.q4_0(256, 4096, 11008)[0][0] == whole


def check_q4_0_beside_a_capture(h):
    """An eager Q4_0 call that takes or grows its workspace while another
    stream is being captured leaves that capture whole."""
    h.set("fake_other_capture", 1)
    h.q4_0(64, 1024, 1024)
    split = h.q4_0(256, 4096, 11008)[-1]
    assert C.c_int.in_dll(h.f, "fake_broken_captures").value == 0
    h.set("fake_other_capture", 0)
    assert h.q4_0(256, 4096, 11008) == [split]


def check_q4_0_grids(h):
    """HIP launches fewer than 2^32 threads in a grid dimension: more channels
    or rows than that take several launches, whose workgroups cover them all."""
    for m, k, n, channels, rows in (
            (1, 32, 2**27 + 40, 16, 1), (2, 32, 2**28, 16, 2),       # a workgroup's outputs
            (1, 256, 2**27 + 40, 8, 1), (1, 256, 2**30, 8, 1),
            (3, 32, 2**28 + 40, 64, 16), (17, 32, 2**28 + 40, 64, 32),
            (1, 32, 2**31 - 1024, 64, 16), (2**29, 32, 1, 128, 128), (2**30, 0, 3, None, None)):
        launched = h.q4_0(m, k, n)
        for name, v in launched:
            assert v[0] * v[3] < 2**32, (m, k, n, name, v)
        if channels:
            need = -(-m // rows) * -(-n // channels)
            got = sum(v[0] for _, v in launched)
            assert need <= got < need + 8, (m, k, n, launched)


def check_q4_0_long_rows(h):
    """Two to four rows whose planes exceed LDS, and a row of few channels, do
    not take the form that was slower for them (kernels of 16 x 16 tiles, and a
    workgroup for 16 channels)."""
    for m, k, n in ((2, 14336, 4096), (2, 28672, 8192), (4, 11008, 4096), (1, 28672, 8192)):
        (name, _), = h.q4_0(m, k, n)
        assert "k_q4_0_gemv" in name, (m, k, n)
    for m, k, n in ((1, 8192, 1024), (1, 8192, 4352), (1, 14336, 2048), (1, 16384, 6144),
                    (2, 8192, 4352), (2, 10240, 5120), (2, 14336, 2048)):
        (name, _), = h.q4_0(m, k, n)
        assert "k_q4_0_lds" in name, (m, k, n)


def check_block_grids(h):
    """As above, for the quantized rows of W4A8 past the LDS-tiled kernel."""
    for m, n in ((2**21, 2**13), (2**21 + 5, 2**13 + 1), (2**17, 2**17), (16, 2**30), (32, 2**30)):
        launched = [(name, v) for name, v in h.w4a8(m, 32, n) if "k_skinny" in name]
        for name, v in launched:
            assert v[0] * v[3] < 2**32, (m, n, name, v)
        assert sum(v[0] * v[3] // 64 for _, v in launched) >= -(-m // 64) * -(-n // 32)


def check_quantize_grids(h):
    """A long tensor that is not whole aligned float4s takes the workgroups of
    one that is: each of them finds the maximum again."""
    def grid(x, n):
        at = h.f.fake_launches()
        h.m.check(h.lib.mri_quantize_symmetric(x, n, OUT, W, STREAM))
        return h.launches(at)[-1][1]
    for n in (1048576, 2**22 - 4):
        assert grid(X, n + 1)[0] <= grid(X, n)[0] + 1 and grid(X + 4, n) == grid(X, n)


CHECKS = [n for n in dir() if n.startswith("check_")]


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["cc", "-O1", "-shared", "-fPIC", "-w", "-I/opt/rocm/include",
                    os.path.join(HERE, "fake_hip.c"), "-o", so], check=True)
    return so


@pytest.mark.parametrize("check", CHECKS)
def test_host(fake, check):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake, check],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    globals()[sys.argv[2]](Host(sys.argv[1]))
