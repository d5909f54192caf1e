"""What the library's host code does when a HIP call fails half-way, on the CPU: its HIP calls land in
tests/native/fake_hip.cc (host memory, kernels not run), which logs them and can make two of them fail.
Each test runs in a process of its own, so that no other test sees the stand-in."""
import os
import subprocess
import sys

import pytest

from diffrg_amd import build as B

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C
fake = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)  # before the library: its HIP calls resolve here
fake.fake_log.restype = C.c_char_p
import diffrg_amd as D
L = D.lib()
D.check(L.dfrg_init(0))
qp = C.c_void_p()
D.check(L.dfrg_qp_create(C.byref(qp), 48, 32, 0))
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    if not os.path.exists(B.HIPCC):
        pytest.skip("hipcc not found")
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run([B.HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++20", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "native", "fake_hip.cc"), "-o", so], check=True, timeout=120)

    def go(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(so=so) + code], cwd=ROOT, capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr

    return go


@pytest.mark.parametrize("call", ["L.dfrg_qp_gl(qp, 64, 0, None, None, None, None)",
                                  "L.dfrg_qp_matsubara(qp, 0.1, 1.0, 0, None, None, None, None, None, None)",
                                  "L.dfrg_qp_matsubara(qp, 0.0, 1.0, 0, None, None, None, None, None, None)"])
def test_rule_whose_staging_fails_has_finished_before_its_room_is_reused(run, call):
    # the kernel that writes the rule's room has been launched when the pinned staging is refused: the
    # room may be handed out again only after the stream was waited for
    run(f"""
fake.fake_fail(1, 0)
fake.fake_clear()
assert {call} != 0
log = fake.fake_log().decode()
assert "L" in log and "M" in log and "S" in log[log.rindex("L"):], log
fake.fake_fail(0, 0)
assert {call} == 0
""")


def test_flow_graph_that_cannot_be_instantiated_is_destroyed(run):
    run("""
fs, fid = C.c_void_p(), C.c_longlong()
D.check(L.dfrg_fs_create(C.byref(fs), qp, 1 << 20, 4, 64, 100, 0.3, 10))
desc = D.FlowDesc(64, 4.0, 0.2, 0.0, 4.0, 0.2, 1.0)
D.check(L.dfrg_fs_submit(fs, C.byref(desc), C.byref(fid)))
fake.fake_clear()
fake.fake_fail(0, 1)
for _ in range(3):
    assert L.dfrg_fs_progress(fs, None, None, None) != 0
log = fake.fake_log().decode()
assert log.count("C") == log.count("D") == 3, log
fake.fake_fail(0, 0)
D.check(L.dfrg_fs_progress(fs, None, None, None))
D.check(L.dfrg_fs_destroy(fs))
log = fake.fake_log().decode()
assert log.count("C") == log.count("D"), log
""")
