"""moe_forward's host side on the CPU: the engine over a stand-in of the HIP runtime and kernel entry points that store what
the real ones promise the host (tests/cpp/forward_slots.cpp)."""
import os
import shutil
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
HIPCC = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc for the host-only build")
@pytest.mark.parametrize("failing", ["table", "launch"])
def test_failed_forward_leaves_no_slot_waiting(failing):
    """The refresh of the slot table fails, or the expert launch is refused: later forwards and the drain go on at once and
    count every hit."""
    r = subprocess.run(["make", "-C", CPP, "forward_slots", "HIPCC=" + HIPCC], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    r = subprocess.run([os.path.join(CPP, "forward_slots"), failing], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc for the host-only build")
def test_an_entry_point_without_a_stand_in_is_named_and_fails_the_forward():
    """A plan that asks for the windows of the w2 pass in the host-only build: the stub's name and an error, not a call of a
    symbol that nothing defines; later forwards go on."""
    r = subprocess.run(["make", "-C", CPP, "forward_slots", "HIPCC=" + HIPCC], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    r = subprocess.run([os.path.join(CPP, "forward_slots"), "windows"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "moe_experts_prefill_windows called" in r.stderr, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
