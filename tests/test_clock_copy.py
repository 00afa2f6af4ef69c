"""The host's copy of the clock equals the device's after every call, halted blocks included."""
import subprocess

from tests.emu import build_emu


def test_host_clock_equals_the_device_clock():
    r = subprocess.run([build_emu.build(main="clock_copy.cpp")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
