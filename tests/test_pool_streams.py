"""A pool's stream is a plain one: nothing in the library makes a stream with a
hardware queue of its own, whose end a pool would have to wait for."""
import subprocess

from nonnewton_amd import build


def test_no_stream_with_a_cu_mask():
    out = subprocess.run(["nm", "-D", "--undefined-only", build.LIB], capture_output=True, text=True, check=True).stdout
    assert "hipStreamCreateWithFlags" in out
    assert "CUMask" not in out
