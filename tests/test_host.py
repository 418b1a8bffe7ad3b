"""The native host module (``logssms_amd._host``): argument conversion and the
checks made before any launch.  No GPU call is made."""

import os
import shutil
import subprocess
import sys
import threading
import time

import pytest
import torch

from logssms_amd import _lib
from logssms_amd.layers import GatedDeltaConfig

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")


def test_typed_entries_convert_or_refuse():
    host = _lib.host()
    assert _lib.entry("gdn_rms_norm_gated") is host.gdn_rms_norm_gated
    assert _lib.entry("gdn_metadata_copy") is _lib.lib().gdn_metadata_copy  # (no typed entry: host tables)
    ok = [None, 1, 0, 128, None, 1, 32, 4096, 128, 1, None, 0, 1e-6, None, None]
    assert host.gdn_rms_norm_gated(*ok) == 0  # no rows: nothing to do
    with pytest.raises(TypeError, match="15 arguments expected, 14 given"):
        host.gdn_rms_norm_gated(*ok[:-1])
    for i, bad in ((1, "bf16"), (1, 1.5), (12, "x"), (0, 1.5), (1, 1 << 40), (2, 1 << 70)):
        args = list(ok)
        args[i] = bad
        with pytest.raises((TypeError, OverflowError)):
            host.gdn_rms_norm_gated(*args)
    # gdn_last_error is the ctypes handle's: one library instance
    assert host.gdn_rms_norm_gated(*(ok[:2] + [4, 0] + ok[4:])) == 1
    assert b"bad shape" in _lib.lib().gdn_last_error()


def test_decode_and_verify_check_their_tensors():
    from logssms_amd.kernel.linear_attention.fused_backend import decode_step, verify_group
    H, HV, d, B = 2, 4, 32, 3
    cfg = GatedDeltaConfig(H, HV, d, d, (2 * H + HV) * d, 3, 0)
    C = cfg.conv_dim

    def args(**other):
        a = dict(mixed=torch.zeros(B, C), gate=torch.zeros(B, HV), beta=torch.zeros(B, HV),
                 weight=torch.zeros(C, 1, 4), A_log=torch.zeros(HV), dt_bias=torch.zeros(HV),
                 conv=torch.zeros(5, 1, C, 3), state=torch.zeros(5, 1, HV, d, d), reads=torch.arange(B),
                 writes=torch.arange(B))
        a.update(other)
        return [a[k] for k in ("mixed", "gate", "beta", "weight", "A_log", "dt_bias")] + [cfg] + [
            a[k] for k in ("conv", "state", "reads", "writes")]

    with pytest.raises(RuntimeError, match="ROCm device"):
        decode_step(*args())
    empty = decode_step(*args(mixed=torch.zeros(0, C), reads=torch.arange(0), writes=torch.arange(0)))
    assert empty.shape == (0, HV, d)
    for bad in (dict(mixed=torch.zeros(B, C + 1)), dict(reads=torch.arange(B + 1)), dict(conv=torch.zeros(5, 1, C, 2)),
                dict(conv=torch.zeros(5, 1, 3, C).transpose(2, 3)), dict(state=torch.zeros(5, HV, d, d)),
                dict(state=torch.zeros(5, 1, HV, d, 2 * d)[..., ::2]), dict(writes=torch.zeros(B, 1, dtype=torch.long))):
        with pytest.raises(AssertionError):
            decode_step(*args(**bad))
    with pytest.raises(AssertionError):
        decode_step(*args(), out=torch.zeros(B, HV, 2 * d))
    with pytest.raises(TypeError):
        decode_step(*args(gate=[0.0]))
    a = args(mixed=torch.zeros(2 * B, C), writes=torch.arange(2 * B).view(B, 2))
    with pytest.raises(RuntimeError, match="ROCm device"):
        verify_group(*a[:9], None, *a[9:], torch.zeros(2 * B, HV, d))
    with pytest.raises(AssertionError):
        verify_group(*a[:9], torch.arange(B), *a[9:], torch.zeros(2 * B, HV, d))


def test_typed_entries_run_without_the_interpreter_lock():
    """Another Python thread gets to run beside a loop of C calls.  (With a
    switch interval that never ends, only a call that gives the lock up lets it:
    the loop below gives it up nowhere else.)"""
    entry = _lib.host().gdn_rms_norm_gated
    args = [None, 1, 0, 128, None, 1, 32, 4096, 128, 1, None, 0, 1e-6, None, None]
    turns, started, stop = [], threading.Event(), []

    def other():
        while not stop:
            turns.append(1)
            started.set()
            time.sleep(0)  # gives the lock up and waits for it

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other, daemon=True)
    sys.setswitchinterval(1000.0)
    try:
        thread.start()
        started.wait()
        seen, until = len(turns), time.monotonic() + 10
        while len(turns) < seen + 2 and time.monotonic() < until:
            assert entry(*args) == 0
        assert len(turns) >= seen + 2
    finally:
        stop.append(1)
        sys.setswitchinterval(interval)
        thread.join()


def test_workspace_is_left_out_where_it_does_not_fit(monkeypatch):
    """The one-launch forms need far less memory: a device with room for those
    alone must still take the call."""
    sizes = (1, 8192, 16, 32, 128, 128)
    ws, n = _lib.workspace("gdn_prefill_workspace_bytes", "cpu", *sizes)
    assert ws.numel() == n > 1 << 27

    def no_room(*args, **kwargs):
        raise torch.OutOfMemoryError("no room")

    monkeypatch.setattr(torch, "empty", no_room)
    assert _lib.workspace("gdn_prefill_workspace_bytes", "cpu", *sizes) == (None, 0)
    assert _lib.workspace("gdn_chunk_workspace_bytes", "cpu", *sizes, 0) == (None, 0)


def test_one_library_instance(tmp_path):
    """With ``LIB_PATH`` on another build of the library (as the stamp tools set
    it), typed entries, ctypes calls and the error text all are of that one
    instance, also after the package's own was in use."""
    other = tmp_path / "libgdn_other.so"
    shutil.copy(_lib.LIB_PATH, other)
    program = f"""
import shutil
import subprocess
import sys
from logssms_amd import _lib
if {{first}}:
    _lib.host()
    _lib._lib = None
_lib.LIB_PATH = {str(other)!r}
bad = [None, 1, 4, 0, None, 1, 32, 4096, 128, 1, None, 0, 1e-6, None, None]
assert _lib.entry("gdn_rms_norm_gated")(*bad) == 1
assert _lib.entry("gdn_rms_norm_gated") is not getattr(_lib.lib(), "gdn_rms_norm_gated")
assert b"bad shape" in _lib.lib().gdn_last_error()
libs = {{{{line.split()[-1] for line in open("/proc/self/maps") if "libgdn" in line}}}}
assert {str(other)!r} in libs and len(libs) == 1 + {{first}}, libs
"""
    for first in (0, 1):
        done = subprocess.run([sys.executable, "-c", program.format(first=first)], capture_output=True, text=True,
                              cwd=os.path.dirname(os.path.dirname(_lib.LIB_PATH)))
        assert done.returncode == 0, done.stderr


def test_an_unbound_module_refuses():
    program = """
import torch
from logssms_amd import _host
try:
    _host.gdn_rms_norm_gated(None, 1, 0, 128, None, 1, 32, 4096, 128, 1, None, 0, 1e-6, None, None)
except RuntimeError as err:
    assert "no library bound" in str(err)
else:
    raise SystemExit("called without a library")
for bad, error in ((0, ValueError), ("x", TypeError)):
    try:
        _host.bind(bad)
    except error:
        continue
    raise SystemExit(f"bound to {bad!r}")
"""
    done = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True,
                          cwd=os.path.dirname(os.path.dirname(_lib.LIB_PATH)))
    assert done.returncode == 0, done.stderr
