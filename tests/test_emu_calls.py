"""Sequences of calls whose mistakes would be accesses to freed memory or
stale results on a GPU, on the CPU build of the product's sources with
AddressSanitizer (tests/emu/run_calls.py, a process per sequence)."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT
from test_emu import _asan_runtime

sys.path.insert(0, os.path.join(ROOT, "tests", "emu"))
import build_emu  # noqa: E402

CASES = ["plastic_log_after_capture", "prescribed_values_after_capture",
         "network_attached_again_after_capture", "state_after_failed_event",
         "state_short_of_memory", "small_state_without_events",
         "lists_short_of_memory", "state_refused",
         "network_without_memory", "materials_without_memory"]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if _asan_runtime() is None:
        pytest.skip("g++ with AddressSanitizer runtime not available")
    return build_emu.build(out=str(tmp_path_factory.mktemp("emu") / "libsps_emu.so"))


@pytest.mark.parametrize("case", CASES)
def test_calls(lib, case):
    env = dict(os.environ, LD_PRELOAD=_asan_runtime(),
               ASAN_OPTIONS="detect_leaks=0:detect_stack_use_after_return=0:halt_on_error=1")
    p = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "emu", "run_calls.py"), lib, case], env=env,
                       capture_output=True, text=True, timeout=600)
    print(p.stdout[-2000:], p.stderr[-3000:])
    assert p.returncode == 0, p.stdout or p.stderr[-3000:]
