"""The blocks of freed buffers, against a system that refuses to take one back: which of them may be handed on, and who waits.

The rule is host code without HIP (ferrum_amd/csrc/freed_blocks.hpp); the program also runs under ThreadSanitizer.
"""
import subprocess

import pytest

from ferrum_amd import build


@pytest.mark.parametrize("sanitize", [False, True])
def test_only_blocks_that_a_free_has_waited_for_are_handed_on(sanitize):
    run = subprocess.run([build.build_freed_blocks_test(sanitize)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout + run.stderr
