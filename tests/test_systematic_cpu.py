"""The resampler's 64-bit thresholds and component keys against their 128-bit
definitions, over the whole range of sizes (host build of
csrc/pf_common.hpp; exact)."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(__file__), "cpp", "test_systematic")


def test_thresholds_and_component_keys_exact():
    if not os.path.exists(BIN):
        pytest.skip("tests/cpp/test_systematic is built by __graft_entry__.build()")
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "comparisons" in r.stdout
