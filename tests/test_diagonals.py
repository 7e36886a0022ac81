"""The diagonals that the host builder finds and its words for the rows
(csrc/format.cpp) against a plain count, on the CPU with the sanitizers
(tests/native/diagonals.cpp)."""
import os

import pytest

from test_sanitizers import CSRC, NATIVE, _build, _run, pytestmark  # noqa: F401


@pytest.mark.parametrize("sanitize", ["address,undefined", "thread"])
def test_diagonals_wherever_they_are(tmp_path, sanitize):
    exe = _build(tmp_path, "diagonals", sanitize,
                 [os.path.join(NATIVE, "diagonals.cpp"), os.path.join(CSRC, "format.cpp")])
    _run([exe])
