"""The synthetic networks' connections, pinned: measurements and the tests' tolerances refer to these networks (CPU)."""
from __future__ import annotations

import hashlib

import numpy as np
import pytest

from flyguy_amd.synth import scaled_3hop, synth_3hop

CROWDED = dict(sizes=(60, 900, 300, 12), edges=(9000, 5000, 400), redrive=(40, 6, 1), sigma=2.0)    # (full rows among them)


@pytest.mark.parametrize("make,want", [
    (lambda: synth_3hop(**CROWDED), "ba6bb6aa08229be3"),
    (lambda: scaled_3hop(64), "f055605b8e584d87"),
    (lambda: scaled_3hop(64, kind="er"), "26e7b44f88ac40be")], ids=["crowded", "lognormal", "er"])
def test_connections_are_the_same_everywhere(make, want):
    m = hashlib.sha256()
    for h in make()[0]["hop"]:
        row = np.repeat(np.arange(len(h["crow"]) - 1), np.diff(h["crow"]))
        assert len(np.unique(row * len(h["tcrow"]) + h["col"])) == len(h["col"])          # no repeated source in a row
        for k in ("crow", "col", "tcrow", "tcol", "twidx", "nid", "drow"):
            m.update(np.ascontiguousarray(h[k], np.int64).tobytes())
    assert m.hexdigest()[:16] == want
