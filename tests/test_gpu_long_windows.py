"""The two phases of a long piece's windows, a wave each (k_long_windows,
k_long_segments, k_repair_merge): letter runs that start and end around the
64-byte windows and their halves, the text's end among them, against the
oracle."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import kit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["qwen3_8b", "llama_3_1_8b"])
@pytest.mark.parametrize("lead", [0, 31, 32, 63])
def test_runs_at_window_edges(name, lead):
    import toktier_amd
    from toktier_amd import workloads
    words = workloads._vocab_lists(kit(name).json)["words"]
    rng = np.random.default_rng(41 + lead)
    t = toktier_amd.load(name)
    for end in (640, 671, 672, 673, 703, 704, 705, 4096, 8191, 8193):
        s = ""
        while len(s) < end:
            s += words[min(len(words) - 1, int(rng.zipf(1.2)) - 1)]
        text = "." * lead + s[: end - lead]
        want = kit(name).expected(text)
        assert not isinstance(want, int)
        assert np.array_equal(t.encode(text).array, want), (lead, end)
    t.close()
