"""Row offsets of a batch (k_doc_offsets, a workgroup a row): documents that
start at, before and after a 16-byte group of token slots, a workgroup's step
and a compaction block, empty documents, and the text's end on a block's
edge; rows and ids against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import kit

pytestmark = pytest.mark.gpu

BLOCK = 8192  # token slots of a compaction block


@pytest.mark.parametrize("total", [1, BLOCK - 1, BLOCK, 3 * BLOCK, 3 * BLOCK + 5])
def test_rows_at_every_edge(total):
    import toktier_amd
    k = kit("gpt2")
    t = toktier_amd.load("gpt2")
    rng = np.random.default_rng(51)
    text = bytes(rng.choice(np.frombuffer(b"ab cd\nef12 .", np.uint8), size=total))
    near = (0, 1, 2, 3, 4, 5, 63, 64, 255, 256, 1023, 1024, 1025, 4097)
    cuts = {b + s * e for b in range(0, total + BLOCK, BLOCK) for e in near
            for s in (-1, 1)}
    cuts = sorted(c for c in cuts if 0 < c < total)
    cuts = [0, 0, *cuts, *cuts[::5], total, total]  # (repeats: empty documents)
    cuts.sort()
    docs = [text[a:b] for a, b in zip(cuts, cuts[1:])]
    ids, rows, status = t.engine.encode_batch(docs)
    assert not status.any() and int(rows[0]) == 0
    for d, doc in enumerate(docs):
        want = k.expected(doc.decode()) if doc else np.empty(0, np.uint32)
        assert np.array_equal(ids[int(rows[d]):int(rows[d + 1])], want), (d, cuts[d])
    t.close()
