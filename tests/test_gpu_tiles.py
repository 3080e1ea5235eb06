"""k_pretok's two tile sizes: texts around the edges of the small tile (768
bytes), at the largest request that takes it and one byte past, and runs whose
state crosses more than 64 tiles (the wave-wide look-back takes two steps),
against the oracle."""

from __future__ import annotations

import re
from pathlib import Path

import numpy as np
import pytest

from conftest import kit

pytestmark = pytest.mark.gpu

# one family per split ruleset (laguna: cl100k inside its newline parts)
NAMES = ["qwen3_8b", "llama_3_1_8b", "gpt2", "deepseek_v3", "gpt_oss_120b",
         "kimi_k3", "laguna_s_2_1"]


def _const(name: str) -> str:
    h = Path(__file__).resolve().parents[1] / "toktier_amd" / "csrc" / "tk_device.h"
    return re.search(rf"constexpr \w+ {name} =\s*([^;]+);", h.read_text()).group(1)


TILE, TILE_S = int(_const("PT_TILE")), int(_const("PT_TILE_S"))
SMALL_MAX = TILE_S * 256 * 7  # PT_SMALL_MAX

_TOKS: dict = {}


def tok(name: str):
    if name not in _TOKS:
        import toktier_amd
        _TOKS[name] = toktier_amd.load(name)
    return _TOKS[name]


def check(name: str, text: str, what) -> None:
    want = kit(name).expected(text)
    assert not isinstance(want, int), (name, what)
    got = tok(name).encode(text).array
    assert np.array_equal(got, want), (name, what)


@pytest.mark.parametrize("name", NAMES)
def test_small_tile_edges(name):
    """Branch atoms of the split at every alignment near a small tile's end."""
    import soak_docs
    rng = np.random.default_rng(71)
    atoms = soak_docs._atoms(name)
    for k in range(48):
        lead = "x" * int(rng.integers(0, 66)) + " "
        body = "".join(atoms[int(i)] for i in rng.integers(0, len(atoms), 700))
        at = k % 8 - 4 + TILE_S * (1 + k % 3)  # the text's last byte
        text = (lead + body).encode()[:at].decode("utf-8", "ignore")
        check(name, text, (k, at))
        check(name, lead + body, k)


@pytest.mark.parametrize("name", NAMES)
def test_runs_across_many_small_tiles(name):
    """Runs whose start or state is over 64 small tiles back: digits, letters
    without case, marks between punctuation, whitespace, line ends."""
    n = 65 * TILE_S + 37
    for run in ("1234567" * (n // 7), "中" * (n // 3), "!́" * (n // 3),
                " " * 3000 + "\n" + "\t" * 3000, "\r\n" * 2000, "Q" * n + "é"):
        for lead in ("", "ab ", "!"):
            check(name, lead + run + " z1", (run[:2], lead))


@pytest.mark.parametrize("name", NAMES)
def test_runs_across_large_tiles(name):
    """Such runs in a request on large tiles, whose o200k / kimi look-back
    takes a tile a step."""
    n = 5 * TILE + 37
    lead = "ab 12 " * (SMALL_MAX // 6 + 1)
    for run in ("1234567" * (n // 7), "中" * (n // 3), "!́" * (n // 3),
                " " * 6000 + "\n" + "\t" * 6000, "\r\n" * 4000, "Q" * n + "é"):
        check(name, lead + run + " z1 " + run + "!", run[:2])


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("past", [0, 1])
def test_largest_small_tile_request(name, past):
    """The last size on small tiles and the first on large ones."""
    from toktier_amd import workloads
    n = SMALL_MAX + past
    text = workloads._ascii_stream(
        np.random.default_rng(5 + past),
        workloads._Words(np.random.default_rng(6), ["the", "Of", "inter", "x9"]), n)
    assert len(text.encode()) == n
    check(name, text, n)


@pytest.mark.parametrize("name", NAMES)
def test_whitespace_runs_across_words(name):
    """Whitespace runs with CR/LF that reach one or more 64-byte words past
    the character asking about them, at drawn alignments, ended by letters,
    punctuation, non-ASCII characters and whitespace, the text's end, and
    (as documents of one batch) a document's start."""
    rng = np.random.default_rng(72)
    unit = ["\n", "\r\n", "\r", "\t", " ", "　", "é", "a", "!", "！", "1", "中"]
    docs = []
    for k in range(160):
        s = "x" * (k % 67)
        for _ in range(int(rng.integers(1, 14))):
            if rng.random() < 0.4:
                s += " " * int(rng.integers(1, 150))
            else:
                s += unit[int(rng.integers(0, len(unit)))] * int(rng.integers(1, 4))
        docs.append(s)
    check(name, "".join(docs), "joined")
    for k, (d, got) in enumerate(zip(docs, tok(name).encode_batch(docs))):
        assert np.array_equal(got.array, kit(name).expected(d)), (name, k)


def _start_showing(js: str) -> str:
    """A variant of an artifact whose only merges join a CR/LF and the blank
    after it: such a blank starts a piece exactly when its id is its own."""
    import json
    from toktier_amd import bpe_tables
    b2u = bpe_tables.bytes_to_unicode()
    spec = json.loads(js)
    merges = [[b2u[a], b2u[b]] for a in b"\n\r" for b in b" \t"]
    toks = [b2u[b] for b in range(256)] + [a + b for a, b in merges]
    spec["model"]["vocab"] = {t: i for i, t in enumerate(toks)}
    spec["model"]["merges"] = merges
    return json.dumps(spec)


@pytest.mark.parametrize("name", NAMES)
def test_crlf_runs_at_every_offset(name):
    """Blanks right after a CR/LF run at each of the 64 offsets of a word,
    after every kind of character, in one text (large tiles), in a request
    that takes the small tiles, and as documents of one batch, each of which
    starts 0 to 127 bytes before its case."""
    import itertools
    import toktier_amd
    from oracle.oracle import Oracle
    from toktier_amd import bpe_tables, classes, families
    js = _start_showing(kit(name).json)
    f, tables = kit(name).family, bpe_tables.load_tables(js)
    o = Oracle(tables, classes.table_named(families.class_table_name(f)),
               classes.nfc_qc_table(), f.ruleset, f.digits_max, f.needs_nfc,
               contractions=f.contractions)
    t = toktier_amd.load(name, tokenizer_json=js)
    o.set_added([a.content.encode() for a in t.added_tokens],
                [a.id for a in t.added_tokens])
    docs, at = [], 0
    for k, unit in enumerate(itertools.product(
            ["a", "!", "！", " ", "1", ""], ["\n", "\r\n", "\n\r" * 33],
            [" ", "    ", "\t" + " " * 65], ["\nfoo", "foo", "\r\n!", "é", "　\n"])):
        body = "".join(unit).encode()
        before = len((unit[0] + unit[1]).encode())
        for off in range(64):  # the first blank's offset in its word
            lead = (off - at - before) % 64 + 64 * (k % 2)
            docs.append(b"x" * lead + body)
            at += len(docs[-1])
    small = docs[::2][:len(docs) * SMALL_MAX // (2 * at)]
    for part in (docs, small):
        joined = b"".join(part)
        assert (len(joined) <= SMALL_MAX) == (part is small)
        got = t.encode(joined.decode()).array
        assert np.array_equal(got, o.encode_bytes(joined)), name
        ids, rows, status = t.engine.encode_batch(part)
        assert not status.any()
        for k, d in enumerate(part):
            want = o.encode_bytes(d)
            assert np.array_equal(ids[int(rows[k]):int(rows[k + 1])], want), (name, k, d)
    t.close()
