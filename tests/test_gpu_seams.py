"""Pieces of 65-512 bytes cut at their seams (k_piece_split, k_bpe_mid,
k_bpe_rows over the parts), the listed pieces of 33-64 bytes merged one a
lane, and long pieces whose seams are cuts without a certificate: against the
oracle, at the counts and lengths where the routes change."""

from __future__ import annotations

import re
from pathlib import Path

import numpy as np
import pytest

from conftest import drop_byte_tokens, kit

pytestmark = pytest.mark.gpu

HEADER = (Path(__file__).resolve().parents[1] / "toktier_amd" / "csrc" /
          "tk_device.h").read_text()
ROWS_MAX = int(re.search(r"PACK_ROWS_MAX = (\d+);", HEADER).group(1))
MID_MAX = int(re.search(r"PACK_MID_MAX = (\d+);", HEADER).group(1))
MID_MAX_SPLIT = int(re.search(r"PACK_MID_MAX_SPLIT = (\d+);", HEADER).group(1))

_TOKS: dict = {}


def tok(name: str):
    if name not in _TOKS:
        import toktier_amd
        _TOKS[name] = toktier_amd.load(name)
    return _TOKS[name]


def _letters(name: str, rng, n_bytes: int) -> str:
    """CJK, Latin or mixed letters of the family's tokens, about n_bytes."""
    from toktier_amd import workloads
    lists = workloads._vocab_lists(kit(name).json)
    pool = [lists["cjk"] or ["中", "文"], lists["words"]][int(rng.integers(0, 2))]
    s = ""
    while len(s.encode()) < n_bytes:
        if rng.random() < 0.1:
            s += "中é한и"[int(rng.integers(0, 4))]
        s += pool[min(len(pool) - 1, int(rng.zipf(1.2)) - 1)]
    return s.encode()[:n_bytes].decode("utf-8", "ignore")


# (llama_3_1_8b, gpt_oss_120b, kimi_k3: the whole-piece vocabulary rule)
@pytest.mark.parametrize("name", ["qwen3_8b", "llama_3_1_8b", "deepseek_v3",
                                  "gpt_oss_120b", "kimi_k3", "gpt2"])
@pytest.mark.parametrize("count", [ROWS_MAX - 40, ROWS_MAX + 40])
def test_pieces_at_every_length(name, count):
    """Just under and just over the count of queued pieces that are split:
    lengths 33-520 bytes, each edge of a part class (8, 16, 32, 64, 128, 256,
    512) among them, and pieces that are whole vocabulary entries."""
    rng = np.random.default_rng(31)
    edges = [33, 63, 64, 65, 66, 127, 128, 129, 255, 256, 257, 511, 512, 513]
    parts, base = [], [_letters(name, rng, 520) for _ in range(200)]
    for k in range(count):
        n = edges[k % len(edges)] if k % 3 == 0 else int(rng.integers(65, 300))
        n = max(n, 66) if k % 5 else n
        s = base[int(rng.integers(0, len(base)))]
        parts.append(s.encode()[:n].decode("utf-8", "ignore"))
        if k % 97 == 0:
            parts.append(" " * int(rng.integers(60, 140)) + "=" * int(rng.integers(60, 140)))
    text = "\n".join(parts)
    want = kit(name).expected(text)
    assert not isinstance(want, int)
    assert np.array_equal(tok(name).encode(text).array, want)


@pytest.mark.parametrize("name", ["qwen3_8b", "llama_3_1_8b", "gpt2"])
@pytest.mark.parametrize("count", [MID_MAX, MID_MAX + 1, 3 * MID_MAX])
def test_listed_pieces_one_a_lane(name, count):
    """The listed pieces of 33-64 bytes at the count where k_bpe_mid takes
    them over from k_bpe_pack, and three times that."""
    rng = np.random.default_rng(32)
    base = [_letters(name, rng, 64) for _ in range(300)]
    parts = []
    for k in range(count):
        s = base[int(rng.integers(0, len(base)))]
        s = s.encode()[:int(rng.integers(33, 65))].decode("utf-8", "ignore")
        parts.append(s + "x" * max(0, 33 - len(s.encode())))
    text = "\n".join(parts)
    want = kit(name).expected(text)
    assert not isinstance(want, int)
    assert np.array_equal(tok(name).encode(text).array, want)


@pytest.mark.parametrize("name", ["qwen3_8b", "gpt_oss_120b"])
@pytest.mark.parametrize("count", [MID_MAX_SPLIT, MID_MAX_SPLIT + 1])
def test_listed_pieces_beside_split_ones(name, count):
    """The same where longer pieces are split, at the count for that."""
    rng = np.random.default_rng(35)
    base = [_letters(name, rng, 130) for _ in range(300)]
    cut = lambda lo, hi: base[int(rng.integers(0, len(base)))].encode()[  # noqa: E731
        :int(rng.integers(lo, hi))].decode("utf-8", "ignore")
    parts = [cut(70, 131) for _ in range(ROWS_MAX + 40)]
    mid = [cut(36, 65) for _ in range(count)]
    for k, s in enumerate(mid):
        parts.insert(2 * k, s + "x" * max(0, 33 - len(s.encode())))
    text = "\n".join(parts)
    want = kit(name).expected(text)
    assert not isinstance(want, int)
    assert np.array_equal(tok(name).encode(text).array, want)


@pytest.mark.parametrize("name", ["qwen3_8b", "llama_3_1_8b", "deepseek_v3", "kimi_k3"])
def test_long_pieces_between_seams(name):
    """Long pieces whose stretches between seams are just under and over 64
    bytes (the window cuts only the longer ones), periodic stretches without
    a seam, and pieces that are one stretch."""
    rng = np.random.default_rng(33)
    for k in range(40):
        s = ""
        while len(s.encode()) < 700 + 150 * (k % 9):
            s += _letters(name, rng, int(rng.integers(3, 160)))
            if rng.random() < 0.5:
                s += ["a" * 70, "ab" * 33, "中" * 22, "Qz" * 40][int(rng.integers(0, 4))]
        for lead in (" ", "!"):
            text = lead + s + " end " + lead + s[::-1]
            want = kit(name).expected(text)
            if isinstance(want, int):
                continue
            assert np.array_equal(tok(name).encode(text).array, want), (name, k)


@pytest.mark.parametrize("name", ["qwen3_8b", "deepseek_v3", "gpt_oss_120b"])
def test_split_with_and_without_long_pieces(name):
    """Split pieces with parts over 128 bytes, in turn without and with a
    piece over 512: the merges of those parts and the long pieces' chain take
    the same side stream."""
    rng = np.random.default_rng(34)
    base = [_letters(name, rng, 512) for _ in range(150)] + ["Qz" * 70, "ab" * 120]
    for turn in range(6):
        parts = [base[int(rng.integers(0, len(base)))].encode()[:int(rng.integers(66, 512))]
                 .decode("utf-8", "ignore") for _ in range(ROWS_MAX + 40)]
        if turn % 2:
            parts[turn * 100] = _letters(name, rng, 3000)
        text = "\n".join(parts)
        want = kit(name).expected(text)
        assert not isinstance(want, int)
        assert np.array_equal(tok(name).encode(text).array, want), (name, turn)


def test_pieces_of_a_table_without_seams(monkeypatch):
    """Rules with an id of two spellings get no seam tables: the pieces that
    would be split go uncut, as one part each, to the same kernels."""
    import dataclasses
    import toktier_amd
    from oracle.oracle import Oracle
    from toktier_amd import bpe_tables, classes, families
    k = kit("qwen3_8b")
    t, f = k.tables, k.family
    used = t.pair_keys[t.pair_keys != 2**64 - 1]
    sides = np.concatenate([used >> np.uint64(32), used & np.uint64(0xFFFFFFFF)])
    prod = t.pair_vals & np.uint64(0xFFFFFFFF)
    # two rules whose products nothing consumes: the first takes the second's
    # product (the ranks' order stays monotone)
    end = np.flatnonzero((t.pair_keys != 2**64 - 1) & ~np.isin(prod, sides))
    end = end[np.argsort(t.pair_vals[end])]
    vals = t.pair_vals.copy()
    vals[end[0]] = (vals[end[0]] >> np.uint64(32) << np.uint64(32)) | prod[end[1]]
    other = dataclasses.replace(t, pair_vals=vals)
    monkeypatch.setattr(bpe_tables, "load_tables", lambda js: other)
    d = toktier_amd.load("qwen3_8b")
    o = Oracle(other, classes.table_named(families.class_table_name(f)),
               classes.nfc_qc_table(), f.ruleset, f.digits_max, f.needs_nfc)
    rng = np.random.default_rng(36)
    base = [_letters("qwen3_8b", rng, 512) for _ in range(150)]
    for hi in (129, 513):  # (the parts over 128 bytes on their own)
        text = "\n".join(base[int(rng.integers(0, len(base)))].encode()[
            :int(rng.integers(68, hi))].decode("utf-8", "ignore")
            for _ in range(ROWS_MAX + 40))
        want = o.encode_bytes(text.encode())
        assert not isinstance(want, int)
        assert np.array_equal(d.encode(text).array, want), hi
    d.close()


def test_dropped_bytes_and_boundary_table_take_no_parts():
    """An artifact that drops bytes and the boundary-format pair table keep
    the general merges, on text that the split would take."""
    import toktier_amd
    from toktier_amd import _ffi, workloads
    k = kit("qwen3_8b")
    text = workloads.config5(k.json, n_chars=1_000_000, n_runs=1, run_chars=4_000)
    want = k.expected(text)
    t = tok("qwen3_8b")
    try:
        t.engine.set_option(_ffi.TK_OPT_COMPACT_PAIRS, 0)
        assert np.array_equal(t.encode(text).array, want)
    finally:
        t.engine.set_option(_ffi.TK_OPT_COMPACT_PAIRS, 1)
    assert np.array_equal(t.encode(text).array, want)
    js = drop_byte_tokens(kit("gpt2").json, b"Q\xe4")
    from tokenizers import Tokenizer
    text = workloads.config5(k.json, n_chars=300_000, n_runs=1, run_chars=2_000)
    d = toktier_amd.load("gpt2", tokenizer_json=js)
    want = Tokenizer.from_str(js).encode(text, add_special_tokens=False).ids
    assert list(d.encode(text).array) == want
    d.close()
