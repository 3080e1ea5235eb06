"""The seam tables that an engine builds when it opens (tk_seams.h), on the
CPU: against a plain restatement on a family's rules, and on tables whose
symbols spell no plain strings or more than any vocabulary holds."""

from __future__ import annotations

import ctypes as C
import shutil
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from conftest import kit

SRC = Path(__file__).resolve().parent / "seam_tables.cpp"
EMPTY = 2**64 - 1
CTX = 4  # SEAM_CTX


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    so = tmp_path_factory.mktemp("seams") / "libseam_tables.so"
    subprocess.run([gxx, "-std=c++17", "-O2", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", str(so), str(SRC)],
                   check=True, capture_output=True, text=True, timeout=120)
    return so


@pytest.fixture(scope="module")
def build(library):
    return lambda *table: seam_tables(library, *table)


def seam_tables(library, keys, vals, byte_id):
    """(mask, bitmap words, shift), or None: no seams."""
    mask, bits = np.zeros(65536, np.uint16), np.zeros(1 << 19, np.uint32)
    words = C.c_uint64()
    keys, vals = np.asarray(keys, np.uint64), np.asarray(vals, np.uint64)
    byte_id = np.asarray(byte_id, np.int32)
    p = [C.c_void_p(a.ctypes.data) for a in (keys, vals, byte_id, mask, bits)]
    shift = C.CDLL(str(library)).seam_tables(p[0], p[1], C.c_uint64(keys.size), *p[2:],
                                             C.byref(words))
    return (mask, bits[:words.value], shift) if shift else None


def _rules(*rules):
    """(left, right, product) ids in rank order, as table words."""
    return ([a << 32 | b for a, b, _ in rules] + [EMPTY],
            [r << 32 | p for r, (_, _, p) in enumerate(rules)] + [0])


def _keys(s: bytes):
    """(bytes before, bytes after, type) at each inner position."""
    for i in range(1, len(s)):
        a, b = min(i, CTX), min(len(s) - i, CTX)
        yield s[i - a:i], s[i:i + b], (a - 1) * CTX + b - 1


def _bit(key, shift: int) -> int:
    left, right, ty = key
    m = 2**32 - 1
    h = (int.from_bytes(left[::-1], "little") * 0x9E3779B1
         + int.from_bytes(right, "little") * 0x85EBCA77 + ty * 0x27D4EB2F) & m
    return ((h ^ (h >> 15)) * 0x2C1B3C6D & m) >> shift


@pytest.mark.parametrize("name", ["gpt2", "deepseek_v3"])
def test_tables_hold_every_inner_position(build, name):
    """Every key of every product and no other; at least 4 bits of the bitmap
    a key."""
    import json
    from toktier_amd import bpe_tables
    t = kit(name).tables
    model = json.loads(kit(name).json)["model"]
    keys = set()
    for a, b in bpe_tables._merge_pairs(model["merges"]):
        keys.update(_keys(bpe_tables.token_to_raw(a + b)))
    mask, bits, shift = build(t.pair_keys, t.pair_vals, t.byte_id)
    assert bits.size == 1 << (27 - shift) and 32 * bits.size >= 4 * len(keys)
    want = np.zeros_like(mask)
    for left, right, ty in keys:
        want[left[-1] << 8 | right[0]] |= 1 << ty
    assert np.array_equal(mask, want)
    words = np.zeros_like(bits)
    at = np.array([_bit(k, shift) for k in keys])
    np.bitwise_or.at(words, at >> 5, (1 << (at & 31)).astype(np.uint32))
    assert np.array_equal(bits, words)


def test_tables_without_plain_strings(build):
    """No seams: a byte without an id, two bytes with one id, an id with two
    spellings; a rule that nothing reaches changes nothing."""
    ids = list(range(256))
    ok = build(*_rules((97, 98, 300), (300, 99, 301)), ids)
    assert ok is not None
    dead = build(*_rules((97, 98, 300), (300, 99, 301), (900, 97, 302)), ids)
    assert np.array_equal(ok[0], dead[0]) and np.array_equal(ok[1], dead[1])
    assert build(*_rules((97, 98, 300)), [-1] + ids[1:]) is None
    assert build(*_rules((97, 98, 300)), [1] + ids[1:]) is None
    assert build(*_rules((97, 98, 300), (98, 97, 300)), ids) is None


def test_memory_of_a_table_of_long_chains(library):
    """Rules that spell 4,096 strings of up to 4,096 bytes a byte, half a
    gigabyte in all: no seams, and a bounded amount of memory (the peak of a
    process of its own)."""
    code = f"""
import resource, sys
sys.path.insert(0, {str(SRC.parent)!r})
import test_seam_tables as t
rules, nid = [], 256
for b in range(60):
    left = b
    for _ in range(4095):
        rules.append((left, 97, nid))
        left, nid = nid, nid + 1
args = (*t._rules(*rules), list(range(256)))
before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
assert t.seam_tables({str(library)!r}, *args) is None
print(resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before)
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    assert int(r.stdout) < 200_000  # KiB
