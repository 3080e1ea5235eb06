"""CPU model of the decision that k_pretok takes from the byte masks of a
64-byte word and of the words beside it, for a whitespace character right
after a CR/LF.

In the cl100k and DeepSeek splits such a character starts a piece unless
another CR/LF follows in its whitespace run and the CR/LF run before it was
not taken by a punctuation match's ``[\\r\\n]*``. The device reads both from
masks: bytes that are blanks (space, tab, VT, FF), CR/LF and above 0x7F, and
the document starts. The masks of the next word are read when the word's last
byte is whitespace, those of the word before when the word's first byte is a
CR/LF or is itself the character that asks. What the masks leave open (a run
past the next word, a non-ASCII character where it matters) is walked. In the
o200k and kimi splits the masks answer only whether another CR/LF follows.

The model restates the decision with the device's bit arithmetic and checks
every answer against the oracle's split, for runs at all 64 offsets of a
word, with and without document starts around them. Planted mistakes must
each answer some position wrongly: the masks of the word before not read for
the word's first character, a mask shifted by 64 that comes out full instead
of empty, document starts in the word before not read, and those in the next
word not read.
"""

from __future__ import annotations

import itertools

import pytest

from conftest import kit

ALL = (1 << 64) - 1
BLANK, CRLF = b" \t\x0b\x0c", b"\r\n"


def ctz(m: int) -> int:
    return (m & -m).bit_length() - 1


def masks(data: bytes, wd: int) -> tuple[int, int, int]:
    """(blanks, CR/LF, bytes above 0x7F) of word wd; bytes outside the text
    are staged as zeros."""
    ws = cr = hi = 0
    for j, b in enumerate(data[64 * wd:64 * wd + 64]):
        ws |= (b in BLANK) << j
        cr |= (b in CRLF) << j
        hi |= (b >= 0x80) << j
    return ws, cr, hi


def doc_word(docs, wd: int) -> int:
    return sum(1 << (d & 63) for d in docs if d >> 6 == wd)


def lanes_from(lo: int, plant=None) -> int:
    """Bits lo..63; none for lo 64 (the planted shift wraps around)."""
    if plant == "shift_by_64":
        lo &= 63
    return ALL & ~((1 << lo) - 1)


def ahead(data, docs, i, plant=None):
    """(f, fd, g, hi): the run's first byte that is not whitespace, the next
    document start and the next CR/LF after i, as offsets in i's word (64 up:
    in the next one; 128: not there), and whether the byte at f is above
    0x7F or unknown."""
    wd, lane = i >> 6, i & 63
    ws, cr, hi = masks(data, wd)
    above = ALL & ~((2 << lane) - 1)
    dm = doc_word(docs, wd) & above
    stop = ~(ws | cr) & above
    f = ctz(stop) if stop else 64
    fd = ctz(dm) if dm else 64
    g = ctz(cr & above) if cr & above else 64
    if f == fd == g == 64:
        nws, ncr, nhi = masks(data, wd + 1) if (ws | cr) >> 63 else (0, 0, 0)
        dmn = 0 if plant == "next_docs" else doc_word(docs, wd + 1)
        f = 64 + ctz(~(nws | ncr) & ALL) if (nws | ncr) != ALL else 128
        fd = 64 + ctz(dmn) if dmn else 128
        g = 64 + ctz(ncr) if ncr else 128
        return f, fd, g, f == 128 or bool((nhi >> (f - 64)) & 1)
    return f, fd, g, bool(f < 64 and (hi >> f) & 1)


def decide(data, docs, i, is_p, plant=None):
    """The device's answer at i (cl100k, DeepSeek): 1, 0, or None (walked)."""
    wd, lane = i >> 6, i & 63
    ws, cr, hi = masks(data, wd)
    dmw = doc_word(docs, wd)
    f, fd, g, fhi = ahead(data, docs, i, plant)
    if g < f and g < fd:
        below = (1 << lane) - 1
        nc = ~cr & below
        h = nc.bit_length() - 1
        if dmw & below & lanes_from(h + 1) or (h < 0 and wd == 0):
            return 0
        if h >= 0:
            if (ws >> h) & 1:
                return 0
            return None if (hi >> h) & 1 else int(is_p(data[64 * wd + h]))
        # (the first character's own CR/LF lies in the word before)
        if cr & 1 or (lane == 0 and plant != "first_char"):
            pws, pcr, phi = masks(data, wd - 1)
        else:
            pws = pcr = phi = 0
        if pcr == ALL:
            return None
        q = (~pcr & ALL).bit_length() - 1
        dmp = 0 if plant == "docs_before" else doc_word(docs, wd - 1)
        if dmp & lanes_from(q + 1, plant) or (pws >> q) & 1:
            return 0
        return None if (phi >> q) & 1 else int(is_p(data[64 * (wd - 1) + q]))
    if fd <= f and fd != 64 and fd < 128:
        return 1
    return None if fhi else 1


def hint(data, docs, i):
    """The o200k / kimi answer: 0 (another CR/LF follows), 1 (none does) or
    None (walked)."""
    wd, lane = i >> 6, i & 63
    ws, cr, hi = masks(data, wd)
    above = ALL & ~((2 << lane) - 1)
    ns, dm = ~(ws | cr) & ALL, doc_word(docs, wd)
    low = (ns | dm) & above
    low &= -low
    if cr & above & (low - 1):
        return 0
    if low & (dm | ~hi):
        return 1
    if low == 0 and (cr > ns or ns == 0):
        ws, cr, hi = masks(data, wd + 1)
        dm = doc_word(docs, wd + 1)
        end = (~(ws | cr) & ALL) | dm
        end &= -end
        return 0 if cr & (end - 1) else 1 if end & (dm | ~hi) else None
    return None


def asking(data, docs):
    """ASCII blanks right after a CR/LF, no document start at them."""
    return [i for i in range(1, len(data))
            if data[i] in BLANK and data[i - 1] in CRLF and i not in docs]


def cases():
    """(data, docs): what precedes the CR/LF run, the run, blanks and what
    follows, its CR/LF at each offset of a word; document starts in the word
    before, at each character of the case, and in the next word."""
    pre = ["a", "!", " ", "é", "！", ""]
    runs = ["\n", "\r\n", "\n\n\r", "\n" * 66]
    blanks = [" ", "    ", "\t" + " " * 63, " " * 70]
    ends = ["\nfoo", "foo", "é\n", "　\n", ""]
    for off, p, r, b, e in itertools.product(range(64), pre, runs, blanks, ends):
        if off % 9 not in (0, 1) and off < 60 and len(r) + len(b) > 9:
            continue  # (long runs cross the word's edges at any offset)
        lead = 128 + off - len(p.encode())
        case = p + r + b + e
        data = ("x" * lead + case).encode()
        at = [lead + len(case[:k].encode()) for k in range(min(len(case), 7))]
        yield data, set()
        yield data, {lead - 3}
        yield data, {70, 100}
        for d in (at[off % len(at)], 64 * ((128 + off + len(r)) // 64 + 1)):
            if d < len(data) and (data[d] & 0xC0) != 0x80:
                yield data, {d}


def oracle_starts(o, data, docs) -> set[int]:
    cuts = sorted(docs | {0, len(data)})
    out = set()
    for a, b in zip(cuts, cuts[1:]):
        out.update(a + s for s in o.pretokenize(data[a:b])[:-1])
    return out


def ascii_p(name: str):
    """Is the ASCII byte punctuation or a symbol to the family's split (not
    a letter, digit, whitespace or, for DeepSeek, a control character)?"""
    from toktier_amd import classes, families
    cls = classes.table_named(families.class_table_name(kit(name).family))
    bang = cls[ord("!")]
    return lambda b: cls[b] == bang


FAMILIES = ["qwen3_8b", "llama_3_1_8b", "deepseek_v3"]


@pytest.mark.parametrize("name", FAMILIES)
def test_decision_matches_the_oracle(name):
    o, is_p = kit(name).oracle, ascii_p(name)
    n = known = 0
    for data, docs in cases():
        want = None
        for i in asking(data, docs):
            got = decide(data, docs, i, is_p)
            n += 1
            if got is None:
                continue
            known += 1
            if want is None:
                want = oracle_starts(o, data, docs)
            assert got == (i in want), (data, docs, i)
    assert known > 0.5 * n > 10_000


def test_hint_matches_a_walk():
    ws = set("\t\n\x0b\x0c\r \x85\xa0     　") | {
        chr(c) for c in range(0x2000, 0x200B)}
    known = 0
    for data, docs in cases():
        for i in asking(data, docs):
            got = hint(data, docs, i)
            if got is None:
                continue
            known += 1
            stop = min((d for d in docs if d > i), default=len(data))
            run = itertools.takewhile(ws.__contains__, data[i:stop].decode("utf-8"))
            assert got == (not set("\r\n") & set(run)), (data, docs, i)
    assert known > 10_000


@pytest.mark.parametrize("plant", ["first_char", "shift_by_64", "docs_before",
                                   "next_docs"])
def test_planted_mask_mistakes_are_caught(plant):
    o, is_p = kit("qwen3_8b").oracle, ascii_p("qwen3_8b")
    for data, docs in cases():
        for i in asking(data, docs):
            got = decide(data, docs, i, is_p, plant)
            if got is not None and got != (i in oracle_starts(o, data, docs)):
                return
    raise AssertionError(plant)
