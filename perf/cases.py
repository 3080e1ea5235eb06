"""Workloads of the fresh-encode engine for timing: requests a program makes
through the public entry points, from a short prompt to 4,194,304 characters.

The texts follow the five benchmark configurations and the chat layout of
``toktier_amd/workloads.py`` (the same element mixes and Zipf(1.1) draws over
the family's vocabulary), drawn with whole-array random calls so that a
4,194,304-char request takes about a second to make. Every seed is another
text.

A case is a dict:

- ``family``: a tokenizer family of ``toktier_amd.families``;
- ``text``: ``ascii`` (plain words), ``mixed`` (accents and whitespace runs),
  ``code``, ``cjk`` (half CJK, a tenth emoji; ``runs`` unbroken letter runs
  of ``run_chars``), ``chat`` (``mixed`` in the family's turn template, with
  its added tokens);
- ``chars``: characters of the request (of a batch: of all its documents);
- ``entry``: ``facade`` (``Tokenizer.encode``), ``host`` (``Engine.encode``,
  host bytes to a reused page-locked id buffer), ``device``
  (``Engine.encode_device``, bytes and ids in HBM), ``seed``
  (``Engine.encode_seed``: ids and span checkpoints in HBM), ``batch``
  (``Engine.encode_batch``: ``docs`` host documents).
"""

from __future__ import annotations

import json
from functools import lru_cache

import numpy as np
import torch

import toktier_amd
from toktier_amd import standin
from toktier_amd.bpe_tables import token_to_raw

MAX_CHARS = 4_194_304
SEED_STRIDE = 4096  # token stride of the session store's checkpoints

#: UTF-8 bytes and token ids per character (means over the generators below)
_BYTES = {"ascii": 1.0, "mixed": 1.02, "code": 1.0, "cjk": 2.22, "chat": 1.02}
_IDS = {"ascii": 0.35, "mixed": 0.42, "code": 0.33, "cjk": 0.41, "chat": 0.42}


def listed() -> list[dict]:
    return [
        # one short user message: the call's latency
        dict(name="prompt_300", family="qwen3_8b", text="mixed", chars=300,
             entry="facade"),
        # a conversation of a few turns with its template's added tokens
        dict(name="chat_6k_llama", family="llama_3_1_8b", text="chat",
             chars=6_001, entry="facade"),
        # a source file handed over by a tool, bytes already on the device
        dict(name="code_20k_device", family="llama_3_1_8b", text="code",
             chars=20_011, entry="device"),
        # one page-sized document, host to host
        dict(name="page_64k_host", family="qwen3_8b", text="ascii",
             chars=65_536, entry="host"),
        # short documents of a serving queue or an embedding job
        dict(name="batch_short_gpt_oss", family="gpt_oss_120b", text="mixed",
             chars=700_000, docs=1_500, entry="batch"),
        # a chat transcript adopted by the session store
        dict(name="chat_1m_seed", family="qwen3_8b", text="chat",
             chars=1_000_003, entry="seed"),
        # multilingual text with unbroken letter runs, another ruleset
        dict(name="cjk_1m_deepseek", family="deepseek_v3", text="cjk",
             chars=1_048_577, runs=2, run_chars=65_536, entry="device"),
        # a ragged batch of 256 documents, host to host
        dict(name="batch_ragged_gpt2", family="gpt2", text="ascii",
             chars=4_300_000, docs=256, entry="batch"),
        # the headline request: long mixed-script text resident in HBM ...
        dict(name="mixed_4m_device", family="qwen3_8b", text="mixed",
             chars=MAX_CHARS, entry="device"),
        # ... and from host bytes to host ids
        dict(name="mixed_4m_host", family="qwen3_8b", text="mixed",
             chars=MAX_CHARS, entry="host"),
        # a repository of source code
        dict(name="code_4m_device", family="llama_3_1_8b", text="code",
             chars=MAX_CHARS, entry="device"),
        # long multilingual text with ten unbroken 65,536-char letter runs
        dict(name="cjk_4m_device", family="qwen3_8b", text="cjk",
             chars=MAX_CHARS, runs=10, run_chars=65_536, entry="device"),
    ]


_FAMILIES = ["qwen3_8b", "llama_3_1_8b", "gpt2", "deepseek_v3", "gpt_oss_120b",
             "kimi_k3", "qwen3_5_08b", "nemotron_3_nano_4b", "laguna_s_2_1"]


def draw(rng) -> dict:
    entry = rng.choice(["facade", "host", "device", "device", "seed", "batch"])
    family = rng.choice(_FAMILIES)
    text = rng.choice(["ascii", "mixed", "code", "cjk", "chat"])
    lo, hi = {"facade": (64, 200_000), "batch": (20_000, 4_000_000),
              "seed": (50_000, 2_000_000)}.get(entry, (256, 4_000_000))
    if text == "cjk":
        hi = min(hi, 1_500_000)  # below the largest listed request
    chars = int(lo * (hi / lo) ** rng.random())
    case = dict(family=family, text=text, chars=chars, entry=entry)
    if entry == "batch":
        case["docs"] = max(2, min(4_000, int(chars / (100 * 300 ** rng.random()))))
    if text == "cjk" and entry != "batch" and chars >= 20_000:
        case["runs"] = rng.randint(0, 3)
        case["run_chars"] = int(600 * 50 ** rng.random())
        case["run_chars"] = min(case["run_chars"], chars // 8)
    return case


# ---- texts

_ACC = {
    "a": "àáâãäå", "e": "èéêë", "i": "ìíîï", "o": "òóôõöø", "u": "ùúûü",
    "y": "ýÿ", "n": "ñ", "c": "ç", "A": "ÀÁÂÃÄÅ", "E": "ÈÉÊË", "O": "ÒÓÔÕÖØ",
}
_PUNCT = list(".,;:!?-()\"'[]/") + ["...", "--", "?!"]
_OPS = ["=", "==", "!=", "+", "-", "*", "/", "%", "<", ">", "<=", ">=", "+=",
        "-=", "->", "=>", "&&", "||", "(", ")", "[", "]", "{", "}", ",", ";",
        ":", ".", "::", "&", "|", "^", "~", "<<", ">>", "@", "#"]
_EMOJI = [chr(c) for c in (*range(0x1F600, 0x1F64F), *range(0x1F300, 0x1F3FF),
                           *range(0x1F680, 0x1F6C5))]


@lru_cache(maxsize=None)
def _vocab(family: str) -> tuple[list[str], list[str]]:
    """The family's ASCII word tokens and CJK tokens in id order."""
    vocab = json.loads(standin.load_artifact_json(family))["model"]["vocab"]
    words, cjk = [], []
    for tok, _ in sorted(vocab.items(), key=lambda kv: kv[1]):
        try:
            w = token_to_raw(tok).decode("utf-8").strip(" ")
        except (KeyError, UnicodeDecodeError):
            continue
        if w and w.isascii() and w.isalpha():
            words.append(w)
        elif w and all(0x4E00 <= ord(ch) <= 0x9FFF for ch in w):
            cjk.append(w)
    return words, cjk


@lru_cache(maxsize=None)
def _zipf_cdf(n: int) -> np.ndarray:
    p = np.arange(1, n + 1, dtype=np.float64) ** -1.1
    return np.cumsum(p) / p.sum()


def _words(rng, toks: list[str], n: int) -> list[str]:
    """n words of one to three Zipf-drawn tokens."""
    k = rng.integers(1, 4, size=n)
    ends = np.cumsum(k).tolist()
    cdf = _zipf_cdf(len(toks))
    idx = np.minimum(np.searchsorted(cdf, rng.random(ends[-1])), len(toks) - 1)
    drawn = [toks[i] for i in idx.tolist()]
    out, at = [], 0
    for e in ends:
        out.append("".join(drawn[at:e]))
        at = e
    return out


def _accent(w: str, pick: int) -> str:
    chars = list(w)
    idx = [i for i, ch in enumerate(chars) if ch in _ACC]
    if not idx:
        return w + "é"
    for i in idx[: max(1, len(idx) // 2)]:
        opts = _ACC[chars[i]]
        chars[i] = opts[pick % len(opts)]
        pick //= 7
    return "".join(chars)


def _digits(rng, n: int, top: int) -> list[str]:
    """n runs of 1..top decimal digits."""
    k = rng.integers(1, top + 1, size=n)
    ends = np.cumsum(k).tolist()
    pool = rng.integers(48, 58, size=ends[-1], dtype=np.uint8).tobytes().decode()
    out, at = [], 0
    for e in ends:
        out.append(pool[at:e])
        at = e
    return out


def _prose(rng, family: str, n_chars: int, latin1: float, ws_runs: float) -> str:
    parts: list[str] = []
    total = col = 0
    while total < n_chars:
        n = (n_chars - total) // 6 + 64
        r, r2 = rng.random(n).tolist(), rng.random(n).tolist()
        acc = (rng.random(n) < latin1).tolist()
        pick = rng.integers(0, 1 << 20, size=n).tolist()
        words, nums = _words(rng, _vocab(family)[0], n), _digits(rng, n, 6)
        ws_len = rng.integers(2, 17, size=n).tolist()
        ws = rng.integers(0, 3, size=17 * n)
        pool = np.array([" ", "\t", "\r\n"], dtype=object)[ws].tolist()
        for j in range(n):
            if r[j] < ws_runs:
                s = "".join(pool[17 * j:17 * j + ws_len[j]])
                parts.append(s)
                total += len(s)
                col = 0 if "\n" in s else col + len(s)
                continue
            if r2[j] < 0.08:
                s = _PUNCT[pick[j] % len(_PUNCT)]
            elif r2[j] < 0.12:
                s = nums[j]
            else:
                s = _accent(words[j], pick[j]) if acc[j] else words[j]
            if col + len(s) + 1 > 80:
                s, col = s + "\n", 0
            else:
                s += " "
                col += len(s)
            parts.append(s)
            total += len(s)
    return "".join(parts)[:n_chars]


def _code(rng, family: str, n_chars: int) -> str:
    parts: list[str] = []
    total = line = 0
    while total < n_chars:
        n = (n_chars - total) // 8 + 64
        r, r2 = rng.random(n).tolist(), rng.random(n).tolist()
        pick = rng.integers(0, 1 << 20, size=n).tolist()
        k3 = rng.integers(1, 4, size=n).tolist()
        words = _words(rng, _vocab(family)[0], 3 * n)
        nums = _digits(rng, n, 20)
        for j in range(n):
            q = r[j]
            if q < 0.20:
                s = _OPS[pick[j] % len(_OPS)]
            elif q < 0.30:
                s = nums[j]
                if r2[j] < 0.5 and len(s) > 2:
                    s = "0x" + ("%x" % int(s))[: len(s) - 2]
            elif q < 0.36:
                esc = ("\\n", "\\t", '\\"', "\\\\")[pick[j] & 3]
                s = f'"{words[3 * j]} {words[3 * j + 1]}{esc}{words[3 * j + 2]}"'
            else:
                toks = [t.lower() for t in words[3 * j:3 * j + k3[j]]]
                if r2[j] < 0.5:
                    s = "_".join(toks)
                else:
                    s = toks[0] + "".join(t[:1].upper() + t[1:] for t in toks[1:])
            line += len(s)
            if line > 70:
                s += "\n" + " " * (4 * (1 + pick[j] % 8))
                line = 0
            elif pick[j] % 10 < 7:
                s += " "
            parts.append(s)
            total += len(s)
    return "".join(parts)[:n_chars]


def _cjk_words(rng, family: str, n: int) -> list[str]:
    """n words of CJK tokens, one in ten a single drawn ideograph."""
    cjk = _vocab(family)[1]
    one = [chr(c) for c in rng.integers(0x4E00, 0xA000, size=n).tolist()]
    if not cjk:
        return one
    rare = (rng.random(n) < 0.1).tolist()
    return [o if x else w for o, x, w in zip(one, rare, _words(rng, cjk, n))]


def _run(rng, words, n_chars: int) -> str:
    out = ""
    while len(out) < n_chars:
        out += "".join(words((n_chars - len(out)) // 2 + 16))
    return out[:n_chars]


def _cjk(rng, family: str, n_chars: int, runs: int, run_chars: int) -> str:
    body = n_chars - runs * run_chars
    latin = lambda n: _words(rng, _vocab(family)[0], n)  # noqa: E731
    cjk = lambda n: _cjk_words(rng, family, n)  # noqa: E731
    # characters of each kind outside the runs (half of them Latin), and the
    # odds of an element of the kind, from its mean length
    half = runs // 2 * run_chars
    want = np.array([0.5 * n_chars - half, 0.1 * n_chars,
                     0.4 * n_chars - (runs * run_chars - half)]).clip(min=1.0)
    odds = want / np.array([32.5, 3.9, 7.0])
    odds /= odds.sum()
    parts: list[str] = []
    total = 0
    while total < body:
        n = (body - total) // 10 + 64
        kinds = rng.choice(3, size=n, p=odds).tolist()
        span = rng.integers(4, 60, size=n).tolist()
        r = rng.random(n).tolist()
        em = rng.integers(0, 1 << 30, size=n).tolist()
        lat, han = latin(n), ""
        at = 0
        for j, kind in enumerate(kinds):
            if kind == 0:
                if at + span[j] > len(han):
                    han, at = "".join(cjk(n + 64)), 0
                s = han[at:at + span[j]] + ("，" if r[j] < 0.6 else "。")
                at += span[j]
            elif kind == 1:
                s, q = "", em[j]
                for _ in range(1 + q % 3):
                    q = q // 3 * 2654435761 % (1 << 30)
                    s += _EMOJI[q % len(_EMOJI)]
                    if q >> 12 & 3 == 0:
                        s += "\u200d" + _EMOJI[(q >> 14) % len(_EMOJI)]
                    if (q >> 22) % 5 == 0:
                        s += "\ufe0f"
                s += " "
            else:
                s = lat[j] + (" " if r[j] < 0.9 else "\n")
            parts.append(s)
            total += len(s)
    text = "".join(parts)[:body]
    cuts = np.sort(rng.integers(0, len(text) + 1, size=runs)).tolist()
    out, prev = [], 0
    for i, c in enumerate(cuts):
        out += [text[prev:c], _run(rng, latin if i % 2 == 0 else cjk, run_chars)]
        prev = c
    return "".join(out) + text[prev:]


#: turn templates: (before everything, open, after the role, close)
_TURNS = {
    "llama_3_1_8b": ("<|begin_of_text|>", "<|start_header_id|>",
                     "<|end_header_id|>\n\n", "<|eot_id|>"),
    "deepseek_v3": ("<｜begin▁of▁sentence｜>", "<｜User｜>", "",
                    "<｜end▁of▁sentence｜>"),
    "gpt_oss_120b": ("", "<|start|>", "<|message|>", "<|end|>"),
    "kimi_k3": ("", "<|im_user|>", "<|im_middle|>", "<|im_end|>"),
    "gpt2": ("", "", "\n", "<|endoftext|>"),
    "laguna_s_2_1": ("", "", "\n", "<|endoftext|>"),
}
_CHATML = ("", "<|im_start|>", "\n", "<|im_end|>\n")


def _chat(rng, family: str, n_chars: int) -> str:
    first, opens, mid, close = _TURNS.get(family, _CHATML)
    body = _prose(rng, family, n_chars, 0.105, 0.05)
    out, total, at, turn = [first], len(first), 0, 0
    while total < n_chars and at < len(body):
        n = int(rng.integers(200, 3001))
        role = ("user", "assistant")[turn % 2]
        piece = opens + role + mid + body[at:at + n] + close
        out.append(piece)
        total += len(piece)
        at += n
        turn += 1
    return "".join(out)[:n_chars]


def _text(case: dict, rng, n_chars: int) -> str:
    fam, kind = case["family"], case["text"]
    if kind == "ascii":
        return _prose(rng, fam, n_chars, 0.0, 0.0)
    if kind == "mixed":
        return _prose(rng, fam, n_chars, 0.105, 0.05)
    if kind == "code":
        return _code(rng, fam, n_chars)
    if kind == "chat":
        return _chat(rng, fam, n_chars)
    return _cjk(rng, fam, n_chars, case.get("runs", 0), case.get("run_chars", 0))


# ---- the calls

@lru_cache(maxsize=None)
def _tokenizer(family: str):
    """A program opens a family's tokenizer once and keeps it."""
    return toktier_amd.load(family)


def _room(case: dict) -> int:
    """Ids a program makes room for: at least the request's bytes, from its
    characters and kind alone (so every seed's buffers have one size)."""
    most = {"ascii": 1.0, "code": 1.0, "cjk": 3.0}.get(case["text"], 1.25)
    return int(case["chars"] * most) + 1024


def prepare(case: dict, seed: int) -> dict:
    rng = np.random.default_rng([seed, case["chars"], 20261204])
    tok = _tokenizer(case["family"])
    text = _text(case, rng, case["chars"])
    entry, room = case["entry"], _room(case)
    state = {"entry": entry, "tok": tok, "engine": tok.engine}
    if entry == "facade":
        state["text"] = text
        state["row"] = np.zeros(room, dtype=np.uint32)
        return state
    data = text.encode("utf-8")
    if entry == "batch":
        # ragged documents, cut between characters
        n = case["docs"]
        w = rng.uniform(0.03, 1.0, size=n)
        ends = np.floor(np.cumsum(w) / w.sum() * len(text)).astype(np.int64).tolist()
        ends[-1] = len(text)
        state["docs"] = [text[a:b].encode("utf-8")
                         for a, b in zip([0] + ends[:-1], ends)]
    if entry in ("host", "batch"):
        # ids land in a page-locked buffer that the program reuses
        pin = torch.zeros(room, dtype=torch.int32, pin_memory=True)
        state["pin"] = pin
        state["out"] = pin.numpy().view(np.uint32)
        state["data"] = data
        return state
    state["data"] = torch.frombuffer(bytearray(data), dtype=torch.uint8).cuda()
    state["ids"] = torch.zeros(room, dtype=torch.int32, device="cuda")
    if entry == "seed":
        state["points"] = torch.zeros((room // SEED_STRIDE + 1, 3),
                                      dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    return state


def run(state: dict):
    """The ids in the program's buffer (zeros past their count) and the
    count; a batch's row offsets and status, a seed's checkpoints."""
    entry, eng = state["entry"], state["engine"]
    if entry == "facade":
        # the ids go into a padded row of the program's model input
        ids = state["tok"].encode(state["text"]).array
        state["row"][: ids.size] = ids
        return state["row"], int(ids.size)
    if entry == "host":
        return state["out"], int(eng.encode(state["data"], out=state["out"]).size)
    if entry == "batch":
        _, rows, status = eng.encode_batch(state["docs"], out=state["out"])
        return state["out"], rows, status
    data, ids = state["data"], state["ids"]
    if entry == "device":
        n = eng.encode_device(data.data_ptr(), data.numel(), ids.data_ptr(),
                              ids.numel())
        return ids, n
    pts = state["points"]
    n, m = eng.encode_seed(data.data_ptr(), data.numel(), ids.data_ptr(),
                           ids.numel(), SEED_STRIDE, pts.data_ptr(), pts.shape[0])
    return ids, pts, n, m


def work(case: dict) -> dict:
    """The text read once and the ids (a batch's rows, a seed's checkpoints)
    written once; the path is integer and byte work, with no products."""
    n = case["chars"]
    ids = n * _IDS[case["text"]]
    by = n * _BYTES[case["text"]] + 4 * ids
    if case["entry"] == "batch":
        by += 12 * case["docs"]
    if case["entry"] == "seed":
        by += 24 * (ids / SEED_STRIDE + 1)
    return {"bytes": int(by), "flops": 0}


def tolerance(case: dict) -> str:
    return "exact"  # token ids, row offsets and byte positions
