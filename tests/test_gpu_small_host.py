"""A small host request's bytes are read by the literal kernel from the pinned
staging: sizes at the edges of the 16-byte loads, of the kernel's blocks and
of the largest such request, from aligned, misaligned and page-locked sources,
each buffer refilled between calls; and the ids of a call are all there when
it returns; against the oracle."""

from __future__ import annotations

import ctypes as C
import re
from pathlib import Path

import numpy as np
import pytest

from conftest import kit

pytestmark = pytest.mark.gpu

ENGINE = (Path(__file__).resolve().parents[1] / "toktier_amd" / "csrc" /
          "tk_engine.cpp").read_text()
MAP_SMALL = eval(re.search(r"constexpr size_t MAP_SMALL = \(size_t\)([^;]+);",
                           ENGINE).group(1))
BLOCK = 4096  # the literal kernel's bytes a block


@pytest.fixture(scope="module")
def qwen():
    import toktier_amd
    from toktier_amd import workloads
    k = kit("qwen3_8b")
    base = workloads.config2(k.json, n_chars=MAP_SMALL + 4096, sample=3).encode()
    return k, toktier_amd.load("qwen3_8b"), base


def _cut(base: bytes, n: int, start: int) -> bytes:
    """n bytes of whole characters with a literal across a block's edge."""
    s = base[start:].decode(errors="ignore").encode()
    lit = b"<|im_start|>"
    at = BLOCK - 5
    if n > at + len(lit):
        s = s[:at].decode(errors="ignore").encode().ljust(at, b"x") + lit + s[at:].decode(
            errors="ignore").encode()
    return s[:n].decode(errors="ignore").encode().ljust(n, b" ")


@pytest.mark.parametrize("n", [1, 15, 16, 17, BLOCK - 1, BLOCK, BLOCK + 1,
                               5 * BLOCK + 9, MAP_SMALL - 1, MAP_SMALL, MAP_SMALL + 1])
def test_sizes_and_sources(qwen, n):
    import torch
    k, t, base = qwen
    E = t.engine
    raw = np.zeros(n + 32, dtype=np.uint8)
    off = -raw.ctypes.data % 16
    out = np.zeros(n + 1, dtype=np.uint32)
    pinned = torch.empty(n + 32, dtype=torch.uint8, pin_memory=True).numpy()
    # aligned and misaligned pageable bytes, then page-locked ones, each with
    # other text than the call before
    for i, src in enumerate((raw[off:off + n], raw[off + 3:off + 3 + n],
                             pinned[:n], pinned[1:1 + n], raw[off:off + n])):
        b = _cut(base, n, 211 * i)
        src[:] = np.frombuffer(b, dtype=np.uint8)
        m = C.c_size_t()
        st = E._L.tk_engine_encode(E._h, C.c_void_p(src.ctypes.data), n, 0,
                                   C.c_void_p(out.ctypes.data), out.size, C.byref(m))
        assert st == 0, (i, E._L.tk_last_error())
        assert np.array_equal(out[:m.value], k.oracle.encode_bytes(b)), i


def test_device_calls_on_two_streams_in_turn(qwen):
    """A call leaves nothing another stream's next call on the same engine could
    meet; the ids are read on a third."""
    import torch
    k, t, base = qwen
    E = t.engine
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    ids = [torch.zeros(3 * BLOCK, dtype=torch.int32, device="cuda") for _ in streams]
    for i in range(12):
        b = _cut(base, 2 * BLOCK + 37 * i, 101 * i)
        x = torch.frombuffer(bytearray(b), dtype=torch.uint8).cuda()
        torch.cuda.synchronize()
        m = C.c_size_t()
        st = E._L.tk_engine_encode_device(
            E._h, C.c_void_p(x.data_ptr()), len(b), 0, C.c_void_p(ids[i & 1].data_ptr()),
            ids[i & 1].numel(), C.byref(m), C.c_void_p(streams[i & 1].cuda_stream))
        assert st == 0, (i, E._L.tk_last_error())
        got = ids[i & 1][:m.value].cpu().numpy().view(np.uint32)
        assert np.array_equal(got, k.oracle.encode_bytes(b)), i


@pytest.mark.parametrize("locked", [False, True])
def test_every_id_is_there_when_a_call_returns(qwen, locked):
    """Small calls in turn whose ids end in a partly filled line of the buffer
    that the device writes, each other than the one before at that place: an id
    still on its way when the call returns would show the earlier call's."""
    import torch
    k, t, base = qwen
    E = t.engine
    texts = [_cut(base, 700 + 37 * i, 977 * i) for i in range(24)]
    want = [k.oracle.encode_bytes(b) for b in texts]
    room = max(len(b) for b in texts)
    out = (torch.zeros(room, dtype=torch.int32, pin_memory=True).numpy().view(np.uint32)
           if locked else np.zeros(room, dtype=np.uint32))
    m = C.c_size_t()
    for i in range(40 * len(texts)):
        j = 7 * i % len(texts)
        b, w = texts[j], want[j]
        st = E._L.tk_engine_encode(E._h, b, len(b), 0, C.c_void_p(out.ctypes.data),
                                   out.size, C.byref(m))
        assert st == 0 and m.value == w.size, (i, E._L.tk_last_error())
        assert np.array_equal(out[:w.size], w), i
