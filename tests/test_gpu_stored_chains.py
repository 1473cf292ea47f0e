"""Chains of stored blocks, whose byte-aligned headers are candidates of their own."""

import zlib

import numpy as np
import pytest

import workloads
from gpu_helpers import capi_decompress
from oracle import oracle

pytestmark = pytest.mark.gpu

KIB = 1 << 10


def _stored(piece, final=False):
    n = len(piece)
    return bytes([int(final)]) + n.to_bytes(2, "little") + (n ^ 0xffff).to_bytes(2, "little") + piece


def _wrap(body, data):
    return b"\x78\x9c" + body + zlib.adler32(data).to_bytes(4, "big")


def _random(n, seed):
    return np.random.default_rng(seed).integers(0, 256, n, dtype=np.uint8).tobytes()


@pytest.mark.parametrize("block", [1, 5, 60, 2043, 2048, 16383, 65535])
@pytest.mark.parametrize("limits", [(), (1, 65536)])
def test_chain(gpu, block, limits):
    """Blocks below and above a discovery range; one candidate allowed."""
    data = _random(min(300 * block, 2500 * KIB) + 3, block)
    pieces = [data[i:i + block] for i in range(0, len(data), block)]
    stream = _wrap(b"".join(_stored(p, i == len(pieces) - 1) for i, p in enumerate(pieces)), data)
    got, status, _ = capi_decompress(stream, len(data), *limits)
    want, want_status = oracle.decompress(stream, len(data), *limits)
    assert (status, got) == (want_status, want)
    assert limits or (status == 0 and got == data)


@pytest.mark.parametrize("level", [0, 6])
def test_chain_between_coded_blocks(gpu, level):
    """Text, a chain of stored blocks whose payload looks like such a chain, text."""
    fake = b"".join(_stored(_random(5, i)) for i in range(400))
    parts = [workloads.text_like(200 * KIB, np.random.default_rng(1)), _random(300 * KIB, 2), fake,
             _random(100 * KIB, 3), workloads.text_like(200 * KIB, np.random.default_rng(4))]
    body, data = b"", b"".join(parts)
    for i, part in enumerate(parts):
        c = zlib.compressobj(6 if i in (0, 4) else level, zlib.DEFLATED, -15)
        body += c.compress(part) + c.flush(zlib.Z_FINISH if i == 4 else zlib.Z_FULL_FLUSH)
    got, status, _ = capi_decompress(_wrap(body, data), len(data))
    assert status == 0
    assert got == data


@pytest.mark.parametrize("cut", [1, 4, 5, 70000])
def test_broken_chain(gpu, cut):
    """A chain cut short, and one whose last header is wrong: the oracle's statuses."""
    data = _random(400 * KIB, cut)
    blocks = [_stored(data[i:i + 65535], False) for i in range(0, len(data), 65535)]
    body = b"".join(blocks)
    for stream in (_wrap(body[:-cut], data),
                   _wrap(body[:-cut] + bytes(cut), data)):
        got, status, _ = capi_decompress(stream, len(data))
        want, want_status = oracle.decompress(stream, len(data))
        assert (status, got) == (want_status, want)


@pytest.mark.parametrize("block", [1500, 2043, 4000])
@pytest.mark.parametrize("order", ["stored first", "stored last", "mixed"])
def test_more_stored_candidates_than_table_slots(gpu, block, order):
    """Thousands of short stored blocks and hundreds of dynamic ones (memLevel 1), whose
    decode tables have a slot per 8 KiB of the stream and 1024 more."""
    noise = _random(7 << 20, block)
    stored = [(_stored(noise[i:i + block]), noise[i:i + block]) for i in range(0, len(noise), block)]
    texts = []
    for i in range(8):
        text = workloads.text_like(256 * KIB, np.random.default_rng(i))
        c = zlib.compressobj(6, zlib.DEFLATED, -15, 1)
        texts.append((c.compress(text) + c.flush(zlib.Z_FULL_FLUSH), text))
    if order == "mixed":
        step = len(stored) // len(texts) + 1
        parts = [p for i, t in enumerate(texts) for p in stored[i * step:(i + 1) * step] + [t]]
    else:
        parts = stored + texts if order == "stored first" else texts + stored
    data = b"".join(raw for _, raw in parts)
    stream = _wrap(b"".join(coded for coded, _ in parts) + _stored(b"end", True), data + b"end")
    assert zlib.decompress(stream) == data + b"end"
    got, status, _ = capi_decompress(stream, len(data) + 3)
    assert status == 0
    assert got == data + b"end"


@pytest.mark.parametrize("tail", [120, 300, 520, 640, 700, 1000])
@pytest.mark.parametrize("size", [30 * KIB, 900 * KIB])
def test_last_header_near_the_end(gpu, size, tail):
    """A small last dynamic block: its header ends close to the body's end."""
    data = workloads.text_like(size, np.random.default_rng(size))
    end = np.random.default_rng(tail).choice(np.frombuffer(b"etaoin shrdlu,.XQ", np.uint8),
                                             tail).tobytes()
    c = zlib.compressobj(9, zlib.DEFLATED, 15, 9, zlib.Z_HUFFMAN_ONLY)
    stream = c.compress(data) + c.flush(zlib.Z_BLOCK) + c.compress(end) + c.flush()
    got, status, _ = capi_decompress(stream, size + tail)
    assert status == 0
    assert got == data + end
