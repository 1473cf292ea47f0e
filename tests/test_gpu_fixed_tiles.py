"""Fixed-Huffman runs around the edges of 1 KiB tiles and groups of 64 tiles:
runs that start and end inside a tile, at its edges, and across groups, at every
alignment of the stream."""

import zlib

import numpy as np
import pytest

import deflate_writer as dw
import workloads
from oracle import oracle

pytestmark = pytest.mark.gpu


def _fixed(data, every=0):
    c = zlib.compressobj(1, zlib.DEFLATED, 15, 8, zlib.Z_FIXED)
    step = every or max(1, len(data))
    out = b""
    for i in range(0, len(data), step):
        out += c.compress(data[i:i + step])
        if every:
            out += c.flush(zlib.Z_SYNC_FLUSH)
    return out + c.flush()


def _literal_run(data, final=True):
    """One fixed block of literals only, as the bits it takes (zlib stores such data)."""
    byte = np.frombuffer(data, np.uint8).astype(np.int64)
    length = np.where(byte < 144, 8, 9)
    code = np.where(byte < 144, byte + 0x30, byte + 256)  # 144 -> 0x190
    bits = (code[:, None] >> (length[:, None] - 1 - np.arange(9))) & 1
    literals = bits[np.arange(9) < length[:, None]]
    return np.concatenate(([int(final), 1, 0], literals, np.zeros(7, np.int64))).astype(np.uint8)


def _literal_stream(data):
    body = np.packbits(_literal_run(data), bitorder="little").tobytes()
    assert body[0] >> 1 & 3 == 1
    stream = dw.wrap(body, data)
    assert zlib.decompress(stream) == data
    return stream


def _content(kind, n):
    rng = np.random.default_rng(n + 17)
    if kind == "text":
        return workloads.text_like(n, rng)
    if kind == "noise":  # 8- and 9-bit literals only, for _literal_stream
        return rng.integers(0, 256, n, dtype=np.uint8).tobytes()
    return workloads.runs_segment(n, rng)  # nearly every token a match of 258


def _check(gpu, stream, raw, skew):
    """Decodes a device tensor that starts `skew` bytes into its storage."""
    import cuda_zlib
    import torch
    held = torch.from_numpy(np.frombuffer(b"\xff" * skew + stream + b"\xff" * 8, np.uint8).copy())
    payload = held.to(gpu)[skew:skew + len(stream)]
    out, meta = cuda_zlib.decompress_zlib_checked(payload, len(raw), gpu)
    assert int(meta.cpu().numpy()[0]) == 0
    assert out.cpu().numpy().tobytes() == raw


@pytest.mark.parametrize("kind", ["text", "noise", "runs"])
@pytest.mark.parametrize("size", [66000, 70001, 131072, 140003, 1000003])
def test_runs_of_every_length(gpu, kind, size):
    raw = _content(kind, size)
    stream = _literal_stream(raw) if kind == "noise" else _fixed(raw)
    assert stream[2] >> 1 & 3 == 1
    _check(gpu, stream, raw, size % 4)


@pytest.mark.parametrize("every", [150, 700, 1024, 1700, 66000, 120001])
def test_runs_that_start_and_end_inside_tiles(gpu, every):
    raw = _content("text", 300007)
    _check(gpu, _fixed(raw, every), raw, every % 4)


@pytest.mark.parametrize("start", [0, 3 * 1024 - 1, 3 * 1024, 3 * 1024 + 1, 64 * 1024])
@pytest.mark.parametrize("end", [70 * 1024, 71 * 1024, 128 * 1024, 192 * 1024])
def test_runs_that_end_at_tile_and_group_edges(gpu, start, end):
    """Literal runs whose end of block lies bits before, at and after the edge of a tile
    or a group, from byte `start` of the body on (behind stored blocks)."""
    rng = np.random.default_rng(start + end)
    prefix, before = b"", b""
    while len(prefix) < start:
        n = min(start - len(prefix) - 5, 60000)
        if 0 < start - len(prefix) - 5 - n < 6:
            n -= 6
        piece = rng.integers(0, 256, n, dtype=np.uint8).tobytes()
        prefix += dw.stored(piece, final=False)
        before += piece
    assert len(prefix) == start
    for delta in (-17, -8, -1, 0, 1, 7, 8, 25):
        bits = 8 * (end - start) + delta - 10  # of the literals
        long = bits % 8 + 8 * (bits // 80)     # with 9-bit codes
        short = (bits - 9 * long) // 8
        data = np.concatenate((rng.integers(144, 256, long), rng.integers(0, 144, short)))
        data = rng.permutation(data.astype(np.uint8)).tobytes()
        run = _literal_run(data)
        assert len(run) == 8 * (end - start) + delta
        raw = before + data
        stream = dw.wrap(prefix + np.packbits(run, bitorder="little").tobytes(), raw)
        assert zlib.decompress(stream) == raw
        _check(gpu, stream, raw, delta & 3)


@pytest.mark.parametrize("keep", [0.02, 0.3, 0.77, 0.999])
def test_cut_runs_match_the_oracle(gpu, keep):
    import cuda_zlib
    raw = _content("text", 150001)
    stream = _fixed(raw, 40000)
    cut = stream[:int(len(stream) * keep)] + stream[-4:]
    _, want = oracle.decompress(cut, len(raw))
    out, meta = cuda_zlib.decompress_zlib_checked(cut, len(raw), gpu)
    assert want and int(meta.cpu().numpy()[0]) == want
    assert not out.any()


def _fixed_tokens(body, bit, count):
    """Whether `count` fixed-code tokens decode from body bit `bit` on, a fixed block's header first."""
    bits = int.from_bytes(body[bit // 8:bit // 8 + 8 * count], "little") >> (bit & 7)

    def code(n, at):
        return int(format((bits >> at) & ((1 << n) - 1), "0%db" % n)[::-1], 2)

    if (bits >> 1) & 3 != 1:
        return False
    at = 3
    for _ in range(count):
        c7, c8 = code(7, at), code(8, at)
        if c7 == 0:
            return False
        if c7 < 24 or 0xc0 <= c8 < 0xc8:
            symbol = 256 + c7 if c7 < 24 else 280 + c8 - 0xc0
            at += 7 if c7 < 24 else 8
            if symbol > 285:
                return False
            at += 0 if symbol < 265 or symbol == 285 else (symbol - 261) // 4
            distance = code(5, at)
            if distance > 29:
                return False
            at += 5 + (0 if distance < 4 else distance // 2 - 1)
        else:
            at += 8 if c8 < 0xc0 else 9
    return True


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_second_walk_over_a_run(gpu, no_cpu_codec, seed):
    """A stored block's payload ends in what looks like stored headers, the last of which
    leads into the fixed run behind it: two walks cover the run's tiles."""
    import cuda_zlib
    text = workloads.text_like(3 << 20, np.random.default_rng(seed))
    c = zlib.compressobj(1, zlib.DEFLATED, -15, 8, zlib.Z_FIXED)
    run = c.compress(text) + c.flush()

    def header(n):
        return b"\0" + n.to_bytes(2, "little") + (n ^ 0xffff).to_bytes(2, "little")

    skip = next(n for n in range(1000 + 7000 * seed, 65000) if _fixed_tokens(run, 8 * n, 400))
    pad = np.random.default_rng(seed).integers(2, 256, 6000, dtype=np.uint8).tobytes()
    payload = pad + header(5) + b"abcde" + header(skip)
    body = header(len(payload)) + payload + run
    data = payload + text
    stream = b"\x78\x9c" + body + zlib.adler32(data).to_bytes(4, "big")
    assert zlib.decompress(stream) == data
    with no_cpu_codec:
        out, meta = cuda_zlib.decompress_zlib_checked(stream, len(data), 0)
    assert int(meta.cpu().numpy()[0]) == 0
    assert out.cpu().numpy().tobytes() == data


@pytest.mark.parametrize("length", [100, 200, 600, 5000, 60000, 66000, 200003])
@pytest.mark.parametrize("gap", [3000, 70000, 131072])
def test_fixed_blocks_between_dynamic_ones(gpu, length, gap):
    """Fixed blocks of literals shorter and longer than a group of tiles, each between
    dynamic blocks and one at the end of the body."""
    rng = np.random.default_rng(length + gap)

    def piece(data, strategy, flush=zlib.Z_FULL_FLUSH):
        c = zlib.compressobj(6, zlib.DEFLATED, -15, 8, strategy)
        return c.compress(data) + c.flush(flush)

    body = raw = b""
    for i in range(6):
        text = workloads.text_like(gap, rng)
        literals = rng.integers(48, 91, length, dtype=np.uint8).tobytes()
        fixed = piece(literals, zlib.Z_FIXED, zlib.Z_FINISH if i == 5 else zlib.Z_FULL_FLUSH)
        assert (fixed[0] >> 1) & 3 == 1
        body += piece(text, zlib.Z_DEFAULT_STRATEGY) + fixed
        raw += text + literals
    stream = b"\x78\x9c" + body + zlib.adler32(raw).to_bytes(4, "big")
    assert zlib.decompress(stream) == raw
    _check(gpu, stream, raw, length % 4)


@pytest.mark.parametrize("length", [3, 19, 58, 130, 257])
@pytest.mark.parametrize("distance_code", [29, 30, 31])
def test_run_that_ends_in_a_match(gpu, length, distance_code):
    """A run's last bits are a match, with a distance code that stands for nothing or cut
    short: the oracle's statuses at every cut."""
    import cuda_zlib
    raw = _content("text", 90000)
    w = dw.BitWriter()
    block = dw.Block(w, True).literals(raw)
    li = max(i for i, base in enumerate(dw.LENGTH_BASE) if base <= length)
    w.code(block.ll[257 + li]).put(length - dw.LENGTH_BASE[li], dw.LENGTH_EXTRA[li])
    w.code((distance_code, 5))
    body = w.getvalue()
    for cut in range(4):
        stream = dw.wrap(body[:len(body) - cut], raw)
        want, status = oracle.decompress(stream, len(raw) + length)
        out, meta = cuda_zlib.decompress_zlib_checked(stream, len(raw) + length, gpu)
        assert status and int(meta.cpu().numpy()[0]) == status
        assert out.cpu().numpy().tobytes() == want


def _final_block_look_alike():
    """The bits of a final dynamic block without output, made so that they also parse as
    tokens of the fixed codes: 105, and three zeros that end the last token."""
    lengths = [0 if s in (3, 5, 14) else 4 for s in range(19)]
    code = dw.canonical(lengths)
    w = dw.BitWriter().put(1, 1).put(2, 2).put(0, 5).put(0, 5).put(15, 4)
    for s in dw.CL_ORDER:
        w.put(lengths[s], 3)
    w.code(code[18]).put(138 - 11, 7).code(code[18]).put(118 - 11, 7)  # 256 lengths of zero
    w.code(code[1]).code(code[0]).put(0, 1)  # the end of block's code, no distances; that code
    assert w.nbits == 105
    return np.unpackbits(np.frombuffer(w.put(0, 3).getvalue(), np.uint8), bitorder="little")[:108]


@pytest.mark.parametrize("members", [False, True])
def test_final_block_look_alike_in_a_run(gpu, members):
    """A run whose tokens hold what reads as a final dynamic block, complete: the run does
    not end there.  (With the rest of it walked tile by tile, 200 times as long.)"""
    import cuda_zlib
    import torch
    rng = np.random.default_rng(23)
    first, rest = (rng.integers(0, 256, n, dtype=np.uint8).tobytes() for n in (40000, 1500000))

    def decode_ms(middle):
        body = np.concatenate((_literal_run(first)[:-7], middle, _literal_run(rest)[3:]))
        body = np.packbits(body.astype(np.uint8), bitorder="little").tobytes()
        raw = zlib.decompress(body, -15)
        assert len(raw) > 1540000
        src = torch.from_numpy(np.frombuffer(dw.wrap(body, raw), np.uint8).copy()).to(gpu)
        times = []
        for _ in range(6):
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            out, meta = cuda_zlib.decompress_zlib_checked(src, len(raw), gpu, members=members)
            stop.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(stop))
            assert int(meta.cpu().numpy()[0]) == 0 and out.cpu().numpy().tobytes() == raw
        return min(times)

    plain = decode_ms(_literal_run(b"middle")[3:-7])
    assert decode_ms(_final_block_look_alike()) < 3 * plain
