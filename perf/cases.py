"""Timed cases of the zlib/DEFLATE codec: decode and encode through ``cuda_zlib``.

Every case is one call a program makes on buffers it already holds in device
memory.  Contents follow the generators of the benchmark's workloads, built on
the GPU from the seed so that inputs are quick to make:

text    Zipf(s=1.1) bytes over 64 symbols, 30 % of them overwritten by
        back-copies of 8-64 bytes from up to 32 KiB behind (logs, tables)
strain  float32 Gaussian noise plus a slow chirp (detector samples; hardly
        compressible, literal-only blocks)
random  uniform bytes (stored blocks)
runs    runs of one byte, 1 to 100000 long (zlib's run-length strategy)
mixed   segments of 1 MiB cycling random (stored), text (fixed Huffman), runs
        (run-length) and strain (level 9), as one stream

Streams to decode come from CPU zlib, as a user's files do.  Above 4 MiB a
stream is written in segments compressed side by side, each primed with the
32 KiB before it and ended by a sync flush: the way parallel compressors write
one stream.  ``writer`` "codec" streams are the framework's own encoder's.
"""

import math
import os
import sys
import zlib
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "cuda-zlib_amd"))

import cuda_zlib  # noqa: E402

KIB, MIB = 1 << 10, 1 << 20
SEGMENT = 4 * MIB
MIXED_SEGMENT = MIB
THREADS = 16

# zlib strategies by name.
STRATEGY = {"default": zlib.Z_DEFAULT_STRATEGY, "fixed": zlib.Z_FIXED, "rle": zlib.Z_RLE,
            "huffman": zlib.Z_HUFFMAN_ONLY}

# Compressed share of each content (zlib level 6, rounded), for work().
SHARE = {"text": 0.54, "strain": 0.926, "random": 1.0, "runs": 0.002, "mixed": 0.64}


def _decode(name, content, size, **options):
    case = {"name": name, "op": "decode", "content": content, "size": size, "format": "zlib",
            "level": 6, "strategy": "default", "writer": "zlib", "wait": False}
    case.update(options)
    return case


def _encode(name, content, size, **options):
    case = {"name": name, "op": "encode", "content": content, "size": size,
            "chunk_bytes": 32768, "independent": False}
    case.update(options)
    return case


def listed():
    return [
        # One small record (an RPC payload, a database cell), waited for.
        _decode("decode_text_4k", "text", 4 * KIB, wait=True),
        # One page or log block: two dynamic blocks.
        _decode("decode_text_64k", "text", 64 * KIB),
        # The headline stream: 64 MiB of float32 samples.
        _decode("decode_strain_64m", "strain", 64 * MIB),
        # A large log or table: most output bytes are back-references.
        _decode("decode_text_64m", "text", 64 * MIB),
        # The stress stream: every block type and strategy in turn.
        _decode("decode_mixed_128m", "mixed", 128 * MIB),
        # A fast writer's stream (fixed Huffman codes only), odd size.
        _decode("decode_fixed_15m", "text", 15999989, level=1, strategy="fixed"),
        # A gzip file of odd size at the strongest level (CRC-32 instead of Adler-32).
        _decode("decode_gzip_5m", "text", 5000011, format="gzip", level=9),
        # One small object compressed on its way out, odd size.
        _encode("encode_text_100k", "text", 100003),
        # The headline's other half.
        _encode("encode_strain_64m", "strain", 64 * MIB),
        # The large encode workload.
        _encode("encode_text_256m", "text", 256 * MIB),
        # Many small files (16 B to 64 KiB, some empty) in one call, each direction.
        {"name": "encode_batch_4096", "op": "encode_batch", "files": 4096, "largest": 64 * KIB,
         "chunk_bytes": 32768},
        {"name": "decode_batch_4096", "op": "decode_batch", "files": 4096, "largest": 64 * KIB,
         "level": 6},
    ]


def _log_size(rng, low, high):
    return int(math.exp(rng.uniform(math.log(low), math.log(high))))


def draw(rng):
    op = rng.choice(["decode"] * 4 + ["encode"] * 2 + ["encode_batch", "decode_batch"])
    if op == "decode":
        content = rng.choice(["text", "text", "strain", "random", "runs", "mixed"])
        strategy = rng.choice(["default"] * 4 + ["fixed", "rle", "huffman"])
        fmt = rng.choice(["zlib"] * 4 + ["gzip", "raw"])
        writer = rng.choice(["zlib"] * 3 + ["codec"]) if fmt == "zlib" else "zlib"
        high = 8 * MIB if strategy == "fixed" else 64 * MIB
        if content == "mixed":
            strategy, writer, size = "default", "zlib", _log_size(rng, 4 * MIB, 64 * MIB)
        else:
            size = _log_size(rng, 256, high)
        return {"op": op, "content": content, "size": size, "format": fmt,
                "level": rng.choice([1, 6, 6, 9]), "strategy": strategy, "writer": writer,
                "wait": rng.choice([False, True])}
    if op == "encode":
        return {"op": op, "content": rng.choice(["text", "text", "strain", "random", "runs"]),
                "size": _log_size(rng, 256, 128 * MIB),
                "chunk_bytes": rng.choice([4096, 16384, 32768, 32768, 32768, 65535]),
                "independent": rng.choice([False, False, True])}
    case = {"op": op, "files": _log_size(rng, 2, 4096), "largest": _log_size(rng, 256, 64 * KIB)}
    if op == "encode_batch":
        case["chunk_bytes"] = rng.choice([8192, 32768, 32768])
    else:
        case["level"] = rng.choice([1, 6, 9])
    return case


# ---- contents, on the GPU ---------------------------------------------------------

def _generator(seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed & 0x7fffffffffffffff)
    return generator


def _uniform(n, g):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _text(n, g):
    weights = torch.arange(1, 65, dtype=torch.float64) ** -1.1
    edges = (torch.cumsum(weights, 0) / weights.sum())[:63].float().cuda()
    data = torch.empty(n, dtype=torch.uint8, device="cuda")
    for start in range(0, n, 32 * MIB):
        part = data[start:start + 32 * MIB]
        draws = torch.rand(part.numel(), generator=g, device="cuda")
        part.copy_((torch.searchsorted(edges, draws, out_int32=True) + 0x20).to(torch.uint8))
    # Copies in passes: a pass's copies keep apart (one per cell) and read what
    # the passes before left, so that copies of copies arise as in real data.
    copies = int(0.3 * n / 36)
    passes = min(16, copies)
    for _ in range(passes):
        count = max(1, copies // passes)
        cell = n // count
        if cell < 130:
            break
        length = 8 + (_uniform(count, g) * 57).long()
        start = torch.arange(count, device="cuda") * cell
        position = start + 1 + (_uniform(count, g) * (cell - 65)).long()
        reach = torch.clamp(position, max=32768)
        distance = 1 + (_uniform(count, g) * reach).long().clamp_(max=reach - 1)
        owner = torch.repeat_interleave(torch.arange(count, device="cuda"), length)
        first = torch.cumsum(length, 0) - length
        step = torch.arange(owner.numel(), device="cuda") - first[owner]
        source = (position - distance)[owner] + step % distance[owner]
        data[position[owner] + step] = data[source]
    return data


def _strain(n, g):
    samples = (n + 3) // 4
    t = torch.arange(samples, dtype=torch.float64, device="cuda") / 4096.0
    duration = max(samples - 1, 1) / 4096.0
    phase = 2 * math.pi * (20.0 * t + 480.0 * t * t / (2 * duration))
    noise = torch.randn(samples, generator=g, device="cuda", dtype=torch.float64)
    x = (1e-21 * noise + 1e-22 * torch.sin(phase)).float()
    return x.view(torch.uint8)[:n].clone()


def _random(n, g):
    return torch.randint(0, 256, (n,), generator=g, device="cuda", dtype=torch.uint8)


def _runs(n, g):
    count = n // 20000 + 8
    length = 1 + (_uniform(count, g) * 100000).long()
    value = _random(count, g)
    data = torch.repeat_interleave(value, length)
    while data.numel() < n:
        data = torch.cat([data, data])
    return data[:n].clone()


CONTENT = {"text": _text, "strain": _strain, "random": _random, "runs": _runs}


def _mixed_kinds(n):
    """Content, level and strategy of each segment of a mixed stream."""
    cycle = [("random", 0, "default"), ("text", 1, "fixed"), ("runs", 6, "rle"),
             ("strain", 9, "default")]
    return [cycle[i % 4] for i in range(-(-n // MIXED_SEGMENT))]


def _content(kind, n, seed):
    g = _generator(seed)
    if kind != "mixed":
        return CONTENT[kind](n, g)
    kinds = _mixed_kinds(n)
    pools = {name: CONTENT[name](MIXED_SEGMENT * sum(k[0] == name for k in kinds), g)
             for name in ("random", "text", "runs", "strain") if any(k[0] == name for k in kinds)}
    taken = dict.fromkeys(pools, 0)
    parts = []
    for name, _, _ in kinds:
        parts.append(pools[name][taken[name]:taken[name] + MIXED_SEGMENT])
        taken[name] += MIXED_SEGMENT
    return torch.cat(parts)[:n].clone()


# ---- streams, by CPU zlib -----------------------------------------------------------

def _deflate(raw, case):
    """Raw DEFLATE of host bytes (segments side by side above SEGMENT bytes)."""
    if case["content"] == "mixed":
        size = MIXED_SEGMENT
        plan = [(level, strategy) for _, level, strategy in _mixed_kinds(len(raw))]
    else:
        size = SEGMENT
        plan = [(case["level"], case["strategy"])] * max(1, -(-len(raw) // size))
    view = memoryview(raw)

    def one(i):
        level, strategy = plan[i]
        history = view[max(0, i * size - 32768):i * size]
        extra = {"zdict": bytes(history)} if i else {}
        c = zlib.compressobj(level, zlib.DEFLATED, -15, 8, STRATEGY[strategy], **extra)
        body = c.compress(view[i * size:(i + 1) * size])
        return body + c.flush(zlib.Z_FINISH if i == len(plan) - 1 else zlib.Z_SYNC_FLUSH)

    if len(plan) == 1:
        return one(0)
    with ThreadPoolExecutor(THREADS) as pool:
        return b"".join(pool.map(one, range(len(plan))))


def _stream(raw, case):
    body = _deflate(raw, case)
    if case["format"] == "zlib":
        return b"\x78\x9c" + body + zlib.adler32(raw).to_bytes(4, "big")
    if case["format"] == "gzip":
        header = b"\x1f\x8b\x08\x08" + b"\0" * 4 + b"\x00\x03" + b"data.txt\0"
        return header + body + zlib.crc32(raw).to_bytes(4, "little") \
            + (len(raw) & 0xffffffff).to_bytes(4, "little")
    return body


def _to_device(data):
    return torch.from_numpy(np.frombuffer(data, dtype=np.uint8).copy()).cuda()


def _batch(case, seed):
    """Files of a batch: log-uniform sizes (the case's own, whatever the seed), one in 64
    empty, text / noise / random in turn."""
    n = case["files"]
    rng = np.random.default_rng([n, case["largest"]])
    sizes = np.floor(np.exp(rng.uniform(np.log(16), np.log(case["largest"]), n))).astype(np.int64)
    sizes[rng.choice(n, n // 64, replace=False)] = 0
    kinds = ("text", "strain", "random")
    pools = [_content(kind, max(4096, int(sizes[i::3].sum())), seed + i)
             for i, kind in enumerate(kinds)]
    at = [0, 0, 0]
    files = []
    for i, size in enumerate(sizes.tolist()):
        files.append(pools[i % 3][at[i % 3]:at[i % 3] + size])
        at[i % 3] += size
    return torch.cat(files), tuple(sizes.tolist())


# ---- the interface --------------------------------------------------------------------

def prepare(case, seed):
    state = {"case": case}
    if case["op"] == "encode":
        state["data"] = _content(case["content"], case["size"], seed)
    elif case["op"] == "decode":
        raw = _content(case["content"], case["size"], seed)
        if case["writer"] == "codec":
            state["payload"] = cuda_zlib.compress_zlib(raw)
        else:
            state["payload"] = _to_device(_stream(raw.cpu().numpy().tobytes(), case))
    else:
        state["data"], state["sizes"] = _batch(case, seed)
        if case["op"] == "decode_batch":
            host = memoryview(state.pop("data").cpu().numpy().tobytes())
            ends = np.cumsum(state["sizes"]).tolist()
            pieces = [host[end - size:end] for end, size in zip(ends, state["sizes"])]
            with ThreadPoolExecutor(THREADS) as pool:
                streams = list(pool.map(lambda p: zlib.compress(p, case["level"]), pieces))
            state["payload"] = _to_device(b"".join(streams))
            state["stream_sizes"] = tuple(len(s) for s in streams)
    return state


def run(state):
    case = state["case"]
    if case["op"] == "encode":
        return cuda_zlib.compress_zlib_padded(state["data"], chunk_bytes=case["chunk_bytes"],
                                              independent_chunks=case["independent"])
    if case["op"] == "encode_batch":
        return cuda_zlib.compress_zlib_batch_padded(state["data"], state["sizes"],
                                                    chunk_bytes=case["chunk_bytes"])
    if case["op"] == "decode_batch":
        return cuda_zlib.decompress_zlib_batch_checked(state["payload"], state["stream_sizes"],
                                                       state["sizes"])
    wait = "" if case["wait"] else "_checked"
    name = {"zlib": "zlib", "gzip": "gzip", "raw": "deflate_raw"}[case["format"]]
    return getattr(cuda_zlib, "decompress_" + name + wait)(state["payload"], case["size"])


def work(case):
    """Input and output once each; no floating-point operations."""
    if case["op"].endswith("batch"):
        # Mean of a log-uniform size; a third each of text, noise and random bytes.
        span = math.log(case["largest"] / 16)
        size = case["files"] * (case["largest"] - 16) / span
        share = (0.62 + 0.95 + 1.0) / 3
    else:
        size, share = case["size"], SHARE[case["content"]]
    return {"bytes": size * (2 if case["op"].startswith("encode") else 1 + share), "flops": 0}


def tolerance(case):
    # Bytes and statuses: decoded output is the stream's, encoded streams are deterministic.
    return "exact"
