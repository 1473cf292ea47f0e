"""gzip CRC-32 from 16 KiB tiles: sizes around tile edges and around 256 tiles,
where a thread's run of tiles gets longer."""

import zlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE = 16384


@pytest.mark.parametrize("size", [256, 259, TILE - 1, TILE, TILE + 1, 3 * TILE + 5, 255 * TILE + 9,
                                  256 * TILE, 256 * TILE + 1, 700 * TILE + 77])
def test_crc_tiles(gpu, size):
    import cuda_zlib
    rng = np.random.default_rng(size)
    raw = rng.integers(0, 256, size, dtype=np.uint8).tobytes()
    c = zlib.compressobj(1, zlib.DEFLATED, -15)
    body = c.compress(raw) + c.flush()
    head = b"\x1f\x8b\x08\0\0\0\0\0\0\x03"
    crc, isize = zlib.crc32(raw), (size & 0xffffffff).to_bytes(4, "little")
    for wanted, status in ((crc, 0), (crc ^ 1, 24), (crc ^ 0x80000000, 24)):
        stream = head + body + wanted.to_bytes(4, "little") + isize
        out, meta = cuda_zlib.decompress_gzip_checked(stream, size, gpu)
        assert int(meta.cpu().numpy()[0]) == status
        if not status:
            assert out.cpu().numpy().tobytes() == raw
