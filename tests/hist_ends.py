"""Sizes of histogram inputs whose ragged ends take each of their paths: no end,
up to four rows of 256 elements, a whole guarded tile, and a second one for the
last of 4096 + 3 elements.  Shared by the emulation and the GPU tests."""

TILE = 4096


def sizes(tiles):
    """(n, words behind a 16-byte boundary) with `tiles` whole 4096-word tiles."""
    out = [(tiles * TILE, 0)]
    for off in (0, 1, 2, 3):
        head = (4 - off) % 4
        for rest in (1, 255, 1023, 1024, 1025, 4095, 4096, 4097, 4098):
            tail = rest - head
            if 0 <= tail < TILE and (tail or head):
                out.append((head + tiles * TILE + tail, off))
    return out
