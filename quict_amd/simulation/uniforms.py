"""Uniform draws from CPython's generator, many at a time."""
import random

import numpy as np


# draws a call of getrandbits (whose argument is a C int); bounds its integer too
BLOCK = 1 << 20


def uniforms(count: int) -> np.ndarray:
    """The next ``count`` values of ``random.random()``, and the same generator state
    after them.  A draw is (a * 2^26 + b) / 2^53 with a, b the top 27 and 26 bits of two
    consecutive 32-bit words, and ``getrandbits`` hands out the words in order, lowest
    first: one call a block instead of one per draw (20480 draws: 1.3 -> 0.4 ms)."""
    owner = getattr(random.random, "__self__", None)
    # (a replaced random.random, or another generator behind it, is asked draw by draw)
    if count <= 0 or type(owner) is not random.Random or getattr(random.getrandbits, "__self__", None) is not owner:
        return np.array([random.random() for _ in range(count)], dtype=np.float64)
    if count <= BLOCK:
        return _draw(count)
    return np.concatenate([_draw(min(BLOCK, count - i)) for i in range(0, count, BLOCK)])


def _draw(k: int) -> np.ndarray:
    w = np.frombuffer(random.getrandbits(64 * k).to_bytes(8 * k, "little"), dtype="<u8")
    return (((w & 0xFFFFFFE0) << 21) | (w >> 38)).astype(np.float64) * 2.0 ** -53
