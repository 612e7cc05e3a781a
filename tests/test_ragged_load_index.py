"""CPU model of the matrix-core kernels' loads of uint8 rows of any width and
alignment (csrc/fa_ssim_mfma.hip, RAG): the three aligned dwords a lane reads,
the byte it starts at in them, and the row pitch of padded pyramid levels.

Every dword read for a row of the image must hold a byte of that plane (such a
dword is mapped whatever follows the plane in memory), and the realigned bytes
must be the lane's samples wherever they lie inside the row.
"""

from __future__ import annotations

import numpy as np
import pytest

MT = 16


def _place(m, pitch, W, n, c0, g):
    """(offset of the dwords from the aligned base, start byte in them)."""
    c = min(c0 + 8 * g, W - 1)
    row = m + n * pitch
    end = ((row + W - 1) & ~3) - 8
    at = min((row + c) & ~3, end)
    return at, row + c - at


def _realign(d, t, any_):
    """The kernel's selects and v_alignbyte on three dwords (as 12 bytes)."""
    d = [d[0:4], d[4:8], d[8:12]]
    if any_:
        s1, s2 = t >= 4, t >= 8
        d[0] = d[2] if s2 else d[1] if s1 else d[0]
        d[1] = d[2] if s1 else d[1]
    k = t & 3
    lo = np.concatenate([d[0], d[1]])[k:k + 4]
    hi = np.concatenate([d[1], d[2]])[k:k + 4]
    return np.concatenate([lo, hi])


@pytest.mark.parametrize("W", [16, 17, 18, 19, 23, 31, 33, 47, 63, 65, 107, 131])
@pytest.mark.parametrize("base", [0, 1, 2, 3])
@pytest.mark.parametrize("extra", [0, 1, 5, 8])
def test_lane_bytes_and_bounds(W, base, extra):
    pitch, H, K = W + extra, 37, 11
    rng = np.random.default_rng(W * 100 + base * 10 + extra)
    ext = (H - 1) * pitch + W
    mem = rng.integers(0, 256, base + ext + 64, dtype=np.uint8)
    first = base & ~3
    last_dword = (base + ext - 1) & ~3          # the dword of the plane's last byte
    m = base & 3
    Wout = W - K + 1
    if Wout < 1:
        Wout = 1
    for r0 in (0, 16, 32):
        bx = r0 * pitch
        limit = ((m + ext + 3) & ~3) - bx       # the buffer's range
        for c0 in range(0, Wout, MT):
            any_ = c0 + 2 * MT + 4 > W
            for n in range(MT):
                for g in range(4):
                    at, t = _place(m, pitch, W, n, c0, g)
                    assert at >= 0 and at % 4 == 0 and 0 <= t < 12
                    assert any_ or t < 4
                    if r0 + n >= H:             # past the image: any value serves
                        continue
                    assert at + 12 <= limit
                    a = first + bx + at
                    assert first <= a and a + 8 <= last_dword
                    got = _realign(mem[a:a + 12], t, any_)
                    c = min(c0 + 8 * g, W - 1)
                    k = min(8, W - c)
                    want = mem[base + (r0 + n) * pitch + c:][:k]
                    assert np.array_equal(got[:k], want), (r0, c0, n, g)


def _pitch(w):
    return (w + 7) // 8 * 8


@pytest.mark.parametrize("K", [3, 11])
def test_first_level_padding_is_written(K):
    """The float16 level's reader takes whole padded rows, so every padded
    column must be stored by some wave: even waves store 16 columns from half
    their first, the row's last active wave its 16 whatever its index."""
    for W in range(2 * K + 16, 420):
        Wout, lp = W - K + 1, _pitch(W // 2)
        seen = np.zeros(lp, bool)
        for w in range((Wout + MT - 1) // MT):
            c0 = w * MT
            if (w & 1) == 0 or c0 + MT >= Wout:
                seen[c0 // 2:min(c0 // 2 + 16, lp)] = True
        assert seen.all(), (W, lp)


def test_deep_level_columns_are_written():
    """Columns of the two levels below the float16 level's next one: lane
    (g, n) stores column (c0 / 2 + n) >> (d + 1) where it is the first of its
    group."""
    K = 11
    for W in range(4 * K, 420):
        Wout = W - K + 1
        for d in (0, 1):
            Wl = W >> (d + 2)
            seen = np.zeros(Wl, bool)
            for w in range((Wout + MT - 1) // MT):
                c0 = w * MT
                if (w & 1) and c0 + MT < Wout:
                    continue
                for n in range(0, 16, 2 << d):
                    col = (c0 // 2 + n) >> (d + 1)
                    if col < Wl:
                        seen[col] = True
            assert seen.all(), (W, d)
