"""The quantiser's three-instruction quotient (``rtn_q8_kernel``; here in C with fmaf)
equals the IEEE division, where its first step is furthest off or the quotient is
hardest to round.

- significands of w at the top (first error next to 1.5 ulp) against every
  significand of s;
- quotients as near to the midpoint of two floats as there are: V 2^k = S M + j for
  small odd j and an odd 25-bit M;
- random pairs.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import cref

ONE = 1 << 23


def _equal(w: np.ndarray, s: np.ndarray) -> None:
    got = cref.rtn_quotients(w, s)
    want = w.astype(np.float32) / s.astype(np.float32)
    bad = np.flatnonzero(got.view(np.int32) != want.view(np.int32))
    assert bad.size == 0, (w[bad[:4]], s[bad[:4]])


@pytest.mark.parametrize("below", [1, 2, 3, 4])
def test_largest_significands_against_every_divisor(below):
    s = np.arange(ONE, 2 * ONE, dtype=np.int64).astype(np.float32)
    _equal(np.full(s.size, 2 * ONE - below, dtype=np.float32), s)


@pytest.mark.parametrize("k", [24, 25])
def test_quotients_beside_midpoints(k):
    rng = np.random.default_rng(k)
    S = (rng.integers(ONE, 2 * ONE, size=300000, dtype=np.uint64) | np.uint64(1))
    inv = S.copy()  # inverse of S modulo 2^25 (Newton, three bits to start with)
    for _ in range(5):
        inv = inv * (np.uint64(2) - S * inv)
    hard = 0
    for j in (1, -1, 3, -3, 5, -5, 7, -7):
        # S M + j = 0 modulo 2^k
        M = (inv * np.uint64((-j) % (1 << 64))) % np.uint64(1 << k)
        M = np.where(M < (1 << 24), M + np.uint64(1 << 24), M) if k == 24 else M
        V = (S * M + np.uint64(j % (1 << 64))) >> np.uint64(k)
        ok = (M >= (1 << 24)) & (M < (1 << 25)) & (M % 2 == 1) & (V >= ONE) & (V < 2 * ONE)
        hard += int(ok.sum())
        _equal(V[ok].astype(np.float32), S[ok].astype(np.float32))
    assert hard > 100000


def test_random_pairs():
    rng = np.random.default_rng(5)
    w = rng.integers(ONE, 2 * ONE, size=1 << 21).astype(np.float32) * np.float32(2.0 ** -30)
    s = rng.integers(ONE, 2 * ONE, size=1 << 21).astype(np.float32) * np.float32(2.0 ** -37)
    _equal(w * rng.choice(np.float32([1, -1]), size=w.size), s)
