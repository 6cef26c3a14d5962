"""Buffer sizes the autograd wrappers give a forward, with the library
replaced by its counting rules: scenes that alternate must fit their pair
stores and slots once each has been seen, counts must find the right key, and
every overflow must end in a forward that fits.
"""
import contextlib

import pytest
import torch

from partgs_amd import _lib
from partgs_amd import rasterizer as R


class _Counter:
    """The library's side of the sizes: posts each forward's counts, `lag` forwards late."""

    def __init__(self, monkeypatch, lag):
        self.posted, self.lag, self.misses, self.runs = [], lag, 0, 0
        for name in ("_capacity_hint", "_pair_hint", "_slot_hint"):
            monkeypatch.setattr(R, name, {})
        monkeypatch.setattr(R._recent, "forwards", R.collections.deque(maxlen=8), raising=False)
        monkeypatch.setattr(torch.cuda, "device", lambda _: contextlib.nullcontext())
        monkeypatch.setattr(_lib, "pair_count", lambda: self._seen(1))
        monkeypatch.setattr(_lib, "slot_count", lambda: self._seen(2))

    def _seen(self, k):
        done = self.posted[:len(self.posted) - self.lag]
        return (done[-1][k], done[-1][0]) if done else None

    def forward(self, n, pairs, slots):
        def run(cap, pcap, scap):
            self.runs += 1
            if 0 < cap < n:
                self.posted.append((n, 0, slots))
                raise _lib.CapacityError(n, cap, slots=False)
            if cap > 0 and 0 < scap < slots:
                self.posted.append((n, 0, slots))
                raise _lib.CapacityError(n, cap, slots=True)
            self.misses += pairs > (pcap if cap > 0 else 8 * n)
            self.posted.append((n, pairs, slots))
            return (n,)
        return run


A, B = (50_000, 150_000, 60_000), (48_000, 420_000, 170_000)  # instances, pairs, slots


@pytest.mark.parametrize("lag", [0, 1])
@pytest.mark.parametrize("keys", [("k",), ("k", "k2")])
def test_alternating_scenes_fit(monkeypatch, lag, keys):
    c = _Counter(monkeypatch, lag)
    for i in range(600):
        if i == 8:
            c.misses = c.runs = 0
        R._forward_sized((0, keys[i % len(keys)]), False, c.forward(*(A, B)[i % 2]))
    assert c.misses == 0 and c.runs == 592


@pytest.mark.parametrize("lag", [0, 1])
def test_outgrown_and_shrunk(monkeypatch, lag):
    c = _Counter(monkeypatch, lag)
    key = (0, "k")
    for _ in range(3):
        R._forward_sized(key, False, c.forward(*A))
    (n,), (cap, _, scap) = R._forward_sized(key, False, c.forward(10 * A[0], 10 * A[1], 10 * A[2]))
    assert n == 500_000 and cap >= n and scap == 0  # outgrew both; every (instance, quadrant) once
    R._forward_sized(key, False, c.forward(2000, 5000, 3000))
    assert R._capacity_hint[key] == R._grown(2000)
    for _ in range(4):
        _, (cap, pcap, scap) = R._forward_sized(key, False, c.forward(2000, 5000, 3000))
    assert cap == R._grown(2000) and pcap <= 8 * cap and scap <= R._grown(3000)
    _, sizes = R._forward_sized(key, True, c.forward(*A))  # debug: exact sizes
    assert sizes == (0, 0, 0)
