"""How a decode launch is split, restated in Python: the host's part against the
library's workspace size, the kernels' part (in 32-bit floats) for what the host
sized: every token of every sequence in exactly one split, no split past the
workspace's, no unit past the grid, no split wider than the kernel's table."""
import math
import random

import numpy as np
import pytest

from lightserve_amd import _lib

f32 = np.float32
SLOTS, SCAN_MAX = 512, 256


def _align(n):
    return (n + 255) // 256 * 256


class Split:
    def __init__(self, batch, hq, hkv, dim, block, maxs):
        g, units = hq // hkv, max(1, batch * hkv)
        wide, mfma, many = dim > 64, block >= 16 and g not in (1, 2, 4, 8), units >= 64
        self.unit = 64 if wide and g >= 4 and not mfma else 128
        self.hkv, self.maxs = hkv, maxs
        self.cap = min((SLOTS - 1) * block // self.unit * self.unit, 1 << 24)
        self.compact, self.scale, self.fill, self.share = batch <= SCAN_MAX, 0.0, 0.0, 0.0
        self.lo, self.hi = self.unit, 1024
        if mfma and units > 128:
            self.whole = self.lo = self.hi = 4096 if wide else 1024
        elif mfma:
            self.whole, self.scale, self.fill = (1024 if wide else 512) if many else 384, 1.8, 1.0 / 192
        elif units >= 4096:
            self.whole = self.lo = self.hi = self.cap
        elif not self.compact:
            n = max(1, min((4096 + units - 1) // units, (maxs + 511) // 512))
            self.whole, self.lo = 512, max(512, -(-maxs // n))
            self.hi = self.lo
        else:
            if wide:
                self.whole = {1: 384, 2: 384, 4: 256, 8: 128}[g] if not many else {1: 512, 2: 512, 4: 512, 8: 256}[g]
            else:
                self.whole = 512 if g <= 4 or many else 256
            if units >= 512 or (units >= 256 and g == 1):
                self.whole = 1024
            self.hi = 512 if g == 8 else 1024
            self.scale, self.fill, self.share = 1.4, 1.0 / 256, 1.0 / 4096
        self.whole = min(self.whole, self.cap)
        self.splits, self.units = 1, 0
        if maxs > self.whole:
            most = min(maxs, 1 << 20) * hkv
            self.splits = math.ceil(maxs / (0.999 * self.size(most)))
            if self.compact:
                self.units = min(math.ceil(batch * maxs / (0.999 * self.size(most * max(1, batch)))) + batch,
                                 batch * self.splits)
        self.compact &= self.splits > 1
        rows = batch * hq * self.splits
        self.bytes = _align(rows * (64 if dim <= 64 else 128) * 4) + _align(rows * 4) + _align(batch * 4) if self.splits > 1 else 0

    def size(self, work):
        fit = min(self.hi, max(self.lo, min(self.scale * math.sqrt(work), work * self.fill)))
        return min(self.cap, max(fit, work * self.share))

    def device_size(self, lens):
        size = f32(self.lo)
        if self.compact:
            work = f32(16) * f32(self.hkv) * f32(sum((min(n, 1 << 20) + 15) >> 4 for n in lens))
            fit = min(f32(self.hi), max(f32(self.lo), min(f32(self.scale) * np.sqrt(work), work * f32(self.fill))))
            size = max(fit, work * f32(self.share))
            if len(lens) == 1 and f32(256) * size < work <= f32(512) * size:
                size = work / f32(256)
        return (int(math.ceil(min(size, f32(self.cap)))) + self.unit - 1) // self.unit * self.unit

    def tokens(self, seq, size):
        n = max(1, min((seq + size - 1) // size, self.splits))
        return max(1, -(-seq // (n * self.unit))) * self.unit


def _check(batch, hq, hkv, dim, block, maxs, lens):
    s = Split(batch, hq, hkv, dim, block, maxs)
    args = _lib.DecodeArgs(batch=batch, heads_q=hq, heads_kv=hkv, head_dim=dim, block_size=block, max_seq_len=maxs)
    assert _lib.decode_workspace_size(args) == s.bytes
    if s.splits == 1:
        assert maxs <= s.cap
        return
    size, total = s.device_size(lens), 0
    assert size % s.unit == 0 and 0 < size <= s.cap
    for n in lens:
        st = s.tokens(n, size)
        have = 1 if n <= st else -(-n // st)
        assert st <= s.cap and have <= s.splits and have * st >= n and (have - 1) * st < max(n, 1)
        total += have
    if s.compact:
        assert total <= s.units


@pytest.mark.parametrize("seed", range(40))
def test_decode_split_covers_every_token(built_library, seed):
    r = random.Random(seed)
    for _ in range(60):
        hkv, g, dim = r.choice([1, 2, 3, 4, 8, 12, 16, 32]), r.choice([1, 2, 4, 8, 3, 7, 16]), r.choice([32, 64, 72, 128])
        block = r.choice([16, 64, 256]) if g not in (1, 2, 4, 8) else r.choice([1, 4, 16, 64, 256, 4096])
        batch = int(2 ** r.uniform(0, 9.5))
        maxs = int(2 ** r.uniform(0, r.choice([10, 14, 21])))
        lens = [r.choice([maxs, 0, r.randint(0, maxs), min(maxs, r.randint(1, 600))]) for _ in range(batch)]
        for lens in (lens, [maxs] * batch, [0] * (batch - 1) + [maxs]):
            _check(batch, g * hkv, hkv, dim, block, maxs, lens)


def test_decode_split_measured_points(built_library):
    """Launches on either side of the rule's lines: whole where a split lost."""
    for batch, hq, hkv, dim, maxs, split in ((1, 32, 8, 64, 200, False), (4, 32, 8, 128, 200, False), (1, 32, 32, 64, 500, False),
                                             (16, 32, 8, 64, 500, False), (55, 28, 4, 128, 1000, False), (1, 16, 2, 128, 200, True),
                                             (1, 32, 8, 128, 1000, True), (16, 28, 4, 128, 4000, True)):
        args = _lib.DecodeArgs(batch=batch, heads_q=hq, heads_kv=hkv, head_dim=dim, block_size=16, max_seq_len=maxs)
        assert (_lib.decode_workspace_size(args) > 0) == split, (batch, hq, hkv, dim, maxs)
