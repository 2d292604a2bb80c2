"""The plan of bwd.hip's dK + dV units restated (plan_key_units(), key_units_before(), key_unit()): which levels
are halved, whether the units are dealt out, and which piece of work a unit is."""
import struct

import numpy as np

FULL_TILE, HALF_TILE, UNIT_FIXED = 175, 100, 700
HALVED_TILES, HALVED_IDLE = 7, 160
DEALT_ROUNDS, MAX_BATCH, MAX_LEVELS = 4, 64, 512
f32 = np.float32


class Plan:
    """lens: tokens of the sequences; workers: workgroups that run at once."""

    def __init__(self, lens, heads_q, heads_kv, causal=True, workers=256):
        self.lens, self.hkv, self.causal, self.workers = list(lens), heads_kv, causal, workers
        self.tiles = [-(-n // 128) for n in lens]
        self.levels = max(self.tiles, default=0)
        self.top = -(-self.levels // 64) * 64
        reach = [sum(a > t for a in self.tiles) for t in range(self.top + 1)]
        self.at_or_above = [sum(reach[t:]) for t in range(self.top + 1)]
        self.weight = [sum((s + 1) * reach[s] for s in range(t, self.top + 1)) for t in range(self.top + 1)]
        self.unit = 2 * (heads_q // heads_kv)   # tiles of 64 queries of a level-0 item
        self.all = self.at_or_above[0]
        self.split_from = self._choose() if causal else 0
        self.dealt = self._worth()

    def _worth(self):
        items = self.all * self.hkv
        dealt = items < DEALT_ROUNDS * self.workers if self.causal else 2 * items <= self.workers
        if items <= self.workers:
            longest = f32(FULL_TILE * self.unit * self.levels + UNIT_FIXED)
            mean = f32(self.hkv) * (f32(FULL_TILE * self.unit) * f32(self.weight[0]) + f32(UNIT_FIXED) * f32(self.all)) / f32(self.workers)
            dealt = dealt and self.unit * self.levels >= HALVED_TILES and max(self.lens, default=0) > 64
            if self.causal:
                dealt = dealt and mean + f32(HALVED_IDLE) <= f32(0.6) * longest
        return bool(dealt)

    def estimate(self, t):
        """What the choice minimises, in hundredths of a microsecond (fp32, as on the device)."""
        a, w = f32(self.at_or_above[t]), f32(self.weight[t])
        unit, workers, hkv = f32(self.unit), f32(self.workers), f32(self.hkv)
        whole = f32(self.all) - a
        units = whole + 2 * a
        total = hkv * (2 * (HALF_TILE * unit * w + UNIT_FIXED * a) + FULL_TILE * unit * (f32(self.weight[0]) - w) + UNIT_FIXED * whole)
        longest = FULL_TILE * unit * f32(t) + UNIT_FIXED if t > 0 else f32(0)
        if t < self.levels:
            longest = max(longest, HALF_TILE * unit * f32(self.levels) + UNIT_FIXED)
        est = total / workers
        if units * hkv > workers:
            est += f32(0.25) * total / (units * hkv)
        return f32(max(est, longest))

    def _choose(self):
        key = [(struct.unpack("I", struct.pack("f", self.estimate(t)))[0] & ~1023) | (1023 - t) for t in range(self.levels + 1)]
        return 1023 - (min(key) & 1023)

    def units(self):
        """How many there are: (sequence, tile or half, kv-head)."""
        return self.hkv * (self.all + self.at_or_above[self.split_from])

    def _before(self, t):
        T, n = self.split_from, self.at_or_above
        if t >= T:   # halves of level t
            return 2 * n[t + 1] + n[min(4 * (t + 1) // 7, T)] - n[T]
        return n[t + 1] - n[T] + 2 * n[min(max((7 * (t + 1) + 3) // 4 - 1, T), self.top)]

    def unit_at(self, u):
        """(sequence, kv-head, tile of 128 keys, half or -1) of unit u, None behind the last."""
        pair = u // self.hkv
        for t in range(self.top):
            n = pair - self._before(t)
            if 0 <= n < (2 if t >= self.split_from else 1) * (self.at_or_above[t] - self.at_or_above[t + 1]):
                half = -1
                if t >= self.split_from:
                    n, half = n >> 1, n & 1
                seq = [b for b, a in enumerate(self.tiles) if a > t][n]
                return seq, u - pair * self.hkv, self.tiles[seq] - 1 - t, half
        return None

    def cost(self, unit):
        seq, _, tile, half = unit
        return (FULL_TILE if half < 0 else HALF_TILE) * self.unit * (self.tiles[seq] - tile)
