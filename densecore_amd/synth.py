"""Deterministic synthetic inputs for the benchmark's configurations.

SplitMix64 (Steele, Lea, Flood 2014) feeds Box-Muller pairs; everything is
vectorised numpy uint64/float64 arithmetic, so a seed gives the same float32
bytes on every x86-64 host running this image. Digests of the generated bytes
are reported with every benchmark result.
"""
import hashlib

import numpy as np

_GAMMA = np.uint64(0x9E3779B97F4A7C15)
_M1 = np.uint64(0xBF58476D1CE4E5B9)
_M2 = np.uint64(0x94D049BB133111EB)


def splitmix64(seed, count):
    """The first `count` outputs of SplitMix64 started at `seed`."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + _GAMMA * np.arange(1, count + 1, dtype=np.uint64)
        z = (z ^ (z >> np.uint64(30))) * _M1
        z = (z ^ (z >> np.uint64(27))) * _M2
        return z ^ (z >> np.uint64(31))


def _splitmix64_range(seed, start, count):
    """Outputs start+1 .. start+count of SplitMix64 started at `seed` (1-based, as splitmix64)."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + _GAMMA * np.arange(start + 1, start + count + 1, dtype=np.uint64)
        z = (z ^ (z >> np.uint64(30))) * _M1
        z = (z ^ (z >> np.uint64(27))) * _M2
        return z ^ (z >> np.uint64(31))


def normal(n, seed, mean=0.0, std=1.0):
    """n float32 samples of N(mean, std^2) via Box-Muller on SplitMix64 (computed in chunks of
    2^20 pairs so the temporaries stay in cache; the values do not depend on the chunking)."""
    pairs = (n + 1) // 2
    out = np.empty(2 * pairs, dtype=np.float32)
    chunk = 1 << 20
    for p0 in range(0, pairs, chunk):
        cnt = min(chunk, pairs - p0)
        z = _splitmix64_range(seed, 2 * p0, 2 * cnt)
        u = ((z >> np.uint64(11)).astype(np.float64) + 1.0) * (1.0 / 9007199254740992.0)
        u1, u2 = u[0::2], u[1::2]
        r = np.sqrt(-2.0 * np.log(u1))
        t = 2.0 * np.pi * u2
        v = np.empty(2 * cnt, dtype=np.float64)
        v[0::2] = r * np.cos(t)
        v[1::2] = r * np.sin(t)
        out[2 * p0:2 * (p0 + cnt)] = (mean + std * v).astype(np.float32)
    return out[:n]


def set_outliers(x, count, value, seed):
    """Set `count` distinct positions of x (seeded shuffle) to +-value in place."""
    n = x.size
    z = splitmix64(seed ^ 0x5DEECE66D, 2 * n)
    order = np.argsort(z[:n], kind="stable")[:count]
    signs = np.where((z[n:n + count] & np.uint64(1)) == 1, -1.0, 1.0).astype(np.float32)
    flat = x.reshape(-1)
    flat[order] = signs * np.float32(value)
    return x


def digest(a):
    return hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()[:16]
