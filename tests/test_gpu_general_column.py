"""The one-workgroup-per-column route of the general speculative acceptance, taken by batches of at least 64
columns: every sequence's outputs equal the oracle's, and those of the same sequence sent alone (the tile
route), bit for bit: both are integer arithmetic over the same weights, so no tolerance applies."""
import numpy as np
import pytest

from ninfer_amd import synthetic as syn

import gpu_runner
from test_gpu_general import _case, _check

pytestmark = pytest.mark.gpu

MASK = 0xFF80  # BF16 -inf


def _columns(kind, t, d):
    rng = np.random.default_rng(5)
    for x in (t, d):
        if kind == "masked":  # most tokens share one value, counted apart
            x[rng.random(x.shape) < 0.8] = MASK
        elif kind == "two_values":  # each more than a histogram counter holds
            x[:] = np.where(rng.random(x.shape) < 0.5, 0x3F80, 0xBF80)
        elif kind == "signed_zeros":  # -0 and +0 are one value
            x[:] = np.where(rng.random(x.shape) < 0.5, 0x8000, np.where(rng.random(x.shape) < 0.5, 0, 0xBF80))
        elif kind == "negative":
            x |= 0x8000
        elif kind == "integers":  # a dozen frequent values, counted apart
            x[:] = syn.f32_to_bf16_bits(np.rint(syn.bf16_bits_to_f32(x)))
        elif kind == "masked_integers":
            x[:] = np.where(rng.random(x.shape) < 0.5, MASK, syn.f32_to_bf16_bits(np.rint(syn.bf16_bits_to_f32(x))))
        elif kind == "fifty_values":  # more frequent values than are counted apart, sharing hash buckets or not
            vals = rng.permutation(np.r_[0x3C00:0x4080, 0xBC00:0xC080])[:50].astype(np.uint16)
            x[:] = vals[rng.integers(0, 50, x.shape)]
        elif kind == "wraps":  # a value that overflows its counter and is at none of the 1,024 sampled places
            rows, bits = x.shape[-1], 0x4049 if x is t else 0xBFC1
            common = rng.random(x.shape, dtype=np.float32) < 0.1
            common[..., np.arange(1024) * rows // 1024] = False
            x[common] = bits
        elif kind == "constant":
            x[:] = 0x3E4D
        elif kind == "nan":
            x[..., 3::97] = 0x7FC0
            x[..., 5::97] = 0xFFC1


@pytest.mark.parametrize("kind,B,K,rows,temp,top_p", [
    ("normal", 13, 2, 7, 0.7, 0.9),           # fewer tokens than a load
    ("normal", 22, 1, 1023, 0.7, 0.95),       # odd rows: columns at any alignment
    ("normal", 10, 3, 65536, 0.7, 0.95),      # one batch exactly
    ("normal", 10, 3, 65544, 1.3, 0.99),      # and 8 tokens more
    ("normal", 6, 5, 131077, 0.5, 1.0),       # no nucleus
    ("normal", 17, 15, 4104, 0.7, 0.5),       # 527 columns: more than compute units
    ("masked", 10, 3, 70000, 0.7, 0.95),
    ("two_values", 10, 3, 150000, 1.0, 0.6),
    ("signed_zeros", 10, 3, 20000, 1.0, 0.6),
    ("negative", 10, 3, 20000, 0.7, 0.95),
    ("integers", 10, 3, 70001, 0.7, 0.95),
    ("integers", 10, 3, 300, 0.7, 0.8),       # fewer tokens than the sample takes
    ("masked_integers", 10, 3, 150000, 0.7, 0.9),
    ("fifty_values", 10, 3, 100000, 1.0, 0.4),
    ("constant", 10, 3, 65552, 0.7, 0.5),
    ("wraps", 22, 1, 700001, 0.7, 0.9),
])
def test_column_route(gpu, oracle, kind, B, K, rows, temp, top_p):
    t, d, dr, ua, ur = _case(60 + rows % 17, B, K, rows)
    _columns(kind, t, d)
    lengths = np.arange(B, dtype=np.int32) * 10 + 3
    got = _check(oracle, t, d, dr, ua, ur, lengths, rows, temp, top_p)
    _compare_alone(got, t, d, dr, ua, ur, lengths, rows, temp, top_p)


def test_column_route_nan_tokens(gpu):
    """NaN is outside the oracle's domain; the tile route leaves it out of the maximum and weighs it as any token."""
    B, K, rows = 10, 3, 9001
    t, d, dr, ua, ur = _case(9, B, K, rows)
    _columns("nan", t, d)
    lengths = np.full(B, 5, np.int32)
    got = gpu_runner.run_general(t, d, dr, ua, ur, lengths, np.zeros((B, 4 + K), np.int64), rows, 0.7, 0.95)
    _compare_alone(got, t, d, dr, ua, ur, lengths, rows, 0.7, 0.95)


@pytest.mark.parametrize("kind", ["integers", "masked_integers", "two_values", "constant"])
def test_few_distinct_values_cost(gpu, kind):
    """Tokens that share a value may not serialize: the call takes at most 1.7 times what it takes on normal
    logits (MI355X: integers 71 us, two values 71, a constant 58, normal logits 62; with atomics that conflict 165,
    463 and, if masked too, 520)."""
    B, K, rows = 10, 3, 248320
    t, d, dr, ua, ur = _case(3, B, K, rows)
    lengths = np.zeros(B, np.int32)
    stats = np.zeros((B, 4 + K), np.int64)
    normal = gpu_runner.run_general(t, d, dr, ua, ur, lengths, stats, rows, 0.7, 0.95, timed=True)
    _columns(kind, t, d)
    few = gpu_runner.run_general(t, d, dr, ua, ur, lengths, stats, rows, 0.7, 0.95, timed=True)
    print(f"{kind}: {few:.1f} us, normal logits {normal:.1f} us")
    assert few <= 1.7 * normal


def _compare_alone(got, t, d, dr, ua, ur, lengths, rows, temp, top_p):
    K = dr.shape[1]
    for b in range(0, len(lengths), 3):
        s = slice(b, b + 1)
        one = gpu_runner.run_general(t[s], d[s], dr[s], ua[s], ur[s], lengths[s], np.zeros((1, 4 + K), np.int64), rows, temp, top_p)
        for k, v in one.items():
            assert np.array_equal(np.asarray(v)[0], np.asarray(got[k])[b]), (b, k)
