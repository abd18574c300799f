"""The one-workgroup-per-column route of the general speculative acceptance, taken by batches of at least 64
columns: every sequence's outputs equal the oracle's, and those of the same sequence sent alone (the tile
route), bit for bit: both are integer arithmetic over the same weights, so no tolerance applies."""
import numpy as np
import pytest

import gpu_runner
from test_gpu_general import _case, _check

pytestmark = pytest.mark.gpu

MASK = 0xFF80  # BF16 -inf


def _columns(kind, t, d):
    rng = np.random.default_rng(5)
    for x in (t, d):
        if kind == "masked":  # most tokens share one value, counted outside the histogram
            x[rng.random(x.shape) < 0.8] = MASK
        elif kind == "two_values":  # one is taken as the common value, the other's counter wraps
            x[:] = np.where(rng.random(x.shape) < 0.5, 0x3F80, 0xBF80)
        elif kind == "signed_zeros":  # -0 and +0 are one value
            x[:] = np.where(rng.random(x.shape) < 0.5, 0x8000, np.where(rng.random(x.shape) < 0.5, 0, 0xBF80))
        elif kind == "negative":
            x |= 0x8000
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


def _compare_alone(got, t, d, dr, ua, ur, lengths, rows, temp, top_p):
    K = dr.shape[1]
    for b in range(0, len(lengths), 3):
        s = slice(b, b + 1)
        one = gpu_runner.run_general(t[s], d[s], dr[s], ua[s], ur[s], lengths[s], np.zeros((1, 4 + K), np.int64), rows, temp, top_p)
        for k, v in one.items():
            assert np.array_equal(np.asarray(v)[0], np.asarray(got[k])[b]), (b, k)
