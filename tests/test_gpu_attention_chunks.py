"""Batch-1 windows whose query rows take several row chunks: every (KV head, split, row chunk) is computed once,
also where KV heads x splits is no multiple of 8 (a grid of its own over BF16 caches), against the FP64
oracle at the verify bars."""
import numpy as np
import pytest

from helpers import AttnCase, rel_l2
import gpu_runner

pytestmark = pytest.mark.gpu

REL_L2_F32 = 1e-3
REL_L2_BF16 = 2e-3


# T = 6: two chunks at group 6 and 8 (5 + 1, 4 + 2 tokens); T = 16: three or four; 2, 3, 5, 9 and 11 splits of
# 256 keys and more: 4 to 44 (KV head, split) units; above 8,192 keys the grid of its own where its XCDs fill evenly
@pytest.mark.parametrize("Hq,Hkv,D,kv", [(24, 4, 256, "i8"), (24, 4, 256, "bf16"), (16, 2, 256, "i8"), (16, 2, 256, "bf16"),
                                         (40, 8, 128, "bf16")])
@pytest.mark.parametrize("L,T", [(300, 7), (700, 16), (1200, 6), (2100, 9), (2700, 16), (8300, 6), (9000, 9), (10300, 16)])
def test_row_chunks(gpu, Hq, Hkv, D, kv, L, T):
    print(f"case row chunks {Hq}/{Hkv}/{D} {kv} L={L} T={T}", flush=True)
    case = AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, kv=kv, seed=900 + L + T + D)
    expected, ref = case.oracle_after_append()
    for f32, bar in ((True, REL_L2_F32), (False, REL_L2_BF16)):
        out, cache = gpu_runner.run_attention(case, out_f32=f32, mode="A1")
        for got, want in zip(cache.download(), expected):
            assert np.array_equal(got, want)
        assert np.all(np.isfinite(out)) and rel_l2(out, ref) <= bar
