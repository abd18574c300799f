"""Windows of at most 256 keys (one split): the attention of one launch that writes its output itself,
at the edges of its chunks, masks and rows, against the FP64 oracle at the verify bars."""
import numpy as np
import pytest

from helpers import AttnCase, rel_l2
import gpu_runner

pytestmark = pytest.mark.gpu

REL_L2_F32 = 1e-3
REL_L2_BF16 = 2e-3


def _run(case, mode="A1"):
    expected, ref = case.oracle_after_append()
    for f32, bar in ((True, REL_L2_F32), (False, REL_L2_BF16)):
        out, cache = gpu_runner.run_attention(case, out_f32=f32, mode=mode)
        for got, want in zip(cache.download(), expected):
            assert np.array_equal(got, want)
        err = rel_l2(out, ref)
        print(f"f32={f32} rel_l2={err:.3e}", flush=True)
        assert np.all(np.isfinite(out)) and err <= bar


# histories around the 32-key chunks and the 128 keys of a step; one row up to 32, two row chunks (T = 6 at
# group 6); 256 keys exactly and 257 (two splits)
@pytest.mark.parametrize("Hq,Hkv,D,kv", [(40, 8, 128, "i8"), (24, 4, 256, "i8"), (40, 8, 128, "bf16"), (16, 2, 256, "bf16"), (8, 8, 128, "i8")])
@pytest.mark.parametrize("L,T", [(0, 1), (0, 6), (31, 1), (32, 4), (100, 2), (127, 3), (128, 4), (250, 6), (251, 6), (255, 1)])
def test_small_windows(gpu, Hq, Hkv, D, kv, L, T):
    print(f"case direct {Hq}/{Hkv}/{D} {kv} L={L} T={T}", flush=True)
    _run(AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, kv=kv, seed=800 + L + T + D))


def _tree(T):
    return np.array([-1] + [(u - 1) // 2 for u in range(1, T)], np.int32)


# 20 nodes: at group 1 one row chunk, at group 5 (100 rows, past the 80-row form) and at head_dim 256 several
@pytest.mark.parametrize("D,Hq,Hkv,kv", [(128, 8, 8, "i8"), (128, 40, 8, "i8"), (256, 16, 2, "i8"), (256, 8, 8, "i8"),
                                         (128, 40, 8, "bf16"), (256, 16, 8, "bf16")])
def test_tree_and_row_chunks(gpu, D, Hq, Hkv, kv):
    print(f"case direct tree {Hq}/{Hkv}/{D} {kv}", flush=True)
    _run(AttnCase([70], T=20, Hq=Hq, Hkv=Hkv, D=D, kv=kv, seed=5, parents=_tree(20)), mode="TREE")


@pytest.mark.parametrize("Hq,Hkv,D,T,parents", [(40, 8, 128, 4, None), (24, 4, 256, 4, None), (8, 8, 128, 20, _tree(20)),
                                                (40, 8, 128, 20, _tree(20)), (24, 4, 256, 9, _tree(9))])
@pytest.mark.parametrize("absmax", [1e5, 1e6])
def test_fp32_range(gpu, Hq, Hkv, D, absmax, T, parents):
    """Groups beyond FP16's range are computed again in FP32 (as in the merge of a split window), a chain's rows and
    a tree's, whose ancestor mask then applies there too."""
    L = 200
    print(f"case direct fp32 range {Hq}/{Hkv}/{D} T={T} {absmax:g}", flush=True)
    case = AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, seed=3, qstd=2e-5, parents=parents)
    rng = np.random.default_rng(8)
    big = np.float16(absmax / 127.0).view(np.uint16)
    for sc in (case.ks, case.vs):
        for _ in range(5):
            sc[0, int(rng.integers(0, Hkv)), int(rng.integers(0, L)), int(rng.integers(0, D // 64))] = big
    _run(case, mode="A1" if parents is None else "TREE")
