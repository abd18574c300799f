"""Prompts through the recurrent-state ops: the chunked gated delta rule (more than 16 tokens at head
dimension 128) at the edges of its 32-token chunks, and the tiled convolution, against the FP64 oracle."""
import numpy as np
import pytest

import ninfer_amd as na
from ninfer_amd import ops
from ninfer_amd.device import DeviceArray, synchronize
from test_gpu_gdn import BF16_REDUCTION, GDN_OUTPUT_BF16, _bf, _dev, _f, _inputs, _ok, run_regular

pytestmark = pytest.mark.gpu

# FP32 sums of products exact in FP32, and one BF16 rounding of v's products: the token-by-token kernel
# is 1.1e-7 to 1.25e-7 from 64 bits in the 2-norm over these ranges, this one 8e-8 to 9e-8.
STATE_REL = 1.5e-7


def _oracle(inp, Hqk, Hv, T, normalize):
    from oracle import pyoracle
    return pyoracle.gdn_recurrent(inp["q"], inp["k"], inp["v"], inp["g"], inp["beta"], inp["state"], 128, Hqk, Hv, T, normalize)


@pytest.mark.parametrize("T", [17, 31, 32, 33, 63, 64, 65, 97, 130])
@pytest.mark.parametrize("Hqk,Hv,normalize,in_place", [(16, 48, True, False), (5, 5, True, True), (2, 18, False, False)])
def test_chunk_edges(gpu, T, Hqk, Hv, normalize, in_place):
    print(f"case gdn chunk T={T} Hqk={Hqk} Hv={Hv} norm={normalize} in_place={in_place}", flush=True)
    inp = _inputs(300 + T + Hv, 128, Hqk, Hv, T, normalized=not normalize, stress_g=T % 2 == 1)
    ref_out, ref_state = _oracle(inp, Hqk, Hv, T, normalize)[:2]
    out, state = run_regular(inp, 128, Hqk, Hv, T, normalize, in_place)
    _ok(_f(out).reshape(T, Hv, 128), ref_out, GDN_OUTPUT_BF16, "out")
    rel = np.linalg.norm(state - ref_state) / np.linalg.norm(ref_state)
    print(f"state rel {rel:.2e}", flush=True)
    assert rel <= STATE_REL


def test_decay_extremes(gpu):
    """Decays of exactly 0 and 1, and long runs of strong decay: no difference of logarithms is lost."""
    T, H = 70, 4
    inp = _inputs(31, 128, H, H, T, normalized=False)
    inp["g"][5] = -np.inf
    inp["g"][6:20] = -0.001
    inp["g"][20:36] = -90.0
    inp["g"][36:50] = 0.0
    ref_out, ref_state = _oracle(inp, H, H, T, True)[:2]
    out, state = run_regular(inp, 128, H, H, T, True, False)
    _ok(_f(out).reshape(T, H, 128), ref_out, GDN_OUTPUT_BF16, "out")
    assert np.linalg.norm(state - ref_state) / np.linalg.norm(ref_state) <= STATE_REL


@pytest.mark.parametrize("where", ["v", "k", "q", "g"])
def test_non_finite_token_leaves_earlier_outputs(gpu, where):
    """A NaN in token 40 reaches no output before it, as token by token."""
    T, H = 66, 3
    inp = _inputs(77, 128, H, H, T, normalized=False)
    clean = _f(run_regular(inp, 128, H, H, T, True, False)[0]).reshape(T, H, 128)
    if where == "g":
        inp["g"][40] = np.nan
    else:
        inp[where].reshape(T, H, 128)[40, :, 7] = 0x7FC0
    out = _f(run_regular(inp, 128, H, H, T, True, False)[0]).reshape(T, H, 128)
    _ok(out[:40], clean[:40], GDN_OUTPUT_BF16, "out before") # the chunk's products in another order
    assert np.isnan(out[40]).any()


@pytest.mark.parametrize("rows", [[(20, "k")], [(33, "q")], [(5, "k"), (40, "k"), (40, "q"), (65, "q")]])
def test_squared_norm_beyond_fp32(gpu, rows):
    """A finite k or q row whose squared norm overflows FP32 is normalized to 0, as token by token: the token decays
    the state and adds nothing, or puts out 0, and no other token sees it."""
    T, H = 66, 3
    inp = _inputs(78, 128, H, H, T, normalized=False)
    zeroed = {n: x.copy() for n, x in inp.items()}
    for t, n in rows:
        inp[n].reshape(T, H, 128)[t, 1, ::3] = _bf(np.array([3.0e38], np.float32))[0]
        zeroed[n].reshape(T, H, 128)[t, 1] = 0
    ref_out, ref_state = _oracle(zeroed, H, H, T, True)[:2]
    out, state = run_regular(inp, 128, H, H, T, True, False)
    _ok(_f(out).reshape(T, H, 128), ref_out, GDN_OUTPUT_BF16, "out")
    assert np.linalg.norm(state - ref_state) / np.linalg.norm(ref_state) <= STATE_REL
    head = {n: x if n == "state" else np.ascontiguousarray(x.reshape(T, -1)[:16]).reshape(16, *x.shape[1:]) for n, x in inp.items()}
    first, _ = run_regular(head, 128, H, H, 16, True, False)
    _ok(_f(out).reshape(T, H, 128)[:16], _f(first).reshape(16, H, 128), GDN_OUTPUT_BF16, "token by token")


@pytest.mark.parametrize("C,T,offset,in_place", [(10240, 17, 0, False), (10240, 1700, 0, True), (1001, 33, 0, True), (64, 16, 0, False),
                                                 (130, 100, 0, False), (512, 40, 1, True), (24, 19, 0, True)])
def test_conv_prompt(gpu, C, T, offset, in_place):
    """Tiles of 16 and 4 tokens, 8, 2 and 1 channels per thread (odd C; tensors one element off), and the
    window read before it is replaced."""
    print(f"case conv prompt C={C} T={T} offset={offset} in_place={in_place}", flush=True)
    from oracle import pyoracle
    rng = np.random.default_rng(C + T)
    x, w, win = (_bf(rng.uniform(-2, 2, n)) for n in (T * C, 4 * C, 3 * C))

    def dev(a, shape):
        d = DeviceArray.from_numpy(na.BF16, np.concatenate([np.zeros(offset, np.uint16), a]))
        return d, na.Tensor.make(d.ptr + 2 * offset, na.BF16, shape)
    keep, (tx, tw, tin, to, tout) = zip(*(dev(a, s) for a, s in ((x, (C, T)), (w, (C, 4)), (win, (C, 3)), (win * 0, (C, 3)), (x * 0, (C, T)))))
    ops.causal_conv1d_silu(tx, tw, tin, tin if in_place else to, tout)
    synchronize()
    ref = pyoracle.causal_conv1d_silu(x, w, win, C, T)
    ref_out = ref[0] if isinstance(ref, tuple) else ref
    _ok(_f(keep[4].numpy()[offset:]).reshape(T, C), np.asarray(ref_out).reshape(T, C), BF16_REDUCTION, "out")
    got = keep[2 if in_place else 3].numpy()[offset:].reshape(3, C)
    assert np.array_equal(got, x.reshape(T, C)[-3:] if T >= 3 else got)
