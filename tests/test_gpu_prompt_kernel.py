"""The prompt kernel (A1/A3 above the verify extents) at the edges of its tiles, against the FP64 oracle
at the verify bars: row tiles of 64, 128 and 256 rows (WK = 4, 2, 1), key tiles of 128 (head_dim 128)
and 64 keys (256), unsplit and split over the keys; the exact recompute of groups beyond FP16's
range in both forms; tensors it cannot address, which the verify launches take; and the flat append."""
import numpy as np
import pytest

import ninfer_amd as na
from ninfer_amd import ops
from ninfer_amd.device import DeviceArray, DeviceBuffer, synchronize
from helpers import AttnCase, rel_l2
import gpu_runner

pytestmark = pytest.mark.gpu

REL_L2_F32 = 1e-3


def _run(case, **kw):
    expected, ref = case.oracle_after_append()
    out, cache = gpu_runner.run_attention(case, out_f32=True, **kw)
    for got, want in zip(cache.download(), expected):
        assert np.array_equal(got, want)
    err = rel_l2(out, ref)
    print(f"rel_l2={err:.3e}", flush=True)
    assert np.all(np.isfinite(out)) and err <= REL_L2_F32, err
    return out


# (heads, D, cache, history, tokens): 5 x 77 = 385 rows end one row past a 64- and 128-row tile; windows one
# key before, at and past a key tile; one long prompt of 256-row tiles; splits (short prompts over
# a longer history); a group of one head and one of eight
@pytest.mark.parametrize("Hq,Hkv,D,kv,L,T", [
    (40, 8, 128, "i8", 0, 65), (40, 8, 128, "i8", 50, 77), (40, 8, 128, "i8", 51, 77), (40, 8, 128, "i8", 52, 77),
    (40, 8, 128, "i8", 3000, 66), (40, 8, 128, "i8", 7, 1100), (40, 8, 128, "bf16", 51, 77), (40, 8, 128, "bf16", 2500, 65),
    (24, 4, 256, "i8", 0, 33), (24, 4, 256, "i8", 31, 33), (24, 4, 256, "i8", 32, 33), (24, 4, 256, "bf16", 2000, 43),
    (16, 2, 256, "i8", 0, 64), (16, 2, 256, "bf16", 1, 64), (16, 2, 256, "i8", 1500, 129), (24, 4, 256, "i8", 3, 700),
    (4, 4, 128, "i8", 129, 130), (64, 2, 128, "i8", 10, 70)])
def test_tile_edges(gpu, Hq, Hkv, D, kv, L, T):
    print(f"case prompt kernel {Hq}/{Hkv}/{D} {kv} L={L} T={T}", flush=True)
    _run(AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, kv=kv, seed=6000 + L + T + Hq))


# A wide envelope: the plan follows its end, the keys the device positions.
@pytest.mark.parametrize("L,T,cap", [(300, 70, 20000), (700, 300, 40000)])
def test_wide_envelope(gpu, L, T, cap):
    print(f"case prompt envelope L={L} T={T} cap={cap}", flush=True)
    case = AttnCase([L], T=T, seed=61 + T, max_context=cap)
    _run(case, envelope=(1, cap))


def _attend64(case, planes, last):
    """Attention in 64 bits of every token over the cache rows [0, last]."""
    f32 = lambda bits: (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)  # noqa: E731
    if case.kv == "bf16":
        k, v = (f32(x[0]) for x in planes)
    else:
        k, v = (c[0].astype(np.float64) * np.repeat(s[0].view(np.float16).astype(np.float64), 64, axis=-1)
                for c, s in ((planes[0], planes[2]), (planes[1], planes[3])))
    n = int(last.max()) + 1
    q = f32(case.q).reshape(case.T, case.Hkv, -1, case.D)
    hidden = np.arange(n)[None, :] > last[:, None]
    out = np.empty(q.shape)
    for h in range(case.Hkv):
        score = np.einsum("tgd,kd->tgk", q[:, h], k[h, :n], optimize=True) * case.scale
        score[np.broadcast_to(hidden[:, None], score.shape)] = -np.inf
        p = np.exp(score - score.max(-1, keepdims=True))
        out[:, h] = np.einsum("tgk,kd->tgd", p / p.sum(-1, keepdims=True), v[h, :n], optimize=True)
    return out.reshape(-1)


# An envelope that ends before the last positions: a token sees the keys up to its position or the envelope's end.
@pytest.mark.parametrize("Hq,Hkv,D,kv,L,T,cap", [
    (40, 8, 128, "i8", 100, 300, 350), (40, 8, 128, "i8", 2500, 80, 2530), (40, 8, 128, "i8", 100, 200, 200), (24, 4, 256, "i8", 30, 300, 301),
    (16, 2, 256, "bf16", 1500, 70, 1510), (40, 8, 128, "bf16", 100, 1000, 1003)])
@pytest.mark.parametrize("rare", [False, True])
def test_envelope_clamps_positions(gpu, Hq, Hkv, D, kv, L, T, cap, rare):
    if rare and kv == "bf16":
        pytest.skip("scales are INT8's")
    print(f"case prompt clamp {Hq}/{Hkv}/{D} {kv} L={L} T={T} cap={cap} rare={rare}", flush=True)
    case = AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, kv=kv, seed=41, qstd=2e-5 if rare else 1.0)
    if rare:
        _rare_scales(case, 3)
    planes, _ = case.oracle_after_append()
    ref = _attend64(case, planes, np.minimum(case.positions, cap - 1))
    out, cache = gpu_runner.run_attention(case, out_f32=True, envelope=(1, cap))
    for got, want in zip(cache.download(), planes):
        assert np.array_equal(got, want)
    err = rel_l2(out, ref)
    print(f"rel_l2={err:.3e}", flush=True)
    assert np.all(np.isfinite(out)) and err <= REL_L2_F32


@pytest.mark.parametrize("Hq,Hkv,D,L,T", [(40, 8, 128, 100, 65), (40, 8, 128, 2600, 65), (24, 4, 256, 150, 40), (24, 4, 256, 1500, 40)])
@pytest.mark.parametrize("absmax", [1e5, 1e6])
def test_fp32_range(gpu, Hq, Hkv, D, L, T, absmax):
    """Scales above 512 in K and V (K' or V' beyond FP16), unsplit and split over the keys: the rows are
    computed again in FP32, as the verify kernels' merge does. K groups and V groups of their own
    positions, so rows with only one kind exist."""
    print(f"case prompt fp32 range {Hq}/{Hkv}/{D} L={L} T={T} absmax={absmax:g}", flush=True)
    case = AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, seed=9, qstd=2e-5)
    rng = np.random.default_rng(5)
    big = np.float16(absmax / 127.0).view(np.uint16)
    for sc in (case.ks, case.vs):
        for _ in range(6):
            sc[0, int(rng.integers(0, Hkv)), int(rng.integers(0, L)), int(rng.integers(0, D // 64))] = big
    _run(case)


def _rare_scales(case, seed, n=6, absmax=1e5, planes=("ks", "vs")):
    rng = np.random.default_rng(seed)
    big = np.float16(absmax / 127.0).view(np.uint16)
    for name in planes:
        for _ in range(n):
            getattr(case, name)[0, int(rng.integers(0, case.Hkv)), int(rng.integers(0, case.Ls[0])), int(rng.integers(0, case.D // 64))] = big


@pytest.mark.parametrize("Hq,Hkv,D,L,T", [
    (40, 8, 128, 130, 1100), (40, 8, 128, 900, 300), (24, 4, 256, 100, 700), (16, 2, 256, 4000, 65), (40, 8, 128, 5000, 70)])
@pytest.mark.parametrize("planes", [("ks",), ("vs",), ("ks", "vs")])
def test_fp32_range_few_tiles(gpu, Hq, Hkv, D, L, T, planes):
    """Such groups in a few key tiles among many, in each form of the kernel (256, 128 and 64 rows, one split and
    several): only those tiles, and the partials that FP16 cannot hold, are computed in FP32."""
    print(f"case prompt rare scales {Hq}/{Hkv}/{D} L={L} T={T} {planes}", flush=True)
    case = AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, seed=19, qstd=2e-5)
    _rare_scales(case, L + T, planes=planes)
    _run(case)


@pytest.mark.parametrize("Hq,Hkv,D,L,T", [(40, 8, 128, 2000, 96), (40, 8, 128, 2000, 512), (24, 4, 256, 2000, 512)])
@pytest.mark.parametrize("plane", ["ks", "vs"])
def test_rare_scales_cost(gpu, Hq, Hkv, D, L, T, plane):
    """One group beyond FP16's range costs its tile and the partials it reaches, not the whole prompt: at most 5 times
    the plain prompt (MI355X: 3 times; a whole prompt computed again row by row took 57 to 250 times)."""
    case = AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, seed=4)
    plain = gpu_runner.attention_us(case)
    for h in range(Hkv):
        getattr(case, plane)[0, h, 3, 0] = np.float16(600.0).view(np.uint16)
    rare = gpu_runner.attention_us(case)
    print(f"{Hq}/{Hkv}/{D} L={L} T={T} {plane}: {rare:.1f} us, plain {plain:.1f} us")
    assert rare <= 5.0 * plain


@pytest.mark.parametrize("Hq,Hkv,D,kv,L,T", [(40, 8, 128, "bf16", 0, 100), (40, 8, 128, "bf16", 300, 600), (40, 8, 128, "bf16", 2500, 65),
                                             (24, 4, 256, "bf16", 20, 300), (40, 8, 128, "i8", 10, 200), (16, 2, 256, "i8", 1500, 70)])
@pytest.mark.parametrize("bits", [0x7F80, 0x7FC0])
def test_non_finite_value_leaves_earlier_outputs(gpu, Hq, Hkv, D, kv, L, T, bits):
    """An infinite or NaN V value reaches the outputs of the tokens that see it and no others."""
    print(f"case prompt non-finite {Hq}/{Hkv}/{D} {kv} L={L} T={T} {bits:#x}", flush=True)
    case = AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, kv=kv, seed=33)
    (planes, ref), at, head = case.oracle_after_append(), T // 2, 1
    cache = gpu_runner.upload_cache(case)
    gpu_runner.append(case, cache)
    dirty = [x.copy() for x in planes]
    if kv == "bf16":
        dirty[1][0, head, L + at, 7] = bits
    else:  # the scale of a group: FP16 infinity or NaN
        dirty[3][0, head, L + at, 0] = 0x7C00 if bits == 0x7F80 else 0x7E00
    cache.upload(*dirty)
    out, _ = gpu_runner.run_attention(case, out_f32=True, mode="A3", cache=cache)
    out, ref = np.asarray(out, np.float64).reshape(T, Hq, D), np.asarray(ref, np.float64).reshape(T, Hq, D)
    G = Hq // Hkv
    reached = np.zeros(out.shape, bool)
    reached[at:, head * G:(head + 1) * G, (7 if kv == "bf16" else slice(0, 64))] = True
    assert np.all(np.isfinite(out[~reached])) and rel_l2(out[~reached], ref[~reached]) <= REL_L2_F32
    assert not np.any(np.isfinite(out[reached]))


@pytest.mark.parametrize("L,T", [(100, 200), (2500, 65)])
def test_nan_key_is_not_dropped(gpu, L, T):
    """A row that sees a NaN key has no defined sum: it is 0 with one key split and with several, never the result
    of the other splits alone."""
    print(f"case prompt NaN key L={L} T={T}", flush=True)
    case = AttnCase([L], T=T, kv="bf16", seed=35)
    (planes, ref), head = case.oracle_after_append(), 2
    cache = gpu_runner.upload_cache(case)
    gpu_runner.append(case, cache)
    dirty = [x.copy() for x in planes]
    dirty[0][0, head, 40, 3] = 0x7FC0
    cache.upload(*dirty)
    out, _ = gpu_runner.run_attention(case, out_f32=True, mode="A3", cache=cache)
    out, ref = np.asarray(out).reshape(T, 8, 5, 128), np.asarray(ref, np.float64).reshape(T, 8, 5, 128)
    others = [h for h in range(8) if h != head]
    assert rel_l2(out[:, others], ref[:, others]) <= REL_L2_F32
    assert not np.any(out[:, head])


@pytest.mark.parametrize("Hq,Hkv,D,kv,L,T", [(16, 2, 256, "i8", 65536, 96), (24, 4, 256, "bf16", 65536, 192), (40, 8, 128, "i8", 65536, 96),
                                             (24, 4, 256, "i8", 16000, 128)])
def test_long_history_cost(gpu, Hq, Hkv, D, kv, L, T):
    """A prompt over a long history takes no longer than the same tokens in calls of 32 (10% for the estimates
    that choose the route; MI355X: 0.5 to 1.0, where the prompt kernel alone took up to 2)."""
    case = AttnCase([L], T=T, Hq=Hq, Hkv=Hkv, D=D, kv=kv, seed=2, gen="pcg")
    whole, parts = gpu_runner.attention_us(case), gpu_runner.attention_us(case, tokens=32)
    print(f"{Hq}/{Hkv}/{D} {kv} L={L} T={T}: {whole:.1f} us, in calls of 32 {parts:.1f} us")
    assert whole <= 1.1 * parts


def test_unaligned_tensors_take_the_verify_launches(gpu):
    """q one element into its buffer: accepted as before, and within the same bar."""
    case = AttnCase([200], T=70, seed=17)
    _, ref = case.oracle_after_append()
    cache = gpu_runner.upload_cache(case)
    gpu_runner.append(case, cache)
    D, Hq, T = case.D, case.Hq, case.T
    raw = DeviceArray.from_numpy(na.BF16, np.concatenate([np.zeros(2, np.uint16), case.q]))
    q = na.Tensor.make(raw.ptr + 4, na.BF16, (D, Hq, T))
    pos = DeviceArray.from_numpy(na.I32, case.positions, (T, 1))
    out = DeviceArray(na.FP32, (D, Hq, T))
    ws = DeviceBuffer(ops.gqa_attention_workspace_bytes(Hq, case.Hkv, D, T, 1, case.max_context))
    ops.gqa_attention_cached(q, pos.tensor(), case.scale, cache.view(), (1, case.max_context), ws, out.tensor())
    synchronize()
    assert rel_l2(out.numpy().astype(np.float64), ref) <= REL_L2_F32


@pytest.mark.parametrize("D,T,B,offset", [(128, 1, 1, 0), (128, 3, 3, 0), (256, 5, 2, 0), (128, 700, 1, 0), (128, 3, 2, 2), (256, 2, 1, 1)])
def test_append_forms(gpu, D, T, B, offset):
    """The flat encoder (aligned) and the one-wave-per-group form (`offset` elements off) write the
    oracle's codes and scales bit for bit, negative positions and zero groups included."""
    print(f"case append D={D} T={T} B={B} offset={offset}", flush=True)
    case = AttnCase([10 * (b + 1) for b in range(B)], T=T, Hq=8, Hkv=4, D=D, seed=T + B)
    case.k_new[:64] = 0
    case.v_new[64:128] = 0x8000
    (kc, vc, ks, vs) = (x.copy() for x in case.cache_planes())
    from oracle import pyoracle
    pyoracle.kv_append(case.k_new, case.v_new, case.positions, T, B, 4, D, case.P, kc, vc, ks, vs)
    if T > 1:  # a negative position is skipped (the oracle takes real ones only): its row stays as it was
        row = int(case.positions[1])
        for got, was in zip((kc, vc, ks, vs), case.cache_planes()):
            got[0, :, row] = was[0, :, row]
        case.positions[1] = -1
    cache = gpu_runner.upload_cache(case)
    pad = np.zeros(offset, np.uint16)
    dk = DeviceArray.from_numpy(na.BF16, np.concatenate([pad, case.k_new]))
    dv = DeviceArray.from_numpy(na.BF16, np.concatenate([pad, case.v_new]))
    pos = DeviceArray.from_numpy(na.I32, case.positions, (T, B))
    ops.gqa_kv_append(na.Tensor.make(dk.ptr + 2 * offset, na.BF16, (D, 4, T, B)),
                      na.Tensor.make(dv.ptr + 2 * offset, na.BF16, (D, 4, T, B)), pos.tensor(), cache.view())
    synchronize()
    for got, want in zip(cache.download(), (kc, vc, ks, vs)):
        assert np.array_equal(got, want)


def test_append_of_several_launches(gpu):
    """2^35 elements of K: more 8-element pieces than one grid holds. Two columns of each of 32 sequences are
    committed, the last ones' by the second launch, with the oracle's codes."""
    from oracle import pyoracle
    T, B, Hkv, D, P, n = 1 << 20, 32, 8, 128, 256, 2
    row = Hkv * D
    src = DeviceArray(na.BF16, (D, Hkv, T, B))  # 64 GiB, only the committed columns written
    rng = np.random.default_rng(12)
    cols = (rng.normal(size=(B, n, row)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    for b in range(B):
        src.buf.upload(cols[b], 2 * row * T * b)
    positions = np.full((B, T), -1, np.int32)
    positions[:, :n] = np.arange(B)[:, None] * 2 + np.arange(n)
    pos = DeviceArray.from_numpy(na.I32, positions, (T, B))
    count = DeviceArray.from_numpy(na.I32, np.full(B, n, np.int32), (B,))
    from ninfer_amd.kv_cache import KVCacheLayer
    cache = KVCacheLayer(P, Hkv, D, B)
    planes = [np.zeros((B, Hkv, P, D), np.int8), np.zeros((B, Hkv, P, D), np.int8),
              np.zeros((B, Hkv, P, D // 64), np.uint16), np.zeros((B, Hkv, P, D // 64), np.uint16)]
    cache.upload(*planes)
    ops.kv_cache_append_prefix(src.tensor(), src.tensor(), pos.tensor(), count.tensor(), (0, n), cache.view())
    synchronize()
    for b in range(B):
        one = cols[b].reshape(-1)
        pyoracle.kv_append(one, one, positions[b, :n].copy(), n, 1, Hkv, D, P, *(x[b] for x in planes))
    for got, want in zip(cache.download(), planes):
        assert np.array_equal(got.reshape(want.shape), want)
