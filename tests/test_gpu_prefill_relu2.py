"""The reference's ReLU² prefill over an int8 cache (one and two 32-row blocks a workgroup, its waves
sharing the key blocks) against the oracle, where it can go wrong: chunks and prefixes at the edges
of the 4-token row groups and 32-key blocks, fewer key blocks than waves, a window, strides and a
base that 16-byte stores cannot take, and scales past the chunk never written (NaN)."""
import numpy as np
import pytest

from conftest import gpu_available
from gpu_util import assert_close, bf16_host, dev, say
from embla_attn import layout, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_gpu():
    if not gpu_available():
        pytest.skip("no GPU")
    import torch
    return torch


# 513 tokens and more take two row blocks a workgroup (258 workgroups of one would need two rounds)
@pytest.mark.parametrize("T,p0,window,tok_stride,off", [
    (1, 0, 0, 2048, 0), (1, 31, 0, 2048, 0), (3, 32, 0, 2048, 0), (4, 250, 0, 2048, 0), (5, 251, 0, 2048, 0),
    (33, 1000, 0, 2048, 0), (37, 999, 100, 2048, 0), (8, 700, 33, 2048, 0), (31, 97, 0, 2049, 0), (16, 300, 0, 2048, 3),
    (512, 0, 0, 2048, 0), (513, 0, 0, 2048, 0), (517, 95, 0, 2048, 0), (530, 64, 130, 2048, 0), (519, 33, 0, 2050, 1)])
def test_relu2_prefill(torch_gpu, orc, T, p0, window, tok_stride, off):
    from embla_attn import ops
    torch = torch_gpu
    n_q, n_kv, S = 16, 2, p0 + T
    max_s = (S + 31) // 32 * 32 + 32
    say(f"relu2 prefill T={T} p0={p0} window={window} stride={tok_stride} offset={off}")
    g = synth.SplitMix64(1000 * T + p0)
    q = synth.bf16_bits(g.normal(T * n_q * 128).astype(np.float32)).reshape(T, n_q, 128)
    K, V = (g.int8(n_kv * S * 128).reshape(n_kv, S, 128) for _ in range(2))
    ks, vs = ((0.005 + 0.02 * g.uniform(n_kv * S)).astype(np.float32).reshape(n_kv, S) for _ in range(2))

    def region(rows, scales, kind):
        r = np.full((n_kv, max_s, 128), 77, np.int8)
        r[:, :S] = rows
        sc = np.full((n_kv, max_s), np.nan, np.float32)
        sc[:, :S] = scales
        return dev(np.concatenate([layout.to_tiles(r, kind).view(np.uint8), sc.reshape(-1).view(np.uint8)]))

    kc, vc = region(K, ks, "k"), region(V, vs, "v")
    out = torch.full((T * tok_stride + 16,), 5.0, dtype=torch.bfloat16, device="cuda")
    ops.prefill_int8(dev(q, torch.bfloat16), kc, vc, T, p0, max_s, n_kv, weights=ops.RELU2_SINK, scale_dtype=ops.F32,
                     window=window, out=out[off:], out_strides=(tok_stride, 128))
    got = bf16_host(out)
    rows = got[off:off + T * tok_stride].reshape(T, tok_stride)
    ref = orc.prefill_int8(synth.bf16_val(q), K, ks, V, vs, p0, weights=1, window=window)
    assert_close(rows[:, :2048].reshape(T, n_q, 128), ref, what=f"T={T} p0={p0}")
    assert (rows[:, 2048:] == 5.0).all() and (got[:off] == 5.0).all() and (got[off + T * tok_stride:] == 5.0).all()


def relu2_f64(q, K, V, p0):
    """q [T][16][128] over K, V [2][S][128], all fp64."""
    T, n_q, _ = q.shape
    S = K.shape[1]
    out = np.empty((T, n_q, 128))
    seen = np.arange(S)[None] <= p0 + np.arange(T)[:, None]
    for h in range(n_q):
        p = np.where(seen, np.maximum(q[:, h] @ K[h // 8].T / np.sqrt(128.0), 0.0) ** 2, 0.0)
        out[:, h] = (p @ V[h // 8]) / (np.sqrt(128.0) + p.sum(1, keepdims=True))
    return out


# sizes of q, of K and of V (V's 1 is an absmax of 2); "rising": later keys' scales up to 2^16 times the
# first ones'; "zeros": the first 300 keys all zero; "heads": each query head's q 8 times the last one's
@pytest.mark.parametrize("T", [5, 520])   # one and two row blocks a workgroup
@pytest.mark.parametrize("qs,ks,vs,shape", [
    (1.0, 1.0, 1.0, ""), (0.1, 1.0, 1.0, ""), (0.1, 1.0, 1e-2, ""), (0.1, 1.0, 1e-3, ""), (0.1, 1.0, 1e-4, ""),
    (1e-3, 1.0, 1e-4, ""), (1e-3, 1e-3, 1e-6, ""), (1.0, 1.0, 1e3, ""), (30.0, 4.0, 1e3, ""), (3e5, 1.0, 1.0, ""),
    (0.1, 1.0, 1e-2, "rising"), (1.0, 1.0, 1.0, "zeros"), (2.0 ** -24, 1.0, 1.0, "heads")])
def test_relu2_prefill_range(torch_gpu, T, qs, ks, vs, shape):
    """Weights far from 1, by small or large q, K or V, against 64 bits: a row's error is that of its
    bf16 outputs (2^-9 of each) and of its fp16 weights (2^-11 of each, whatever their size; weights
    and results of random sign add up alike), 2^-8 of its 2-norm with room for the second."""
    from embla_attn import ops
    torch = torch_gpu
    p0, n_kv = 1001, 2
    S = p0 + T
    max_s = (S + 31) // 32 * 32
    say(f"relu2 prefill range T={T} q {qs} k {ks} v {vs} {shape}")
    g = synth.SplitMix64(T + int(1000 * vs) + len(shape))
    x = g.normal(T * 16 * 128).reshape(T, 16, 128) * qs
    if shape == "heads":
        x *= 8.0 ** np.arange(16)[None, :, None]
    q = synth.bf16_bits(x.astype(np.float32))
    K, V = (g.int8(n_kv * S * 128).reshape(n_kv, S, 128) for _ in range(2))
    sk, sv = (((0.5 + g.uniform(n_kv * S)).astype(np.float32) * np.float32(s / 64)).reshape(n_kv, S) for s in (ks, vs))
    if shape == "rising":
        sk, sv = (s * np.exp2(np.arange(S) * 16 / S / 2 - 8).astype(np.float32)[None] for s in (sk, sv))
    if shape == "zeros":
        sk[:, :300] = 0
        sv[:, :300] = 0

    def region(rows, scales, kind):
        r, sc = np.zeros((n_kv, max_s, 128), np.int8), np.full((n_kv, max_s), np.nan, np.float32)
        r[:, :S], sc[:, :S] = rows, scales
        return dev(np.concatenate([layout.to_tiles(r, kind).view(np.uint8), sc.reshape(-1).view(np.uint8)]))

    out = torch.empty((T, 16, 128), dtype=torch.bfloat16, device="cuda")
    ops.prefill_int8(dev(q, torch.bfloat16), region(K, sk, "k"), region(V, sv, "v"), T, p0, max_s, n_kv,
                     weights=ops.RELU2_SINK, scale_dtype=ops.F32, out=out)
    got = bf16_host(out).astype(np.float64)
    ref = relu2_f64(synth.bf16_val(q).astype(np.float64), K * sk.astype(np.float64)[..., None],
                    V * sv.astype(np.float64)[..., None], p0)
    assert np.isfinite(got).all()
    err = np.linalg.norm(got - ref, axis=2) / np.linalg.norm(ref, axis=2)
    print(f"[gpu-case] worst row {err.max():.2e}, rms {np.sqrt((err ** 2).mean()):.2e}", flush=True)
    assert err.max() <= 2.0 ** -8


def test_relu2_prefill_nonfinite_q(torch_gpu):
    """A row with an infinity has no finite output, one with a NaN no weight (0); its neighbours keep theirs."""
    from embla_attn import ops
    torch = torch_gpu
    T, S = 4, 64
    say("relu2 prefill non-finite q")
    g = synth.SplitMix64(5)
    rows = layout.to_tiles(g.int8(2 * S * 128).reshape(2, S, 128), "k").view(np.uint8)
    cache = dev(np.concatenate([rows, np.full(2 * S, 0.01, np.float32).view(np.uint8)]))
    q = torch.randn(T, 16, 128, generator=torch.Generator("cuda").manual_seed(1), device="cuda").bfloat16()
    bad = q.clone()
    bad[1, 3, 7], bad[2, 9, 100] = float("inf"), float("nan")
    a, b = (ops.prefill_int8(x, cache, cache, T, S - T, S, 2, weights=ops.RELU2_SINK, scale_dtype=ops.F32) for x in (q, bad))
    torch.cuda.synchronize()
    assert torch.isnan(b[1, 3]).all() and (b[2, 9] == 0).all()
    b[1, 3], b[2, 9] = a[1, 3], a[2, 9]
    assert torch.equal(a, b)
