"""Short chunks' key-range splits (up to 64, a 128-key tile each at least) against the oracle: the split
counts at which the merge changes or a group of its lanes has no record, a workspace of four fp32
records (as sized before a call's own split count), rows whose every key lies in a few splits,
types, and output strides that no 16-byte store takes."""
import numpy as np
import pytest

from conftest import gpu_available
from gpu_util import assert_close, bf16_host, dev, f16_host, say
from embla_attn import layout, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_gpu():
    if not gpu_available():
        pytest.skip("no GPU")
    import torch
    return torch


# 64-key tiles (p0 + T) / 64, halved: the splits of a chunk of few workgroups
@pytest.mark.parametrize("T,p0,window,f16,small_ws,tok_stride", [
    (20, 236, 0, False, False, 2048),      # 2
    (20, 492, 0, True, False, 2048),       # 4: the last of the merge of a row a lane group
    (20, 620, 0, False, False, 2050),      # 5: the first of a row a wave
    (7, 2042, 0, True, False, 2048),       # 16: the last of them
    (20, 2156, 0, False, False, 2048),     # 17: the first of a row a workgroup
    (1, 8191, 0, False, False, 2048),      # 64, one token
    (65, 5000, 0, False, False, 2049),     # two row blocks: 32 splits
    (20, 8200, 0, False, True, 2048),      # 64 wanted, room for 4
    (33, 3000, 700, False, False, 2048),   # a window: 12 tiles, splits that some rows do not see
    (130, 0, 0, True, False, 2048)])       # no prefix
def test_prefill_splits(torch_gpu, orc, T, p0, window, f16, small_ws, tok_stride):
    from embla_attn import ops
    torch = torch_gpu
    n_q, n_kv, S = 16, 4, p0 + T
    max_s = (S + 31) // 32 * 32
    say(f"prefill splits T={T} p0={p0} window={window} f16={f16} small_ws={small_ws}")
    g = synth.SplitMix64(31 * T + p0)
    bits = synth.f16_bits if f16 else synth.bf16_bits
    q = bits(g.normal(T * n_q * 128).astype(np.float32)).reshape(T, n_q, 128)
    K, V = (g.int8(n_kv * S * 128).reshape(n_kv, S, 128) for _ in range(2))
    ks, vs = (synth.f16_bits(0.005 + 0.015 * g.uniform(n_kv * S)).reshape(n_kv, S) for _ in range(2))
    kc, vc = dev(layout.pack_region(K, ks, max_s, "k")), dev(layout.pack_region(V, vs, max_s, "v"))
    dt, code = (torch.float16, ops.F16) if f16 else (torch.bfloat16, ops.BF16)
    ws = ops.PrefillWorkspace(T, n_q)
    if small_ws:
        ws.nbytes = 4 * T * n_q * 132 * 4
    out = torch.full((T * tok_stride,), 3.0, dtype=dt, device="cuda")
    ops.prefill_int8(dev(q, dt), kc, vc, T, p0, max_s, n_kv, window=window, q_dtype=code, out_dtype=code, out=out,
                     out_strides=(tok_stride, 128), ws=ws)
    got = (f16_host if f16 else bf16_host)(out).reshape(T, tok_stride)
    val = synth.f16_val if f16 else synth.bf16_val
    ref = orc.prefill_int8(val(q), K, synth.f16_val(ks), V, synth.f16_val(vs), p0, window=window)
    assert_close(got[:, :2048].reshape(T, n_q, 128), ref, what=f"T={T} p0={p0}")
    assert (got[:, 2048:] == 3.0).all()


@pytest.mark.parametrize("T,p0", [(193, 130), (60, 440), (193, 800), (60, 5000), (20, 8200)])   # 2, 3, 7, 39, 64 splits at most
def test_prefill_splits_precision(torch_gpu, T, p0):
    """A split's sums stay in fp32 on their way to the merge: with fp16 outputs, the error against 64
    bits is the unsplit call's (1.08 to 1.1 times that with each split's O / l rounded to fp16 too)."""
    from embla_attn import ops
    torch = torch_gpu
    n_q, n_kv, S = 16, 4, p0 + T
    max_s = (S + 31) // 32 * 32
    say(f"prefill splits precision T={T} p0={p0}")
    g = synth.SplitMix64(T + p0)
    q = synth.f16_bits(g.normal(T * n_q * 128)).reshape(T, n_q, 128)
    K, V = (g.int8(n_kv * S * 128).reshape(n_kv, S, 128) for _ in range(2))
    ks, vs = (synth.f16_bits(0.005 + 0.01 * g.uniform(n_kv * S)).reshape(n_kv, S) for _ in range(2))
    kc, vc = dev(layout.pack_region(K, ks, max_s, "k")), dev(layout.pack_region(V, vs, max_s, "v"))
    qf = synth.f16_val(q).astype(np.float64)
    Kf, Vf = (x * synth.f16_val(s).astype(np.float64)[..., None] for x, s in ((K, ks), (V, vs)))
    ref = np.empty((T, n_q, 128))
    for h in range(n_q):
        s = qf[:, h] @ Kf[h // 4].T / np.sqrt(128.0)
        s[np.arange(S)[None] > p0 + np.arange(T)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        ref[:, h] = p @ Vf[h // 4] / p.sum(1, keepdims=True)
    err = []
    for ws in (None, ops.PrefillWorkspace(T, n_q)):
        o = ops.prefill_int8(dev(q, torch.float16), kc, vc, T, p0, max_s, n_kv, q_dtype=ops.F16, out_dtype=ops.F16, ws=ws)
        err.append(np.linalg.norm(f16_host(o) - ref) / np.linalg.norm(ref))
    print(f"[gpu-case] unsplit {err[0]:.3e} split {err[1]:.3e}", flush=True)
    assert err[1] <= 1.03 * err[0]


@pytest.mark.parametrize("T,window", [(12, 1024), (193, 1024), (60, 4096)])
def test_prefill_ring_without_a_prefix_is_one_pass(torch_gpu, T, window):
    """A ring's splits follow the keys there are, not the window: a conversation's first message fills
    a tile or two, and the call with a workspace is the unsplit one, bit for bit."""
    from embla_attn import ops
    torch = torch_gpu
    R = (window + T + 127) // 128 * 128
    say(f"prefill ring without a prefix T={T} window={window}")
    g = torch.Generator("cuda").manual_seed(T)
    k, v = (torch.randn(4 * R * 128, generator=g, device="cuda").half() for _ in range(2))
    q = torch.randn(T, 16, 128, generator=g, device="cuda").half()
    a, b = (ops.prefill_ring(q, k, v, T, 0, R, window, 4, dtype=ops.F16, ws=ws) for ws in (None, ops.PrefillWorkspace(T, 16)))
    torch.cuda.synchronize()
    assert torch.equal(a, b)
