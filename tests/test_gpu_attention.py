"""GPU parity: the attention core and KV cache (aero_hip_attention /
aero_hip_kv_write / aero_hip_softmax_rows and the reference-compatible
aero_attention_tiled / aero_attention / aero_softmax*) against the oracle's
restatement of src/transformer.cpp:120-214, src/tensor.cpp:167-178 and
src/kv.cpp:13-46, and the reference's own outputs (tests/golden/ref_vectors.npz).

Attention and softmax: <= 1e-5 relative to the output's scale, the
reference's RTOL (tests/test_transformer_native.py:34-37,52-61); the GPU sums
in another order and uses its own exp. KV quantisation (integer codes and
scales): bit-exact.
"""
import numpy as np
import pytest

from conftest import RTOL, bits_equal, golden, rel_to_scale
from aero_amd import ops
from aero_amd import transformer_native as TN
from aero_amd.device import DeviceArray as DA, Event, tune_set

pytestmark = pytest.mark.gpu


def gpu_attention(q, k, v, scale, qpos=None, kpos=None, window=0, kv_dt=0, ks=None, vs=None,
                  head_dim=None, value_dim=None):
    T, H, D = q.shape
    S, HK = k.shape[0], k.shape[1]
    D = head_dim or D
    DV = value_dim or v.shape[2]
    out = DA.empty((T, H, DV))
    dq = DA.from_numpy(np.ascontiguousarray(q, np.float32))
    dk, dv = DA.from_numpy(np.ascontiguousarray(k)), DA.from_numpy(np.ascontiguousarray(v))
    dqp = None if qpos is None else DA.from_numpy(np.asarray(qpos, np.int32))
    dkp = None if kpos is None else DA.from_numpy(np.asarray(kpos, np.int32))
    dks = None if ks is None else DA.from_numpy(np.asarray(ks, np.float32))
    dvs = None if vs is None else DA.from_numpy(np.asarray(vs, np.float32))
    ops.attention(dq, dk, dv, out, T, H, HK, D, DV, S, scale, qpos=dqp, kpos=dkp, window=window,
                  kv_dt=kv_dt, k_scale=dks, v_scale=dvs)
    return out.numpy()


def rand_qkv(rng, T, H, HK, D, DV, S):
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    k = rng.standard_normal((S, HK, D)).astype(np.float32)
    v = rng.standard_normal((S, HK, DV)).astype(np.float32)
    return q, k, v


def test_attention_golden(hip):
    """The reference's own attention outputs: causal with positions (one query
    at a position below every key), a window, shuffled key positions."""
    g = golden("ref_vectors.npz")
    q, k, v, qpos = g["att_q"], g["att_k"], g["att_v"], g["att_qpos"]
    assert rel_to_scale(gpu_attention(q, k, v, 0.125, qpos=qpos), g["att_out"]) <= RTOL
    assert rel_to_scale(gpu_attention(q, k, v, 0.125, qpos=qpos, window=8),
                        g["att_out_win8"]) <= RTOL
    assert rel_to_scale(gpu_attention(q, k, v, 0.125, qpos=qpos, kpos=g["att_kpos"]),
                        g["att_out_kpos"]) <= RTOL
    # host ABI (engine/transformer_native.py shapes)
    assert rel_to_scale(TN.attention_tiled(q, k, v, 0.125, qpos=qpos), g["att_out"]) <= RTOL
    assert rel_to_scale(TN.softmax(g["softmax_x"]), g["softmax_y"]) <= RTOL


@pytest.mark.parametrize("T,H,HK,D,DV,S,window", [
    (1, 32, 8, 128, 128, 1, 0),        # decode, one key
    (1, 32, 8, 128, 128, 300, 0),      # decode, Llama-3-8B heads
    (1, 32, 8, 128, 128, 4096, 0),     # decode, 4k cache (key chunks + combine)
    (1, 64, 8, 128, 128, 2000, 0),     # 8 query heads per kv head
    (1, 14, 2, 64, 64, 777, 0),        # Qwen2-0.5B heads
    (1, 16, 2, 256, 256, 513, 0),      # head_dim 256 (Gemma-3 / Qwen3-next)
    (1, 32, 8, 128, 128, 1000, 64),    # sliding window
    (257, 8, 2, 128, 128, 257, 0),     # causal prefill
    (100, 6, 6, 80, 48, 130, 0),       # MHA, dims not a multiple of 16, value_dim < head_dim
    (33, 4, 1, 32, 32, 40, 7),         # MQA with a window
    (200, 8, 2, 128, 128, 300, 50),    # prefill after a cached prefix, with a window
    (3, 16, 4, 64, 64, 2500, 100),     # three tokens at once, head_dim 64, window
    (1, 8, 8, 128, 128, 5000, 0),      # MHA decode
    (100, 8, 4, 256, 256, 300, 0),     # head_dim 256 prefill after a cached prefix (matrix cores)
    (77, 16, 2, 256, 256, 77, 40),     # head_dim 256, 8 query heads a kv head, a window
    (1024, 8, 4, 256, 256, 1024, 0),   # Gemma-3-4B heads, 1024-token causal prefill
])
def test_attention_vs_oracle(hip, oracle, T, H, HK, D, DV, S, window):
    rng = np.random.default_rng(T * 7 + H + S + D + window)
    q, k, v = rand_qkv(rng, T, H, HK, D, DV, S)
    qpos = np.arange(S - T, S, dtype=np.int32)      # the last T positions (prefill / decode)
    scale = 1.0 / np.sqrt(D)
    print(f"attention T={T} H={H} HK={HK} D={D} DV={DV} S={S} window={window}", flush=True)
    got = gpu_attention(q, k, v, scale, qpos=qpos, window=window)
    want = oracle.attention_tiled(q, k, v, scale, qpos=qpos, window=window or None)
    assert rel_to_scale(got, want) <= RTOL


@pytest.mark.parametrize("D", [64, 256])
def test_attention_positions_and_masks(hip, oracle, D):
    """Arbitrary query / key positions (a shuffled cache), a query before every
    key (exact zeros), and the decode entry of the host ABI; head dims 64 and
    256 (both on the fp32 matrix-core kernel)."""
    rng = np.random.default_rng(5 + D)
    T, H, HK, S = 9, 8, 4, 70
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    qpos = np.array([-3, 0, 5, 69, 12, 40, 41, 100, 2], np.int32)
    kpos = rng.permutation(S).astype(np.int32)
    got = gpu_attention(q, k, v, 0.2, qpos=qpos, kpos=kpos)
    assert rel_to_scale(got, oracle.attention_tiled(q, k, v, 0.2, qpos=qpos, kpos=kpos)) <= RTOL
    assert not got[0].any()
    got_w = gpu_attention(q, k, v, 0.2, qpos=qpos, kpos=kpos, window=5)
    assert rel_to_scale(got_w, oracle.attention_tiled(q, k, v, 0.2, qpos=qpos, kpos=kpos,
                                                      window=5)) <= RTOL
    dq = rng.standard_normal((H, D)).astype(np.float32)
    assert rel_to_scale(TN.attention(dq, k, v, 0.2), oracle.attention(dq, k, v, 0.2)) <= RTOL


@pytest.mark.parametrize("dt", [0, 1, 2])
def test_kv_write_bit_exact_and_ring(hip, oracle, dt):
    """Device quantisation of (token, head) vectors equals the reference's
    aero_kv_write_vec code for code and scale for scale, at ring positions
    (phys0 + t) % cap; includes a zero vector (scale 1) and a tiny one."""
    rng = np.random.default_rng(11 + dt)
    T, HK, D, cap, phys0 = 6, 3, 128, 8, 5
    x = (rng.standard_normal((T, HK, D)) * 4).astype(np.float32)
    x[1, 2] = 0.0
    x[3, 0] *= 1e-20
    vb = {0: 4 * D, 1: D, 2: D // 2}[dt]
    q = DA.empty(cap * HK * vb, np.uint8)
    sc = DA.empty(cap * HK)
    ops.kv_write(dt, DA.from_numpy(x), T, HK, D, q, sc, phys0, cap)
    qh = q.numpy().reshape(cap, HK, vb)
    sh = sc.numpy().reshape(cap, HK)
    for t in range(T):
        p = (phys0 + t) % cap
        for h in range(HK):
            want_q, want_s = oracle.kv_write_vec(dt, x[t, h])
            assert np.array_equal(qh[p, h], want_q), (t, h)
            if dt:
                assert np.float32(sh[p, h]) == np.float32(want_s), (t, h)
    if dt:  # host ABI, one vector
        from aero_amd import _lib
        import ctypes
        qb = np.zeros(vb, np.uint8)
        s1 = np.zeros(1, np.float32)
        assert _lib.lib().aero_kv_write_vec(dt, x[0, 0].ctypes.data_as(
            ctypes.POINTER(ctypes.c_float)), D, qb.ctypes.data, s1.ctypes.data_as(
            ctypes.POINTER(ctypes.c_float))) == 1
        wq, ws = oracle.kv_write_vec(dt, x[0, 0])
        assert np.array_equal(qb, wq) and np.float32(s1[0]) == np.float32(ws)


@pytest.mark.parametrize("dt,T,H,HK,D,S", [(1, 3, 32, 8, 128, 1500), (2, 3, 32, 8, 128, 1500),
                                           (1, 40, 14, 2, 64, 700), (2, 1, 14, 2, 64, 3000),
                                           # several 32-key steps a wave (4 a chunk of 512),
                                           # a partial last chunk
                                           (1, 64, 32, 8, 128, 2048), (2, 64, 32, 8, 128, 2048),
                                           (1, 1, 32, 8, 128, 32768), (2, 1, 32, 8, 64, 20000),
                                           # head_dim 256 (the fp32 matrix-core kernel
                                           # reading the codes): decode and prefill
                                           (1, 1, 8, 4, 256, 3000), (2, 1, 8, 4, 256, 3000),
                                           (1, 70, 16, 2, 256, 300), (2, 70, 16, 2, 256, 300)])
def test_attention_over_quantised_cache(hip, oracle, dt, T, H, HK, D, S):
    """Attention reading an int8 / int4 cache (the fp16 matrix-core kernel at
    head dims 64 and 128) equals the oracle's attention over the cache read
    back with the reference's aero_kv_read_vec."""
    rng = np.random.default_rng(23 + dt + T)
    print(f"quantised-cache attention dt={dt} T={T} H={H}/{HK} D={D} S={S}", flush=True)
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    vb = D if dt == 1 else D // 2
    kq, vq = DA.empty(S * HK * vb, np.uint8), DA.empty(S * HK * vb, np.uint8)
    ks, vs = DA.empty(S * HK), DA.empty(S * HK)
    ops.kv_write(dt, DA.from_numpy(k), S, HK, D, kq, ks, 0, S)
    ops.kv_write(dt, DA.from_numpy(v), S, HK, D, vq, vs, 0, S)
    kqh, vqh = kq.numpy().reshape(S * HK, vb), vq.numpy().reshape(S * HK, vb)
    ksh, vsh = ks.numpy(), vs.numpy()
    kd = np.stack([oracle.kv_read_vec(dt, kqh[i], ksh[i], D) for i in range(S * HK)])
    vd = np.stack([oracle.kv_read_vec(dt, vqh[i], vsh[i], D) for i in range(S * HK)])
    kd, vd = kd.reshape(S, HK, D), vd.reshape(S, HK, D)
    qpos = np.arange(S - T, S, dtype=np.int32)
    out = DA.empty((T, H, D))
    ops.attention(DA.from_numpy(q), kq, vq, out, T, H, HK, D, D, S, 0.09,
                  qpos=DA.from_numpy(qpos), kv_dt=dt, k_scale=ks, v_scale=vs)
    want = oracle.attention_tiled(q, kd, vd, 0.09, qpos=qpos)
    assert rel_to_scale(out.numpy(), want) <= RTOL


@pytest.mark.parametrize("dt,D,H,HK,S", [(1, 64, 8, 2, 700), (2, 64, 8, 2, 700),
                                          (1, 128, 32, 8, 6000), (2, 128, 32, 8, 6000),
                                          (1, 256, 8, 4, 700), (2, 256, 8, 4, 700)])
def test_quantised_cache_positions_and_masks(hip, oracle, dt, D, H, HK, S):
    """The integer-cache kernels (fp16 matrix steps at head dims 64 and 128,
    the fp32 matrix-core kernel reading the codes at 256) under arbitrary
    positions: a shuffled cache (700 keys: one 32-key step a wave; 6000 keys:
    chunks of 384, three steps a wave), a query before every key (exact
    zeros), positions past the cache, then the same with a window of 37."""
    rng = np.random.default_rng(11 * dt + D)
    T = 9
    print(f"quantised-cache positions dt={dt} D={D} S={S}", flush=True)
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    vb = D if dt == 1 else D // 2
    kq, vq = DA.empty(S * HK * vb, np.uint8), DA.empty(S * HK * vb, np.uint8)
    ks, vs = DA.empty(S * HK), DA.empty(S * HK)
    ops.kv_write(dt, DA.from_numpy(k), S, HK, D, kq, ks, 0, S)
    ops.kv_write(dt, DA.from_numpy(v), S, HK, D, vq, vs, 0, S)
    kqh, vqh = kq.numpy().reshape(S * HK, vb), vq.numpy().reshape(S * HK, vb)
    ksh, vsh = ks.numpy(), vs.numpy()
    kd = np.stack([oracle.kv_read_vec(dt, kqh[i], ksh[i], D) for i in range(S * HK)])
    vd = np.stack([oracle.kv_read_vec(dt, vqh[i], vsh[i], D) for i in range(S * HK)])
    kd, vd = kd.reshape(S, HK, D), vd.reshape(S, HK, D)
    qpos = np.array([-3, 0, 5, S - 1, 120, 400, 401, S + 300, 2], np.int32)
    kpos = rng.permutation(S).astype(np.int32)
    for window in (0, 37):
        out = DA.empty((T, H, D))
        ops.attention(DA.from_numpy(q), kq, vq, out, T, H, HK, D, D, S, 0.11,
                      qpos=DA.from_numpy(qpos), kpos=DA.from_numpy(kpos), window=window,
                      kv_dt=dt, k_scale=ks, v_scale=vs)
        want = oracle.attention_tiled(q, kd, vd, 0.11, qpos=qpos, kpos=kpos,
                                      window=window or None)
        got = out.numpy()
        assert rel_to_scale(got, want) <= RTOL, window
        assert not got[0].any()


@pytest.mark.parametrize("dt", [1, 2])
@pytest.mark.parametrize("case", ["late_jump", "tiny_block"])
@pytest.mark.parametrize("one_chunk", [False, True])
def test_quantised_cache_scale_ranges(hip, oracle, dt, case, one_chunk):
    """Value vectors in blocks of 1e-30, 1e24, 1, 1e-20 and 3 along the cache
    (value scales 2^-100 .. 2^80), keys of the 1e24 block (and, for
    tiny_block, of every block but 1e-20) pointing away from the queries so
    their weights vanish, and a late key whose score jumps far above the
    running max (late_jump) or an output carried by the 1e-20 block alone
    (tiny_block). The integer-cache kernel keeps its value sums in units of a
    per-step power of two and its probabilities against a reference max that
    moves only on large changes; with one chunk every wave walks ~23 steps in
    one pass and meets each change. Against the oracle's attention over the
    read-back cache."""
    from aero_amd.device import tune_set
    rng = np.random.default_rng(91 + dt + 2 * one_chunk)
    T, H, HK, D, S = 1, 8, 2, 128, 3000
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    mags = np.ones(S, np.float32)
    mags[0:400], mags[400:800], mags[1600:2400], mags[2400:] = 1e-30, 1e24, 1e-20, 3.0
    v = (v * mags[:, None, None]).astype(np.float32)
    qdir = q[0].reshape(HK, H // HK, D).sum(1)
    qdir = qdir / np.linalg.norm(qdir, axis=-1, keepdims=True)
    away = list(range(400, 800)) if case == "late_jump" else \
        list(range(400, 1600)) + list(range(2400, S))
    k[away] = -qdir[None] * 4000.0
    if case == "late_jump":
        k[2990] = qdir * 30.0
    else:
        k[1600:2400] = k[1600:2400] * 0.2 + qdir[None] * 10.0
    vb = D if dt == 1 else D // 2
    kq, vq = DA.empty(S * HK * vb, np.uint8), DA.empty(S * HK * vb, np.uint8)
    ks, vs = DA.empty(S * HK), DA.empty(S * HK)
    ops.kv_write(dt, DA.from_numpy(k.astype(np.float32)), S, HK, D, kq, ks, 0, S)
    ops.kv_write(dt, DA.from_numpy(v), S, HK, D, vq, vs, 0, S)
    kqh, vqh = kq.numpy().reshape(S * HK, vb), vq.numpy().reshape(S * HK, vb)
    ksh, vsh = ks.numpy(), vs.numpy()
    kd = np.stack([oracle.kv_read_vec(dt, kqh[i], ksh[i], D) for i in range(S * HK)])
    vd = np.stack([oracle.kv_read_vec(dt, vqh[i], vsh[i], D) for i in range(S * HK)])
    kd, vd = kd.reshape(S, HK, D), vd.reshape(S, HK, D)
    qpos = np.array([S - 1], np.int32)
    want = oracle.attention_tiled(q, kd, vd, 0.09, qpos=qpos)
    scale = np.abs(want).max()
    if case == "tiny_block":
        assert 1e-24 < scale < 1e-16   # carried by the 1e-20 block
    else:
        assert 0.5 < scale < 20.0      # carried by the late key (3.0 block)
    print(f"scale ranges dt={dt} {case} one_chunk={one_chunk}", flush=True)
    out = DA.empty((T, H, D))
    if one_chunk:
        tune_set("attn_wgs", 1)
    try:
        ops.attention(DA.from_numpy(q), kq, vq, out, T, H, HK, D, D, S, 0.09,
                      qpos=DA.from_numpy(qpos), kv_dt=dt, k_scale=ks, v_scale=vs)
        got = out.numpy()
    finally:
        if one_chunk:
            tune_set("attn_wgs", None)
    assert np.isfinite(got).all()
    assert rel_to_scale(got, want) <= RTOL


@pytest.mark.parametrize("combine4", [1, 0])
@pytest.mark.parametrize("dt,H,HK,D,DV,S", [(0, 32, 8, 128, 128, 4096), (0, 16, 2, 256, 256, 3000),
                                             (0, 14, 2, 64, 48, 2500), (1, 8, 2, 42, 42, 3000),
                                             (1, 32, 8, 128, 128, 9000)])
def test_chunk_merge_kernels(hip, oracle, combine4, dt, H, HK, D, DV, S):
    """Decode over many key chunks: the chunk merge with float4 lanes (value
    widths of a multiple of 4) and the scalar one (attn_combine4=0, and the
    42-wide int8 value rows, which always take it) both equal the oracle."""
    from aero_amd.device import tune_set
    rng = np.random.default_rng(31 + D + S)
    q, k, v = rand_qkv(rng, 1, H, HK, D, DV, S)
    qpos = np.array([S - 1], np.int32)
    print(f"chunk merge combine4={combine4} dt={dt} H={H}/{HK} D={D} DV={DV} S={S}", flush=True)
    if dt == 0:
        kd, vd, args = k, v, {}
    else:
        kq, vq = DA.empty(S * HK * D, np.uint8), DA.empty(S * HK * DV, np.uint8)
        ks, vs = DA.empty(S * HK), DA.empty(S * HK)
        ops.kv_write(dt, DA.from_numpy(k), S, HK, D, kq, ks, 0, S)
        ops.kv_write(dt, DA.from_numpy(v), S, HK, DV, vq, vs, 0, S)
        kqh, vqh = kq.numpy().reshape(S * HK, D), vq.numpy().reshape(S * HK, DV)
        ksh, vsh = ks.numpy(), vs.numpy()
        kd = np.stack([oracle.kv_read_vec(dt, kqh[i], ksh[i], D)
                       for i in range(S * HK)]).reshape(S, HK, D)
        vd = np.stack([oracle.kv_read_vec(dt, vqh[i], vsh[i], DV)
                       for i in range(S * HK)]).reshape(S, HK, DV)
        args = dict(kv_dt=dt, k_scale=ks, v_scale=vs)
    out = DA.empty((1, H, DV))
    dk = DA.from_numpy(k) if dt == 0 else kq
    dv = DA.from_numpy(v) if dt == 0 else vq
    tune_set("attn_combine4", combine4)
    try:
        ops.attention(DA.from_numpy(q), dk, dv, out, 1, H, HK, D, DV, S, 0.11,
                      qpos=DA.from_numpy(qpos), **args)
        got = out.numpy()
    finally:
        tune_set("attn_combine4", None)
    want = oracle.attention_tiled(q, kd, vd, 0.11, qpos=qpos)
    assert rel_to_scale(got, want) <= RTOL


def test_softmax_rows(hip, oracle):
    """Rows of 1..100k values, large and tiny ranges; the flat-vector host ABI."""
    rng = np.random.default_rng(31)
    for rows, cols, s in ((1, 1, 1.0), (3, 7, 50.0), (64, 4096, 3.0), (2, 100000, 10.0)):
        x = (rng.standard_normal((rows, cols)) * s).astype(np.float32)
        dx, dy = DA.from_numpy(x), DA.empty((rows, cols))
        ops.softmax_rows(dx, dy, rows, cols)
        assert rel_to_scale(dy.numpy(), oracle.softmax(x)) <= RTOL
    from aero_amd import tensor_native
    x = (rng.standard_normal(1000) * 5).astype(np.float32)
    xc = x.copy()
    y = tensor_native.softmax(xc)
    # in place on a contiguous float32 input, as engine/tensor_native.py:153-160
    assert np.shares_memory(y, xc)
    assert rel_to_scale(y, oracle.softmax(x)) <= RTOL


def test_attention_decode_full_size(hip, oracle):
    """Llama-3-8B decode at a 16k-token cache (H=32, HK=8, D=128): the key split
    into chunks and their combine against the oracle; and the 512-token causal
    prefill of the same heads."""
    rng = np.random.default_rng(37)
    q, k, v = rand_qkv(rng, 1, 32, 8, 128, 128, 16384)
    got = gpu_attention(q, k, v, 1 / np.sqrt(128), qpos=[16383])
    assert rel_to_scale(got, oracle.attention_tiled(q, k, v, 1 / np.sqrt(128),
                                                    qpos=[16383])) <= RTOL
    q, k, v = rand_qkv(rng, 512, 32, 8, 128, 128, 512)
    got = gpu_attention(q, k, v, 1 / np.sqrt(128))
    assert rel_to_scale(got, oracle.attention_tiled(q, k, v, 1 / np.sqrt(128))) <= RTOL


def _random_attention_cases(n, seed):
    rng = np.random.default_rng(seed)
    cases = []
    for i in range(n):
        dt = int(rng.integers(0, 3))
        D = int(rng.choice([64, 128]))
        HK = int(rng.choice([1, 2, 4, 8]))
        H = HK * int(rng.choice([1, 2, 4, 7, 8]))
        T = int(rng.integers(1, 71))
        S = int(rng.integers(T, 3001))
        window = int(rng.choice([0, 0, int(rng.integers(1, S + 1))]))
        cases.append((i, dt, T, H, HK, D, S, window))
    return cases


@pytest.mark.parametrize("i,dt,T,H,HK,D,S,window", _random_attention_cases(24, 2026))
def test_attention_random_shapes(hip, oracle, i, dt, T, H, HK, D, S, window):
    """Seeded random shapes over every cache type and both matrix-core kernels:
    1-70 queries at the last positions of 1-3000 keys, 1-8 query heads a kv
    head, head dims 64 / 128, with and without a window."""
    rng = np.random.default_rng(100 + i)
    print(f"random attention {i}: dt={dt} T={T} H={H}/{HK} D={D} S={S} window={window}",
          flush=True)
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    qpos = np.arange(S - T, S, dtype=np.int32)
    scale = 1.0 / np.sqrt(D)
    if dt == 0:
        got = gpu_attention(q, k, v, scale, qpos=qpos, window=window)
        want = oracle.attention_tiled(q, k, v, scale, qpos=qpos, window=window or None)
    else:
        vb = D if dt == 1 else D // 2
        kq, vq = DA.empty(S * HK * vb, np.uint8), DA.empty(S * HK * vb, np.uint8)
        ks, vs = DA.empty(S * HK), DA.empty(S * HK)
        ops.kv_write(dt, DA.from_numpy(k), S, HK, D, kq, ks, 0, S)
        ops.kv_write(dt, DA.from_numpy(v), S, HK, D, vq, vs, 0, S)
        kqh, vqh = kq.numpy().reshape(S * HK, vb), vq.numpy().reshape(S * HK, vb)
        ksh, vsh = ks.numpy(), vs.numpy()
        kd = np.stack([oracle.kv_read_vec(dt, kqh[j], ksh[j], D)
                       for j in range(S * HK)]).reshape(S, HK, D)
        vd = np.stack([oracle.kv_read_vec(dt, vqh[j], vsh[j], D)
                       for j in range(S * HK)]).reshape(S, HK, D)
        out = DA.empty((T, H, D))
        ops.attention(DA.from_numpy(q), kq, vq, out, T, H, HK, D, D, S, scale,
                      qpos=DA.from_numpy(qpos), window=window, kv_dt=dt, k_scale=ks,
                      v_scale=vs)
        got = out.numpy()
        want = oracle.attention_tiled(q, kd, vd, scale, qpos=qpos, window=window or None)
    assert rel_to_scale(got, want) <= RTOL


@pytest.fixture
def split_always(hip):
    """attn_split_kernel whatever the sizes."""
    tune_set("attn_split", 2)
    yield
    tune_set("attn_split", None)


@pytest.mark.parametrize("T,H,HK,D,S,window,kpos", [
    (1, 4, 4, 64, 1, 0, False),          # one query, one key
    (32, 4, 1, 64, 129, 0, False),       # 128 vectors exactly, one key past a tile
    (33, 8, 2, 64, 127, 0, True),        # one token past a workgroup, shuffled keys
    (65, 8, 2, 128, 65, 0, False),       # one key past the 64-key tile
    (40, 6, 2, 128, 300, 33, False),     # 3 heads a kv head, a window across tiles
    (70, 16, 2, 128, 190, 64, True),     # window and shuffled keys
    (31, 4, 2, 256, 33, 0, False),       # one key past the 32-key tile
    (90, 8, 4, 256, 200, 50, False),
    (17, 16, 2, 256, 64, 0, True),
])
def test_split_vs_oracle(split_always, oracle, T, H, HK, D, S, window, kpos):
    """The fp16-split kernel at the edges of its tiles; queries that keep no
    key give exact zeros, and blocks of K / V of very different sizes meet."""
    rng = np.random.default_rng(T + H + D + S + window)
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    k[S // 2:] *= 2.0 ** -20              # block exponents that move
    v[S // 3:] *= 2.0 ** 12
    qpos = np.arange(S - T, S, dtype=np.int32)
    if T > 4:
        qpos[0], qpos[1] = -3, S + 100
    kp = rng.permutation(S).astype(np.int32) if kpos else None
    print(f"split attention T={T} H={H} HK={HK} D={D} S={S} window={window}", flush=True)
    scale = -1.0 / np.sqrt(D) if T == 40 else 1.0 / np.sqrt(D)
    got = gpu_attention(q, k, v, scale, qpos=qpos, kpos=kp, window=window)
    want = oracle.attention_tiled(q, k, v, scale, qpos=qpos, kpos=kp, window=window or None)
    assert rel_to_scale(got, want) <= RTOL
    if T > 4:
        assert not got[0].any()


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 3.0e38])
@pytest.mark.parametrize("where", ["q", "k", "v"])
def test_split_non_finite(split_always, oracle, D, bad, where):
    """A non-finite or huge operand touches the queries that keep it and no
    other: those agree with the oracle's result without it. The touched ones
    are the fp32-step kernel's where its row is finite; where it is not, the
    split's is not either, and each element is the NaN or infinity that the
    fp32-step kernel gives it."""
    rng = np.random.default_rng(D)
    T, H, HK, S = 70, 4, 2, 100
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    qpos = np.arange(S - T, S, dtype=np.int32)
    scale = 1.0 / np.sqrt(D)
    want = oracle.attention_tiled(q, k, v, scale, qpos=qpos)
    {"q": q, "k": k, "v": v}[where][60, 1, 5] = bad
    print(f"split attention D={D} {where} = {bad}", flush=True)
    got = gpu_attention(q, k, v, scale, qpos=qpos)
    touched = np.zeros((T, H), bool)
    if where == "q":
        touched[60, 1] = True
    else:
        touched[qpos >= 60, 2:] = True   # the heads of kv head 1
    assert rel_to_scale(got[~touched], want[~touched]) <= RTOL
    tune_set("attn_split", 0)
    general = gpu_attention(q, k, v, scale, qpos=qpos)
    tune_set("attn_split", 2)
    for t, h in np.argwhere(touched):
        if np.isfinite(general[t, h]).all():
            assert rel_to_scale(got[t, h].astype(np.float64),
                                general[t, h].astype(np.float64)) <= RTOL
        else:
            assert np.array_equal(np.isnan(got[t, h]), np.isnan(general[t, h])), (t, h)
            inf = np.isinf(general[t, h])
            assert np.array_equal(got[t, h][inf], general[t, h][inf]), (t, h)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("T,S,window,turned,up", [
    (8, 8, 0, False, 40),      # a few keys
    (100, 100, 3, False, 40),  # queries that keep none of the large rows
    (100, 100, 3, True, 40),   # the same, keys stored last to first
    (100, 100, 3, False, 24),
    (100, 100, 3, False, 14),
])
def test_split_value_rows(split_always, oracle, D, T, S, window, turned, up):
    """Every fourth row of V 2^up above the others, so that every block of keys
    that shares a scale holds both: a query that keeps small rows alone gets
    them whole (each query against its own scale)."""
    rng = np.random.default_rng(D + T + up)
    q, k, v = rand_qkv(rng, T, 4, 2, D, D, S)
    v[3::4] *= 2.0 ** up
    qpos = np.arange(S - T, S, dtype=np.int32)
    kpos = np.arange(S, dtype=np.int32)[::-1] if turned else None
    scale = 1.0 / np.sqrt(D)
    print(f"split attention D={D} T={T} S={S} V rows 2^{up} apart", flush=True)
    got = gpu_attention(q, k, v, scale, qpos=qpos, kpos=kpos, window=window)
    want = oracle.attention_tiled(q, k, v, scale, qpos=qpos, kpos=kpos, window=window or None)
    for t in range(T):
        assert rel_to_scale(got[t], want[t]) <= RTOL, t


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("up", [12, 18, 24, 60])
def test_split_value_channels(split_always, D, up):
    """A dimension of V 2^up above the others, with dimensions of zeros (a
    padded head) among these: each is as good against its own scale as without
    it (2-norm against float64 2.6e-7 to 4e-7 on either kernel; 2^-25 of the
    dimension's scale more at the ratio that the split takes)."""
    rng = np.random.default_rng(D + up)
    T, H, HK, S = 150, 4, 2, 150
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    v[:, 1, 5] *= 2.0 ** up
    v[:, :, D - 7:] = 0.0
    scale = 1.0 / np.sqrt(D)
    print(f"split attention D={D} a V channel 2^{up} up", flush=True)
    got = gpu_attention(q, k, v, scale, qpos=np.arange(T, dtype=np.int32)).astype(np.float64)
    mask = np.arange(S)[None] > np.arange(T)[:, None]
    for h in range(H):
        s = q[:, h].astype(np.float64) @ k[:, h // 2].T.astype(np.float64) * np.float32(scale)
        s[mask] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        want = p @ v[:, h // 2].astype(np.float64) / p.sum(1, keepdims=True)
        assert not got[:, h, D - 7:].any()
        err = np.linalg.norm(got[:, h] - want, axis=0)[:D - 7]
        assert (err <= 1e-6 * np.linalg.norm(want, axis=0)[:D - 7]).all(), err.max()


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("e", [10, 12, 13, 14])
def test_split_score_products(split_always, D, e):
    """Large q values against small K values whose parts drop a remainder of
    one sign, next to K values (met by zeros of q) that set the scale, the
    maxima's product just below 2^e log2 units: at most D / 2 * 2^(e - 39) off
    in the scores, D / 2 * 2^-27 where the split takes them (e <= 12), so that
    times ln 2 / 2 in a result that is a mean of zeros and ones near 1/2 and
    twice that relative to it; the kernels' own 1e-7 on top."""
    rng = np.random.default_rng(0)
    S, T = 64, 40
    scale = 1.0 / np.sqrt(D)
    up = 2.0 ** (e - e // 2)
    sign = np.where(rng.permutation(S) % 2 == 0, 1.0, -1.0)
    q = np.zeros((T, 1, D), np.float32)
    q[..., :D // 2] = 0.99 * 2.0 ** (e // 2) / (scale * np.log2(np.e))
    k = np.zeros((S, 1, D), np.float32)
    k[..., D // 2:] = 0.99 * up
    # (in units of up / 2^14: 2^-5 and up to 2^-18 more, 0.48 of the last fp16 bit over)
    k[..., :D // 2] = (2.0 ** -5 + rng.integers(-64, 64, (S, 1, D // 2)) * 2.0 ** -24 +
                       sign[:, None, None] * 0.48 * 2.0 ** -24) * up / 2 ** 14
    v = np.zeros((S, 1, D), np.float32)
    v[sign > 0] = 1.0
    print(f"split attention D={D} products 2^{e}", flush=True)
    got = gpu_attention(q, k, v, scale, qpos=np.full(T, S, np.int32))[:, 0].astype(np.float64)
    s = q[:, 0].astype(np.float64) @ k[:, 0].T.astype(np.float64) * np.float32(scale)
    p = np.exp(s - s.max(1, keepdims=True))
    want = p @ v[:, 0].astype(np.float64) / p.sum(1, keepdims=True)
    assert np.abs(got - want).max() <= (D / 2 * 2.0 ** -27 * np.log(2) + 1e-7) * np.abs(want).max()


@pytest.mark.parametrize("T,H,HK,D,S,window,kpos", [
    (512, 16, 4, 64, 512, 0, False),
    (500, 8, 2, 128, 700, 300, False),    # a partial last tile, a window
    (300, 8, 2, 128, 300, 0, True),
    (509, 8, 4, 256, 509, 0, False),
])
def test_split_redo(split_always, T, H, HK, D, S, window, kpos):
    """Queries and keys whose products pass what the fp16 parts carry: the
    workgroups do such rows again on fp32 matrix steps, with the sums of the
    fp32-step kernel over one chunk (the same partial sums, merged in the same
    order but for the sum of the probabilities, an fp32 rounding: 1e-7), in a
    small multiple of its time (on MI355X 1.1 to 3 times, by how much of the
    chip the workgroups fill; 26 to 65 times with a row at a time)."""
    rng = np.random.default_rng(T + D)
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    for x, up, down in ((q, 3, 7), (k, 7, 3)):
        x[..., up] *= 256.0
        x[..., down] /= 256.0
    dq, dk, dv = DA.from_numpy(q), DA.from_numpy(k), DA.from_numpy(v)
    qpos = DA.from_numpy(np.arange(S - T, S, dtype=np.int32))
    kp = DA.from_numpy(rng.permutation(S).astype(np.int32)) if kpos else None
    print(f"split attention redo T={T} H={H} HK={HK} D={D} S={S}", flush=True)
    res, ms = [], []
    for use in (0, 2):
        tune_set("attn_split", use)
        tune_set("attn_wgs", 1 if use == 0 else None)    # one chunk
        out = DA.empty((T, H, D))

        def call():
            ops.attention(dq, dk, dv, out, T, H, HK, D, D, S, 1.0 / np.sqrt(D), qpos=qpos,
                          kpos=kp, window=window)
        call()
        best = []
        for _ in range(5):
            a, b = Event(), Event()
            a.record()
            call()
            b.record()
            b.synchronize()
            best.append(a.elapsed_ms(b))
        res.append(out.numpy().astype(np.float64))
        ms.append(min(best))
    assert np.isfinite(res[1]).all()
    assert np.linalg.norm(res[1] - res[0]) <= 1e-7 * np.linalg.norm(res[0])
    assert ms[1] <= 10 * ms[0], ms


@pytest.mark.parametrize("T,H,HK,D,S,window,kpos,split", [
    (255, 64, 8, 128, 255, 0, False, True),      # 128 workgroups, 128 keys a query
    (239, 64, 8, 128, 239, 0, False, False),     # 120
    (508, 32, 8, 64, 508, 0, False, True),       # 128 over 255
    (600, 32, 8, 64, 700, 128, False, True),     # 152 in a window of 128
    (508, 32, 8, 64, 700, 128, False, False),    # 128 in a window of 128
    (480, 32, 8, 64, 480, 0, False, False),      # 120 over 241
    (255, 32, 8, 64, 1300, 0, False, False),     # 64 over 1173
    (288, 32, 8, 64, 1300, 0, False, True),      # 72
    (284, 32, 8, 128, 1100, 0, False, False),    # 72 over 959
    (600, 14, 2, 64, 1700, 0, True, False),      # 66, shuffled keys
    (700, 16, 2, 256, 1700, 0, True, False),     # 88 over 1350, shuffled keys
    (700, 16, 2, 256, 1700, 0, False, True),
    (1024, 16, 2, 256, 1024, 300, True, True),   # 128, shuffled keys in a window
])
def test_split_rule_matches_general(hip, T, H, HK, D, S, window, kpos, split):
    """Calls on both sides of the rule's lines run the kernel that they are
    meant to (both are deterministic: their bits tell) and agree with the
    other, a window, shuffled keys and cached prefixes among them."""
    rng = np.random.default_rng(3)
    q, k, v = rand_qkv(rng, T, H, HK, D, D, S)
    qpos = np.arange(S - T, S, dtype=np.int32)
    kp = rng.permutation(S).astype(np.int32) if kpos else None
    print(f"attention rule T={T} H={H} HK={HK} D={D} S={S} window={window}", flush=True)
    out = []
    for use in (None, 0, 2):
        tune_set("attn_split", use)
        try:
            out.append(gpu_attention(q, k, v, 1.0 / np.sqrt(D), qpos=qpos, kpos=kp,
                                     window=window))
        finally:
            tune_set("attn_split", None)
    assert not bits_equal(out[1], out[2])
    assert bits_equal(out[0], out[2 if split else 1])
    assert rel_to_scale(out[2], out[1]) <= RTOL


def test_split_output_past_2_32_elements(hip, oracle):
    """An output of more than 2^32 elements (the first rows, the last ones and
    those around the 2^32nd element), over 8 keys: nothing wraps onto the
    first rows."""
    H, D, S = 33, 128, 8
    T = 2 ** 32 // (H * D) + 500
    rng = np.random.default_rng(5)
    k = rng.standard_normal((S, H, D)).astype(np.float32)
    v = rng.standard_normal((S, H, D)).astype(np.float32)
    edge = 2 ** 32 // (H * D)
    spots = [0, 40, edge - 6, edge + 1, T - 5]
    q, out = DA.empty((T, H, D)), DA.empty((T, H, D))    # 17 GB each
    row = H * D * 4
    ops.fill_f32(q, 0.0)
    ops.fill_f32(out, -7.0)
    part = {}
    for t in spots:
        part[t] = rng.standard_normal((5, H, D)).astype(np.float32)
        q.view((5, H, D), offset_bytes=t * row).copy_from(part[t])
    print(f"split attention T={T} H={H} D={D} S={S}", flush=True)
    ops.attention(q, DA.from_numpy(k), DA.from_numpy(v), out, T, H, H, D, D, S, 0.125)
    for t in spots:
        got = out.view((5, H, D), offset_bytes=t * row).numpy()
        want = oracle.attention_tiled(part[t], k, v, 0.125, qpos=np.arange(t, t + 5, dtype=np.int32))
        assert rel_to_scale(got, want) <= RTOL, t
    q.free()
    out.free()
