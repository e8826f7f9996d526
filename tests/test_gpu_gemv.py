"""GPU parity: the quantised GEMV / small-batch GEMM (aero_hip_matvec) and the
reference-compatible aero_matvec / aero_matmul, against the oracle's
restatement of src/kernels.cpp:78-250,497-538 and the reference's own outputs
(tests/golden/ref_vectors.npz). The GPU sums in a different order from the
reference's serial loops, so results agree to a tolerance relative to the
output's scale: 1e-5 (observed ~1e-7), the reference's own RTOL for fp32 ops
(tests/test_transformer_native.py:34-37).
"""
import numpy as np
import pytest

from conftest import RTOL, golden, rel_to_scale
from aero_amd import native, ops
from aero_amd import workloads as W
from aero_amd.device import DeviceArray as DA, Event, Plan, tune_set

pytestmark = pytest.mark.gpu

TYPES = [W.Q8_0, W.Q4_K, W.Q5_K, W.Q6_K, W.IQ4_XS]


def gpu_matvec(t, w, X, n_rows):
    X = np.atleast_2d(np.ascontiguousarray(X, np.float32))
    T, n_cols = X.shape
    y = DA.empty((T, n_rows))
    ops.matvec(t, DA.from_numpy(w), DA.from_numpy(X), y, n_rows, n_cols, T)
    return y.numpy()


@pytest.mark.parametrize("t", TYPES)
def test_matvec_golden(hip, t):
    """The reference's own matvec / matmul outputs (24 x 512, 3 tokens)."""
    g = golden("ref_vectors.npz")
    w, X = g[f"mv{t}_w"], g[f"mv{t}_x"]
    n_rows = g[f"mv{t}_y"].size
    assert rel_to_scale(gpu_matvec(t, w, X[:1], n_rows)[0], g[f"mv{t}_y"]) <= RTOL
    assert rel_to_scale(gpu_matvec(t, w, X, n_rows), g[f"mm{t}_y"]) <= RTOL


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("n_rows,n_cols,n_tok", [
    (1, 256, 1), (37, 1024, 1), (4096, 4096, 1), (1000, 14336, 1),   # decode shapes
    (4103, 4096, 2), (513, 2048, 3), (130, 4096, 8), (67, 1024, 13),  # token groups
    (300, 14336, 5), (64, 8192, 4),  # rows of several 4096-column steps, token groups
    # 5-24 tokens: Q4_K / Q5_K take the split GEMM (5+ tokens from 32M
    # weights, 12+ from 8M, else 16+), the other types the GEMV
    (8200, 1024, 8), (100, 2048, 16), (33, 512, 24), (8192, 4096, 5),
])
def test_matvec_vs_oracle(hip, oracle, t, n_rows, n_cols, n_tok):
    rng = np.random.default_rng(n_rows * 31 + n_cols + n_tok + t)
    bv, bb = W.BLOCK[t]
    w = W.make_table(t, n_rows * n_cols // bv, rng)
    X = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    print(f"matvec type={t} rows={n_rows} cols={n_cols} tokens={n_tok}", flush=True)
    got = gpu_matvec(t, w, X, n_rows)
    want = oracle.matmul(t, w, X, n_rows)
    assert rel_to_scale(got, want) <= RTOL


@pytest.mark.parametrize("n_rows,n_cols,n_tok", [
    (896, 896, 1), (128, 896, 3), (4864, 896, 1), (127, 896, 2), (64, 640, 5),
])
def test_matvec_q8_0_rows_of_8_bytes(hip, oracle, n_rows, n_cols, n_tok):
    """Q8_0 rows of a multiple of 8 bytes but not of 16 (896 columns: 952
    bytes, Qwen2-0.5B; 640: 680) alternate between 16- and 8-byte aligned
    starts: the 64-column lane kernel places each lane's 16-byte window from
    the absolute address. With an odd row count the last row ends 8 bytes
    short of a 16-byte boundary, past the weights: that matrix takes the
    word kernel. Both match the oracle."""
    t = W.Q8_0
    rng = np.random.default_rng(n_rows + n_cols + n_tok)
    w = W.make_table(t, n_rows * n_cols // 32, rng)
    X = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    print(f"matvec Q8_0 rows={n_rows} cols={n_cols} tokens={n_tok}", flush=True)
    assert rel_to_scale(gpu_matvec(t, w, X, n_rows), oracle.matmul(t, w, X, n_rows)) <= RTOL


@pytest.mark.parametrize("t", [W.Q8_0, W.Q6_K])
def test_matvec_rows_off_word_boundary(hip, oracle, t):
    """Row sizes that are not a multiple of 4 bytes (Q8_0 with 45 blocks per row,
    Q6_K with 5): every other row starts 2 bytes past a 4-byte word."""
    rng = np.random.default_rng(61 + t)
    bv, bb = W.BLOCK[t]
    nb = 45 if t == W.Q8_0 else 5
    n_rows, n_cols = 301, nb * bv
    assert (nb * bb) % 4 == 2
    w = W.make_table(t, n_rows * nb, rng)
    X = rng.standard_normal((3, n_cols)).astype(np.float32)
    assert rel_to_scale(gpu_matvec(t, w, X, n_rows), oracle.matmul(t, w, X, n_rows)) <= RTOL


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("n_rows,n_cols,n_tok", [
    (100, 1024, 40), (130, 2048, 33), (257, 4096, 100), (64, 14336, 64),
])
def test_matmul_many_tokens_vs_oracle(hip, oracle, t, n_rows, n_cols, n_tok):
    """32 or more tokens take the matrix-core GEMM (64 x 64 tiles, partial
    row and token tiles, rows of 1 to 56 blocks)."""
    rng = np.random.default_rng(n_rows * 17 + n_cols + n_tok + t)
    bv, bb = W.BLOCK[t]
    w = W.make_table(t, n_rows * n_cols // bv, rng)
    X = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    print(f"matmul type={t} rows={n_rows} cols={n_cols} tokens={n_tok}", flush=True)
    got = gpu_matvec(t, w, X, n_rows)
    want = oracle.matmul(t, w, X, n_rows)
    assert rel_to_scale(got, want) <= RTOL


def test_matmul_prefill_size_matches_gemv(hip):
    """At Llama-3-8B FFN size with 512 tokens (14336 x 4096 Q4_K, the prefill
    shape), every token's GEMM row equals that token's GEMV (one-token launch)
    to the tolerance; sampled tokens cover every 64-token tile."""
    rng = np.random.default_rng(91)
    n_rows, n_cols, n_tok = 14336, 4096, 512
    w = W.make_table(W.Q4_K, n_rows * n_cols // 256, rng)
    X = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    Y = gpu_matvec(W.Q4_K, w, X, n_rows)
    for i in (0, 63, 64, 200, 383, 511):
        assert rel_to_scale(Y[i], gpu_matvec(W.Q4_K, w, X[i], n_rows)[0]) <= RTOL


def test_matvec_linearity_at_full_size(hip):
    """At Llama-3-8B FFN-down size (4096 x 14336 Q4_K): W(a*x1 + x2) equals
    a*W(x1) + W(x2) to the tolerance, and a zero x gives exactly zero."""
    rng = np.random.default_rng(71)
    n_rows, n_cols = 4096, 14336
    w = W.make_table(W.Q4_K, n_rows * n_cols // 256, rng)
    x1, x2 = rng.standard_normal((2, n_cols)).astype(np.float32)
    a = np.float32(0.75)
    X = np.stack([x1, x2, a * x1 + x2, np.zeros(n_cols, np.float32)])
    Y = gpu_matvec(W.Q4_K, w, X, n_rows).astype(np.float64)
    assert rel_to_scale(Y[2], a * Y[0] + Y[1]) <= RTOL
    assert not Y[3].any()


def test_host_abi_matvec_matmul(hip, oracle):
    """engine/native.py-shaped calls (host arrays, bytes) and the reference's
    refusals (tests/test_kernels.cpp:242-250)."""
    rng = np.random.default_rng(81)
    for t in TYPES:
        bv, bb = W.BLOCK[t]
        n_rows, n_cols = 29, 4 * 256
        w = W.make_table(t, n_rows * n_cols // bv, rng)
        x = rng.standard_normal(n_cols).astype(np.float32)
        X = rng.standard_normal((5, n_cols)).astype(np.float32)
        y = native.matvec(t, w.tobytes(), x)
        assert y.shape == (n_rows,)
        assert rel_to_scale(y, oracle.matvec(t, w, x, n_rows)) <= RTOL
        Y = native.matmul(t, bytearray(w.tobytes()), X)
        assert Y.shape == (5, n_rows)
        assert rel_to_scale(Y, oracle.matmul(t, w, X, n_rows)) <= RTOL
    with pytest.raises(ValueError):
        native.matvec(W.F32, bytes(64), np.zeros(16, np.float32))
    with pytest.raises(ValueError):
        native.matvec(W.Q4_K, bytes(144 * 4), np.zeros(255, np.float32))


@pytest.mark.parametrize("t", [W.Q4_K, W.Q8_0, W.Q6_K, W.IQ4_XS, W.Q5_K])
@pytest.mark.parametrize("n_rows,n_cols", [(1, 2048), (3, 1024), (37, 2048), (129, 512)])
@pytest.mark.parametrize("n_tok", [1, 2, 4])
def test_matvec_half_wave_rows(hip, oracle, t, n_rows, n_cols, n_tok):
    """Rows of at most 2048 columns, one a half-wave: odd row counts leave the
    last wave's upper half on a clamped row whose sum is not stored, and rows
    of 512 columns use 8 of a half-wave's 32 column slots."""
    rng = np.random.default_rng(n_rows * 7 + n_cols + n_tok + t)
    w = W.make_table(t, n_rows * n_cols // W.BLOCK[t][0], rng)
    X = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    got = gpu_matvec(t, w, X, n_rows)
    assert rel_to_scale(got, oracle.matmul(t, w, X, n_rows)) <= RTOL


@pytest.mark.parametrize("n_tok", [1, 3])
def test_norm_matvec_half_wave_odd_rows(hip, oracle, n_tok):
    """The fused decode GEMV over three matrices of odd row counts and 2048
    columns (a row a half-wave), with the RMSNorm in its prologue."""
    t, n_cols, rows = W.Q4_K, 2048, [37, 5, 1]
    rng = np.random.default_rng(61 + n_tok)
    ws = [W.make_table(t, r * n_cols // 256, rng) for r in rows]
    x = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(n_cols)).astype(np.float32)
    ys = [DA.empty((n_tok, r)) for r in rows]
    ops.norm_matvec(t, [DA.from_numpy(w) for w in ws], DA.from_numpy(x), ys, rows, n_cols,
                    n_tok, norm_w=DA.from_numpy(nw), eps=1e-5)
    h = oracle.rmsnorm_rows(x, nw, 1e-5)
    for w, r, y in zip(ws, rows, ys):
        assert rel_to_scale(y.numpy(), oracle.matmul(t, w, h, r)) <= RTOL


@pytest.mark.parametrize("tile", range(1, 8))
@pytest.mark.parametrize("n_rows,n_cols,n_tok", [
    (1, 32, 5),        # one block a row: seven of the eight waves have none
    (17, 96, 17),      # an odd block count: rows start 2 bytes off a dword
    (65, 896, 64),     # one row past four tiles, whole token tiles
    (130, 4864, 65),   # one token past four tiles
    (33, 544, 6),
])
def test_gemm_q8_tiles(hip, oracle, n_rows, n_cols, n_tok, tile):
    """gemm_q8_kernel's tiles at their edges (split=False: no workspace)."""
    rng = np.random.default_rng(n_rows + n_cols + n_tok)
    w = W.make_table(W.Q8_0, n_rows * n_cols // 32, rng)
    X = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    X *= np.exp2(rng.integers(-30, 30, (n_tok, 1))).astype(np.float32)
    y = DA.empty((n_tok, n_rows))
    print(f"gemm_q8 tile={tile} rows={n_rows} cols={n_cols} tokens={n_tok}", flush=True)
    tune_set("gemm_q8_tile", tile)
    try:
        ops.matvec(W.Q8_0, DA.from_numpy(w), DA.from_numpy(X), y, n_rows, n_cols, n_tok,
                   split=False)
    finally:
        tune_set("gemm_q8_tile", None)
    want = oracle.matmul(W.Q8_0, w, X, n_rows)
    for t in range(n_tok):                # a token's scale is its own
        assert rel_to_scale(y.numpy()[t], want[t]) <= RTOL


def test_gemm_q8_non_finite(hip, oracle):
    """An infinity or NaN in x reaches its token only, an infinity with the
    sign that the exact product has."""
    rng = np.random.default_rng(9)
    n_rows, n_cols, n_tok = 40, 896, 20
    w = W.make_table(W.Q8_0, n_rows * n_cols // 32, rng)
    X = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    clean = oracle.matmul(W.Q8_0, w, X, n_rows)
    X[3, 100], X[7, 5], X[11, 800] = np.inf, -np.inf, np.nan
    y = DA.empty((n_tok, n_rows))
    ops.matvec(W.Q8_0, DA.from_numpy(w), DA.from_numpy(X), y, n_rows, n_cols, n_tok, split=False)
    got = y.numpy()
    with np.errstate(all="ignore"):
        want = oracle.matmul(W.Q8_0, w, X, n_rows)
    keep = [t for t in range(n_tok) if t not in (3, 7, 11)]
    assert rel_to_scale(got[keep], clean[keep]) <= RTOL
    assert np.isnan(got[11]).all()
    for t in (3, 7):
        assert np.array_equal(np.isnan(got[t]), np.isnan(want[t]))
        assert np.array_equal(np.sign(got[t]), np.sign(want[t]), equal_nan=True)


@pytest.mark.parametrize("tile", range(1, 8))
@pytest.mark.parametrize("e", [-140, -121, -113, 110, 122, 126])
def test_gemm_q8_far_x(hip, tile, e):
    """x near either end of fp32's range against float64: every other token's
    values are 2^e (ordinary tokens between them, and an ordinary group of 8
    columns in each), d such that no result leaves that range. x, codes and d are exact; a step's sum of 32 and 28
    such steps leave 60 roundings of 2^-24 of the sum of magnitudes at most."""
    rng = np.random.default_rng(tile)
    n_rows, n_cols, n_tok = 70, 896, 66
    d = 2.0 ** -20 if e > 0 else 2.0 ** 10
    code = rng.integers(-127, 128, (n_rows, n_cols // 32, 32), dtype=np.int8)
    raw = np.empty((n_rows, n_cols // 32, 34), np.uint8)
    raw[..., :2] = np.full((n_rows, n_cols // 32, 1), d, np.float16).view(np.uint8)
    raw[..., 2:] = code.view(np.uint8)
    X = rng.standard_normal((n_tok, n_cols)).clip(-3.9, 3.9).astype(np.float32)
    far = np.arange(n_tok) % 2 == 1
    X[far] = np.ldexp(X[far], e - 1 if e == 126 else e)
    X[far, 40:48] = rng.standard_normal((far.sum(), 8))
    y = DA.empty((n_tok, n_rows))
    print(f"gemm_q8 tile={tile} x 2^{e}", flush=True)
    tune_set("gemm_q8_tile", tile)
    try:
        ops.matvec(W.Q8_0, DA.from_numpy(raw.reshape(-1)), DA.from_numpy(X), y, n_rows, n_cols,
                   n_tok, split=False)
    finally:
        tune_set("gemm_q8_tile", None)
    w = code.astype(np.float64).reshape(n_rows, n_cols) * d
    want = X.astype(np.float64) @ w.T
    size = np.abs(X.astype(np.float64)) @ np.abs(w.T)
    got = y.numpy().astype(np.float64)
    assert np.isfinite(got).all()
    assert (np.abs(got - want) <= 60 * 2.0 ** -24 * size).all()
    if e < 0:        # without the ordinary columns a tiny token stands alone
        X[far, 40:48] = np.ldexp(X[far, 40:48], e)
        want = X.astype(np.float64) @ w.T
        tune_set("gemm_q8_tile", tile)
        try:
            ops.matvec(W.Q8_0, DA.from_numpy(raw.reshape(-1)), DA.from_numpy(X), y, n_rows,
                       n_cols, n_tok, split=False)
        finally:
            tune_set("gemm_q8_tile", None)
        got = y.numpy().astype(np.float64)
        lim = np.maximum(60 * 2.0 ** -24 * (np.abs(X.astype(np.float64)) @ np.abs(w.T)),
                         30 * 2.0 ** -149)
        assert (np.abs(got - want) <= lim).all()


@pytest.mark.parametrize("n_rows,n_cols,n_tok", [(896, 4864, 16), (896, 4864, 100),
                                                 (1024, 4096, 12), (1024, 4096, 13),
                                                 (512, 2048, 5), (130, 5120, 5), (130, 2304, 5)])
def test_q8_routes_agree(hip, oracle, n_rows, n_cols, n_tok):
    """Q8_0 calls on both sides of the lines between GEMV, gemm_q8_kernel and
    the split GEMM, with and without the workspace."""
    rng = np.random.default_rng(n_rows + n_cols + n_tok)
    w = W.make_table(W.Q8_0, n_rows * n_cols // 32, rng)
    X = rng.standard_normal((n_tok, n_cols)).astype(np.float32)
    want = oracle.matmul(W.Q8_0, w, X, n_rows)
    dw, dx, y = DA.from_numpy(w), DA.from_numpy(X), DA.empty((n_tok, n_rows))
    for split in (True, False):
        ops.matvec(W.Q8_0, dw, dx, y, n_rows, n_cols, n_tok, split=split)
        assert rel_to_scale(y.numpy(), want) <= RTOL


@pytest.mark.parametrize("n_rows,n_cols,n_tok", [
    (11008, 2816, 12), (4864, 3328, 10), (11008, 4864, 4), (4864, 7424, 77),   # workspace
    (896, 4864, 16), (4864, 2816, 12),
    (11008, 2048, 5), (896, 8192, 5), (128, 28672, 8), (896, 4864, 5), (4864, 896, 5),
])
def test_q8_route_is_no_slow_one(hip, n_rows, n_cols, n_tok):
    """A Q8_0 call with a workspace takes no route that is much slower than
    another one it could take (GEMV, gemm_q8_kernel, the split GEMM), one
    without none that is much slower than the GEMV (measured within 1.15; calls
    sent to a wrong one took 1.4 to 2.5 times)."""
    rng = np.random.default_rng(1)
    dw = DA.from_numpy(W.make_table(W.Q8_0, n_rows * n_cols // 32, rng))
    dx = DA.from_numpy(rng.standard_normal((n_tok, n_cols)).astype(np.float32))
    y = DA.empty((n_tok, n_rows))
    print(f"Q8_0 routes {n_rows} x {n_cols}, {n_tok} tokens", flush=True)

    def us(split, **tunes):
        for key, value in tunes.items():
            tune_set(key, value)
        try:
            plan = Plan()
            with plan:
                for _ in range(10):
                    ops.matvec(W.Q8_0, dw, dx, y, n_rows, n_cols, n_tok, split=split)
        finally:
            for key in tunes:
                tune_set(key, None)
        best = []
        for _ in range(6):
            a, b = Event(), Event()
            a.record()
            plan.launch()
            b.record()
            b.synchronize()
            best.append(a.elapsed_ms(b) * 100)
        plan.destroy()
        return min(best)

    gemv, gemm = us(False, gemm_min_tokens=1000), us(False, gemm_min_tokens=1)
    split = us(True, gemm_q8_split=0, gemm_min_tokens=1000)
    own, own_ws = us(False), us(True)
    assert own <= 1.3 * gemv, (own, gemv, gemm)
    assert own_ws <= 1.3 * min(gemv, gemm, split), (own_ws, gemv, gemm, split)
