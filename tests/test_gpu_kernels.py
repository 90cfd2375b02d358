"""Kernel-level parity: HIP path (through the C ABI) vs the CPU oracle.

Bars: dequantisation bit-exact; f32 path within 1e-5 relative L2 of the
oracle's f32 arithmetic; f16 path (f16 operands, f32 accumulation) within
2e-3 relative L2 for a single GEMM.
"""
import numpy as np
import pytest

import oracle
import pk_model as pm
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _rng(seed=7):
    return np.random.default_rng(seed)


@pytest.mark.parametrize("gtype,n", [(pm.GGML_Q8_0, 32 * 1000), (pm.GGML_Q4_K, 256 * 300),
                                     (pm.GGML_F16, 4096)])
def test_dequantize_bit_exact(gpu, stream, gtype, n):
    rng = _rng()
    if gtype == pm.GGML_Q8_0:
        raw = pm.synth_q8_0(rng, n)
    elif gtype == pm.GGML_Q4_K:
        raw = pm.synth_q4_k(rng, n)
    else:
        raw = rng.normal(0, 1, n).astype(np.float16).view(np.uint16)
    print(f"[dequant] type={gtype} n={n}", flush=True)
    ref = oracle.dequantize(gtype, raw, n)
    d_raw = gpu.DeviceArray.from_numpy(raw.view(np.uint8), stream)
    out = gpu.DeviceArray((n,), np.float32)
    gpu.dequantize(gtype, d_raw, n, out, stream)
    got = out.numpy(stream)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


def _weights(gtype, N, K, rng):
    if gtype == pm.GGML_F32:
        w = rng.normal(0, 0.05, (N, K)).astype(np.float32)
        return w, w
    if gtype == pm.GGML_F16:
        h = rng.normal(0, 0.05, (N, K)).astype(np.float16)
        return h.view(np.uint16), h.astype(np.float32)
    raw = pm.synth_q8_0(rng, N * K) if gtype == pm.GGML_Q8_0 else pm.synth_q4_k(rng, N * K)
    return raw, oracle.dequantize(gtype, raw, N * K).reshape(N, K)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("gtype", [pm.GGML_F32, pm.GGML_F16, pm.GGML_Q8_0, pm.GGML_Q4_K])
@pytest.mark.parametrize("M,N,K", [(77, 96, 256), (300, 200, 512), (1, 64, 256), (130, 1030, 768)])
def test_linear(gpu, stream, prec, gtype, M, N, K):
    rng = _rng(M + N + K)
    raw, wf = _weights(gtype, N, K, rng)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 0.1, N).astype(np.float32)
    print(f"[linear] prec={prec} type={gtype} M={M} N={N} K={K}", flush=True)
    ref = oracle.linear(x, wf, b)
    dx = gpu.DeviceArray.from_numpy(x, stream)
    db = gpu.DeviceArray.from_numpy(b, stream)
    dy = gpu.DeviceArray((M, N), np.float32)
    gpu.linear(prec, gtype, N, K, raw, dx, M, dy, db, stream)
    got = dy.numpy(stream)
    err = rel_l2(got, ref)
    tol = 1e-5 if prec == 0 else 2e-3
    assert err < tol, err


@pytest.mark.parametrize("M,D", [(1, 64), (257, 512), (2000, 1024), (33, 640)])
def test_layernorm(gpu, stream, M, D):
    rng = _rng(M * D)
    x = (rng.normal(0, 2, (M, D)) + rng.normal(0, 3, (M, 1))).astype(np.float32)
    g = (1 + rng.normal(0, 0.1, D)).astype(np.float32)
    b = rng.normal(0, 0.1, D).astype(np.float32)
    ref = oracle.layer_norm(x, g, b)
    dx, dg, db = (gpu.DeviceArray.from_numpy(a, stream) for a in (x, g, b))
    dy = gpu.DeviceArray((M, D), np.float32)
    gpu.layernorm(dx, dg, db, dy, M, D, 1e-5, stream)
    got = dy.numpy(stream)
    assert rel_l2(got, ref) < 1e-6
    assert np.abs(got - ref).max() < 1e-5


@pytest.mark.parametrize("T,D", [(1, 64), (125, 1024), (375, 512), (26, 512)])
def test_rel_pos_encoding(gpu, stream, T, D):
    ref = oracle.rel_pos_encoding(T, D)
    out = gpu.DeviceArray((2 * T - 1, D), np.float32)
    gpu.rel_pos_encoding(T, D, out, stream)
    got = out.numpy(stream)
    # f64 sin/cos then one rounding to f32: equal up to at most 1 f32 ulp
    ulp = np.abs(got.view(np.int32).astype(np.int64) - ref.view(np.int32).astype(np.int64))
    assert ulp.max() <= 1


@pytest.mark.parametrize("gtype", [pm.GGML_F16, pm.GGML_Q8_0, pm.GGML_Q4_K])
@pytest.mark.parametrize("M,N,K", [(1000, 3072, 512), (2000, 4096, 256), (333, 2048, 1024), (129, 320, 1280),
                                   (2000, 1024, 4096), (700, 1000, 2048), (2000, 3072, 1024), (1900, 2880, 512),
                                   (2000, 2832, 256)])
def test_linear_tile_shapes(gpu, stream, gtype, M, N, K):
    """f16 path at shapes that select each MFMA tile (64x64, 128x64, 128x128,
    and 128x64 with two K groups for long K; the register-B 128x256 tiles) and
    leave partial tiles on both edges (N = 2832: the last 256-column tile holds
    16 columns, one lane half's store group of one wave)."""
    rng = _rng(M * 7 + N + K)
    raw, wf = _weights(gtype, N, K, rng)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 0.1, N).astype(np.float32)
    print(f"[linear-tiles] type={gtype} M={M} N={N} K={K}", flush=True)
    ref = oracle.linear(x, wf, b)
    dx = gpu.DeviceArray.from_numpy(x, stream)
    db = gpu.DeviceArray.from_numpy(b, stream)
    dy = gpu.DeviceArray((M, N), np.float32)
    gpu.linear(1, gtype, N, K, raw, dx, M, dy, db, stream)
    err = rel_l2(dy.numpy(stream), ref)
    assert err < 2e-3, err


def _residual_calls(gpu, stream, gtype, K, shapes, rng, tag):
    """linear_residual (y += alpha (x W^T + b)) on fresh random inputs at each
    (M, N) of shapes.  Every element is checked against a float64 product of
    the exact f16 operands the kernel multiplies (activations rounded to f16;
    q8_0 weights f16(d q), f16 weights as stored), within the worst-case f32
    summation bound of its K terms, and the first element outside it fails
    the test."""
    alpha = 0.5
    for call, (M, N) in enumerate(shapes):
        raw, wf = _weights(gtype, N, K, rng)
        if gtype == pm.GGML_Q8_0:
            blk = raw.reshape(-1, 34)
            d = blk[:, :2].copy().view(np.float16).astype(np.float32).reshape(-1, 1)
            q = blk[:, 2:].view(np.int8).astype(np.float32)
            w16 = (d * q).astype(np.float16).astype(np.float64).reshape(N, K)
        else:
            w16 = wf.astype(np.float64)
        x = rng.normal(0, 1, (M, K)).astype(np.float32)
        b = rng.normal(0, 0.1, N).astype(np.float32)
        y0 = rng.normal(0, 1, (M, N)).astype(np.float32)
        x16 = x.astype(np.float16).astype(np.float64)
        acc = x16 @ w16.T
        ref = y0.astype(np.float64) + alpha * (acc + b)
        # |f32 sum - exact| <= K 2^-24 sum|x w| (+ the rounding of the last adds)
        bound = K * 2.0 ** -24 * (np.abs(x16) @ np.abs(w16).T) + 2.0 ** -22 * (np.abs(ref) + 1.0)
        print(f"[{tag}] call {call} type={gtype} M={M} N={N} K={K}", flush=True)
        dx = gpu.DeviceArray.from_numpy(x, stream)
        db = gpu.DeviceArray.from_numpy(b, stream)
        dy = gpu.DeviceArray.from_numpy(y0, stream)
        gpu.linear_residual(1, gtype, N, K, raw, dx, M, dy, alpha, db, stream)
        got = dy.numpy(stream).astype(np.float64)
        bad = np.abs(got - ref) > bound
        if bad.any():
            i, j = np.argwhere(bad)[0]
            raise AssertionError(f"call {call}: y[{i}][{j}] = {got[i, j]!r}, float64 {ref[i, j]!r}, "
                                 f"bound {bound[i, j]:.3g} ({int(bad.sum())} elements outside)")
        dx.free(), db.free(), dy.free()


@pytest.mark.parametrize("gtype", [pm.GGML_Q8_0, pm.GGML_F16])
def test_residual_few_rows_fresh_inputs(gpu, stream, gtype):
    """The residual product of few rows (K split over the waves of a workgroup,
    the partial tiles summed in a fixed order) on fresh random inputs at every
    call, the calls of different sizes, so a stale or missing partial cannot
    repeat the previous result; and with N no multiple of 32, which the K-split
    tiles do not take (64 x 64 tiles with two K groups)."""
    _residual_calls(gpu, stream, gtype, 2048, ((512, 1024), (200, 1024), (128, 320), (192, 448), (512, 1024),
                                               (128, 312), (512, 488), (125, 1000)),
                    _rng(2048), "few-rows")


@pytest.mark.parametrize("gtype", [pm.GGML_Q8_0, pm.GGML_F16])
@pytest.mark.parametrize("K", [4096, 1024, 512])
def test_residual_two_k_groups(gpu, stream, gtype, K):
    """The residual products at N = 1024, M = 2000 (FFN linear2 and attention
    output shapes): q8_0 weights on the register-B kernel with two K groups
    (64 x 128 tiles, one per CU), f16 weights on the LDS-B kernel with two K
    groups.  In the former group g sums the other group's partial into row
    block g; M = 2040 leaves the last tile's second row block 24 rows,
    M = 1990 leaves it none (the first 6), and N = 960 leaves the last column
    tile's two right waves no columns."""
    _residual_calls(gpu, stream, gtype, K, ((2000, 1024), (2040, 1024), (1990, 1024), (2000, 960)),
                    _rng(K + gtype), "two-k-groups")



@pytest.mark.parametrize("M,N,K", [(1, 33, 8), (17, 31, 1000), (125, 512, 2048), (16, 32, 1024), (249, 2048, 520),
                                   (33, 1025, 40), (33, 1025, 264), (1, 31, 256), (1000, 1030, 1032), (700, 512, 512), (513, 640, 1024)])
def test_linear_f32_k_split(gpu, stream, M, N, K):
    """f32 weights on the K-split tiles (16 x 32 with four and eight K groups,
    32 x 32 with four): partial tiles on both edges, K that is no whole number
    of 32-column steps; and K below the K-split kernel's 256.  Every element within the
    worst-case f32 summation bound of the float64 product, for the store and
    for the residual update."""
    rng = _rng(M + 3 * N + K)
    w = rng.normal(0, 0.05, (N, K)).astype(np.float32)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 0.1, N).astype(np.float32)
    y0 = rng.normal(0, 1, (M, N)).astype(np.float32)
    print(f"[linear-f32-ks] M={M} N={N} K={K}", flush=True)
    acc = x.astype(np.float64) @ w.T.astype(np.float64) + b
    bound = K * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T) + 2.0 ** -22 * (np.abs(acc) + 1.0)
    dx = gpu.DeviceArray.from_numpy(x, stream)
    db = gpu.DeviceArray.from_numpy(b, stream)
    dy = gpu.DeviceArray((M, N), np.float32)
    gpu.linear(0, pm.GGML_F32, N, K, w, dx, M, dy, db, stream)
    assert (np.abs(dy.numpy(stream) - acc) <= bound).all()
    dr = gpu.DeviceArray.from_numpy(y0, stream)
    gpu.linear_residual(0, pm.GGML_F32, N, K, w, dx, M, dr, 0.5, db, stream)
    assert (np.abs(dr.numpy(stream) - (y0 + 0.5 * acc)) <= bound + 2.0 ** -22 * np.abs(y0)).all()


@pytest.mark.parametrize("gtype", [pm.GGML_F32, pm.GGML_F16, pm.GGML_Q8_0, pm.GGML_Q4_K])
@pytest.mark.parametrize("M", [827, 1019, 1147, 1211, 1403, 1787])
def test_linear_f32_mode_tiles(gpu, stream, gtype, M):
    """f32 mode past one round of 64 x 128 tiles (N = 3072): 1.2 to 1.8 rounds,
    where the 64 x 128 and the 32 x 64 tiles alternate by weight type, and 2.1
    and 2.6."""
    N, K = 3072, 256
    rng = _rng(M)
    raw, wf = _weights(gtype, N, K, rng)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 0.1, N).astype(np.float32)
    print(f"[linear-f32-tiles] type={gtype} M={M}", flush=True)
    ref = oracle.linear(x, wf, b)
    dx = gpu.DeviceArray.from_numpy(x, stream)
    db = gpu.DeviceArray.from_numpy(b, stream)
    dy = gpu.DeviceArray((M, N), np.float32)
    gpu.linear(0, gtype, N, K, raw, dx, M, dy, db, stream)
    assert rel_l2(dy.numpy(stream), ref) < 1e-5


@pytest.mark.parametrize("gtype", [pm.GGML_F16, pm.GGML_Q8_0, pm.GGML_Q4_K])
@pytest.mark.parametrize("M,N,K", [(1, 32, 256), (2, 2048, 512), (17, 64, 768), (125, 1024, 4096), (130, 2048, 512),
                                   (250, 1024, 2048), (257, 1536, 1024), (500, 1024, 1024), (129, 4096, 256),
                                   (129, 3072, 256), (200, 4032, 512), (1000, 1024, 1024), (3, 96, 1280)])
def test_linear_few_rows(gpu, stream, gtype, M, N, K):
    """f16 path on the K-split row tiles: 16-, 32- and 64-row tiles, partial
    row tiles, fewer and more 64-column steps than K groups; the store, and
    the residual update twice in a row on the same inputs (bit-identical)."""
    rng = _rng(M + 5 * N + K)
    raw, wf = _weights(gtype, N, K, rng)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    b = rng.normal(0, 0.1, N).astype(np.float32)
    y0 = rng.normal(0, 1, (M, N)).astype(np.float32)
    print(f"[linear-rows] type={gtype} M={M} N={N} K={K}", flush=True)
    ref = oracle.linear(x, wf, b)
    dx = gpu.DeviceArray.from_numpy(x, stream)
    db = gpu.DeviceArray.from_numpy(b, stream)
    dy = gpu.DeviceArray((M, N), np.float32)
    gpu.linear(1, gtype, N, K, raw, dx, M, dy, db, stream)
    assert rel_l2(dy.numpy(stream), ref) < 2e-3
    outs = []
    for _ in range(2):
        dr = gpu.DeviceArray.from_numpy(y0, stream)
        gpu.linear_residual(1, gtype, N, K, raw, dx, M, dr, 0.5, db, stream)
        outs.append(dr.numpy(stream))
    assert np.array_equal(outs[0], outs[1])
    assert rel_l2(outs[0] - y0, 0.5 * ref) < 2e-3
