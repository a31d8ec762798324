"""GPU parity of the GEMM on 16 x 16 tiles (q8_gemm16.hip) at the edges of its
tiles, rings and workgroup shapes: bit for bit the oracle's serial block order
with the platform's epilogue (Q8Matmul.cpp:204-223, Q8Scalar.cpp:192-199).
The shapes below lie where the dispatch takes it (gemm16_takes, shape16)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def same(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32),
                          np.asarray(b, np.float32).view(np.uint32))


def weights(oracle, rng, n, k):
    return oracle.pack_q8_0_p4((rng.standard_normal((n, k)) * 0.02).astype(np.float32))


# (m, n, k): row tiles 1 / 2 / 4 and ragged last ones; columns that end inside
# a tile and inside a workgroup's group of tiles (one, two, four or three);
# K of one unit more or less, ragged units, and the S = 4 and S = 6 layouts
@pytest.mark.parametrize("m,n,k", [
    (2, 8, 2560), (16, 40, 2592), (15, 5000, 2560), (3, 9000, 2560),
    (17, 24, 2528), (32, 5000, 2560), (31, 5016, 2208),
    (33, 1000, 2208), (64, 2568, 2560), (50, 5000, 2560), (65, 264, 2560), (130, 2568, 2560),
    (7, 136, 4096), (29, 136, 4096), (41, 264, 4096), (200, 2600, 4096),
    (5, 136, 9216), (18, 136, 9216), (70, 264, 9216), (210, 2600, 9216)])
def test_gemm16_bitwise(ctx, oracle, m, n, k):
    rng = np.random.default_rng(m * 31 + n + k)
    p4 = weights(oracle, rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[m // 2, 32:64] = 0.0
    t = ctx.upload_p4(p4, n, k)
    try:
        xd, yd = ctx.to_device(x), ctx.to_device(np.full((m, n), np.nan, np.float32))
        ctx.linear(xd, t, yd, m, mode="prefill")
        assert same(ctx.to_host(yd, (m, n), np.float32),
                    oracle.linear(x, p4, n, epilogue=ctx.epilogue, colpar=m < 16))
    finally:
        ctx.release(t)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("m,h,f", [(5, 2560, 264), (16, 2560, 5000), (9, 2560, 9000),
                                   (20, 2560, 264), (32, 2560, 5000), (40, 2560, 264),
                                   (6, 4096, 136), (21, 4096, 136), (12, 9216, 136),
                                   (30, 9216, 136)])
def test_gemm16_swiglu(ctx, oracle, m, h, f, dtype):
    rng = np.random.default_rng(m + h + f)
    pg, pu = weights(oracle, rng, f, h), weights(oracle, rng, f, h)
    x = rng.standard_normal((m, h)).astype(np.float32)
    bits, wide = oracle.f32_to_bf16_bits, oracle.bf16_bits_to_f32
    if dtype == "bf16":
        x = wide(bits(x))
    tg, tu = ctx.upload_p4(pg, f, h), ctx.upload_p4(pu, f, h)
    try:
        xd = ctx.to_device(bits(x) if dtype == "bf16" else x)
        hd = ctx.alloc(m * f * 4)
        ctx.swiglu(xd, tg, tu, hd, m, mode="prefill", dtype=dtype)
        g = oracle.linear(x, pg, f, activation="silu", epilogue=ctx.epilogue, colpar=m < 16)
        u = oracle.linear(x, pu, f, epilogue=ctx.epilogue, colpar=m < 16)
        if dtype == "bf16":
            ref = bits(wide(bits(g)) * wide(bits(u)))
            assert np.array_equal(ctx.to_host(hd, (m, f), np.uint16), ref)
        else:
            assert same(ctx.to_host(hd, (m, f), np.float32), g * u)
    finally:
        ctx.release(tg)
        ctx.release(tu)


@pytest.mark.parametrize("m", [2, 19, 40])
def test_gemm16_group_and_residual(ctx, oracle, m):
    """One launch over weights of different widths and activations (each
    with columns of its own in the last tile), bf16 rows, and the
    residual add in place."""
    rng = np.random.default_rng(m)
    k, widths, acts = 2560, (1000, 32, 8, 520), ("none", "sigmoid", "softplus", "silu")
    ps = [weights(oracle, rng, n, k) for n in widths]
    x = rng.standard_normal((m, k)).astype(np.float32)
    bits, wide = oracle.f32_to_bf16_bits, oracle.bf16_bits_to_f32
    xb = bits(x)
    ts = [ctx.upload_p4(p, n, k) for p, n in zip(ps, widths)]
    try:
        xd = ctx.to_device(xb)
        ys = [ctx.alloc(m * n * 2) for n in widths]
        ctx.linear_group(xd, ts, ys, m, activations=acts, mode="prefill", dtype="bf16")
        for p, n, act, y in zip(ps, widths, acts, ys):
            ref = bits(oracle.linear(wide(xb), p, n, activation=act, epilogue=ctx.epilogue,
                                     colpar=m < 16))
            assert np.array_equal(ctx.to_host(y, (m, n), np.uint16), ref), (n, act)
        r = rng.standard_normal((m, widths[0])).astype(np.float32)
        xf, rd = ctx.to_device(x), ctx.to_device(r)
        ctx.linear_add(xf, ts[0], rd, rd, m, mode="prefill")
        lin = oracle.linear(x, ps[0], widths[0], epilogue=ctx.epilogue, colpar=m < 16)
        assert same(ctx.to_host(rd, (m, widths[0]), np.float32), r + lin)
    finally:
        for t in ts:
            ctx.release(t)
