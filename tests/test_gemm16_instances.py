"""Every instance of the GEMM on 16 x 16 tiles (q8_gemm16.hip), bit for bit the
oracle's serial block order: the ring depths, the unrolled period and the wait
counts differ with S, the workgroup's row and column tiles and the SwiGLU
pair.  gemm_plan says which instance a shape runs on, so a shape that the
dispatch moves to another one shows as a failure.  And the other GEMM
(q8_gemm.hip) at small shapes, which the dispatch gives to this one."""
import numpy as np
import pytest

# (S, row tiles, column tiles), SwiGLU pair, m, widths, k: rows that end inside
# a row tile and, with two or four row tiles, inside the workgroup; columns
# that end inside a tile and inside the workgroup's tiles; K of ragged units
LINEARS = [
    ((1, 1, 1), 15, (136,), 2528), ((1, 1, 2), 5, (4136,), 2560), ((1, 1, 4), 13, (8264,), 2560),
    ((1, 2, 1), 29, (136,), 2528), ((1, 2, 2), 18, (4136,), 2560),
    ((1, 2, 4), 20, (4104, 4104, 40), 2560), ((1, 4, 1), 41, (264,), 2208),
    ((1, 4, 2), 70, (2072,), 2560), ((1, 4, 3), 66, (4120,), 2560),
    ((4, 1, 1), 15, (136,), 4064), ((4, 1, 2), 5, (4136,), 4096), ((4, 1, 4), 3, (8264,), 4064),
    ((4, 2, 1), 29, (136,), 4064), ((4, 2, 2), 18, (4136,), 4096),
    ((4, 2, 4), 20, (4104, 4104, 40), 4064), ((4, 4, 1), 41, (264,), 4064),
    ((4, 4, 2), 70, (2072,), 4096), ((4, 4, 3), 66, (4120,), 4064),
    ((6, 1, 1), 15, (136,), 8864), ((6, 1, 2), 5, (4136,), 9216), ((6, 1, 4), 3, (8264,), 9184),
    ((6, 2, 1), 29, (136,), 9184), ((6, 2, 2), 18, (4136,), 8864),
    ((6, 2, 4), 17, (8264,), 9216), ((6, 4, 1), 41, (264,), 9184),
    ((6, 4, 2), 70, (2072,), 8864), ((6, 4, 2), 100, (2560,), 9216), ((6, 4, 3), 66, (4120,), 9216)]
SWIGLUS = [
    ((1, 1, 1), 13, 264, 2528), ((1, 2, 1), 29, 264, 2560), ((1, 2, 3), 20, 4136, 2528),
    ((1, 4, 1), 41, 264, 2560), ((1, 4, 1), 70, 136, 2208),
    ((4, 1, 1), 13, 264, 4096), ((4, 2, 1), 29, 264, 4064), ((4, 2, 3), 20, 4136, 4096),
    ((4, 4, 1), 41, 264, 4064), ((4, 4, 1), 70, 136, 4096),
    ((6, 1, 1), 13, 264, 8864), ((6, 2, 1), 29, 264, 9216), ((6, 2, 1), 20, 4136, 9184),
    ((6, 4, 1), 41, 264, 9216), ((6, 4, 1), 70, 136, 9184)]


def same(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32),
                          np.asarray(b, np.float32).view(np.uint32))


def weights(oracle, rng, n, k):
    return oracle.pack_q8_0_p4((rng.standard_normal((n, k)) * 0.02).astype(np.float32))


def test_the_cases_reach_every_instance(q8):
    for inst, m, widths, k in LINEARS:
        assert q8.gemm_plan(m, widths, k)[0] == inst, (m, widths, k)
    for inst, m, f, h in SWIGLUS:
        assert q8.gemm_plan(m, [f], h, dual=True)[0] == inst, (m, f, h)
    shapes = {(1, 1), (1, 2), (1, 4), (2, 1), (2, 2), (2, 4), (4, 1), (4, 2), (4, 3)}
    pairs = {(1, 1), (2, 1), (2, 3), (4, 1)}
    assert {c[0] for c in LINEARS} == {(s,) + t for s in (1, 4, 6) for t in shapes}
    assert {c[0] for c in SWIGLUS} == {(s,) + t for s in (1, 4, 6) for t in pairs} - {(6, 2, 3)}


@pytest.mark.gpu
@pytest.mark.parametrize("inst,m,widths,k", LINEARS)
def test_linear_instance_bitwise(ctx, q8, oracle, inst, m, widths, k):
    assert q8.gemm_plan(m, widths, k)[0] == inst
    rng = np.random.default_rng(m * 31 + sum(widths) + k)
    ps = [weights(oracle, rng, n, k) for n in widths]
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[m // 2, 32:64] = 0.0
    ts = [ctx.upload_p4(p, n, k) for p, n in zip(ps, widths)]
    try:
        xd = ctx.to_device(x)
        ys = [ctx.to_device(np.full((m, n), np.nan, np.float32)) for n in widths]
        ctx.linear_group(xd, ts, ys, m, mode="prefill")
        for p, n, y in zip(ps, widths, ys):
            assert same(ctx.to_host(y, (m, n), np.float32),
                        oracle.linear(x, p, n, epilogue=ctx.epilogue, colpar=True)), n
    finally:
        for t in ts:
            ctx.release(t)


@pytest.mark.gpu
@pytest.mark.parametrize("inst,m,f,h", SWIGLUS)
def test_swiglu_instance_bitwise(ctx, q8, oracle, inst, m, f, h):
    assert q8.gemm_plan(m, [f], h, dual=True)[0] == inst
    rng = np.random.default_rng(m + h + f)
    pg, pu = weights(oracle, rng, f, h), weights(oracle, rng, f, h)
    x = rng.standard_normal((m, h)).astype(np.float32)
    tg, tu = ctx.upload_p4(pg, f, h), ctx.upload_p4(pu, f, h)
    try:
        xd, hd = ctx.to_device(x), ctx.to_device(np.full((m, f), np.nan, np.float32))
        ctx.swiglu(xd, tg, tu, hd, m, mode="prefill")
        ref = (oracle.linear(x, pg, f, activation="silu", epilogue=ctx.epilogue, colpar=True)
               * oracle.linear(x, pu, f, epilogue=ctx.epilogue, colpar=True))
        assert same(ctx.to_host(hd, (m, f), np.float32), ref)
    finally:
        ctx.release(tg)
        ctx.release(tu)


# the 16-row quantizer in front of it: four waves a tile (up to 1024 tiles) and
# one, rows on and off an aligned address, values of extreme scale
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("m", [40, 260])
def test_quantized_rows_bitwise(ctx, q8, oracle, m, shift, dtype):
    n, k = 136, 4096
    assert q8.gemm_plan(m, [n], k)[0] == (4, 4, 1)
    rng = np.random.default_rng(m + shift)
    p4 = weights(oracle, rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[3, 0:32] *= np.float32(1e-36)
    x[m - 1, k - 32:] *= np.float32(1e37)
    x[m // 2] = 0.0
    dt = np.float32
    if dtype == "bf16":
        dt = np.uint16
        xb = oracle.f32_to_bf16_bits(x)
        x = oracle.bf16_bits_to_f32(xb)
    rows = xb if dtype == "bf16" else x
    t = ctx.upload_p4(p4, n, k)
    try:
        xd = ctx.to_device(np.concatenate([np.zeros(shift, dt), rows.reshape(-1)]))
        yd = ctx.alloc(m * n * np.dtype(dt).itemsize)
        ctx.linear(xd.ptr + shift * np.dtype(dt).itemsize, t, yd, m, mode="prefill", dtype=dtype)
        ref = oracle.linear(x, p4, n, epilogue=ctx.epilogue, colpar=True)
        if dtype == "bf16":
            assert np.array_equal(ctx.to_host(yd, (m, n), np.uint16), oracle.f32_to_bf16_bits(ref))
        else:
            assert same(ctx.to_host(yd, (m, n), np.float32), ref)
    finally:
        ctx.release(t)


# one forced split is the serial order on the other GEMM: its 64 x 64 and 128 x
# 96 workgroups at S = 1, 4 and 6
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(2, 136, 288), (45, 264, 2208), (33, 136, 4096), (17, 264, 8864),
                                   (130, 520, 1056), (97, 264, 4064), (256, 1024, 2560),
                                   (129, 264, 9184)])
def test_other_gemm_bitwise(ctx, oracle, m, n, k):
    rng = np.random.default_rng(m * 7 + n + k)
    p4 = weights(oracle, rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[m // 2, 32:64] = 0.0
    t = ctx.upload_p4(p4, n, k)
    ctx.set_accumulation("split_k", splits=1)
    try:
        xd, yd = ctx.to_device(x), ctx.to_device(np.full((m, n), np.nan, np.float32))
        ctx.linear(xd, t, yd, m, mode="prefill")
        assert same(ctx.to_host(yd, (m, n), np.float32),
                    oracle.linear(x, p4, n, epilogue=ctx.epilogue, colpar=True))
    finally:
        ctx.set_accumulation("exact")
        ctx.release(t)


# K = 2560 is five passes of 512 values: splits 0 (its own choice, three) and 1
# (the serial order), the epilogue once on the sum
@pytest.mark.gpu
@pytest.mark.parametrize("splits", [0, 1])
@pytest.mark.parametrize("m", [40, 100])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("op", ["none", "silu", "sigmoid", "softplus", "add", "swiglu"])
def test_other_gemm_epilogues_bitwise(ctx, q8, oracle, op, dtype, m, splits):
    n, k = 264, 2560
    assert q8.gemm_plan(m, [n], k)[1] == 3
    cuts = [0, 512, 1536, 2560] if splits == 0 else [0, 2560]  # passes 0, 1-2, 3-4
    rng = np.random.default_rng(m + len(op))
    ws = [(rng.standard_normal((n, k)) * 0.02).astype(np.float32) for _ in range(2)]
    bits, wide = oracle.f32_to_bf16_bits, oracle.bf16_bits_to_f32
    bf16 = dtype == "bf16"
    stored = (lambda v: wide(bits(v))) if bf16 else (lambda v: v)
    x, r = (stored(rng.standard_normal(s).astype(np.float32)) for s in ((m, k), (m, n)))

    def sums(w):
        parts = [oracle.linear(x[:, a:b], oracle.pack_q8_0_p4(w[:, a:b]), n,
                               epilogue=ctx.epilogue, colpar=True) for a, b in zip(cuts, cuts[1:])]
        total = parts[0]
        for part in parts[1:]:
            total = total + part
        return total

    act = {"none": lambda v: v, "add": lambda v: v, "silu": oracle.silu, "swiglu": oracle.silu,
           "sigmoid": oracle.sigmoid, "softplus": oracle.softplus}[op]
    ref = act(sums(ws[0]))
    if op == "add":
        ref = stored(ref) + r
    if op == "swiglu":
        ref = stored(ref) * stored(sums(ws[1]))
    ts = [ctx.upload_p4(oracle.pack_q8_0_p4(w), n, k) for w in ws]
    put = (lambda v: ctx.to_device(bits(v))) if bf16 else ctx.to_device
    ctx.set_accumulation("split_k", splits=splits)
    try:
        xd, yd = put(x), put(r)
        if op == "add":
            ctx.linear_add(xd, ts[0], yd, yd, m, mode="prefill", dtype=dtype)
        elif op == "swiglu":
            ctx.swiglu(xd, ts[0], ts[1], yd, m, mode="prefill", dtype=dtype)
        else:
            ctx.linear(xd, ts[0], yd, m, activation=op, mode="prefill", dtype=dtype)
        if bf16:
            assert np.array_equal(ctx.to_host(yd, (m, n), np.uint16), bits(ref))
        else:
            assert same(ctx.to_host(yd, (m, n), np.float32), ref)
    finally:
        ctx.set_accumulation("exact")
        for t in ts:
            ctx.release(t)
