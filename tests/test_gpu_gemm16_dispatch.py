"""The choice between the two GEMMs (gemm16_takes) must change neither what a
call returns nor what an earlier call has prepared for it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def weights(oracle, rng, n, k):
    return oracle.pack_q8_0_p4((rng.standard_normal((n, k)) * 0.02).astype(np.float32))


# groups of which a member alone would split K, or run in the serial order,
# while the group's column tiles together would be priced otherwise
@pytest.mark.parametrize("m,k,widths", [
    (200, 2560, (2560, 1024, 1024)), (256, 2560, (8192, 4096, 32, 32)),
    (40, 4096, (264, 2048)), (20, 9216, (136, 1024, 2560))])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_split_group_equals_single_calls(ctx, oracle, m, k, widths, dtype):
    rng = np.random.default_rng(m + k)
    ps = [weights(oracle, rng, n, k) for n in widths]
    x = rng.standard_normal((m, k)).astype(np.float32)
    esz, view = (2, np.uint16) if dtype == "bf16" else (4, np.uint32)
    ts = [ctx.upload_p4(p, n, k) for p, n in zip(ps, widths)]
    ctx.set_accumulation("split_k")
    try:
        xd = ctx.to_device(oracle.f32_to_bf16_bits(x) if dtype == "bf16" else x)
        group, single = ([ctx.alloc(m * n * esz) for n in widths] for _ in range(2))
        ctx.linear_group(xd, ts, group, m, mode="prefill", dtype=dtype)
        for t, y in zip(ts, single):
            ctx.linear(xd, t, y, m, mode="prefill", dtype=dtype)
        for n, a, b in zip(widths, group, single):
            assert np.array_equal(ctx.to_host(a, (m, n), view), ctx.to_host(b, (m, n), view)), n
    finally:
        ctx.set_accumulation("exact")
        for t in ts:
            ctx.release(t)


# the counts of gemm_splits_for on 256 CUs
@pytest.mark.parametrize("m,n,k,splits", [
    (2, 136, 1024, 2), (40, 264, 4096, 3), (16, 512, 16384, 10), (64, 2560, 9216, 6),
    (256, 2560, 9216, 4), (512, 2560, 9216, 2), (200, 2560, 2560, 3)])
def test_split_shapes_run_in_their_splits(ctx, oracle, m, n, k, splits):
    """SPLIT_K sums a shape that it splits in the splits of its own choice: the
    bits of that count forced, and not those of the serial order."""
    rng = np.random.default_rng(m + n + k)
    t = ctx.upload_p4(weights(oracle, rng, n, k), n, k)
    xd = ctx.to_device(rng.standard_normal((m, k)).astype(np.float32))
    yd = ctx.alloc(m * n * 4)

    def linear(mode, forced=0):
        ctx.set_accumulation(mode, splits=forced)
        ctx.linear(xd, t, yd, m, mode="prefill")
        return ctx.to_host(yd, (m, n), np.uint32)

    try:
        chosen, serial = linear("split_k"), linear("exact")
        assert np.array_equal(chosen, linear("split_k", splits))
        assert not np.array_equal(chosen, serial)
    finally:
        ctx.set_accumulation("exact")
        ctx.release(t)


@pytest.mark.parametrize("entry", ["swiglu", "mlp"])
def test_warm_up_with_more_rows_prepares_fewer(q8, oracle, entry):
    """A call of more rows prepares the scratch of one with fewer, also where
    the two run on different GEMMs: H = 1024, F = 4352 in bf16 takes the 16 x
    16 tiles at 100 rows and the 64 x 64 ones, which need a buffer for the
    gate, at 40.  Each replay equals the eager result."""
    h, f, rng = 1024, 4352, np.random.default_rng(3)
    with q8.Context(0) as c:
        ts = [c.upload_p4(weights(oracle, rng, n, k), n, k) for n, k in ((f, h), (f, h), (h, f))]
        x = oracle.f32_to_bf16_bits(rng.standard_normal((100, h)).astype(np.float32))
        xd, hd, yd = c.to_device(x), c.alloc(100 * f * 2), c.alloc(100 * h * 2)

        def call(m):
            if entry == "swiglu":
                c.swiglu(xd, ts[0], ts[1], hd, m, mode="prefill", dtype="bf16")
            else:
                c.mlp(xd, ts[0], ts[1], ts[2], yd, h=hd, m=m, mode="prefill", dtype="bf16")

        def result():
            return (c.to_host(hd, (40, f), np.uint16) if entry == "swiglu"
                    else c.to_host(yd, (40, h), np.uint16))

        call(100)
        c.sync()
        c.graph_begin()
        call(40)
        graph = c.graph_end()
        replays = []
        for _ in range(3):
            c.graph_launch(graph)
            c.sync()
            replays.append(result())
        call(40)
        c.sync()
        for got in replays:
            assert np.array_equal(got, result())
        c.graph_destroy(graph)
