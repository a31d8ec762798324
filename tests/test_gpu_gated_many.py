"""The gated RMSNorm of many groups (sixteen per workgroup), bit for bit the
oracle's serial sums, at the group sizes and counts around its dispatch line
and with a last workgroup that is not full."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("m,h,group,activated,shift", [
    (17, 4064, 32, False, 0), (16, 4096, 32, True, 1), (75, 4032, 96, False, 0),
    (129, 4096, 128, True, 0), (128, 4096, 128, False, 1), (483, 4352, 256, False, 0)])
def test_gated_rmsnorm_many(ctx, oracle, m, h, group, activated, shift, dtype):
    rng = np.random.default_rng(m + h + group)
    x, z = rng.standard_normal((m, h)).astype(np.float32), rng.standard_normal((m, h)).astype(np.float32)
    x[m // 2] = 0.0
    w = (rng.standard_normal(group) * 0.1 + 1.0).astype(np.float32)
    dt = np.uint16 if dtype == "bf16" else np.float32
    if dtype == "bf16":
        x, z = oracle.f32_to_bf16_bits(x), oracle.f32_to_bf16_bits(z)

    def place(a):  # `shift` values past an aligned address
        return ctx.to_device(np.concatenate([np.zeros(shift, dt), a.reshape(-1)]))

    size = np.dtype(dt).itemsize
    xd, zd, wd = place(x), place(z), ctx.to_device(w)
    yd = ctx.alloc((m * h + shift) * size)
    ctx.gated_rmsnorm(xd.ptr + shift * size, zd.ptr + shift * size, wd, yd.ptr + shift * size, m, h,
                      group, eps=1e-6, gate_activated=activated, dtype=dtype)
    got = ctx.to_host(yd, (m, h), dt, offset=shift * size)
    ref = oracle.gated_rmsnorm(x, z, w, group, 1e-6, gate_activated=activated,
                               out_bf16=dtype == "bf16")
    bits = np.uint16 if dtype == "bf16" else np.uint32
    assert np.array_equal(got.view(bits), np.asarray(ref, dt).view(bits))
