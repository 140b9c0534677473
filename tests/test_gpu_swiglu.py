"""The expert kernels' clamped SwiGLU (hardware base-2 exponential and reciprocal) against the op-by-op bf16 rounding of
the oracle.  At the model's alpha and limit: every finite bf16 gate value, with the up values +-0, +-1, the limit and
beyond it.  With alpha = +-1 and no limit the sigmoid's argument is +-gate: every bf16 argument, the same bits as the fp32
expression 1 / (1 + exp(-t)) with correctly rounded steps, infinite and NaN gates and ups included (the clamps return the
other operand for a NaN).  A limit below zero is the clamp's result for every up value, as min(max(u, -limit), limit) has
it.  The paired form gives the single form's bits."""
import numpy as np
import pytest

from oracle.bf16 import bf16_bits_to_f32, f32_to_bf16_bits

pytestmark = pytest.mark.gpu


def test_swiglu_every_gate_value():
    import torch
    from neural_amd import _native as N
    ups = f32_to_bf16_bits(np.array([0.0, -0.0, 1.0, -1.0, 0.3, 7.0, 9.0, -12.0], np.float32))
    g = np.repeat(np.arange(65536, dtype=np.uint16), len(ups))
    u = np.tile(ups, 65536)
    ok = np.isfinite(bf16_bits_to_f32(g))
    g, u = g[ok], u[ok]
    print(f"case swiglu self-check, {g.size} pairs", flush=True)
    gd, ud = (torch.from_numpy(v.view(np.int16).copy()).cuda() for v in (g, u))
    out, out2 = torch.empty_like(gd), torch.empty_like(gd)
    N.call("na_selftest_swiglu", gd.data_ptr(), ud.data_ptr(), 1.702, 7.0, out.data_ptr(), out2.data_ptr(), g.size,
           N.stream(gd.device))
    got, got2 = (t.cpu().numpy().view(np.uint16) for t in (out, out2))
    assert np.array_equal(got, got2)
    rb = lambda v: bf16_bits_to_f32(f32_to_bf16_bits(v.astype(np.float32)))  # noqa: E731
    gf, uf = bf16_bits_to_f32(g), bf16_bits_to_f32(u)
    gate, up = np.minimum(gf, np.float32(7.0)), np.clip(uf, np.float32(-7.0), np.float32(7.0))
    with np.errstate(over="ignore", under="ignore"):
        t = rb(gate * np.float32(1.702))
        s = rb(1.0 / (1.0 + np.exp(-t.astype(np.float64))))
        want = rb(rb(up + np.float32(1.0)) * rb(gate * s))
    tiny = t < -87.3
    assert np.array_equal(f32_to_bf16_bits(want)[~tiny], got[~tiny])
    assert np.abs(bf16_bits_to_f32(got)[tiny].astype(np.float64) - want[tiny]).max() < 2.0 ** -120 * 8


# No limit of 0: the minimum of two zeros of opposite sign may be either (numpy's and the hardware's differ).
@pytest.mark.parametrize("alpha,limit", [(1.0, np.inf), (-1.0, np.inf), (1.702, 7.0), (1.702, -3.0)])
def test_swiglu_every_sigmoid_argument(alpha, limit):
    import torch
    from neural_amd import _native as N
    ups = f32_to_bf16_bits(np.array([0.0, -1.0, 0.3, 7.0, -12.0, np.inf, -np.inf], np.float32))
    ups = np.append(ups, np.uint16([0x7FC0])).astype(np.uint16)
    g = np.repeat(np.arange(65536, dtype=np.uint16), len(ups))
    u = np.tile(ups, 65536)
    print(f"case swiglu alpha={alpha} limit={limit}, {g.size} pairs", flush=True)
    gd, ud = (torch.from_numpy(v.view(np.int16).copy()).cuda() for v in (g, u))
    out, out2 = torch.empty_like(gd), torch.empty_like(gd)
    N.call("na_selftest_swiglu", gd.data_ptr(), ud.data_ptr(), alpha, limit, out.data_ptr(), out2.data_ptr(), g.size,
           N.stream(gd.device))
    got, got2 = (t.cpu().numpy().view(np.uint16) for t in (out, out2))
    rb = lambda v: bf16_bits_to_f32(f32_to_bf16_bits(v))  # noqa: E731
    one, lim = np.float32(1.0), np.float32(limit)
    with np.errstate(all="ignore"):
        gate = np.fmin(bf16_bits_to_f32(g), lim)
        up = np.fmin(np.fmax(bf16_bits_to_f32(u), -lim), lim)
        t = rb(gate * np.float32(alpha))
        e = np.exp(-t.astype(np.float64)).astype(np.float32)
        want = f32_to_bf16_bits(rb(rb(up + one) * rb(gate * rb(one / (one + e)))))
    nan = np.isnan(bf16_bits_to_f32(want))
    for v in (got, got2):
        assert np.array_equal(np.isnan(bf16_bits_to_f32(v)), nan)
        bad = (v != want) & ~nan
        assert not bad.any(), sorted(set(t[bad].tolist()))[:20]
