"""The expert kernels' clamped SwiGLU (hardware base-2 exponential and reciprocal) against the op-by-op bf16 rounding of
the oracle, over every bf16 gate value, with the up values +-0, +-1, the limit and beyond it: the same bits, except that
a sigmoid below 2^-126 (gates whose bf16(alpha gate) is below -87.3) may become +0, which moves the result by less than
2^-120.  The paired form gives the single form's bits."""
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
