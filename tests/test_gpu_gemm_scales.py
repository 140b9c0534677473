"""The GEMM entry points (plain and grouped, raw and PS4 scales) at the ends of the E8M0 range, against products formed
in 64 bits from the codes and scale bytes: bytes 0 .. 2 (weights below bf16's normal range), 253 and 254 (weights past
bf16's largest value, whose products with small x are finite), 255 (NaN), side by side within a k-tile and within a row
block; x that is subnormal, infinite or NaN.  The t950 layout gives the raw layout's bits.

Bar, per element: one bf16 rounding (at most 2^-8 of the value) of the exact product, and fp32 accumulation of 2,880
exact products, each added in at most four equal parts: below 4 x 2 x 2,880 x 2^-24 of the sum of their magnitudes.
Elements whose magnitudes sum past 2^126 are left out (fp32 accumulation may overflow on the way)."""
import numpy as np
import pytest

from oracle import mxfp4_oracle as mo
from neural_amd import synth

pytestmark = pytest.mark.gpu

N_ROWS, K, GK = 384, 2880, 90
BANDS = {                                               # scale bytes of group g of row r: band[(g + r) % len(band)]
    "raw_mixed": (False, lambda r: [0, 1, 2, 126, 252, 253, 254]),
    "raw_high": (False, lambda r: [252, 253, 254]),
    "raw_low": (False, lambda r: [0, 1, 2]),
    "raw_nan": (False, lambda r: [126, 254, 127] if r % 5 else [126, 255, 127]),
    "ps4_high": (True, lambda r: [239, 252, 253, 254]),
    "ps4_low": (True, lambda r: [0, 1, 2, 15]),
    "ps4_rows": (True, lambda r: [[0, 1, 2], [126, 127], [252, 253, 254], [241, 254, 255]][r % 4]),
}
# x rows: standard normal values times 2^k, (one element infinite or NaN), or only in the groups of the given bytes
X_EXP = (-130, -110, -100, 0, 100, 110)


def _matrix(rng, band):
    s = np.empty((N_ROWS, GK), np.uint8)
    for r in range(N_ROWS):
        b = band(r)
        s[r] = [b[(g + r // 16) % len(b)] for g in range(GK)]
    return rng.integers(0, 256, (N_ROWS, GK, 16), dtype=np.uint8), s


def _weights64(codes, scales):
    v = mo.dequant_rows(codes, np.full_like(scales, 127)).astype(np.float64).reshape(N_ROWS, GK, 32)
    w = np.ldexp(v, scales.astype(np.int32)[..., None] - 127)
    w[scales == 255] = np.nan
    return w.reshape(N_ROWS, K)


def _rows(rng, scales):
    """[M, K] bf16 rows: every exponent over all elements, then only where row 0's groups hold a byte below 3 / above
    252, then one with an infinity and one with a NaN."""
    import torch
    base = rng.standard_normal((len(X_EXP) + 4, K)) * 0.5
    x = base * 2.0 ** np.array(list(X_EXP) + [100, -120, -100, -100])[:, None]
    per = np.repeat(scales[0], 32)
    x[len(X_EXP)] *= per < 3
    x[len(X_EXP) + 1] *= per > 252
    x[len(X_EXP) + 2, 77] = np.inf
    x[len(X_EXP) + 3, 1234] = np.nan
    return torch.from_numpy(x.astype(np.float32)).to(torch.bfloat16)


@pytest.mark.parametrize("name", sorted(BANDS))
def test_gemm_scale_range(name):
    import torch
    from neural_amd.q80 import mxfp4_kernels as mk
    packed, band = BANDS[name]
    rng = np.random.default_rng(sorted(BANDS).index(name))
    codes, scales = _matrix(rng, band)
    w = _weights64(codes, scales)
    x = _rows(rng, scales)
    M = x.shape[0]
    blocks = torch.from_numpy(codes)[None].cuda()
    sc = torch.from_numpy(mo.ps4_pack_rows(scales) if packed else scales)[None].cuda()
    xd = x.repeat(7, 1).cuda()                          # 70 rows: a full tile and a short one
    out = torch.empty(7 * M, N_ROWS, dtype=torch.bfloat16, device="cuda")
    print(f"case gemm scale bytes {name}", flush=True)
    got = mk.mxfp4_gemm(xd, blocks, sc, torch.zeros(1, dtype=torch.int64, device="cuda"))[0]
    mk.mxfp4_gemm_grouped_into([(xd, 0, out)], blocks, sc)
    for v in (got, out):                                # the same bits for a row wherever it lies
        assert torch.equal(v.view(torch.int16).view(7, M, N_ROWS), got[:M].view(torch.int16).expand(7, M, N_ROWS))
    got = got[:M]
    got = got.float().cpu().numpy().astype(np.float64)
    x64 = x.float().numpy().astype(np.float64)
    checked = 0
    for m in range(M):
        with np.errstate(invalid="ignore"):
            terms = w * x64[m]                          # inf * 0 is NaN
        special = ~np.isfinite(terms).all(1)
        if special.any():
            with np.errstate(invalid="ignore"):
                want = terms[special].sum(1)
            fin = np.where(np.isfinite(terms[special]), np.abs(terms[special]), 0).sum(1) < 2.0 ** 126
            assert np.array_equal(want[fin], got[m][special][fin], equal_nan=True), (name, m)
            checked += int(fin.sum())
        t = terms[~special]
        mag = np.abs(t).sum(1)
        ok = mag < 2.0 ** 126
        want, g = t.sum(1)[ok], got[m][~special][ok]
        bound = 2.0 ** -8 * np.abs(want) + 4 * 5760 * 2.0 ** -24 * mag[ok] + 2.0 ** -133
        worst = (np.abs(g - want) / bound).max(initial=0.0)
        assert worst <= 1.0, (name, m, worst)
        checked += int(ok.sum())
    assert checked > 3 * N_ROWS, (name, checked)


@pytest.mark.parametrize("high", [False, True])
def test_gemm_t950_equals_raw(high):
    """The C entry points over a t950 pool (layout 2): the raw pool's bits, with the model's scale bytes and with bytes
    252 .. 254 in every seventh row; two slots, gate_up and down, full and short tiles, plain and grouped."""
    import torch
    from neural_amd import _native as N
    from neural_amd import tiles
    from neural_amd.moe.layout import GPTOSS_LAYOUT, GPTOSS_LAYOUT_T950, mxfp4_pool_views
    from neural_amd.q80 import mxfp4_kernels as mk
    rng = np.random.default_rng(40 + high)
    slots = np.stack([synth.slot_raw(rng) for _ in range(2)])
    if high:
        sc = slots[:, synth.CODE_BYTES:].reshape(2, -1, GK)
        sc[:, ::7] = rng.integers(252, 255, sc[:, ::7].shape, dtype=np.uint8)
    raw = torch.from_numpy(slots).cuda()
    t950 = torch.empty(2, GPTOSS_LAYOUT_T950.slot_bytes, dtype=torch.uint8, device="cuda")
    tiles.repack_to_t950(raw, t950)
    gb, db, gs, ds = mxfp4_pool_views(raw, GPTOSS_LAYOUT)
    x = (synth.bf16_normal(rng, (83, K)).float() * (2.0 ** -100 if high else 1.0)).to(torch.bfloat16).cuda()
    sl = torch.tensor([1, 0], dtype=torch.int64, device="cuda")
    for blocks, scales, off, n in ((gb, gs, 0, 5760), (db, ds, 360 * 24576, 2880)):
        print(f"case gemm t950 n={n} high={high}", flush=True)
        want = mk.mxfp4_gemm(x, blocks, scales, sl)
        assert torch.isfinite(want).all()
        base, s = t950.data_ptr() + off, N.stream(x.device)
        got = torch.full_like(want, 7.0)
        N.call("na_mxfp4_gemm", x.data_ptr(), 83, K, base, t950.stride(0), None, 0, 2, sl.data_ptr(), 2, got.data_ptr(), n,
               s)
        assert torch.equal(got, want)
        out = torch.full_like(want, 7.0)
        plan = mk.GroupedGemmPlan([(x, 1, out[0]), (x, 0, out[1])])
        N.call("na_mxfp4_gemm_grouped", base, t950.stride(0), None, 0, 2, plan.metadata.data_ptr(), plan.ntiles,
               plan.block_m, n, K, s)
        assert torch.equal(out, want)
