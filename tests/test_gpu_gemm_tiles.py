"""The GEMM entry points at the edges of their tiles: 1 to 4 16-row blocks per tile (full and one row over), column
counts on both sides of the XCD order's rule (192 and 384 columns take the plain order, 1,536, 2,880 and 5,760 the XCD
order), scale views that are not 16-byte aligned, and grouped tiles of more than 64 rows.

Bar, per element: one bf16 rounding (8 significant bits: half a unit in the last place is at most 2^-8 of the value,
reached just above a power of two) of the exact product and fp32 accumulation of 2,880 exact
products (below 5,760 x 2^-24 of the sum of their magnitudes)."""
import numpy as np
import pytest

from oracle import mxfp4_oracle as mo
from neural_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def slots():
    rng = np.random.default_rng(91)
    raw = [synth.slot_raw(rng) for _ in range(2)]
    return raw, [mo.expert_weights(s)[0].astype(np.float64) for s in raw]


def _views(slots, packed, n, odd):
    """gate_up views of the first n rows; odd: the scale rows copied to an odd address."""
    import torch
    from neural_amd.moe.layout import GPTOSS_LAYOUT, GPTOSS_LAYOUT_PS4, mxfp4_pool_views
    pool = torch.from_numpy(np.stack([mo.ps4_pack_slot(s) if packed else s for s in slots[0]])).cuda()
    gb, _, gs, _ = mxfp4_pool_views(pool, GPTOSS_LAYOUT_PS4 if packed else GPTOSS_LAYOUT)
    gb, gs = gb[:, :n], gs[:, :n]
    if odd:
        buf = torch.empty(gs.numel() + 1, dtype=torch.uint8, device="cuda")
        own = buf[1:].view(gs.shape)
        own.copy_(gs)
        gs = own
    return gb, gs


def _check(got, x, w, tag):
    want = x @ w.T
    bound = 2.0 ** -8 * np.abs(want) + 5760 * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T) + 1e-30
    worst = (np.abs(got - want) / bound).max(initial=0.0)
    assert worst <= 1.0, (tag, worst)


@pytest.mark.parametrize("n,packed,odd", [(5760, False, False), (2880, True, False), (1536, False, True),
                                          (384, True, True), (192, False, False)])
def test_gemm_tile_edges(slots, n, packed, odd):
    import torch
    from neural_amd.q80 import mxfp4_kernels as mk
    gb, gs = _views(slots, packed, n, odd)
    sl = torch.tensor([1, 0], dtype=torch.int64, device="cuda")
    rng = np.random.default_rng(n)
    for M in (1, 16, 17, 32, 33, 48, 49, 65):
        print(f"case gemm n={n} packed={packed} odd={odd} M={M}", flush=True)
        x = synth.bf16_normal(rng, (M, 2880))
        got = mk.mxfp4_gemm(x.cuda(), gb, gs, sl).float().cpu().numpy().astype(np.float64)
        xf = x.float().numpy().astype(np.float64)
        for e, s in enumerate((1, 0)):
            _check(got[e], xf, slots[1][s][:n], (n, packed, odd, M, e))


@pytest.mark.parametrize("block_m", [16, 32, 256])
def test_grouped_sub_tiles(slots, block_m):
    import torch
    from neural_amd.q80 import mxfp4_kernels as mk
    n = 2880
    gb, gs = _views(slots, False, n, False)
    rng = np.random.default_rng(block_m)
    ms = [300, 1, 40, 0, 256, 257]
    xs = [synth.bf16_normal(rng, (m, 2880)) for m in ms]
    outs = [torch.full((m, n), 7.0, dtype=torch.bfloat16, device="cuda") for m in ms]
    print(f"case grouped block_m={block_m} M={ms}", flush=True)
    mk.mxfp4_gemm_grouped_into([(x.cuda(), i % 2, o) for i, (x, o) in enumerate(zip(xs, outs))], gb, gs,
                               block_m=block_m)
    for i, (x, o) in enumerate(zip(xs, outs)):
        _check(o.float().cpu().numpy().astype(np.float64), x.float().numpy().astype(np.float64),
               slots[1][i % 2][:n], (block_m, i))


def test_more_tiles_than_one_grid_holds(slots):
    """Tiles past 2^32 threads of one grid: 1,048,584 one-row tiles of 16 column groups, and 16,400 grouped tiles of
    4,096 rows (64 x 16 workgroups each); every row equals the same row of a small call, bit for bit."""
    import torch
    from neural_amd.q80 import mxfp4_kernels as mk
    n = 2880
    gb, gs = _views(slots, False, n, False)
    x = synth.bf16_normal(np.random.default_rng(5), (1, n)).cuda()
    two = mk.mxfp4_gemm(x, gb, gs, torch.tensor([0, 1], device="cuda"))[:, 0]
    E = 1_048_576 + 8
    print(f"case gemm E={E} M=1", flush=True)
    got = mk.mxfp4_gemm(x, gb, gs, torch.arange(E, device="cuda") % 2).view(E // 2, 2, n)
    assert all(torch.equal(c, two.expand_as(c)) for c in got.split(1 << 16))
    del got
    P = 16_400
    out = torch.full((P, 1, n), 7.0, dtype=torch.bfloat16, device="cuda")
    print(f"case grouped pairs={P} block_m=4096", flush=True)
    mk.mxfp4_gemm_grouped_into([(x, i % 2, out[i]) for i in range(P)], gb, gs, block_m=4096)
    assert torch.equal(out.view(P // 2, 2, n), two.expand(P // 2, 2, n))


@pytest.mark.parametrize("packed", [False, True])
def test_codes_past_32_bit_offsets(packed):
    """Row blocks on both sides of 2^31 and 2^32 code bytes (1,440 a row), and the last one: the same bits, bit for bit,
    as the product with those 192 rows alone.  The reference product of the rows just past 4 GiB is checked in 64 bits."""
    import torch
    from neural_amd.q80 import mxfp4_kernels as mk
    n = 192 * (2 ** 32 // (192 * 1440) + 2)
    w = 46 if packed else 90
    print(f"case gemm N={n} packed={packed}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(17)
    codes = torch.empty(n * 1440 // 8, dtype=torch.int64, device="cuda").random_(generator=g).view(torch.uint8)
    codes = codes.view(1, n, 90, 16)
    scales = torch.randint(0 if packed else 119, 126, (1, n, w), generator=g, dtype=torch.uint8, device="cuda")
    if packed:
        scales[:, :, 0] = 119                           # base byte; the others hold two 4-bit deltas each
        scales[:, :, 1:] &= 0x33
    x = synth.bf16_normal(np.random.default_rng(6), (5, 2880)).cuda()
    slot = torch.zeros(1, dtype=torch.int64, device="cuda")
    full = mk.mxfp4_gemm(x, codes, scales, slot)[0]
    out = torch.empty_like(full)
    mk.mxfp4_gemm_grouped_into([(x, 0, out)], codes, scales)
    assert torch.equal(full, out)
    for r0 in (0, 2 ** 31 // 1440 // 192 * 192, 2 ** 32 // 1440 // 192 * 192, n - 192):
        cb, sb = codes[:, r0:r0 + 192].clone(), scales[:, r0:r0 + 192].clone()
        assert torch.equal(full[:, r0:r0 + 192], mk.mxfp4_gemm(x, cb, sb, slot)[0]), r0
    sc = sb[0].cpu().numpy()
    wts = mo.dequant_rows(cb[0].cpu().numpy(), mo.ps4_unpack_rows(sc) if packed else sc).astype(np.float64)
    _check(full[:, n - 192:].float().cpu().numpy().astype(np.float64), x.float().cpu().numpy().astype(np.float64), wts,
           (packed, n))
