"""na_core_router_pack against na_core_router followed by na_core_route_pack: the same bits in every output, with and
without a slot table (some experts not resident), near misses, bx and pack, with logits that tie; and the counter is
zero again after each call."""
import pytest

pytestmark = pytest.mark.gpu

H, NE, K = 2880, 128, 4


@pytest.mark.parametrize("table,near,bx_on,pack_on,ties", [(False, False, True, True, False), (True, True, True, True, False),
                                                           (True, True, False, True, True), (True, False, True, False, True)])
def test_equals_two_launches(table, near, bx_on, pack_on, ties):
    import torch
    from neural_amd import _native as N
    g = torch.Generator(device="cuda")
    g.manual_seed(17 + table + 2 * near + 4 * ties)
    bf = torch.bfloat16
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    mid, post_w, wr, br = rn(H).to(bf), (1 + 0.1 * rn(H)).to(bf), (0.02 * rn(NE, H)).to(bf), (0.02 * rn(NE)).to(bf)
    if ties:                                            # experts in equal pairs, and half the logits equal
        wr[1::2], br[1::2] = wr[0::2], br[0::2]
        wr[64:], br[64:] = wr[:1], br[:1]
    tab = torch.arange(3 * NE, device="cuda")
    tab[torch.rand(3 * NE, generator=g, device="cuda") < 0.4] = -1
    for layer in (0, 2):
        print(f"case router_pack table={table} near={near} ties={ties} layer={layer}", flush=True)
        res = []
        for fused in (False, True):
            z = lambda n, dt: torch.full((n,), 7, dtype=dt, device="cuda")  # noqa: E731
            o = dict(hn=z(H, bf), logits=z(NE, torch.float32), ids=z(K, torch.int64), wts=z(K, bf), bx=z(H, bf),
                     pack=z(H + 4 * K, torch.float32), bslots=z(K, torch.int64), bgids=z(K, torch.int64), bw=z(K, bf))
            counter = torch.zeros(1, dtype=torch.int32, device="cuda")
            s = N.stream(mid.device)
            p = lambda k: o[k].data_ptr()  # noqa: E731
            head = (mid.data_ptr(), post_w.data_ptr(), 1e-5, wr.data_ptr(), br.data_ptr(), p("hn"), p("logits"),
                    counter.data_ptr(), p("ids"), p("wts"))
            tail = (tab.data_ptr() if table else None, layer * NE, p("bx") if bx_on else None,
                    p("pack") if pack_on else None, int(near), p("bslots"), p("bgids"), p("bw"), s)
            if fused:
                N.call("na_core_router_pack", *head, *tail)
            else:
                N.call("na_core_router", *head, s)
                N.call("na_core_route_pack", p("hn"), p("logits"), p("ids"), p("wts"), *tail)
            assert int(counter.item()) == 0
            res.append(o)
        for k in res[0]:
            assert torch.equal(res[0][k], res[1][k]), k
