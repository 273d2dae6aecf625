"""Experts of many tokens on the matrix cores: the tiles whose operands travel into LDS by direct transfers, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


# pairs of an expert below, at and beyond half a tile and a tile of 160 and none at all, more pairs than the
# grouping holds and more experts than it numbers at a time; widths of one step of 64 and of half a one, of fewer
# steps than the ring has stages, of odd halves behind whole steps, outputs that end inside a block of 128 and of 256
@pytest.mark.parametrize("N,top,E", [(80, 1, 1), (160, 1, 1), (161, 1, 1), (177, 2, 2), (40, 2, 5), (300, 3, 4), (33, 1, 40), (3000, 3, 70)])
@pytest.mark.parametrize("W,F", [(32, 32), (64, 96), (96, 160), (352, 224), (512, 288)])
@pytest.mark.parametrize("form", ["table", "router", "one matrix", "bounded"])
def test_experts_in_tiles(ops, N, top, E, W, F, form):
    g = torch.Generator().manual_seed(N * 100 + top + W)
    r = lambda *s: torch.randn(*s, generator=g).to("cuda:0")     # noqa: E731
    bf = torch.bfloat16
    gated = form != "one matrix"
    gu, dn = (r(E, (2 if gated else 1) * F, W) * W ** -0.5).to(bf), (r(E, W, F) * F ** -0.5).to(bf)
    h, base = r(N, W).to(bf), r(N, W).to(bf)
    assert ops.lib.lmsf_table_moe_grouped(1, N, top, E, F, W, h.stride(0))
    vocab = 11 if form == "table" else N
    table = torch.randint(0, E, (vocab, top), generator=g, dtype=torch.int32).to("cuda:0")
    ids = torch.randint(0, vocab, (N,), generator=g, dtype=torch.int32).to("cuda:0") if form == "table" else None
    ps = r(N, top).abs() if form == "router" else None
    got = ops.table_moe(h, gu, dn, ids, table, 0.5, base=base, pair_scale=ps, gated=gated, limit=3.0 if form == "bounded" else 0.0)
    chosen = table[ids.long()] if ids is not None else table
    rnd = lambda t: t.to(bf).double()      # noqa: E731  (stored activations)
    want = base.double()
    for k in range(top):
        for e in range(E):
            mine = (chosen[:, k] == e).nonzero()[:, 0]
            x = h.double()[mine] * (ps.double()[mine, k:k + 1] if ps is not None else 1)
            a = rnd(x @ gu[e, :F].double().T)
            if not gated:
                a = a.clamp(min=0) ** 2
            else:
                u = rnd(x @ gu[e, F:].double().T)
                if form == "bounded":
                    a, u = a.clamp(max=3.0), u.clamp(-3.0, 3.0)
                    a = a * torch.sigmoid(1.702 * a) * (u + 1)
                else:
                    a = a * torch.sigmoid(a) * u
            want[mine] += 0.5 * rnd(a) @ dn[e].double().T
    # the result's own rounding, 2^-9 of it, and an activation of up to 10 (a square: 20) whose rounding falls the other way: 2^-8 of
    # it times the weight of 0.5 and an entry of up to 0.2 of a matrix; all entries together differ by less than one place of eight bits
    diff = got.double() - want
    assert (diff.abs() <= (6e-3 if gated else 1e-2) * (1 + want.abs())).all()
    assert diff.norm() <= 2.0 ** -8 * want.norm()
