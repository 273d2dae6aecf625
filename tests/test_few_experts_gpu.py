"""Experts of few tokens: the kernels that read 16 bytes a load beside those that take any row (the same tokens, off a
16-byte boundary): every output is added up in the same order, so the bits are the same; and against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


# one pair, pairs that all share an expert (more than the four that share a read), as many as a wave has lanes, widths
# below, at and beyond four pieces of 512 (256) entries, odd numbers of outputs a wave
@pytest.mark.parametrize("N,top,E", [(1, 1, 1), (1, 2, 16), (9, 1, 1), (8, 2, 16), (15, 2, 3), (3, 8, 8), (31, 1, 2), (64, 1, 5)])
@pytest.mark.parametrize("W,F", [(8, 8), (520, 264), (2048, 1024), (2056, 16), (24, 1032)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["table", "router", "one matrix", "bounded"])
def test_experts_of_few_tokens(ops, N, top, E, W, F, dtype, form):
    g = torch.Generator().manual_seed(N * 100 + top + W)
    r = lambda *s: torch.randn(*s, generator=g).to("cuda:0")     # noqa: E731
    gated = form != "one matrix"
    gu = (r(E, (2 if gated else 1) * F, W) * W ** -0.5).to(dtype)
    dn = (r(E, W, F) * F ** -0.5).to(dtype)
    h, base = r(N, W).to(dtype), r(N, W).to(dtype)
    identity = 1 if form == "bounded" else 0
    vocab = 11 if form == "table" else N
    table = torch.randint(0, E + identity, (vocab, top), generator=g, dtype=torch.int32).to("cuda:0")
    ids = torch.randint(0, vocab, (N,), generator=g, dtype=torch.int32).to("cuda:0") if form == "table" else None
    ps = r(N, top).abs() if form == "router" else None
    os = r(N, top).abs() if form == "bounded" else None
    bs = r(N) if form == "router" else None
    args = dict(base=base, pair_scale=ps, base_scale=bs, out_scale=os, gated=gated, limit=3.0 if form == "bounded" else 0.0,
                identity=identity)
    got = ops.table_moe(h, gu, dn, ids, table, 0.5, **args)
    off = torch.empty(N * (W + 16) + 1, dtype=dtype, device="cuda:0")[1:].view(N, W + 16)[:, :W]
    off.copy_(h)
    if N * top < 32 or dtype == torch.float32:
        other = ops.table_moe(off, gu, dn, ids, table, 0.5, **args)
        if os is None:
            assert torch.equal(got, other)
        else:       # (a factor on the results may or may not be contracted with their addition: a rounding of a few units)
            step = 2.0 ** -22 if dtype == torch.float32 else 2.0 ** -7
            assert ((got.double() - other.double()).abs() <= step * (8 + other.double().abs())).all()
    hd, want = h.double(), base.double() * (bs.double()[:, None] if bs is not None else 1)
    rnd = lambda t: t.to(dtype).double()      # noqa: E731  (stored activations)
    for n in range(N):
        for k in range(top):
            e = int(table[int(ids[n]) if ids is not None else n, k])
            x = hd[n] * (float(ps[n, k]) if ps is not None else 1)
            if e >= E:
                y = x
            elif not gated:
                y = dn[e].double() @ rnd(rnd(gu[e].double() @ x).clamp(min=0) ** 2)
            else:
                a, u = rnd(gu[e, :F].double() @ x), rnd(gu[e, F:].double() @ x)
                if form == "bounded":
                    a, u = a.clamp(max=3.0), u.clamp(-3.0, 3.0)
                    a = a * torch.sigmoid(1.702 * a) * (u + 1)
                else:
                    a = a * torch.sigmoid(a) * u
                y = dn[e].double() @ rnd(a)
            want[n] += 0.5 * (float(os[n, k]) if os is not None else 1) * y
    # float32: sums of a few thousand products of unit size; bfloat16: activations of up to 10 whose rounding to 2^-9 may fall
    # the other way, and the result's own rounding
    tol = 1e-4 if dtype == torch.float32 else 6e-2
    assert ((got.double() - want).abs() <= tol * (1 + want.abs())).all()


@pytest.mark.parametrize("W,F", [(8, 8), (520, 264), (2048, 1024), (392, 2056)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scaled_results_of_experts_have_the_same_bits(ops, W, F, dtype):
    """Factors on what experts return, experts without matrices among them: rows on and off a 16-byte boundary."""
    g = torch.Generator().manual_seed(W)
    N, top, E = 9, 3, 4
    r = lambda *s: torch.randn(*s, generator=g).to("cuda:0")     # noqa: E731
    gu, dn = (r(E, 2 * F, W) * W ** -0.5).to(dtype), (r(E, W, F) * F ** -0.5).to(dtype)
    h, scale = r(N, W).to(dtype), r(N, top).abs()
    table = torch.randint(0, E + 2, (N, top), generator=g, dtype=torch.int32).to("cuda:0")
    off = torch.empty(N * (W + 16) + 1, dtype=dtype, device="cuda:0")[1:].view(N, W + 16)[:, :W]
    off.copy_(h)
    args = dict(out_scale=scale, limit=3.0, identity=2)
    assert torch.equal(ops.table_moe(h, gu, dn, None, table, 0.5, **args), ops.table_moe(off, gu, dn, None, table, 0.5, **args))


# experts on both sides of the line to those whose rows are shared (786,432 entries), odd pieces of rows
@pytest.mark.parametrize("N,top,E", [(1, 1, 1), (9, 1, 1), (15, 2, 3), (31, 1, 2), (64, 1, 5)])
@pytest.mark.parametrize("W,F", [(1024, 760), (1024, 768), (1032, 776), (392, 2056), (2056, 392)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["table", "router", "one matrix", "bounded"])
def test_experts_about_the_line_to_shared_rows(ops, N, top, E, W, F, dtype, form):
    test_experts_of_few_tokens(ops, N, top, E, W, F, dtype, form)
